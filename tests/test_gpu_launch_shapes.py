"""Results do not depend on the launch shape, the placement of a working set in
LDS or the way the state crosses to the host: the same bits on both sides of
each line where one of them changes."""
import numpy as np
import pytest

from conftest import say
from odemi import scenes as sc

pytestmark = pytest.mark.gpu


def _pile(n, seed, spread=1.0):
    """n spheres and boxes in a packed lattice, resting on a plane."""
    rng = np.random.default_rng(seed)
    b = sc._Builder()
    b.geom(sc.PLANE, (0.0, 0.0, 1.0, 0.0))
    side = max(1, int(np.ceil(n ** (1 / 3))))
    for i in range(n):
        x, y, z = i % side, (i // side) % side, i // side ** 2
        p = (0.98 * spread * x, 0.98 * spread * y, 0.49 + 0.98 * z)
        if rng.random() < 0.5:
            b.sphere_body(p, 0.5, 1.0)
        else:
            b.box_body(p, (1.0, 1.0, 1.0), 1.0)
    s = b.scene(dt=0.01, mu=0.5, seed=seed)
    s.body_lvel = rng.normal(0, 0.1, (n, 3)).astype(np.float32).astype(np.float64)
    return s


@pytest.mark.parametrize("order", ["reference", "coloured"])
@pytest.mark.parametrize("worlds", [1, 257, 513, 1025])
def test_default_shape_gives_the_bits_of_256_lanes(odemi_mod, order, worlds):
    """The default shape on both sides of one, two and four worlds per CU, by
    the number of small worlds."""
    o = odemi_mod.ORDER_REFERENCE if order == "reference" else odemi_mod.ORDER_COLORED
    base = [_pile(n, n) for n in ((30,) if worlds == 1 else (1, 3, 9, 20, 27))]
    ws = [base[w % len(base)] for w in range(worlds)]
    out = []
    for fixed in (False, True):
        b = odemi_mod.Batch(ws, o)
        if fixed:
            b.set_launch_config(256, 1.0)
        say("shape", order, worlds, b.launch_config()["wg"])
        b.step(3)
        out.append(b.state())
        b.close()
    assert np.array_equal(out[0], out[1])


def test_wide_coloured_world(odemi_mod):
    """512 lanes (the default of a large coloured world) and 256: colours stay
    capped at 256, in every placement of the bodies' colouring state and of the
    solver's (fixed sweeps)."""
    s = _pile(2200, 5)
    out = []
    for lds in ("default", None, 60000, 20000, 0):
        b = odemi_mod.Batch([s], odemi_mod.ORDER_COLORED)
        if lds != "default":
            b.set_launch_config(256, 1.0, lds)
        say("wide", lds, b.launch_config()["wg"])
        b.step(2)
        out.append((b.state(), b.counters()["groups"]))
        b.close()
    for st, g in out[1:]:
        assert g == out[0][1]
        assert np.array_equal(st, out[0][0])


@pytest.mark.parametrize("n", [1, 2, 12])
def test_exact_lcp_placements_agree(odemi_mod, n):
    """An island's workspace in LDS, all but its matrix, and in global memory."""
    ws = [sc.box_stack(n, gap=-1e-3, seed=n), _pile(n, n, spread=1.5)]
    out = []
    for wg, lds in ((256, None), (64, 60000), (256, 30000), (128, 8192), (256, 0)):
        say("exact", n, wg, lds)
        b = odemi_mod.Batch(ws, odemi_mod.ORDER_REFERENCE)
        b.set_launch_config(wg, 1.0, lds)
        b.set_exact_lcp(15 * n + 15)
        b.step(2)
        assert b.counters()["overflow"] == 0
        out.append(b.state())
        b.close()
    for st in out[1:]:
        assert np.array_equal(st, out[0])


@pytest.mark.parametrize("n", [1, 100, 20200])
def test_state_crosses_unchanged(odemi_mod, n):
    """set_state / state below and above the size that goes through pinned
    memory (1 MB: 20 164 bodies), and a step from a state that was set."""
    b1 = sc._Builder()
    b1.geom(sc.PLANE, (0.0, 0.0, 1.0, 0.0))
    per = min(n, 101)
    for i in range(per):
        b1.sphere_body((2.0 * i, 0.0, 1.0), 0.5, 1.0)
    s = b1.scene(dt=0.01, mu=0.5, seed=1)
    say("state", n)
    a, b = (odemi_mod.Batch([s] * (n // per), odemi_mod.ORDER_COLORED) for _ in range(2))
    st = a.state()
    rng = np.random.default_rng(n)
    q = rng.normal(0, 1, (len(st), 4))
    st[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
    st[:, 7:] = rng.normal(0, 1, (len(st), 6))
    for x in (a, b):
        x.set_state(st)
        assert np.array_equal(x.state(), st)
    a.step(2)
    b.step(1)
    b.set_state(b.state())
    b.step(1)
    assert np.array_equal(a.state(), b.state())


@pytest.mark.parametrize("order", ["reference", "coloured"])
@pytest.mark.parametrize("worlds,bodies", [(1, 30), (1, 2200), (257, 9), (1025, 9)])
def test_a_shape_that_is_read_can_be_set(odemi_mod, order, worlds, bodies):
    """What launch_config() gives is accepted, with and without its pool and
    grid, stays, and is the same shape."""
    o = odemi_mod.ORDER_REFERENCE if order == "reference" else odemi_mod.ORDER_COLORED
    ws = [_pile(bodies, 3)] * worlds
    out = []
    for again in (None, "all", "width"):
        b = odemi_mod.Batch(ws, o)
        c = b.launch_config()
        say("read and set", order, worlds, bodies, again, c)
        if again == "all":
            b.set_launch_config(c["wg"], c["cell_scale"], c["lds"], grid=c["grid"])
        elif again:
            b.set_launch_config(c["wg"], c["cell_scale"])
        assert b.launch_config() == c
        b.step(1)
        out.append(b.state())
        b.close()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


@pytest.mark.parametrize("wg", [0, 32, 320, 384, 1024])
def test_other_widths_are_refused(odemi_mod, wg):
    b = odemi_mod.Batch([_pile(2, 1)], odemi_mod.ORDER_REFERENCE)
    c = b.launch_config()
    with pytest.raises(RuntimeError):
        b.set_launch_config(wg, 1.0)
    assert b.launch_config() == c


def test_widest_workgroup_at_a_tolerance(odemi_mod):
    """512 lanes set by hand while iterating to a tolerance, which takes 256 by
    itself.  A bed of touching spheres (a pile of boxes has no single solution
    and does not converge): forces within a few hundred times the residual of
    1e-5 of the solution, so velocities within 1e-4 (dt = 0.01, mass 1)."""
    b = sc._Builder()
    b.geom(sc.PLANE, (0.0, 0.0, 1.0, 0.0))
    for i in range(324):
        b.sphere_body((0.998 * (i % 18), 0.998 * (i // 18), 0.499), 0.5, 1.0)
    s = b.scene(dt=0.01, mu=0.5, seed=4)
    s.body_lvel = np.random.default_rng(4).normal(0, 0.05, (324, 3)).astype(np.float32).astype(np.float64)
    out = []
    for wg in (256, 512):
        b = odemi_mod.Batch([s], odemi_mod.ORDER_COLORED)
        b.set_tolerance(1e-5, 100000, 10, accel=True)
        assert b.launch_config()["wg"] == 256
        b.set_launch_config(wg, 1.0, 65536)
        say("tolerance", wg)
        b.step(1)
        unconverged, residual = b.solve_stats()
        out.append(b.state())
        say("residual", residual[0], "sweeps", b.world_counters()[0, 5], "differs", np.abs(out[0] - out[-1]).max())
        assert unconverged[0] == 0 and residual[0] <= 1e-5
        b.close()
    assert np.abs(out[0] - out[1]).max() <= 1e-4


@pytest.mark.parametrize("keep_cell", [False, True])
def test_tuning_is_not_slower_than_the_default(odemi_mod, keep_cell):
    """One large world in the reference order, whose default is the widest
    workgroup: the tuned shape is the default or a faster one (fastest of 12
    steps; the runs of one shape differ by about 2 %)."""
    s = _pile(1400, 11)
    ms = []
    for tuned in (False, True):
        b = odemi_mod.Batch([s], odemi_mod.ORDER_REFERENCE)
        if tuned:
            b.autotune(2, keep_cell=keep_cell)
        b.step(2)
        st = b.state()
        times = []
        for _ in range(12):
            b.set_state(st)
            times.append(b.step_timed(1))
        ms.append(min(times))
        say("tuned" if tuned else "default", b.launch_config(), ms[-1])
        b.close()
    assert ms[1] <= 1.1 * ms[0]


@pytest.mark.parametrize("worlds", [1, 300, 600, 1100])
def test_pool_and_tolerance_in_either_order(odemi_mod, worlds):
    """A pool set by hand leaves the width to the solver mode, whichever is set
    first: 256 lanes at a tolerance, and the same bits."""
    base = [_pile(n, n) for n in (1, 9, 20, 27)]
    ws = [base[w % len(base)] for w in range(worlds)]
    out = []
    for first in ("pool", "tolerance"):
        b = odemi_mod.Batch(ws, odemi_mod.ORDER_COLORED)
        for what in (first, "tolerance" if first == "pool" else "pool"):
            if what == "pool":
                b.L.dBatchSetLds(b.h, 40960)
            else:
                b.set_tolerance(1e-5, 400, 10, accel=True)
        say("pool and tolerance", worlds, first, b.launch_config())
        assert b.launch_config()["wg"] == 256 and b.launch_config()["lds"] == 40960
        b.step(2)
        out.append(b.state())
        b.close()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("bodies,worlds,wg", [(64, 1025, 64), (65, 1025, 128), (128, 513, 128), (129, 513, 256)])
def test_narrow_workgroups_hold_a_whole_colour(odemi_mod, bodies, worlds, wg):
    """Coloured order: the largest world at the width's bound, all its bodies
    apart on a plane, so that one colour has a constraint of every body; the
    bits and colours of 256 lanes."""
    def spheres(n):
        b = sc._Builder()
        b.geom(sc.PLANE, (0.0, 0.0, 1.0, 0.0))
        for i in range(n):
            b.sphere_body((1.5 * (i % 12), 1.5 * (i // 12), 0.49), 0.5, 1.0)
        s = b.scene(dt=0.01, mu=0.5, seed=n)
        s.body_lvel = np.random.default_rng(n).normal(0, 0.2, (n, 3)).astype(np.float32).astype(np.float64)
        s.body_lvel[:, 2] = 0
        return s
    ws = [spheres(bodies)] + [spheres(3)] * (worlds - 1)
    out = []
    for fixed in (False, True):
        b = odemi_mod.Batch(ws, odemi_mod.ORDER_COLORED)
        if fixed:
            b.set_launch_config(256, 1.0)
        else:
            assert b.launch_config()["wg"] == wg
        say("whole colour", bodies, worlds, b.launch_config()["wg"])
        b.step(1)
        wc = b.world_counters()
        assert wc[0, 1] == bodies and wc[0, 3] == 1
        b.step(2)
        out.append((b.state(), wc[:, 3]))
        b.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


def test_scratch_is_the_batches_orders(odemi_mod):
    """The solver's working set of a world is sized for the batch's order (a
    row takes 200 bytes of it in the reference order and 108 in the coloured):
    512 worlds of 64 bodies and 1474 rows' room differ by 68 MB."""
    import torch
    say("scratch")
    ws = [_pile(64, 2)] * 512
    used = []
    for o in (odemi_mod.ORDER_COLORED, odemi_mod.ORDER_REFERENCE):
        odemi_mod.Batch(ws[:1], o).close()
        before = torch.cuda.mem_get_info()[0]
        b = odemi_mod.Batch(ws, o)
        used.append(before - torch.cuda.mem_get_info()[0])
        b.close()
    say("bytes", used)
    assert used[0] < used[1] - (48 << 20)


@pytest.mark.parametrize("worlds,lds,wg", [(1, 1024, 512), (600, 4096, 128), (600, 49152, 256), (1100, 16384, 64),
                                           (1100, 32768, 128), (1100, 65536, 256)])
def test_width_that_goes_with_a_pool(odemi_mod, worlds, lds, wg):
    """A pool set by hand takes the narrow workgroups of which a CU has room
    for four (128 lanes) or eight (64); the bits are those of 256 lanes."""
    base = [_pile(n, n) for n in (9, 20, 27)]
    ws = [base[w % 3] for w in range(worlds)]
    out = []
    for fixed in (False, True):
        b = odemi_mod.Batch(ws, odemi_mod.ORDER_REFERENCE)
        if fixed:
            b.set_launch_config(256, 1.0, lds)
        else:
            b.L.dBatchSetLds(b.h, lds)
        c = b.launch_config()
        say("width and pool", worlds, c)
        assert (c["wg"], c["lds"]) == (256 if fixed else wg, lds)
        b.step(2)
        out.append(b.state())
        b.close()
    assert np.array_equal(out[0], out[1])
