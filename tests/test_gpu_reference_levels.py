"""The reference-order solve by levels: worlds whose levels are at the edges of
what one wavefront, one workgroup and each placement of the working set takes."""
import numpy as np
import pytest

import pyoracle as po
from conftest import say
from odemi import scenes as sc

pytestmark = pytest.mark.gpu


def _scene(kind):
    b = sc._Builder()
    b.geom(sc.PLANE, (0.0, 0.0, 1.0, 0.0))
    if kind == "one":                       # one body, 3 rows
        b.sphere_body((0.0, 0.0, 0.499), 0.5, 1.0)
    elif kind == "islands":                 # 70 islands of 3 rows: levels wider than a wavefront takes
        for i in range(70):
            b.sphere_body((1.5 * i, 0.0, 0.499), 0.5, 1.0)
    elif kind == "platform":                # one body with most of the rows: one row per level
        b.box_body((0.0, 0.0, 0.249), (16.0, 16.0, 0.5), 1.0)
        for i in range(25):
            b.box_body((3.0 * (i % 5) - 6.0, 3.0 * (i // 5) - 6.0, 0.997), (1.0, 1.0, 1.0), 1.0)
    else:                                   # a bed of 324 spheres, 2808 rows: wide levels
        for i in range(324):
            b.sphere_body((0.998 * (i % 18), 0.998 * (i // 18), 0.499), 0.5, 1.0)
    s = b.scene(dt=0.01, mu=0.5, seed=77)
    rng = np.random.default_rng(3)
    s.body_lvel = rng.normal(0, 0.2, (s.nb, 3)).astype(np.float32).astype(np.float64)
    s.body_avel = rng.normal(0, 0.2, (s.nb, 3)).astype(np.float32).astype(np.float64)
    return s


@pytest.mark.parametrize("iters", [1, 8, 9, 20])
@pytest.mark.parametrize("kind", ["one", "islands", "platform", "bed"])
def test_levels_keep_the_sequence(odemi_mod, kind, iters):
    """One step equals the restatement's sequential sweep (4x what its single
    and double builds differ by, plus 1e-5 of the fastest body: 20 sweeps of
    sums in 32 bits), with the same bits for every pool and workgroup size."""
    s = _scene(kind)
    s.iterations = iters
    want32, want64 = (po.run(po.oracle_lib(p), s, 1, 1)["traj"][1] for p in ("f32", "f64"))
    tol = 4 * np.abs(want32 - want64).max() + 1e-5 * max(1.0, np.abs(want64[:, 7:]).max())
    first = None
    for wg, lds in ((256, None), (64, None), (256, 0), (64, 4096), (128, 16384), (256, 60000)):
        say("levels", kind, iters, wg, lds)
        b = odemi_mod.Batch([s, s], odemi_mod.ORDER_REFERENCE)
        b.set_launch_config(wg, 1.0, lds)
        b.step(1)
        st = b.state()
        b.close()
        assert np.array_equal(st[:s.nb], st[s.nb:])
        if first is None:
            first = st
            err = np.abs(st[:s.nb] - want32).max()
            say("error", err, "tolerance", tol)
            assert err <= tol
        assert np.array_equal(first, st)
