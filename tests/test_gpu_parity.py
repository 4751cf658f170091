"""Parity of the HIP path against the reference (golden fixtures written from
the reference double build) and the CPU restatement, through the C ABI.

Tolerances (FP32 device arithmetic against the FP64 reference):
* pair sets, pair order and contact counts: exact;
* contact position/normal/depth: |a-b| <= 2e-5 * max(1, |b|);
* contact impulses of one step from the same state: |f-g| <= 2e-3 * max(1, |g|);
* trajectories: within 4x the distance between the reference's own
  single-precision build and its double build at the same step, plus 1e-3 m.
"""
import ctypes as C
import math
import os

import numpy as np
import pytest

import pyoracle as po
from conftest import ROOT, golden, say
from odemi import scenes

pytestmark = pytest.mark.gpu




# ------------------------------------------------------------------ narrowphase

class Api:
    """ctypes view of the ODE API subset of libodemi.so."""

    def __init__(self):
        import odemi
        L = odemi.lib()
        V, F = C.c_void_p, C.c_float
        for name, res, args in [
            ("dCreateBox", V, [V, F, F, F]), ("dCreateSphere", V, [V, F]), ("dCreatePlane", V, [V, F, F, F, F]),
            ("dCreateCapsule", V, [V, F, F]), ("dCreateRay", V, [V, F]), ("dCreateCylinder", V, [V, F, F]),
            ("dGeomSetPosition", None, [V, F, F, F]), ("dGeomSetRotation", None, [V, C.POINTER(F)]),
            ("dCollide", C.c_int, [V, V, C.c_int, V, C.c_int]), ("dGeomDestroy", None, [V])]:
            f = getattr(L, name)
            f.restype = res
            f.argtypes = args
        self.L = L

    def geom(self, t, prm, p, R4):
        L = self.L
        if t == 0:
            g = L.dCreateSphere(None, prm[0])
        elif t == 1:
            g = L.dCreateBox(None, prm[0], prm[1], prm[2])
        elif t == 3:
            g = L.dCreateCapsule(None, prm[0], prm[1])
        elif t == 4:
            g = L.dCreateRay(None, prm[0])
        elif t == 5:
            g = L.dCreateCylinder(None, prm[0], prm[1])
        else:
            return L.dCreatePlane(None, *prm)
        L.dGeomSetPosition(g, *p)
        R = (C.c_float * 12)(*R4)
        L.dGeomSetRotation(g, R)
        return g

    def collide(self, g1, g2, maxc):
        buf = (C.c_byte * (64 * maxc))()
        n = self.L.dCollide(g1, g2, maxc, buf, 64)
        raw = np.frombuffer(bytes(buf), dtype=np.float32).reshape(maxc, 16)[:n]
        return np.concatenate([raw[:, 0:3], raw[:, 4:7], raw[:, 8:9]], axis=1)


def _rot(q):
    w, x, y, z = q / np.linalg.norm(q)
    R = np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)],
                  [2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)],
                  [2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)]])
    R4 = np.zeros((3, 4))
    R4[:, :3] = R
    return R4.reshape(12)


def test_narrowphase_pairs_vs_oracle(odemi_mod):
    from test_oracle_pins import collide as orc_collide
    api = Api()
    rng = np.random.default_rng(11)
    combos = [(0, 0), (0, 1), (1, 0), (0, 2), (2, 0), (1, 1), (1, 2), (2, 1)]
    n_cmp = n_disc = 0
    for t1, t2 in combos:
        say("narrowphase case", t1, t2)
        for trial in range(60):
            def shape(t):
                if t == 0:
                    return [rng.uniform(0.1, 0.6), 0, 0, 0]
                if t == 1:
                    return [*rng.uniform(0.2, 1.2, 3), 0]
                n = rng.normal(size=3)
                n /= np.linalg.norm(n)
                return [*n, rng.uniform(-0.3, 0.3)]
            s1, s2 = shape(t1), shape(t2)
            q1, q2 = rng.normal(size=4), rng.normal(size=4)
            p1, p2 = rng.uniform(-0.4, 0.4, 3), rng.uniform(-0.4, 0.4, 3)
            if t1 == 2:
                p1 = np.zeros(3); q1 = np.array([1.0, 0, 0, 0])
            if t2 == 2:
                p2 = np.zeros(3); q2 = np.array([1.0, 0, 0, 0])
            maxc = 4
            g1 = api.geom(t1, s1, p1, _rot(q1))
            g2 = api.geom(t2, s2, p2, _rot(q2))
            got = api.collide(g1, g2, maxc)
            api.L.dGeomDestroy(g1)
            api.L.dGeomDestroy(g2)
            ref32 = orc_collide(t1, p1, q1, s1, t2, p2, q2, s2, maxc, prec="f32")
            ref64 = orc_collide(t1, p1, q1, s1, t2, p2, q2, s2, maxc, prec="f64")
            if len(ref32) != len(ref64):
                n_disc += 1      # a precision tie: the decision flips between f32 and f64
                continue
            assert len(got) == len(ref64), (t1, t2, trial, got, ref64)
            if len(got):
                # 1e-5 relative, widened to 4x the reference FP32 build's own
                # error on the same case (ill-conditioned normals of nearly
                # touching shapes)
                scale = np.maximum(1.0, np.abs(ref64))
                err = np.abs(got - ref64) / scale
                e32 = np.abs(ref32 - ref64) / scale
                tol = max(1e-5, 4.0 * float(e32.max()))
                assert err.max() <= tol, (t1, t2, trial, err.max(), tol)
                n_cmp += 1
    say("narrowphase compared", n_cmp, "precision ties skipped", n_disc)
    assert n_cmp > 150 and n_disc < 10


def test_capsule_narrowphase_vs_oracle(odemi_mod):
    """The four capsule colliders (capsule-sphere, -box, -capsule, -plane,
    capsule.cpp:130-409) through dCollide on random overlapping poses, both
    argument orders, including capsules with parallel axes (the two-contact
    branch), against the restatement: the bar of the narrowphase test above."""
    from test_oracle_pins import collide as orc_collide
    api = Api()
    rng = np.random.default_rng(17)
    combos = [(3, 0), (0, 3), (3, 1), (1, 3), (3, 3), (3, 2), (2, 3)]
    n_cmp = n_disc = n_two = 0
    for t1, t2 in combos:
        say("capsule narrowphase case", t1, t2)
        for trial in range(60):
            def shape(t):
                if t == 0:
                    return [rng.uniform(0.1, 0.6), 0, 0, 0]
                if t == 1:
                    return [*rng.uniform(0.2, 1.2, 3), 0]
                if t == 3:
                    return [rng.uniform(0.1, 0.4), rng.uniform(0.2, 1.0), 0, 0]
                n = rng.normal(size=3)
                n /= np.linalg.norm(n)
                return [*n, rng.uniform(-0.3, 0.3)]
            s1, s2 = shape(t1), shape(t2)
            q1, q2 = rng.normal(size=4), rng.normal(size=4)
            if t1 == 3 and t2 == 3 and trial % 3 == 0:
                q2 = q1.copy() * (1 if trial % 2 else -1)   # parallel or antiparallel axes
            p1, p2 = rng.uniform(-0.4, 0.4, 3), rng.uniform(-0.4, 0.4, 3)
            if t1 == 2:
                p1 = np.zeros(3); q1 = np.array([1.0, 0, 0, 0])
            if t2 == 2:
                p2 = np.zeros(3); q2 = np.array([1.0, 0, 0, 0])
            maxc = 4
            g1 = api.geom(t1, s1, p1, _rot(q1))
            g2 = api.geom(t2, s2, p2, _rot(q2))
            got = api.collide(g1, g2, maxc)
            api.L.dGeomDestroy(g1)
            api.L.dGeomDestroy(g2)
            ref32 = orc_collide(t1, p1, q1, s1, t2, p2, q2, s2, maxc, prec="f32")
            ref64 = orc_collide(t1, p1, q1, s1, t2, p2, q2, s2, maxc, prec="f64")
            if len(ref32) != len(ref64):
                n_disc += 1
                continue
            assert len(got) == len(ref64), (t1, t2, trial, got, ref64)
            if len(got):
                scale = np.maximum(1.0, np.abs(ref64))
                err = np.abs(got - ref64) / scale
                e32 = np.abs(ref32 - ref64) / scale
                tol = max(1e-5, 4.0 * float(e32.max()))
                assert err.max() <= tol, (t1, t2, trial, err.max(), tol)
                n_cmp += 1
                n_two += int(len(got) == 2 and t1 == 3 and t2 == 3)
    say("capsule narrowphase compared", n_cmp, "two-contact capsule pairs", n_two, "precision ties skipped", n_disc)
    assert n_cmp > 150 and n_two > 0 and n_disc < 10


def test_ray_narrowphase_vs_reference_fixture(odemi_mod):
    """The ray colliders (ray-sphere, -box, -capsule, -plane in both argument
    orders, ray.cpp:196-497) through dCollide on the reference's own cases
    (tests/golden/rays.npz, from its double build): the same hit or miss and
    the contact within the FP32 envelope, except where the restatement in
    FP32 and in FP64 disagree on hit or miss (a ray grazing a surface or
    ending on it)."""
    from test_oracle_pins import _case, _ray_fixture, collide as orc_collide
    api = Api()
    cases, count, contacts = _ray_fixture()
    n_cmp = n_tie = 0
    say("ray narrowphase cases", len(cases))
    for i, row in enumerate(cases):
        t1, p1, q1, s1, t2, p2, q2, s2 = _case(row)
        g1 = api.geom(t1, s1, p1, _rot(q1))
        g2 = api.geom(t2, s2, p2, _rot(q2))
        got = api.collide(g1, g2, 4)
        api.L.dGeomDestroy(g1)
        api.L.dGeomDestroy(g2)
        ref32 = orc_collide(t1, p1, q1, s1, t2, p2, q2, s2, 4, prec="f32")
        if len(ref32) != count[i]:
            # rays exactly parallel to a capsule's axis from inside it: the
            # quadratic's leading term is a rounding residue in FP64 (a miss)
            # and exactly zero in FP32 (the end cap is hit)
            assert len(got) in (len(ref32), count[i]), (i, t1, t2, got)
            n_tie += 1
            continue
        assert len(got) == count[i], (i, t1, t2, got, contacts[i])
        if count[i]:
            scale = np.maximum(1.0, np.abs(contacts[i]))
            err = np.abs(got[0] - contacts[i]) / scale
            e32 = np.abs(ref32[0] - contacts[i]) / scale
            assert err.max() <= max(1e-5, 4.0 * float(e32.max())), (i, t1, t2, err.max(), e32.max())
            n_cmp += 1
    say("ray contacts compared", n_cmp, "precision ties skipped", n_tie)
    assert n_cmp > 300 and n_tie < 16


def test_cylinder_narrowphase_vs_reference_fixture(odemi_mod):
    """The cylinder colliders (cylinder-sphere, -plane, -box, ray-cylinder,
    both argument orders, maxc 1-8; cylinder-cylinder and capsule-cylinder
    without a collider) through dCollide on the reference's own cases
    (tests/golden/cylinder_colliders.npz, from its double build): the same number of
    contacts, and contacts within 4x the restatement's FP32 distance from the
    reference (at least 1e-5 relative), except where the restatement in FP32
    and the reference disagree on the count (a feature at a tolerance
    boundary)."""
    from test_oracle_pins import _cyl_case, _cyl_fixture, collide as orc_collide
    api = Api()
    cases, count, contacts = _cyl_fixture()
    n_cmp = n_tie = n_many = n_face_tie = n_face_off = 0
    say("cylinder narrowphase cases", len(cases))
    for i, row in enumerate(cases):
        t1, p1, q1, s1, t2, p2, q2, s2, maxc = _cyl_case(row)
        g1 = api.geom(t1, s1, p1, _rot(q1))
        g2 = api.geom(t2, s2, p2, _rot(q2))
        got = api.collide(g1, g2, maxc)
        api.L.dGeomDestroy(g1)
        api.L.dGeomDestroy(g2)
        ref32 = orc_collide(t1, p1, q1, s1, t2, p2, q2, s2, maxc, prec="f32")
        if len(ref32) != count[i]:
            assert len(got) in (len(ref32), count[i]), (i, t1, t2, got)
            n_tie += 1
            continue
        assert len(got) == count[i], (i, t1, t2, maxc, got, contacts[i, :count[i]])
        if count[i]:
            ref = contacts[i, :count[i]]
            scale = np.maximum(1.0, np.abs(ref))
            err = float((np.abs(got - ref) / scale).max())
            e32 = float((np.abs(ref32 - ref) / scale).max())
            if e32 < 1e-4:
                assert err <= max(1e-5, 4.0 * e32), (i, t1, t2, err, e32)
            else:
                # a disc resting on a box face: separating axes of equal depth
                # in exact arithmetic, the winner set by rounding (FP32 and
                # FP64 pick different faces); the device must agree with one
                # of the two
                e_dev32 = float((np.abs(got - ref32) / scale).max())
                n_face_tie += 1
                n_face_off += int(min(err, e_dev32) > 1e-3)
            n_cmp += 1
            n_many += int(count[i] > 2)
    say("cylinder contacts compared", n_cmp, "cases with more than two contacts", n_many, "count ties", n_tie,
        "face ties", n_face_tie, "of them matching neither precision", n_face_off)
    assert n_cmp > 800 and n_many > 50 and n_tie < 30 and n_face_off <= max(2, n_face_tie // 10)


def test_dcollide_refusals_match_the_reference(odemi_mod):
    """dCollide returns 0 for a request of no contacts, a geom against itself
    and two geoms on one body (collision_kernel.cpp:306-311); the flag bits
    above the contact count (CONTACTS_UNIMPORTANT) do not change the count."""
    say("dCollide refusals")
    api = Api()
    L = api.L
    V, F = C.c_void_p, C.c_float
    for name, res, args in [("dWorldCreate", V, []), ("dWorldDestroy", None, [V]), ("dBodyCreate", V, [V]),
                            ("dBodySetPosition", None, [V, F, F, F]), ("dGeomSetBody", None, [V, V])]:
        f = getattr(L, name)
        f.restype = res
        f.argtypes = args
    R0 = _rot(np.array([1.0, 0, 0, 0]))
    s1 = api.geom(0, [0.5, 0, 0, 0], np.zeros(3), R0)
    s2 = api.geom(0, [0.5, 0, 0, 0], np.array([0.6, 0, 0]), R0)
    assert len(api.collide(s1, s2, 1)) == 1
    buf = (C.c_byte * 256)()
    assert L.dCollide(s1, s2, 0, buf, 64) == 0
    assert L.dCollide(s1, s2, 0x80000000 | 4, buf, 64) == 1
    assert L.dCollide(s1, s1, 4, buf, 64) == 0
    w = L.dWorldCreate()
    body = L.dBodyCreate(w)
    L.dGeomSetBody(s1, body)
    L.dGeomSetBody(s2, body)
    assert L.dCollide(s1, s2, 4, buf, 64) == 0
    L.dGeomDestroy(s1)
    L.dGeomDestroy(s2)
    L.dWorldDestroy(w)


# ------------------------------------------------------------------ broadphase + contacts


def _batch(odemi_mod, scs, order=None):
    return odemi_mod.Batch(scs, odemi_mod.ORDER_REFERENCE if order is None else order)


@pytest.mark.parametrize("name", ["pile4096", "pile256_dense", "chains", "vehicle", "surfaces", "capsules",
                                  "cylinders"])
def test_first_step_pairs_and_contacts_match_reference(odemi_mod, name):
    say("first-step parity", name)
    from test_golden import CASES
    sc = CASES[name][0]()
    g = golden(name)
    b = _batch(odemi_mod, [sc])
    if sc.step_ctrl is not None:
        b.set_controls(sc.step_ctrl[0])
    b.step(1)
    n0 = int(g["pair_step_count"][0])
    k0 = int(g["contact_step_count"][0])
    pairs = b.pairs(0)
    assert np.array_equal(pairs, g["pairs"][:n0]), "pair order/set differs from the reference"
    con = b.contacts(0)
    assert len(con) == k0
    ref = g["contacts"][:k0]
    if k0:
        assert np.array_equal(con[:, 7:9].astype(int), ref[:, 7:9].astype(int))
        con, nre = _match_within_pairs(con, ref)
        err = np.abs(con[:, :7] - ref[:, :7]) / np.maximum(1.0, np.abs(ref[:, :7]))
        say(name, "pairs", n0, "contacts", k0, "max rel err", float(err.max()), "reordered ties", nre)
        assert err.max() <= 2e-5
    assert b.counters()["overflow"] == 0


@pytest.mark.parametrize("wg,lds", [(256, 8192), (64, 2048), (128, 0)])
def test_broadphase_sort_paths_keep_reference_pair_order(odemi_mod, wg, lds):
    """The 4096-body pile's first-step pairs with small LDS pools: cell keys
    and pair keys sorted by the block radix sort in global memory (pools of
    8 KB and 2 KB), or by the bitonic sort in global memory (no pool); the
    pair order must stay the reference's, bit for bit."""
    say("broadphase sort path", wg, lds)
    from test_golden import CASES
    sc = CASES["pile4096"][0]()
    g = golden("pile4096")
    b = _batch(odemi_mod, [sc])
    b.set_launch_config(wg, 1.0, lds)
    b.step(1)
    n0 = int(g["pair_step_count"][0])
    assert np.array_equal(b.pairs(0), g["pairs"][:n0])
    assert b.counters()["contacts"] == int(g["contact_step_count"][0])


def _match_within_pairs(con, ref):
    """Contacts of one pair whose depths tie (a box resting flat on a plane:
    its four lowest vertices) come out in an order decided by the last bit of
    the face projections; match such contacts by position within their pair
    before comparing.  Returns the reordered GPU contacts and the number of
    contacts that moved."""
    out = con.copy()
    moved = 0
    i = 0
    n = len(ref)
    while i < n:
        j = i
        while j < n and ref[j, 7] == ref[i, 7] and ref[j, 8] == ref[i, 8]:
            j += 1
        if j - i > 1:
            used = set()
            for a in range(i, j):
                d = [np.abs(con[c, :3] - ref[a, :3]).max() if c not in used else np.inf for c in range(i, j)]
                c = i + int(np.argmin(d))
                used.add(c)
                out[a] = con[c]
                moved += int(c != a)
        i = j
    return out, moved


def _plane_space(n):
    if abs(n[2]) > math.sqrt(0.5):
        a = n[1] ** 2 + n[2] ** 2
        k = 1 / math.sqrt(a)
        p = np.array([0, -n[2] * k, n[1] * k])
        q = np.array([a * k, -n[0] * p[2], n[0] * p[1]])
    else:
        a = n[0] ** 2 + n[1] ** 2
        k = 1 / math.sqrt(a)
        p = np.array([-n[1] * k, n[0] * k, 0])
        q = np.array([-n[2] * p[1], n[2] * p[0], a * k])
    return p, q


@pytest.mark.parametrize("name", ["pile4096", "chains"])
def test_first_step_contact_impulses_match_reference(odemi_mod, name):
    say("impulse parity", name)
    from test_golden import CASES
    sc = CASES[name][0]()
    g = golden(name)
    b = _batch(odemi_mod, [sc])
    b.step(1)
    con = b.contacts(0)
    k0 = int(g["contact_step_count"][0])
    fb = g["feedback"][:k0]
    if k0 == 0:
        pytest.skip("no contacts in the first step")
    # force on body 1 of each contact joint: J_l1^T lambda = n l0 + t1 l1 + t2 l2
    f = np.zeros((k0, 3))
    bodies = sc.geom_body
    for i, c in enumerate(con):
        n = c[3:6].astype(np.float64)
        g1 = int(c[7])
        if bodies[g1] < 0:
            n = -n   # contact attached with the static geom first: reversed
        t1, t2 = _plane_space(n)
        f[i] = n * c[9] + t1 * c[10] + t2 * c[11]
    scale = np.maximum(1.0, np.abs(fb[:, :3]).max())
    err = np.abs(f - fb[:, :3]).max() / scale
    say(name, "contacts", k0, "max impulse err (rel to max force)", float(err))
    assert err <= 2e-3


def _envelope(sc, n, every):
    """Distance of the reference's own FP32 build from its FP64 build."""
    a = po.run(po.oracle_lib("f64"), sc, n, every)["traj"]
    b = po.run(po.oracle_lib("f32"), sc, n, every)["traj"]
    return np.abs(a[:, :, :3] - b[:, :, :3]).max(axis=(1, 2))


@pytest.mark.parametrize("name", ["box_stack", "chains", "vehicle", "chains200", "vehicle200", "joints", "surfaces",
                                  "frictionless", "capsules", "cylinders"])
def test_trajectory_within_fp32_envelope(odemi_mod, name):
    say("trajectory", name)
    from test_golden import CASES
    fac, n, every, _ = CASES[name]
    sc = fac()
    g = golden(name)
    env = _envelope(sc, n, every)
    b = _batch(odemi_mod, [sc])
    worst = 0.0
    for k in range(n // every):
        for s in range(every):
            if sc.step_ctrl is not None:
                b.set_controls(sc.step_ctrl[k * every + s])
            b.step(1)
        st = b.state()
        err = float(np.abs(st[:, :3] - g["traj"][k + 1][:, :3]).max())
        tol = 4 * env[k + 1] + 1e-3
        worst = max(worst, err / tol)
        assert err <= tol, (name, k, err, env[k + 1])
    say(name, "worst err/tol", worst)


def test_dropin_driver_runs_the_reference_frame_loop(odemi_mod):
    """The unchanged ODE-API application (oracle/scene_driver.cpp) linked
    against libodemi.so: callback pair order, contacts and trajectories."""
    say("drop-in driver")
    lib = po.load(os.path.join(ROOT, "tests", "_build", "libscene_odemi.so"))
    assert lib.scene_dreal_size() == 4
    for name in ("box_stack", "vehicle"):
        from test_golden import CASES
        fac, n, every, diag = CASES[name]
        sc = fac()
        n = min(n, 60)
        g = golden(name)
        r = po.run(lib, sc, n, every, diag_steps=min(diag, 5), max_pairs=100000, max_contacts=100000,
                   feedback=True)
        np_ = int(g["pair_step_count"][:5].sum())
        assert np.array_equal(r["pairs"], g["pairs"][:np_]), name
        env = _envelope(sc, n, every)
        err = np.abs(r["traj"][:, :, :3] - g["traj"][: n // every + 1, :, :3]).max(axis=(1, 2))
        say(name, "drop-in traj err", err.max())
        assert np.all(err <= 4 * env + 1e-3)


@pytest.mark.parametrize("name", ["box_stack_ws", "chains_ws", "vehicle_ws", "joints_ws"])
def test_dropin_world_step_matches_reference(odemi_mod, name):
    """dWorldStep through the unchanged ODE-API application linked against
    libodemi.so (each island's LCP solved exactly on the device) against the
    reference double build's dWorldStep (Dantzig's LCP solver, lcp.cpp):
    every step's callback pairs bit-exact; trajectories within 4x the FP32
    restatement's distance from the reference + 1e-3 m; the contact joints'
    feedback summed per geom pair on every diagnostic step within 4x the
    FP32 restatement's distance + 2e-3 of the step's largest force."""
    say("drop-in dWorldStep", name)
    from test_golden import CASES
    fac, n, every, diag = CASES[name]
    sc = fac()
    g = golden(name)
    lib = po.load(os.path.join(ROOT, "tests", "_build", "libscene_odemi.so"))
    kw = dict(diag_steps=diag, max_pairs=400000, max_contacts=400000, feedback=True)
    r = po.run(lib, sc, n, every, **kw)
    assert r["status"] == 0
    r32 = po.run(po.oracle_lib("f32"), sc, n, every, **kw)
    if not np.array_equal(r32["pairs"], g["pairs"]):
        # an AABB pair touching exactly at the boundary (the joint zoo's
        # first steps) is reported one step later in FP32 than in FP64, by
        # the FP32 restatement too: only the trajectories are compared
        say(name, "pair sets differ in FP32 (boundary touch); trajectories only")
        diag = 0
    else:
        assert np.array_equal(r["pair_step_count"], g["pair_step_count"])
        assert np.array_equal(r["pairs"], g["pairs"])
        assert np.array_equal(r["contact_step_count"], g["contact_step_count"])
    env = np.abs(r32["traj"][:, :, :3] - g["traj"][:, :, :3]).max(axis=(1, 2))
    err = np.abs(r["traj"][:, :, :3] - g["traj"][:, :, :3]).max(axis=(1, 2))
    say(name, "traj err", float(err.max()), "FP32 envelope", float(env.max()))
    assert np.all(err <= 4 * env + 1e-3)
    k0 = np.concatenate([[0], np.cumsum(g["contact_step_count"])])
    worst = 0.0
    same32 = np.array_equal(r32["contact_step_count"], g["contact_step_count"])
    for s in range(diag):
        if k0[s + 1] == k0[s] or not same32:
            continue
        ref = g["contacts"][k0[s]:k0[s + 1]]
        perm = _tie_order(r["contacts"][k0[s]:k0[s + 1]], ref)
        p32 = _tie_order(r32["contacts"][k0[s]:k0[s + 1]], ref)
        fref = g["feedback"][k0[s]:k0[s + 1]]
        # per geom pair: the sum over its contacts (boxes resting on four
        # coplanar contacts split their load as FP32 rounding decides -- the
        # matrix is singular up to cfm along those directions -- while the
        # sum is determined)
        keys = ref[:, 7] * 100003 + ref[:, 8]
        _, grp = np.unique(keys, return_inverse=True)
        def pair_sum(f):
            out = np.zeros((grp.max() + 1, f.shape[1]))
            np.add.at(out, grp, f)
            return out
        fg = pair_sum(r["feedback"][k0[s]:k0[s + 1]][perm])
        f32 = pair_sum(r32["feedback"][k0[s]:k0[s + 1]][p32])
        fr = pair_sum(fref)
        fe = float(np.abs(fg - fr).max())
        env_f = float(np.abs(f32 - fr).max())
        tol = 4 * env_f + 2e-3 * max(1.0, float(np.abs(fr).max()))
        worst = max(worst, fe / tol)
        assert fe <= tol, (name, s, fe, env_f)
    say(name, "feedback (per pair) worst err/tol", worst)


def test_batch_exact_lcp_matches_world_step(odemi_mod):
    """dBatchSetExactLCP: the box stack, chains in a pile and the vehicle
    (per-step controls) stepped together in one batch with each island's LCP
    solved exactly -- the batch form of dWorldStep -- against the reference
    double build's dWorldStep fixtures: trajectories within 4x the FP32
    restatement's distance + 1e-3 m, no world flagged; and each world of the
    batch bit-identical to the same world stepped alone."""
    from test_golden import CASES
    names = ["box_stack_ws", "chains_ws", "vehicle_ws"]
    scs = [CASES[k][0]() for k in names]
    n, every = 60, 10
    b = _batch(odemi_mod, scs, odemi_mod.ORDER_REFERENCE)
    b.set_exact_lcp(256)
    nb = [sc.nb for sc in scs]
    off = np.concatenate([[0], np.cumsum(nb)])
    trajs = [[] for _ in scs]
    for k in range(n + 1):
        if k % every == 0:
            st = b.state().reshape(-1, 13)
            for w in range(len(scs)):
                trajs[w].append(st[off[w]:off[w + 1]].copy())
        if k == n:
            break
        # per joint: lostop, histop (NaN: unchanged), torque1, torque2
        b.set_controls(np.concatenate([sc.step_ctrl[k].reshape(-1) if sc.step_ctrl is not None
                                       else np.tile([np.nan, np.nan, 0.0, 0.0], sc.nj) for sc in scs]))
        b.step(1)
    cnt = b.world_counters()
    assert np.all((cnt[:, 4] & 32) == 0), cnt[:, 4]
    for w, name in enumerate(names):
        g = golden(name)
        got = np.array(trajs[w])[:, :, :3]
        ref = g["traj"][: n // every + 1, :, :3]
        r32 = po.run(po.oracle_lib("f32"), scs[w], n, every)["traj"][:, :, :3]
        env = np.abs(r32 - ref).max(axis=(1, 2))
        err = np.abs(got - ref).max(axis=(1, 2))
        say(name, "batch exact LCP traj err", float(err.max()), "envelope", float(env.max()))
        assert np.all(err <= 4 * env + 1e-3), name
    alone = _batch(odemi_mod, [scs[0]], odemi_mod.ORDER_REFERENCE)
    alone.set_exact_lcp(256)
    alone.step(n)
    assert np.array_equal(alone.state().reshape(-1, 13), b.state().reshape(-1, 13)[off[0]:off[1]])


def _tie_order(con, ref):
    """Permutation of this step's GPU contacts onto the reference's: within a
    pair, contacts whose depths tie come out in an order decided by the last
    bit of the arithmetic, so they are matched by position."""
    perm = np.arange(len(ref))
    i, n = 0, len(ref)
    while i < n:
        j = i
        while j < n and ref[j, 7] == ref[i, 7] and ref[j, 8] == ref[i, 8]:
            j += 1
        if j - i > 1:
            used = set()
            for a in range(i, j):
                d = [np.abs(con[c, :3] - ref[a, :3]).max() if c not in used else np.inf for c in range(i, j)]
                c = i + int(np.argmin(d))
                used.add(c)
                perm[a] = c
        i = j
    return perm


@pytest.mark.parametrize("name", ["box_stack", "chains", "surfaces", "vehicle", "vehicle_spaces", "capsules",
                                  "cylinders"])
def test_dropin_joint_feedback_every_step(odemi_mod, name):
    """dJointFeedback written back by dWorldQuickStep (quickstep.cpp:918-957)
    for every contact joint of every diagnostic step of the drop-in run,
    against the reference double build's: within 4x the distance of the
    reference's own single build (its CPU restatement) from the double build
    at the same step, plus 2e-3 of the step's largest force (a box resting
    on four coplanar contacts splits its load among them in a way the
    rounding decides, in the reference's own builds as here).  A step is
    compared when its callback pairs and contact counts equal the
    reference's in this run and in the single build's (the runs then hold
    the same joints in the same order) and its contacts are as close to the
    reference's as the single build's (a step over the bar whose pair
    contacts came out in another order than in the single build's is
    counted apart: the 20 sweeps relaxed its rows in another order), on at
    least half of the steps with contacts or 25 steps."""
    say("drop-in feedback", name)
    from test_golden import CASES
    fac, n, every, diag = CASES[name]
    sc = fac()
    g = golden(name)
    lib = po.load(os.path.join(ROOT, "tests", "_build", "libscene_odemi.so"))
    kw = dict(diag_steps=diag, max_pairs=400000, max_contacts=400000, feedback=True)
    r = po.run(lib, sc, diag, 0, **kw)
    r32 = po.run(po.oracle_lib("f32"), sc, diag, 0, **kw)
    pc, cc = g["pair_step_count"], g["contact_step_count"]
    p0 = np.concatenate([[0], np.cumsum(pc)])
    k0 = np.concatenate([[0], np.cumsum(cc)])
    rp0 = np.concatenate([[0], np.cumsum(r["pair_step_count"])])
    rk0 = np.concatenate([[0], np.cumsum(r["contact_step_count"])])
    sp0 = np.concatenate([[0], np.cumsum(r32["pair_step_count"])])
    sk0 = np.concatenate([[0], np.cumsum(r32["contact_step_count"])])
    compared, drifted, reordered, worst = 0, 0, 0, 0.0
    for s in range(diag):
        if cc[s] == 0:
            continue
        same = (r["pair_step_count"][s] == pc[s] and r["contact_step_count"][s] == cc[s] and
                np.array_equal(r["pairs"][rp0[s]:rp0[s + 1]], g["pairs"][p0[s]:p0[s + 1]]))
        if not same:
            continue
        ref = g["contacts"][k0[s]:k0[s + 1]]
        fref = g["feedback"][k0[s]:k0[s + 1]]
        perm = _tie_order(r["contacts"][rk0[s]:rk0[s + 1]], ref)
        fgpu = r["feedback"][rk0[s]:rk0[s + 1]][perm]
        scale = max(1.0, float(np.abs(fref).max()))
        err = float(np.abs(fgpu - fref).max())
        if not (r32["contact_step_count"][s] == cc[s] and
                np.array_equal(r32["pairs"][sp0[s]:sp0[s + 1]], g["pairs"][p0[s]:p0[s + 1]])):
            continue   # no FP32 envelope at this step
        p32 = _tie_order(r32["contacts"][sk0[s]:sk0[s + 1]], ref)
        # the step's inputs: compared only while this run's contacts are as
        # close to the reference's as the single restatement's (4x its
        # distance, at least 1e-5); later the trajectories have drifted apart
        # by their own rounding (bounded by the trajectory tests) and the
        # forces of different states are not comparable
        cg = float(np.abs(r["contacts"][rk0[s]:rk0[s + 1]][perm][:, :7] - ref[:, :7]).max())
        c32 = float(np.abs(r32["contacts"][sk0[s]:sk0[s + 1]][p32][:, :7] - ref[:, :7]).max())
        if cg > 4 * c32 + 1e-5:
            drifted += 1
            continue
        env = float(np.abs(r32["feedback"][sk0[s]:sk0[s + 1]][p32] - fref).max())
        tol = 4 * env + 2e-3 * scale
        if err > tol and not np.array_equal(perm, p32):
            # a pair's contacts came out in another order here than in the
            # single restatement (a tie the last bit decides, e.g. a box
            # resting flat): the 20 sweeps relaxed the rows in another order,
            # which the restatement's distance does not cover
            reordered += 1
            continue
        worst = max(worst, err / tol)
        assert err <= tol, (name, s, err, env, scale, fgpu[:, :3].tolist(), fref[:, :3].tolist())
        compared += 1
    with_contacts = int((cc > 0).sum())
    say(name, "steps compared", compared, "of", with_contacts, "(contacts drifted apart on", drifted,
        ", contacts of a pair reordered on", reordered, ") worst err/tol", worst)
    # chaotic piles (cylinders pass through each other here as in the
    # reference) leave the reference's pair sets after a few dozen steps
    assert compared >= min(0.5 * with_contacts, 25)


@pytest.mark.parametrize("name", ["box_stack", "chains", "pile256_dense", "surfaces"])
def test_reference_order_residual_matches_restatement(odemi_mod, name):
    """The LCP residual after each reference-order solve (20 iterations, the
    reference's row order and shuffle) against the residual of the double
    restatement's impulses, which equal the reference double build's (the
    reference computes no residual): within 4x the single restatement's
    distance from the double one, plus 5 % and 1e-4."""
    say("reference-order residual", name)
    from test_golden import CASES
    sc = CASES[name][0]()
    nsteps = 20
    r64 = po.run(po.oracle_lib("f64"), sc, nsteps, 0, residual=True)["residual"]
    r32 = po.run(po.oracle_lib("f32"), sc, nsteps, 0, residual=True)["residual"]
    b = _batch(odemi_mod, [sc])
    b.track_residual(True)
    got = []
    for k in range(nsteps):
        if sc.step_ctrl is not None:
            b.set_controls(sc.step_ctrl[k])
        b.step(1)
        got.append(float(b.residual()[0]))
    got = np.array(got)
    tol = 4 * np.abs(r32 - r64) + 0.05 * r64 + 1e-4
    say(name, "residuals", np.round(got[:5], 6), "restatement", np.round(r64[:5], 6),
        "worst err/tol", float((np.abs(got - r64) / tol).max()))
    assert np.all(np.abs(got - r64) <= tol)


def test_plain_path_equals_batched_path(odemi_mod):
    say("plain vs batched")
    ws = scenes.uneven_worlds(24, seed=3)
    a = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
    b = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
    a.step(15)
    b.step_plain(15)
    assert np.array_equal(a.state(), b.state())
    r1 = _batch(odemi_mod, ws[:6])
    r2 = _batch(odemi_mod, ws[:6])
    r1.step(10)
    r2.step_plain(10)
    assert np.array_equal(r1.state(), r2.state())


def test_reference_order_independent_of_launch_shape(odemi_mod):
    say("launch shapes")
    ws = scenes.uneven_worlds(8, seed=5)
    outs = []
    # the last shapes have a 16 KB pool (rows streamed from global memory,
    # impulses and forces in LDS) and no LDS pool (sorts, ordering and the
    # solve in global scratch); the others solve the worlds whose rows fit
    # in LDS there
    for wg, cs, lds in ((256, 1.0, None), (64, 2.0, None), (128, 1.5, None), (128, 1.0, 16384), (128, 1.0, 0)):
        b = _batch(odemi_mod, ws)
        b.set_launch_config(wg, cs, lds)
        b.step(12)
        outs.append(b.state())
    for o in outs[1:]:
        assert np.array_equal(outs[0], o)


def test_colored_solver_converges_with_iterations(odemi_mod):
    say("coloured convergence")
    res = {}
    for iters in (20, 400):
        sc = scenes.pile_world(np.random.default_rng(8), 48, 2, seed=2)
        sc.iterations = iters
        b = _batch(odemi_mod, [sc], odemi_mod.ORDER_COLORED)
        b.step(60)
        b.track_residual(True)
        b.step(1)
        res[iters] = float(b.residual().max())
    say("residual", res)
    assert res[400] < 0.5 * res[20]


def test_autotune_keeps_state(odemi_mod):
    say("autotune")
    ws = scenes.uneven_worlds(16, seed=9)
    a = _batch(odemi_mod, ws)
    a.step(3)
    st = a.state()
    wg = a.autotune(1)
    assert wg in (64, 128, 256, 512)
    assert np.array_equal(a.state(), st)
    b = _batch(odemi_mod, ws)
    b.step(3)
    a.step(5)
    b.step(5)
    assert np.array_equal(a.state(), b.state())
    # the two-kernel step is switched off: refused, never chosen
    assert a.launch_config()["split"] == 0
    with pytest.raises(RuntimeError):
        a.set_launch_config(wg, 1.0, split=1)
    assert a.launch_config()["split"] == 0


@pytest.mark.parametrize("wg", [256, 64], ids=["wg256", "wg64-capped"])
def test_coloured_order_matches_coloured_restatement(odemi_mod, wg):
    """Coloured order against its CPU restatement (oracle coloured mode, the
    same pair order and colouring, colours capped at the workgroup width):
    first-step pairs and contacts exact, trajectories over 40 steps within 4x
    the restatement's own FP32-FP64 distance + 1e-3 m.  At width 64 the
    worlds include 144 boxes on a plane, whose colours the cap splits."""
    ws = scenes.uneven_worlds(6, seed=11)
    if wg == 64:
        ws = [scenes.box_floor(12)] + ws[:3]

    def batch():
        b = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
        if wg != 256:
            b.set_launch_config(wg, 1.0)
        return b

    lib32, lib64 = po.oracle_lib("f32"), po.oracle_lib("f64")
    b = batch()
    b.step(1)
    n = 40
    refs = []
    try:
        for lib in (lib32, lib64):
            lib.orc_set_colored(1)
            lib.orc_set_colour_width(wg)
        for w, sc in enumerate(ws):
            say("coloured parity world", w, "nb", sc.nb, "nj", sc.nj)
            r = po.run(lib64, sc, 1, 1, diag_steps=1, max_pairs=100000, max_contacts=100000)
            pairs = b.pairs(w)
            assert np.array_equal(pairs, r["pairs"]), "coloured pair order differs"
            con = b.contacts(w)
            assert len(con) == len(r["contacts"])
            if len(con):
                assert np.array_equal(con[:, 7:9].astype(int), r["contacts"][:, 7:9].astype(int))
                err = np.abs(con[:, :7] - r["contacts"][:, :7]) / np.maximum(1.0, np.abs(r["contacts"][:, :7]))
                assert err.max() <= 2e-5
            t32 = po.run(lib32, sc, n, 10)["traj"]
            t64 = po.run(lib64, sc, n, 10)["traj"]
            refs.append((t32, t64))
    finally:
        for lib in (lib32, lib64):
            lib.orc_set_colored(0)
            lib.orc_set_colour_width(256)
    b.close()
    b = batch()
    offs = np.concatenate([[0], np.cumsum([w.nb for w in ws])])
    worst = 0.0
    for k in range(n // 10):
        b.step(10)
        st = b.state()
        for w, (t32, t64) in enumerate(refs):
            env = float(np.abs(t32[k + 1][:, :3] - t64[k + 1][:, :3]).max())
            err = float(np.abs(st[offs[w]:offs[w + 1], :3] - t32[k + 1][:, :3]).max())
            tol = 4 * env + 1e-3
            worst = max(worst, err / tol)
            assert err <= tol, (w, k, err, env)
    say("coloured trajectories: worst err/tol", worst)


@pytest.mark.parametrize("warm", [0.0, 1.0], ids=["cold", "warm"])
def test_accelerated_tolerance_solver_matches_restatement(odemi_mod, warm):
    """Coloured order iterated to a residual tolerance with the conjugate-
    gradient steps (cold, or warm-started from the previous step's impulses),
    against the same solver in the CPU restatement: 20 steps within 4x the
    restatement's FP32-FP64 distance + 1e-3 m; every world reaches the
    tolerance."""
    ws = scenes.uneven_worlds(4, seed=13)
    lib32, lib64 = po.oracle_lib("f32"), po.oracle_lib("f64")
    n, tol = 20, 1e-3
    refs = []
    try:
        for lib in (lib32, lib64):
            lib.orc_set_colored_solver.argtypes = [C.c_double, C.c_int, C.c_int, C.c_int]
            lib.orc_set_warm_start.argtypes = [C.c_double]
            lib.orc_set_colored(1)
            lib.orc_set_colored_solver(tol, 3000, 10, 1)
            lib.orc_set_warm_start(warm)
        for sc in ws:
            refs.append((po.run(lib32, sc, n, n)["traj"][-1], po.run(lib64, sc, n, n)["traj"][-1]))
    finally:
        for lib in (lib32, lib64):
            lib.orc_set_colored(0)
            lib.orc_set_colored_solver(0.0, 0, 10, 0)
            lib.orc_set_warm_start(0.0)
    b = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
    b.set_tolerance(tol, 3000, 10, accel=True)
    b.set_warm_start(warm)
    b.track_residual(True)
    its = np.zeros(len(ws), np.int64)
    for _ in range(n):
        b.step(1)
        its += b.world_counters()[:, 5]
    res = b.residual()
    st = b.state()
    wc = b.world_counters()
    b.close()
    say(f"accelerated solver (warm {warm}): residual", res.tolist(), "iterations", wc[:, 5].tolist(),
        "total sweeps", its.tolist())
    assert (res <= tol).all() and (wc[:, 5] < 3000).all()
    offs = np.concatenate([[0], np.cumsum([w.nb for w in ws])])
    for w, (t32, t64) in enumerate(refs):
        env = float(np.abs(t32[:, :3] - t64[:, :3]).max())
        err = float(np.abs(st[offs[w]:offs[w + 1], :3] - t32[:, :3]).max())
        say(f"world {w}: err {err:.3g} envelope {env:.3g}")
        assert err <= 4 * env + 1e-3


@pytest.mark.skip(reason="split sweep kernel switched off: a 4096-world timing run with it did not finish; "
                         "cause not found")
def test_split_sweep_kernel_matches_fused(odemi_mod):
    """The coloured solver at a tolerance with its sweeps in a kernel of their
    own (collide + set-up | sweeps | integration) runs the same arithmetic as
    the one-kernel step: states agree bit for bit, with an LDS pool that holds
    every world and with one so small that the integration kernel solves the
    worlds it cannot hold.  (Same workgroup size as the one-kernel step: the
    block sums of the conjugate-gradient step follow the workgroup size.)"""
    ws = scenes.uneven_worlds(24, seed=17)
    n = 12
    ref = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
    ref.set_launch_config(128, 1.0, 65536, 0, 0)
    ref.set_tolerance(1e-4, 400, 10, accel=True)
    ref.set_warm_start(1.0)
    ref.step(n)
    want = ref.state()
    want_it = ref.world_counters()[:, 5]
    ref.close()
    for wg, lds, grid in ((128, 65536, 0), (128, 8192, 0), (128, 32768, 64)):
        say("split sweep kernel", wg, lds, grid)
        b = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
        b.set_launch_config(128, 1.0, 65536, 0, 0)
        b.set_tolerance(1e-4, 400, 10, accel=True)
        b.set_warm_start(1.0)
        b.set_sor_launch(True, wg, lds, grid)
        b.step(n)
        got = b.state()
        got_it = b.world_counters()[:, 5]
        cfg = b.launch_config()
        b.close()
        assert cfg["sor"]["on"] == 1
        assert np.array_equal(got_it, want_it)
        assert np.array_equal(got, want), float(np.abs(got - want).max())


def _free_fall_world(v0=(1.0, -0.5, 2.0)):
    from odemi.scenes import _Builder
    b = _Builder()
    b.sphere_body((0.5, 0.25, 3.0), 0.2, 1.0, lvel=v0)
    return b.scene(dt=0.01, mu=0.5, seed=1)


def _nan_world():
    """Two spheres over a plane; the test makes the first one's velocity NaN
    through dBatchSetState (dBatchCreate refuses non-finite input)."""
    from odemi.scenes import _Builder, PLANE
    b = _Builder()
    b.geom(PLANE, (0.0, 0.0, 1.0, 0.0))
    b.sphere_body((0.0, 0.0, 0.5), 0.3, 1.0)
    b.sphere_body((2.0, 0.0, 0.25), 0.3, 1.0)
    return b.scene(dt=0.01, mu=0.5, seed=2)


def test_ragged_batch_worlds_step_independently(odemi_mod):
    """Worlds of very different kinds and sizes in one batch (a lone body in
    free fall with no geoms to meet, the box stack, uneven piles with chains, a
    vehicle, a world whose state is made non-finite before the first step),
    reference order: every finite world ends bit-identical to the same world
    stepped alone; the non-finite world is frozen and flagged without touching the
    others; the free-falling body follows the integrator's closed form
    (v += h g, x += h v: x_n = x_0 + n h v_0 + h^2 g n (n + 1) / 2) within
    FP32 rounding (1e-4 m)."""
    from odemi import scenes as S
    worlds = [_free_fall_world(), S.box_stack(10), *S.uneven_worlds(3, seed=2),
              S.vehicle_world(np.random.default_rng(4), 40, seed=9), _nan_world()]
    nsteps = 25
    say("ragged batch", [w.nb for w in worlds])
    b = _batch(odemi_mod, worlds)
    st0 = b.state()
    st0[sum(w.nb for w in worlds[:-1]), 7] = np.nan      # lvel.x of the last world's first body
    b.set_state(st0)
    b.step(nsteps)
    st = b.state()
    wc = b.world_counters()
    off = np.cumsum([0] + [w.nb for w in worlds])
    for k, w in enumerate(worlds[:-1]):
        say("solo world", k, w.nb)
        s = _batch(odemi_mod, [w])
        s.step(nsteps)
        assert np.array_equal(s.state(), st[off[k]:off[k + 1]]), k
        assert wc[k, 4] == 0, (k, wc[k])
        s.close()
    assert wc[-1, 4] & 16, wc[-1]            # non-finite: frozen and flagged
    frozen = st[off[-2]:off[-1]].copy()
    b.step(3)
    assert np.array_equal(b.state()[off[-2]:off[-1]], frozen, equal_nan=True)
    # closed form of the lone body
    h, n = 0.01, nsteps
    g = np.array([0.0, 0.0, -9.81])
    x = np.array([0.5, 0.25, 3.0]) + n * h * np.array([1.0, -0.5, 2.0]) + h * h * g * n * (n + 1) / 2
    assert np.abs(st[0, :3] - x).max() <= 1e-4, (st[0, :3], x)
    b.close()


def _packed_spheres():
    """252 spheres (r 0.3 m) on a 0.5 m lattice over a plane: every sphere
    overlaps its lattice neighbours, ~700 candidate pairs on the first step."""
    from odemi.scenes import _Builder, PLANE
    b = _Builder()
    b.geom(PLANE, (0.0, 0.0, 1.0, 0.0))
    for x in range(6):
        for y in range(6):
            for z in range(7):
                b.sphere_body((0.5 * x, 0.5 * y, 0.35 + 0.5 * z), 0.3, 1.0)
    return b.scene(dt=0.01, mu=0.5, seed=3)


def test_capacity_overflow_is_flagged_and_deterministic(odemi_mod, monkeypatch):
    """Packed spheres with pair, contact and row capacities cut to 5 %
    (ODEMI_CAPACITY_SCALE): the first step flags the pair overflow, keeps
    exactly as many pairs as there are slots, all of them pairs of the
    full-capacity step, and two runs agree bit for bit (the pairs kept when
    they overflow are chosen in entry order, not by the order lanes finish)."""
    sc = _packed_spheres()
    say("capacity overflow: full capacity")
    full = _batch(odemi_mod, [sc])
    full.step(1)
    full_pairs = {tuple(p) for p in full.pairs(0)}
    full.close()
    monkeypatch.setenv("ODEMI_CAPACITY_SCALE", "0.05")
    runs = []
    for rep in range(2):
        say("capacity overflow: run", rep)
        b = _batch(odemi_mod, [sc])
        b.step(1)
        p1 = b.pairs(0)
        f1 = int(b.world_counters()[0, 4])
        b.step(2)
        runs.append((p1, f1, b.state()))
        b.close()
    p1, f1, _ = runs[0]
    assert f1 & 2, f1                                   # OVF_PAIRS
    pcap = 1
    while pcap < int(0.05 * (16 * sc.ng + 64)):   # the library's capacity rule
        pcap <<= 1
    assert len(p1) == pcap and len(full_pairs) > pcap
    assert {tuple(p) for p in p1} <= full_pairs
    assert np.array_equal(runs[0][0], runs[1][0]) and runs[0][1] == runs[1][1]
    assert np.array_equal(runs[0][2], runs[1][2], equal_nan=True)


def test_coloured_order_is_reproducible(odemi_mod):
    """The coloured order at a tolerance (CG steps, warm start) gives the same
    bits on every run at one launch shape: pair slots are taken in any order
    but sorted by key, colours are bucketed stably, and the block sums of the
    stopping test and the CG step run in a fixed order."""
    ws = scenes.uneven_worlds(12, seed=11)
    outs = []
    for rep in range(2):
        say("coloured reproducibility run", rep)
        b = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
        b.set_launch_config(128, 1.5, None, 0, 256)
        b.set_tolerance(1e-4, 400, 10, accel=True)
        b.set_warm_start(1.0)
        b.step(15)
        outs.append((b.state(), b.world_counters()))
        b.close()
    assert np.array_equal(outs[0][0], outs[1][0], equal_nan=True)
    assert np.array_equal(outs[0][1], outs[1][1])


def test_coloured_solver_placements_agree(odemi_mod):
    """The coloured solver's working set placed in the LDS pool, with only its
    rows in global scratch, with its rows and the bodies' conjugate-gradient
    state in global scratch, with its rows and all of the conjugate-gradient
    state in global scratch, or all in global scratch (the pool size decides
    per world): the same bits at one workgroup size, at a tolerance with CG
    steps and warm start, over 15 steps of uneven worlds."""
    ws = scenes.uneven_worlds(12, seed=11)
    outs = []
    for lds in (None, 32768, 16384, 12288, 9216, 6144, 4096, 3072, 0):
        say("coloured placement, pool", lds)
        b = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
        b.set_launch_config(128, 1.5, lds, 0, 256)
        b.set_tolerance(1e-4, 400, 10, accel=True)
        b.set_warm_start(1.0)
        b.step(15)
        outs.append((b.state(), b.world_counters()))
        b.close()
    for st, wc in outs[1:]:
        assert np.array_equal(outs[0][0], st, equal_nan=True)
        assert np.array_equal(outs[0][1], wc)


def test_queue_order_by_cost_keeps_every_world(odemi_mod):
    """The persistent queue ordered by estimated solver work and by size (the
    default): every world is stepped exactly once per step either
    way, so the states and counters are the same bits, over 20 steps of 48
    uneven worlds at a tolerance with warm start, on a grid smaller than the
    batch (workgroups pull several worlds each)."""
    ws = scenes.uneven_worlds(48, seed=13)
    outs = []
    for by_cost in (True, False):
        say("queue order by cost:", by_cost)
        b = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
        b.set_launch_config(64, 1.5, 38400, 0, 16)
        b.set_queue_order(by_cost)
        assert b.queue_order() == by_cost
        b.set_tolerance(1e-4, 400, 10, accel=True)
        b.set_warm_start(1.0)
        b.step(20)
        outs.append((b.state(), b.world_counters()))
        b.close()
    assert np.array_equal(outs[0][0], outs[1][0], equal_nan=True)
    assert np.array_equal(outs[0][1], outs[1][1])


def test_uneven_worlds_rollout_at_tolerance(odemi_mod):
    """The batched-uneven-worlds configuration at the metric's operating
    point on 24 worlds: 200 steps, coloured order iterated to an LCP residual
    of 1e-4 (cap 2000, CG steps, warm start).  Every world stays finite (none
    frozen); whenever the solver reports a solve converged, the residual
    recomputed afterwards from the rows and the final impulses is within the
    tolerance (the stopping test is sound); the fraction of converged solves
    is reported and must be at least half."""
    ws = scenes.uneven_worlds(24, seed=5)
    say("uneven worlds at tolerance:", len(ws), "worlds,", sum(w.nb for w in ws), "bodies, 200 steps")
    b = _batch(odemi_mod, ws, odemi_mod.ORDER_COLORED)
    b.set_tolerance(1e-4, 2000, 10, accel=True)
    b.set_warm_start(1.0)
    b.track_residual(True)
    solves = conv = 0
    worst_conv = 0.0
    prev = np.zeros(len(ws), np.int64)
    for k in range(200):
        b.step(1)
        res = b.residual()
        unconv, _ = b.solve_stats()
        newly = unconv.astype(np.int64) - prev
        prev = unconv.astype(np.int64)
        ok = newly == 0
        solves += len(ws)
        conv += int(ok.sum())
        if ok.any():
            worst_conv = max(worst_conv, float(res[ok].max()))
        assert (res[ok] <= 1.05e-4).all(), (k, res[ok].max())
    st = b.state()
    wc = b.world_counters()
    assert np.isfinite(st).all()
    assert not ((wc[:, 4] & 16) != 0).any()
    say("converged solves", conv, "of", solves, f"({conv / solves:.3f}); largest residual of a converged solve "
        f"{worst_conv:.3g}")
    assert conv >= 0.5 * solves
