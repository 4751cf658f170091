"""An ODE API world on both sides of the size up to which its results come
back through pinned memory (1 MB)."""
import numpy as np
import pytest

import pyoracle as po
from conftest import ROOT, say
from odemi import scenes as sc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [100, 3000])
def test_frame_loop_equals_the_batch(odemi_mod, n):
    """The frame loop of an application (dSpaceCollide, contacts, quickstep)
    gives the batch's states: the same device code on the same contacts.  3000
    spheres apart on a plane: 65 536 pairs' room, 1.9 MB of outputs."""
    b = sc._Builder()
    b.geom(sc.PLANE, (0.0, 0.0, 1.0, 0.0))
    for i in range(n):
        b.sphere_body((1.5 * (i % 60), 1.5 * (i // 60), 0.499), 0.5, 1.0)
    s = b.scene(dt=0.01, mu=0.5, seed=9)
    s.body_lvel = np.random.default_rng(n).normal(0, 0.2, (n, 3)).astype(np.float32).astype(np.float64)
    say("frame loop", n)
    api = po.run(po.load(f"{ROOT}/tests/_build/libscene_odemi.so"), s, 3, 1)["traj"][3]
    w = odemi_mod.Batch([s], odemi_mod.ORDER_REFERENCE)
    w.step(3)
    assert np.array_equal(api.astype(np.float32), w.state())
