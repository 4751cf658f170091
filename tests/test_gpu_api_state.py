"""What the ODE API reads after a step that did not end well."""
import ctypes as C

import pytest

from conftest import say

pytestmark = pytest.mark.gpu

V, F, I = C.c_void_p, C.c_float, C.c_int


def _lib(odemi_mod):
    L = C.CDLL(odemi_mod.capi.LIB_PATH)
    for name, res, args in [
            ("dInitODE2", I, [C.c_uint]), ("dWorldCreate", V, []), ("dWorldDestroy", None, [V]),
            ("dWorldSetGravity", None, [V, F, F, F]), ("dBodyCreate", V, [V]),
            ("dBodySetLinearVel", None, [V, F, F, F]), ("dBodyGetPosition", C.POINTER(F), [V]),
            ("dWorldQuickStep", I, [V, F])]:
        f = getattr(L, name)
        f.restype, f.argtypes = res, args
    L.hipSetDevice.argtypes = [I]
    L.hipGetLastError.argtypes = []
    return L


def test_state_after_a_step_that_failed_late(odemi_mod):
    """A step whose kernel ran and that then returned with an error (here the
    runtime's last error, left by a call of the application's own): the bodies
    are where the device has them, not where the step before left them."""
    L = _lib(odemi_mod)
    L.dInitODE2(0)
    w = L.dWorldCreate()
    L.dWorldSetGravity(w, 0.0, 0.0, 0.0)
    b = L.dBodyCreate(w)
    L.dBodySetLinearVel(b, 1.0, 0.0, 0.0)
    say("late failure")
    assert L.dWorldQuickStep(w, 0.25)
    assert L.hipSetDevice(-1) != 0
    ok = L.dWorldQuickStep(w, 0.25)
    L.hipGetLastError()
    x = L.dBodyGetPosition(b)[0]
    L.dWorldDestroy(w)
    say("second step", ok, "x", x)
    assert not ok and x == 0.5
