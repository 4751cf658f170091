"""dSpaceCollide past the capacities of its world: the overflow is reported and
what is handed out is what the device found room for, on both sides of the size
up to which the results come back through pinned memory (1 MB)."""
import ctypes as C

import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu

V, F, I = C.c_void_p, C.c_float, C.c_int
CB = C.CFUNCTYPE(None, V, V, V)
MSG = C.CFUNCTYPE(None, I, C.c_char_p, V)
PAIRS, CONTACTS = 2, 4      # overflow flags


def _lib(odemi_mod):
    L = C.CDLL(odemi_mod.capi.LIB_PATH)
    for name, res, args in [
            ("dInitODE2", I, [C.c_uint]), ("dWorldCreate", V, []), ("dWorldDestroy", None, [V]),
            ("dHashSpaceCreate", V, [V]), ("dSpaceDestroy", None, [V]), ("dBodyCreate", V, [V]),
            ("dBodySetPosition", None, [V, F, F, F]), ("dCreateBox", V, [V, F, F, F]), ("dGeomSetBody", None, [V, V]),
            ("dSpaceCollide", None, [V, V, CB]), ("dCollide", I, [V, V, I, V, I]), ("dSetErrorHandler", None, [V])]:
        f = getattr(L, name)
        f.restype, f.argtypes = res, args
    return L


def _collide(L, near, overlapping, apart):
    """One dSpaceCollide of `overlapping` unit boxes within a centimetre of
    each other and `apart` ones on their own; the messages it gave."""
    libc = C.CDLL(None)
    messages = []

    def message(num, fmt, ap):
        buf = C.create_string_buffer(256)
        libc.vsnprintf(buf, C.c_size_t(256), C.c_char_p(fmt), V(ap))
        messages.append(buf.value.decode())

    handler, cb = MSG(message), CB(near)
    L.dInitODE2(0)
    w, s = L.dWorldCreate(), L.dHashSpaceCreate(None)
    for i in range(overlapping + apart):
        b = L.dBodyCreate(w)
        k = i - overlapping
        if k < 0:
            L.dBodySetPosition(b, 0.0001 * i, 0.00007 * i, 0.00005 * i)
        else:
            L.dBodySetPosition(b, 3.0 * (1 + k % 50), 3.0 * (1 + k // 50), 0.0)
        L.dGeomSetBody(L.dCreateBox(s, 1.0, 1.0, 1.0), b)
    L.dSetErrorHandler(C.cast(handler, V))
    L.dSpaceCollide(s, None, cb)
    L.dSetErrorHandler(None)
    L.dSpaceDestroy(s)
    L.dWorldDestroy(w)
    return messages


# room of a world of n geoms: 16 n + 64 pairs, rounded up to a power of two, and
# 6 n + 64 contacts, at least 4096
@pytest.mark.parametrize("overlapping,apart,pairs,flags", [
    (20, 0, 190, 0),                    # 190 pairs, at most 760 contacts: all fit
    (64, 0, 2016, CONTACTS),            # 2048 pairs' room
    (65, 0, 2048, PAIRS | CONTACTS),    # 2080 pairs
    (20, 2080, 190, 0),                 # 65 536 pairs' room: through device memory
    (120, 1980, 7140, CONTACTS),        # 12 664 contacts' room
])
def test_overflow_is_reported(odemi_mod, overlapping, apart, pairs, flags):
    say("overflow", overlapping, apart)
    seen = []
    messages = _collide(_lib(odemi_mod), lambda _, a, b: seen.append((a, b)), overlapping, apart)
    assert len(seen) == pairs and len(set(seen)) == pairs
    assert messages == ([f"dSpaceCollide: device capacity exceeded (flags {flags})"] if flags else [])


@pytest.mark.parametrize("overlapping,apart,contacts", [
    (20, 0, 760),          # four a pair
    (32, 0, 1984), (64, 0, 4096), (65, 0, 4096), (120, 1980, 12664),
])
def test_contacts_handed_out_are_the_devices(odemi_mod, overlapping, apart, contacts):
    """dCollide in the callback gives contacts as far as there was room, and
    none for the pairs after that."""
    say("contacts", overlapping, apart)
    L = _lib(odemi_mod)
    rec = np.zeros((4, 32), np.float32)       # dContactGeom: pos 4, normal 4, depth, ...
    counts, at = [], []

    def near(_, g1, g2):
        n = L.dCollide(g1, g2, 4, rec.ctypes.data, 128)
        counts.append(n)
        at.append(rec[:n, :9].copy())

    _collide(L, near, overlapping, apart)
    at = np.concatenate(at)
    assert len(at) == sum(counts) == contacts
    full = contacts // 4
    assert counts[:full] == [4] * full and not any(counts[full:])
    assert np.abs(at[:, :3]).max() < 0.6 and at[:, 8].min() > 0
    assert np.allclose(np.linalg.norm(at[:, 4:7], axis=1), 1.0, atol=1e-5)
