"""Every form of the MCTF level kernel (block side, fractional rounds, range,
integer, fractional, missing and far candidates) on planes of any sample
alignment and on ragged sizes, against the oracle, bit-exact."""
import ctypes

import numpy as np
import pytest

from tests.helpers import ptr
from xin26x_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs,rng,frac,lower,factor,pad,shift,size", [
    (8, 0, 1, "int", 1, 80, 0, (64, 96)), (8, 0, 1, "frac", 1, 80, 1, (53, 71)), (8, 0, 1, None, 1, 12, 1, (40, 72)),
    (8, 0, 0, "int", 4, 40, 1, (64, 80)), (8, 8, 1, "int", 2, 9, 1, (48, 61)), (8, 3, 0, "frac", 3, 30, 0, (33, 50)),
    (16, 0, 1, "int", 1, 80, 1, (64, 96)), (16, 8, 1, "frac", 1, 80, 0, (53, 71)), (16, 5, 1, None, 1, 0, 1, (48, 80)),
    (16, 8, 0, None, 1, 16, 0, (96, 112)), (16, 5, 0, "int", 2, 5, 1, (70, 90)), (16, 1, 0, "frac", 4, 60, 1, (35, 49)),
    (8, 2, 1, "far", 4, 20, 1, (48, 64)), (16, 2, 1, "far", 4, 20, 0, (48, 64)), (8, 1, 1, "int", 1, 3, 0, (8, 8)),
    (16, 8, 1, "int", 1, 7, 1, (16, 16))])
@pytest.mark.parametrize("kind", ["texture", "extreme"])
def test_level(oracle, kind, bs, rng, frac, lower, factor, pad, shift, size):
    import torch
    lib = capi.load()
    h, w = size
    r = np.random.default_rng(bs + 3 * rng + 7 * pad)
    m = pad + 24                                             # held past the declared padding
    if kind == "texture":
        yy, xx = np.mgrid[0:h + 2 * m, 0:w + 2 * m]
        full = 500 + 260 * np.sin(xx / 5.0 + yy / 9.0) + 180 * np.cos(yy / 4.0 - xx / 13.0) + r.normal(0, 20, xx.shape)
    else:
        full = r.integers(0, 2, (h + 2 * m, w + 2 * m)) * 1023
    full = np.clip(full, 0, 1023).astype(np.uint16)
    d = min(3, m)
    cur = full[m + d:m + d + h, m - 2:m - 2 + w].copy()
    if kind == "texture":
        cur = np.clip(0.5 * cur + 0.5 * full[m + d:m + d + h, m - 1:m - 1 + w] + r.normal(0, 3, cur.shape), 0, 1023)
    cur = np.ascontiguousarray(cur.astype(np.uint16))

    def shifted(a):                                          # odd start and odd stride when shift, both even if not
        st = a.shape[1] + (a.shape[1] % 2 != shift)
        b = np.zeros(shift + st * a.shape[0] + 2, np.uint16)
        b[shift:shift + st * a.shape[0]].reshape(a.shape[0], st)[:, :a.shape[1]] = a
        return torch.from_numpy(b.view(np.int16)).cuda(), st

    dc, cs = shifted(cur)
    dr, rs = shifted(full)
    pc = capi.XgPlane(dc.data_ptr() + 2 * shift, cs, w, h, 0)
    pr = capi.XgPlane(dr.data_ptr() + 2 * (shift + m * rs + m), rs, w, h, pad)
    nbx, nby = w // bs, h // bs
    low = None
    if lower:
        low = r.integers(-4, 5, (max(1, nby // 2), max(1, nbx // 2), 2)).astype(np.int32) * 16
        if lower == "frac":
            low += r.integers(0, 16, low.shape).astype(np.int32)
        elif lower == "far":
            low = r.integers(-3, 4, low.shape).astype(np.int32) * 16 * 40
        low = np.ascontiguousarray(low)
    emv, eerr = np.zeros(2 * nbx * nby, np.int32), np.zeros(nbx * nby, np.uint32)
    oracle.or_MctfMeLevel(ptr(cur), w, ptr(full, m * full.shape[1] + m), full.shape[1], w, h, pad, bs, rng,
                          None if low is None else ptr(low), 0 if low is None else low.shape[1],
                          0 if low is None else low.shape[0], factor, frac, 0, nby, ptr(emv), ptr(eerr))
    dl = None if low is None else torch.from_numpy(low).cuda()
    mv = torch.zeros(2 * nbx * nby, dtype=torch.int32, device="cuda")
    err = torch.zeros(nbx * nby, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), 1) == 0
    try:
        assert lib.xg_mctf_me_level(s, ctypes.byref(pc), ctypes.byref(pr), bs, rng,
                                    None if dl is None else ctypes.c_void_p(dl.data_ptr()),
                                    0 if low is None else low.shape[1], 0 if low is None else low.shape[0], factor, frac,
                                    ctypes.c_void_p(mv.data_ptr()), ctypes.c_void_p(err.data_ptr())) == 0
        assert lib.xg_session_sync(s) == 0
    finally:
        lib.xg_session_destroy(s)
    assert np.array_equal(mv.cpu().numpy(), emv)
    assert np.array_equal(err.cpu().numpy().view(np.uint32), eerr)
