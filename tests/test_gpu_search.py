"""Integer full / diamond search and the half+quarter-pel refinement through
the per-call C-ABI, and the frame-level full search of the 416x240 workload,
against the CPU oracle.  Bit-exact MVs, costs and SADs."""
import ctypes

import numpy as np
import pytest

from tests.helpers import ptr, rand_pixels
from tests.oracle_lib import OrMe
from xin26x_amd import capi, workloads as wl
from xin26x_amd.device import DevicePicture

pytestmark = pytest.mark.gpu

PAD = 80


def _me_pair(rng, plane, cur, w, h, bx, by, pred, sw, lam, mn, mx, cands=()):
    stride = plane.shape[1]
    ref_ptr = plane.ctypes.data + 2 * ((PAD + by) * stride + PAD + bx)
    cur_ptr = cur.ctypes.data + 2 * (by * cur.shape[1] + bx)
    xm = capi.XgMeStruct()
    om = OrMe()
    for m in (xm, om):
        m.width, m.height = w, h
        m.searchWidth = m.searchHeight = sw
        m.sadLambda = lam
        m.inputStride = cur.shape[1]
        m.refStride = stride
        m.candNum = len(cands)
        m.bestCost = 0xFFFFFFFF
    xm.input, xm.ref = cur_ptr, ref_ptr
    om.input, om.ref = cur_ptr, ref_ptr
    xm.minMv = capi.XgMv(*mn)
    xm.maxMv = capi.XgMv(*mx)
    om.minMvX, om.minMvY = mn
    om.maxMvX, om.maxMvY = mx
    xm.predMv = capi.XgMv(*pred)
    om.predMvX, om.predMvY = pred
    for i, (cx, cy) in enumerate(cands):
        xm.meCand[i] = capi.XgMv(cx, cy)
        om.candX[i], om.candY[i] = cx, cy
    return xm, om


def _planes(seed):
    rng = np.random.default_rng(seed)
    ref = wl.smooth_field(180, 260, seed).astype(np.uint16)
    cur = np.clip(np.roll(ref, (2, -3), axis=(0, 1)).astype(np.int64) + rng.integers(-6, 7, ref.shape), 0, 1023).astype(np.uint16)
    return rng, np.pad(ref, PAD, mode="edge"), cur


def test_full_search_matches_oracle(oracle):
    lib = capi.load()
    rng, plane, cur = _planes(31)
    for (w, h, sw, pred, lam) in ((16, 16, 16, (0, 0), 1024), (8, 8, 8, (5, -7), 2048), (32, 16, 12, (-9, 3), 512),
                                  (4, 8, 20, (2, 2), 4096), (64, 64, 6, (0, 0), 8192), (16, 32, 10, (13, -6), 0)):
        bx, by = int(rng.integers(0, 260 - w)), int(rng.integers(0, 180 - h))
        mn = (-bx - 72, -by - 72)
        mx = (260 + 72 - w - bx, 180 + 72 - h - by)
        xm, om = _me_pair(rng, plane, cur, w, h, bx, by, pred, sw, lam, mn, mx)
        lib.Xg26xMotionEstFull(ctypes.byref(xm))
        oracle.or_MotionEstFull(ctypes.byref(om))
        assert (xm.bestMv.mvX, xm.bestMv.mvY, xm.bestCost, xm.bestSad) == \
               (om.bestMvX, om.bestMvY, om.bestCost, om.bestSad), (w, h, sw)
    assert lib.xg_last_error() == 0


def test_full_search_window_clipped_at_edges(oracle):
    lib = capi.load()
    rng, plane, cur = _planes(32)
    w = h = 16
    for (bx, by) in ((0, 0), (244, 164)):
        mn = (-bx - 72, -by - 72)
        mx = (260 + 72 - w - bx, 180 + 72 - h - by)
        # tight MV window: the search range is cut by [minMv, maxMv]
        mn = (max(mn[0], -3), max(mn[1], -5))
        mx = (min(mx[0], 4), min(mx[1], 2))
        xm, om = _me_pair(rng, plane, cur, w, h, bx, by, (0, 0), 16, 1024, mn, mx)
        lib.Xg26xMotionEstFull(ctypes.byref(xm))
        oracle.or_MotionEstFull(ctypes.byref(om))
        assert (xm.bestMv.mvX, xm.bestMv.mvY, xm.bestCost, xm.bestSad) == \
               (om.bestMvX, om.bestMvY, om.bestCost, om.bestSad)


def test_diamond_matches_oracle(oracle):
    lib = capi.load()
    rng, plane, cur = _planes(33)
    for k in range(8):
        w, h = [(8, 8), (16, 16), (16, 8), (32, 32)][k % 4]
        bx, by = int(rng.integers(0, 260 - w)), int(rng.integers(0, 180 - h))
        mn = (-bx - 72, -by - 72)
        mx = (260 + 72 - w - bx, 180 + 72 - h - by)
        cands = [(0, 0)] + [(int(a), int(b)) for a, b in rng.integers(-20, 21, size=(int(rng.integers(1, 6)), 2))]
        pred = (int(rng.integers(-30, 30)), int(rng.integers(-30, 30)))
        xm, om = _me_pair(rng, plane, cur, w, h, bx, by, pred, 16, 1024, mn, mx, cands)
        lib.Xg26xMotionEstDia(ctypes.byref(xm))
        oracle.or_MotionEstDia(ctypes.byref(om))
        assert (xm.bestMv.mvX, xm.bestMv.mvY, xm.bestCost, xm.bestSad) == \
               (om.bestMvX, om.bestMvY, om.bestCost, om.bestSad), k
    assert lib.xg_last_error() == 0


def test_subpel_matches_oracle(oracle):
    lib = capi.load()
    rng, plane, cur = _planes(34)
    for k in range(12):
        w, h = [(8, 8), (16, 16), (16, 8), (4, 16), (32, 32), (64, 64)][k % 6]
        bx, by = int(rng.integers(0, 260 - w)), int(rng.integers(0, 180 - h))
        mn = (-bx - 72, -by - 72)
        mx = (260 + 72 - w - bx, 180 + 72 - h - by)
        pred = (int(rng.integers(-40, 40)), int(rng.integers(-40, 40)))
        xm, om = _me_pair(rng, plane, cur, w, h, bx, by, pred, 8, 1024, mn, mx)
        lib.Xg26xMotionEstFull(ctypes.byref(xm))
        oracle.or_MotionEstFull(ctypes.byref(om))
        lib.Xg266FullSubPelMe(ctypes.byref(xm))
        oracle.or_FullSubPelMe(ctypes.byref(om))
        assert (xm.bestMv.mvX, xm.bestMv.mvY, xm.bestCost) == (om.bestMvX, om.bestMvY, om.bestCost), k
    assert lib.xg_last_error() == 0


def test_frame_full_search_416x240(oracle):
    """The 416x240 workload: every 16x16 block, +/-16, lambda 4 (sadLambda 1024)."""
    import torch
    lib = capi.load()
    cur, ref = wl.frame_pair_416x240()
    W, H = 416, 240
    nb = (W // 16) * (H // 16)
    dc = DevicePicture([cur, cur[::2, ::2].copy(), cur[::2, ::2].copy()], pad=0)
    dr = DevicePicture([ref, ref[::2, ::2].copy(), ref[::2, ::2].copy()], pad=PAD)
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), 1024) == 0
    mv = torch.zeros(2 * nb, dtype=torch.int16, device="cuda")
    cost = torch.zeros(nb, dtype=torch.int32, device="cuda")
    sad = torch.zeros(nb, dtype=torch.int32, device="cuda")
    rc = lib.xg_full_search_frame(s, ctypes.byref(dc.pic.plane[0]), ctypes.byref(dr.pic.plane[0]), 16, 16, 16,
                                  1024, 64, mv.data_ptr(), cost.data_ptr(), sad.data_ptr())
    assert rc == 0 and lib.xg_session_sync(s) == 0
    refp = np.ascontiguousarray(np.pad(ref, PAD, mode="edge"))
    emx = np.zeros(nb, np.int16)
    emy = np.zeros(nb, np.int16)
    ec = np.zeros(nb, np.uint32)
    es = np.zeros(nb, np.uint32)
    oracle.or_FullSearchFrame(ptr(cur), W, ptr(refp, PAD * (W + 2 * PAD) + PAD), W + 2 * PAD, W, H, 16, 16, 16,
                              1024, 64, 0, nb, ptr(emx), ptr(emy), ptr(ec), ptr(es))
    g = mv.cpu().numpy().reshape(nb, 2)
    assert np.array_equal(g[:, 0], emx) and np.array_equal(g[:, 1], emy)
    assert np.array_equal(cost.cpu().numpy().view(np.uint32), ec)
    assert np.array_equal(sad.cpu().numpy().view(np.uint32), es)
    # the global motion (+13, -7) quarter-pel is found at integer precision
    inner = g.reshape(H // 16, W // 16, 2)[2:-2, 2:-2].reshape(-1, 2)
    assert np.median(inner[:, 0]) == 12 and np.median(inner[:, 1]) == -8
    lib.xg_session_destroy(s)


@pytest.mark.parametrize("bw,bh,rng", [(8, 8, 7), (32, 16, 24), (16, 32, 3), (8, 16, 60), (64, 8, 10), (4, 4, 5),
                                       (32, 32, 0)])
def test_frame_full_search_shapes(oracle, bw, bh, rng):
    """Packed kernel (widths 8, 16, 32) and the general one (4, 64) against the
    oracle on a 128x96 crop: costs, SADs, MVs and the raster tie order."""
    import torch
    lib = capi.load()
    cur, ref = wl.frame_pair_416x240()
    W, H, pad = 128, 96, 72
    cur = np.ascontiguousarray(cur[40:40 + H, 96:96 + W])
    ref = np.ascontiguousarray(ref[40:40 + H, 96:96 + W])
    nb = (W // bw) * (H // bh)
    dc = DevicePicture([cur, cur[::2, ::2].copy(), cur[::2, ::2].copy()], pad=0)
    dr = DevicePicture([ref, ref[::2, ::2].copy(), ref[::2, ::2].copy()], pad=pad)
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), 1024) == 0
    mv = torch.zeros(2 * nb, dtype=torch.int16, device="cuda")
    cost = torch.zeros(nb, dtype=torch.int32, device="cuda")
    sad = torch.zeros(nb, dtype=torch.int32, device="cuda")
    rc = lib.xg_full_search_frame(s, ctypes.byref(dc.pic.plane[0]), ctypes.byref(dr.pic.plane[0]), bw, bh, rng,
                                  1024, 64, mv.data_ptr(), cost.data_ptr(), sad.data_ptr())
    assert rc == 0 and lib.xg_session_sync(s) == 0
    refp = np.ascontiguousarray(np.pad(ref, pad, mode="edge"))
    emx = np.zeros(nb, np.int16)
    emy = np.zeros(nb, np.int16)
    ec = np.zeros(nb, np.uint32)
    es = np.zeros(nb, np.uint32)
    oracle.or_FullSearchFrame(ptr(cur), W, ptr(refp, pad * (W + 2 * pad) + pad), W + 2 * pad, W, H, bw, bh, rng,
                              1024, 64, 0, nb, ptr(emx), ptr(emy), ptr(ec), ptr(es))
    g = mv.cpu().numpy().reshape(nb, 2)
    assert np.array_equal(g[:, 0], emx) and np.array_equal(g[:, 1], emy)
    assert np.array_equal(cost.cpu().numpy().view(np.uint32), ec)
    assert np.array_equal(sad.cpu().numpy().view(np.uint32), es)
    lib.xg_session_destroy(s)


def test_search_blocks_every_width(oracle):
    """The session search of the serving path (packed core) for block widths
    4..64 and heights 4..64 around non-zero predictors, against the oracle's
    Xg26xMotionEstFull; the searched MVs are read back through a one-candidate
    (0, 0) refinement."""
    from xin26x_amd.device import blocks_to_struct, refine_cfg
    lib = capi.load()
    cur, ref = wl.frame_pair_416x240()
    W, H, pad = 256, 192, 80
    cur = np.ascontiguousarray(cur[24:24 + H, 80:80 + W])
    ref = np.ascontiguousarray(ref[24:24 + H, 80:80 + W])
    chroma = lambda p: np.ascontiguousarray(p[::2, ::2])
    dc = DevicePicture([cur, chroma(cur), chroma(cur)], pad)
    dr = DevicePicture([ref, chroma(ref), chroma(ref)], pad)
    pred = DevicePicture.empty(W, H)
    rng = np.random.default_rng(5)
    blocks = []
    for w in (4, 8, 16, 32, 64):
        for h in (4, 8, 16, 32, 64):
            for _ in range(2):
                x = int(rng.integers(0, (W - w) // 4 + 1)) * 4
                y = int(rng.integers(0, (H - h) // 4 + 1)) * 4
                blocks.append((x, y, w, h, 0, 0, int(rng.integers(-300, 301)), int(rng.integers(-300, 301))))
    n = len(blocks)
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), n) == 0
    try:
        assert lib.xg_session_set_picture(s, 0, dc.ref()) == 0
        assert lib.xg_session_set_picture(s, 1, dr.ref()) == 0
        barr = blocks_to_struct(blocks)
        assert lib.xg_session_set_blocks(s, barr.ctypes.data, n) == 0
        assert lib.xg_search_blocks(s, 16, 1024, 64) == 0
        cfg = refine_cfg([(0, 0)], wl.LAMBDA_REFINE)
        assert lib.xg_refine_frac(s, ctypes.byref(cfg), pred.ref(), capi.MODE_BATCHED) == 0
        best = np.zeros(n * 4, np.int32)
        assert lib.xg_session_read(s, None, best.ctypes.data) == 0
    finally:
        lib.xg_session_destroy(s)
    got = best.reshape(n, 4)[:, :2]
    refp = np.ascontiguousarray(np.pad(ref, pad, mode="edge"))
    rs = W + 2 * pad
    for i, (x, y, w, h, _, _, mvpx, mvpy) in enumerate(blocks):
        m = OrMe()
        m.width, m.height = w, h
        m.minMvX, m.minMvY = -x - 72, -y - 72
        m.maxMvX, m.maxMvY = W + 72 - w - x, H + 72 - h - y
        m.predMvX, m.predMvY = mvpx >> 2, mvpy >> 2
        m.searchWidth = m.searchHeight = 16
        m.sadLambda = 1024
        m.input = cur.ctypes.data + 2 * (y * W + x)
        m.inputStride = W
        m.ref = refp.ctypes.data + 2 * ((y + pad) * rs + x + pad)
        m.refStride = rs
        oracle.or_MotionEstFull(ctypes.byref(m))
        assert (got[i, 0], got[i, 1]) == (4 * m.bestMvX, 4 * m.bestMvY), (i, blocks[i])


@pytest.mark.parametrize("unit,rng_", [(16, 16), (8, 24)])
def test_lookahead_me(oracle, unit, rng_):
    """Half-resolution lookahead search: the 2x2-mean downscale of both
    pictures (the reference over its padding) then the frame full search of
    every whole unit, against the oracle's downscale and full search."""
    import torch
    lib = capi.load()
    cur, ref = wl.frame_pair_416x240()
    W, H, pad = 416, 240, 2 * (rng_ + 4) + 8
    dc = DevicePicture([cur, cur[::2, ::2].copy(), cur[::2, ::2].copy()], pad=0)
    dr = DevicePicture([ref, ref[::2, ::2].copy(), ref[::2, ::2].copy()], pad=pad)
    hw, hh, hp = W // 2, H // 2, pad // 2
    nb = (hw // unit) * (hh // unit)
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), 1024) == 0
    mv = torch.zeros(2 * nb, dtype=torch.int16, device="cuda")
    cost = torch.zeros(nb, dtype=torch.int32, device="cuda")
    sad = torch.zeros(nb, dtype=torch.int32, device="cuda")
    rc = lib.xg_lookahead_me(s, ctypes.byref(dc.pic.plane[0]), ctypes.byref(dr.pic.plane[0]), unit, rng_, 1024,
                             mv.data_ptr(), cost.data_ptr(), sad.data_ptr())
    assert rc == 0 and lib.xg_session_sync(s) == 0
    hcur = np.zeros((hh, hw), np.uint16)
    oracle.or_Downscale2x2(ptr(cur), W, ptr(hcur), hw, hw, hh)
    refp = np.ascontiguousarray(np.pad(ref, pad, mode="edge"))
    href = np.zeros((hh + 2 * hp, hw + 2 * hp), np.uint16)
    oracle.or_Downscale2x2(ptr(refp), W + 2 * pad, ptr(href), hw + 2 * hp, hw + 2 * hp, hh + 2 * hp)
    emx = np.zeros(nb, np.int16)
    emy = np.zeros(nb, np.int16)
    ec = np.zeros(nb, np.uint32)
    es = np.zeros(nb, np.uint32)
    oracle.or_FullSearchFrame(ptr(hcur), hw, ptr(href, hp * (hw + 2 * hp) + hp), hw + 2 * hp, hw, hh, unit, unit,
                              rng_, 1024, rng_, 0, nb, ptr(emx), ptr(emy), ptr(ec), ptr(es))
    g = mv.cpu().numpy().reshape(nb, 2)
    assert np.array_equal(g[:, 0], emx) and np.array_equal(g[:, 1], emy)
    assert np.array_equal(cost.cpu().numpy().view(np.uint32), ec)
    assert np.array_equal(sad.cpu().numpy().view(np.uint32), es)
    # an odd padding is refused
    dr2 = DevicePicture([ref, ref[::2, ::2].copy(), ref[::2, ::2].copy()], pad=pad + 1)
    assert lib.xg_lookahead_me(s, ctypes.byref(dc.pic.plane[0]), ctypes.byref(dr2.pic.plane[0]), unit, rng_, 1024,
                               mv.data_ptr(), cost.data_ptr(), sad.data_ptr()) == capi.XG_ERR_ARG
    lib.xg_clear_error()
    lib.xg_session_destroy(s)


@pytest.mark.parametrize("w,h,sw,sh", [(1, 1, 3, 2), (3, 5, 8, 1), (5, 3, 2, 9), (7, 7, 0, 0), (17, 13, 11, 6), (4, 4, 84, 84),
                                       (16, 16, 104, 60), (127, 33, 4, 5), (128, 96, 5, 3), (64, 127, 9, 2)])
def test_full_search_staging_sizes(oracle, w, h, sw, sh):
    """The per-call full search at odd sizes (window and block past whole 16-byte loads), large blocks and the largest
    window it takes (16x16 at +/-104 x +/-60 is 60 KB of samples); one column more is refused."""
    lib = capi.load()
    lib.xg_clear_error()
    rng, plane, cur = _planes(36)
    bx, by = 118, 52
    xm, om = _me_pair(rng, plane, cur, w, h, bx, by, (2, -3), sw, 512, (-180, -130), (180, 130))
    xm.searchHeight = om.searchHeight = sh
    lib.Xg26xMotionEstFull(ctypes.byref(xm))
    oracle.or_MotionEstFull(ctypes.byref(om))
    assert (xm.bestMv.mvX, xm.bestMv.mvY, xm.bestCost, xm.bestSad) == \
           (om.bestMvX, om.bestMvY, om.bestCost, om.bestSad)
    assert lib.xg_last_error() == 0
    if sw == 104:
        xm.searchWidth = 105
        lib.Xg26xMotionEstFull(ctypes.byref(xm))
        assert lib.xg_last_error() == capi.XG_ERR_ARG
        lib.xg_clear_error()


def test_full_search_stages_as_fast_as_the_diamond():
    """A one-sample block has next to nothing to cost, so the time of its search is that of its window's staging, which
    the diamond does for the same window."""
    import time
    lib = capi.load()
    rng, plane, cur = _planes(37)
    xm, _ = _me_pair(rng, plane, cur, 1, 1, 130, 90, (0, 0), 80, 1024, (-180, -130), (180, 130), [(0, 0)])

    def us(call, n=20):
        t = []
        for _ in range(8):
            t0 = time.perf_counter()
            for _ in range(n):
                call(ctypes.byref(xm))
            t.append((time.perf_counter() - t0) / n * 1e6)
        return float(np.median(t[1:]))

    full, dia = us(lib.Xg26xMotionEstFull), us(lib.Xg26xMotionEstDia)
    print(f"1x1 at +/-80: full {full:.1f} us, diamond {dia:.1f} us", flush=True)
    assert full < 2.5 * dia


@pytest.mark.parametrize("w,h,sw", [(128, 128, 8), (128, 64, 8), (64, 128, 20), (96, 100, 12), (100, 70, 64), (127, 128, 3),
                                    (64, 64, 64), (64, 64, 6), (8, 8, 78)])
def test_diamond_and_subpel_of_large_blocks_and_windows(oracle, w, h, sw):
    """The forms of the per-call diamond and rings on either side of their LDS limit: regions read in place because
    they do not fit, first passes in several strips (128x128), widths over a wave and no powers of two."""
    lib = capi.load()
    lib.xg_clear_error()
    rng, plane, cur = _planes(38)
    for k in range(4):
        bx, by = int(rng.integers(0, 260 - w)), int(rng.integers(0, 180 - h))
        mn = (-bx - 72, -by - 72)
        mx = (260 + 72 - w - bx, 180 + 72 - h - by)
        cands = [(0, 0)] + [(int(a), int(b)) for a, b in rng.integers(-sw, sw + 1, size=(int(rng.integers(1, 12)), 2))]
        pred = (int(rng.integers(-30, 30)), int(rng.integers(-30, 30)))
        xm, om = _me_pair(rng, plane, cur, w, h, bx, by, pred, sw, 256, mn, mx, cands)
        lib.Xg26xMotionEstDia(ctypes.byref(xm))
        oracle.or_MotionEstDia(ctypes.byref(om))
        assert (xm.bestMv.mvX, xm.bestMv.mvY, xm.bestCost, xm.bestSad) == \
               (om.bestMvX, om.bestMvY, om.bestCost, om.bestSad), k
        lib.Xg266FullSubPelMe(ctypes.byref(xm))
        oracle.or_FullSubPelMe(ctypes.byref(om))
        assert (xm.bestMv.mvX, xm.bestMv.mvY, xm.bestCost) == (om.bestMvX, om.bestMvY, om.bestCost), k
    assert lib.xg_last_error() == 0
