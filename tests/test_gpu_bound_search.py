"""The bounded integer searches (block-sum elimination) against the oracle's
exhaustive one, on content that takes each of their paths: textures (few
candidates left), flat noise (too many left: the exhaustive list), extreme
samples (the largest sums), repeated texture and constant planes (ties in
raster order), windows cut at an odd column, and rate weights past the rule."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from tests.helpers import ptr
from xin26x_amd import capi, workloads as wl
from xin26x_amd.device import DevicePicture, refine_cfg

pytestmark = pytest.mark.gpu


def content(kind, h, w, seed=3):
    """Current plane and two reference planes."""
    r = np.random.default_rng(seed)
    if kind == "texture":
        f = wl.smooth_field(h + 80, w + 80, seed)
        cut = lambda dy, dx: f[40 + dy:40 + dy + h, 40 + dx:40 + dx + w]
        out = [cut(0, 0) + r.integers(-4, 5, (h, w)), cut(9, -23), cut(-31, 14) + r.integers(-2, 3, (h, w))]
    elif kind == "flat":
        out = [500 + np.rint(r.normal(0, 4, (h, w))) for _ in range(3)]
    elif kind == "noise":
        out = [p + np.rint(r.normal(0, 64, (h, w))) for p in content("texture", h, w, seed)]
    elif kind == "half":
        a, b = content("texture", h, w, seed), content("flat", h, w, seed)
        out = [np.where(np.arange(w) < w // 2, p, q) for p, q in zip(a, b)]
    elif kind == "extreme":
        out = [r.integers(0, 2, (h // 8 + 1, w // 8 + 1)).repeat(8, 0).repeat(8, 1)[:h, :w] * 1023 for _ in range(3)]
    elif kind == "periodic":
        t = r.integers(0, 1024, (8, 12))
        out = [np.tile(np.roll(t, k, 1), (h // 8 + 1, w // 12 + 1))[:h, :w] for k in range(3)]
    else:
        out = [np.full((h, w), v) for v in (1023, 0, 1023)]
    return [np.ascontiguousarray(np.clip(p, 0, 1023).astype(np.uint16)) for p in out]


def oracle_search(oracle, cur, ref, bw, bh, rng, lam, ctu, pad):
    h, w = cur.shape
    nb = (w // bw) * (h // bh)
    refp = np.ascontiguousarray(np.pad(ref, pad, mode="edge"))
    mx, my = np.zeros(nb, np.int16), np.zeros(nb, np.int16)
    c, s = np.zeros(nb, np.uint32), np.zeros(nb, np.uint32)
    # block ranges in threads: these are whole frames
    step = -(-nb // 8)

    def part(b0):
        oracle.or_FullSearchFrame(ptr(cur), w, ptr(refp, pad * (w + 2 * pad) + pad), w + 2 * pad, w, h, bw, bh, rng, lam,
                                  ctu, b0, min(nb, b0 + step), ptr(mx), ptr(my), ptr(c), ptr(s))

    with ThreadPoolExecutor(8) as ex:
        list(ex.map(part, range(0, nb, step)))
    return mx, my, c, s


@pytest.mark.parametrize("kind,rng,ctu,lam", [
    ("texture", 64, 64, 1024), ("texture", 33, 64, 0), ("texture", 7, 16, 300), ("texture", 64, 33, 1024),
    ("texture", 0, 64, 1024), ("texture", 64, 64, 1 << 21), ("texture", 40, 64, (1 << 21) + 1), ("flat", 64, 64, 1024),
    ("half", 64, 64, 1024), ("extreme", 64, 64, 1024), ("periodic", 50, 64, 0), ("constant", 64, 31, 0)])
def test_pipeline_full_search(oracle, kind, rng, ctu, lam):
    lib = capi.load()
    h, w, pad = 496, 848, 152          # 1,643 blocks: the bounded form's sizes, CTUs cut at both edges
    planes = content(kind, h, w)
    half = lambda p: np.ascontiguousarray(p[::2, ::2])
    pics = [DevicePicture([p, half(p), half(p)], pad) for p in planes]
    pred = DevicePicture.empty(w, h)
    nb = (w // 16) * (h // 16)
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), nb) == 0
    try:
        cfg = capi.XgPipelineCfg()
        cfg.range, cfg.sadLambda, cfg.ctuSize = rng, lam, ctu
        cfg.refine = refine_cfg([(0, 0)], wl.LAMBDA_REFINE)
        exp = [oracle_search(oracle, planes[0], planes[1 + r], 16, 16, rng, lam, ctu, pad)[:2] for r in (0, 1)]
        for mode in (capi.MODE_BATCHED, capi.MODE_GRAPH, capi.MODE_GRAPH):
            assert lib.xg_me_pipeline(s, ctypes.byref(cfg), pics[0].ref(), pics[1].ref(), pics[2].ref(), pred.ref(),
                                      mode) == 0
            full = np.zeros((nb, 2, 2), np.int16)
            assert lib.xg_me_pipeline_read(s, full.ctypes.data, None, None, None, None, None) == 0
            for r in (0, 1):
                mx, my = exp[r]
                # the frame search reports quarter pel, the pipeline integer pel
                assert np.array_equal(full[:, r, 0], mx >> 2) and np.array_equal(full[:, r, 1], my >> 2), (mode, r)
    finally:
        lib.xg_session_destroy(s)


def test_pipeline_graph_follows_the_references(oracle):
    """Reference pictures that change from frame to frame, other buffers and strides among them: every replay
    searches the pictures it was given, and the graph is captured once.  A call that only changes its pictures
    takes the time of one that does not, and not of one that changes the rate weight, which is captured again."""
    import time
    lib = capi.load()
    h, w, lam = 496, 848, 1024
    planes = content("texture", h, w)
    planes.append(np.ascontiguousarray(planes[1][::-1]))
    half = lambda p: np.ascontiguousarray(p[::2, ::2])
    pads = (152, 152, 96, 120)
    pics = [DevicePicture([p, half(p), half(p)], pad) for p, pad in zip(planes, pads)]
    pred = DevicePicture.empty(w, h)
    nb = (w // 16) * (h // 16)
    exp = {k: oracle_search(oracle, planes[0], planes[k], 16, 16, 24, lam, 64, 152)[:2] for k in (1, 2, 3)}
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), nb) == 0
    try:
        cfg = capi.XgPipelineCfg()
        cfg.range, cfg.ctuSize = 24, 64
        cfg.refine = refine_cfg([(0, 0)], wl.LAMBDA_REFINE)

        def call(a, b, weight):
            assert lib.xg_session_sync(s) == 0
            cfg.sadLambda = weight
            t = time.perf_counter()
            assert lib.xg_me_pipeline(s, ctypes.byref(cfg), pics[0].ref(), pics[a].ref(), pics[b].ref(), pred.ref(),
                                      capi.MODE_GRAPH) == 0
            return time.perf_counter() - t

        for k in range(6):
            a, b = 1 + k % 3, 1 + (k + 1) % 3
            call(a, b, lam)
            full = np.zeros((nb, 2, 2), np.int16)
            assert lib.xg_me_pipeline_read(s, full.ctypes.data, None, None, None, None, None) == 0
            for r, e in enumerate((exp[a], exp[b])):
                assert np.array_equal(full[:, r, 0], e[0] >> 2) and np.array_equal(full[:, r, 1], e[1] >> 2), (k, r)
        same, other, again = [], [], []
        for k in range(60):
            call(1, 2, lam)
            same.append(call(1, 2, lam))
            other.append(call(1 + k % 2, 3, lam))
            again.append(call(1, 2, lam + 1))
        same, other, again = (1e6 * float(np.median(v)) for v in (same, other, again))
        print(f"host us a call: same references {same:.1f}, others {other:.1f}, captured again {again:.1f}", flush=True)
        assert other - same < 0.5 * (again - same)
    finally:
        lib.xg_session_destroy(s)


@pytest.mark.parametrize("kind,size,bs,rng,ctu,lam,shift", [
    ("texture", (560, 816), 16, 16, 64, 1024, 0), ("texture", (489, 485), 8, 24, 64, 1024, 1),
    ("texture", (713, 709), 16, 32, 32, 0, 1), ("texture", (480, 480), 8, 48, 48, 500, 0),
    ("texture", (713, 709), 16, 40, 7, 1024, 1), ("texture", (479, 800), 16, 16, 64, 1024, 0),
    ("texture", (560, 816), 16, 15, 64, 1024, 0), ("texture", (560, 816), 16, 49, 64, 1024, 1),
    ("texture", (28007, 24), 16, 17, 64, 1024, 1), ("texture", (13, 28004), 8, 16, 64, 1024, 0),
    ("texture", (480, 480), 8, 16, 64, 1 << 21, 0), ("texture", (480, 480), 8, 16, 64, (1 << 21) + 1, 0),
    ("flat", (713, 709), 16, 32, 64, 1024, 0), ("flat", (489, 485), 8, 17, 64, 0, 1), ("half", (713, 709), 16, 30, 64, 1024, 0),
    ("extreme", (560, 816), 16, 24, 64, 1024, 0), ("extreme", (489, 485), 8, 24, 64, 1024, 1),
    ("periodic", (480, 480), 8, 20, 64, 0, 0), ("periodic", (713, 709), 16, 31, 64, 0, 1),
    ("constant", (560, 816), 16, 33, 13, 0, 0), ("constant", (489, 485), 8, 33, 9, 0, 1)])
def test_frame_search(oracle, kind, size, bs, rng, ctu, lam, shift):
    """shift: the reference plane starts at an odd sample and has an odd stride (rows of every alignment)."""
    import torch
    lib = capi.load()
    h, w = size
    pad = rng + 5
    cur, ref, _ = content(kind, h, w)
    refp = np.pad(ref, pad, mode="edge")
    rs = refp.shape[1] + (1 - refp.shape[1] % 2 if shift else refp.shape[1] % 2)      # odd when shifted, else even
    buf = np.zeros(shift + rs * refp.shape[0], np.uint16)
    buf[shift:].reshape(refp.shape[0], rs)[:, :refp.shape[1]] = refp
    cs = w + w % 2
    cbuf = np.zeros((h, cs), np.uint16)
    cbuf[:, :w] = cur
    dr, dc = (torch.from_numpy(b.view(np.int16)).cuda() for b in (buf, cbuf))
    pc = capi.XgPlane(dc.data_ptr(), cs, w, h, 0)
    pr = capi.XgPlane(dr.data_ptr() + 2 * (shift + pad * rs + pad), rs, w, h, pad)
    nb = (w // bs) * (h // bs)
    mv = torch.zeros(2 * nb, dtype=torch.int16, device="cuda")
    cost, sad = (torch.zeros(nb, dtype=torch.int32, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), 16) == 0
    try:
        assert lib.xg_full_search_frame(s, ctypes.byref(pc), ctypes.byref(pr), bs, bs, rng, lam, ctu, mv.data_ptr(),
                                        cost.data_ptr(), sad.data_ptr()) == 0
        assert lib.xg_session_sync(s) == 0
    finally:
        lib.xg_session_destroy(s)
    emx, emy, ec, es = oracle_search(oracle, cur, ref, bs, bs, rng, lam, ctu, pad)
    g = mv.cpu().numpy().reshape(nb, 2)
    assert np.array_equal(g[:, 0], emx) and np.array_equal(g[:, 1], emy)
    assert np.array_equal(cost.cpu().numpy().view(np.uint32), ec)
    assert np.array_equal(sad.cpu().numpy().view(np.uint32), es)


@pytest.mark.parametrize("kind,rng,ctu,lam,n", [
    ("texture", 16, 64, 1024, 4400), ("texture", 32, 48, 1024, 4000), ("texture", 16, 64, 1024, 3999),
    ("texture", 15, 64, 1024, 4000), ("texture", 16, 64, (1 << 21) + 1, 4000), ("half", 21, 64, 1024, 4100),
    ("flat", 16, 7, 0, 4000), ("extreme", 24, 64, 1024, 4000), ("extreme", 16, 64, 1 << 21, 4000),
    ("periodic", 19, 64, 0, 4000), ("constant", 16, 31, 0, 4000)])
def test_block_search(oracle, kind, rng, ctu, lam, n):
    """Session blocks of every shape, the large ones in their own launch, on both sides of the rule."""
    from tests.oracle_lib import OrMe
    from xin26x_amd.device import blocks_to_struct
    lib = capi.load()
    h, w, pad = 136, 200, 96
    cur, ref, _ = content(kind, h, w)
    half = lambda p: np.ascontiguousarray(p[::2, ::2])
    pics = [DevicePicture([p, half(p), half(p)], pad) for p in (cur, ref)]
    pred = DevicePicture.empty(w, h)
    r = np.random.default_rng(n + rng)
    sides, p = (4, 8, 16, 32, 64), (0.2, 0.3, 0.25, 0.15, 0.1)
    blocks = []
    for _ in range(n):
        bw, bh = (int(v) for v in r.choice(sides, 2, p=p))
        x, y = int(r.integers(0, (w - bw) // 4 + 1)) * 4, int(r.integers(0, (h - bh) // 4 + 1)) * 4
        blocks.append((x, y, bw, bh, 0, 0, int(r.integers(-600, 601)), int(r.integers(-600, 601))))
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), n) == 0
    try:
        for k in (0, 1):
            assert lib.xg_session_set_picture(s, k, pics[k].ref()) == 0
        barr = blocks_to_struct(blocks)
        assert lib.xg_session_set_blocks(s, barr.ctypes.data, n) == 0
        assert lib.xg_search_blocks(s, rng, lam, ctu) == 0
        cfg = refine_cfg([(0, 0)], wl.LAMBDA_REFINE, ctu)
        assert lib.xg_refine_frac(s, ctypes.byref(cfg), pred.ref(), capi.MODE_BATCHED) == 0
        best = np.zeros(n * 4, np.int32)
        assert lib.xg_session_read(s, None, best.ctypes.data) == 0
    finally:
        lib.xg_session_destroy(s)
    got = best.reshape(n, 4)[:, :2]
    refp = np.ascontiguousarray(np.pad(ref, pad, mode="edge"))
    rs, m = w + 2 * pad, ctu + 8

    def check(i):
        x, y, bw, bh, _, _, mvpx, mvpy = blocks[i]
        o = OrMe()
        o.width, o.height = bw, bh
        o.minMvX, o.minMvY, o.maxMvX, o.maxMvY = -x - m, -y - m, w + m - bw - x, h + m - bh - y
        # the search centre kept inside the window, as the block search keeps it
        o.predMvX, o.predMvY = mvpx >> 2, mvpy >> 2
        o.searchWidth = o.searchHeight = rng
        o.sadLambda = lam
        o.input = cur.ctypes.data + 2 * (y * w + x)
        o.inputStride = w
        o.ref = refp.ctypes.data + 2 * ((y + pad) * rs + x + pad)
        o.refStride = rs
        oracle.or_MotionEstFull(ctypes.byref(o))
        return (got[i, 0], got[i, 1]) == (4 * o.bestMvX, 4 * o.bestMvY)

    # predictors whose centre lies outside the window are not the oracle's form
    inside = [i for i, (x, y, bw, bh, _, _, px, py) in enumerate(blocks)
              if -x - m <= ((px >> 2) + 2) >> 2 <= w + m - bw - x and -y - m <= ((py >> 2) + 2) >> 2 <= h + m - bh - y]
    with ThreadPoolExecutor(8) as ex:
        bad = [i for i, ok in zip(inside, ex.map(check, inside)) if not ok]
    assert not bad, [blocks[i] for i in bad[:5]]
    assert len(inside) > n // 2


def search_session(lib, pics, blocks):
    """A session over the two pictures with these blocks installed."""
    from xin26x_amd.device import blocks_to_struct
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), len(blocks)) == 0
    for k in (0, 1):
        assert lib.xg_session_set_picture(s, k, pics[k].ref()) == 0
    barr = blocks_to_struct(blocks)
    assert lib.xg_session_set_blocks(s, barr.ctypes.data, len(blocks)) == 0
    return s


def searched(lib, pics, pred, blocks, rng, lam, ctu):
    """Best MVs of xg_search_blocks, read back through a refinement of one candidate at offset 0."""
    s = search_session(lib, pics, blocks)
    try:
        assert lib.xg_search_blocks(s, rng, lam, ctu) == 0
        cfg = refine_cfg([(0, 0)], wl.LAMBDA_REFINE, ctu)
        assert lib.xg_refine_frac(s, ctypes.byref(cfg), pred.ref(), capi.MODE_BATCHED) == 0
        best = np.zeros((len(blocks), 4), np.int32)
        assert lib.xg_session_read(s, None, best.ctypes.data) == 0
        return best[:, :2]
    finally:
        lib.xg_session_destroy(s)


@pytest.mark.parametrize("kind,rng,ctu,n,large,reach", [
    ("texture", 16, 64, 3700, 0.15, 2600), ("half", 24, 16, 6200, 0.5, 1500), ("periodic", 32, 33, 9100, 0.66, 2600),
    ("texture", 17, 64, 3001, 0.0, 2600), ("flat", 16, 7, 3500, 0.1, 600), ("flat", 25, 40, 3300, 0.0, 2600),
    ("noise", 32, 64, 3200, 0.0, 1500), ("constant", 19, 64, 3100, 0.0, 300)])
def test_block_search_is_that_of_short_lists(kind, rng, ctu, n, large, reach):
    """A long list of blocks in one call against the same blocks in calls below the rule, which search exhaustively:
    predictors far outside the window, many or no blocks too large for the bounds, at both ends of the list."""
    lib = capi.load()
    h, w, pad = 136, 200, 160
    cur, ref, _ = content(kind, h, w)
    half = lambda p: np.ascontiguousarray(p[::2, ::2])
    pics = [DevicePicture([p, half(p), half(p)], pad) for p in (cur, ref)]
    pred = DevicePicture.empty(w, h)
    r = np.random.default_rng(n)
    small, big = ((4, 4), (8, 8), (16, 8), (16, 16), (4, 32), (32, 16)), ((32, 32), (64, 64), (64, 8), (16, 64))
    blocks = []
    for i in range(n):
        t = big if (r.random() < large or (large and i in (0, n - 1))) else small
        bw, bh = t[int(r.integers(len(t)))]
        x, y = int(r.integers(0, (w - bw) // 4 + 1)) * 4, int(r.integers(0, (h - bh) // 4 + 1)) * 4
        blocks.append((x, y, bw, bh, 0, 0, int(r.integers(-reach, reach + 1)), int(r.integers(-reach, reach + 1))))
    assert sum((b[2] + 2 * rng) * (b[3] + 2 * rng) <= (16 + 2 * rng) * (32 + 2 * rng) for b in blocks) >= 3000
    m = ctu + 8
    outside = sum(not (-x - m <= ((px >> 2) + 2) >> 2 <= w + m - bw - x and -y - m <= ((py >> 2) + 2) >> 2 <= h + m - bh - y)
                  for x, y, bw, bh, _, _, px, py in blocks)
    assert outside > n // 20 or reach < 2000
    got = searched(lib, pics, pred, blocks, rng, 1024, ctu)
    exp = np.concatenate([searched(lib, pics, pred, blocks[k:k + 2500], rng, 1024, ctu) for k in range(0, n, 2500)])
    bad = np.flatnonzero((got != exp).any(1))
    assert bad.size == 0, [(blocks[i], got[i].tolist(), exp[i].tolist()) for i in bad[:4]]


def test_large_blocks_take_one_launch():
    """Blocks that the bounds do not take: a list of them is searched at once, and takes less time than its thirds in
    three sessions, which the rule leaves to the exhaustive search for their number."""
    import time
    lib = capi.load()
    h, w, pad = 2160, 3840, 96
    f = wl.smooth_field(h, w, 5)
    cur, ref = np.ascontiguousarray(f.astype(np.uint16)), np.ascontiguousarray(np.roll(f, 3, 1).astype(np.uint16))
    half = lambda p: np.ascontiguousarray(p[::2, ::2])
    pics = [DevicePicture([p, half(p), half(p)], pad) for p in (cur, ref)]
    blocks = [(x, y, 32, 32, 0, 0, 0, 0) for y in range(0, h - 31, 32) for x in range(0, w, 32)][:7500]
    parts = [[search_session(lib, pics, blocks)],
             [search_session(lib, pics, blocks[k:k + 2500]) for k in range(0, 7500, 2500)]]

    def us(sessions):
        t = []
        for _ in range(7):
            t0 = time.perf_counter()
            for s in sessions:                                # one after the other, several calls in flight
                for _ in range(6):
                    assert lib.xg_search_blocks(s, 16, 1024, 64) == 0
                assert lib.xg_session_sync(s) == 0
            t.append((time.perf_counter() - t0) / 6 * 1e6)
        return float(np.median(t[1:]))

    try:
        whole, thirds = us(parts[0]), us(parts[1])
        print(f"7,500 blocks of 32x32: whole {whole:.0f} us, in thirds {thirds:.0f}", flush=True)
        assert whole < 0.97 * thirds
    finally:
        for s in parts[0] + parts[1]:
            lib.xg_session_destroy(s)


def call_us(lib, s, call, n=4, reps=7):
    """Median time in us of a call, n in flight."""
    import time
    t = []
    for _ in range(reps):
        t0 = time.perf_counter()
        for _ in range(n):
            assert call() == 0
        assert lib.xg_session_sync(s) == 0
        t.append((time.perf_counter() - t0) / n * 1e6)
    return float(np.median(t[1:]))


EXHAUSTIVE = (1 << 21) + 1             # a rate weight past the rules: the same call, every SAD


def test_flat_frames_cost_little_more_in_the_pipeline():
    """A flat noisy frame, whose blocks all end in the exhaustive search, against the exhaustive form."""
    lib = capi.load()
    h, w, pad = 1088, 1920, 96
    half = lambda p: np.ascontiguousarray(p[::2, ::2])
    pics = [DevicePicture([p, half(p), half(p)], pad) for p in content("flat", h, w)]
    pred = DevicePicture.empty(w, h)
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), (w // 16) * (h // 16)) == 0
    try:
        us = []
        for lam in (1024, EXHAUSTIVE):
            cfg = capi.XgPipelineCfg()
            cfg.range, cfg.sadLambda, cfg.ctuSize = 64, lam, 64
            cfg.refine = refine_cfg([(0, 0)], wl.LAMBDA_REFINE)
            us.append(call_us(lib, s, lambda: lib.xg_me_pipeline(s, ctypes.byref(cfg), pics[0].ref(), pics[1].ref(),
                                                                 pics[2].ref(), pred.ref(), capi.MODE_BATCHED)))
        print(f"flat 1920x1088 +/-64: bounded {us[0]:.0f} us, exhaustive {us[1]:.0f}", flush=True)
        assert us[0] < 1.24 * us[1]
    finally:
        lib.xg_session_destroy(s)


def test_noisy_frames_cost_little_more():
    """Frame search of content whose bounds exclude little, against the exhaustive form."""
    import torch
    lib = capi.load()
    h, w = 720, 1280
    cur, ref = (DevicePicture([p, p[::2, ::2].copy(), p[::2, ::2].copy()], 96) for p in content("noise", h, w)[:2])
    nb = (w // 16) * (h // 16)
    out = [torch.zeros(2 * nb, dtype=torch.int32, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    s = ctypes.c_void_p()
    assert lib.xg_session_create(ctypes.byref(s), 16) == 0
    try:
        us = [call_us(lib, s, lambda: lib.xg_full_search_frame(
            s, ctypes.byref(cur.pic.plane[0]), ctypes.byref(ref.pic.plane[0]), 16, 16, 16, lam, 64,
            *[t.data_ptr() for t in out]), n=20) for lam in (1024, EXHAUSTIVE)]
    finally:
        lib.xg_session_destroy(s)
    print(f"noise, 1280x720 16x16 +/-16: bounded {us[0]:.0f} us, exhaustive {us[1]:.0f}", flush=True)
    assert us[0] < 1.5 * us[1]


def test_flat_blocks_cost_little_more():
    """Block search of flat noisy content, where the bounds exclude nothing, against the exhaustive form."""
    lib = capi.load()
    h, w = 1088, 1920
    half = lambda p: np.ascontiguousarray(p[::2, ::2])
    pics = [DevicePicture([p, half(p), half(p)], 96) for p in content("flat", h, w)[:2]]
    s = search_session(lib, pics, [(x, y, 16, 16, 0, 0, 0, 0) for y in range(0, h, 16) for x in range(0, w, 16)])
    try:
        us = [call_us(lib, s, lambda: lib.xg_search_blocks(s, 16, lam, 64), n=10) for lam in (1024, EXHAUSTIVE)]
    finally:
        lib.xg_session_destroy(s)
    print(f"flat 1920x1088 16x16 blocks +/-16: bounded {us[0]:.0f} us, exhaustive {us[1]:.0f}", flush=True)
    assert us[0] < 1.2 * us[1]
