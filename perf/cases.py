"""The work that programs have this library do, as cases that can be timed and compared.

A case names a path (a group of public entry points of include/xg266.h, called through
xin26x_amd.capi as any program would) and its sizes.  listed() are the fixed cases, draw()
gives more of the same ranges.  Pictures are 10-bit 4:2:0, made on the GPU from the seed:
textures with energy at every scale (strong coarse, weaker fine detail, flat and busy areas),
motion that is constant per 64x64 CTU at 1/16-pel precision, and sensor noise on the current
picture.  Partitions are the QTMT splits of xin26x_amd.workloads.  Every output is a whole
number and has one right value, so the tolerance of every case is "exact".
"""
import ctypes
import math
import os
import random

import numpy as np
import torch

from xin26x_amd import capi, workloads as wl
from xin26x_amd.capi import XgPicture, XgPlane
from xin26x_amd.device import BLOCK_DTYPE, refine_cfg
from xin26x_amd.serve import Server, server_cfg

PAD = 80                      # luma padding of a picture for 64x64 CTUs
LAMBDA_INT = 1024             # sadLambda of the integer searches
DEV = "cuda"


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one CU through the drop-in table, host buffers, one call after the other, as an encoder's worker
        # thread makes them: diamond search, half/quarter-pel refinement, interpolation, SATD
        {"name": "slots_16x16", "path": "slots", "w": 16, "h": 16, "noise": 4},
        # a small picture's fractional refinement, replayed from the captured graph: latency
        {"name": "refine_416x240", "path": "refine", "width": 416, "height": 240, "ncand": 32, "chroma": 1,
         "mode": "graph", "tuned": 0, "noise": 4},
        # the headline: a 1080p frame's QTMT blocks, 32 fractional candidates each, luma and chroma, with MC
        {"name": "refine_1080p", "path": "refine", "width": 1920, "height": 1080, "ncand": 32, "chroma": 1,
         "mode": "batched", "tuned": 1, "noise": 4},
        # integer full search of a small picture on the 16x16 grid
        {"name": "search_416x240", "path": "search", "width": 416, "height": 240, "bw": 16, "bh": 16, "range": 16,
         "noise": 4},
        # a 720p frame's QTMT blocks: AMVP predictor choice, then the integer search around the predictors
        {"name": "blocks_720p", "path": "blocks", "width": 1280, "height": 720, "range": 16, "imv": 0, "noise": 4},
        # lookahead of a 1080p pair: half-resolution pictures, +/-32
        {"name": "lookahead_1080p", "path": "lookahead", "width": 1920, "height": 1080, "unit": 16, "range": 32,
         "noise": 4},
        # temporal-filter motion of a 1080p pair, four levels down to 1/16 pel
        {"name": "mctf_1080p", "path": "mctf", "width": 1920, "height": 1080, "noise": 4},
        # the whole motion search of a 4K frame against two references, one graph per frame: the largest
        {"name": "pipeline_4k", "path": "pipeline", "width": 3840, "height": 2160, "range": 64, "mode": "graph",
         "noise": 4},
        # a 1080p B frame: decoder-side refinement of its bi-predicted blocks, then their bi-prediction cost
        {"name": "bi_1080p", "path": "bi", "width": 1920, "height": 1080, "satd": 1, "noise": 4},
        # a frame's TUs through transform, quantiser and reconstruction as three calls (RDOQ reads the coefficients)
        {"name": "residual_20k", "path": "residual", "blocks": 20000, "fused": 0, "qp": 27, "noise": 4},
        # a batch of frames' TUs with the quantiser fused into the transform
        {"name": "residual_200k", "path": "residual", "blocks": 200000, "fused": 1, "qp": 22, "noise": 4},
        # the serving mix: two frames of each of 16 streams offered at once, results back in pinned memory
        {"name": "serve_16", "path": "serve", "s360": 6, "s720": 6, "s1080": 4, "ticks": 2, "noise": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["slots", "refine", "refine", "search", "blocks", "lookahead", "mctf", "pipeline", "bi",
                       "residual", "residual", "serve"])
    noise = rng.randint(1, 8)

    def frame(lo, hi, step):
        area = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        aspect = rng.uniform(1.0, 2.2)
        w = max(64, int(math.sqrt(area * aspect)) // step * step)
        h = max(64, int(math.sqrt(area / aspect)) // step * step)
        return w, h

    if path == "slots":
        return {"path": path, "w": rng.choice([4, 8, 16, 32, 64, 128]), "h": rng.choice([4, 8, 12, 16, 32, 64, 128]),
                "noise": noise}
    if path == "refine":
        w, h = frame(64 * 64, 2560 * 1440, 8)
        return {"path": path, "width": w, "height": h, "ncand": rng.choice([5, 8, 9, 17, 24, 32, 32, 48]),
                "chroma": rng.choice([0, 1, 1, 1]), "mode": rng.choice(["batched", "graph"]), "tuned": rng.randint(0, 1),
                "noise": noise}
    if path == "search":
        w, h = frame(64 * 64, 1920 * 1080, 1)
        return {"path": path, "width": w, "height": h, "bw": rng.choice([4, 8, 16, 16, 32]),
                "bh": rng.choice([4, 8, 12, 16, 16, 32]), "range": _log(rng, 4, 48), "noise": noise}
    if path == "blocks":
        w, h = frame(64 * 64, 1920 * 1080, 4)
        return {"path": path, "width": w, "height": h, "range": _log(rng, 4, 24), "imv": rng.randint(0, 3),
                "noise": noise}
    if path == "lookahead":
        w, h = frame(128 * 128, 3840 * 2160, 1)
        return {"path": path, "width": w, "height": h, "unit": rng.choice([8, 16]), "range": _log(rng, 8, 40),
                "noise": noise}
    if path == "mctf":
        w, h = frame(128 * 128, 3840 * 2160, 1)
        return {"path": path, "width": w, "height": h, "noise": noise}
    if path == "pipeline":
        w, h = frame(128 * 128, 2560 * 1440, 16)
        return {"path": path, "width": w, "height": h, "range": _log(rng, 8, 64),
                "mode": rng.choice(["batched", "graph"]), "noise": noise}
    if path == "bi":
        w, h = frame(128 * 128, 3840 * 2160, 8)
        return {"path": path, "width": w, "height": h, "satd": rng.randint(0, 1), "noise": noise}
    if path == "residual":
        return {"path": path, "blocks": _log(rng, 30, 160000), "fused": rng.randint(0, 1), "qp": rng.randint(12, 45),
                "noise": noise}
    return {"path": path, "s360": rng.randint(1, 7), "s720": rng.randint(0, 5), "s1080": rng.randint(0, 3),
            "ticks": rng.randint(1, 3), "noise": rng.randint(1, 4)}


# ---------------------------------------------------------------------------
# Pictures
# ---------------------------------------------------------------------------
def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)
    return g


def _texture(g, h, w):
    """float32 h x w: noise octaves, the fine ones scaled by a smooth activity map."""
    out = torch.full((1, 1, h, w), 500.0, device=DEV)
    act = torch.nn.functional.interpolate(torch.rand((1, 1, h // 96 + 3, w // 96 + 3), generator=g, device=DEV),
                                          size=(h, w), mode="bilinear")
    for scale, amp in ((64, 85.0), (32, 70.0), (16, 55.0), (8, 40.0), (4, 26.0), (2, 14.0), (1, 7.0)):
        n = torch.randn((1, 1, -(-h // scale) + 2, -(-w // scale) + 2), generator=g, device=DEV)
        if scale > 1:
            n = torch.nn.functional.interpolate(n, size=(n.shape[2] * scale, n.shape[3] * scale), mode="bicubic")
        n = n[:, :, :h, :w] * amp
        out += n * (2 * act) if scale <= 16 else n
    return out


def _sample(canvas, margin, dx, dy):
    """The h x w window of a canvas (margin samples around it) displaced per sample by (dx, dy)."""
    h, w = dx.shape
    ys = torch.arange(h, device=DEV, dtype=torch.float32)[:, None] + margin + dy
    xs = torch.arange(w, device=DEV, dtype=torch.float32)[None, :] + margin + dx
    H, W = canvas.shape[2:]
    grid = torch.stack(((xs + 0.5) * (2.0 / W) - 1, (ys + 0.5) * (2.0 / H) - 1), dim=-1)[None]
    return torch.nn.functional.grid_sample(canvas, grid, mode="bicubic", padding_mode="border", align_corners=False)


def _finish(p, g, noise, pad):
    if noise:
        p = p + torch.randn(p.shape, generator=g, device=DEV) * noise
    p = p.round().clamp(0, 1023)
    if pad:
        p = torch.nn.functional.pad(p, (pad, pad, pad, pad), mode="replicate")
    return p[0, 0].to(torch.int16).contiguous()


class Pic:
    """Planes on the GPU and their xg_picture (chroma planes at half size and half padding)."""

    def __init__(self, tensors, pads, sizes):
        self.t = tensors
        self.pic = XgPicture()
        for p, (t, pad, (h, w)) in enumerate(zip(tensors, pads, sizes)):
            st = t.shape[1]
            self.pic.plane[p] = XgPlane(t.data_ptr() + 2 * (pad * st + pad), st, w, h, pad)

    def luma(self):
        return ctypes.byref(self.pic.plane[0])

    def ref(self):
        return ctypes.byref(self.pic)


def _sizes(w, h, luma_only):
    return [(h, w)] if luma_only else [(h, w), (h // 2, w // 2), (h // 2, w // 2)]


def _scene(seed, w, h, noise, frames=2, luma_only=False, pad=PAD, reach=32):
    """`frames` pictures, oldest first: the last is the current one (noisy), the others are references; and the
    MV of every CTU of the current picture against the newest reference (1/16 pel, ncty x nctx x 2)."""
    g = _gen(seed, 1)
    ncx, ncy = -(-w // 64), -(-h // 64)
    r = 16 * reach
    # regional motion: a global pan, most CTUs near it, some of their own
    pan = torch.randint(-r // 2, r // 2 + 1, (2,), generator=g, device=DEV)
    mv = pan + torch.randint(-48, 49, (ncy, ncx, 2), generator=g, device=DEV)
    own = torch.rand((ncy, ncx, 1), generator=g, device=DEV) < 0.2
    mv = torch.where(own, torch.randint(-r, r + 1, (ncy, ncx, 2), generator=g, device=DEV), mv).clamp(-r, r)
    out = [[] for _ in range(frames)]
    for p, (ph, pw) in enumerate(_sizes(w, h, luma_only)):
        sub = 2 if p else 1
        m = (2 * reach + 16) // sub
        canvas = _texture(g, ph + 2 * m, pw + 2 * m)
        if p:
            canvas = 512 + (canvas - 500) * 0.5
        d = mv.float() / (16 * sub)
        d = d.repeat_interleave(64 // sub, 0).repeat_interleave(64 // sub, 1)[:ph, :pw]
        pp = pad if not p else pad // 2
        for f in range(frames):
            k = frames - 2 - f               # newest reference is the window itself, older ones the opposite way
            s = _sample(canvas, m, -d[..., 0] * k, -d[..., 1] * k)
            out[f].append(_finish(s, g, noise if f == frames - 1 else 0.5 * noise, pp))
    pads = [pad, pad // 2, pad // 2]
    pics = [Pic(t, pads, _sizes(w, h, luma_only)) for t in out]
    return pics, mv.cpu().numpy().astype(np.int64)


_PARTS = {}


def _ctu_bank(w, h):
    """Partitions of a CTU of which w x h samples lie in the picture."""
    if (w, h) not in _PARTS:
        n = 48 if (w, h) == (64, 64) else 4
        _PARTS[w, h] = [np.array(wl.qtmt_partition(0, 0, w, h, 977 * k + 31 * w + h), np.int64).reshape(-1, 4)
                        for k in range(n)]
    return _PARTS[w, h]


def _blocks(seed, w, h, mv, jitter=0):
    """QTMT blocks (struct array as xg_block) with their CTU's MV rounded to integer pel as base and predictor (plus
    up to jitter sixteenths).  A picture size has one partition, so outputs have the same size for every seed."""
    r = np.random.default_rng(w * 8191 + h)
    parts = []
    for cy in range(-(-h // 64)):
        for cx in range(-(-w // 64)):
            bank = _ctu_bank(min(64, w - 64 * cx), min(64, h - 64 * cy))
            b = bank[int(r.integers(len(bank)))]
            q = np.zeros((len(b), 6), np.int64)
            q[:, :4] = b
            q[:, 0] += 64 * cx
            q[:, 1] += 64 * cy
            q[:, 4:] = mv[cy, cx]
            parts.append(q)
    q = np.concatenate(parts)
    a = np.zeros(len(q), BLOCK_DTYPE)
    for i, n in enumerate(("x", "y", "w", "h")):
        a[n] = q[:, i]
    a["ref"] = 1
    r = np.random.default_rng(seed * 7 + 5)
    e = r.integers(-jitter, jitter + 1, (len(q), 2)) if jitter else np.zeros((len(q), 2), np.int64)
    for i, n in enumerate(("x", "y")):
        a["mv" + n] = ((q[:, 4 + i] + 8) >> 4) << 4
        a["mvp" + n] = a["mv" + n] + e[:, i]
    return a


def _offsets(n):
    """The first n candidates of: the zero offset for odd counts, then rings at 8, 4, 12, 2, 6, 1 sixteenths."""
    ring = [(-1, 0), (1, 0), (0, -1), (0, 1), (-1, -1), (1, -1), (-1, 1), (1, 1)]
    if n == 17:
        return list(wl.CAND17_SIXTEENTH)
    out = [(0, 0)] if n % 2 else []
    for r in (8, 4, 12, 2, 6, 1):
        out += [(dx * r, dy * r) for dx, dy in ring]
    return out[:n]


# ---------------------------------------------------------------------------
# States
# ---------------------------------------------------------------------------
class _Ptr:
    """A device array of a session, for torch.as_tensor; the tensor keeps the session's handle alive."""

    def __init__(self, ptr, n, handle, typestr="<i4"):
        self.handle = handle
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (n,), "typestr": typestr, "version": 2}


class _Handle:
    """Owns an xg_session: destroyed with the last state or output that refers to it."""

    def __init__(self, max_blocks):
        self.lib = capi.load()
        self.s = ctypes.c_void_p()
        capi.check(self.lib.xg_session_create(ctypes.byref(self.s), max_blocks), "session")

    def __del__(self):
        if self.s:
            self.lib.xg_session_destroy(self.s)


class Session:
    def __init__(self, max_blocks=16):
        self.handle = _Handle(max_blocks)
        self.lib, self.s = self.handle.lib, self.handle.s

    def outputs(self, n, ncand):
        c, b = ctypes.c_void_p(), ctypes.c_void_p()
        capi.check(self.lib.xg_session_outputs(self.s, ctypes.byref(c), ctypes.byref(b)), "outputs")
        return [torch.as_tensor(_Ptr(c.value, n * ncand, self.handle), device=DEV),
                torch.as_tensor(_Ptr(b.value, 4 * n, self.handle), device=DEV)]


def _empty(n, dtype=torch.int32):
    return torch.zeros(n, dtype=dtype, device=DEV)


def _empty_pic(w, h):
    t = [torch.zeros(s, dtype=torch.int16, device=DEV) for s in _sizes(w, h, False)]
    return Pic(t, [0, 0, 0], _sizes(w, h, False))


class Refine(Session):
    def __init__(self, c, seed):
        (ref, cur), mv = _scene(seed, c["width"], c["height"], c["noise"])
        b = _blocks(seed, c["width"], c["height"], mv)
        super().__init__(len(b))
        self.keep = (ref, cur, b)
        self.pred = _empty_pic(c["width"], c["height"])
        self.cfg = refine_cfg(_offsets(c["ncand"]), wl.LAMBDA_REFINE, use_chroma=c["chroma"])
        self.mode = capi.MODE_GRAPH if c["mode"] == "graph" else capi.MODE_BATCHED
        if c["tuned"]:
            path = os.path.join(os.path.dirname(capi.__file__), "tuned", "refine_1080p_cand32.txt")
            capi.check(self.lib.xg_session_load_tiles(self.s, path.encode()), "tiles")
        capi.check(self.lib.xg_session_set_picture(self.s, 0, cur.ref()), "set_picture")
        capi.check(self.lib.xg_session_set_picture(self.s, 1, ref.ref()), "set_picture")
        capi.check(self.lib.xg_session_set_blocks(self.s, b.ctypes.data, len(b)), "set_blocks")
        self.out = self.outputs(len(b), c["ncand"]) + self.pred.t

    def run(self):
        capi.check(self.lib.xg_refine_frac(self.s, ctypes.byref(self.cfg), self.pred.ref(), self.mode), "refine")
        return self.out


class Search(Session):
    def __init__(self, c, seed):
        super().__init__()
        (self.ref, self.cur), _ = _scene(seed, c["width"], c["height"], c["noise"], luma_only=True,
                                         reach=min(32, c["range"]))
        self.c = c
        n = (c["width"] // c["bw"]) * (c["height"] // c["bh"])
        self.out = [_empty(2 * n, torch.int16), _empty(n), _empty(n)]

    def run(self):
        c, o = self.c, self.out
        capi.check(self.lib.xg_full_search_frame(self.s, self.cur.luma(), self.ref.luma(), c["bw"], c["bh"], c["range"],
                                                 LAMBDA_INT, 64, *[t.data_ptr() for t in o]), "full search")
        return o


class Blocks(Session):
    """xg_amvp_select of every block's two candidates, and xg_search_blocks of the session's blocks, whose base
    MVs the following xg_refine_frac (here with one candidate, costs and MC) starts from."""

    def __init__(self, c, seed):
        (ref, cur), mv = _scene(seed, c["width"], c["height"], c["noise"], reach=24)
        b = _blocks(seed, c["width"], c["height"], mv, jitter=6 * 16)
        super().__init__(len(b))
        n = len(b)
        r = np.random.default_rng(seed * 11 + 3)
        a = (capi.XgAmvpBlock * n)()
        v = np.frombuffer(a, dtype=np.dtype([("x", "<i2"), ("y", "<i2"), ("w", "u1"), ("h", "u1"), ("pic", "u1"),
                                             ("ref", "u1"), ("ncand", "<i4"), ("cand", "<i4", (4,))]))
        for k in ("x", "y", "w", "h", "pic", "ref"):
            v[k] = b[k]
        v["ncand"] = np.where(r.random(n) < 0.15, 1, 2)
        base = np.stack([b["mvpx"], b["mvpy"]], 1)
        v["cand"] = np.concatenate([base + r.integers(-40, 41, (n, 2)), base + r.integers(-80, 81, (n, 2))], 1)
        self.amvp = torch.from_numpy(np.frombuffer(a, np.uint8).copy()).to(DEV)
        self.n, self.c, self.keep = n, c, (ref, cur, b)
        self.sel = _empty(5 * n)
        self.pred = _empty_pic((c["width"] + 7) & ~7, (c["height"] + 7) & ~7)
        self.cfg = refine_cfg([(0, 0)], wl.LAMBDA_REFINE, use_chroma=0)
        capi.check(self.lib.xg_session_set_picture(self.s, 0, cur.ref()), "set_picture")
        capi.check(self.lib.xg_session_set_picture(self.s, 1, ref.ref()), "set_picture")
        capi.check(self.lib.xg_session_set_blocks(self.s, b.ctypes.data, n), "set_blocks")
        self.out = [self.sel] + self.outputs(n, 1) + self.pred.t

    def run(self):
        lib, s, c = self.lib, self.s, self.c
        capi.check(lib.xg_amvp_select(s, self.amvp.data_ptr(), self.n, c["imv"], 64, self.sel.data_ptr()), "amvp")
        capi.check(lib.xg_search_blocks(s, c["range"], LAMBDA_INT, 64), "search")
        capi.check(lib.xg_refine_frac(s, ctypes.byref(self.cfg), self.pred.ref(), capi.MODE_BATCHED), "refine")
        return self.out


class Lookahead(Session):
    def __init__(self, c, seed):
        super().__init__()
        pad = max(PAD, 2 * (c["range"] + 4))
        (self.ref, self.cur), _ = _scene(seed, c["width"], c["height"], c["noise"], luma_only=True, pad=pad)
        self.c = c
        n = (c["width"] // 2 // c["unit"]) * (c["height"] // 2 // c["unit"])
        self.out = [_empty(2 * n, torch.int16), _empty(n), _empty(n)]

    def run(self):
        c, o = self.c, self.out
        capi.check(self.lib.xg_lookahead_me(self.s, self.cur.luma(), self.ref.luma(), c["unit"], c["range"], LAMBDA_INT,
                                            *[t.data_ptr() for t in o]), "lookahead")
        return o


class Mctf(Session):
    def __init__(self, c, seed):
        super().__init__()
        (self.ref, self.cur), _ = _scene(seed, c["width"], c["height"], c["noise"], luma_only=True, reach=16)
        n = (c["width"] // 8) * (c["height"] // 8)
        self.out = [_empty(2 * n), _empty(n)]

    def run(self):
        o = self.out
        capi.check(self.lib.xg_mctf_me(self.s, self.cur.luma(), self.ref.luma(), o[0].data_ptr(), o[1].data_ptr()), "mctf")
        return o


class Pipeline(Session):
    def __init__(self, c, seed):
        w, h = c["width"], c["height"]
        n = (w // 16) * (h // 16)
        super().__init__(n)
        (self.ref1, self.ref0, self.cur), _ = _scene(seed, w, h, c["noise"], frames=3, reach=min(32, c["range"]))
        self.pred = _empty_pic(w, h)
        self.cfg = capi.XgPipelineCfg()
        self.cfg.range, self.cfg.sadLambda, self.cfg.ctuSize = c["range"], LAMBDA_INT, 64
        self.cfg.refine = refine_cfg(wl.CAND17_SIXTEENTH, wl.LAMBDA_REFINE)
        self.mode = capi.MODE_GRAPH if c["mode"] == "graph" else capi.MODE_BATCHED
        self.out = self.outputs(n, 17) + self.pred.t

    def run(self):
        capi.check(self.lib.xg_me_pipeline(self.s, ctypes.byref(self.cfg), self.cur.ref(), self.ref0.ref(),
                                           self.ref1.ref(), self.pred.ref(), self.mode), "pipeline")
        return self.out


class Bi(Session):
    def __init__(self, c, seed):
        super().__init__()
        w, h = c["width"], c["height"]
        (self.ref1, self.ref0, self.cur), mv = _scene(seed, w, h, c["noise"], frames=3, luma_only=True, reach=16)
        b = _blocks(seed, w, h, mv)
        r = np.random.default_rng(seed * 13 + 1)
        sel = b[(b["w"] >= 8) & (b["h"] >= 8) & (b["w"].astype(int) * b["h"] >= 128)]
        n = len(sel)
        d = (capi.XgDmvrBlock * n)()
        v = np.frombuffer(d, dtype=np.dtype([("x", "<i4"), ("y", "<i4"), ("w", "<i4"), ("h", "<i4"), ("mv", "<i4", (4,)),
                                             ("win", "<i2", (4,))]))
        for k in ("x", "y", "w", "h"):
            v[k] = sel[k]
        off = r.integers(-12, 13, (n, 4))
        base = np.stack([sel["mvx"], sel["mvy"]], 1).astype(np.int64)
        v["mv"] = np.concatenate([base, -base], 1) + off
        v["win"] = np.stack([-72 - v["x"], -72 - v["y"], w - v["x"] - v["w"] + 72, h - v["y"] - v["h"] + 72], 1)
        sub = np.zeros(n + 1, np.int32)
        capi.check(self.lib.xg_dmvr_plan(self.s, d, n, sub.ctypes.data), "dmvr plan")
        capi.check(self.lib.xg_bipred_plan(self.s, b.ctypes.data, len(b)), "bipred plan")
        self.c, self.b = c, b
        self.out = [_empty(2 * int(sub[-1]), torch.int16), _empty(len(b))]

    def run(self):
        lib, s, o = self.lib, self.s, self.out
        capi.check(lib.xg_dmvr_run(s, self.ref0.luma(), self.ref1.luma(), o[0].data_ptr()), "dmvr")
        capi.check(lib.xg_bipred_run(s, self.cur.luma(), self.ref0.luma(), self.ref1.luma(), self.c["satd"],
                                     o[1].data_ptr()), "bipred")
        return o


def _tus(n):
    """n TUs: descriptors, offsets and the sample count (shapes as workloads.residual_blocks draws them)."""
    r = np.random.default_rng(n * 17 + 9)
    sides = np.array(sorted(wl.SIDE_WEIGHTS))
    p = np.array([wl.SIDE_WEIGHTS[s] for s in sides])
    w, h = sides[r.choice(len(sides), n, p=p / p.sum())], sides[r.choice(len(sides), n, p=p / p.sum())]
    mts = np.where((w <= 32) & (h <= 32), np.array([0, 0, 2, 3, 4, 5])[r.integers(0, 6, n)], 0)
    desc = (np.log2(w).astype(np.int64) | np.log2(h).astype(np.int64) << 4 | mts << 8).astype(np.uint32)
    size = w * h
    offs = np.concatenate([[0], np.cumsum(size)[:-1]]).astype(np.int64)
    return desc, offs, int(size.sum())


class Residual(Session):
    def __init__(self, c, seed):
        super().__init__()
        n = c["blocks"]
        desc, offs, total = _tus(n)
        g = _gen(seed, 2)
        u = torch.rand(total, generator=g, device=DEV) - 0.5
        lap = -3.0 * c["noise"] * torch.sign(u) * torch.log((1 - 2 * u.abs()).clamp_min(1e-30))
        self.resid = lap.round().clamp(-1023, 1023).to(torch.int16)
        self.pred = torch.randint(0, 1024, (total,), generator=g, device=DEV).to(torch.int16)
        q = ((desc & 0xFFF) | 2 << 12 | 2 << 15 | (c["qp"] + 12) << 18).astype(np.uint32)
        self.q, self.r, self.rec = (_empty(total, torch.int16) for _ in range(3))
        self.nz = _empty(n, torch.int64)
        self.coeff = None if c["fused"] else _empty(total)
        if c["fused"]:
            capi.check(self.lib.xg_fdct_quant_plan(self.s, offs.ctypes.data, desc.ctypes.data, q.ctypes.data, n), "plan")
        else:
            capi.check(self.lib.xg_fdct_plan(self.s, offs.ctypes.data, desc.ctypes.data, n), "plan")
            capi.check(self.lib.xg_quant_plan(self.s, offs.ctypes.data, q.ctypes.data, n), "plan")
        capi.check(self.lib.xg_recon_plan(self.s, offs.ctypes.data, desc.ctypes.data, n), "plan")
        self.out = [self.q, self.r, self.nz, self.rec] + ([] if c["fused"] else [self.coeff])

    def run(self):
        lib, s = self.lib, self.s
        if self.coeff is None:
            capi.check(lib.xg_fdct_quant_run(s, self.resid.data_ptr(), self.q.data_ptr(), self.r.data_ptr(),
                                             self.nz.data_ptr()), "fdct + quant")
        else:
            capi.check(lib.xg_fdct_run(s, self.resid.data_ptr(), self.coeff.data_ptr()), "fdct")
            capi.check(lib.xg_quant_run(s, self.coeff.data_ptr(), self.q.data_ptr(), self.r.data_ptr(),
                                        self.nz.data_ptr()), "quant")
        capi.check(lib.xg_recon_run(s, self.r.data_ptr(), self.pred.data_ptr(), self.rec.data_ptr()), "recon")
        return self.out


class Slots:
    """Host buffers of one CU, as an encoder's worker holds them."""

    def __init__(self, c, seed):
        self.lib, self.c = capi.load(), c
        w, h = c["w"], c["h"]
        g = torch.Generator().manual_seed(int(seed) * 5 + 1)
        W, H = w + 2 * PAD, h + 2 * PAD
        t = 500 + sum(torch.nn.functional.interpolate(torch.randn(1, 1, H // s + 2, W // s + 2, generator=g), size=(H, W),
                                                      mode="bicubic") * a for s, a in ((32, 90), (8, 50), (3, 20)))
        m = (3 + seed % 5, -2 - seed % 3)
        ref = t[0, 0]
        cur = torch.roll(ref, (m[1], m[0]), (0, 1)) + torch.randn(H, W, generator=g) * c["noise"]
        conv = lambda x: np.ascontiguousarray(x.round().clamp(0, 1023).to(torch.int16).numpy().view(np.uint16))  # noqa: E731
        self.refb, self.curb, self.stride = conv(ref), conv(cur), W
        self.at = PAD * W + PAD
        self.dst = np.zeros((h, w), np.uint16)
        self.satd = np.zeros(1, np.uint32)
        me = capi.XgMeStruct()
        me.width, me.height = w, h
        me.minMv, me.maxMv = capi.XgMv(-32, -32), capi.XgMv(32, 32)
        for k, (x, y) in enumerate(((0, 0), (-2, 1), (4, -4))):
            me.meCand[k] = capi.XgMv(x, y)
        me.candNum, me.predMv = 3, capi.XgMv(2, -3)
        me.searchWidth = me.searchHeight = 16
        me.sadLambda = LAMBDA_INT
        me.input, me.inputStride = self.curb.ctypes.data + 2 * self.at, W
        me.ref, me.refStride = self.refb.ctypes.data + 2 * self.at, W
        self.me = me
        self.pcur, self.pref = me.input, me.ref
        self.frac = ((1 + 3 * (seed % 5)) << 4) | (2 + 2 * (seed % 7))

    def run(self):
        lib, c, me, W = self.lib, self.c, self.me, self.stride
        lib.Xg26xMotionEstDia(ctypes.byref(me))
        ix, iy, icost, isad = me.bestMv.mvX, me.bestMv.mvY, me.bestCost, me.bestSad
        lib.Xg266FullSubPelMe(ctypes.byref(me))
        lib.Xg266LumaInterpHorVet(self.pref, W, self.dst.ctypes.data, c["w"], self.frac, c["w"], c["h"], 0)
        lib.Xg266ComputeSatd(self.pcur, W, self.dst.ctypes.data, c["w"], c["w"], c["h"], self.satd.ctypes.data)
        return {"int": np.array([ix, iy, icost, isad], np.int64),
                "sub": np.array([me.bestMv.mvX, me.bestMv.mvY, me.bestCost], np.int64),
                "pred": self.dst.astype(np.int32), "satd": self.satd.astype(np.int64)}


class Serve:
    RING = 4

    def __init__(self, c, seed):
        sizes = [(640, 360)] * c["s360"] + [(1280, 720)] * c["s720"] + [(1920, 1080)] * c["s1080"]
        self.frames, self.blocks = [], []
        for k, (w, h) in enumerate(sizes):
            g = _gen(seed, 100 + k)
            r = random.Random(seed * 31 + k)
            vx, vy = r.uniform(-6, 6), r.uniform(-4, 4)
            ring = [[] for _ in range(self.RING)]
            for p, (ph, pw) in enumerate(_sizes(w, h, False)):
                sub = 2 if p else 1
                canvas = _texture(g, ph + 64 // sub, pw + 64 // sub)
                one = torch.ones((ph, pw), device=DEV)
                for f in range(self.RING):
                    s = _sample(canvas, 32 // sub, one * (vx * f / sub), one * (vy * f / sub))
                    ring[f].append(_finish(s, g, c["noise"], 0))
            self.frames.append(ring)
            self.blocks.append(_blocks(seed + k, w, h, np.zeros((-(-h // 64), -(-w // 64), 2), np.int64)))
        n = [len(b) for b in self.blocks]
        cap = min([max(sum(n[:k]), sum(n[k:])) for k in range(1, len(n))] or [sum(n)])
        self.srv = Server(server_cfg(cap))
        self.sizes, self.c, self.t = sizes, c, 0
        self.sid = []
        for w, h in sizes:
            rc, sid = self.srv.open(w, h)
            capi.check(rc, "open_stream")
            self.sid.append(sid)
        self.res = torch.zeros((c["ticks"], 4 * sum(n)), dtype=torch.int32).pin_memory()
        self.at = np.concatenate([[0], np.cumsum(n)])
        self.first = True

    def __del__(self):
        if getattr(self, "srv", None):
            self.srv.destroy()

    def run(self):
        srv, ticks = self.srv, self.c["ticks"]
        for k in range(ticks):
            for i, (w, h) in enumerate(self.sizes):
                f = self.frames[i][self.t % self.RING]
                capi.check(srv.submit_frame(self.sid[i], [p.data_ptr() for p in f], [w, w // 2, w // 2],
                                            capi.XG_MEM_DEVICE, self.res[k].data_ptr() + 16 * int(self.at[i]),
                                            capi.XG_MEM_HOST_PINNED, self.blocks[i] if self.first else None), "submit")
            self.first = False
            self.t += 1
        left = ticks * len(self.sizes)
        while left > 0:
            for r in srv.poll(64, 100):
                capi.check(r.status, "frame")
                left -= 1
        return self.res


PATHS = {"slots": Slots, "refine": Refine, "search": Search, "blocks": Blocks, "lookahead": Lookahead, "mctf": Mctf,
         "pipeline": Pipeline, "bi": Bi, "residual": Residual, "serve": Serve}


def prepare(case, seed):
    st = PATHS[case["path"]](case, int(seed))
    torch.cuda.synchronize()
    return st


def run(state):
    return state.run()


def tolerance(case):
    """Integer arithmetic throughout: every implementation has the same outputs."""
    return "exact"


# ---------------------------------------------------------------------------
# What one pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Inputs read once, outputs written once (bytes), and the arithmetic of the path's definition (an absolute
    difference, an addition or a multiplication counts as one)."""
    c, path = case, case["path"]
    if path == "slots":
        px = c["w"] * c["h"]
        return {"bytes": 2 * ((c["w"] + 2 * 20) * (c["h"] + 2 * 20) + 5 * px), "flops": px * (2 * 20 + 16 * 34 + 32 + 14)}
    if path == "serve":
        px = c["ticks"] * (c["s360"] * 640 * 360 + c["s720"] * 1280 * 720 + c["s1080"] * 1920 * 1080)
        return {"bytes": px * 9, "flops": px * (2 * 33 * 33 + 32 * 1.5 * 46)}
    if path == "residual":
        px = c["blocks"] * 210          # mean TU area of the shape weights
        return {"bytes": px * (2 + 4 + 4) + px * (0 if c["fused"] else 8), "flops": px * 4 * 16}
    px = c["width"] * c["height"]
    if path == "refine":
        k = 1.5 if c["chroma"] else 1.0
        return {"bytes": px * (6 * k + 3) + px / 108 * (4 * c["ncand"] + 16), "flops": px * k * c["ncand"] * 46}
    if path == "search":
        return {"bytes": px * 4, "flops": px * 2 * (2 * c["range"] + 1) ** 2}
    if path == "blocks":
        return {"bytes": px * 7, "flops": px * (2 * (2 * c["range"] + 1) ** 2 + 2 * 34 + 46)}
    if path == "lookahead":
        return {"bytes": px * 4, "flops": px / 4 * (8 + 2 * (2 * c["range"] + 1) ** 2)}
    if path == "mctf":
        return {"bytes": px * 4, "flops": px * (3 * (289 / 16 + 131 / 4 + 131 + 11) + 98 * 34)}
    if path == "pipeline":
        return {"bytes": px * 12, "flops": px * (2 * 2 * (2 * c["range"] + 1) ** 2 + 2 * 16 * 34 + 17 * 1.5 * 46)}
    return {"bytes": px * 6, "flops": px * (25 * 2 + 14 + 16)}


# ---------------------------------------------------------------------------
# The same from plain torch / numpy
# ---------------------------------------------------------------------------
def _eg(v):
    k = np.where(v > 0, 2 * v - 1, -2 * v).astype(np.int64) + 1
    return 2 * np.floor(np.log2(k)).astype(np.int64) + 1


def _exact_search(c, seed):
    st = Search(c, seed)
    torch.cuda.synchronize()
    w, h, bw, bh, r = c["width"], c["height"], c["bw"], c["bh"], c["range"]
    nbx, nby = w // bw, h // bh
    W, H = nbx * bw, nby * bh
    cur = st.cur.t[0][PAD:PAD + H, PAD:PAD + W].to(torch.int32)
    ref = st.ref.t[0].to(torch.int32)
    x = np.arange(nbx) * bw
    y = np.arange(nby) * bh
    best = torch.full((nby, nbx), 1 << 62, dtype=torch.int64, device=DEV)
    bsad = torch.zeros((nby, nbx), dtype=torch.int64, device=DEV)
    bmv = torch.zeros((nby, nbx, 2), dtype=torch.int64, device=DEV)
    for dy in range(-r, r + 1):
        oky = torch.from_numpy((dy >= -y - 72) & (dy <= h + 72 - bh - y)).to(DEV)[:, None]
        for dx in range(-r, r + 1):
            okx = torch.from_numpy((dx >= -x - 72) & (dx <= w + 72 - bw - x)).to(DEV)[None]
            d = (cur - ref[PAD + dy:PAD + dy + H, PAD + dx:PAD + dx + W]).abs()
            sad = d.view(nby, bh, nbx, bw).sum((1, 3))
            cost = (sad << 8) + int(_eg(np.array(4 * dx)) + _eg(np.array(4 * dy))) * LAMBDA_INT
            m = (cost < best) & oky & okx
            best = torch.where(m, cost, best)
            bsad = torch.where(m, sad, bsad)
            bmv = torch.where(m[..., None], torch.tensor([4 * dx, 4 * dy], device=DEV), bmv)
    return [bmv.reshape(-1), best.reshape(-1), bsad.reshape(-1)]


def _hada(n):
    m = np.array([[1.0]])
    while len(m) < n:
        m = np.block([[m, m], [m, -m]])
    return m


def _satd(d):
    """SATD of a difference block: 8x8 Hadamard tiles, 4x4 where a side is not a multiple of 8."""
    n = 8 if d.shape[0] % 8 == 0 and d.shape[1] % 8 == 0 else 4
    t = d.reshape(d.shape[0] // n, n, d.shape[1] // n, n).transpose(0, 2, 1, 3)
    s = np.abs(_hada(n) @ t @ _hada(n)).sum((2, 3)).astype(np.int64)
    return int(((s + n // 4) >> (n // 4)).sum())


def _exact_slots(c, seed):
    st = Slots(c, seed)
    w, h = c["w"], c["h"]
    fx, fy = st.frac & 15, st.frac >> 4
    a = st.refb.astype(np.int64)
    reg = a[PAD - 3:PAD + h + 4, PAD - 3:PAD + w + 4]
    t = sum(int(wl.LUMA_FILTER[fx][j]) * reg[:, j:j + w] for j in range(8))
    t = (t - (8192 << 2)) >> 2
    p = sum(int(wl.LUMA_FILTER[fy][j]) * t[j:j + h] for j in range(8))
    p = np.clip((p + 512 + (8192 << 6)) >> 10, 0, 1023)
    d = (st.curb[PAD:PAD + h, PAD:PAD + w].astype(np.int64) - p).astype(np.float64)
    return {"int": None, "sub": None, "pred": p.astype(np.float64), "satd": np.array([_satd(d)], np.float64)}


def _exact_bi(c, seed):
    st = Bi(c, seed)
    torch.cuda.synchronize()
    w, h = c["width"], c["height"]
    win = lambda p: p.t[0][PAD:PAD + h, PAD:PAD + w].cpu().numpy().astype(np.int64)  # noqa: E731
    d = (win(st.cur) - ((win(st.ref0) + win(st.ref1) + 1) >> 1)).astype(np.float64)
    out = np.zeros(len(st.b), np.float64)
    for i, (x, y, bw, bh) in enumerate(zip(*[st.b[k].tolist() for k in ("x", "y", "w", "h")])):
        t = d[y:y + bh, x:x + bw]
        out[i] = _satd(t) if c["satd"] else np.abs(t).sum()
    return [None, out]


def exact(case, seed):
    """Searches, interpolation and distortions from their definitions; the other paths end in integer transforms
    with rounding inside, or take too long this way."""
    c = case
    if c["path"] == "search" and c["width"] * c["height"] * (2 * c["range"] + 1) ** 2 < 4e9:
        return _exact_search(c, int(seed))
    if c["path"] == "slots":
        return _exact_slots(c, int(seed))
    if c["path"] == "bi" and c["width"] * c["height"] <= 1920 * 1080:
        return _exact_bi(c, int(seed))
    return None
