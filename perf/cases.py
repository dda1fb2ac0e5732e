"""Performance cases: the calls users of this library make, over the sizes they make them at.

Each case is a dict of plain values.  `prepare` makes what a program holds before the call
(inputs on the GPU or, where the call takes host data, on the host; the context), `run` is one
pass through public entry points of `bimp_amd`, `work` the bytes and operations a pass cannot do
without, and `exact` the same results in FP64 from plain torch and numpy.

Kinds of case (field "kind"):
  detect     one uint8 frame -> keypoints, from a host array (the video loop) or a device frame,
             gray or, with "colour", a device BGR frame prepared by getGPUImage's steps first
  responses  one frame -> the double- and single-stopped response maps of every scale
  batch      several frames of mixed sizes as one graph launch
  diff       float images -> differentiable responses, forward only
  fit        a training step on images and Gabor parameters: forward, loss, backward, update
  describe   a BGR frame and its keypoints -> SURF and colour descriptors
  match      two descriptor sets -> two nearest neighbours of every query
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "cuda-bimp_amd"))

import bimp_amd as B  # noqa: E402

# Banks: eight wavelengths from 4 to 13.5 (four to an octave, the benchmark's) and Context's
# default makeLambdasLog(4, 64, 2), nine wavelengths down to the fourth pyramid level.
BANKS = {
    "octaves2": [4.0 * 2.0 ** (k / 4.0) for k in range(8)],
    "context": [4.0 * 2.0 ** (k / 2.0) for k in range(9)],
}
PRECISIONS = {"fp32": B.PRECISION_FP32, "bf16": B.PRECISION_BF16, "fp16": B.PRECISION_FP16}
MAX_KEYPOINTS = 65536
DESCRIPTOR = 152  # floats per descriptor row: 64 SURF, 64 unused, 24 colour


def listed():
    return [
        # a small colour picture or thumbnail: upscaled to 350 rows, converted, detected; the
        # fewest and smallest launches of the path
        dict(name="small_colour", kind="detect", width=320, height=240, bank="context",
             precision="fp32", source="device", colour=True, shapes=20),
        # one frame of a camera loop: host frame in, keypoints back on the host
        dict(name="video_vga", kind="detect", width=640, height=480, bank="octaves2",
             precision="fp32", source="host", colour=False, shapes=40),
        # the headline workload: a device-resident 1080p frame
        dict(name="frame_1080p", kind="detect", width=1920, height=1080, bank="octaves2",
             precision="fp32", source="device", colour=False, shapes=300),
        # the same frame in the matrix-core precision form
        dict(name="frame_1080p_bf16", kind="detect", width=1920, height=1080, bank="octaves2",
             precision="bf16", source="device", colour=False, shapes=300),
        # the largest frame the transforms are built for in practice
        dict(name="frame_2160p", kind="detect", width=3840, height=2160, bank="octaves2",
             precision="fp32", source="device", colour=False, shapes=300),
        # a photograph of no standard size, all response maps (Context's bank, five levels)
        dict(name="responses_odd", kind="responses", width=1237, height=701, bank="context",
             precision="fp32", shapes=120),
        # a dataset chunk: frames of several sizes in one launch
        dict(name="batch_mixed", kind="batch", frames=16, largest=1920, bank="octaves2",
             precision="fp32", shapes=40),
        # differentiable responses at inference, images of an odd size
        dict(name="diff_odd", kind="diff", width=333, height=251, images=3, bank="octaves2"),
        # a training step of the differentiation form
        dict(name="fit_512", kind="fit", width=512, height=512, images=8, bank="octaves2"),
        # descriptors of a full keypoint list (the keypoint matrix's capacity) on a 1080p frame
        dict(name="describe_1080p", kind="describe", width=1920, height=1080, keypoints=8000,
             shapes=300),
        # matching two full lists, and two short ones
        dict(name="match_8000", kind="match", queries=8000, trains=8000),
        dict(name="match_small", kind="match", queries=517, trains=433),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _frame_size(rng, lo, hi):
    """A frame of lo to hi pixels (over the logarithm), upright or wide, any side up to 3840."""
    area = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    ratio = rng.uniform(0.75, 1.9)
    w = min(3840, int(round(math.sqrt(area * ratio))))
    return w, min(2160, int(round(area / w)))


def draw(rng):
    kind = rng.choice(["detect", "detect", "detect", "responses", "batch", "diff", "fit",
                       "describe", "match"])
    bank = rng.choice(["octaves2", "context"])
    if kind in ("detect", "responses"):
        w, h = _frame_size(rng, 160 * 120, 3840 * 2160 if kind == "detect" else 1920 * 1080)
        case = dict(kind=kind, width=w, height=h, bank=bank,
                    precision=rng.choice(["fp32", "fp32", "bf16", "fp16"]),
                    shapes=rng.randint(20, 300))
        if kind == "detect":
            case["source"] = rng.choice(["host", "device"])
            case["colour"] = case["source"] == "device" and rng.random() < 0.3
        return case
    if kind == "batch":
        return dict(kind=kind, frames=_log_int(rng, 3, 24), largest=rng.choice([640, 1280, 1920]),
                    bank="octaves2", precision=rng.choice(["fp32", "bf16"]),
                    shapes=rng.randint(20, 80))
    if kind in ("diff", "fit"):
        return dict(kind=kind, width=rng.randint(130, 512), height=rng.randint(130, 512),
                    images=rng.randint(1, 8), bank="octaves2")
    if kind == "describe":
        w, h = _frame_size(rng, 160 * 120, 1920 * 1080)
        return dict(kind=kind, width=w, height=h, keypoints=_log_int(rng, 60, 8000),
                    shapes=rng.randint(20, 300))
    return dict(kind=kind, queries=_log_int(rng, 60, 8000), trains=_log_int(rng, 60, 8000))


# ---------------------------------------------------------------- inputs
def _frame(width, height, shapes, seed):
    """uint8 scene: rectangles and ellipses on a flat background, camera noise of sigma 5."""
    r = np.random.default_rng(seed)
    img = np.full((height, width), float(r.integers(0, 256)), np.float32)
    for _ in range(shapes):
        rx = max(2, int(r.uniform(0.01, 0.12) * min(width, height)))
        ry = max(2, int(r.uniform(0.01, 0.12) * min(width, height)))
        cx, cy = int(r.integers(0, width)), int(r.integers(0, height))
        x0, x1 = max(0, cx - rx), min(width, cx + rx + 1)
        y0, y1 = max(0, cy - ry), min(height, cy + ry + 1)
        level = float(r.integers(0, 256))
        if r.random() < 0.5:
            img[y0:y1, x0:x1] = level
        else:
            yy, xx = np.ogrid[y0:y1, x0:x1]
            inside = ((xx - cx) / rx) ** 2 + ((yy - cy) / ry) ** 2 <= 1.0
            img[y0:y1, x0:x1][inside] = level
    img += 5.0 * r.standard_normal((height, width), dtype=np.float32)
    return np.clip(np.rint(img), 0, 255).astype(np.uint8)


def _bgr(width, height, shapes, seed):
    """A colour scene: one layout, a tint per channel and independent noise."""
    base = _frame(width, height, shapes, seed).astype(np.float32)
    r = np.random.default_rng(seed + 7919)
    gain = r.uniform(0.4, 1.0, 3).astype(np.float32)
    noise = 3.0 * r.standard_normal((height, width, 3), dtype=np.float32)
    return np.clip(np.rint(base[:, :, None] * gain + noise), 0, 255).astype(np.uint8)


def _batch_sizes(case):
    sides = [(320, 240), (640, 480), (1280, 720), (1920, 1080)]
    sides = [s for s in sides if s[0] <= case["largest"]]
    return [sides[(5 * i + i // 3) % len(sides)] for i in range(case["frames"])]


def _images(case, seed):
    return np.stack([_frame(case["width"], case["height"], 30, 1000 * seed + i)
                     for i in range(case["images"])]).astype(np.float32) / np.float32(255.0)


def _keypoint_matrix(case, seed):
    """7 x n SURF_CUDA matrix of keypoints in list order: by scale, then row, then column."""
    r = np.random.default_rng(seed + 31)
    n = case["keypoints"]
    lam = np.asarray(BANKS["octaves2"], np.float32)
    scale = np.sort(r.choice(len(lam), n, p=np.linspace(2.0, 0.5, len(lam)) / 10.0))
    y = r.uniform(4.0, case["height"] - 5.0, n)
    x = r.uniform(4.0, case["width"] - 5.0, n)
    order = np.lexsort((x, y, scale))
    m = np.zeros((7, n), np.float32)
    m[0], m[1] = x[order], y[order]
    m[2] = np.ones(n, np.int32).view(np.float32)
    m[3] = lam[scale].astype(np.int32).view(np.float32)
    m[4], m[5], m[6] = lam[scale], -1.0, r.uniform(0.01, 0.1, n)
    return m


def _descriptors(case, seed):
    """Query and train rows as descriptors are: unit SURF part, unused columns, colour part;
    half the queries are noisy copies of train rows."""
    r = np.random.default_rng(seed + 57)
    nq, nt = case["queries"], case["trains"]

    def rows(n):
        d = np.zeros((n, DESCRIPTOR), np.float32)
        s = r.standard_normal((n, 64), dtype=np.float32)
        d[:, :64] = s / np.linalg.norm(s, axis=1, keepdims=True)
        d[:, 128:] = r.integers(0, 5, (n, 24)).astype(np.float32) / 24.0
        return d

    t, q = rows(nt), rows(nq)
    half = r.permutation(nq)[: nq // 2]
    q[half] = t[r.integers(0, nt, half.size)]
    q[half, :64] += 0.05 * r.standard_normal((half.size, 64), dtype=np.float32)
    return q, t


def _learning_rate(case):
    """A step of about 1e-6 on the parameters (the loss and its gradients are sums over pixels),
    so that each pass of a training run has new parameters and a long run stays near them."""
    return 2e-7 / (case["images"] * case["width"] * case["height"])


def _context(case):
    opt = B.default_options()
    opt.precision = PRECISIONS[case["precision"]]
    return B.CudaStuff(case["width"], case["height"], np.asarray(BANKS[case["bank"]], np.float32),
                       opt)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("detect", "responses"):
        s["cs"] = _context(case)
        w, h = case["width"], case["height"]
        if kind == "detect" and case["colour"]:
            s["bgr"] = torch.from_numpy(_bgr(w, h, case["shapes"], seed)).cuda()
            ow, oh, _ = B.min_size_shape(w, h)
            s["gray"] = torch.empty((oh, ow), dtype=torch.uint8, device="cuda")
        elif kind == "detect" and case["source"] == "host":
            s["img"] = _frame(w, h, case["shapes"], seed)
        else:
            s["img"] = torch.from_numpy(_frame(w, h, case["shapes"], seed)).cuda()
        if kind == "detect" and case["source"] == "host":
            s["out"] = np.zeros(B.KP_MAX_POINTS, B.KEYPOINT_DTYPE)
        elif kind == "detect":
            s["out"] = torch.zeros((MAX_KEYPOINTS, 7), dtype=torch.float32, device="cuda")
    elif kind == "batch":
        sizes = _batch_sizes(case)
        opt = B.default_options()
        opt.precision = PRECISIONS[case["precision"]]
        s["batch"] = B.Batch(sizes, np.asarray(BANKS[case["bank"]], np.float32), opt)
        for i, (w, h) in enumerate(sizes):
            s["batch"].upload(i, _frame(w, h, case["shapes"], 1000 * seed + i))
        s["out"] = np.zeros((len(sizes), B.KP_MAX_POINTS), B.KEYPOINT_DTYPE)
    elif kind in ("diff", "fit"):
        from bimp_amd.autograd import BimpResponses
        s["model"] = BimpResponses(case["width"], case["height"],
                                   np.asarray(BANKS[case["bank"]], np.float32))
        s["images"] = torch.from_numpy(_images(case, seed)).cuda()
        s["params"] = torch.tensor([0.56, 0.5], dtype=torch.float64)
        if kind == "fit":
            s["params"].requires_grad_(True)
            with torch.no_grad():
                other = torch.from_numpy(_images(case, seed + 500)).cuda()
                s["target"] = s["model"](other, torch.tensor([0.56, 0.5], dtype=torch.float64))
            s["opt"] = torch.optim.SGD([s["params"]], lr=_learning_rate(case))
    elif kind == "describe":
        w, h = case["width"], case["height"]
        s["bgr"] = torch.from_numpy(_bgr(w, h, case["shapes"], seed)).cuda()
        s["kp"] = torch.from_numpy(_keypoint_matrix(case, seed)).cuda()
        s["gray"] = torch.empty((h, w), dtype=torch.uint8, device="cuda")
        s["integral"] = torch.empty((h + 1, w + 1), dtype=torch.int32, device="cuda")
        n = case["keypoints"]
        s["desc"] = torch.zeros((n, DESCRIPTOR), dtype=torch.float32, device="cuda")
        s["angle"] = torch.empty(n, dtype=torch.float32, device="cuda")
    else:
        q, t = _descriptors(case, seed)
        s["q"], s["t"] = torch.from_numpy(q).cuda(), torch.from_numpy(t).cuda()
        s["idx"] = torch.empty((len(q), 2), dtype=torch.int32, device="cuda")
        s["dist"] = torch.empty((len(q), 2), dtype=torch.float32, device="cuda")
    return s


# ---------------------------------------------------------------- one pass
def _p(t):
    return C.c_void_p(t.data_ptr())


def _ok(status):
    if status < 0:
        raise RuntimeError("bimp status %d" % status)


def _fields(k):
    """Keypoint records (structured array) as one array per field."""
    return {f: k[f] for f in k.dtype.names}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "detect":
        cs, n = state["cs"], C.c_int(0)
        if case["source"] == "host":
            img, out = state["img"], state["out"]
            _ok(B.lib.bimp_detect_u8(cs.ctx, img.ctypes.data, case["width"], 0, out.ctypes.data,
                                     len(out), 0, C.byref(n), None))
            return {"keypoints": _fields(out), "count": n.value}
        if case["colour"]:
            img, w = state["gray"], state["gray"].shape[1]
            _ok(B.lib.bimp_get_gpu_image(_p(state["bgr"]), 3 * case["width"], case["width"],
                                         case["height"], 3, 1, _p(img), w, None))
        else:
            img, w = state["img"], case["width"]
        out = state["out"]
        _ok(B.lib.bimp_detect_u8(cs.ctx, _p(img), w, 1, _p(out), MAX_KEYPOINTS, 1, C.byref(n),
                                 None))
        # the records past the count stay as prepare() left them
        return {"keypoints": {"values": out[:, :5], "labels": out[:, 5:].view(torch.int32)},
                "count": n.value}
    if kind == "responses":
        cs = state["cs"]
        _ok(B.lib.bimp_filter_u8(cs.ctx, _p(state["img"]), case["width"], 1, None))
        _ok(B.lib.bimp_cells(cs.ctx, None))
        out = []
        for i, si in enumerate(cs.ks):
            maps = torch.empty((2, si.data_h, si.data_w), dtype=torch.float32, device="cuda")
            for k, which in enumerate((B.MAP_DOUBLE, B.MAP_SINGLE)):
                _ok(B.lib.bimp_get_map(cs.ctx, i, which, 0, _p(maps[k]), si.data_w, 1, None))
            out.append(maps)
        return out
    if kind == "batch":
        b, out, counts, n = state["batch"], state["out"], [], C.c_int(0)
        b.run()
        for i in range(case["frames"]):
            _ok(B.lib.bimp_batch_results(b.b, i, out[i].ctypes.data, b.cap, C.byref(n)))
            counts.append(n.value)
        return {"keypoints": _fields(out), "counts": np.array(counts, np.int32)}
    if kind == "diff":
        with torch.no_grad():
            return state["model"](state["images"], state["params"])
    if kind == "fit":
        x = state["images"].detach().requires_grad_(True)
        p = state["params"]
        state["opt"].zero_grad()
        resp = state["model"](x, p)
        ((resp - state["target"]) ** 2).sum().backward()
        grad = p.grad.clone()
        state["opt"].step()
        return {"responses": resp.detach(), "image_grad": x.grad, "param_grad": grad,
                "params": p.detach().clone()}
    if kind == "describe":
        w, h, n = case["width"], case["height"], case["keypoints"]
        _ok(B.lib.bimp_bgr_to_gray(_p(state["bgr"]), 3 * w, w, h, 1, _p(state["gray"]), w, None))
        _ok(B.lib.bimp_integral_image(_p(state["gray"]), w, w, h, _p(state["integral"]), None))
        _ok(B.lib.bimp_surf_descriptors(_p(state["integral"]), w, h, _p(state["kp"]), n, n, 0,
                                        _p(state["desc"]), DESCRIPTOR, _p(state["angle"]), None))
        _ok(B.lib.bimp_color_features(_p(state["kp"]), n, n, _p(state["bgr"]), 3 * w, w, h,
                                      _p(state["desc"][:, 128:]), DESCRIPTOR, None))
        return {"descriptors": state["desc"], "angles": state["angle"], "gray": state["gray"],
                "integral": state["integral"]}
    nq, nt = case["queries"], case["trains"]
    _ok(B.lib.bimp_match_knn2(_p(state["q"]), nq, DESCRIPTOR, _p(state["t"]), nt, DESCRIPTOR,
                              DESCRIPTOR, _p(state["idx"]), _p(state["dist"]), None))
    return {"index": state["idx"], "distance": state["dist"]}


# ---------------------------------------------------------------- geometry (CudaStuff's rules)
def _snap(n):
    m = (n + 15) // 16 * 16
    p = 16
    while p < m:
        p *= 2
    return p if p == m or p <= 1024 else (m + 511) // 512 * 512


class _Scale:
    def __init__(self, lambda2, width, height):
        step = 1.0
        while float(np.float32(np.float32(lambda2) / np.float32(step))) >= 7.5:
            step *= 2.0
        lam = np.float32(np.float32(lambda2) / np.float32(step))
        fs = np.float32(7.0) * lam
        if int(fs) % 2 == 0:
            fs = np.float32(fs + np.float32(1.0))
        self.step, self.lam, self.fs = step, float(lam), float(fs)
        self.kw, self.kx, self.off = int(fs), int(float(fs) / 2), int(lam)
        self.level = int(round(math.log2(step)))
        self.h, self.w = int(height / step), int(width / step)
        self.fh, self.fw = _snap(self.h), _snap(self.w)

    def offsets(self, o):
        def away(v):
            return int(math.copysign(math.floor(abs(v) + 0.5), v))
        th = float(np.float32(o * math.pi / 8))
        ea, eb = away(0.6 * self.lam * math.cos(th)), away(0.6 * self.lam * math.sin(th))
        return ea, eb, eb, ea, away(0.5 * eb), away(0.5 * ea)


def _scales(case):
    lam = sorted(np.asarray(BANKS[case["bank"]], np.float32).tolist())
    return [_Scale(v, case["width"], case["height"]) for v in lam]


def _frame_work(scales, pixels):
    """One frame's filter bank and stencil: image read, the five stored orientations of each
    bank read; a real forward transform, eight complex inverse ones, about 25 operations per
    pixel and orientation after them."""
    b, f = pixels, 0.0
    for s in scales:
        n = s.fh * s.fw
        b += 4 * 5 * n
        f += (0.5 + 8) * 5 * n * math.log2(n) + 8 * 25 * s.h * s.w
    return b, f


def work(case):
    kind = case["kind"]
    if kind in ("detect", "responses"):
        b, f = _frame_work(_scales(case), case["width"] * case["height"])
        if kind == "responses":
            b += sum(2 * 4 * s.h * s.w for s in _scales(case))
        elif case["colour"]:
            b += 2 * case["width"] * case["height"]
        return {"bytes": b, "flops": f}
    if kind == "batch":
        tot = [0, 0.0]
        banks = set()
        for w, h in _batch_sizes(case):
            c = dict(case, width=w, height=h)
            b, f = _frame_work(_scales(c), w * h)
            tot[0] += b if (w, h) not in banks else w * h  # a size's bank is read once
            tot[1] += f
            banks.add((w, h))
        return {"bytes": tot[0], "flops": tot[1]}
    if kind in ("diff", "fit"):
        sc = _scales(case)
        b, f = _frame_work(sc, 4 * case["width"] * case["height"])
        resp = 4 * sum(s.h * s.w for s in sc)
        n = case["images"]
        banks = 4 * 5 * sum(s.fh * s.fw for s in sc)
        byts = banks + n * (4 * case["width"] * case["height"] + resp)
        if kind == "fit":
            # the adjoint: eight forward transforms and one inverse per scale beside the
            # recomputed responses; responses, target and upstream gradient pass once more
            byts += n * (4 * case["width"] * case["height"] + 3 * resp)
            return {"bytes": byts, "flops": 3.0 * n * f}
        return {"bytes": byts, "flops": n * f}
    if kind == "describe":
        px, n = case["width"] * case["height"], case["keypoints"]
        # 113 orientation samples and 400 descriptor samples of four box sums, 72 windows
        return {"bytes": 3 * px + px + 4 * px + n * (28 + 4 * (64 + 24 + 1)),
                "flops": 2.0 * px + n * (513 * 40.0 + 72 * 113 * 3.0)}
    nq, nt = case["queries"], case["trains"]
    return {"bytes": 4 * DESCRIPTOR * (nq + nt) + 16 * nq, "flops": 3.0 * nq * nt * DESCRIPTOR}


# ---------------------------------------------------------------- FP64 results
_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_INPUT_SCALE = float(np.float32(255.0 / 65536.0))


def _pyramid_matrix(n):
    dn = (n + 1) // 2
    a = torch.zeros((dn, n), dtype=torch.float64)
    for d in range(dn):
        for i, w in zip(range(-2, 3), (1.0, 4.0, 6.0, 4.0, 1.0)):
            t = abs(2 * d + i)
            a[d, 2 * (n - 1) - t if t >= n else t] += w / 16.0
    return a.to(_DEV)


def _levels(img, top, rounded):
    lev = [img]
    for _ in range(top):
        a = lev[-1]
        b = _pyramid_matrix(a.shape[0]) @ a @ _pyramid_matrix(a.shape[1]).T
        lev.append(torch.round(b) if rounded else b)
    return lev


def _bank_spectra(s, ratio, gamma):
    """FFT of the eight quadrature kernels placed on the transform's torus."""
    c = torch.arange(s.kw, dtype=torch.float64, device=_DEV) - s.kx
    y, x = torch.meshgrid(c, c, indexing="ij")
    iy, ix = (y.long() % s.fh).reshape(-1), (x.long() % s.fw).reshape(-1)
    sig2 = 2.0 * (s.lam * ratio) ** 2
    out = []
    for o in range(8):
        th = o * math.pi / 8
        xr, yr = x * math.cos(th) + y * math.sin(th), y * math.cos(th) - x * math.sin(th)
        env = torch.exp(-(xr * xr + gamma * yr * yr) / sig2)
        f = 2.0 * math.pi * xr / s.lam
        even, odd = env * torch.cos(f), env * torch.sin(f)
        even = even - even.sum() / s.fs ** 2
        k = torch.zeros((s.fh, s.fw), dtype=torch.complex128, device=_DEV)
        k = k.index_put((iy, ix), torch.complex(even, odd).reshape(-1), accumulate=True)
        out.append(torch.fft.fft2(k))
    return torch.stack(out)


def _pad_index(n, size, k):
    i = torch.arange(size, device=_DEV)
    return torch.where(i < n, i, torch.where(i < n + k, torch.full_like(i, n - 1), 0 * i))


def _stencil(s, level, bank, gain):
    """(D, S) of one scale from its level image (FP64)."""
    pd = gain * level[: s.h, : s.w][_pad_index(s.h, s.fh, s.kx)][:, _pad_index(s.w, s.fw, s.kx)]
    cells = torch.fft.ifft2(torch.fft.fft2(pd.to(torch.complex128))[None] * bank).abs()
    flat = cells.reshape(8, -1)
    p = s.fh * s.fw
    y = torch.arange(s.h, device=_DEV)[:, None]
    x = torch.arange(s.w, device=_DEV)[None, :]
    g = (y * s.fw + x).reshape(-1)

    def at(o, d):
        return flat[o][(g + d) % p].reshape(s.h, s.w)

    def valid(a, b):
        return ((x >= 2 * abs(b)) & (x <= s.w - 2 * abs(b)) & (y >= 2 * abs(a))
                & (y <= s.h - 2 * abs(a)))

    zero = torch.zeros((s.h, s.w), dtype=torch.float64, device=_DEV)
    dd, ss, inhib = zero, zero, zero
    for o in range(8):
        ea, eb, ia, ib, ra, rb = s.offsets(o)
        centre, e = at(o, 0), -ea * s.fw + eb
        ok = valid(ea, eb)
        ss = ss + torch.where(ok, torch.relu(at(o, e) - at(o, -e)), zero)
        dd = dd + torch.where(ok, torch.relu(centre - 0.5 * at(o, 2 * e) - 0.5 * at(o, -2 * e)),
                              zero)
        r = ra * s.fw + rb
        o2 = (o + 4) % 8
        radial = torch.relu(torch.relu(centre - 16.0 * at(o2, r)) + centre - 16.0 * at(o2, -r))
        tangential = torch.relu(at(o, -ia * s.fw - ib) - centre)
        inhib = inhib + torch.where(valid(ia, ib), radial + tangential, zero)
    return dd - inhib, ss - inhib


def _resized_gray(bgr, ow, oh, factor):
    """cv::resize's fixed-point bilinear upscale and the Q14 gray conversion, in integers."""
    img = bgr.astype(np.int64)
    if factor != 1.0:
        def taps(n, out):
            f = ((np.arange(out) + 0.5) * (1.0 / factor) - 0.5).astype(np.float32)
            i = np.floor(f).astype(np.int64)
            f = f - i.astype(np.float32)
            f = np.where((i < 0) | (i >= n - 1), np.float32(0), f)
            i = np.clip(i, 0, n - 1)
            return (i, np.minimum(i + 1, n - 1), np.rint((1 - f) * np.float32(2048)).astype(np.int64),
                    np.rint(f * np.float32(2048)).astype(np.int64))
        y0, y1, v0, v1 = taps(img.shape[0], oh)
        x0, x1, u0, u1 = taps(img.shape[1], ow)
        h = img[:, x0] * u0[None, :, None] + img[:, x1] * u1[None, :, None]
        v = h[y0] * v0[:, None, None] + h[y1] * v1[:, None, None]
        img = np.clip((v + (1 << 21)) >> 22, 0, 255)
    return ((1868 * img[..., 0] + 9617 * img[..., 1] + 4899 * img[..., 2] + (1 << 13)) >> 14)


def _exact_maps(case, img):
    lev_img = torch.as_tensor(np.ascontiguousarray(img), device=_DEV).double()
    sc = _scales(case)
    lev = _levels(lev_img, max(s.level for s in sc), True)
    ratio, gamma = torch.tensor(0.56, dtype=torch.float64), torch.tensor(0.5, dtype=torch.float64)
    for s in sc:
        bank = _bank_spectra(s, ratio.to(_DEV), gamma.to(_DEV))
        yield s, _stencil(s, lev[s.level], bank, _INPUT_SCALE)


def _exact_keypoints(case, img):
    values, labels = [], []
    for s, (d, _) in _exact_maps(case, img):
        thresh = float(np.float32(0.104 * float(d.max())))
        near = torch.nn.functional.max_pool2d(d[None, None], 3, 1, 1)[0, 0]
        inner = torch.zeros_like(d, dtype=torch.bool)
        inner[s.off + 1: s.h - s.off, s.off + 1: s.w - s.off] = True
        y, x = torch.nonzero(inner & (d > thresh) & (d >= near), as_tuple=True)
        c, size = d[y, x], s.lam * s.step

        def peak(a, b):
            den = a + b - 2.0 * c
            return torch.where(den != 0, 0.5 * (a - b) / den, 0.0 * den)

        px = (x + peak(d[y, x - 1], d[y, x + 1])) * s.step
        py = (y + peak(d[y - 1, x], d[y + 1, x])) * s.step
        values.append(torch.stack([px, py, 0 * c + size, 0 * c - 1.0, c], 1))
        labels.append(torch.tensor([[int(size), 1]], dtype=torch.int32).repeat(len(c), 1))
    return torch.cat(values).cpu(), torch.cat(labels)


def _exact_fit(case, seed):
    sc = _scales(case)
    top = max(s.level for s in sc)
    gain = 255.0 * _INPUT_SCALE

    def responses(img, banks):
        lev = _levels(img, top, False)
        return torch.cat([_stencil(s, lev[s.level], b, gain)[0].reshape(-1)
                          for s, b in zip(sc, banks)])

    p = torch.tensor([0.56, 0.5], dtype=torch.float64, device=_DEV)
    imgs = torch.from_numpy(_images(case, seed)).to(_DEV).double()
    with torch.no_grad():
        banks = [_bank_spectra(s, p[0], p[1]) for s in sc]
        if case["kind"] == "diff":
            return torch.stack([responses(im, banks) for im in imgs]).cpu()
        other = torch.from_numpy(_images(case, seed + 500)).to(_DEV).double()
        target = [responses(im, banks) for im in other]
    out, gx = [], []
    gp = torch.zeros(2, dtype=torch.float64, device=_DEV)
    for im, t in zip(imgs, target):
        # one scale at a time: the graph of a whole image's bank is large
        x = im.clone().requires_grad_(True)
        parts, at = [], 0
        for s in sc:
            q = p.clone().requires_grad_(True)
            r = _stencil(s, _levels(x, s.level, False)[-1], _bank_spectra(s, q[0], q[1]), gain)[0]
            r = r.reshape(-1)
            ((r - t[at: at + r.numel()]) ** 2).sum().backward()
            gp += q.grad
            parts.append(r.detach())
            at += r.numel()
        out.append(torch.cat(parts).cpu())
        gx.append(x.grad.cpu())
    gp = gp.cpu()
    return {"responses": torch.stack(out), "image_grad": torch.stack(gx), "param_grad": gp,
            "params": p.cpu() - _learning_rate(case) * gp}


def _exact_describe(case, seed):
    bgr = _bgr(case["width"], case["height"], case["shapes"], seed)
    gray = _resized_gray(bgr, case["width"], case["height"], 1.0)
    w, h, n = case["width"], case["height"], case["keypoints"]
    ii = np.zeros((h + 1, w + 1), np.int64)
    ii[1:, 1:] = gray.cumsum(0).cumsum(1)
    m = _keypoint_matrix(case, seed)
    x, y = m[0].astype(np.float64)[:, None], m[1].astype(np.float64)[:, None]
    s = 1.2 * m[4].astype(np.float64)[:, None] / 9.0

    def away(v):
        return (np.sign(v) * np.floor(np.abs(v) + 0.5)).astype(np.int64)

    def box(c0, r0, c1, r1):
        c0, c1, r0, r1 = np.clip(c0, 0, w), np.clip(c1, 0, w), np.clip(r0, 0, h), np.clip(r1, 0, h)
        v = ii[r1, c1] - ii[r0, c1] - ii[r1, c0] + ii[r0, c0]
        return np.where((c1 > c0) & (r1 > r0), v, 0).astype(np.float64)

    def haar(px, py, k):
        return (box(px, py - k, px + k, py + k) - box(px - k, py - k, px, py + k),
                box(px - k, py, px + k, py + k) - box(px - k, py - k, px + k, py))

    i, j = np.array([(i, j) for j in range(-6, 7) for i in range(-6, 7) if i * i + j * j <= 36]).T
    # which pixel a sample falls on and which window its angle are decided in FP32, as the
    # method states them; the sums and everything after them are FP64
    s32 = np.float32(1.2) * m[4][:, None] / np.float32(9)
    px = away(m[0][:, None] + i.astype(np.float32) * s32)
    py = away(m[1][:, None] + j.astype(np.float32) * s32)
    dx, dy = haar(px, py, np.maximum(1, away(2.0 * s)))
    g = np.exp(-(i * i + j * j) / 8.0)
    turn = np.float32(2.0) * np.float32(math.pi)
    ang = np.arctan2(dy.astype(np.float32), dx.astype(np.float32))
    ang = np.where(ang < 0, ang + turn, ang)
    best, theta = np.full(n, -1.0), np.zeros(n)
    for k in range(72):
        d = ang - np.float32(k) * (turn / np.float32(72))
        inside = np.where(d < 0, d + turn, d) < np.float32(math.pi) / np.float32(3)
        sx, sy = (g * dx * inside).sum(1), (g * dy * inside).sum(1)
        longer = sx * sx + sy * sy > best
        best = np.where(longer, sx * sx + sy * sy, best)
        theta = np.where(longer, np.arctan2(sy, sx), theta)
    co, si = np.cos(theta)[:, None], np.sin(theta)[:, None]
    v, u = np.divmod(np.arange(400), 20)
    u, v = u - 9.5, v - 9.5
    px, py = away(x + co * u * s - si * v * s), away(y + si * u * s + co * v * s)
    dx, dy = haar(px, py, np.maximum(1, away(s)))
    g = np.exp(-(u * u + v * v) / (2 * 3.3 * 3.3))
    ru, rv = g * (dx * co + dy * si), g * (dy * co - dx * si)
    cells = np.stack([ru, rv, np.abs(ru), np.abs(rv)], -1).reshape(n, 4, 5, 4, 5, 4).sum((2, 4))
    cells = cells.reshape(n, 64)
    norm = np.sqrt((cells * cells).sum(1, keepdims=True))
    desc = np.zeros((n, DESCRIPTOR))
    desc[:, :64] = cells / np.where(norm > 0, norm, 1.0)
    # colour: bins 0..3 of each channel over a 2p x 2p window (bytes 1..127 only)
    cx, cy = m[0].astype(np.int64), m[1].astype(np.int64)
    half = (np.log2(m[4].astype(np.float64)) / 2.0).astype(np.int64)
    for k in range(n):
        x0, x1 = max(0, cx[k] - half[k]), min(w, cx[k] + half[k])
        y0, y1 = max(0, cy[k] - half[k]), min(h, cy[k] + half[k])
        win = bgr[y0:y1, x0:x1].reshape(-1, 3).astype(np.int64)
        for ch in range(3):
            b = win[:, ch][(win[:, ch] >= 1) & (win[:, ch] <= 127)]
            desc[k, 128 + 8 * ch: 136 + 8 * ch] = (0.5 * np.bincount(8 * b // 255, minlength=8)
                                                   / (3 * len(win)))
    return {"descriptors": desc, "angles": theta, "gray": None, "integral": None}


def _exact_match(case, seed):
    q, t = (torch.from_numpy(a).to(_DEV).double() for a in _descriptors(case, seed))
    idx, dist = [], []
    for k in range(0, len(q), 64):
        d = torch.cdist(q[k: k + 64], t, compute_mode="donot_use_mm_for_euclid_dist")
        v, i = d.topk(2, dim=1, largest=False, sorted=True)
        idx.append(i.int().cpu())
        dist.append(v.cpu())
    return {"index": torch.cat(idx), "distance": torch.cat(dist)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "detect":
        if case["precision"] != "fp32":
            return None  # the precision forms find other keypoints than FP64 does
        if case["colour"]:
            ow, oh, f = B.min_size_shape(case["width"], case["height"])
            gray = _resized_gray(_bgr(case["width"], case["height"], case["shapes"], seed), ow, oh,
                                 float(np.float32(f)))
            img = gray[: case["height"], : case["width"]].astype(np.uint8)
        else:
            img = _frame(case["width"], case["height"], case["shapes"], seed)
        values, labels = _exact_keypoints(case, img)
        count = len(values)
        cap = B.KP_MAX_POINTS if case["source"] == "host" else MAX_KEYPOINTS
        pad = (0, 0, 0, max(0, cap - count))
        values = torch.nn.functional.pad(values, pad)[:cap]
        labels = torch.nn.functional.pad(labels, pad)[:cap]
        if case["source"] == "host":
            names = ("x", "y", "size", "angle", "response")
            fields = {f: values[:, i].contiguous() for i, f in enumerate(names)}
            fields |= {"octave": labels[:, 0].contiguous(), "class_id": labels[:, 1].contiguous()}
            return {"keypoints": fields, "count": count}
        return {"keypoints": {"values": values, "labels": labels}, "count": count}
    if kind == "responses":
        img = _frame(case["width"], case["height"], case["shapes"], seed)
        return [torch.stack(m).cpu() for _, m in _exact_maps(case, img)]
    if kind == "batch":
        return None  # its frames are those of the detect cases
    if kind in ("diff", "fit"):
        return _exact_fit(case, seed)
    if kind == "describe":
        return _exact_describe(case, seed)
    return _exact_match(case, seed)
