"""The work that users of libmc3 have it do, as measurable cases.

Whole calls go through Context.align_movie / align_movies / load_frames /
load_eer; single stages through the C entry points of include/mc_abi.h with
buffers that the caller keeps, as a program that binds the C ABI calls them.

Torch is imported before the library is loaded, so both run on the HIP runtime
that torch brings; library buffers are handed out as torch tensors over the
same memory.

Ranges:
  movies, measured without patches: any frame size from 512 x 512 up, 6 to 64
    frames, FP32 / FP16 / BF16 spectra, with and without dose weighting, split
    sums and Fourier binning;
  movies, measured with patches: 5760 x 4092 and its 2x super-resolution size
    with 5 x 5 patches, one movie or several per call.  A patch shift that
    moves by 1e-5 px flips the nearest-pixel warp over whole regions, so sums
    can be compared between two builds only while every rounding of the
    alignment is the same; at other sizes the stages of patch mode are
    measured one by one, and its correction with given shifts;
  movies corrected with given shifts (-InAln): any size, with and without
    patches;
  2-D FFTs (both directions): 64 to 8192 points a side, smooth and ragged, one
    transform to a movie's frames;
  local warp, patch extraction, frame loading (8-bit, 16-bit, 4-bit, float,
    with and without references), EER rendering.
"""
import ctypes as C
import functools

import numpy as np
import torch

from motioncor3_amd import lib as L
from motioncor3_amd.synth import MovieRecipe, eer_stream_7bit

# frame sizes of cameras in use (counting and super-resolution modes, and a
# movie whose frames are stored turned by 90 degrees; 5760 rows are not a
# supported height)
FRAMES = [(3838, 3710), (4096, 4096), (5760, 4092), (3710, 3838), (7676, 7420), (8192, 8192)]
# the patch sizes of movies with a 2048-row alignment size
GRIDS = [(5, 5), (7, 5), (6, 4), (3, 3)]


def _movie(name, W, H, N, count=1, px=0, py=0, dose=0.0, ft_bin=1.0, split=False, fmt=0, replay=False):
    return {"name": name, "kind": "movie", "W": W, "H": H, "N": N, "count": count, "px": px, "py": py,
            "dose": dose, "ft_bin": ft_bin, "split": split, "fmt": fmt, "replay": replay}


def _fft(name, W, H, batch, inverse):
    return {"name": name, "kind": "fft", "W": W, "H": H, "batch": batch, "inverse": inverse}


def listed():
    return [
        # a session's movies in one call: patch alignment with dose weighting
        _movie("movies_patch", 5760, 4092, 50, count=3, px=5, py=5, dose=1.0),
        # super-resolution frames, binned back by the output
        _movie("movie_superres", 11520, 8184, 12, px=5, py=5, dose=1.2, ft_bin=2.0),
        # whole-frame alignment of a camera size with prime factors 101 and 53
        _movie("movie_ragged", 3838, 3710, 40, dose=1.0),
        # the same on a power-of-two camera, spectra stored in FP16, half sets
        _movie("movie_f16", 4096, 4096, 40, dose=1.3, split=True, fmt=1),
        # the smallest whole call: a few small frames (screening, tilt images)
        _movie("movie_small", 512, 512, 8),
        # correction with shifts from an earlier run (-InAln), patch mode
        _movie("replay_patch", 4096, 4096, 40, px=7, py=5, dose=1.2, replay=True),
        # one small transform: the smallest stage call
        _fft("fft_small", 512, 512, 1, False),
        # forward transforms of frames
        _fft("fft_frames", 5760, 4092, 10, False),
        # inverse transforms of a ragged size
        _fft("ifft_ragged", 3838, 3710, 10, True),
        # local-motion correction of real frames
        {"name": "warp", "kind": "warp", "W": 5760, "H": 4092, "N": 24, "px": 5, "py": 5, "bad": True},
        # patch windows of a movie and their transforms, 7 x 5 patches of 292 x 408
        {"name": "patches", "kind": "patches", "W": 2048, "H": 2048, "N": 40, "px": 7, "py": 5},
        # 8-bit counts in pinned host memory to gain-corrected frames
        {"name": "load_u8", "kind": "load", "W": 5760, "H": 4092, "N": 24, "mode": 0, "gain": True, "dark": False},
    ]


def _log_int(rng, lo, hi, step=1):
    return max(lo, int(round(lo * (hi / lo) ** rng.random() / step)) * step)


def _length(rng, lo, hi, step=1):
    """A side without a prime factor above 151: cameras, crops and patch grids
    give ragged sides, but not large primes."""
    while True:
        n = m = _log_int(rng, lo, hi, step)
        for f in range(2, 152):
            while m % f == 0:
                m //= f
        if m == 1 and n != 5760:
            return n


def _size(rng, lo=512, hi=6000):
    if rng.random() < 0.6:
        return rng.choice(FRAMES)
    return _length(rng, lo, hi, 2), _length(rng, lo, hi, 2)


def _frames(rng, W, H, budget, hi=64):
    """A frame count with at most `budget` pixels in all."""
    return max(6, min(_log_int(rng, 6, hi), int(budget / (W * H))))


def draw(rng):
    kind = rng.choice(["global", "global", "patch", "replay", "replay", "fft", "fft", "warp", "patches", "load", "eer"])
    dose = rng.choice([0.0, round(rng.uniform(0.5, 2.0), 2), round(rng.uniform(0.5, 2.0), 2)])
    if kind == "global":
        W, H = _size(rng)
        c = _movie("", W, H, _frames(rng, W, H, 0.8e9), dose=dose, ft_bin=rng.choice([1.0, 1.0, 1.0, 2.0, 1.5]),
                   split=rng.random() < 0.25, fmt=rng.choice([0, 0, 0, 1, 2]))
    elif kind == "patch":
        W, H = rng.choice([(5760, 4092), (5760, 4092), (11520, 8184)])
        c = _movie("", W, H, _frames(rng, W, H, 1.2e9, 50), px=5, py=5, dose=dose,
                   ft_bin=rng.choice([1.0, 2.0]), split=rng.random() < 0.25)
    elif kind == "replay":
        px, py = rng.choice([(0, 0)] + GRIDS)
        W, H = _size(rng) if not px else rng.choice(FRAMES[:4]) if rng.random() < 0.6 else _size(rng, 512, 4000)
        W, H = (W, H) if not px or W * H < 24e6 else FRAMES[0]
        c = _movie("", W, H, _frames(rng, W, H, 0.3e9 if px else 0.8e9), px=px, py=py, dose=dose,
                   ft_bin=rng.choice([1.0, 1.0, 2.0]), split=rng.random() < 0.25, replay=True)
    elif kind == "fft":
        if rng.random() < 0.4:
            W, H = rng.choice(FRAMES + [(576, 408), (292, 408), (2882, 2048), (1024, 1024)])
        else:
            W, H = _length(rng, 64, 8192, 2), _length(rng, 64, 8192)
        c = _fft("", W, H, max(1, min(_log_int(rng, 1, 200), int(0.3e9 / (W * H)))), rng.random() < 0.5)
    elif kind == "warp":
        W, H = (_size(rng) if rng.random() < 0.7 else (_log_int(rng, 500, 6000), _log_int(rng, 500, 6000)))
        px, py = rng.choice(GRIDS + [(8, 8)])
        c = {"kind": "warp", "W": W, "H": H, "N": _frames(rng, W, H, 0.8e9), "px": px, "py": py,
             "bad": rng.random() < 0.5}
    elif kind == "patches":
        W, H = rng.choice([(2882, 2048), (2048, 2048), (2118, 2048), (2048, 2882)])
        px, py = rng.choice(GRIDS)
        c = {"kind": "patches", "W": W, "H": H, "N": _log_int(rng, 6, 50), "px": px, "py": py}
    elif kind == "load":
        W, H = _size(rng)
        mode = rng.choice([0, 0, 1, 6, 2, 101])
        c = {"kind": "load", "W": W, "H": H, "N": _frames(rng, W, H, 0.6e9 if mode != 2 else 0.3e9),
             "mode": mode, "gain": rng.random() < 0.7, "dark": rng.random() < 0.4}
    else:
        W = rng.choice([2048, 4096, 4096])
        c = {"kind": "eer", "W": W, "N": rng.choice([40, 80, 120]), "electrons": _log_int(rng, 20000, 80000),
             "out": rng.choice([10, 20, 40]), "sampling": rng.choice([1, 2]) if W == 4096 else 1,
             "gain": rng.random() < 0.5}
    c.pop("name", None)
    return c


# ---- what a program keeps -------------------------------------------------
@functools.lru_cache(maxsize=None)
def _ctx():
    """One context for all movies of a process, as a session keeps it."""
    torch.cuda.init()
    return L.Context(0)


class _View:
    def __init__(self, dev):
        self.dev = dev  # keeps the buffer alive
        self.__cuda_array_interface__ = {"shape": dev.shape, "typestr": dev.dtype.str, "data": (dev.ptr, False),
                                         "version": 2}


def _tensor(dev):
    """A torch tensor over a library buffer."""
    return torch.as_tensor(_View(dev), device="cuda")


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _counts(shape, seed, mean=1.0):
    """Poisson counts with a smooth image below them, as movie frames hold."""
    H, W = shape[-2:]
    y = torch.linspace(0, 9.0, H, device="cuda")[:, None]
    x = torch.linspace(0, 11.0, W, device="cuda")[None, :]
    rate = mean * (1.0 + 0.2 * torch.sin(x + 0.7 * y) * torch.cos(y))
    out = torch.empty(shape, device="cuda")
    g = _gen(seed)
    for f in out.view(-1, H, W):
        f.copy_(torch.poisson(rate, generator=g))
    return out


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _check(ctx, rc):
    if rc != L.MC_OK:
        raise RuntimeError(ctx.lib.mc_last_error(ctx.ptr).decode())


def _params(c):
    return L.default_params(patch=(c["px"], c["py"]), pix_size=0.83, fm_dose=c["dose"], ft_bin=c["ft_bin"],
                            split_sum=int(c["split"]), frame_fmt=c["fmt"], spectra_fmt=c["fmt"])


def _recipe(c, seed):
    W, H = c["W"], c["H"]
    return MovieRecipe(W, H, c["N"], min(20000, max(200, W * H // 1200)), seed=seed, dose=1.0,
                       local_max=3.0 if c["px"] else 0.0)


def _centres(c):
    W, H, px, py = c["W"], c["H"], c["px"], c["py"]
    return np.array([[(i % px + 0.5) * W / px, (i // px + 0.5) * H / py] for i in range(px * py)], np.float32)


def _local_shifts(c, seed):
    """Smooth local motion per patch, frame and axis, [N, P, 2], and bad flags."""
    rng = np.random.default_rng(seed + 17)
    cen = _centres(c) / np.array([c["W"], c["H"]]) - 0.5
    t = np.linspace(-0.5, 0.5, c["N"])
    k = rng.normal(0.0, 2.0, (6, 2))
    a = k[0] + cen[:, :1] * k[1] + cen[:, 1:] * k[2] + cen[:, :1] * cen[:, 1:] * k[3]
    sh = t[:, None, None] * a + (t ** 2)[:, None, None] * (k[4] + cen[:, :1] * k[5])
    sh = sh + rng.normal(0.0, 0.05, sh.shape)
    bad = (rng.random(sh.shape[:2]) < 0.01).astype(np.uint8)
    return sh.astype(np.float32), bad


def _windows(c, seed):
    g = L.geometry(c["W"], c["H"], c["px"], c["py"])
    pw, ph = g["patch"]
    rng = np.random.default_rng(seed + 5)
    st = np.stack([rng.integers(0, c["W"] - pw + 1, c["px"] * c["py"]),
                   rng.integers(0, c["H"] - ph + 1, c["px"] * c["py"])], 1).astype(np.int32)
    return st, pw, ph


def _values(c, seed):
    """The counts of a raw movie, in the range of its mode."""
    v = _counts((c["N"], c["H"], c["W"]), seed, 1.5)
    return v.clamp_(max=15.0) if c["mode"] == 101 else v


def _raw(c, seed):
    """Raw frames as a file of the MRC mode holds them, [N, H, samples or bytes a row]."""
    v, mode = _values(c, seed), c["mode"]
    if mode == 2:
        return v.cpu().numpy()
    if mode == 101:
        q = torch.nn.functional.pad(v, (0, c["W"] % 2)).to(torch.uint8)
        return (q[..., 0::2] | (q[..., 1::2] << 4)).cpu().numpy()
    return v.to(torch.uint8 if mode == 0 else torch.int16).cpu().numpy()


@functools.lru_cache(maxsize=4)
def _refs(W, H, gain, dark):
    """A camera's references: the same for all its movies."""
    rng = np.random.default_rng(W + H)
    return (rng.uniform(0.8, 1.2, (H, W)).astype(np.float32) if gain else None,
            rng.uniform(0.0, 0.2, (H, W)).astype(np.float32) if dark else None)


def _use_refs(ctx, refs):
    """Set once, as a program does for a session's camera."""
    if getattr(ctx, "refs_in_use", None) is not refs:
        ctx.set_refs(*refs)
        ctx.refs_in_use = refs


def _events(c, seed):
    """Sorted pixel indices of each EER fraction's electrons, their sub-pixel
    nibbles, and the fractions of each rendered frame."""
    rng = np.random.default_rng(seed)
    n = c["W"] * c["W"]
    ev = []
    for _ in range(c["N"]):
        q = np.unique(rng.integers(0, n, c["electrons"]))
        ev.append((q, rng.integers(0, 16, len(q))))
    size = c["N"] // c["out"]
    return ev, (np.arange(c["out"]) * size).astype(np.int32), np.full(c["out"], size, np.int32)


# ---- the cases ------------------------------------------------------------
def prepare(case, seed):
    c, ctx = case, _ctx()
    s = {"case": c, "ctx": ctx}
    k = c["kind"]
    if k == "movie":
        p = s["params"] = _params(c)
        ns, ow, oh = ctx.output_geometry(p, c["W"], c["H"], c["N"])
        s["frames"], s["sums"], s["views"] = [], [], []
        for m in range(c["count"]):
            f = ctx.empty((c["N"], c["H"], c["W"]), np.float32)
            ctx.synth_render(f, _recipe(c, 1000 * seed + m))
            s["frames"].append(f)
            s["sums"].append([ctx.empty((oh, ow), np.float32) for _ in range(ns)])
            s["views"].append([_tensor(x) for x in s["sums"][-1]])
        if c["replay"]:
            d = _recipe(c, 1000 * seed).displacement
            kw = {"replay_global": np.round(-d, 2).astype(np.float32)}
            if c["px"]:
                sh, bad = _local_shifts(c, seed)
                kw.update(replay_patch=sh, replay_centers=_centres(c), replay_bad=bad)
            s["replay"] = kw
        return s
    if k == "fft":
        W, H, B = c["W"], c["H"], c["batch"]
        x = _counts((B, H, W), seed)
        spec = torch.empty((B, W // 2 + 1, H), dtype=torch.complex64, device="cuda")
        if c["inverse"]:
            for b in range(B):
                spec[b] = (torch.fft.rfft2(x[b]) / (W * H)).t()
            s["in"], s["out"] = spec, torch.empty_like(x)
        else:
            s["in"], s["out"] = x, spec
    elif k == "warp":
        s["in"] = _counts((c["N"], c["H"], c["W"]), seed)
        s["out"] = torch.empty_like(s["in"])
        s["cen"] = _centres(c)
        s["shifts"], bad = _local_shifts(c, seed)
        s["bad"] = bad if c["bad"] else None
    elif k == "patches":
        st, pw, ph = _windows(c, seed)
        s["in"] = _counts((c["N"], c["H"], c["W"]), seed)
        s["starts"], s["size"] = st, (pw, ph)
        s["out"] = torch.empty((len(st) * c["N"], pw // 2 + 1, ph), dtype=torch.complex64, device="cuda")
    elif k == "load":
        raw = _raw(c, seed)
        s["raw"] = ctx.host_array(raw.shape, raw.dtype)
        s["raw"].a[...] = raw
        _use_refs(ctx, _refs(c["W"], c["H"], c["gain"], c["dark"]))
        s["out"] = ctx.empty((c["N"], c["H"], c["W"]), np.float32)
        s["view"] = _tensor(s["out"])
    else:
        ev, st, sz = _events(c, seed)
        parts = [eer_stream_7bit(q, sub, c["W"] * c["W"]) for q, sub in ev]
        s["offsets"] = np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.int64)
        s["data"] = ctx.host_array((int(s["offsets"][-1]),), np.uint8)
        s["data"].a[...] = np.concatenate(parts)
        s["groups"] = (st, sz)
        n = c["W"] * (2 if c["sampling"] == 2 else 1)
        _use_refs(ctx, _refs(n, n, c["gain"], False))
        s["out"] = ctx.empty((c["out"], n, n), np.float32)
        s["view"] = _tensor(s["out"])
    torch.cuda.synchronize()
    return s


def run(state):
    s = state
    c, ctx = s["case"], s["ctx"]
    k = c["kind"]
    if k == "movie":
        p = s["params"]
        if c["replay"]:
            ctx.align_movie(s["frames"][0], p, sums=s["sums"][0], **s["replay"])
            return {"sums": s["views"][0]}
        if c["count"] > 1:
            res = ctx.align_movies(s["frames"], p, sums=s["sums"])
        else:
            res = [ctx.align_movie(s["frames"][0], p, sums=s["sums"][0])]
        keys = ["global_shift", "global_iters"]
        if c["px"]:
            keys += ["patch_shift", "patch_bad", "patch_center", "patch_starts", "patch_iters"]
        return [dict({q: r[q] for q in keys}, sums=v) for r, v in zip(res, s["views"])]
    lib = ctx.lib
    if k == "fft":
        W, H, B = c["W"], c["H"], c["batch"]
        if c["inverse"]:
            _check(ctx, lib.mc_irfft2(ctx.ptr, _ptr(s["in"]), W, H, B, _ptr(s["out"]), C.c_longlong(W),
                                      C.c_longlong(W * H), 0))
        else:
            _check(ctx, lib.mc_rfft2(ctx.ptr, _ptr(s["in"]), W, H, C.c_longlong(W), C.c_longlong(W * H), B,
                                     C.c_float(1.0 / (W * H)), _ptr(s["out"])))
        return s["out"]
    if k == "warp":
        f = C.POINTER(C.c_float)
        bad = None if s["bad"] is None else s["bad"].ctypes.data_as(C.POINTER(C.c_ubyte))
        _check(ctx, lib.mc_local_warp(ctx.ptr, _ptr(s["in"]), _ptr(s["out"]), c["W"], c["H"], c["N"],
                                      len(s["cen"]), s["cen"].ctypes.data_as(f), s["shifts"].ctypes.data_as(f), bad))
        return s["out"]
    if k == "patches":
        st, (pw, ph) = s["starts"], s["size"]
        _check(ctx, lib.mc_extract_patches(ctx.ptr, _ptr(s["in"]), c["W"], c["H"], c["N"],
                                           st.ctypes.data_as(C.POINTER(C.c_int)), len(st), pw, ph, _ptr(s["out"])))
        return s["out"]
    if k == "load":
        ctx.load_frames(s["raw"], c["mode"], c["W"], c["H"], c["N"], s["out"])
    else:
        st, sz = s["groups"]
        ctx.load_eer(s["data"], s["offsets"], c["W"], c["W"], 7, c["sampling"], s["out"], int_start=st, int_size=sz)
    return s["view"]


def _num_sums(c):
    n = c["dose"] > 0
    return 1 + (2 if c["split"] else 0) + (2 if n else 0)


def work(case):
    c = case
    k = c["kind"]
    if k == "movie":
        n = c["W"] * c["H"]
        sums = _num_sums(c) * n / c["ft_bin"] ** 2
        ffts = c["N"] * (3 if c["px"] else 1)
        return {"bytes": c["count"] * 4.0 * (c["N"] * n + sums),
                "flops": c["count"] * (ffts * 2.5 * n * np.log2(n) + 10.0 * c["N"] * n)}
    if k == "fft":
        n = c["W"] * c["H"]
        return {"bytes": c["batch"] * (4.0 * n + 8.0 * (c["W"] // 2 + 1) * c["H"]),
                "flops": c["batch"] * 2.5 * n * np.log2(n)}
    if k == "warp":
        n = c["W"] * c["H"]
        return {"bytes": 8.0 * n * c["N"], "flops": 4.0 * n * c["N"]}
    if k == "patches":
        g = L.geometry(c["W"], c["H"], c["px"], c["py"])
        pw, ph = g["patch"]
        P = c["px"] * c["py"]
        return {"bytes": c["N"] * (4.0 * c["W"] * c["H"] + P * 8.0 * (pw // 2 + 1) * ph),
                "flops": c["N"] * P * 2.5 * pw * ph * np.log2(pw * ph)}
    if k == "load":
        n = c["W"] * c["H"]
        per = {0: 1.0, 1: 2.0, 6: 2.0, 2: 4.0, 101: 0.5}[c["mode"]]
        return {"bytes": n * (c["N"] * (per + 4.0) + 4.0 * (c["gain"] + c["dark"])), "flops": 2.0 * n * c["N"]}
    n = (c["W"] * (2 if c["sampling"] == 2 else 1)) ** 2
    return {"bytes": 4.0 * n * (c["out"] + c["gain"]) + 2.2 * c["N"] * c["electrons"], "flops": 1.0 * c["N"] * c["electrons"]}


# ---- the same in 64 bits --------------------------------------------------
def _warp_field(c, cen, sh, bad):
    """The source offsets of mGCorrect3D: a function of the frame's number."""
    W, H = c["W"], c["H"]
    x = torch.arange(W, device="cuda", dtype=torch.float64)
    y = torch.arange(H, device="cuda", dtype=torch.float64)
    cen = torch.from_numpy(cen.astype(np.float64)).cuda()
    w = torch.empty((len(cen), H, W), device="cuda", dtype=torch.float64)
    for p in range(len(cen)):
        r = torch.sqrt(((x - cen[p, 0]) / W)[None, :] ** 2 + ((y - cen[p, 1]) / H)[:, None] ** 2)
        w[p] = torch.where(r > 0.6, 0.0, torch.exp(-100.0 * r))

    def source(i):
        ok = torch.from_numpy(1.0 - (bad[i] if bad is not None else np.zeros(len(cen)))).cuda()
        s = torch.from_numpy(sh[i].astype(np.float64)).cuda() * ok[:, None]
        v = w.view(len(cen), -1)
        den, sx, sy = (torch.mv(v.t(), u.contiguous()).view(H, W) for u in (ok, s[:, 0], s[:, 1]))
        ok = den > 0
        xs = (x[None, :] - torch.where(ok, sx / den, sx)).trunc().long()
        ys = (y[:, None] - torch.where(ok, sy / den, sy)).trunc().long()
        out = (xs < 0) | (ys < 0) | (xs >= W) | (ys >= H)
        xs, ys = (torch.where(out, (811 * q.abs()) % n, q) for q, n in ((xs, W), (ys, H)))
        return ys, xs

    return source


def _exact_sums(c, seed):
    """A corrected movie's output sums for given shifts."""
    W, H, N = c["W"], c["H"], c["N"]
    ctx = _ctx()
    st = prepare(c, seed)
    frames, rep = _tensor(st["frames"][0]), st["replay"]
    g = rep["replay_global"].astype(np.float64)
    source = None
    if c["px"]:
        g = g - g[N // 2]
        source = _warp_field(c, rep["replay_centers"], rep["replay_patch"], rep["replay_bad"])
    kx = torch.arange(W // 2 + 1, device="cuda", dtype=torch.float64)
    ky = torch.arange(H, device="cuda", dtype=torch.float64)
    ky = torch.where(ky > H // 2, ky - H, ky)
    dose = c["dose"]
    if dose:
        fy = torch.arange(H, device="cuda", dtype=torch.float64) / H
        fy = torch.where(fy >= 0.5, fy - 1.0, fy)
        f = torch.sqrt((kx * 0.5 / (W // 2))[None, :] ** 2 + fy[:, None] ** 2) / float(np.float32(0.83))
        f[0, 0] = 1.0
        d = float(np.float32(dose))
        q = torch.exp(-0.5 * d / (0.24499 * f ** -1.6649 + 2.8141))
        q[0, 0] = 1.0
        norm = torch.sqrt(sum(q ** (2 * (i + 1)) for i in range(N)))
        norm[0, 0] = 1.0
    acc = [torch.zeros((H, W // 2 + 1), dtype=torch.complex128, device="cuda") for _ in range(_num_sums(c))]
    for i in range(N):
        F = torch.fft.rfft2(frames[i].double(), norm="forward")
        if np.hypot(*g[i]) >= 0.1:
            ph = -(kx * (g[i, 0] * 2 * np.pi / W))[None, :] - (ky * (g[i, 1] * 2 * np.pi / H))[:, None]
            F = F * torch.polar(torch.ones_like(ph), ph)
        if source is not None:
            ys, xs = source(i)
            F = torch.fft.rfft2(torch.fft.irfft2(F, s=(H, W), norm="forward")[ys, xs], norm="forward")
        acc[0] += F
        n = 1
        if dose:
            F = F * (q ** (i + 1) / norm)
            acc[1] += F
            if 3.0 <= d * (i + 1) <= 25.0:
                acc[2] += F
            n = 3
        if c["split"]:
            acc[n + (i & 1)] += F
    del frames, st
    _, ow, oh = ctx.output_geometry(_params(c), W, H, N)
    out = []
    for a in acc:
        if (ow, oh) != (W, H):
            rows = torch.arange(oh, device="cuda")
            rows = torch.where(rows > oh // 2, rows - oh + H, rows)
            a = a[rows, : ow // 2 + 1]
        out.append(torch.fft.irfft2(a, s=(oh, ow), norm="forward").clamp_(min=0.0))
    return {"sums": out}


def exact(case, seed):
    c = case
    k = c["kind"]
    if k == "movie":
        # a measured movie is an iterative fit; only its correction is a formula
        return _exact_sums(c, seed) if c["replay"] and not c["fmt"] else None
    if k == "fft":
        st = prepare(c, seed)
        W, H, x = c["W"], c["H"], st["in"]
        if c["inverse"]:
            return torch.stack([torch.fft.irfft2(v.t().to(torch.complex128), s=(H, W), norm="forward") for v in x])
        scale = float(np.float32(1.0 / (W * H)))
        return torch.stack([torch.fft.rfft2(v.double()).t() * scale for v in x])
    if k == "warp":
        st = prepare(c, seed)
        source = _warp_field(c, st["cen"], st["shifts"], st["bad"])
        out = torch.empty_like(st["in"])
        for i in range(c["N"]):
            ys, xs = source(i)
            out[i] = st["in"][i][ys, xs]
        return out
    if k == "patches":
        st = prepare(c, seed)
        pw, ph = st["size"]
        out = torch.empty(st["out"].shape, dtype=torch.complex128, device="cuda")
        for q, (x0, y0) in enumerate(st["starts"].tolist()):
            win = st["in"][:, y0:y0 + ph, x0:x0 + pw].double()
            out[q * c["N"]:(q + 1) * c["N"]] = torch.fft.rfft2(win).transpose(1, 2)
        return out
    if k == "load":
        gain, dark = _refs(c["W"], c["H"], c["gain"], c["dark"])
        v = _values(c, seed).double()
        if dark is not None:
            v = v - torch.from_numpy(dark).cuda()
        return v if gain is None else v * torch.from_numpy(gain).cuda()
    ev, st, sz = _events(c, seed)
    W, up = c["W"], 2 if c["sampling"] == 2 else 1
    n = W * up
    out = torch.zeros((c["out"], n * n), dtype=torch.float64, device="cuda")
    for o in range(c["out"]):
        for i in range(st[o], st[o] + sz[o]):
            q, sub = (torch.from_numpy(np.asarray(a, np.int64)).cuda() for a in ev[i])
            x, y = q % W, q // W
            if up == 2:
                x, y = 2 * x + ((sub >> 1) & 1), 2 * y + ((sub >> 3) & 1)
            out[o] += torch.bincount(y * n + x, minlength=n * n)
    out = out.view(c["out"], n, n)
    gain, _ = _refs(n, n, c["gain"], False)
    return out if gain is None else out * torch.from_numpy(gain).cuda()
