"""The work that users of this library have it do, as cases that can be timed.

A case is a dict of plain values; prepare() makes its inputs on the device
from a seed, run() takes them once through the library's C entry points as a
user's program calls them, exact() gives the same outputs in 64 bits from
torch alone, work() the bytes and operations that the case cannot do without.

The sizes are those of the repository's own workloads: the 64- and 256-volume
batches (axes U{128..288} and U{96..320}), the 256x256x176 and 512x512x320
head volumes, the 64^3 volume of the reference's own demonstration, and their
working grids and lattices for the stage calls.
"""
from __future__ import annotations

import ctypes as C
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-n4_amd"))

import n4amd  # noqa: E402

DEV = "cuda"
LOW = 10.0  # the library's default low_value


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # a night's worth of head scans corrected at once, the library's
        # headline workload: whole corrections, mixed sizes, one shrink
        dict(name="batch64_bf16", kind="batch", nvol=64, lo=128, hi=288, shrink=4, mixed=False, precision="bf16",
             levels=4, iters=50, mask="f32", bias=False, dims_seed=0),
        # a small study of scans of several scanners: mixed sizes and
        # shrinks, byte masks, the precise matrix-core fit
        dict(name="batch12_mixed_split", kind="batch", nvol=12, lo=96, hi=320, shrink=2, mixed=True,
             precision="split_bf16", levels=4, iters=50, mask="u8", bias=False, dims_seed=4),
        # one subject at the default precision, the drop-in call as shipped
        dict(name="head256_fp32", kind="single", x=256, y=256, z=176, shrink=4, precision="fp32", levels=4, iters=50,
             mask="f32", ncpt=4, bias=False),
        # one large 7T-like volume on a fine working grid
        dict(name="head512_bf16", kind="single", x=512, y=512, z=320, shrink=2, precision="bf16", levels=4, iters=50,
             mask="f32", ncpt=4, bias=False),
        # the reference demonstration's size, without a shrink: the smallest
        # whole correction, where latency counts
        dict(name="demo64_fp32", kind="single", x=64, y=64, z=64, shrink=1, precision="fp32", levels=3, iters=50,
             mask="f32", ncpt=4, bias=False),
        # an odd-sized volume with a confidence image and the bias field as
        # an output
        dict(name="odd_weighted_fp32", kind="single", x=181, y=217, z=163, shrink=3, precision="fp32", levels=3,
             iters=30, mask="weights", ncpt=5, bias=True),
        # the command line's call: image and mask in host memory, results
        # back in host memory
        dict(name="host256_fp32", kind="host", x=256, y=256, z=176, shrink=4, precision="fp32", levels=4, iters=50,
             mask="f32", ncpt=4, bias=False),
        # the stage calls of programs that run their own loop, on the
        # working grids of the volumes above: B-spline fit of a residual,
        dict(name="fit_64x64x44", kind="fit", x=64, y=64, z=44, c=7),
        dict(name="fit_256x256x160", kind="fit", x=256, y=256, z=160, c=11),
        # histogram sharpening,
        dict(name="sharpen_64x64x44", kind="sharpen", x=64, y=64, z=44, bins=200),
        # the field of a stored lattice at full resolution,
        dict(name="evaluate_256x256x176", kind="evaluate", x=256, y=256, z=176, c=11),
        # and the convergence measure between two fields
        dict(name="convergence_64x64x44", kind="convergence", x=64, y=64, z=44),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """One more case of the same kinds, over the same ranges."""
    kind = rng.choice(["batch", "batch", "single", "single", "single", "single", "host", "fit", "sharpen", "evaluate",
                       "convergence"])
    precision = rng.choice(["fp32", "bf16", "split_bf16"])
    mask = rng.choice(["f32", "f32", "u8", "none"])
    if kind == "batch":
        lo, s, mixed = rng.randint(96, 160), rng.choice([2, 3, 4, 4, 4]), rng.random() < 0.3
        most = 12 if mixed else {2: 6, 3: 20, 4: 48}[s]
        return dict(kind=kind, nvol=_log_uniform(rng, 2, most), lo=lo, hi=rng.randint(lo + 16, 288), shrink=s,
                    mixed=mixed, precision=precision, levels=4, iters=50, mask=rng.choice(["f32", "u8"]),
                    bias=rng.random() < 0.25, dims_seed=rng.randrange(1 << 20))
    if kind in ("single", "host"):
        s = rng.choice([1, 2, 3, 4, 4])
        lo, hi = {1: (40, 96), 2: (96, 320), 3: (120, 352), 4: (128, 400)}[s]
        if kind == "host":
            hi = min(hi, 256)
        if kind == "single" and rng.random() < 0.2:
            mask, precision = "weights", "fp32"
        return dict(kind=kind, x=_log_uniform(rng, lo, hi), y=_log_uniform(rng, lo, hi), z=_log_uniform(rng, lo, hi),
                    shrink=s, precision=precision, levels=rng.choice([2, 3, 4, 4]), iters=rng.choice([20, 50, 50]),
                    mask=mask if kind == "single" else rng.choice(["f32", "none"]), ncpt=rng.choice([4, 4, 5]),
                    bias=rng.random() < 0.25)
    lo, hi = (64, 320) if kind == "evaluate" else (36, 256)
    d = dict(kind=kind, x=_log_uniform(rng, lo, hi), y=_log_uniform(rng, lo, hi), z=_log_uniform(rng, lo, hi))
    if kind in ("fit", "evaluate"):
        d["c"] = rng.choice([4, 5, 7, 11])
    if kind == "sharpen":
        d["bins"] = rng.choice([200, 200, 128, 256])
    return d


def _dims(case):
    return (case["x"], case["y"], case["z"])


def _volumes(case):
    """(dims, shrink) of every volume of a whole-correction case."""
    if case["kind"] != "batch":
        return [(_dims(case), case["shrink"])]
    r = random.Random(case["dims_seed"])
    out = []
    for _ in range(case["nvol"]):
        dims = tuple(r.randint(case["lo"], case["hi"]) for _ in range(3))
        out.append((dims, r.choice([2, 3, 4]) if case["mixed"] else case["shrink"]))
    return out


def _params(case):
    return n4amd.default_params(levels=case["levels"], max_iter=case["iters"], threshold=0.001,
                                ncpt=case.get("ncpt", 4), shrink=case["shrink"], precision=case["precision"],
                                weighted_mask=case["mask"] == "weights")


def _final_c(case):
    return (case.get("ncpt", 4) - 3) * 2 ** (case["levels"] - 1) + 3


# ---------------------------------------------------- B-splines in 64 bits --
def _weights(n, c, domain=None):
    """[n, c] banded cubic B-spline weights of positions i + 0.5 over c - 3
    spans of the domain, in FP64."""
    span = float(n if domain is None else domain) / (c - 3)
    pos = torch.arange(n, dtype=torch.float64, device=DEV) + 0.5
    b = torch.floor(pos / span)
    t = (pos - b * span) / span
    b = b.clamp(0, c - 4).long()
    w = torch.stack([(1 - t) ** 3 / 6, (3 * t ** 3 - 6 * t ** 2 + 4) / 6,
                     (-3 * t ** 3 + 3 * t ** 2 + 3 * t + 1) / 6, t ** 3 / 6], 1)
    m = torch.zeros(n, c, dtype=torch.float64, device=DEV)
    m.scatter_(1, b[:, None] + torch.arange(4, device=DEV), w)
    return m


def _modes(t, ms):
    """t contracted with ms[d] ([in, out]) along each axis d in turn."""
    for m in ms:
        t = torch.tensordot(t, m, dims=([0], [0]))  # the contracted axis goes last: three turns restore the order
    return t


def _evaluate(lat, dims, domain=None):
    return _modes(lat, [_weights(dims[d], lat.shape[d], None if domain is None else domain[d]).T.contiguous()
                        for d in range(3)])


def _fit_tables(dims, c, domain=None):
    ws = [_weights(dims[d], c[d]) for d in range(3)]
    return [w ** 3 / (w ** 2).sum(1, keepdim=True) for w in ws], [w ** 2 for w in ws]


# ----------------------------------------------------------------- inputs --
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _phantom(dims, g, frac, sigma=5.0, bias_c=5, bias_sigma=0.3):
    """Head-class phantom (image, ellipsoid radius): three nested tissue
    classes, noise, a smooth multiplicative bias; frac: the mask's share."""
    k = (frac * 6.0 / math.pi / (0.5 * 0.45 * 0.48 * 8)) ** (1 / 3)
    ax = [(torch.arange(n, device=DEV, dtype=torch.float32) + 0.5 - n / 2.0) / (k * f * n)
          for n, f in zip(dims, (0.5, 0.45, 0.48))]
    rho = (ax[0][:, None, None] ** 2 + ax[1][None, :, None] ** 2 + ax[2][None, None, :] ** 2).sqrt_()
    im = (rho <= 1.0).float().mul_(100.0).add_((rho <= 0.75).float(), alpha=100.0)
    im.add_((rho <= 0.45).float(), alpha=100.0)
    n1 = torch.randn(dims, generator=g, device=DEV).mul_(sigma)
    im = im.add_(n1).square_().add_(n1.normal_(0.0, sigma, generator=g).square_()).sqrt_()
    lat = torch.randn((bias_c,) * 3, generator=g, device=DEV, dtype=torch.float64) * bias_sigma
    im.mul_(_modes(lat.float(), [_weights(dims[d], bias_c).T.float().contiguous() for d in range(3)]).exp_())
    return im, rho


def _mask(rho, kind):
    if kind == "none":
        return None
    if kind == "u8":
        return (rho <= 1.0).to(torch.uint8)
    if kind == "weights":  # a soft edge, as tissue probabilities have
        return ((1.15 - rho) * 4.0).clamp_(0.0, 1.0)
    return (rho <= 1.0).float()


def _offsets(vols):
    """Start of every volume in one flat buffer (64-voxel aligned) and its size."""
    o, out = 0, []
    for dims, _ in vols:
        out.append(o)
        o += (math.prod(dims) + 63) // 64 * 64
    return out, o


def _image_inputs(case, seed):
    """One flat image (and mask) buffer holding every volume of the case."""
    vols = _volumes(case)
    offs, total = _offsets(vols)
    g = _gen(seed)
    r = random.Random(seed)
    im = torch.zeros(total, device=DEV)
    mask = None if case["mask"] == "none" else torch.zeros(
        total, device=DEV, dtype=torch.uint8 if case["mask"] == "u8" else torch.float32)
    for (dims, _), o in zip(vols, offs):
        n = math.prod(dims)
        v, rho = _phantom(dims, g, r.uniform(0.3, 0.55), r.uniform(3.0, 8.0), r.choice([4, 5, 6]))
        im[o:o + n] = v.reshape(-1)
        if mask is not None:
            mask[o:o + n] = _mask(rho, case["mask"]).reshape(-1)
    return vols, offs, total, im, mask


def _stage_inputs(case, seed):
    """Log intensities of a phantom, its mask and a smooth residual-like field."""
    dims = _dims(case)
    g = _gen(seed)
    im, rho = _phantom(dims, g, random.Random(seed).uniform(0.3, 0.55))
    mask = ((rho <= 1.0) & (im > LOW)).to(torch.uint8)
    return im.clamp_min(1.0).log_(), mask, g


def prepare(case, seed):
    lib = n4amd.load()
    st = dict(case=case, lib=lib)
    kind = case["kind"]
    if kind in ("batch", "single"):
        vols, offs, total, im, mask = _image_inputs(case, seed)
        c = _final_c(case)
        st.update(im=im, mask=mask, params=_params(case), out=torch.zeros(total, device=DEV),
                  log_bias=torch.zeros(total, device=DEV), lattice=torch.zeros(len(vols), c, c, c, device=DEV),
                  bias=torch.zeros(total, device=DEV) if case["bias"] else None)
        mk = n4amd.MASK_NONE if mask is None else n4amd.MASK_U8 if case["mask"] == "u8" else n4amd.MASK_F32
        arr = (n4amd.Volume * len(vols))()
        for v, (dims, s), o, k in zip(arr, vols, offs, range(len(vols))):
            v.d_im = im.data_ptr() + 4 * o
            v.d_mask = None if mask is None else mask.data_ptr() + mask.element_size() * o
            v.mask_kind = mk
            for d in range(3):
                v.dims[d] = dims[d]
            v.shrink_factor = s
            v.d_im_normalized = st["out"].data_ptr() + 4 * o
            v.d_lattice = st["lattice"][k].data_ptr()
            v.d_bias_field = None if st["bias"] is None else st["bias"].data_ptr() + 4 * o
            v.d_log_bias_field = st["log_bias"].data_ptr() + 4 * o
        st.update(volumes=arr, reports=(n4amd.Report * len(vols))())
    elif kind == "host":
        _, _, _, im, mask = _image_inputs(case, seed)
        n, c = math.prod(_dims(case)), _final_c(case)
        st.update(im=im[:n].cpu().numpy(), mask=None if mask is None else mask[:n].cpu().numpy(), params=_params(case),
                  out=np.zeros(n, np.float32), lattice=np.zeros((c, c, c), np.float32), report=n4amd.Report())
    else:
        x, mask, g = _stage_inputs(case, seed)
        st.update(x=x, mask=mask)
        if kind == "fit":
            lat = torch.randn((6, 6, 6), generator=g, device=DEV, dtype=torch.float64) * 0.05
            st["x"] = (_evaluate(lat, _dims(case)) + 0.05 * torch.randn(_dims(case), generator=g, device=DEV)).float()
            st["out"] = torch.zeros((case["c"],) * 3, device=DEV)
        elif kind == "sharpen":
            st["out"] = torch.zeros_like(x)
        elif kind == "evaluate":
            st["x"] = torch.randn((case["c"],) * 3, generator=g, device=DEV) * 0.3
            st["out"] = torch.zeros(_dims(case), device=DEV)
        elif kind == "convergence":
            lat = torch.randn((6, 6, 6), generator=g, device=DEV, dtype=torch.float64) * 0.02
            st["y"] = (x.double() + _evaluate(lat, _dims(case))).float()
            st["value"] = C.c_double()
    return st


def run(st):
    case, lib = st["case"], st["lib"]
    kind, L, h = case["kind"], lib.L, lib.h
    if kind == "batch":
        lib._check(L.n4_correct_batch(h, st["volumes"], len(st["volumes"]), C.byref(st["params"]), st["reports"], None))
    elif kind == "single":
        v = st["volumes"][0]
        lib._check(L.n4_correct(h, v.d_im, v.d_mask, v.mask_kind, v.dims[0], v.dims[1], v.dims[2],
                                C.byref(st["params"]), v.d_im_normalized, v.d_lattice, v.d_bias_field,
                                v.d_log_bias_field, C.byref(st["reports"][0]), None))
    elif kind == "host":
        lib._check(L.n4_correct_host(h, st["im"].ctypes.data, None if st["mask"] is None else st["mask"].ctypes.data,
                                     *_dims(case), C.byref(st["params"]), st["out"].ctypes.data,
                                     st["lattice"].ctypes.data, None, C.byref(st["report"])))
        its = [int(i) for i in st["report"].iterations[:case["levels"]]]
        return {"normalized": st["out"], "lattice": st["lattice"], "iterations": np.array(its)}
    if kind in ("batch", "single"):
        its = np.array([r.iterations[:case["levels"]] for r in st["reports"]], np.int64)
        out = {"normalized": st["out"], "log_bias": st["log_bias"], "lattice": st["lattice"], "iterations": its}
        if st["bias"] is not None:
            out["bias"] = st["bias"]
        return out
    dims = (C.c_uint32 * 3)(*_dims(case))
    if kind == "fit":
        nc = (C.c_uint32 * 3)(*(case["c"],) * 3)
        lib._check(L.n4_fit_bspline3d(h, st["x"].data_ptr(), st["mask"].data_ptr(), nc, dims, 1e-3,
                                      st["out"].data_ptr()))
    elif kind == "sharpen":
        lib._check(L.n4_sharpen_image(h, st["x"].data_ptr(), st["mask"].data_ptr(), st["x"].numel(), case["bins"],
                                      0.01, 0.15, st["out"].data_ptr(), None))
    elif kind == "evaluate":
        nc = (C.c_uint32 * 3)(*(case["c"],) * 3)
        lib._check(L.n4_evaluate_bspline3d(h, st["x"].data_ptr(), nc, dims, st["out"].data_ptr()))
    else:
        lib._check(L.n4_convergence_measurement(h, st["x"].data_ptr(), st["y"].data_ptr(), st["mask"].data_ptr(),
                                                st["x"].numel(), C.byref(st["value"])))
        return {"cv": st["value"].value}
    return {"out": st["out"]}


def work(case):
    """Inputs read once and outputs written once.  Operations of a whole
    correction: a nominal 30 iterations over the working grid's foreground
    (45%), about 60 a voxel (bin, remap, 8 products each of fit and field,
    exp and its two sums), besides 12 a full-resolution voxel."""
    kind = case["kind"]
    if kind in ("batch", "single", "host"):
        vols = _volumes(case)
        full = sum(math.prod(d) for d, _ in vols)
        grid = sum(math.prod((n + s - 1) // s for n in d) for d, s in vols)
        per = 4 + {"none": 0, "u8": 1}.get(case["mask"], 4) + 4 + (0 if kind == "host" else 4) + 4 * bool(case["bias"])
        return {"bytes": per * full + 4 * len(vols) * _final_c(case) ** 3, "flops": 12 * full + 0.45 * grid * 30 * 60}
    n = math.prod(_dims(case))
    return {"fit": lambda: {"bytes": 5 * n + 4 * case["c"] ** 3, "flops": 32 * n},
            "sharpen": lambda: {"bytes": 9 * n, "flops": 20 * n},
            "evaluate": lambda: {"bytes": 4 * n + 4 * case["c"] ** 3, "flops": 8 * n},
            "convergence": lambda: {"bytes": 9 * n, "flops": 10 * n}}[kind]()


# ------------------------------------------------------------------ exact --
def _e_table(x, bins, noise, fwhm):
    """(E table, bin minimum, slope) of masked FP64 values (the Wiener
    deconvolution of N4's sharpening step); None where it is undefined."""
    if not x.numel():
        return None
    mn, mx = x.min(), x.max()
    slope = (mx - mn) / (bins - 1)
    if not bool(slope > 0):
        return None
    c = (x - mn) / slope
    i = torch.floor(c)
    off = c - i
    hit = (i >= 0) & (i < bins)
    i = i.long().clamp(0, bins - 1)
    whole, part = hit & (off == 0), hit & (off != 0) & (i < bins - 1)
    w0 = torch.where(whole, torch.ones_like(off), torch.where(part, 1 - off, torch.zeros_like(off)))
    w1 = torch.where(part, off, torch.zeros_like(off))
    hist = torch.bincount(i, w0, bins) + torch.bincount((i + 1).clamp_max(bins - 1), w1, bins)
    P = 2 << max(0, (bins - 1).bit_length())
    o = (P - bins) // 2
    V = torch.zeros(P, dtype=torch.float64, device=DEV)
    V[o:o + bins] = hist
    j = torch.arange(P, device=DEV, dtype=torch.float64)
    j = torch.minimum(j, P - j)
    s = fwhm / slope
    F = 2 * math.sqrt(math.log(2) / math.pi) / s * torch.exp(-j * j * 4 * math.log(2) / (s * s))
    Ff = torch.fft.fft(F)
    gain = (Ff.conj() / (Ff.conj() * Ff + noise)).real
    U = torch.fft.ifft(torch.fft.fft(V) * gain).real.clamp_min(0)
    at = mn + (torch.arange(P, device=DEV, dtype=torch.float64) - o) * slope
    num = torch.fft.ifft(torch.fft.fft(at * U) * Ff).real
    den = torch.fft.ifft(torch.fft.fft(U) * Ff).real
    E = torch.where(den != 0, num / den, torch.zeros_like(num))[o:o + bins]
    return E, mn, slope


def _remap(x, table):
    E, mn, slope = table
    c = ((x - mn) / slope).clamp(0, E.numel())
    i = torch.floor(c).long().clamp_max(E.numel() - 1)
    return torch.where(i < E.numel() - 1, E[i] + (E[(i + 1).clamp_max(E.numel() - 1)] - E[i]) * (c - i), E[-1])


def _cv(d):
    """Coefficient of variation of exp(-d)."""
    u = torch.expm1(-d)
    mu = u.mean()
    return float(((u * u).mean() - mu * mu).clamp_min(0).sqrt() / (1 + mu))


def _refine(lat):
    """Lattice of twice the spans with the same field."""
    for _ in range(3):
        n = lat.shape[0] - 3
        m = torch.zeros(lat.shape[0], 2 * n + 3, dtype=torch.float64, device=DEV)
        for o in range(2 * n + 3):  # the child at index o - 1 in [-1, 2n + 1]
            par = (o - 1) // 2 + 1
            taps = ((par, 0.5), (par + 1, 0.5)) if (o - 1) % 2 else ((par - 1, 0.125), (par, 0.75), (par + 1, 0.125))
            for p, w in taps:
                m[min(max(p, 0), n + 2), o] += w
        lat = torch.tensordot(lat, m, dims=([0], [0]))
    return lat


def _correct(im, mask, s, case):
    """(normalised image, log bias, final lattice) of one volume in FP64."""
    dims = im.shape
    W = [(n + s - 1) // s for n in dims]
    fg = (im > LOW) & torch.isfinite(im)
    conf = None
    if mask is not None:
        m = mask.double()
        fg &= (m > 0) & torch.isfinite(m) if case["mask"] == "weights" else m != 0
        conf = m if case["mask"] == "weights" else None

    def blocks(v):
        out = torch.zeros([w * s for w in W], dtype=torch.float64, device=DEV)
        out[:dims[0], :dims[1], :dims[2]] = v
        return out.view(W[0], s, W[1], s, W[2], s).sum((1, 3, 5))

    nm, nb = blocks(fg), blocks(torch.ones_like(fg))
    fgw = (nm > 0) & (2 * nm >= nb)
    one = nm.clamp_min(1)
    imlog = blocks(torch.where(fg, im.double().clamp_min(1e-30).log(), torch.zeros((), dtype=torch.float64, device=DEV))) / one
    wgt = fgw.double() if conf is None else torch.where(fgw, blocks(conf * fg) / one, torch.zeros_like(one))
    at = fgw.reshape(-1).nonzero().reshape(-1)
    x0 = imlog.reshape(-1)[at]
    field = torch.zeros_like(x0)
    lat = None
    c0 = case.get("ncpt", 4)
    for level in range(case["levels"]):
        c = (c0 - 3) * 2 ** level + 3
        lat = torch.zeros(c, c, c, dtype=torch.float64, device=DEV) if lat is None else _refine(lat)
        p, q = _fit_tables(W, (c, c, c))
        den = _modes(wgt, q) + 1e-3
        wts = [_weights(W[d], c).T.contiguous() for d in range(3)]
        for _ in range(case["iters"]):
            x = x0 - field
            table = _e_table(x, 200, 0.01, 0.15)
            r = torch.zeros_like(imlog)
            if table is not None:
                r.view(-1)[at] = x - _remap(x, table)
            inc = _modes(r * wgt, p) / den
            lat = lat + inc
            d = _modes(inc, wts).reshape(-1)[at]
            field = field + d
            if not x.numel() or _cv(d) <= 0.001:
                break
    f = _evaluate(lat, dims, [w * s for w in W])
    return torch.where(im > LOW, im.double(), torch.zeros((), dtype=torch.float64, device=DEV)) * torch.exp(-f), f, lat


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "single", "host"):
        vols, offs, total, im, mask = _image_inputs(case, seed)
        out = torch.zeros(total, dtype=torch.float64, device=DEV)
        lb, lats = torch.zeros_like(out), []
        for (dims, s), o in zip(vols, offs):
            n = math.prod(dims)
            v, b, lat = _correct(im[o:o + n].view(dims), None if mask is None else mask[o:o + n].view(dims), s, case)
            out[o:o + n], lb[o:o + n] = v.reshape(-1), b.reshape(-1)
            lats.append(lat)
        if kind == "host":
            return {"normalized": out[:math.prod(_dims(case))], "lattice": lats[0], "iterations": None}
        r = {"normalized": out, "log_bias": lb, "lattice": torch.stack(lats), "iterations": None}
        if case["bias"]:
            r["bias"] = torch.exp(lb)
            for (dims, _), o, e in zip(vols, offs, offs[1:] + [total]):
                r["bias"][o + math.prod(dims):e] = 0.0
        return r
    st = prepare(case, seed)
    x = st["x"].double()
    if kind == "fit":
        p, q = _fit_tables(_dims(case), (case["c"],) * 3)
        m = st["mask"].double()
        return {"out": _modes(x * m, p) / (_modes(m, q) + 1e-3)}
    if kind == "sharpen":
        m = st["mask"] != 0
        v = torch.zeros_like(x)
        v[m] = _remap(x[m], _e_table(x[m], case["bins"], 0.01, 0.15))
        return {"out": v}
    if kind == "evaluate":
        return {"out": _evaluate(x, _dims(case))}
    return {"cv": _cv(st["y"].double()[st["mask"] != 0] - x[st["mask"] != 0])}
