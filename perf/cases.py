"""Cases of the framework's main paths, from the smallest single-coil NUFFT to
the 3D kooshball: ``listed`` names them, ``draw`` gives more of the same
ranges, ``prepare`` makes what a program holds before the call, ``run`` is one
pass through the public entry points, ``work`` its unavoidable bytes and
operations, and ``exact`` the same result in 64 bits from plain torch.
"""

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "deep-mr_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "deep-mr_amd"))

import tilenufft  # noqa: E402
from tilenufft.batch import BatchedNUFFT  # noqa: E402

GOLDEN = math.pi * (math.sqrt(5.0) - 1.0) / 2.0


def listed():
    return [
        # the smallest call: one coil, one radial image, forward then adjoint (launch latency)
        _nufft("radial2d_1coil", "both", (128, 128), 1, 1, "radial", 128, 256, 2.0, 4, False),
        # one slice of a multi-coil radial scan, density-weighted adjoint (the gridding reconstruction)
        _nufft("radial2d_adj_dcf", "adj", (320, 320), 12, 1, "radial", 503, 640, 1.25, 4, True),
        # a dynamic series, one plan of many frames, the wider kernel that the Gram operator defaults to
        _nufft("dynamic2d_fwd_w6", "fwd", (192, 192), 8, 20, "radial", 34, 384, 1.25, 6, False),
        # batched ragged spirals, forward and adjoint (the benchmark's workload)
        {"name": "spiral2d_batch", "kind": "batch", "n": 256, "coils": 16, "frames": 8, "arms_lo": 24, "arms_hi": 48,
         "samples": 2048, "osf": 2.0, "width": 4},
        # 3D golden-means kooshball, 8 coils: the largest forward and adjoint
        _nufft("koosh3d_fwd", "fwd", (128, 128, 128), 8, 1, "koosh", 20000, 256, 2.0, 4, False),
        _nufft("koosh3d_adj_dcf", "adj", (128, 128, 128), 8, 1, "koosh", 20000, 256, 2.0, 4, True),
        # an odd, anisotropic volume at the default oversampling, forward and adjoint
        _nufft("aniso3d_odd", "both", (61, 101, 84), 4, 1, "koosh", 3001, 193, 1.25, 4, False),
        # subspace (low-rank) fingerprinting: one spiral arm per frame, 5 coefficients, both directions
        {"name": "lowrank2d", "kind": "lowrank", "n": 192, "coils": 8, "frames": 400, "arms": 1, "samples": 1000,
         "coeffs": 5, "osf": 1.25, "width": 4},
        # the Toeplitz normal operator of an iterative multi-coil reconstruction
        {"name": "gram2d", "kind": "gram", "n": 256, "nz": 1, "coils": 24, "views": 201, "samples": 512, "width": 4},
        # undersampled Cartesian cine: sparse FFT and its adjoint
        {"name": "cartesian2d", "kind": "sparse", "ny": 256, "nx": 256, "coils": 8, "frames": 12, "lines": 48},
        # differentiable unrolled CG-SENSE, captured, forward and backward (a training step's core)
        {"name": "cgsense_unrolled", "kind": "cg", "n": 256, "coils": 8, "views": 201, "samples": 512, "iters": 10,
         "osf": 1.25, "width": 4},
        # the functional interface, which plans on every call
        {"name": "functional2d", "kind": "functional", "n": 256, "coils": 8, "views": 128, "samples": 512,
         "osf": 1.25, "width": 4},
    ]


def _nufft(name, direction, shape, coils, frames, traj, views, samples, osf, width, dcf):
    c = {"kind": "nufft", "direction": direction, "ndim": len(shape), "nz": 1, "ny": shape[-2], "nx": shape[-1],
         "coils": coils, "frames": frames, "traj": traj, "views": views, "samples": samples, "osf": osf,
         "width": width, "dcf": dcf}
    if len(shape) == 3:
        c["nz"] = shape[0]
    if name:
        c["name"] = name
    return c


def draw(rng):
    def lograndint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["nufft2d", "nufft2d", "nufft2d", "nufft3d", "nufft3d", "batch", "lowrank", "gram", "sparse",
                       "functional", "cg"])
    if kind == "nufft2d":
        n = lograndint(64, 384)
        ny = n if rng.random() < 0.7 else lograndint(64, 384)
        frames = 1 if rng.random() < 0.5 else lograndint(2, 24)
        coils = lograndint(1, 32)
        views = lograndint(16, 400) if frames == 1 else lograndint(8, 64)
        return _nufft("", rng.choice(["fwd", "adj", "both"]), (ny, n), coils, frames,
                      rng.choice(["radial", "spiral"]), views, lograndint(128, 1024),
                      rng.choice([1.25, 1.25, 1.5, 2.0]), rng.choice([3, 4, 4, 4, 5, 6]), rng.random() < 0.5)
    if kind == "nufft3d":
        n = lograndint(24, 128)
        shape = (n, n, n) if rng.random() < 0.6 else (lograndint(24, 128), lograndint(24, 128), n)
        return _nufft("", rng.choice(["fwd", "adj", "both"]), shape, lograndint(1, 8), 1, "koosh",
                      lograndint(400, 10000), lograndint(64, 256), rng.choice([1.25, 1.5, 2.0]),
                      rng.choice([3, 4, 4, 4]), rng.random() < 0.5)
    if kind == "batch":
        lo = lograndint(4, 32)
        return {"kind": "batch", "n": rng.choice([64, 96, 128, 160, 192, 256, 320]), "coils": lograndint(1, 16),
                "frames": lograndint(2, 8), "arms_lo": lo, "arms_hi": 2 * lo, "samples": lograndint(256, 2048),
                "osf": rng.choice([1.25, 1.5, 2.0]), "width": 4}
    if kind == "lowrank":
        return {"kind": "lowrank", "n": lograndint(64, 256), "coils": lograndint(1, 12), "frames": lograndint(24, 400),
                "arms": rng.choice([1, 1, 2]), "samples": lograndint(256, 1000), "coeffs": rng.choice([3, 4, 5, 6]),
                "osf": rng.choice([1.25, 2.0]), "width": 4}
    if kind == "gram":
        threed = rng.random() < 0.3
        return {"kind": "gram", "n": lograndint(32, 80) if threed else lograndint(64, 320),
                "nz": lograndint(16, 64) if threed else 1, "coils": lograndint(1, 8) if threed else lograndint(1, 32),
                "views": lograndint(50, 400), "samples": lograndint(128, 512), "width": rng.choice([4, 6])}
    if kind == "sparse":
        ny = lograndint(64, 320)
        return {"kind": "sparse", "ny": ny, "nx": lograndint(64, 320), "coils": lograndint(1, 16),
                "frames": lograndint(1, 16), "lines": max(4, ny // rng.choice([2, 3, 4, 6]))}
    if kind == "functional":
        return {"kind": "functional", "n": lograndint(48, 320), "coils": lograndint(1, 16),
                "views": lograndint(24, 300), "samples": lograndint(128, 640), "osf": 1.25, "width": 4}
    return {"kind": "cg", "n": lograndint(96, 288), "coils": lograndint(2, 12), "views": lograndint(64, 256),
            "samples": lograndint(192, 512), "iters": rng.choice([3, 5, 8]), "osf": 1.25, "width": 4}


# ---- inputs -----------------------------------------------------------------


def _radius(samples, n):
    return (np.arange(samples) - samples // 2) * (n / samples)


def _radial(views, samples, ny, nx, offset):
    a = offset + np.arange(views) * GOLDEN
    return np.stack([np.outer(np.cos(a), _radius(samples, nx)), np.outer(np.sin(a), _radius(samples, ny))],
                    -1).astype(np.float32)


def _spiral(arms, samples, ny, nx, offset):
    tau = np.arange(samples) / samples
    turns = max(ny, nx) / float(arms)
    ph = 2 * np.pi * turns * tau + offset + 2 * np.pi * np.arange(arms)[:, None] / arms
    r = tau**2
    return np.stack([(nx / 2 - 0.5) * r * np.cos(ph), (ny / 2 - 0.5) * r * np.sin(ph)], -1).astype(np.float32)


def _koosh(spokes, samples, shape, offset):
    s = np.arange(spokes) + offset
    z = np.mod(s * 0.4656, 1.0) * 2.0 - 1.0
    phi = 2.0 * np.pi * np.mod(s * 0.6823, 1.0)
    st = np.sqrt(np.clip(1.0 - z**2, 0.0, None))
    r = _radius(samples, 1.0)[None, :]
    nz, ny, nx = shape
    return np.stack([nx * (st * np.cos(phi))[:, None] * r, ny * (st * np.sin(phi))[:, None] * r,
                     nz * z[:, None] * r], -1).astype(np.float32)


def _coords(case, seed):
    """(frames, views, samples, ndim) float32, or without the frame axis for
    one frame; the seed turns the whole trajectory."""
    off = 0.1 + 2.0 * math.pi * ((seed * 0.61803398875) % 1.0)
    k = case["kind"]
    if k == "nufft":
        shape = _shape(case)
        frames = []
        for f in range(case["frames"]):
            o = off + f * GOLDEN * (1.0 if case["traj"] != "radial" else case["views"])
            if case["traj"] == "radial":
                frames.append(_radial(case["views"], case["samples"], *shape, o))
            elif case["traj"] == "spiral":
                frames.append(_spiral(case["views"], case["samples"], *shape, o))
            else:
                frames.append(_koosh(case["views"], case["samples"], shape, 1000.0 * off))
        return frames[0] if len(frames) == 1 else np.stack(frames)
    if k == "batch":
        r = np.random.default_rng(case["frames"] * 131 + case["arms_lo"])  # the scan's arm counts, not its data
        arms = r.integers(case["arms_lo"], case["arms_hi"] + 1, case["frames"])
        return [_spiral(int(a), case["samples"], case["n"], case["n"], off + f * GOLDEN) for f, a in enumerate(arms)]
    if k == "lowrank":
        return np.stack([_spiral(case["arms"] * 24, case["samples"], case["n"], case["n"], off + f * GOLDEN)
                         [:: 24][: case["arms"]] for f in range(case["frames"])])
    if k == "gram" and case["nz"] > 1:
        return _koosh(case["views"], case["samples"], _shape(case), 1000.0 * off)
    return _radial(case["views"], case["samples"], case["n"], case["n"], off)


def _shape(case):
    if case["kind"] == "nufft":
        return (case["nz"], case["ny"], case["nx"]) if case["ndim"] == 3 else (case["ny"], case["nx"])
    if case["kind"] == "gram" and case["nz"] > 1:
        return (case["nz"], case["n"], case["n"])
    if case["kind"] == "sparse":
        return (case["ny"], case["nx"])
    return (case["n"], case["n"])


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _gen(seed):
    g = torch.Generator(device=_device())
    g.manual_seed(int(seed))
    return g


def _cnormal(shape, g):
    re = torch.randn(shape, generator=g, device=_device())
    return torch.complex(re, torch.randn(shape, generator=g, device=_device()))


def _grid_axes(shape):
    return torch.meshgrid(*[torch.linspace(-1, 1, s, device=_device()) for s in shape], indexing="ij")


def _maps(coils, shape, g):
    """Smooth complex coil sensitivities with a sum of squares of one."""
    ax = _grid_axes(shape)
    c = torch.rand((coils, len(shape)), generator=g, device=_device()) * 2.4 - 1.2
    ph = torch.rand((coils, len(shape)), generator=g, device=_device()) * 4 - 2
    out = []
    for k in range(coils):
        d2 = sum((a - c[k, i]) ** 2 for i, a in enumerate(ax))
        out.append(torch.polar(torch.exp(-d2 / 0.9), sum(ph[k, i] * a for i, a in enumerate(ax))))
    m = torch.stack(out)
    return m / m.abs().square().sum(0, keepdim=True).sqrt()


def _object(lead, shape, g):
    """Smooth-edged discs with a slow phase and a little noise: (*lead, *shape)."""
    ax = _grid_axes(shape)
    n = int(np.prod(lead)) if lead else 1
    noise = 0.02 * _cnormal((n, *shape), g)
    par = torch.rand((n, 3, len(shape) + 2), generator=g, device=_device())
    img = torch.zeros((n, *shape), dtype=torch.complex64, device=_device())
    view = (n,) + (1,) * len(shape)
    for b in range(3):
        p = par[:, b]
        r2 = sum((a - (p[:, i].view(view) - 0.5)) ** 2 for i, a in enumerate(ax))
        disc = torch.sigmoid(30.0 * ((0.25 + 0.5 * p[:, -2].view(view)) - r2.sqrt()))
        img += torch.polar((0.3 + p[:, -1].view(view)) * disc, 1.5 * p[:, 0].view(view) * ax[-1].expand(n, *shape))
    return (img + noise).reshape(*lead, *shape)


def _kspace(lead, coord, shape, g):
    """k-space samples: Gaussian, falling off with the distance from the centre as measured data do."""
    c = torch.as_tensor(coord, device=_device())
    r = sum((c[..., d] * (2.0 / shape[::-1][d])) ** 2 for d in range(c.shape[-1])).sqrt()
    return _cnormal((*lead, *c.shape[:-1]), g) * (0.01 + 1.0 / (1.0 + 40.0 * r))


def _density(coord, shape):
    c = torch.as_tensor(coord)
    r = sum((c[..., d] * (2.0 / shape[::-1][d])) ** 2 for d in range(c.shape[-1])).sqrt()
    return (r ** (c.shape[-1] - 1) + 1e-3).to(torch.float32)


def _basis(case, seed):
    """Orthonormal temporal basis of decaying signals, (coeffs, frames) complex64."""
    r = np.random.default_rng(seed)
    t = np.linspace(0, 1, case["frames"])
    sig = np.exp(-t[None] * r.uniform(0.5, 12, (64, 1))) * np.exp(2j * np.pi * t[None] * r.uniform(-1, 1, (64, 1)))
    _, _, v = np.linalg.svd(sig, full_matrices=False)
    return np.ascontiguousarray(v[: case["coeffs"]].conj()).astype(np.complex64)


def _lines(case, seed):
    """Cartesian sampling indexes (frames, lines, nx, 2), x first: a full centre and random outer lines."""
    r = np.random.default_rng(seed)
    ny, nx, lines = case["ny"], case["nx"], case["lines"]
    centre = np.arange(ny // 2 - lines // 6, ny // 2 - lines // 6 + lines // 3)
    rest = np.setdiff1d(np.arange(ny), centre)
    idx = []
    for _ in range(case["frames"]):
        y = np.sort(np.concatenate([centre, r.choice(rest, lines - len(centre), replace=False)]))
        yy, xx = np.meshgrid(y, np.arange(nx), indexing="ij")
        idx.append(np.stack([xx, yy], -1))
    return np.stack(idx) if len(idx) > 1 else idx[0]


def _inputs(case, seed):
    """The tensors of a case (on the GPU) and its host-side coordinates."""
    g, kind, shape = _gen(seed), case["kind"], _shape(case)
    if kind == "nufft":
        coord = _coords(case, seed)
        frames = () if case["frames"] == 1 else (case["frames"],)
        d = {"coord": coord}
        if case["direction"] != "adj":
            obj = _object(frames, shape, g)
            maps = _maps(case["coils"], shape, g)
            d["image"] = (maps.reshape(case["coils"], *([1] * len(frames)), *shape) * obj).contiguous()
        else:
            d["kspace"] = _kspace((case["coils"],), coord, shape, g)
        if case["dcf"]:
            d["weight"] = _density(coord, shape).to(_device())
        return d
    if kind == "batch":
        return {"coord": _coords(case, seed), "maps": _maps(case["coils"], shape, g),
                "frames": _object((case["frames"],), shape, g)}
    if kind == "lowrank":
        coord = _coords(case, seed)
        maps = _maps(case["coils"], shape, g)
        coef = _object((case["coeffs"],), shape, g)
        return {"coord": coord, "image": (maps[:, None] * coef[None]).contiguous(),
                "kspace": _kspace((case["coils"],), coord, shape, g), "basis": _basis(case, seed)}
    if kind == "gram":
        coord = _coords(case, seed)
        return {"coord": coord, "image": (_maps(case["coils"], shape, g) * _object((), shape, g)).contiguous(),
                "weight": _density(coord, shape)}
    if kind == "sparse":
        lead = () if case["frames"] == 1 else (case["frames"],)
        obj = _object(lead, shape, g)
        maps = _maps(case["coils"], shape, g).reshape(case["coils"], *([1] * len(lead)), *shape)
        return {"index": _lines(case, seed), "image": (maps * obj).contiguous()}
    if kind == "functional":
        return {"coord": torch.from_numpy(_coords(case, seed)),
                "image": (_maps(case["coils"], shape, g) * _object((), shape, g)).contiguous()}
    coord = _coords(case, seed)  # cg
    return {"coord": coord, "maps": _maps(case["coils"], shape, g), "kspace": _kspace((case["coils"],), coord, shape, g),
            "target": _object((), shape, g), "weight": _density(coord, shape)}


def prepare(case, seed):
    d, kind, dev, shape = _inputs(case, seed), case["kind"], _device(), _shape(case)
    st = {"case": case}
    if kind == "nufft":
        st["plan"] = tilenufft.fft.plan_nufft(d["coord"], list(shape), case["width"], case["osf"], device=dev)
        st.update({k: d[k] for k in ("image", "kspace", "weight") if k in d})
    elif kind == "batch":
        plans = [tilenufft.fft.plan_nufft(c, case["n"], case["width"], case["osf"], device=dev) for c in d["coord"]]
        b = BatchedNUFFT(plans, case["coils"])
        for k in range(case["frames"]):
            b.image_view(k).copy_((d["maps"] * d["frames"][k])[:, None])
        st["batch"] = b
    elif kind == "lowrank":
        st["plan"] = tilenufft.fft.plan_nufft(d["coord"], case["n"], case["width"], case["osf"], device=dev)
        st["image"], st["kspace"] = d["image"], d["kspace"]
        st["basis"] = torch.from_numpy(d["basis"]).to(dev)
        st["basis_adjoint"] = st["basis"].conj().T.resolve_conj().contiguous()
    elif kind == "gram":
        st["kern"] = tilenufft.fft.plan_toeplitz_nufft(d["coord"], list(shape), dcf=d["weight"], width=case["width"],
                                                       device=dev)
        st["image"] = d["image"]
    elif kind == "sparse":
        st["mask"] = tilenufft.fft.prepare_sampling(d["index"], list(shape), device=dev)
        st["image"] = d["image"]
    elif kind == "functional":
        st["coord"], st["image"] = d["coord"], d["image"]
    else:
        m = tilenufft.recon.UnrolledCGSENSE(torch.from_numpy(d["coord"]), shape, d["maps"], niter=case["iters"],
                                            dcf=d["weight"].to(dev), device=dev, width=case["width"],
                                            oversamp=case["osf"])
        st["model"] = tilenufft.recon.capture_unrolled(m, d["kspace"].clone().requires_grad_(True))
        st["kspace"], st["target"] = d["kspace"], d["target"]
    return st


def run(st):
    case, kind, fft = st["case"], st["case"]["kind"], tilenufft.fft
    if kind == "nufft":
        w = st.get("weight")
        if case["direction"] == "fwd":
            return fft.apply_nufft(st["image"], st["plan"], weight=w)
        if case["direction"] == "adj":
            return fft.apply_nufft_adj(st["kspace"], st["plan"], weight=w)
        y = fft.apply_nufft(st["image"], st["plan"])
        return y, fft.apply_nufft_adj(y, st["plan"], weight=w)
    if kind == "batch":
        b = st["batch"]
        return b.forward(), b.adjoint()
    if kind == "lowrank":
        return (fft.apply_nufft(st["image"], st["plan"], st["basis_adjoint"]),
                fft.apply_nufft_adj(st["kspace"], st["plan"], st["basis"]))
    if kind == "gram":
        return fft.apply_nufft_selfadj(st["image"], st["kern"])
    if kind == "sparse":
        y = fft.apply_sparse_fft(st["image"], st["mask"])
        return y, fft.apply_sparse_ifft(y, st["mask"])
    if kind == "functional":
        dev = st["image"].device
        y = fft.nufft(st["image"], st["coord"], device=dev, width=case["width"], oversamp=case["osf"])
        return y, fft.nufft_adj(y, st["coord"], list(st["image"].shape[-2:]), device=dev, width=case["width"],
                                oversamp=case["osf"])
    y = st["kspace"].detach().requires_grad_(True)
    x = st["model"](y)
    (x - st["target"]).abs().square().mean().backward()
    return x.detach(), y.grad


def work(case):
    """Bytes: every input and output once (images, samples, coordinates,
    weights, maps). Operations: 5 G log2 G for a transform of G cells and 4
    per kernel tap and sample (a complex value times a real weight, added)."""
    kind, shape = case["kind"], _shape(case)
    ndim, nvox = len(shape), int(np.prod(shape))

    def fft(g):
        return 5.0 * g * math.log2(g)

    def nufft(nimg, ncoord, nsamp, osf, w):
        g = int(np.prod([math.ceil(osf * s) for s in shape]))
        return 8 * nimg * nvox + 8 * nsamp + 4 * ndim * ncoord, nimg * fft(g) + 4 * nsamp * w**ndim

    if kind in ("nufft", "functional", "batch"):
        f = case.get("frames", 1)
        if kind == "batch":
            m = sum(c.shape[0] * c.shape[1] for c in _coords(case, 0))
        else:
            m = f * case["views"] * case["samples"]
        b, o = nufft(case["coils"] * f, m, case["coils"] * m, case["osf"], case["width"])
        passes = 1 if case.get("direction", "both") in ("fwd", "adj") else 2
        return {"bytes": passes * b + (4 * m if case.get("dcf") else 0), "flops": passes * o}
    if kind == "lowrank":
        m = case["frames"] * case["arms"] * case["samples"]
        b, o = nufft(case["coils"] * case["coeffs"], m, case["coils"] * m, case["osf"], case["width"])
        per = 4 * case["width"] ** 2 * (case["coeffs"] - 1) * case["coils"] * m + 8 * case["coeffs"] * case["coils"] * m
        return {"bytes": 2 * (b + 8 * case["coeffs"] * case["frames"]), "flops": 2 * (o + per)}
    if kind == "gram":
        g = int(np.prod([2 * s for s in shape]))
        return {"bytes": 16 * case["coils"] * nvox + 8 * g, "flops": case["coils"] * (2 * fft(g) + 6 * g)}
    if kind == "sparse":
        m = case["frames"] * case["lines"] * case["nx"]
        nimg = case["coils"] * case["frames"]
        return {"bytes": 2 * (8 * nimg * nvox + 8 * case["coils"] * m + 8 * m), "flops": 2 * nimg * fft(nvox)}
    m = case["views"] * case["samples"]  # cg: forward and backward, 2 transforms per application of E^H E
    b, o = nufft(case["coils"], m, case["coils"] * m, case["osf"], case["width"])
    return {"bytes": 2 * 8 * case["coils"] * m + 8 * case["coils"] * nvox + 24 * nvox + 8 * m,
            "flops": 2 * (2 * case["iters"] + 1) * o}


# ---- the same in 64 bits -------------------------------------------------------


class _Exact:
    """Kaiser-Bessel NUFFT of one frame in float64: apodize, pad, centred FFT
    and W taps per axis, with the grid positions rounded to float32 as the
    plan's coordinates are."""

    def __init__(self, coord, shape, width, osf):
        dev = _device()
        self.shape, self.ndim, self.w = tuple(shape), len(shape), width
        osf32 = np.float32(osf)
        self.g = tuple(int(np.ceil(osf32 * np.float32(s))) for s in shape)
        inner = np.float32((np.float32(width) / osf32 * (osf32 - np.float32(0.5))) ** 2 - np.float32(0.8))
        self.beta = float(np.float32(np.float32(math.pi) * np.sqrt(inner)))
        c = np.array(coord, dtype=np.float32).reshape(-1, self.ndim)
        self.m = c.shape[0]
        i0 = torch.special.i0
        first = math.ceil(-width / 2)
        node = torch.tensor([(first + k) / (width / 2) for k in range(width)], dtype=torch.float64)
        self.scale = float(i0(self.beta * (1 - node**2).clamp(min=0).sqrt()).sum()) ** self.ndim
        self.idx, self.wt, self.apod = [], [], []
        for d in range(self.ndim):  # x first
            n, gd = self.shape[self.ndim - 1 - d], self.g[self.ndim - 1 - d]
            x = (c[:, d] * np.float32(np.float32(gd) / np.float32(n))).astype(np.float32)
            x = torch.from_numpy((x + np.float32(gd // 2)).astype(np.float32)).to(dev).double()
            x0 = torch.ceil(x - width / 2)
            k = torch.arange(width, device=dev, dtype=torch.float64)
            u = (x0[:, None] + k - x[:, None]) / (width / 2)
            wt = torch.where(u.abs() <= 1, i0(self.beta * (1 - u * u).clamp(min=0).sqrt()), 0.0)
            self.wt.append(wt)
            self.idx.append(torch.remainder((x0[:, None] + k).long(), gd))
            i = torch.arange(n, device=dev, dtype=torch.float64) - n // 2
            s = (self.beta**2 - (math.pi * width * i / gd) ** 2).sqrt()
            a = s / torch.sinh(s)
            self.apod.append(a / a[n // 2])

    def _taps(self):
        for t in range(self.w**self.ndim):
            cell, wt = 0, 1.0
            for d in reversed(range(self.ndim)):
                k = (t // self.w**d) % self.w
                cell = cell * self.g[self.ndim - 1 - d] + self.idx[d][:, k]
                wt = wt * self.wt[d][:, k]
            yield cell, wt / self.scale

    def _crop(self):
        return tuple(slice(g // 2 - n // 2, g // 2 - n // 2 + n) for g, n in zip(self.g, self.shape))

    def _apodize(self, x):
        for d, a in enumerate(self.apod):
            x = x * a.view((-1,) + (1,) * d)
        return x

    def forward(self, img):
        """(B, *shape) -> (B, M) complex128."""
        ax = tuple(range(1, self.ndim + 1))
        big = torch.zeros((img.shape[0], *self.g), dtype=torch.complex128, device=img.device)
        big[(slice(None),) + self._crop()] = self._apodize(img.to(torch.complex128))
        k = torch.fft.fftshift(torch.fft.fftn(torch.fft.ifftshift(big, dim=ax), dim=ax), dim=ax)
        return self.gather(k)

    def gather(self, k):
        k = torch.view_as_real(k.reshape(k.shape[0], -1).T.contiguous()).reshape(-1, 2 * k.shape[0])
        out = torch.zeros((self.m, k.shape[1]), dtype=torch.float64, device=k.device)
        for cell, wt in self._taps():
            out += wt[:, None] * k[cell]
        return torch.view_as_complex(out.view(self.m, -1, 2)).T

    def adjoint(self, y):
        """(B, M) -> (B, *shape) complex128, with the 1 / G of the inverse FFT."""
        y = torch.view_as_real(y.to(torch.complex128).T.contiguous()).reshape(self.m, -1)
        grid = torch.zeros((int(np.prod(self.g)), y.shape[1]), dtype=torch.float64, device=y.device)
        for cell, wt in self._taps():
            grid.index_add_(0, cell, wt[:, None] * y)
        grid = torch.view_as_complex(grid.view(grid.shape[0], -1, 2)).T.reshape(-1, *self.g)
        ax = tuple(range(1, self.ndim + 1))
        img = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(grid, dim=ax), dim=ax), dim=ax)
        return self._apodize(img[(slice(None),) + self._crop()])


def _exact_nufft(frames, image, kspace, weight, direction):
    """Frame by frame: (coils, F, *shape) and (coils, F, M)."""
    ys, xs = [], []
    for f, e in enumerate(frames):
        wt = None if weight is None else weight[f]
        y = kspace[:, f] if direction == "adj" else e.forward(image[:, f])
        if direction == "both":
            ys.append(y)
        if direction == "fwd":
            ys.append(y if wt is None else y * wt)
        else:
            # the adjoint reads the forward's samples as they are handed over, in 32 bits
            yy = y.to(torch.complex64).to(torch.complex128)
            xs.append(e.adjoint(yy if wt is None else yy * wt))
    return (torch.stack(ys, 1) if ys else None), (torch.stack(xs, 1) if xs else None)


def exact(case, seed):
    d, kind, shape = _inputs(case, seed), case["kind"], _shape(case)
    if kind == "nufft":
        f, coils = case["frames"], case["coils"]
        coord = np.asarray(d["coord"]).reshape(f, -1, len(shape))
        fr = [_Exact(c, shape, case["width"], case["osf"]) for c in coord]
        img = d["image"].reshape(coils, f, *shape) if "image" in d else None
        ksp = d["kspace"].reshape(coils, f, -1) if "kspace" in d else None
        wt = d["weight"].double().reshape(f, -1) if "weight" in d else None
        y, x = _exact_nufft(fr, img, ksp, wt, case["direction"])
        lead = (coils,) if f == 1 else (coils, f)
        y = None if y is None else y.reshape(*lead, case["views"], case["samples"])
        x = None if x is None else x.reshape(*lead, *shape)
        return y if case["direction"] == "fwd" else x if case["direction"] == "adj" else (y, x)
    if kind == "batch":
        ks, xs = [], []
        for c, obj in zip(d["coord"], d["frames"]):
            y, x = _exact_nufft([_Exact(c, shape, case["width"], case["osf"])], (d["maps"] * obj)[:, None], None, None,
                                "both")
            ks.append(y.reshape(-1))
            xs.append(x.reshape(-1, *shape))
        return torch.cat(ks), torch.cat(xs)
    if kind == "lowrank":
        f, nc, coils = case["frames"], case["coeffs"], case["coils"]
        e = _Exact(np.asarray(d["coord"]).reshape(-1, 2), shape, case["width"], case["osf"])
        b = torch.from_numpy(d["basis"]).to(_device()).to(torch.complex128)
        k = e.forward(d["image"].reshape(coils * nc, *shape)).reshape(coils, nc, f, -1)
        y = (k * b.conj()[None, :, :, None]).sum(1).reshape(coils, f, case["arms"], case["samples"])
        ks = d["kspace"].to(torch.complex128).reshape(coils, 1, f, -1) * b[None, :, :, None]
        return y, e.adjoint(ks.reshape(coils * nc, -1)).reshape(coils, nc, *shape)
    if kind == "gram":
        ndim, dev = len(shape), _device()
        big = tuple(2 * s for s in shape)
        e = _Exact(2.0 * np.asarray(d["coord"]).reshape(-1, ndim), big, case["width"], 1.25)
        ax = tuple(range(ndim))
        kern = torch.fft.fftn(torch.fft.ifftshift(e.adjoint(d["weight"].to(dev).reshape(1, -1))[0], dim=ax), dim=ax)
        kern = kern / kern[kern != 0].abs().mean()
        img = torch.zeros((case["coils"], *big), dtype=torch.complex128, device=dev)
        sl = (slice(None),) + tuple(slice(s - s // 2, s - s // 2 + s) for s in shape)
        img[sl] = d["image"].to(torch.complex128)
        ax = tuple(range(1, ndim + 1))
        return torch.fft.ifftn(kern * torch.fft.fftn(img, dim=ax), dim=ax)[sl]
    if kind == "sparse":
        f, coils = case["frames"], case["coils"]
        idx = torch.from_numpy(np.asarray(d["index"])).to(_device()).reshape(f, -1, 2)
        img = d["image"].to(torch.complex128).reshape(coils, f, *shape)
        k = torch.fft.fftshift(torch.fft.fftn(torch.fft.ifftshift(img, dim=(2, 3)), dim=(2, 3)), dim=(2, 3))
        fr = torch.arange(f, device=_device())[:, None]
        y = k[:, fr, idx[..., 1], idx[..., 0]]
        grid = torch.zeros_like(k)
        grid[:, fr, idx[..., 1], idx[..., 0]] = y.to(torch.complex64).to(torch.complex128)
        x = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(grid, dim=(2, 3)), dim=(2, 3)), dim=(2, 3))
        lead = (coils,) if f == 1 else (coils, f)
        return y.reshape(*lead, case["lines"], case["nx"]), x.reshape(*lead, *shape)
    e = _Exact(np.asarray(d["coord"]), shape, case["width"], case["osf"])
    if kind == "functional":
        y, x = _exact_nufft([e], d["image"][:, None], None, None, "both")
        return y.reshape(case["coils"], case["views"], case["samples"]), x.reshape(case["coils"], *shape)
    return _exact_cg(case, d, e, shape)


def _exact_cg(case, d, e, shape):
    """Unrolled CG-SENSE and the gradient of its loss, by torch's autograd in 64 bits."""
    nos = float(np.prod(e.g))

    class Fwd(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return e.forward(x)

        @staticmethod
        def backward(ctx, gy):
            return e.adjoint(gy) * nos

    class Adj(torch.autograd.Function):
        @staticmethod
        def forward(ctx, y):
            return e.adjoint(y)

        @staticmethod
        def backward(ctx, gx):
            return e.forward(gx) / nos

    maps = d["maps"].to(torch.complex128)
    # the operators hold the square root of the weight forward and the weight
    # itself in the adjoint's, which takes the root again
    w = d["weight"].to(_device()).double().reshape(-1)
    wf = w.sqrt()

    def eh(y):
        return (maps.conj() * Adj.apply(wf * y)).sum(0)

    y = d["kspace"].to(torch.complex128).reshape(case["coils"], -1).requires_grad_(True)
    b = eh(wf * y)
    x, r, p = torch.zeros_like(b), b, b
    rs = (r.conj() * r).sum().real
    for _ in range(case["iters"]):
        q = eh(wf * Fwd.apply(maps * p))
        alpha = rs / (p.conj() * q).sum()
        x, r = x + alpha * p, r - alpha * q
        new = (r.conj() * r).sum().real
        p, rs = r + (new / rs) * p, new
    (x - d["target"].to(torch.complex128)).abs().square().mean().backward()
    return x.detach(), y.grad.reshape(case["coils"], case["views"], case["samples"])
