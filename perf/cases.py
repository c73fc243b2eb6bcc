"""The workloads this library is timed on, through its public entry points.

Every case is one call (or one forward + backward pass) as a program makes it
with its inputs resident on the GPU: ``nufft1`` / ``nufft2`` / ``nufft3`` with
new points on every call, a guru ``Plan`` with new points on every pass
(``setpts`` + ``execute``), a ragged batch through a kept ``RaggedPlan``, and a
least-squares gradient through ``torch.autograd``.

``exact`` evaluates the defining sums in float64 (as matrix products over
chunks of points) wherever that takes a few seconds at most.
"""

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "jax-finufft_amd"))

from jax_finufft_amd import Plan, RaggedPlan, nufft1, nufft2, nufft3  # noqa: E402
from jax_finufft_amd.options import Opts  # noqa: E402

DEVICE = "cuda"
# most multiply-adds (points x modes x transforms) exact() evaluates
EXACT_LIMIT = 1.5e13


def _case(kind, dim, M, n=(1, 1, 1), T=1, sets=1, single=True, eps=1e-6, points="uniform",
          modeord=0, **more):
    n = tuple(n) + (1,) * (3 - len(n))
    return dict(kind=kind, dim=dim, M=int(M), n1=int(n[0]), n2=int(n[1]), n3=int(n[2]), T=int(T),
                sets=int(sets), single=bool(single), eps=float(eps), points=points,
                modeord=int(modeord), **more)


def listed():
    return [
        # The smallest call: a few thousand visibilities onto a small image, as
        # in a test or an inner loop over many small problems; launches and host
        # work are all of it.
        dict(_case("type1", 2, 4000, (48, 40)), name="type1_2d_small"),
        # A double-precision irregularly sampled series evaluated at its times,
        # odd sizes: small, a handful of launches.
        dict(_case("type2", 1, 30011, (1001,), single=False, eps=1e-9), name="type2_1d_f64_small"),
        # The double-precision 1D configuration of the benchmark: the spectrum
        # of a long irregular series (periodogram).
        dict(_case("type1", 1, 1 << 20, (1 << 16,), single=False, eps=1e-9), name="type1_1d_f64"),
        # An ordinary multi-coil / multi-channel call: four strength vectors on
        # shared, centre-dense points, odd image sizes, FFT-ordered modes, low
        # accuracy.
        dict(_case("type1", 2, 300007, (301, 255), T=4, eps=1e-4, points="gauss", modeord=1),
             name="type1_2d_multi_odd"),
        # Double precision at high accuracy (kernel width above 8).
        dict(_case("type1", 2, 1_000_000, (512, 512), single=False, eps=1e-9),
             name="type1_2d_f64"),
        # The headline benchmark: 2D type 1, 1e7 uniform points, 1024^2 modes,
        # as setpts + execute on a kept plan.
        dict(_case("plan1", 2, 10_000_000, (1024, 1024)), name="type1_2d_large"),
        # Its forward model, through nufft2.
        dict(_case("type2", 2, 10_000_000, (1024, 1024)), name="type2_2d_large"),
        # 3D MRI, koosh-ball trajectory (radially dense centre): evaluation at
        # 16.8M samples of a 256^3 volume, and gridding 2.1M samples onto 128^3.
        dict(_case("type2", 3, 8192 * 2048, (256, 256, 256), eps=1e-5, points="koosh"),
             name="type2_3d_koosh"),
        dict(_case("type1", 3, 2048 * 1024, (128, 128, 128), eps=1e-5, points="koosh"),
             name="type1_3d_koosh"),
        # 3D type 3, sources and targets both irregular, in one pair of
        # fine grids.
        dict(_case("type3", 3, 1 << 20, points="box", extent=16.0, targets=1 << 20),
             name="type3_3d"),
        # Training step on image and trajectory: loss and gradients of
        # sum |nufft2(f, x, y) - d|^2 w.r.t. f, x, y (the benchmark's gradient
        # workload).
        dict(_case("grad2", 2, 4_000_000, (512, 512)), name="grad_type2_2d"),
        # The benchmark's ragged batch: 64 problems of different point counts,
        # grids and stacked transforms in one plan.
        dict(_case("ragged", 2, 2_000_000, (512, 512), T=8, problems=64, sizes_seed=7),
             name="ragged_64"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi], odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["type1", "type1", "type1", "type2", "type2", "plan1", "type3", "grad2",
                       "ragged"])
    single = rng.random() < 0.7
    eps = 10.0 ** -(rng.randint(2, 6) if single else rng.choice([6, 8, 9, 10, 12]))
    modeord = rng.randint(0, 1)
    if kind == "ragged":
        top = _log(rng, 5e4, 2e6)
        return _case("ragged", 2, top, (512, 512), T=rng.randint(1, 8),
                     problems=rng.randint(3, 48), sizes_seed=rng.randint(100, 1 << 20))
    if kind == "type3":
        dim = rng.randint(1, 3)
        M, N = _log(rng, 2e3, 1 << 20), _log(rng, 2e3, 1 << 20)
        extent = rng.uniform(4.0, 16.0) if dim == 3 else rng.uniform(4.0, 40.0)
        return _case("type3", dim, M, single=True, eps=10.0 ** -rng.randint(3, 6), points="box",
                     extent=round(extent, 3), targets=N)
    if kind in ("plan1", "grad2"):
        n = [_log(rng, 48, 512 if kind == "grad2" else 1024) for _ in range(2)]
        M = _log(rng, 1e5, 4e6 if kind == "grad2" else 1e7)
        return _case(kind, 2, M, n, eps=10.0 ** -rng.randint(3, 6),
                     points=rng.choice(["uniform", "gauss"]))
    dim = rng.randint(1, 3)
    if dim == 1:
        n, M = [_log(rng, 256, 1 << 16)], _log(rng, 4e3, 1 << 20)
    elif dim == 2:
        n, M = [_log(rng, 40, 1024) for _ in range(2)], _log(rng, 4e3, 4e6 if single else 1e6)
    else:
        top = (256 if single else 96) if kind == "type2" else (128 if single else 64)
        n = [_log(rng, 24, top) for _ in range(3)]
        M = _log(rng, 1e4, (8e6 if kind == "type2" else 1e6) if single else 3e5)
    T = rng.choice([1, 1, 1, 2, 4]) if M * n[0] ** (dim - 1) < 3e9 and dim < 3 else 1
    sets = rng.choice([2, 5]) if kind == "type1" and dim == 2 and M <= 1e6 and T == 1 and \
        rng.random() < 0.3 else 1
    points = rng.choice(["uniform", "gauss"] if dim < 3 else ["uniform", "gauss", "koosh"])
    return _case(kind, dim, M, n, T=T, sets=sets, single=single, eps=eps, points=points,
                 modeord=modeord)


# ------------------------------------------------------------------ inputs


def _modes(case):
    return (case["n1"], case["n2"], case["n3"])[:case["dim"]]


def _types(case):
    return (torch.float32, torch.complex64) if case["single"] else (torch.float64,
                                                                    torch.complex128)


def _complex(shape, g, dtype):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=dtype)


def _points(case, g, shape):
    """`dim` coordinate arrays of `shape`; the last axis counts points."""
    real, _ = _types(case)
    dim, M = case["dim"], shape[-1]
    rand = lambda: torch.rand(shape, generator=g, device=DEVICE, dtype=real)  # noqa: E731
    if case["points"] == "uniform":
        return [(rand() * 2 - 1) * math.pi for _ in range(dim)]
    if case["points"] == "box":
        return [(rand() * 2 - 1) * case["extent"] for _ in range(dim)]
    if case["points"] == "gauss":
        # centre-dense: Gaussian about the origin, wrapped to [-pi, pi)
        return [torch.remainder(torch.randn(shape, generator=g, device=DEVICE, dtype=real) * 0.4
                                + math.pi, 2 * math.pi) - math.pi for _ in range(dim)]
    # koosh ball: golden-angle spokes of equidistant samples, acquisition order,
    # turned by a random angle per seed
    samples = max(16, int(round(math.sqrt(M / 4))))
    spokes = -(-M // samples)
    turn = float(torch.rand(1, generator=g, device=DEVICE, dtype=torch.float64)) * 2 * math.pi
    s = torch.arange(spokes, device=DEVICE, dtype=torch.float64)
    zc = 1 - (2 * s + 1) / spokes
    rc = torch.sqrt(1 - zc * zc)
    phi = s * math.pi * (3 - math.sqrt(5)) + turn
    r = -math.pi + 2 * math.pi * torch.arange(samples, device=DEVICE, dtype=torch.float64) / samples
    return [(d[:, None] * r[None, :]).reshape(-1)[:M].to(real).contiguous()
            for d in (rc * torch.cos(phi), rc * torch.sin(phi), zc)]


def _ragged_sizes(case):
    """Point counts (log-uniform from 1e4), grids and stacked transforms."""
    rng = np.random.default_rng(case["sizes_seed"])
    k = case["problems"]
    Ms = np.round(10 ** rng.uniform(4, math.log10(case["M"]), k)).astype(int)
    Ns = rng.choice([64, 128, 256, 512], k)
    Ts = rng.integers(1, case["T"] + 1, k)
    return [int(m) for m in Ms], [(int(n), int(n)) for n in Ns], [int(t) for t in Ts]


def _data(case, seed):
    """Inputs from the seed alone: points, source and what else the call takes."""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    _, cplx = _types(case)
    kind, M, T, sets = case["kind"], case["M"], case["T"], case["sets"]
    if kind == "ragged":
        Ms, _, Ts = _ragged_sizes(case)
        pts = [_points(case, g, (m,)) for m in Ms]
        return {"x": [p[0] for p in pts], "y": [p[1] for p in pts],
                "c": [_complex((t, m), g, cplx) for m, t in zip(Ms, Ts)]}
    pts = _points(case, g, (M,) if sets == 1 else (sets, M))
    if kind == "type3":
        tgt = _points(case, g, (case["targets"],))
        return {"pts": pts, "tgt": tgt, "src": _complex((M,), g, cplx)}
    if kind in ("type1", "plan1"):
        shape = (M,) if T == 1 else (T, M)
        return {"pts": pts, "src": _complex((sets,) + shape if sets > 1 else shape, g, cplx)}
    modes = _modes(case)
    if kind == "grad2":
        # a smooth image observed with noise
        k = [torch.arange(n, device=DEVICE, dtype=torch.float32) - n // 2 for n in modes]
        f = torch.exp(-(k[0][:, None] ** 2 + k[1][None, :] ** 2) / (2 * 64.0**2)).to(cplx)
        return {"pts": pts, "src": f, "d": _complex((M,), g, cplx)}
    return {"pts": pts, "src": _complex(modes if T == 1 else (T,) + modes, g, cplx)}


def prepare(case, seed):
    st = _data(case, seed)
    kind = case["kind"]
    st["case"] = case
    # keyword arguments a user's program holds beside its arrays
    st["kw"] = dict(eps=case["eps"], opts=Opts(modeord=case["modeord"]))
    if kind == "plan1":
        st["plan"] = Plan(1, _modes(case), iflag=1, eps=case["eps"], dtype=_types(case)[1],
                          device=DEVICE)
        st["fk"] = torch.empty(_modes(case), dtype=_types(case)[1], device=DEVICE)
    if kind == "ragged":
        Ms, shapes, Ts = _ragged_sizes(case)
        st["plan"] = RaggedPlan(shapes, Ms, Ts, eps=case["eps"], dtype=_types(case)[1])
    if kind == "grad2":
        st["leaves"] = [t.requires_grad_(True) for t in (st["src"], *st["pts"])]
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "type1":
        return nufft1(_modes(case), st["src"], *st["pts"], **st["kw"])
    if kind == "type2":
        return nufft2(st["src"], *st["pts"], **st["kw"])
    if kind == "type3":
        return nufft3(st["src"], *st["pts"], *st["tgt"], eps=case["eps"])
    if kind == "plan1":
        st["plan"].setpts(*st["pts"])
        st["plan"].execute(st["src"], st["fk"])
        return st["fk"]
    if kind == "ragged":
        return st["plan"].run(st["x"], st["y"], st["c"])
    f, x, y = st["leaves"]
    loss = (nufft2(f, x, y, eps=case["eps"]) - st["d"]).abs().pow(2).sum()
    gf, gx, gy = torch.autograd.grad(loss, [f, x, y])
    return {"loss": loss.detach(), "f": gf, "x": gx, "y": gy}


# ------------------------------------------------------------------ work


def _width(eps):
    return max(2, math.ceil(math.log10(20 / eps)))


def _transform_work(M, modes, T, sets, single, eps):
    """Bytes in and out and the arithmetic of the method (taps and FFT) of one
    type-1 or type-2 call."""
    dim, real = len(modes), 4 if single else 8
    ntot = math.prod(modes)
    nbytes = sets * (M * real * dim + T * 2 * real * (M + ntot))
    F = ntot * 2**dim
    return nbytes, sets * T * (4 * M * _width(eps) ** dim + 5 * F * math.log2(max(F, 2)))


def work(case):
    kind, M, eps = case["kind"], case["M"], case["eps"]
    if kind == "ragged":
        w = [_transform_work(m, s, t, 1, case["single"], eps)
             for m, s, t in zip(*_ragged_sizes(case))]
        return {"bytes": sum(a for a, _ in w), "flops": sum(b for _, b in w)}
    if kind == "type3":
        dim, N, ns = case["dim"], case["targets"], _width(eps)
        real = 4 if case["single"] else 8
        nf = 4 * case["extent"] ** 2 / math.pi + ns + 1
        Fi = (2 * nf) ** dim
        return {"bytes": (M + N) * real * (dim + 2),
                "flops": 4 * (M + N) * ns**dim + 5 * Fi * math.log2(Fi)}
    b, f = _transform_work(M, _modes(case), case["T"], case["sets"], case["single"], eps)
    if kind == "grad2":
        # forward, adjoint and the point gradients; inputs and outputs once
        return {"bytes": 2 * b + M * 8, "flops": 2 * f + 12 * M * _width(eps) ** 2}
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------ exact


def _freqs(n, modeord):
    k = torch.arange(n, device=DEVICE, dtype=torch.float64)
    if modeord == 0:
        return k - n // 2
    return torch.where(k < (n + 1) // 2, k, k - n)


def _phases(x, k, sign):
    ph = sign * x.double()[:, None] * k[None, :]
    return torch.polar(torch.ones_like(ph), ph)


def _khatri(E):
    """Row-wise product of the phase matrices of several axes, (m, prod n)."""
    out = E[0]
    for e in E[1:]:
        out = (out[:, :, None] * e[:, None, :]).reshape(out.shape[0], -1)
    return out


def _chunks(M, modes, T=1):
    step = max(256, int(4e7 // max(math.prod(modes[1:]), sum(modes), 1)))
    return [(a, min(M, a + step)) for a in range(0, M, step)]


def _sum1(pts, c, modes, modeord):
    """f[t, k] = sum_j c[t, j] exp(+i k.x_j), c (T, M)."""
    ks = [_freqs(n, modeord) for n in modes]
    out = torch.zeros((c.shape[0], modes[0], math.prod(modes[1:])), dtype=torch.complex128,
                      device=DEVICE)
    one = torch.ones((1, 1), dtype=torch.complex128, device=DEVICE)
    for a, b in _chunks(c.shape[1], modes):
        E0 = _phases(pts[0][a:b], ks[0], 1).t().contiguous()
        rest = _khatri([_phases(p[a:b], k, 1) for p, k in zip(pts[1:], ks[1:])]) \
            if len(modes) > 1 else one.expand(b - a, 1)
        for t in range(c.shape[0]):
            out[t] += E0 @ (c[t, a:b].to(torch.complex128)[:, None] * rest)
    return out.reshape((c.shape[0],) + tuple(modes))


def _sum2(pts, f, modeord, sign=-1, along=None):
    """c[t, j] = sum_k f[t, k] exp(i sign k.x_j), f (T, *modes); with `along`,
    its derivative with respect to that coordinate."""
    modes = tuple(f.shape[1:])
    ks = [_freqs(n, modeord) for n in modes]
    F = f.to(torch.complex128)
    if along is not None:
        shape = [1] * len(modes)
        shape[along] = -1
        F = F * (1j * sign * ks[along]).reshape(shape)
    F = F.reshape(f.shape[0], modes[0], -1)
    M = pts[0].shape[0]
    out = torch.empty((f.shape[0], M), dtype=torch.complex128, device=DEVICE)
    for a, b in _chunks(M, modes):
        E0 = _phases(pts[0][a:b], ks[0], sign)
        rest = _khatri([_phases(p[a:b], k, sign) for p, k in zip(pts[1:], ks[1:])]) \
            if len(modes) > 1 else None
        for t in range(f.shape[0]):
            v = E0 @ F[t]
            out[t, a:b] = v[:, 0] if rest is None else (v * rest).sum(1)
    return out


def exact(case, seed):
    kind, M, T, sets = case["kind"], case["M"], case["T"], case["sets"]
    if kind == "ragged":
        Ms, shapes, Ts = _ragged_sizes(case)
        if sum(m * math.prod(s) * t for m, s, t in zip(Ms, shapes, Ts)) > EXACT_LIMIT:
            return None
        d = _data(case, seed)
        return [_sum1((x, y), c, s, 0)
                for x, y, c, s in zip(d["x"], d["y"], d["c"], shapes)]
    if kind == "type3":
        if M * case["targets"] > 1.5e11:
            return None
        d = _data(case, seed)
        c = d["src"].to(torch.complex128)
        out = torch.empty(case["targets"], dtype=torch.complex128, device=DEVICE)
        step = max(1, int(1e8 // M))
        x = torch.stack([p.double() for p in d["pts"]], 1)
        s = torch.stack([t.double() for t in d["tgt"]], 1)
        for a in range(0, case["targets"], step):
            ph = -(s[a:a + step] @ x.t())
            out[a:a + step] = torch.polar(torch.ones_like(ph), ph) @ c
        return out
    modes = _modes(case)
    cost = M * math.prod(modes) * T * sets * (4 if kind == "grad2" else 1)
    if cost > EXACT_LIMIT:
        return None
    d = _data(case, seed)
    pts = d["pts"]
    if kind in ("type1", "plan1"):
        if sets > 1:
            return torch.stack([_sum1([p[i] for p in pts], d["src"][i][None], modes,
                                      case["modeord"])[0] for i in range(sets)])
        f = _sum1(pts, d["src"].reshape(T, M), modes, case["modeord"])
        return f[0] if T == 1 else f
    if kind == "type2":
        c = _sum2(pts, d["src"].reshape((T,) + modes), case["modeord"])
        return c[0] if T == 1 else c
    # loss = sum |r|^2, r = B f - d: grad_f = 2 B^H r (a type 1 with the
    # opposite sign), grad_x = 2 Re(conj(r) dB/dx f)
    f = d["src"][None]
    r = _sum2(pts, f, 0)[0] - d["d"].to(torch.complex128)
    out = {"loss": r.abs().pow(2).sum(), "f": 2 * _sum1(pts, r[None], modes, 0)[0]}
    for i, name in enumerate("xy"):
        out[name] = 2 * (r.conj() * _sum2(pts, f, 0, along=i)[0]).real
    return out
