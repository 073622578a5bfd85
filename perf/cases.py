"""Timed cases of the transforms, over the range that programs use them in.

A case is a dict of plain values:

* ``kind``: "scalar" (synthesis and analysis of real fields), "sphtor" (the
  spheroidal/toroidal vector pair), "qst" (3-D vector fields: a scalar and a
  vector transform on one grid), "grad" (a loss on the grid and its gradient
  with respect to the coefficients) or "uneven" (one batch object over several
  truncations);
* ``lmax, nlat, nlon, grid, norm, mres``: the configuration;
* ``nf``: fields (0: the single-field entry points, no batch axis);
* ``dtype``: "f64" or "f32" arrays; ``precision``: the batch contraction;
* ``way``: "both" (coefficients to the grid and back), "synthesis" or "analysis".

``exact`` evaluates the same transforms from their definition in 64 bits: nodes
and sectoral values in extended precision, the three-term recurrence in the
degree for every order at once, theta derivatives from the neighbouring orders,
and torch's FFT.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The package lives in a folder whose name has a dot: loaded by its place."""
    name = "shtnskit_jl_amd"
    if name not in sys.modules:
        folder = os.path.join(_ROOT, "shtnskit.jl_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        module = importlib.util.module_from_spec(spec)
        sys.modules[name] = module
        spec.loader.exec_module(module)
    return sys.modules[name]


def _case(kind, lmax, nlat, nlon, nf=0, dtype="f64", precision="fp64", way="both", grid="gauss",
          norm="orthonormal", mres=1):
    return {"kind": kind, "lmax": lmax, "nlat": nlat, "nlon": nlon, "nf": nf, "dtype": dtype,
            "precision": precision, "way": way, "grid": grid, "norm": norm, "mres": mres}


def listed():
    named = {
        # A small field, transformed in every step of a long run or in a unit test: latency.
        "scalar_63": _case("scalar", 63, 64, 128),
        # One field on the grid that create_config gives by default (nlat = lmax + 2,
        # nlon = 2 lmax + 2, here 2^5 * 19: not a power of two).
        "scalar_303_default": _case("scalar", 303, 305, 608),
        # The benchmark's headline: one field, there and back.
        "scalar_1023": _case("scalar", 1023, 1024, 2048),
        # The largest truncation in the tests: one high-resolution field.
        "scalar_2047": _case("scalar", 2047, 2048, 4096),
        # A wind or flow field of a model step, on the dealiased grid (3/2 rule, odd nlat).
        "sphtor_340": _case("sphtor", 340, 511, 1024),
        # Radial shells of a 3-D flow (Q, S, T), all transformed at once.
        "qst_170x24": _case("qst", 170, 256, 512, nf=24),
        # Pressure levels of a scalar field in one call.
        "scalar_255x37": _case("scalar", 255, 256, 512, nf=37),
        # The benchmark's vector batch, on the matrix cores.
        "sphtor_511x32_split": _case("sphtor", 511, 512, 1024, nf=32, precision="split"),
        # The benchmark's scalar batches, on the matrix cores in both precisions.
        "scalar_1023x16_split": _case("scalar", 1023, 1024, 2048, nf=16, precision="split"),
        "scalar_1023x16_fp32": _case("scalar", 1023, 1024, 2048, nf=16, precision="fp32"),
        # Loss and gradient through the synthesis, single precision: fitting coefficients to grids.
        "grad_511x16_f32": _case("grad", 511, 512, 1024, nf=16, dtype="f32"),
        # Fields of several truncations in one batch object.
        "uneven_64_split": dict(_case("uneven", 1023, 1024, 2048, precision="split"),
                                groups="1023:10,511:13,255:12,127:13,63:16"),
    }
    return [dict(c, name=n) for n, c in named.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _orders(case):
    return range(0, case["lmax"] + 1, case["mres"])


def _folded(lmax, nlat, mres=1):
    """(latitude pair, degree, order) triples of one field in one direction."""
    return (nlat + 1) // 2 * sum(lmax - m + 1 for m in range(0, lmax + 1, mres))


_MOST_TRIPLES = 16 * 1024 * 512 * 1025 // 2  # the batch of 16 at lmax 1023


def _size(rng, lmax, grid):
    if grid != "gauss":
        nlat = max(2 * lmax + 1, 2)  # the equiangular default
    else:
        nlat = rng.choice([lmax + 1, lmax + 2, (3 * lmax + 1) // 2 + 1])
    nlon = rng.choice([2 * lmax + 1, 2 * lmax + 2, 2 * lmax + 2, 2 * (nlat + nlat % 2)])
    if nlon > 4096:
        nlon = 2 * lmax + 2
    return nlat, nlon


def draw(rng):
    kind = rng.choices(["scalar", "sphtor", "qst", "grad", "uneven"], [8, 4, 2, 2, 1])[0]
    if kind == "uneven":
        while True:
            sizes = sorted({_log_int(rng, 31, 1023) for _ in range(rng.randint(2, 5))}, reverse=True)
            counts = [rng.randint(1, 16) for _ in sizes]
            if sum(n * _folded(l, l + 1) for l, n in zip(sizes, counts)) <= _MOST_TRIPLES // 2:
                break
        c = _case("uneven", sizes[0], sizes[0] + 1, 2 * sizes[0] + 2, precision=rng.choice(["fp64", "split", "fp32"]))
        return dict(c, groups=",".join("%d:%d" % p for p in zip(sizes, counts)))
    components = {"scalar": 1, "grad": 1, "sphtor": 4, "qst": 5}[kind]
    while True:
        lmax = _log_int(rng, 31, 2047)
        single = kind in ("scalar", "sphtor") and rng.random() < 0.4
        nf = 0 if single else _log_int(rng, 2, 64)
        grid = rng.choices(["gauss", "regular", "regular_poles"], [8, 2, 1])[0]
        if grid == "regular_poles" and kind != "scalar":
            grid = "regular"
        if grid != "gauss" and lmax > 700:
            continue
        nlat, nlon = _size(rng, lmax, grid)
        mres = rng.choices([1, 2, 3], [8, 1, 1])[0]
        if components * max(nf, 1) * _folded(lmax, nlat, mres) > _MOST_TRIPLES or \
                components * max(nf, 1) * nlat * nlon > 16 * 1024 * 2048:
            continue
        break
    dtype = rng.choices(["f64", "f32"], [2, 1])[0]
    precision = "fp64" if nf < 2 or kind == "grad" else rng.choice(["fp64", "split", "fp32"])
    way = "both" if kind == "grad" else rng.choices(["both", "synthesis", "analysis"], [4, 1, 1])[0]
    norm = rng.choices(["orthonormal", "schmidt", "fourpi"], [6, 1, 1])[0]
    return _case(kind, lmax, nlat, nlon, nf=nf, dtype=dtype, precision=precision, way=way, grid=grid, norm=norm,
                 mres=mres)


# --------------------------------------------------------------------------- inputs
def _groups(case):
    """The (lmax, nlat, nlon, fields) of an uneven batch."""
    out = []
    for text in case["groups"].split(","):
        l, n = (int(v) for v in text.split(":"))
        out.append((l, l + 1, 2 * l + 2, n))
    return out


def _real(case):
    return torch.float32 if case["dtype"] == "f32" else torch.float64


def _spectrum(gen, lmax, mres, nf, power, rdt, lmin=0):
    """Complex Gaussian coefficients with a power-law spectrum, degree fastest in memory."""
    dev = gen.device
    n = max(nf, 1)
    a = torch.randn(n, lmax + 1, lmax + 1, 2, dtype=torch.float64, device=dev, generator=gen)
    l = torch.arange(lmax + 1, device=dev, dtype=torch.float64)
    m = l[:, None]
    keep = (l >= m) & (l >= lmin) & (torch.remainder(m, mres) == 0)
    a = a * torch.where(keep, (l + 1.0) ** -power, torch.zeros((), device=dev, dtype=torch.float64))[None, :, :, None]
    a[:, 0, :, 1] = 0.0
    a = torch.view_as_complex(a).to(torch.complex64 if rdt == torch.float32 else torch.complex128)
    return (a if nf else a[0]).permute(*((2, 1, 0) if nf else (1, 0)))


def _grid_noise(gen, nlat, nlon, nf, rdt):
    f = torch.randn(max(nf, 1), nlon, nlat, dtype=torch.float64, device=gen.device, generator=gen).to(rdt)
    return (f if nf else f[0]).permute(*((2, 1, 0) if nf else (1, 0)))


def _inputs(case, seed):
    """The arrays of a case: a list of spectra (or of grids for an analysis alone)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rdt, kind = _real(case), case["kind"]
    if kind == "uneven":
        return [_spectrum(gen, l, 1, n, 1.5, rdt) for l, _, _, n in _groups(case)]
    lmax, nf, mres = case["lmax"], case["nf"], case["mres"]
    comps = {"scalar": 1, "grad": 2, "sphtor": 2, "qst": 3}[kind]
    if case["way"] == "analysis":
        return [_grid_noise(gen, case["nlat"], case["nlon"], nf, rdt) for _ in range(comps)]
    if kind == "grad":
        return [_spectrum(gen, lmax, mres, nf, 1.0, rdt),
                _grid_noise(gen, case["nlat"], case["nlon"], nf, rdt)]
    out = []
    if kind != "sphtor":
        out.append(_spectrum(gen, lmax, mres, nf, 1.5, rdt))
    if kind != "scalar":
        out += [_spectrum(gen, lmax, mres, nf, 2.0, rdt, lmin=1) for _ in range(2)]
    return out


def _config(shtk, lmax, nlat, nlon, grid="gauss", norm="orthonormal", mres=1):
    kw = {"nlon": nlon, "norm": norm, "mres": mres}
    if grid == "gauss":
        cfg = shtk.create_gauss_config(lmax, nlat, **kw)
    else:
        cfg = shtk.create_regular_config(lmax, nlat, include_poles=grid == "regular_poles", **kw)
    cfg.plan  # made now, as a program that transforms many fields does
    return cfg


def prepare(case, seed):
    shtk = _package()
    state = {"case": case, "lib": shtk, "in": _inputs(case, seed)}
    if case["kind"] == "uneven":
        cfgs = [_config(shtk, l, nlat, nlon) for l, nlat, nlon, _ in _groups(case)]
        state["batch"] = shtk.UnevenBatch(cfgs, [g[3] for g in _groups(case)], precision=case["precision"])
        return state
    cfg = state["cfg"] = _config(shtk, case["lmax"], case["nlat"], case["nlon"], case["grid"], case["norm"],
                                 case["mres"])
    if case["kind"] == "grad":
        w = torch.as_tensor(cfg.w, dtype=_real(case), device="cuda")
        state["w"] = w.reshape((-1, 1) + ((1,) if case["nf"] else ()))
    return state


# --------------------------------------------------------------------------- one pass
def run(state):
    case, lib, x = state["case"], state["lib"], state["in"]
    kind, way = case["kind"], case["way"]
    if kind == "uneven":
        grids = state["batch"].synthesis(x)
        return {"grid": grids, "spec": state["batch"].analysis(grids)}
    cfg = state["cfg"]
    if kind == "grad":
        a = x[0].detach().requires_grad_(True)
        f = lib.ad.synthesis(cfg, a)
        loss = (state["w"] * (f - x[1]) ** 2).sum()
        g, = torch.autograd.grad(loss, a)
        return {"grid": f.detach(), "loss": loss.detach(), "grad": g}
    if case["nf"]:
        kw = {"precision": case["precision"]}
        to_grid = {"scalar": lib.synthesis_batch, "sphtor": lib.synthesis_sphtor_batch,
                   "qst": lib.synthesis_qst_batch}[kind]
        to_spec = {"scalar": lib.analysis_batch, "sphtor": lib.analysis_sphtor_batch,
                   "qst": lib.analysis_qst_batch}[kind]
    else:
        kw = {}
        to_grid = {"scalar": lib.synthesis, "sphtor": lib.synthesis_sphtor}[kind]
        to_spec = {"scalar": lib.analysis, "sphtor": lib.analysis_sphtor}[kind]
    out = {}
    if way != "analysis":
        x = to_grid(cfg, *x, **kw)
        x = x if isinstance(x, tuple) else (x,)
        out["grid"] = x
    if way != "synthesis":
        out["spec"] = to_spec(cfg, *x, **kw)
    return out


def work(case):
    """Arrays in and out once; two real columns per field and component against the folded
    Legendre functions (2 flop each for real and imaginary part), the recurrence (4 flop)
    once per direction however many fields share it, and 2.5 n log2 n per grid row."""
    if case["kind"] == "uneven":
        parts = [dict(case, kind="scalar", lmax=l, nlat=nlat, nlon=nlon, nf=n) for l, nlat, nlon, n in _groups(case)]
        each = [work(p) for p in parts]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    kind, nf = case["kind"], max(case["nf"], 1)
    comps = {"scalar": 1, "grad": 1, "sphtor": 2, "qst": 3}[kind]
    size = 4 if case["dtype"] == "f32" else 8
    spec = 2 * size * sum(case["lmax"] - m + 1 for m in _orders(case))
    grid = size * case["nlat"] * case["nlon"]
    both = case["way"] == "both"
    ways = 2 if both else 1
    triples = _folded(case["lmax"], case["nlat"], case["mres"])
    rows = 2.5 * case["nlat"] * case["nlon"] * math.log2(max(case["nlon"], 2))
    flops = ways * (4.0 * triples * comps * nf + 4.0 * triples + rows * comps * nf)
    if kind == "grad":
        moved = nf * (2 * spec + 2 * grid)  # coefficients and target in, grid and gradient out
    else:
        moved = comps * nf * (spec + grid + (spec if both else 0))
    return {"bytes": float(moved), "flops": float(flops)}


# --------------------------------------------------------------------------- 64-bit values
def _nodes(grid, n):
    """cos(theta), sin(theta) (north first) and weights in extended precision."""
    ld = np.longdouble
    pi = ld("3.14159265358979323846264338327950288")
    if grid == "gauss":
        k = np.arange(1, n + 1, dtype=ld)
        z = np.cos(pi * (k - ld(0.25)) / (n + ld(0.5)))
        for _ in range(8):
            p0, p1 = np.ones_like(z), z.copy()
            for l in range(2, n + 1):
                p0, p1 = p1, ((2 * l - 1) * z * p1 - (l - 1) * p0) / ld(l)
            d = n * (z * p1 - p0) / (z * z - 1)
            z = z - p1 / d
        return z, np.sqrt((1 - z) * (1 + z)), 2 / ((1 - z * z) * d * d)
    if grid == "regular":
        th = (np.arange(n, dtype=ld) + ld(0.5)) * pi / n
        w = np.ones(n, dtype=ld)
        for k in range(1, n // 2 + 1):
            w -= 2 * np.cos(2 * k * th) / ld(4 * k * k - 1)
        return np.cos(th), np.sin(th), 2 * w / n
    N = n - 1
    th = np.arange(n, dtype=ld) * pi / N
    w = np.ones(n, dtype=ld)
    for k in range(1, (N - 1) // 2 + 1):
        w -= 2 * np.cos(2 * k * th) / ld(4 * k * k - 1)
    if N % 2 == 0:
        w -= np.cos(N * th) / ld(N * N - 1)
    w = 2 * w / N
    w[0] = w[-1] = 1 / ld(N * N - 1) if N % 2 == 0 else 1 / ld(N * N)
    x, s = np.cos(th), np.sin(th)
    x[0], x[-1], s[0], s[-1] = 1, -1, 0, 0
    return x, s, w


def _rows(grid, nlat, lmax, mtop):
    """For each degree l the array P_l^m(x_i) (orthonormal, Condon-Shortley) of shape
    (min(l, mtop) + 1, nlat), as a generator; values under 2^-360 may be given as zero."""
    x_, s_, _ = _nodes(grid, nlat)
    # sectoral values as mantissa and exponent
    man = np.empty((mtop + 1, nlat), dtype=np.longdouble)
    ex = np.empty((mtop + 1, nlat), dtype=np.int64)
    cur, e = np.full(nlat, 1 / np.sqrt(4 * np.longdouble("3.14159265358979323846264338327950288"))), np.zeros(nlat, np.int64)
    for m in range(mtop + 1):
        if m:
            cur = -cur * s_ * np.sqrt(np.longdouble(2 * m + 1) / (2 * m))
        cur, d = np.frexp(cur)
        e = e + d
        man[m], ex[m] = cur, e
    k = np.where(ex < -400, (-ex - 400 + 511) // 512, 0)
    start = torch.from_numpy(np.ldexp(man, np.clip(ex + 512 * k, -1000, 1000)).astype(np.float64)).cuda()
    k = torch.from_numpy(k).cuda()
    x = torch.from_numpy(x_.astype(np.float64)).cuda()
    m2 = torch.arange(mtop + 1, device="cuda", dtype=torch.float64)[:, None] ** 2
    prev = torch.zeros(mtop + 1, nlat, dtype=torch.float64, device="cuda")
    cur = torch.zeros_like(prev)
    for l in range(lmax + 1):
        if l > 0:
            # orders below l step on; order l starts from its sectoral value
            n = min(l, mtop + 1)
            den = l * l - m2[:n]
            a = torch.sqrt((4.0 * l * l - 1.0) / den)
            b = torch.sqrt((2.0 * l + 1.0) * ((l - 1.0) ** 2 - m2[:n]) / ((2.0 * l - 3.0) * den)) if l > 1 else 0.0 * den
            nxt = torch.addcmul(-b * prev[:n], a * x, cur[:n])
            prev[:n] = cur[:n]
            cur[:n] = nxt
            if l % 8 == 0:
                big = (k[:n] > 0) & (torch.maximum(cur[:n].abs(), prev[:n].abs()) > 2.0 ** 100)
                for q in (cur, prev):
                    q[:n] = torch.where(big, q[:n] * 2.0 ** -512, q[:n])
                k[:n] -= big.to(k.dtype)
        if l <= mtop:
            cur[l] = start[l]
        n = min(l, mtop) + 1
        yield torch.where(k[:n] == 0, cur[:n], torch.zeros((), dtype=torch.float64, device="cuda"))


def _scale(norm, l):
    return {"orthonormal": 1.0, "fourpi": math.sqrt(4 * math.pi), "schmidt": math.sqrt(4 * math.pi / (2 * l + 1))}[norm]


def _derivatives(P, l, mmax, s):
    """dP/dtheta and m P / sin(theta) of the orders 0 .. min(l, mmax) from P of the orders up to mmax + 1."""
    n = min(l, mmax) + 1
    m = torch.arange(n, device="cuda", dtype=torch.float64)[:, None]
    up = torch.zeros(n, P.shape[1], dtype=torch.float64, device="cuda")
    k = min(n, P.shape[0] - 1)
    up[:k] = P[1:k + 1]
    down = torch.zeros_like(up)
    if n > 1:
        down[1:] = P[:n - 1]
    if l >= 1:
        down[0] = -up[0]
    d = 0.5 * (torch.sqrt((l - m) * (l + m + 1.0)) * up - torch.sqrt((l + m) * (l - m + 1.0)) * down)
    return d, m * P[:n] / s


def _columns(a):
    """A spectrum (l, m[, field]) as (l, m, field, re/im) doubles."""
    a = a if a.dim() == 3 else a[..., None]
    return torch.view_as_real(a.to(torch.complex128).contiguous())


def _to_grid(F, nlon):
    """Orders (m, lat, field, re/im) -> real grid (lat, lon, field)."""
    c = torch.view_as_complex(F.contiguous())
    full = torch.zeros(nlon // 2 + 1, c.shape[1], c.shape[2], dtype=torch.complex128, device="cuda")
    full[:c.shape[0]] = c
    return torch.fft.irfft(full, n=nlon, dim=0, norm="forward").permute(1, 0, 2)


def _to_orders(f, mmax):
    """Real grid (lat, lon, field) -> Fourier sums (m, lat, re/im x field) without a factor."""
    f = (f if f.dim() == 3 else f[..., None]).to(torch.float64)
    c = torch.fft.rfft(f.permute(1, 0, 2).contiguous(), dim=0)[:mmax + 1]
    return torch.view_as_real(c)


def _synth(case, spectra):
    """Exact grids of one scalar spectrum or of a vector pair."""
    lmax, nlat, nlon = case["lmax"], case["nlat"], case["nlon"]
    cols = [_columns(a) for a in spectra]
    vector = len(cols) == 2
    F = [torch.zeros(lmax + 1, nlat, cols[0].shape[2], 2, dtype=torch.float64, device="cuda") for _ in cols]
    s = torch.from_numpy(_nodes(case["grid"], nlat)[1].astype(np.float64)).cuda()

    def add(k, n, row, coef):
        F[k][:n].addcmul_(row[:, :, None, None], coef[:, None])

    def turned(c):  # i c
        return torch.stack((-c[..., 1], c[..., 0]), dim=-1)

    for l, P in enumerate(_rows(case["grid"], nlat, lmax, lmax + (1 if vector else 0))):
        n = l + 1
        c = [q[l, :n] * _scale(case["norm"], l) for q in cols]
        if not vector:
            add(0, n, P, c[0])
            continue
        d, q = _derivatives(P, l, lmax, s)
        add(0, n, d, c[0])
        add(0, n, q, -turned(c[1]))
        add(1, n, q, turned(c[0]))
        add(1, n, d, c[1])
    grids = [_to_grid(f, nlon) for f in F]
    return [g if case["nf"] or case["kind"] == "uneven" else g[..., 0] for g in grids]


def _anal(case, grids, weights=True, double=False):
    """Exact coefficients of one real grid or of a vector pair. ``weights=False``: plain sums
    over the grid; ``double``: orders m > 0 count twice (the gradient of a real synthesis)."""
    lmax, nlat, nlon, mres = case["lmax"], case["nlat"], case["nlon"], case["mres"]
    _, s, w = _nodes(case["grid"], nlat)
    s = torch.from_numpy(s.astype(np.float64)).cuda()
    w = torch.from_numpy(w.astype(np.float64)).cuda() * (2 * math.pi / nlon) if weights else torch.ones_like(s)
    G = [_to_orders(f, lmax) * w[None, :, None, None] for f in grids]
    nf = G[0].shape[2]
    G = [g.reshape(lmax + 1, nlat, 2 * nf) for g in G]
    out = [torch.zeros(lmax + 1, lmax + 1, nf, dtype=torch.complex128, device="cuda") for _ in G]
    kept = (torch.arange(lmax + 1, device="cuda") % mres == 0).to(torch.float64)
    twice = torch.full((lmax + 1,), 2.0 if double else 1.0, dtype=torch.float64, device="cuda")
    twice[0] = 1.0

    def dot(row, k):
        n = row.shape[0]
        return torch.view_as_complex(torch.bmm(row[:, None, :], G[k][:n])[:, 0].reshape(n, nf, 2).contiguous())

    for l, P in enumerate(_rows(case["grid"], nlat, lmax, lmax + (1 if len(G) == 2 else 0))):
        n = l + 1
        sc = _scale(case["norm"], l)
        f = (kept * twice)[:n, None] * (1.0 / sc if weights else sc)
        if len(G) == 1:
            out[0][l, :n] = f * dot(P, 0)
        elif l > 0:
            d, q = _derivatives(P, l, lmax, s)
            f = f / (l * (l + 1.0))
            out[0][l, :n] = f * (dot(d, 0) - 1j * dot(q, 1))
            out[1][l, :n] = f * (1j * dot(q, 0) + dot(d, 1))
    return [o if case["nf"] else o[..., 0] for o in out]


def exact(case, seed):
    x = _inputs(case, seed)
    kind, way = case["kind"], case["way"]
    if kind == "uneven":
        grids = [_synth(dict(case, lmax=l, nlat=nlat, nlon=nlon, nf=n), [a])[0]
                 for a, (l, nlat, nlon, n) in zip(x, _groups(case))]
        return {"grid": grids, "spec": [a.to(torch.complex128) for a in x]}
    if kind == "grad":
        f, = _synth(case, x[:1])
        w = torch.from_numpy(_nodes(case["grid"], case["nlat"])[2].astype(np.float64)).cuda()
        w = w.reshape((-1, 1) + ((1,) if case["nf"] else ()))
        r = f - x[1].to(torch.float64)
        g, = _anal(case, [2.0 * w * r], weights=False, double=True)
        return {"grid": f, "loss": (w * r * r).sum(), "grad": g}
    parts = [x[:1], x[1:]] if kind == "qst" else [x]
    out = {}
    if way != "analysis":
        out["grid"] = tuple(g for p in parts for g in _synth(case, p))
        # every grid here integrates the products of two functions of the truncation exactly
        spec = [a.to(torch.complex128) for a in x]
    else:
        spec = [a for p in parts for a in _anal(case, p)]
    if way != "synthesis":
        out["spec"] = spec[0] if kind == "scalar" else tuple(spec)
    return out
