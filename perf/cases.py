"""The work that programs using shtns_amd have it do, as cases that can be timed.

A case is one call, or one short sequence of calls, of the torch interface on fields that
already are on the GPU: synthesis (spectrum to grid), analysis (grid to spectrum), both, or a
differentiated synthesis.  Its keys:

  kind    scalar, vector (spheroidal/toroidal pairs), cplx (complex-valued fields)
  step    synth, analys, pair (synthesis then analysis of its result), grad (synthesis with
          loss and gradient through shtns_amd.autograd)
  dtype   f64 or f32 (single-precision arrays; scalar fields only)
  lmax, mres, nlat, nphi, nf (fields or vector pairs per call), ltr (0: no truncation)
  layout  theta (the C interface's native layout) or phi (the Python default)
  polar   the polar threshold given to set_grid (1e-10 is its default)

listed() has one case for each kind of program; draw() gives more of the same ranges.
"""
import functools
import math

import numpy as np
import torch

import shtns_amd
from shtns_amd import autograd

DEV = "cuda"


def _case(name, kind, step, dtype, lmax, nlat, nphi, nf, layout, polar=0.0, mres=1, ltr=0):
    c = {"kind": kind, "step": step, "dtype": dtype, "lmax": lmax, "mres": mres, "nlat": nlat, "nphi": nphi, "nf": nf,
         "ltr": ltr, "layout": layout, "polar": polar}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one low-resolution field on the dealiased grid, Python defaults
        _case("synth_l63_f1", "scalar", "synth", "f64", 63, 96, 192, 1, "phi", polar=1e-10),
        # one field of a small simulation or a data set on a 1.4-degree grid
        _case("analys_l127_f1", "scalar", "analys", "f64", 127, 192, 384, 1, "theta"),
        # training through a synthesis: loss and gradient of a mini-batch
        _case("grad_l127_f8", "scalar", "grad", "f64", 127, 192, 384, 8, "phi", polar=1e-10),
        # the grid set_grid picks by itself for a ragged lmax (nphi = 720, not a power of two),
        # three fields truncated below lmax: filtering
        _case("synth_l340_f3_ltr", "scalar", "synth", "f64", 340, 342, 720, 3, "phi", polar=1e-10, ltr=301),
        # the same kind of grid, a handful of fields of a data set analysed at once
        _case("analys_l250_f5", "scalar", "analys", "f64", 250, 252, 512, 5, "phi", polar=1e-10),
        # the shells of a simulation at moderate resolution, Python's layout
        _case("analys_l255_f32", "scalar", "analys", "f64", 255, 384, 768, 32, "phi", polar=1e-10),
        # flow fields: spheroidal/toroidal pairs at lmax = 511
        _case("vpair_l511_f32", "vector", "pair", "f64", 511, 768, 1536, 32, "theta"),
        # single-precision fields in the C interface's layout
        _case("synth_f32_l511_f16", "scalar", "synth", "f32", 511, 768, 1536, 16, "theta"),
        # complex-valued fields (waves, spin-weighted quantities)
        _case("cplx_pair_l511_f4", "cplx", "pair", "f64", 511, 768, 1536, 4, "theta"),
        # a high-resolution batch, each direction
        _case("synth_l1023_f16", "scalar", "synth", "f64", 1023, 1536, 3072, 16, "theta"),
        _case("analys_l1023_f16", "scalar", "analys", "f64", 1023, 1536, 3072, 16, "theta"),
        # the largest: one very high-resolution field there and back
        _case("pair_l4095_f1", "scalar", "pair", "f64", 4095, 6144, 12288, 1, "theta"),
    ]


def _smooth(n):
    """Smallest even number >= n with no prime factor above 5, as set_grid picks nphi."""
    n += n & 1
    while True:
        t = n
        for p in (2, 3, 5):
            while t % p == 0:
                t //= p
        if t == 1:
            return n
        n += 2


#: a drawn case does at most this much Legendre work (flop per pass)
_DRAW_FLOPS = 5.0e10


def draw(rng):
    kind, step, dtype = rng.choice([("scalar", "synth", "f64"), ("scalar", "analys", "f64"), ("scalar", "pair", "f64"),
                                    ("scalar", "grad", "f64"), ("vector", "synth", "f64"), ("vector", "analys", "f64"),
                                    ("cplx", "synth", "f64"), ("cplx", "analys", "f64"), ("scalar", "synth", "f32"),
                                    ("scalar", "analys", "f32")])
    lmax = int(round(math.exp(rng.uniform(math.log(40), math.log(1400)))))
    if rng.random() < 0.35:   # 2^k - 1 and the like are common
        lmax = min((63, 95, 127, 191, 255, 383, 511, 767, 1023), key=lambda v: abs(math.log(v / lmax)))
    mres = rng.choice((2, 3, 4)) if kind != "cplx" and rng.random() < 0.15 else 1
    mmax = lmax // mres
    if rng.random() < 0.6:   # dealiased: 3/2 of the degrees
        nlat = 3 * (lmax + 1) // 2
        nphi = _smooth(3 * mmax + 3)
    else:                    # the sizes set_grid picks
        nlat = lmax + 2 + (lmax & 1)
        nphi = _smooth(2 * mmax + 2)
    nlat += nlat & 1
    if rng.random() < 0.15:
        nlat += 1            # an odd grid has a row on the equator
    c = _case(None, kind, step, dtype, lmax, nlat, nphi, 1, rng.choice(("theta", "phi")), rng.choice((0.0, 1e-10)), mres)
    most = max(1.0, min(48.0, _DRAW_FLOPS / work(c)["flops"]))
    c["nf"] = int(round(math.exp(rng.uniform(0.0, math.log(most)))))
    if rng.random() < 0.1 and kind != "cplx":
        c["ltr"] = int(lmax * rng.uniform(0.5, 0.95))
    return c


# ---- sizes and work ----------------------------------------------------------------------
def _nlm(lmax, mmax, mres):
    return sum(lmax + 1 - im * mres for im in range(mmax + 1))


def work(case):
    """One pass's inputs read and outputs written once, and the contraction's and the FFTs'
    operations (one complex x real multiply-add per degree, order and latitude pair and
    parity; 2.5 n log2 n per real FFT of n points)."""
    L, mres, nlat, nphi, nf = case["lmax"], case["mres"], case["nlat"], case["nphi"], case["nf"]
    mmax = L // mres
    parts = {"scalar": 1, "vector": 2, "cplx": 2}[case["kind"]]   # real fields per field
    times = 2 if case["step"] in ("pair", "grad") else 1
    real = 4 if case["dtype"] == "f32" else 8
    ltr = case["ltr"] or L
    leg = 2.0 * nlat * _nlm(ltr, min(mmax, ltr // mres), mres)
    fft = 2.5 * nlat * nphi * math.log2(nphi)
    spec, spat = 2.0 * real * _nlm(L, mmax, mres), float(real * nlat * nphi)
    flops = nf * parts * times * (leg + fft)
    nbytes = nf * parts * (spec + spat) * times
    return {"bytes": nbytes, "flops": flops}


@functools.lru_cache(maxsize=4)
def _lm(L, mres):
    """Degrees and orders of the spectral layout (order by order)."""
    ls = [np.arange(m, L + 1) for m in range(0, L + 1, mres)]
    ms = [np.full(L + 1 - m, m) for m in range(0, L + 1, mres)]
    return torch.from_numpy(np.concatenate(ls)).to(DEV), torch.from_numpy(np.concatenate(ms)).to(DEV)


# ---- inputs ------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 7919 + 17)
    return g


def _spectrum(case, g):
    """Coefficients of a field with a decaying spectrum, real at m = 0; complex-valued fields:
    all (l, m), -l <= m <= l, degree by degree."""
    L, nf = case["lmax"], case["nf"]
    if case["kind"] == "cplx":
        l = torch.arange((L + 1) ** 2, device=DEV, dtype=torch.float64).sqrt_().floor_()
        m = None
    else:
        l, m = _lm(L, case["mres"])
    q = torch.randn((nf, l.numel(), 2), generator=g, device=DEV, dtype=torch.float64)
    q /= (l + 1.0)[:, None]
    if m is not None:
        q[..., 1] *= (m > 0).to(q.dtype)
    q = torch.view_as_complex(q)
    return q.to(torch.complex64) if case["dtype"] == "f32" else q


def _grid_field(case, g):
    """A rough field on the grid: random waves with amplitudes falling as k^-1.5, every field."""
    nlat, nphi = case["nlat"], case["nphi"]
    parts = 2 if case["kind"] == "cplx" else 1
    ky = torch.fft.fftfreq(nlat, 1.0 / nlat, device=DEV, dtype=torch.float64)
    kx = torch.fft.rfftfreq(nphi, 1.0 / nphi, device=DEV, dtype=torch.float64)
    amp = (1.0 + ky[:, None] ** 2 + kx[None, :] ** 2) ** -0.75 * math.sqrt(nlat * nphi)
    out = torch.empty((case["nf"], parts, nlat, nphi), device=DEV, dtype=torch.float64)
    for f in range(case["nf"]):
        for p in range(parts):
            a = torch.randn((nlat, kx.numel(), 2), generator=g, device=DEV, dtype=torch.float64)
            out[f, p] = torch.fft.irfft2(torch.view_as_complex(a) * amp, s=(nlat, nphi))
    v = torch.complex(out[:, 0], out[:, 1]) if parts == 2 else out[:, 0]
    if case["layout"] == "theta":
        v = v.transpose(-1, -2)
    v = v.contiguous()
    return v.float() if case["dtype"] == "f32" else v


def _inputs(case, seed):
    g = _gen(seed)
    two = case["kind"] == "vector"
    if case["step"] == "analys":
        return tuple(_grid_field(case, g) for _ in range(2 if two else 1))
    q = tuple(_spectrum(case, g) for _ in range(2 if two else 1))
    if two:
        for x in q:
            x[:, 0] = 0.0   # a vector field has no degree 0
    if case["step"] == "grad":
        return q[0], _grid_field(case, g)
    return q


def prepare(case, seed):
    sh = shtns_amd.sht(case["lmax"], case["lmax"] // case["mres"], case["mres"])
    layout = shtns_amd.SHT_THETA_CONTIGUOUS if case["layout"] == "theta" else shtns_amd.SHT_PHI_CONTIGUOUS
    sh.set_grid(case["nlat"], case["nphi"], flags=layout | shtns_amd.sht_gauss, polar_opt=case["polar"])
    x = _inputs(case, seed)
    if case["step"] == "grad":
        x[0].requires_grad_(True)
    return {"sh": sh, "x": x, "kind": case["kind"], "step": case["step"], "ltr": case["ltr"] or -1}


def run(state):
    sh, x, step, ltr = state["sh"], state["x"], state["step"], state["ltr"]
    if step == "grad":
        v = autograd.synth(sh, x[0], ltr=ltr)
        loss = 0.5 * (v - x[1]).square().sum()
        (g,) = torch.autograd.grad(loss, x[0])
        return {"loss": loss.detach(), "field": v.detach(), "grad": g}
    if state["kind"] == "cplx":
        if step == "synth":
            return sh.synth_cplx(*x)
        if step == "analys":
            return sh.analys_cplx(*x)
        z = sh.synth_cplx(*x)
        return z, sh.analys_cplx(z)
    if step == "synth":
        return sh.synth(*x, ltr=ltr)
    if step == "analys":
        return sh.analys(*x, ltr=ltr)
    v = sh.synth(*x, ltr=ltr)
    return v, sh.analys(*(v if isinstance(v, tuple) else (v,)), ltr=ltr)


# ---- the same in plain torch, 64 bits ----------------------------------------------------
@functools.lru_cache(maxsize=2)
def _gauss(n):
    """cos(theta), sin(theta) and weights of the (n + 1) // 2 northern Gauss latitudes (Newton's
    method on the colatitude, long double)."""
    k = np.arange((n + 1) // 2, dtype=np.longdouble)
    pi = np.longdouble("3.14159265358979323846264338327950288")
    th = pi * (4 * k + 3) / (4 * n + 2)
    th = th + np.longdouble(n - 1) / (8 * np.longdouble(n) ** 3) / np.tan(th)
    for _ in range(4):
        x, s = np.cos(th), np.sin(th)
        p0, p1 = np.ones_like(x), x
        for l in range(2, n + 1):
            p0, p1 = p1, ((2 * l - 1) * x * p1 - (l - 1) * p0) / l
        d = n * (p0 - x * p1) / s          # -dP_n/dtheta
        th = th + p1 / d
    w = 2 / (d * d)
    if n % 2:
        x[-1] = 0
    return tuple(torch.from_numpy(np.asarray(a, dtype=np.float64)).to(DEV) for a in (x, np.sin(th), w))


def _legendre(L, mres, x, s):
    """Yields (l, P, Pm1, c) for l = 0 .. L: P[im, k] = P_lm(x_k) of the orders im*mres <= l
    (orthonormal, Condon-Shortley phase), Pm1 the same of degree l - 1 (zero where l = m), and
    c[im] = sqrt((2l+1)/(2l-1) (l^2 - m^2)).  Values carry a separate power of 2^256."""
    M = L // mres + 1
    m = torch.arange(M, device=DEV, dtype=torch.float64) * mres
    j = np.arange(1, M * mres, dtype=np.longdouble)   # log2 |a_mm sin^m|, long double
    lg = np.concatenate([np.zeros(1, np.longdouble), np.cumsum(np.log2((2 * j + 1) / (2 * j)))])[::mres]
    lg = (lg - np.log2(4 * np.longdouble("3.14159265358979323846264338327950288"))) / 2
    ld = lg[:, None] + np.arange(0, M * mres, mres, dtype=np.longdouble)[:, None] * np.log2(s.cpu().numpy().astype(np.longdouble))
    e = np.minimum(np.floor(ld / 256), 0)
    frac = torch.from_numpy((ld - 256 * e).astype(np.float64)).to(DEV)
    e = torch.from_numpy(e.astype(np.float64)).to(DEV)
    sign = 1.0 - 2.0 * torch.remainder(m, 2)
    cur = torch.zeros((M, x.numel()), device=DEV, dtype=torch.float64)
    old = torch.zeros_like(cur)
    first = sign[:, None] * torch.exp2(frac)
    one = torch.ones((), device=DEV, dtype=torch.float64)
    down = one * 2.0 ** -256
    for l in range(L + 1):
        n = l // mres + 1
        mm = m[:n]
        den = (l * l - mm * mm).clamp_(min=1.0)
        a = torch.sqrt((4.0 * l * l - 1) / den)
        b = torch.sqrt(((l - 1.0) ** 2 - mm * mm).clamp_(min=0.0) / (4.0 * (l - 1.0) ** 2 - 1)) if l else a
        new = a[:, None] * (x * cur[:n] - b[:, None] * old[:n]) if l else cur[:n].clone()
        if l % mres == 0:
            new[n - 1] = first[n - 1]
        big = new.abs() > 2.0 ** 128
        sc = torch.where(big & (e[:n] < 0), down, one)
        old[:n] = cur[:n] * sc
        cur[:n] = new * sc
        e[:n] += (sc != 1.0).to(e.dtype)
        f = torch.exp2(256 * e[:n].clamp(min=-4.0))
        yield l, cur[:n] * f, old[:n] * f, torch.sqrt((2.0 * l + 1) / max(2.0 * l - 1, 1.0) * (l * l - mm * mm))


def _rows(L, mres):
    """index[im] = place of degree 0 of order im in the spectral layout."""
    return torch.tensor([(im * (2 * L + 2 - (im + 1) * mres)) // 2 for im in range(L // mres + 1)], device=DEV)


def _to_grid(F, case):
    """Fourier rows F[f, im, lat] -> fields in the case's layout."""
    nphi = case["nphi"]
    X = torch.zeros((F.shape[0], F.shape[2], nphi // 2 + 1), device=DEV, dtype=torch.complex128)
    X[:, :, : F.shape[1]] = F.transpose(1, 2)
    v = torch.fft.irfft(X, n=nphi) * nphi
    return v.transpose(-1, -2).contiguous() if case["layout"] == "theta" else v


def _to_rows(v, case):
    """Fields -> unnormalised Fourier rows [f, im, lat], im <= mmax."""
    v = v.double()
    v = v.transpose(-1, -2) if case["layout"] == "theta" else v
    F = torch.fft.rfft(v)[..., : case["lmax"] // case["mres"] + 1]
    return F.transpose(1, 2).contiguous()


def _sum_up(case, A, nlat):
    """A[parity of l + m of the functions' even (0) and odd (1) parts][f, im, k] -> all rows."""
    N, S = A[0] + A[1], A[0] - A[1]
    return torch.cat([N, S.flip(-1)[..., nlat % 2:]], -1)


def _exact_synth(case, spectra):
    L, mres, nlat, ltr = case["lmax"], case["mres"], case["nlat"], case["ltr"] or case["lmax"]
    x, s, _ = _gauss(nlat)
    M, base = L // mres + 1, _rows(L, mres)
    vec = case["kind"] == "vector"
    nf = spectra[0].shape[0]
    A = [[torch.zeros((nf, M, x.numel()), device=DEV, dtype=torch.complex128) for _ in range(2)] for _ in spectra]
    odd = (torch.arange(M, device=DEV) * mres) % 2
    m = torch.arange(M, device=DEV, dtype=torch.float64) * mres
    for l, P, Pm1, c in _legendre(ltr, mres, x, s):
        n = P.shape[0]
        q = [z[:, base[:n] + l].to(torch.complex128) for z in spectra]
        for par in (0, 1):
            sel = torch.nonzero(odd[:n] == (l + par) % 2).flatten()   # rows with l + m of this parity
            if not sel.numel():
                continue
            if not vec:
                A[0][par][:, sel] += q[0][:, sel, None] * P[sel]
                continue
            Y = (1j * m[sel])[:, None] * (P[sel] / s)
            D = (l * x * P[sel] - c[sel, None] * Pm1[sel]) / s
            S, T = q[0][:, sel, None], q[1][:, sel, None]
            A[0][par][:, sel] += T * Y
            A[1][par][:, sel] += S * Y
            A[0][1 - par][:, sel] += S * D
            A[1][1 - par][:, sel] -= T * D
    out = []
    for a in A:
        F = _sum_up(case, a, nlat)
        F[:, 0].imag.zero_()
        out.append(_to_grid(F, case))
    return out


def _exact_analys(case, fields, adjoint=False):
    """adjoint: the transpose of the synthesis (unit weights, orders m > 0 twice)."""
    L, mres, nlat, ltr = case["lmax"], case["mres"], case["nlat"], case["ltr"] or case["lmax"]
    x, s, w = _gauss(nlat)
    K, M, base = x.numel(), L // mres + 1, _rows(L, mres)
    vec = case["kind"] == "vector"
    w = torch.ones_like(w) if adjoint else w * (2 * math.pi / case["nphi"])
    G = []
    for v in fields:
        F = _to_rows(v, case)
        N, S = F[..., :K] * w, F.flip(-1)[..., :K] * w
        if nlat % 2:
            N[..., -1] *= 0.5
            S[..., -1] *= 0.5
        G.append((N + S, N - S))
        del F, N, S
    nf = fields[0].shape[0]
    out = [torch.zeros((nf, _nlm(L, M - 1, mres)), device=DEV, dtype=torch.complex128) for _ in fields]
    odd = (torch.arange(M, device=DEV) * mres) % 2
    m = torch.arange(M, device=DEV, dtype=torch.float64) * mres
    for l, P, Pm1, c in _legendre(ltr, mres, x, s):
        n = P.shape[0]
        for par in (0, 1):
            sel = torch.nonzero(odd[:n] == (l + par) % 2).flatten()
            if not sel.numel():
                continue
            at = base[sel] + l
            if not vec:
                z = (G[0][par][:, sel] * P[sel]).sum(-1)
                if adjoint:
                    z *= torch.where(m[sel] > 0, 2.0, 1.0)
                out[0][:, at] = z
                continue
            if l == 0:
                continue
            Y = (-1j * m[sel])[:, None] * (P[sel] / s)
            D = (l * x * P[sel] - c[sel, None] * Pm1[sel]) / s
            vt, vp = G
            out[0][:, at] = ((vt[1 - par][:, sel] * D).sum(-1) + (vp[par][:, sel] * Y).sum(-1)) / (l * (l + 1.0))
            out[1][:, at] = ((vt[par][:, sel] * Y).sum(-1) - (vp[1 - par][:, sel] * D).sum(-1)) / (l * (l + 1.0))
    for z in out:
        z[:, : L + 1].imag.zero_()
    return out


def _cplx_order(L):
    """For every (l, m >= 0) of the real layout: places of (l, m) and (l, -m) in the complex one,
    and (-1)^m."""
    l, m = _lm(L, 1)
    return l * (l + 1) + m, l * (l + 1) - m, 1.0 - 2.0 * (m % 2).double()


def exact(case, seed):
    x = _inputs(case, seed)
    L = case["lmax"]
    if case["kind"] == "cplx":
        plus, minus, sg = _cplx_order(L)
        z = x[0]
        if case["step"] != "analys":
            a, b = x[0][:, plus], sg * x[0][:, minus]
            re, im = (a + b.conj()) / 2, (a - b.conj()) / 2j
            re[:, : L + 1] = a[:, : L + 1].real.to(re.dtype)
            im[:, : L + 1] = a[:, : L + 1].imag.to(im.dtype)
            both = _exact_synth(case, [torch.cat([re, im])])[0]
            z = torch.complex(*both.chunk(2))
            if case["step"] == "synth":
                return z
        re, im = _exact_analys(case, [torch.cat([z.real, z.imag])])[0].chunk(2)
        out = torch.empty((z.shape[0], (L + 1) ** 2), device=DEV, dtype=torch.complex128)
        out[:, minus] = sg * (re.conj() + 1j * im.conj())
        out[:, plus] = re + 1j * im
        return out if case["step"] == "analys" else (z, out)
    if case["step"] == "analys":
        out = _exact_analys(case, x)
        return out[0] if len(out) == 1 else tuple(out)
    if case["step"] == "grad":
        v = _exact_synth(case, x[:1])[0]
        d = v - x[1]
        return {"loss": 0.5 * d.square().sum(), "field": v, "grad": _exact_analys(case, [d], adjoint=True)[0]}
    v = _exact_synth(case, x)
    if case["step"] == "synth":
        return v[0] if len(v) == 1 else tuple(v)
    q = _exact_analys(case, v)
    return (v[0], q[0]) if len(v) == 1 else (tuple(v), tuple(q))
