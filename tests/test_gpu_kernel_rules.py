"""GPU: the kernels that the dispatch rules choose by size, at the edges of their ranges, against
the CPU oracle (FP64, rel-L2 <= 1e-12; where single-precision arrays or contractions take part,
2e-6: 6e-8 of rounding per value, summed over at most 800 latitudes or 150 degrees in FP32).

Latitude tiles hold 64 north-south pairs, so nlat sets the tile count at any degree."""
import numpy as np
import pytest

import shtns_amd
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
TOL, TOL_F32 = 1e-12, 2e-6


def rel_l2(a, b):
    return float(np.linalg.norm((np.asarray(a) - b).ravel()) / np.linalg.norm(np.asarray(b).ravel()))


def make(lmax, nlat, nphi, mmax=None, mres=1, phi=False):
    mmax = lmax // mres if mmax is None else mmax
    layout = shtns_amd.SHT_PHI_CONTIGUOUS if phi else shtns_amd.SHT_THETA_CONTIGUOUS
    s = shtns_amd.sht(lmax, mmax, mres)
    s.set_grid(nlat, nphi, flags=layout | shtns_amd.sht_gauss, polar_opt=0.0)
    o = Oracle(lmax, mmax, mres, nlat, nphi)
    return s, o


def spectra(s, nf, mres=1, seed=0):
    """nf spectra with 1/(l+1) decay, real at m = 0"""
    rng = np.random.default_rng(seed)
    q = (rng.standard_normal((nf, s.nlm)) + 1j * rng.standard_normal((nf, s.nlm))) / (s.l + 1.0)
    q[:, s.m == 0] = q[:, s.m == 0].real
    return q


def run(f, *a, **k):
    import torch
    r = f(*[torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in a], **k)
    return [x.cpu().numpy() for x in r] if isinstance(r, tuple) else r.cpu().numpy()


# one to three fields: 64 steps per coefficient chunk (lmax 127 / 128: one full, one step over),
# one and two tiles per wave (12 / 13 tiles), full and single-lane last tiles, the middle row of
# odd grids, orders that a truncation empties, m = 0 mod mres
@pytest.mark.parametrize("lmax,nlat,nphi,mres,ltr", [
    (2, 3, 8, 1, -1), (16, 128, 36, 1, -1), (127, 130, 256, 1, -1), (128, 131, 270, 1, 127), (40, 1024, 84, 1, -1),
    (40, 1026, 84, 1, 17), (30, 1536, 64, 1, -1), (140, 1537, 288, 1, 131), (60, 1666, 64, 2, -1), (150, 3073, 64, 5, 1)])
def test_few_field_synthesis(lmax, nlat, nphi, mres, ltr, device):
    s, o = make(lmax, nlat, nphi, mres=mres)
    q = spectra(s, 3, mres, seed=nlat)
    ref = np.stack([o.synth(q[f], ltr) for f in range(3)])
    for nf in (1, 2, 3):
        v = run(s.synth, q[:nf], ltr=ltr)
        assert rel_l2(v, ref[:nf]) <= TOL, nf
    q[:, s.l == 0] = 0
    vt, vp = run(s.synth, q[0], q[1], ltr=ltr)
    rt, rp = o.synth_sphtor(q[0], q[1], ltr)
    assert rel_l2(vt, rt) <= TOL and rel_l2(vp, rp) <= TOL


# every block shape of the shared analysis and of the matrix synthesis: tile counts 1 to 13 (13
# and 25 in parts that add up), one to four groups of four fields, remainders of 16-field shapes
@pytest.mark.parametrize("prec", [shtns_amd.SHT_PREC_AUTO, shtns_amd.SHT_PREC_F32, shtns_amd.SHT_PREC_SPLIT])
@pytest.mark.parametrize("tiles", [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 25])
def test_shapes_by_tiles_and_fields(tiles, prec, device):
    lmax, nlat = 37, 128 * tiles - (37 if tiles % 2 else 0)   # odd grids, partly empty last tiles
    s, o = make(lmax, nlat, 80)
    s.set_precision(prec)
    tol = TOL if prec == shtns_amd.SHT_PREC_AUTO else TOL_F32
    q = spectra(s, 24, seed=tiles)
    v = np.stack([o.synth(x) for x in q])
    for nf in (3, 4, 5, 9, 16, 17, 24):
        assert rel_l2(run(s.synth, q[:nf]), v[:nf]) <= tol, nf
        back = run(s.analys, v[:nf])
        errs = [rel_l2(back[f], q[f]) for f in range(nf)]   # band-limited: the analysis inverts
        assert max(errs) <= tol, (nf, errs)
    if prec == shtns_amd.SHT_PREC_AUTO:
        w = np.random.default_rng(tiles).standard_normal((6, 80, nlat))   # unfiltered
        got, gotv = run(s.analys, w, ltr=30), run(s.analys, w[:3], w[3:])
        for f in range(6):
            assert rel_l2(got[f], o.analys(w[f], 30)) <= TOL
        for f in range(3):
            for x, r in zip(gotv, o.analys_sphtor(w[f], w[3 + f])):
                assert rel_l2(x[f], r) <= TOL


# longitude FFTs: half-lengths of every radix of the runtime plan (2 to 10, 12, 15, 16), of the
# register and the split-exchange kernels (24 to 1536) and beyond, both layouts, few fields
# (small blocks) and many
@pytest.mark.parametrize("phi", [False, True])
@pytest.mark.parametrize("half", [9, 14, 21, 25, 35, 45, 49, 60, 81, 96, 105, 135, 192, 225, 240, 256, 343, 384, 441, 625,
                                  640, 1080, 1536, 1600, 2187, 3072])
def test_longitude_fft(half, phi, device):
    lmax, nlat = 8, 19
    s, o = make(lmax, nlat, 2 * half, phi=phi)
    rng = np.random.default_rng(half)
    for nf in (1, 150):
        q = spectra(s, nf, seed=half)
        w = rng.standard_normal((nf, 2 * half, nlat))
        sw = (lambda a: np.swapaxes(a, -1, -2)) if phi else (lambda a: a)
        pick = sorted({0, nf // 2, nf - 1})
        v, a = sw(run(s.synth, q)), run(s.analys, sw(w))
        v4, a4 = sw(run(s.synth, q.astype(np.complex64))), run(s.analys, sw(w).astype(np.float32))
        for f in pick:
            ref, refa = o.synth(q[f]), o.analys(w[f])
            assert rel_l2(v[f], ref) <= TOL and rel_l2(a[f], refa) <= TOL, (nf, f)
            assert rel_l2(v4[f], ref) <= TOL_F32 and rel_l2(a4[f], refa) <= TOL_F32, (nf, f)


@pytest.mark.parametrize("nphi", [42, 70, 90, 98, 162, 192, 210, 360, 768, 1280])
def test_complex_fields_at_general_lengths(nphi, device):
    lmax, nlat = 12, 20
    s, o = make(lmax, nlat, nphi)
    rng = np.random.default_rng(nphi)
    alm = rng.standard_normal((2, o.nlm_cplx)) + 1j * rng.standard_normal((2, o.nlm_cplx))
    z = run(s.synth_cplx, alm)
    back = run(s.analys_cplx, z)
    for f in range(2):
        assert rel_l2(z[f], o.synth_cplx(alm[f])) <= TOL and rel_l2(back[f], alm[f]) <= TOL


@pytest.mark.parametrize("lmax,nlat,nphi", [(63, 96, 192), (100, 131, 210), (150, 1026, 320)])
def test_float_data_of_few_fields_in_fp64(lmax, nlat, nphi, device):
    """No precision chosen: the error of one to three (synthesis) and one (analysis) fields is
    the FP32 rounding of the arrays, 6e-8; beyond, and where FP32 is chosen, the FP32 contraction's."""
    s, o = make(lmax, nlat, nphi)
    q = spectra(s, 4, seed=lmax).astype(np.complex64)
    v = np.stack([o.synth(x.astype(np.complex128)) for x in q])
    v4 = v.astype(np.float32)
    for nf in (1, 2, 3, 4):
        assert rel_l2(run(s.synth, q[:nf]), v[:nf]) <= (1e-7 if nf <= 3 else TOL_F32), nf
        ref = np.stack([o.analys(x.astype(np.float64)) for x in v4[:nf]])
        assert rel_l2(run(s.analys, v4[:nf]), ref) <= (1e-7 if nf == 1 else TOL_F32), nf
    s.set_precision(shtns_amd.SHT_PREC_F32)
    assert rel_l2(run(s.synth, q[:1]), v[:1]) <= TOL_F32
