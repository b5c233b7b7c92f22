"""GPU parity of the individual HIP kernels against the CPU oracle / numpy.

Each test calls the kernels through the C ABI (ctypes binding) on torch device
buffers and compares with the FP64 oracle restatement of the reference.
"""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    return torch


def test_gemm_f64_matches_numpy():
    """FP64 MFMA GEMM (also checks the 16x16x4 lane layout) against numpy."""
    torch = _torch()
    from magic_amd import _lib
    from magic_amd.device import ptr, stream_handle
    rng = np.random.default_rng(1)
    for (M, Nn, K, batch) in ((16, 64, 4, 1), (37, 91, 53, 3), (97, 291, 97, 2)):
        A = rng.standard_normal((batch, M, K))
        B = rng.standard_normal((batch, K, Nn))
        dA = torch.from_numpy(A).cuda()
        dB = torch.from_numpy(B).cuda()
        dC = torch.zeros(batch, M, Nn, dtype=torch.float64, device="cuda")
        g = _lib.GemmArgs()
        g.A, g.B, g.C = ptr(dA), ptr(dB), ptr(dC)
        g.sAr, g.sAc, g.sAb = K, 1, M * K
        g.sBr, g.sBc, g.sBb = Nn, 1, K * Nn
        g.sCr, g.sCc, g.sCb = Nn, 1, M * Nn
        g.M, g.Nn, g.K, g.batch, g.alpha = M, Nn, K, batch, 1.0
        _lib.call("mh_gemm_f64", _lib.ref(g), stream_handle())
        ref = A @ B
        err = np.abs(dC.cpu().numpy() - ref).max() / np.abs(ref).max()
        assert err < 1e-14, (M, Nn, K, err)


@pytest.mark.parametrize("l_max,minc", [(16, 1), (32, 1), (63, 1), (16, 2), (32, 4)])
def test_plm_tables_match_oracle(l_max, minc):
    """Device P_lm / dP_lm tables against the oracle's recurrence (plms.py);
    minc > 1: the tables of the orders m = 0, minc, ... in the run's lm order."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from oracle.params import Params as OP
    from oracle import horizontal
    p = Params({"l_max": l_max, "n_r_max": 9, "minc": minc})
    res = Resolution(p)
    op = OP({"l_max": l_max, "n_r_max": 9, "minc": minc})
    tab = horizontal.plm_tables(op)
    lay = res.lay
    info = lay["mp_info"].reshape(p.n_m, 2, 4)
    synP = res.synP.cpu().numpy()
    synD = res.synD.cpu().numpy()
    anaW = res.anaW.cpu().numpy()
    H, Hp = lay["H"], lay["Hp"]
    lm = 0
    worst = 0.0
    for mi in range(p.n_m):
        m = mi * minc
        for l in range(m, l_max + 1):
            par, k = (l - m) % 2, (l - m) // 2
            K, so, ao, K16 = info[mi, par]
            gP = synP[so + k * Hp: so + k * Hp + H]
            gD = synD[so + k * Hp: so + k * Hp + H]
            gW = anaW[ao + np.arange(H) * K16 + k]
            scale = max(np.abs(tab["Plm"][lm]).max(), 1e-300)
            worst = max(worst, np.abs(gP - tab["Plm"][lm]).max() / scale,
                        np.abs(gD - tab["dPlm"][lm]).max() / max(np.abs(tab["dPlm"][lm]).max(), 1e-300),
                        np.abs(gW - tab["wPlm"][lm]).max() / max(np.abs(tab["wPlm"][lm]).max(), 1e-300))
            lm += 1
    assert lm == p.lm_max
    assert worst < 1e-12, worst


def _oracle_sht(l_max, minc=1):
    from oracle.params import Params as OP
    from oracle.sht import SHT as OSHT
    return OSHT(OP({"l_max": l_max, "n_r_max": 9, "minc": minc}))


def _rand_spec(L, B, lmaps, seed):
    rng = np.random.default_rng(seed)
    l = lmaps["l"]
    x = (rng.standard_normal((L, B)) + 1j * rng.standard_normal((L, B))) / (l[:, None] + 1.0) ** 2
    x[lmaps["m"] == 0] = x[lmaps["m"] == 0].real
    return x


@pytest.mark.parametrize("l_max,B,minc", [(16, 1, 1), (16, 7, 1), (32, 33, 1), (64, 20, 1),
                                          (16, 7, 2), (12, 5, 3), (32, 9, 4)])
def test_sht_matches_oracle(l_max, B, minc):
    """scal_to_spat / scal_to_SH / torpol_to_spat / spat_to_sphertor vs the
    oracle; minc > 1: the orders m = 0, minc, ... on one 2 pi / minc sector."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    p = Params({"l_max": l_max, "n_r_max": 9, "minc": minc})
    res = Resolution(p)
    sht = SHT(res)
    osht = _oracle_sht(l_max, minc)
    L = p.lm_max
    S = _rand_spec(L, B, res.maps, 1)
    Q = _rand_spec(L, B, res.maps, 2)
    T = _rand_spec(L, B, res.maps, 3)
    dev = lambda a: torch.from_numpy(a).cuda()
    # scalar synthesis
    g = sht.scal_to_spat(dev(S)).cpu().numpy()
    go = osht.scal_to_spat(S)
    assert np.abs(g - go).max() / np.abs(go).max() < 1e-13
    # scalar analysis of the oracle grid
    s2 = sht.scal_to_SH(dev(go)).cpu().numpy()
    so = osht.scal_to_SH(go)
    assert np.abs(s2 - so).max() / np.abs(so).max() < 1e-13
    assert np.abs(s2 - S).max() / np.abs(S).max() < 1e-12   # round trip
    # vector synthesis
    br, bt, bp = (x.cpu().numpy() for x in sht.torpol_to_spat(dev(Q), dev(S), dev(T)))
    obr, obt, obp = osht.torpol_to_spat(Q, S, T)
    for a, b in ((br, obr), (bt, obt), (bp, obp)):
        assert np.abs(a - b).max() / np.abs(b).max() < 1e-13
    # vector analysis
    Sv, Tv = (x.cpu().numpy() for x in sht.spat_to_sphertor(dev(obt), dev(obp)))
    oS, oT = osht.spat_to_sphertor(obt, obp)
    assert np.abs(Sv - oS).max() / np.abs(oS).max() < 1e-12
    assert np.abs(Tv - oT).max() / np.abs(oT).max() < 1e-12


def test_sht_round_trip_lmax383():
    """Config-2 shapes (l_max=383, n_theta=576, n_phi=1152), reduced batch: round trip."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    p = Params({"l_max": 383, "n_r_max": 9})
    assert (p.n_theta, p.n_phi, p.lm_max) == (576, 1152, 73920)
    res = Resolution(p)
    sht = SHT(res)
    S = _rand_spec(p.lm_max, 6, res.maps, 5)
    dS = torch.from_numpy(S).cuda()
    back = sht.scal_to_SH(sht.scal_to_spat(dS)).cpu().numpy()
    assert np.abs(back - S).max() / np.abs(S).max() < 1e-11
    T = _rand_spec(p.lm_max, 6, res.maps, 6)
    T[0] = 0.0
    S[0] = 0.0
    Z = np.zeros_like(S)
    _, vt, vp = sht.torpol_to_spat(torch.from_numpy(Z).cuda(), torch.from_numpy(S).cuda(),
                                   torch.from_numpy(T).cuda())
    S2, T2 = (x.cpu().numpy() for x in sht.spat_to_sphertor(vt, vp))
    assert np.abs(S2 - S).max() / np.abs(S).max() < 1e-11
    assert np.abs(T2 - T).max() / np.abs(T).max() < 1e-11


@pytest.mark.parametrize("l_max", [63, 383])
def test_sht_mixed_precision_against_fp64(l_max):
    """FP32-MFMA Legendre transforms ("mixed") against the FP64 transforms on
    (l+1)^-2 spectra (the config-2 input law): each of the four transforms and
    the round trip stay within 1e-5 of the largest value (FP32 tables, inputs
    rounded to FP32, FP32 accumulation over at most l_max/2 degrees or n_theta/2
    nodes).  The FP64 transforms are pinned against the oracle above."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    p = Params({"l_max": l_max, "n_r_max": 9})
    res = Resolution(p)
    s64, s32 = SHT(res), SHT(res, precision="mixed")
    rel = lambda a, b: float((a - b).abs().max() / b.abs().max())
    S = torch.from_numpy(_rand_spec(p.lm_max, 5, res.maps, 7)).cuda()
    T = torch.from_numpy(_rand_spec(p.lm_max, 5, res.maps, 8)).cuda()
    Q = torch.from_numpy(_rand_spec(p.lm_max, 5, res.maps, 9)).cuda()
    g64 = s64.scal_to_spat(S)
    assert rel(s32.scal_to_spat(S), g64) < 1e-5
    assert rel(s32.scal_to_SH(g64), s64.scal_to_SH(g64)) < 1e-5
    v64 = s64.torpol_to_spat(Q, S, T)
    for a, b in zip(s32.torpol_to_spat(Q, S, T), v64):
        assert rel(a, b) < 1e-5
    for a, b in zip(s32.spat_to_sphertor(v64[1], v64[2]), s64.spat_to_sphertor(v64[1], v64[2])):
        assert rel(a, b) < 1e-5
    assert rel(s32.scal_to_SH(s32.scal_to_spat(S)), S) < 1e-5


@pytest.mark.parametrize("l_max,precision,tol", [(63, "mixed_bf16", 1e-4), (63, "mixed_bf16x3", 1e-5),
                                                  (383, "mixed_bf16", 1e-4), (383, "mixed_bf16x3", 1e-5)])
def test_sht_bf16_split_against_fp64(l_max, precision, tol):
    """BF16 split-precision Legendre transforms (tables and inputs as two or
    three bf16 planes, the plane products i + j < planes on the BF16 MFMA, FP32
    accumulation) against the FP64 transforms on (l+1)^-2 spectra: every
    transform, both directions, scalar and vector, within `tol` of the largest
    value.  Two planes keep about 16 significant bits per operand (dropped
    products below 2^-16 relative), three about 24 (FP32 inputs)."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    p = Params({"l_max": l_max, "n_r_max": 9})
    res = Resolution(p)
    s64, sbf = SHT(res), SHT(res, precision=precision)
    rel = lambda a, b: float((a - b).abs().max() / b.abs().max())
    S = torch.from_numpy(_rand_spec(p.lm_max, 5, res.maps, 7)).cuda()
    T = torch.from_numpy(_rand_spec(p.lm_max, 5, res.maps, 8)).cuda()
    Q = torch.from_numpy(_rand_spec(p.lm_max, 5, res.maps, 9)).cuda()
    g64 = s64.scal_to_spat(S)
    errs = [rel(sbf.scal_to_spat(S), g64), rel(sbf.scal_to_SH(g64), s64.scal_to_SH(g64))]
    v64 = s64.torpol_to_spat(Q, S, T)
    errs += [rel(a, b) for a, b in zip(sbf.torpol_to_spat(Q, S, T), v64)]
    errs += [rel(a, b) for a, b in zip(sbf.spat_to_sphertor(v64[1], v64[2]),
                                       s64.spat_to_sphertor(v64[1], v64[2]))]
    errs.append(rel(sbf.scal_to_SH(sbf.scal_to_spat(S)), S))
    print(f"bf16 split {precision} l_max={l_max}: max errors {['%.1e' % e for e in errs]}")
    assert max(errs) < tol, errs
    # the split is doing its work: an error far below one bf16 rounding (2^-9)
    assert max(errs) < 2.0 ** -12


@pytest.mark.parametrize("n", [5, 97, 112, 113, 194, 208, 230])
def test_gj_inverse_matches_numpy(n):
    """Batched equilibrated Gauss-Jordan inverse (register-resident for n <= 208,
    global-memory kernel above) against numpy.linalg.inv, for every
    equilibration mode, on badly scaled random matrices; the batch is done in
    place (A and out alias), as the operator rebuild calls it."""
    torch = _torch()
    from magic_amd import _lib
    from magic_amd.device import ptr, stream_handle
    rng = np.random.default_rng(n)
    batch = 3
    A = rng.standard_normal((batch, n, n)) + n * np.eye(n) * (rng.random((batch, 1, 1)) > 0.5)
    A *= np.exp(rng.uniform(-6, 6, (batch, n, 1)))  # row scales
    A *= np.exp(rng.uniform(-3, 3, (batch, 1, n)))  # column scales
    ref = np.linalg.inv(A)
    for precond in (0, 1, 2):
        d = torch.from_numpy(A.copy()).cuda()
        work = torch.empty(batch * 2 * n * n, dtype=torch.float64, device="cuda")
        scal = torch.empty(batch * 2 * n, dtype=torch.float64, device="cuda")
        info = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
        _lib.call("mh_gj_inverse", ptr(d), ptr(d), ptr(work), ptr(scal), n, batch, precond,
                  ptr(info), None, stream_handle())
        got = d.cpu().numpy()
        assert np.all(info.cpu().numpy() == 0)
        for b in range(batch):
            cond = np.linalg.cond(A[b])
            res = np.abs(got[b] @ A[b] - np.eye(n)).max()
            assert res < 1e-14 * cond * n, (n, precond, b, res, cond)
            err = np.abs(got[b] - ref[b]).max() / np.abs(ref[b]).max()
            assert err < 1e-15 * cond * n, (n, precond, b, err, cond)


def test_gj_inverse_reports_singular_pivot():
    """A matrix with a zero column reports the first zero pivot (1-based)."""
    torch = _torch()
    from magic_amd import _lib
    from magic_amd.device import ptr, stream_handle
    for n in (9, 150):
        A = np.random.default_rng(3).standard_normal((1, n, n))
        A[0, :, 0] = 0.0
        d = torch.from_numpy(A).cuda()
        work = torch.empty(2 * n * n, dtype=torch.float64, device="cuda")
        scal = torch.empty(2 * n, dtype=torch.float64, device="cuda")
        info = torch.zeros(1, dtype=torch.int32, device="cuda")
        _lib.call("mh_gj_inverse", ptr(d), ptr(d), ptr(work), ptr(scal), n, 1, 1, ptr(info),
                  None, stream_handle())
        assert int(info.cpu()[0]) == 1


def test_sht_round_trip_config2_full_batch():
    """Config 2 at its full batch: 3 fields x 97 radial levels = 291 columns at
    l_max=383 (n_theta=576, n_phi=1152), coefficients ~ N(0,1) (l+1)^-2.  Scalar
    and vector round trips in FP64 return the input to 1e-11 of its largest
    coefficient; the mixed-precision (FP32 MFMA) transforms stay within 1e-5
    of the FP64 ones, both for the grid values and after the round trip."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    p = Params({"l_max": 383, "n_r_max": 9})
    res = Resolution(p)
    f64, mix = SHT(res), SHT(res, "mixed")
    B = 291
    S = torch.from_numpy(_rand_spec(p.lm_max, B, res.maps, 21)).cuda()
    S[0] = 0.0
    g64 = f64.scal_to_spat(S)
    gmx = mix.scal_to_spat(S)
    assert tuple(g64.shape) == (B, 576, 1152)
    gs = g64.abs().max()
    assert float((gmx - g64).abs().max() / gs) < 1e-5
    back = f64.scal_to_SH(g64)
    ss = S.abs().max()
    assert float((back - S).abs().max() / ss) < 1e-11
    back_mx = mix.scal_to_SH(gmx)
    assert float((back_mx - back).abs().max() / ss) < 1e-5
    del g64, gmx, back, back_mx
    T = torch.from_numpy(_rand_spec(p.lm_max, B, res.maps, 22)).cuda()
    T[0] = 0.0
    Z = torch.zeros_like(S)
    _, vt, vp = f64.torpol_to_spat(Z, S, T)
    S2, T2 = f64.spat_to_sphertor(vt, vp)
    assert float((S2 - S).abs().max() / ss) < 1e-11
    assert float((T2 - T).abs().max() / T.abs().max()) < 1e-11
    _, vtm, vpm = mix.torpol_to_spat(Z, S, T)
    assert float((vtm - vt).abs().max() / vt.abs().max()) < 1e-5
    S3, T3 = mix.spat_to_sphertor(vtm, vpm)
    assert float((S3 - S2).abs().max() / ss) < 1e-5
    assert float((T3 - T2).abs().max() / T.abs().max()) < 1e-5


@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed_bf16x3"])
def test_sht_batch_wider_than_the_radial_grid(precision):
    """A transform of more columns than the resolution has radial levels reads no
    radial profile: each column equals its transform alone."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    res = Resolution(Params({"l_max": 16, "n_r_max": 9}))
    sht = SHT(res, precision)
    rng = np.random.default_rng(4)
    x = [torch.from_numpy(rng.standard_normal((res.L, 40)) + 0j).cuda() for _ in range(3)]
    wide = sht.torpol_to_spat(*x)
    for c in (0, 9, 39):
        one = sht.torpol_to_spat(*[v[:, c].contiguous() for v in x])
        assert all(torch.equal(a[c], b) for a, b in zip(wide, one))


@pytest.mark.parametrize("l_max,B,minc", [(126, 25, 1), (20, 8, 1), (48, 9, 2)])
def test_fp64_transforms_at_tile_edges(l_max, B, minc):
    """FP64 vector and scalar transforms where the work split has edges: orders
    with one and with two analysis windows (l_max = 126: 121 or 122 degrees at m =
    6 and 5), an odd number of theta tiles, column counts at and past a tile of 8
    and 24; against the oracle to rounding (sums of up to l_max terms)."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    res = Resolution(Params({"l_max": l_max, "n_r_max": 9, "minc": minc}))
    sht, osht = SHT(res), _oracle_sht(l_max, minc)
    Q, S, T = (_rand_spec(res.L, B, res.maps, k) for k in (1, 2, 3))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    tol = 4 * l_max * np.finfo(float).eps
    grids = osht.torpol_to_spat(Q, S, T)
    for a, b in zip(sht.torpol_to_spat(dev(Q), dev(S), dev(T)), grids):
        assert np.abs(a.cpu().numpy() - b).max() < tol * np.abs(b).max()
    sc = osht.scal_to_spat(Q)
    assert np.abs(sht.scal_to_spat(dev(Q)).cpu().numpy() - sc).max() < tol * np.abs(sc).max()
    back = osht.scal_to_SH(sc)
    assert np.abs(sht.scal_to_SH(dev(sc)).cpu().numpy() - back).max() < tol * np.abs(back).max()
    for a, b in zip(sht.spat_to_sphertor(dev(grids[1]), dev(grids[2])),
                    osht.spat_to_sphertor(grids[1], grids[2])):
        assert np.abs(a.cpu().numpy() - b).max() < tol * np.abs(b).max()


@pytest.mark.parametrize("l_max,B", [(16, 1500), (27, 20), (31, 300), (48, 520), (85, 300), (91, 210),
                                     (127, 200), (200, 41), (341, 40)])
def test_fp64_work_splits_give_identical_results(l_max, B):
    """The FP64 Legendre kernels choose their work split by sizes and batch: one or
    three column tiles of the scalar synthesis (three from B > 16 where the launch is
    large, as at these B), one to three theta tiles a wave (l_max 16, 48, 127), and the
    analysis of few columns or low degrees (two windows from l_max = 31, four from 91).
    Every column of a large batch equals the column in a small one bit for bit."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    res = Resolution(Params({"l_max": l_max, "n_r_max": 9}))
    sht = SHT(res)
    gen = torch.Generator(device="cuda").manual_seed(l_max)
    x = [torch.randn(res.L, B, dtype=torch.complex128, device="cuda", generator=gen) for _ in range(3)]
    g = [torch.randn(B, res.T, res.P, dtype=torch.float64, device="cuda", generator=gen)
         for _ in range(2)]
    big = (sht.scal_to_spat(x[0]), *sht.torpol_to_spat(*x))
    ana = (sht.scal_to_SH(g[0]), *sht.spat_to_sphertor(*g))
    for c in (slice(0, 1), slice(3, 11), slice(B - 9, B), slice(0, 16), slice(B - 17, B)):
        y = [v[:, c].contiguous() for v in x]
        part = (sht.scal_to_spat(y[0]), *sht.torpol_to_spat(*y))
        assert all(torch.equal(a[c], b) for a, b in zip(big, part)), c
        h = [v[c].contiguous() for v in g]
        part = (sht.scal_to_SH(h[0]), *sht.spat_to_sphertor(*h))
        assert all(torch.equal(a[:, c], b) for a, b in zip(ana, part)), c
    # outputs inside wider rows: the columns around them stay as they were
    F = res.fourier_buffer(4, 7).normal_()
    for N in (9, 16):
        out = [torch.full((res.L, N), 5.0, dtype=torch.complex128, device="cuda") for _ in range(3)]
        p = [o.data_ptr() + 16 for o in out]
        res.analysis(F, 7, 7, [(0, 1)], p[:1], p[1:2], N, vector=True)
        res.analysis(F, 7, 7, [2], p[2:], [None], N, vector=False)
        for o in out:
            assert (o[:, 0] == 5.0).all() and (o[:, 8:] == 5.0).all() and (o[:, 1:8] != 5.0).all()


def _long_double_vector_sums(th, l_max, S, T, ft, fp):
    """In long double, from the same nodes: the Fourier rows (M, T, B) of the vector
    synthesis of S and T, and S, T of the vector analysis of the Fourier rows ft, fp
    (weighted by 1/sin^2), by the products with P and sin(theta) dP (the recurrence of the
    tables)."""
    LD = np.longdouble
    c, s, w = (np.asarray(th[k], dtype=LD) for k in ("cos_n", "sin_n", "w_n"))
    H, M = c.size, l_max + 1
    rows = np.zeros((2, M, 2 * H, S.shape[1]), np.clongdouble)
    sol = np.zeros((2, *S.shape), np.clongdouble)
    r = lambda a, b: np.sqrt(LD(a) / LD(b))
    start = 0
    for m in range(M):
        n = l_max + 1 - m
        pi = LD("3.14159265358979323846264338327950288")
        p0, pm1 = np.sqrt(LD(0.25) / pi) * np.ones(H, LD), np.zeros(H, LD)
        for q in range(1, m + 1):
            p0 = p0 * s * r(2 * q + 1, 2 * q)
        P, D = np.zeros((n, H), LD), np.zeros((n, H), LD)
        for i in range(n):
            l = m + i
            up, dn = r((l + 1 - m) * (l + 1 + m), (2 * l + 1) * (2 * l + 3)), \
                r((l - m) * (l + m), (2 * l - 1) * (2 * l + 1)) if l > m else LD(0)
            p1 = (c * p0 - dn * pm1) / up
            P[i], D[i] = p0, l * up * p1 - (l + 1) * dn * pm1
            pm1, p0 = p0, p1
        sl = slice(start, start + n)
        start += n
        for e in (0, 1):        # parity of l - m: P keeps it across the equator, dP flips it
            a, b = S[sl][e::2], T[sl][e::2]
            q, d = P[e::2].T, D[e::2].T
            pt, dt = 1j * m * (q @ b), d @ a
            pp, dp = 1j * m * (q @ a), -(d @ b)
            sg = 1 - 2 * e
            rows[0, m, 0::2] += pt + dt
            rows[0, m, 1::2] += sg * pt - sg * dt
            rows[1, m, 0::2] += pp + dp
            rows[1, m, 1::2] += sg * pp - sg * dp
            fold = lambda f, g: (2 * pi * w)[:, None] * (f[m, 0::2] + g * f[m, 1::2])
            l = np.arange(m, l_max + 1)[e::2].astype(LD)
            inv = np.where(l > 0, 1 / np.maximum(l * (l + 1), 1), 0)[:, None]
            sol[0, sl][e::2] = inv * (d.T @ fold(ft, -sg) - 1j * m * (q.T @ fold(fp, sg)))
            sol[1, sl][e::2] = inv * (-(d.T @ fold(fp, -sg)) - 1j * m * (q.T @ fold(ft, sg)))
    return rows, sol


@pytest.mark.parametrize("l_max", [33, 85])
def test_fp64_vector_transforms_row_by_row(l_max):
    """The FP64 vector transforms combine neighbouring degrees where the oracle multiplies
    by sin(theta) dP; a cancellation in that would show in single latitudes near the
    poles or single degrees, not in the largest value.  Errors against long double sums:
    every latitude (synthesis) and every degree (analysis) within 6 times the oracle's
    of that row, or of a few roundings of the row's largest value (both come from the
    rounding of the tables, largest of a few hundred values a row; the ratio is below 3)."""
    import scipy.fft
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    res = Resolution(Params({"l_max": l_max, "n_r_max": 9}))
    sht, osht = SHT(res), _oracle_sht(l_max)
    S, T = (_rand_spec(res.L, 3, res.maps, k) for k in (21, 22))
    S[0] = T[0] = 0.0
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    four = lambda g: scipy.fft.rfft(np.asarray(g, np.longdouble), axis=2, norm="forward")[
        :, :, :res.M].transpose(2, 1, 0)
    _, ot, op = osht.torpol_to_spat(0 * S, S, T)
    gpu = [x.cpu().numpy() for x in sht.torpol_to_spat(dev(0 * S), dev(S), dev(T))[1:]]
    ost2 = (1 / np.asarray(res.th["sin_grid"], np.longdouble) ** 2)[None, :, None]
    rows, sol = _long_double_vector_sums(res.th, l_max, S, T, four(ot) * ost2, four(op) * ost2)
    eps = np.finfo(float).eps
    for a, b, ref in zip(gpu, (ot, op), rows):
        err = [np.abs(four(g) - ref).max(axis=(0, 2)) for g in (a, b)]
        bound = 6 * np.maximum(err[1], 4 * eps * np.abs(ref).max(axis=(0, 2)))
        print("synthesis", l_max, float((err[0] / np.maximum(err[1], bound / 6)).max()))
        assert (err[0] <= bound).all(), (err[0] / bound).max()
    l = res.maps["l"]
    by_l = lambda x: np.array([np.abs(x[l == k]).max() for k in range(1, l_max + 1)])
    for a, b, ref in zip(sht.spat_to_sphertor(dev(ot), dev(op)), osht.spat_to_sphertor(ot, op), sol):
        err = [by_l(v - ref) for v in (a.cpu().numpy(), b)]
        bound = 6 * np.maximum(err[1], 4 * eps * by_l(ref))
        print("analysis", l_max, float((err[0] / np.maximum(err[1], bound / 6)).max()))
        assert (err[0] <= bound).all(), (err[0] / bound).max()


def test_fp64_resolution_holds_no_derivative_tables():
    """FP64 transforms read the P_lm tables alone, so a resolution keeps the other two
    only as the FP32 and BF16 copies of a mixed run."""
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    res = Resolution(Params({"l_max": 42, "n_r_max": 9}))
    big = [k for k, v in vars(res).items() if getattr(v, "nbytes", 0) >= res.anaW.nbytes // 2]
    assert sorted(big) == ["anaW", "synP"], big
    synD, anaWd = res.derivative_tables()
    t = res.f32_tables()
    assert (t["synD"] == synD.float()).all() and (t["anaWd"] == anaWd.float()).all()
    assert not {"synD", "anaWd"} & set(vars(res))


def test_fp64_legendre_rows_past_32_bit_offsets():
    """The last 9 columns of arrays whose orders span more than 2^31 bytes (l_max = 4, 40
    and 22.5 million columns, 10 GB each) transform as they do alone, bit for bit:
    scalar, and vector with every input mode."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    res = Resolution(Params({"l_max": 4, "n_r_max": 9}))
    B = 9
    gen = torch.Generator(device="cuda").manual_seed(1)
    ld = 40_000_000
    wide = torch.empty(res.L, ld, dtype=torch.complex128, device="cuda")
    x = torch.randn(res.L, B, dtype=torch.complex128, device="cuda", generator=gen)
    v = wide[:, ld - B:]
    v.copy_(x)
    outs = []
    for y, ldx in ((v, ld), (x, B)):
        Fs, Fv = res.fourier_buffer(1, B).fill_(7.0), res.fourier_buffer(3, 2 * B).fill_(7.0)
        res.synth([[(y, None, 0)]], B, ldx, Fs, B, vector=False)
        res.synth([[(y, None, 1), (y, None, 0), (y, y, 2)], [(y, None, 0)] * 3], B, ldx, Fv, 2 * B,
                  vector=True)
        outs.append((Fs, Fv))
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    del wide, v
    torch.cuda.empty_cache()
    n = 22_500_000
    wide = torch.empty(res.M * res.T, n, 2, dtype=torch.float64, device="cuda")
    F = torch.randn(res.M * res.T, B, 2, dtype=torch.float64, device="cuda", generator=gen)
    wide[:, n - B:].copy_(F)
    outs = []
    for G, Bin in ((wide[:, n - B:], n), (F, B)):
        o = [torch.full((res.L, B), 7.0, dtype=torch.complex128, device="cuda") for _ in range(3)]
        res.analysis(G, Bin, B, [0], o[:1], [None], B, vector=False)
        res.analysis(G, Bin, B, [(0, 0)], o[1:2], o[2:], B, vector=True)
        outs.append(o)
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    del wide, G
    torch.cuda.empty_cache()


@pytest.mark.parametrize("Mh", [2, 3, 5, 12, 24, 30, 45, 48, 54, 64, 72, 81, 90, 96, 100, 128, 150, 192,
                                225, 288, 300, 384, 400, 500, 576, 648, 720, 768, 800, 1000])
def test_fft_lengths_match_numpy(Mh):
    """mh_fft both ways for compiled, run-time, short and long (> 768) plans (the
    workgroup's passes below 50, and with a factor 5 below 100), odd and even half
    lengths, batches that do not fill a workgroup's rows, orders up to Mh; error of a
    few roundings per pass against numpy."""
    torch = _torch()
    from magic_amd import _lib, grid
    from magic_amd.device import ptr, stream_handle
    rng = np.random.default_rng(Mh)
    T, n = 2, 2 * Mh
    up = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    k = np.arange(Mh)
    tw, tw2 = np.exp(-2j * np.pi * k / Mh), np.exp(-2j * np.pi * k / n)
    dtw, dtw2 = up(tw.view(np.float64)), up(tw2.view(np.float64))
    ost2 = up(np.array([2.0, 3.0]))
    scale = torch.tensor([0, 1], dtype=torch.int32, device="cuda")
    for B, M in ((1, max(1, Mh // 3)), (9, Mh), (35, max(1, 2 * Mh // 3))):
        F = rng.standard_normal((2, M, T, B)) + 1j * rng.standard_normal((2, M, T, B))
        F[:, 0] = F[:, 0].real
        full = np.zeros((2, Mh + 1, T, B), complex)
        full[:, :M] = F
        g = np.fft.irfft(full, n=n, axis=1, norm="forward").transpose(0, 3, 2, 1)  # (2, B, T, n)
        dF, dG = up(F), torch.full((2, B, T, n), 7.0, dtype=torch.float64, device="cuda")
        a = _lib.FftArgs()
        rad = grid.fft_radices(Mh)
        a.Mh, a.nstage, a.n_m, a.T, a.B, a.ncomp, a.RB = Mh, len(rad), M, T, B, 2, 1
        for i, r in enumerate(rad):
            a.radix[i] = r
        a.tw, a.tw2, a.ost2 = ptr(dtw), ptr(dtw2), ptr(ost2)
        a.F, a.Fm_stride, a.Fc_stride, a.FB = ptr(dF), 2 * T * B, 2 * T * B * M, B
        a.G, a.Gc_stride = ptr(dG), B * T * n
        tol = 8 * np.finfo(float).eps * np.log2(n)
        _lib.call("mh_fft", 0, _lib.ref(a), stream_handle())
        out = dG.cpu().numpy()
        assert np.abs(out - g).max() < tol * np.abs(g).max(), (B, M)
        G = rng.standard_normal((2, B, T, n))
        H = np.fft.rfft(G, axis=3, norm="forward").transpose(0, 3, 2, 1)[:, :M].copy()
        H[1] *= np.array([2.0, 3.0])[None, :, None]
        dG.copy_(torch.from_numpy(G))
        a.comp_scale = ptr(scale)
        _lib.call("mh_fft", 1, _lib.ref(a), stream_handle())
        assert np.abs(dF.cpu().numpy() - H).max() < tol * np.abs(H).max(), (B, M)


def test_sphertor_inputs_of_any_layout():
    """spat_to_sphertor reads the grids in place: a strided view, a view that does
    not start on 16 bytes and one phi field for a batch of theta fields give the
    results of plain copies."""
    torch = _torch()
    from magic_amd.params import Params
    from magic_amd.device import Resolution
    from magic_amd.sht import SHT
    res = Resolution(Params({"l_max": 16, "n_r_max": 9}))
    sht = SHT(res)
    T, P = res.T, res.P
    base = torch.randn(3 * T * P + 1, dtype=torch.float64, device="cuda")
    vt = base[1:].view(3, T, P)
    vp = torch.randn(P, 3, T, dtype=torch.float64, device="cuda").permute(1, 2, 0)
    ref = sht.spat_to_sphertor(vt.clone(), vp.contiguous().clone())
    assert all(torch.equal(a, b) for a, b in zip(sht.spat_to_sphertor(vt, vp), ref))
    one = sht.spat_to_sphertor(vt, vp[:1])
    full = sht.spat_to_sphertor(vt, vp[:1].expand(3, T, P).contiguous())
    assert all(torch.equal(a, b) for a, b in zip(one, full))
