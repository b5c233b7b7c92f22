"""GPU parity of the full CNAB2 dynamo step against the reference trajectory.

The golden fixtures (``tests/golden/traj_*.npz``) were written by running the
reference's own ``step_time.one_step`` on the CPU (``make_golden.py``); the
oracle reproduces them to ~1e-13.  The bar (north star): spectral
coefficients within 1e-10 relative and energies within 1e-9 relative.
"""

import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _load(name):
    with open(os.path.join(GOLD, f"traj_{name}.json")) as f:
        case = json.load(f)
    return case, np.load(os.path.join(GOLD, f"traj_{name}.npz"))


def _run(case, fused=True, precision="fp64"):
    from magic_amd.dynamo import DynamoRun
    run = DynamoRun(dict(case["cfg"], precision=precision), fused_grid=fused)
    nz = case["noise"]
    if nz:
        run.initialize_fields(noise_amp=nz["amp"], noise_seed=nz["seed"])
    else:
        run.initialize_fields()
    run.setup_initial_state()
    run.initialize_dt(case["dt"])
    return run


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


P_TOL_ANEL = 1e-9


@pytest.mark.parametrize("name,fused", [("bench16", True), ("bench16", False), ("c1", True),
                                        ("dtchange", True), ("bpr16", True), ("bprdt", True),
                                        ("minc2", True), ("minc2", False),
                                        ("bprminc4", True), ("condic", True),
                                        ("bprcondic", True), ("rotic", True), ("rotic", False),
                                        ("bprrotic4", True), ("anel21", True), ("anelmag16", True),
                                        ("bpranel2", True), ("amc16", True), ("amc16", False),
                                        ("rotom8", True), ("fd2mhd", True), ("fd2mhd", False),
                                        ("fd4mhd", True), ("fdanel", True), ("fdanelmhd", True),
                                        ("fd4anel", True), ("fdcondic", True), ("fdrotic", True),
                                        ("fdbpr", True)])
def test_step_matches_reference_trajectory(name, fused):
    """fused: one grid-space kernel; otherwise separate FFT / products / FFT kernels.
    The dt each step returns is passed to the next (dtchange: the reference
    changes dt five times in 30 steps, each with a rebuild and variable-step
    CNAB2 weights).  bpr16 / bprdt: the BPR353 four-stage DIRK step of the
    reference at constant dt and with Courant-driven dt changes.  minc2 /
    bprminc4: azimuthal symmetry minc = 2 (CNAB2) and 4 (BPR353), the orders
    m = 0, minc, ... on one 2 pi / minc sector of longitudes.  condic /
    bprcondic: a conducting inner core (coupled outer/inner B and J solves),
    with the inner-core fields b_ic and aj_ic checked too.  rotic / bprrotic4:
    the conducting core also rotates (omega_ic integrated in time from the
    Lorentz torque, CNAB2 and BPR353 with minc = 4), its rotation rate checked
    at every step.  anel21 / anelmag16 / bpranel2: the anelastic step (the
    hydrodynamic benchmark's physics with angular-momentum corrections, a
    magnetic run, BPR353 with minc = 2); the pressure within P_TOL_ANEL (the
    l = 0 pressure's system under the integral condition has a condition number
    near 3e9: two LAPACK inverses differ by 3e-10 there).  amc16: Boussinesq,
    stress-free, with the axial and equatorial angular-momentum corrections.
    rotom8: a rotating core started at omega_ic1 = 2.  fd2mhd / fd4mhd / fdanel /
    fdanelmhd / fdbpr: the finite-difference radial scheme with the
    double-curl poloidal equation (second- and fourth-order stencils on the
    stretched grid, n_r even in fd4mhd, anelastic hydrodynamic and magnetic
    runs, BPR353)."""
    case, g = _load(name)
    run = _run(case, fused)
    dt = case["dt"]
    for n in range(1, case["steps"] + 1):
        dt = run.one_step(n, dt)
        assert dt == pytest.approx(g["dt"][n - 1], rel=1e-12)
        e = np.array(run.energies())
        ge = g["energies"][n - 1]
        assert np.all(np.abs(e - ge) <= 1e-9 * np.abs(ge)), (n, e, ge)
        if "omega_ic" in g.files:
            assert run.omega_ic == pytest.approx(g["omega_ic"][n - 1], rel=1e-10), n
        if n in case["field_steps"]:
            for k in ("s", "z", "w", "p", "b", "aj"):
                got, ref = run.f[k].cpu().numpy(), g[f"{k}_step{n}"]
                if not np.abs(ref).max():
                    assert not np.abs(got).max(), (n, k)
                    continue
                tol = P_TOL_ANEL if (k == "p" and run.anel) else 1e-10
                assert _rel(got, ref) < tol, (n, k, _rel(got, ref))
            if run.cond_ic:
                for k in ("b_ic", "aj_ic"):
                    got = run.fic[k].cpu().numpy()
                    assert _rel(got, g[f"{k}_step{n}"]) < 1e-10, (n, k, _rel(got, g[f"{k}_step{n}"]))


@pytest.mark.parametrize("name,precision,etol,ftol", [
    ("bench16", "mixed", 1e-6, 1e-5), ("c1", "mixed", 1e-6, 1e-5),
    ("c1", "mixed_bf16x3", 1e-6, 1e-5), ("c1", "mixed_bf16", 1e-4, 1e-4),
    ("bprminc4", "mixed", 1e-6, 1e-5), ("condic", "mixed_bf16x3", 1e-6, 1e-5),
    ("rotic", "mixed", 1e-6, 1e-5), ("fd2mhd", "mixed_bf16x3", 1e-6, 1e-5),
    ("fd4mhd", "mixed", 1e-6, 1e-5), ("anel21", "mixed_bf16x3", 1e-6, 1e-5),
    ("anelmag16", "mixed", 1e-6, 1e-5), ("fdanel", "mixed_bf16x3", 1e-6, 1e-5)])
def test_mixed_precision_step_tracks_reference(name, precision, etol, ftol):
    """Mixed precision (Legendre transforms on FP32 MFMA, or on BF16 MFMA with
    operands split into three or two bf16 planes; everything else FP64) against
    the FP64 reference trajectory: energies within `etol` relative and fields
    within `ftol` of their largest coefficient at every recorded step (a
    conducting and a rotating inner core, the finite-difference step and the
    anelastic step, whose grid path keeps FP64 Fourier buffers, included).  1e-6 is
    the mixed-precision target; two bf16 planes (about 16 significant bits)
    miss it by design and are held to 1e-4."""
    case, g = _load(name)
    run = _run(case, precision=precision)
    dt = case["dt"]
    worst = [0.0, 0.0]
    for n in range(1, case["steps"] + 1):
        dt = run.one_step(n, dt)
        assert dt == pytest.approx(g["dt"][n - 1], rel=1e-6)
        e = np.array(run.energies())
        ge = g["energies"][n - 1]
        nz = ge != 0   # a hydrodynamic run's magnetic energies are zero
        worst[0] = max(worst[0], float(np.max(np.abs(e - ge)[nz] / np.abs(ge[nz]))))
        assert np.all(np.abs(e - ge) <= etol * np.abs(ge)), (n, e, ge)
        if n in case["field_steps"]:
            for k in ("s", "z", "w", "p", "b", "aj"):
                got, ref = run.f[k].cpu().numpy(), g[f"{k}_step{n}"]
                if not np.abs(ref).max():   # zero in the reference (z at step 1, B of a
                    # hydrodynamic run): rounding-level values against the flow's scale
                    scale = np.abs(g[f"w_step{n}"]).max()
                    assert np.abs(got).max() <= ftol * scale, (n, k, np.abs(got).max())
                    continue
                worst[1] = max(worst[1], _rel(got, ref))
                assert _rel(got, ref) < ftol, (n, k, _rel(got, ref))
    print(f"{name} {precision}: worst energy rel. error {worst[0]:.2e}, field {worst[1]:.2e}")


@pytest.mark.parametrize("name", ["bench16", "fd2mhd", "fdanel"])
def test_first_step_explicit_terms(name):
    """Explicit terms after the first radial loop (get_nl + get_td in context);
    fd2mhd and fdanel: the double-curl poloidal term (Coriolis form with w'',
    z' and the radial derivative of the horizontal advection) and a zero
    pressure term."""
    case, g = _load(name)
    run = _run(case)
    run.one_step(1, case["dt"])
    for k in ("s", "z", "w", "p", "b", "j"):
        ref = g[f"expl_{k}_step1"]
        got = run.expl_prev[k].cpu().numpy()
        scale = max(np.abs(ref).max(), 1e-300)
        assert np.abs(got - ref).max() / scale < 1e-10 or np.abs(ref).max() == 0.0, k


_GRID_CFG = dict(ek=1e-3, ra=1e5, pr=1.0, prmag=5.0, radratio=0.35)
_SPEC = dict(Advr="AdvrLM", Advt="AdvtLM", Advp="AdvpLM", dVSr="dVSrLM", VSt="VStLM",
             VxBr="VxBrLM", VxBt="VxBtLM", VxBp="VxBpLM")


def _random_fields(shape, seed):
    from magic_amd.dynamo import _FIELDS
    rng = np.random.default_rng(seed)
    return {k: rng.standard_normal(shape) + 1j * rng.standard_normal(shape) for k in _FIELDS}


def _radial_loop_outputs(l_max, mode, seed=11, precision="fp64", rb=None):
    """One radial loop on random spectral fields; mode: fused, generic or separate;
    rb: radial levels per workgroup of the grid step (the tuner's by default)."""
    import torch
    from magic_amd.dynamo import DynamoRun
    run = DynamoRun(dict(_GRID_CFG, l_max=l_max, n_r_max=9, precision=precision),
                    fused_grid=(mode != "separate"))
    run.grid_generic = mode == "generic"
    if rb is not None:
        run.grid_rb = rb
    for k, a in _random_fields(tuple(run.f["s"].shape), seed).items():
        run.f[k].copy_(torch.as_tensor(a))
    cour = run.radial_loop()
    torch.cuda.synchronize()
    return {k: run.nl[k].cpu().numpy() for k in _SPEC}, np.array(cour)


_VECTOR_OF = dict(Advr="Adv", Advt="Adv", Advp="Adv", dVSr="VS", VSt="VS",
                  VxBr="VxB", VxBt="VxB", VxBp="VxB")


def _rel_errs(out, ref):
    """Max error of each output relative to the largest coefficient of its vector
    (advection, entropy flux, induction): on random fields one component can be
    far smaller than the others through cancellation."""
    scale = {}
    for k, g in _VECTOR_OF.items():
        scale[g] = max(scale.get(g, 1e-300), np.abs(ref[k]).max())
    return {k: float(np.abs(out[k] - ref[k]).max() / scale[_VECTOR_OF[k]]) for k in ref}


@pytest.mark.parametrize("l_max", [63, 85])
def test_grid_step_matches_oracle_on_random_fields(l_max):
    """All three grid-space paths (fused with compiled FFT plan, fused with the
    run-time plan, separate kernels) against the oracle's radial loop
    (irfft / get_nl / rfft of step_time.py:931-1212) on O(1) random spectral
    fields, through the same Legendre transforms.  l_max=63 gives n_phi/2 = 96
    (radix-3 register pass, compiled plan); l_max=85 gives n_phi/2 = 128
    (radix-8 passes)."""
    from oracle.dynamo import OracleRun
    orun = OracleRun(dict(_GRID_CFG, l_max=l_max, n_r_max=9))
    fields = _random_fields((orun.prm.lm_max, 9), 11)
    for k, a in fields.items():
        setattr(orun, k, a.copy())
    ocour = np.array(orun.radial_loop())
    ref = {k: orun.last_spec[v] for k, v in _SPEC.items()}
    for mode in ("fused", "generic", "separate"):
        out, cour = _radial_loop_outputs(l_max, mode)
        errs = _rel_errs(out, ref)
        assert max(errs.values()) < 1e-11, (mode, errs)
        assert np.allclose(cour, ocour, rtol=1e-12, atol=0), (mode, cour, ocour)


@pytest.mark.parametrize("l_max", [63, 85, 383])
def test_mixed_radial_loop_against_fp64(l_max):
    """Mixed precision radial loop (FP32 Legendre transforms, FP32 Fourier
    buffers, FP32 azimuthal FFTs and nonlinear products in the fused grid
    kernel, compiled and run-time FFT plans) against the FP64 loop on O(1)
    random fields: every explicit term within 5e-5 of the largest coefficient
    of its vector (FP32 rounding, 6e-8, grown by the Legendre sums over up to
    l_max/2 degrees, the length-n_phi FFTs and the 1/sin^2(theta) weighting of
    the theta/phi terms near the poles: 2.1e-5 measured at l_max=383), Courant
    maxima within 1e-5 relative."""
    ref, cref = _radial_loop_outputs(l_max, "fused")
    for mode in ("fused", "generic"):
        out, cour = _radial_loop_outputs(l_max, mode, precision="mixed")
        errs = _rel_errs(out, ref)
        assert max(errs.values()) < 5e-5, (mode, errs)
        assert np.allclose(cour, cref, rtol=1e-5, atol=0), (mode, cour, cref)


@pytest.mark.parametrize("l_max", [16, 127, 383])
def test_fp32_grid_step_vector_batches_match_single_transforms(l_max):
    """The FP32 grid step of the compiled plans (the three components of each
    vector transformed together over 3*RB LDS rows) against the kernel that
    transforms one component at a time (run-time plan): the same arithmetic per
    value, so FP32 outputs within 1e-6 of each vector's largest coefficient and
    Courant maxima within 1e-6 (l_max 16, 127, 383: n_phi/2 = 24, 192, 576)."""
    out, cour = _radial_loop_outputs(l_max, "fused", precision="mixed")
    ref, cref = _radial_loop_outputs(l_max, "generic", precision="mixed")
    errs = _rel_errs(out, ref)
    assert max(errs.values()) < 1e-6, errs
    assert np.allclose(cour, cref, rtol=1e-6, atol=0), (cour, cref)
    print(f"l_max={l_max}: max rel diff {max(errs.values()):.2e}, "
          f"Courant identical: {np.array_equal(cour, cref)}")


@pytest.mark.parametrize("l_max", [16, 383])
def test_fused_grid_step_matches_separate_kernels(l_max):
    """Fused grid-space kernel (compiled and run-time FFT plans) against the
    separate inverse FFT / get_nl / forward FFT kernels on random fields.
    l_max 16 and 383 give n_phi/2 = 24 and 576.  The two fused variants run the
    same arithmetic; against the separate kernels the summation order differs.
    Errors are relative to the largest coefficient of each vector."""
    ref, cref = _radial_loop_outputs(l_max, "separate")
    fused, cf = _radial_loop_outputs(l_max, "fused")
    gen, cg = _radial_loop_outputs(l_max, "generic")
    e_sep = _rel_errs(fused, ref)
    e_gen = _rel_errs(fused, gen)
    assert max(e_sep.values()) < 1e-11, e_sep
    assert max(e_gen.values()) < 1e-12, e_gen
    assert np.allclose(cf, cref, rtol=1e-12, atol=0), (cf, cref)
    assert np.allclose(cf, cg, rtol=1e-14, atol=0), (cf, cg)


@pytest.mark.parametrize("rb", [0, 1, 2])
@pytest.mark.parametrize("l_max,mh", [(42, 64), (48, 72), (85, 128), (96, 144), (170, 256)])
def test_grid_step_plan_lengths_match_run_time_plan(l_max, mh, rb):
    """Row lengths whose compiled plans have radix-8 passes, padded rows or (FP64,
    n_phi/2 <= 128, one or two levels) the three components of a vector in one pass,
    against the run-time plan of the same length and the separate kernels, at the
    level blocks that have a kernel of their own: FP64 within 1e-12 and 1e-11, FP32
    within 1e-6 of each vector's largest coefficient (the bounds of the tests above:
    the arithmetic per value is the same up to the order of sums)."""
    from magic_amd.params import Params
    assert Params(dict(l_max=l_max, n_r_max=17)).n_phi == 2 * mh
    fused, cf = _radial_loop_outputs(l_max, "fused", rb=rb)
    for other, tol, ctol in (("generic", 1e-12, 1e-14), ("separate", 1e-11, 1e-12)):
        ref, cref = _radial_loop_outputs(l_max, other, rb=0)
        errs = _rel_errs(fused, ref)
        assert max(errs.values()) < tol, (other, errs)
        assert np.allclose(cf, cref, rtol=ctol, atol=0), (other, cf, cref)
    out, cour = _radial_loop_outputs(l_max, "fused", precision="mixed", rb=rb)
    ref, cref = _radial_loop_outputs(l_max, "generic", precision="mixed", rb=0)
    errs = _rel_errs(out, ref)
    assert max(errs.values()) < 1e-6, errs
    assert np.allclose(cour, cref, rtol=1e-6, atol=0), (cour, cref)


@pytest.mark.parametrize("name", ["bench16", "c1", "bprdt", "fd2mhd", "fdbpr", "fdanel", "anel21",
                                  "bpranel2", "condic", "rotic", "bprrotic4"])
def test_graph_replay_matches_eager(name):
    """The step's radial and lm phases captured as HIP graphs (one per parity of
    the explicit-history buffers, weights read from device memory) and replayed
    every step, with the host Courant decision, rebuilds and energy reads in
    between: every step equals the eager step bit for bit."""
    import torch
    case, g = _load(name)
    eager = _run(case)
    graph = _run(case)
    graph.use_graphs = True
    dt_e = dt_g = case["dt"]
    for n in range(1, case["steps"] + 1):
        dt_e = eager.one_step(n, dt_e)
        dt_g = graph.one_step(n, dt_g)
        assert dt_g == dt_e
        assert graph.energies() == eager.energies(), n
        for k in ("s", "z", "w", "p", "b", "aj"):
            assert torch.equal(graph.f[k], eager.f[k]), (n, k)
    # two phases x two parities (CNAB2), or 3 radial + 4 lm stage graphs (BPR353)
    assert len(graph._graphs) == (7 if graph.dirk else 4)


# Courant-limited case: noise of amplitude 1 on s makes the flow strong enough
# that the Courant rule changes dt six times in 30 steps (l_max=16, n_r=33)
_DT_CASE = dict(cfg=dict(l_max=16, n_r_max=33, ek=1e-3, ra=1e5, pr=1.0, prmag=5.0,
                         radratio=0.35, dtmax=1e-3),
                dt=1e-3, noise=dict(amp=1.0, seed=7), steps=30)


def test_device_step_control_matches_host_steps_bpr353():
    """BPR353 under device step control: each step one captured sequence of the
    three radial loops, the dt decision at stage 1 (this scheme's Courant
    factors) with the stage weights and wimp_lin0 = dt/2 written on the device,
    the rebuild when dt changed, and the four lm loops; against host-decided
    steps bit for bit (dt sequence, rebuilds, time, fields) and the reference's
    dt sequence of traj_bprdt (the same case)."""
    import torch
    case = dict(_DT_CASE, cfg=dict(_DT_CASE["cfg"], time_scheme="BPR353"))
    host = _run(case)
    dev = _run(case)
    dev.use_graphs = True
    dt = case["dt"]
    for n in range(1, case["steps"] + 1):
        dt = host.one_step(n, dt)
    dev.run_steps(10, case["dt"])
    dev.run_steps(case["steps"] - 10, dev.dt_log[-1])
    assert dev.dt_log == host.dt_log
    assert dev.n_rebuild == host.n_rebuild and host.n_rebuild >= 4, host.n_rebuild
    assert dev.time == host.time and dev.n_step == host.n_step == case["steps"]
    for k in ("s", "z", "w", "p", "b", "aj", "db", "ddw"):
        assert torch.equal(dev.f[k], host.f[k]), k
    _, g = _load("bprdt")
    np.testing.assert_allclose(dev.dt_log, g["dt"], rtol=1e-12, atol=0)
    e, ge = np.array(dev.energies()), g["energies"][-1]
    assert np.all(np.abs(e - ge) <= 1e-9 * np.abs(ge)), (e, ge)
    assert [k for k in dev._graphs if k[0] == "step"] == [("step", "dirk")]


def test_device_step_control_matches_host_steps_anelastic():
    """The anelastic Chebyshev step under device step control: noise of
    amplitude 1 makes the Courant rule change dt six times in 20 steps, and each
    rebuild (A0 + w A1 of the anelastic S, Z and (w, p) matrices, inverses,
    folds, the fixed l = 0 pressure block) runs inside the captured step; dt
    sequence, rebuild count and fields equal the host-decided eager steps bit
    for bit, and the dt sequence and energies follow the oracle."""
    import torch
    case = dict(cfg=dict(l_max=16, n_r_max=33, strat=1.0, polind=2.0, g1=1.0, ra=1e5,
                         ek=1e-3, pr=1.0, prmag=5.0, dtmax=1e-3),
                dt=1e-3, noise=dict(amp=1.0, seed=7), steps=20)
    host = _run(case)
    dev = _run(case)
    dev.use_graphs = True
    dt = case["dt"]
    for n in range(1, case["steps"] + 1):
        dt = host.one_step(n, dt)
    dev.run_steps(8, case["dt"])
    dev.run_steps(case["steps"] - 8, dev.dt_log[-1])
    assert dev.dt_log == host.dt_log
    assert dev.n_rebuild == host.n_rebuild and host.n_rebuild >= 5, host.n_rebuild
    for k in ("s", "z", "w", "p", "b", "aj", "dw", "ddw"):
        assert torch.equal(dev.f[k], host.f[k]), k
    from oracle.dynamo import OracleRun
    orc = OracleRun(dict(case["cfg"]))
    orc.initialize_fields()
    orc.add_noise(case["noise"]["seed"], case["noise"]["amp"])
    orc.setup_initial_state()
    orc.initialize_dt(case["dt"])
    dt = case["dt"]
    odts = []
    for n in range(1, case["steps"] + 1):
        dt = orc.one_step(n, dt)
        odts.append(dt)
    np.testing.assert_allclose(dev.dt_log, odts, rtol=1e-9)
    e, oe = np.array(dev.energies()), np.array(orc.energies())
    assert np.all(np.abs(e - oe) <= 1e-9 * np.abs(oe)), (e, oe)


def test_device_step_control_matches_host_steps_rotating_inner_core():
    """A conducting, rotating inner core under device step control: the coupled
    outer/inner B and J operators and the z(l=1, m=0) operator are rebuilt on the
    device (A0 + w A1, inverses, folds) inside the captured step whenever the
    Courant rule changes dt; dt sequence, rebuild count, omega_ic and fields
    (outer and inner) equal the host-decided eager steps bit for bit."""
    import torch
    case = dict(cfg=dict(l_max=16, n_r_max=33, n_cheb_max=31, n_cheb_ic_max=15,
                         sigma_ratio=1.0, kbotb=3, nRotIC=1, dtmax=1e-3),
                dt=1e-3, noise=dict(amp=1.0, seed=7), steps=20)
    host = _run(case)
    dev = _run(case)
    dev.use_graphs = True
    dt = case["dt"]
    for n in range(1, case["steps"] + 1):
        dt = host.one_step(n, dt)
    dev.run_steps(8, case["dt"])
    dev.run_steps(case["steps"] - 8, dev.dt_log[-1])
    assert dev.dt_log == host.dt_log
    assert dev.n_rebuild == host.n_rebuild and host.n_rebuild >= 3, host.n_rebuild
    assert dev.omega_ic == host.omega_ic
    for k in ("s", "z", "w", "p", "b", "aj", "db", "ddw"):
        assert torch.equal(dev.f[k], host.f[k]), k
    for k in ("b_ic", "aj_ic"):
        assert torch.equal(dev.fic[k], host.fic[k]), k


def test_device_step_control_matches_host_steps_finite_differences():
    """The finite-difference (double-curl) step under device step control: the
    Courant rule changes dt six times in 30 steps and every rebuild (affine
    assembly, inverses, folds) runs inside the captured step; dt sequence,
    rebuild count and fields equal the host-decided eager steps bit for bit,
    and the dt sequence and energies follow the oracle."""
    import torch
    case = dict(_DT_CASE, cfg=dict(_DT_CASE["cfg"], radial_scheme="FD", fd_order=2,
                                   fd_order_bound=2))
    host = _run(case)
    dev = _run(case)
    dev.use_graphs = True
    dt = case["dt"]
    for n in range(1, case["steps"] + 1):
        dt = host.one_step(n, dt)
    dev.run_steps(10, case["dt"])
    dev.run_steps(case["steps"] - 10, dev.dt_log[-1])
    assert dev.dt_log == host.dt_log
    assert dev.n_rebuild == host.n_rebuild and host.n_rebuild >= 6, host.n_rebuild
    for k in ("s", "z", "w", "p", "b", "aj", "dw", "ddw"):
        assert torch.equal(dev.f[k], host.f[k]), k
    from oracle.dynamo import OracleRun
    orc = OracleRun(dict(case["cfg"]))
    orc.initialize_fields()
    orc.add_noise(case["noise"]["seed"], case["noise"]["amp"])
    orc.setup_initial_state()
    orc.initialize_dt(case["dt"])
    dt = case["dt"]
    odts = []
    for n in range(1, case["steps"] + 1):
        dt = orc.one_step(n, dt)
        odts.append(dt)
    np.testing.assert_allclose(dev.dt_log, odts, rtol=1e-9)
    e, oe = np.array(dev.energies()), np.array(orc.energies())
    assert np.all(np.abs(e - oe) <= 1e-9 * np.abs(oe)), (e, oe)


def test_device_step_control_matches_host_steps():
    """Steps with the dt decision on the device, each step one HIP graph (radial
    loop, step control, rebuild launches that run only when dt changed, lm loop),
    against host-decided eager steps: same dt sequence, rebuild count, time and
    fields bit for bit, in two batches (state read back and pushed again in
    between); the dt sequence also follows the oracle's."""
    import torch
    case = _DT_CASE
    host = _run(case)
    dev = _run(case)
    dev.use_graphs = True
    dt = case["dt"]
    for n in range(1, case["steps"] + 1):
        dt = host.one_step(n, dt)
    dev.run_steps(10, case["dt"])
    dev.run_steps(case["steps"] - 10, dev.dt_log[-1])
    assert dev.dt_log == host.dt_log
    # the same case as the reference fixture traj_dtchange: the reference's dt sequence
    _, g = _load("dtchange")
    np.testing.assert_allclose(dev.dt_log, g["dt"], rtol=1e-12, atol=0)
    assert dev.n_rebuild == host.n_rebuild and host.n_rebuild >= 6, host.n_rebuild
    assert dev.time == host.time and dev.n_step == host.n_step == case["steps"]
    for k in ("s", "z", "w", "p", "b", "aj", "db", "ddw"):
        assert torch.equal(dev.f[k], host.f[k]), k
    assert dev.energies() == host.energies()
    assert sorted(k[0] for k in dev._graphs) == ["step", "step"]
    # the oracle's decisions on the same initial state
    from oracle.dynamo import OracleRun
    orc = OracleRun(dict(case["cfg"]))
    orc.initialize_fields()
    orc.add_noise(case["noise"]["seed"], case["noise"]["amp"])
    orc.setup_initial_state()
    orc.initialize_dt(case["dt"])
    dt = case["dt"]
    odts = []
    for n in range(1, case["steps"] + 1):
        dt = orc.one_step(n, dt)
        odts.append(dt)
    np.testing.assert_allclose(dev.dt_log, odts, rtol=1e-9)
    e, oe = np.array(dev.energies()), np.array(orc.energies())
    assert np.all(np.abs(e - oe) <= 1e-9 * np.abs(oe)), (e, oe)


def test_device_step_control_replays_schedule_with_timers():
    """dt_schedule replay through the device step control, run eagerly with
    section timers (the step's launch sequence outside a graph), equals the
    host-decided run on the same schedule."""
    import torch
    case = _DT_CASE
    sched = [4e-5] * 4 + [3e-5] * 3 + [2.5e-5] * 5  # below the case's Courant limits
    host = _run(case)
    dev = _run(case)
    host.dt_schedule = dev.dt_schedule = sched
    dt = case["dt"]
    for n in range(1, len(sched) + 1):
        dt = host.one_step(n, dt)
    dev.enable_timers(True)
    dev.run_steps(len(sched), case["dt"])
    assert dev.dt_log == host.dt_log == sched
    assert dev.n_rebuild == host.n_rebuild == 3
    for k in ("s", "z", "w", "b", "aj"):
        assert torch.equal(dev.f[k], host.f[k]), k
    t = dev.timer_summary()
    assert "step_ctl" in t and "rebuild" in t


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("l_max", [20, 32, 40, 42, 48, 63, 72, 85, 96, 127, 170, 191, 255, 383])
def test_grid_level_blocks_give_identical_results(l_max, precision):
    """Every level block the tuner may choose (1, 2, 4, ... up to the plan's own), and
    blocks between those, give the same Fourier outputs and Courant maxima bit for
    bit: compiled plans (n_phi/2 = 48, 64, 72, 96, 128, 144, 192, 256, 288, 384, 576,
    their own, 1- and 2-level instantiations) and the run-time plan (30, 60, 108)."""
    import torch
    from magic_amd import tune
    from magic_amd.device import Resolution
    from magic_amd.params import Params
    N = 9
    p = Params(dict(_GRID_CFG, l_max=l_max, n_r_max=N, precision=precision))
    res = Resolution(p, "cuda")
    fdt = torch.float32 if precision == "mixed" else torch.float64
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    Fs = torch.randn(res.fourier_buffer(1, N, fdt).shape, generator=gen, device="cuda",
                     dtype=fdt) * 1e-2
    Fv = torch.randn(res.fourier_buffer(3, 4 * N, fdt).shape, generator=gen, device="cuda",
                     dtype=fdt) * 1e-2
    own = res.grid_plan()[2]
    outs = {}
    for rb in sorted({*tune.grid_candidates(own), min(3, own), max(1, own - 1)}):
        Fo = res.fourier_buffer(9, N - 2, fdt).zero_()
        cfl = torch.zeros(2 * N, dtype=torch.int64, device="cuda")
        res.grid_step(Fs, Fv, Fo, N, cfl, p, rb=0 if rb == own else rb)
        torch.cuda.synchronize()
        outs[rb] = (Fo, cfl)
    ref_Fo, ref_cfl = outs[own]
    assert torch.isfinite(ref_Fo).all() and (ref_cfl > 0).all()
    for rb, (Fo, cfl) in outs.items():
        assert torch.equal(Fo, ref_Fo), rb
        assert torch.equal(cfl, ref_cfl), rb


@pytest.mark.parametrize("l_max,prec", [(32, 1), (85, 1), (383, 1)])
def test_synthesis_workgroup_sizes_give_identical_results(l_max, prec):
    """The FP32 vector and scalar Legendre synthesis (FP32 tables, FP32 Fourier
    buffer) with 4 and 6 waves per workgroup, and the vector synthesis with one or two
    column tiles per workgroup (the tuner's candidates), write the same Fourier
    coefficients bit for bit."""
    import torch
    from magic_amd.device import Resolution
    from magic_amd.params import Params
    N = 9
    p = Params(dict(_GRID_CFG, l_max=l_max, n_r_max=N, precision="mixed" if prec else "fp64"))
    res = Resolution(p, "cuda")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    xs = [torch.randn(res.L, N, dtype=torch.complex128, generator=gen, device="cuda")
          for _ in range(4)]
    fdt = torch.float32 if prec else torch.float64
    groups = [[(xs[0], None, 1), (xs[1], None, 0), (xs[2], xs[3], 2)] for _ in range(4)]
    outs = {}
    shapes = [(4, 1), (6, 1)] + ([(4, 2), (6, 2)] if prec else [])
    for w, nct in shapes:
        Fv = res.fourier_buffer(3, 4 * N, fdt).zero_()
        Fs = res.fourier_buffer(1, N, fdt).zero_()
        res.synth(groups, N, N, Fv, 4 * N, vector=True, prec=prec, waves=w, nct=nct)
        res.synth([[(xs[0], None, 0)]], N, N, Fs, N, vector=False, prec=prec, waves=w)
        torch.cuda.synchronize()
        outs[(w, nct)] = (Fv, Fs)
    ref = outs[(4, 1)]
    assert torch.isfinite(ref[0]).all() and ref[0].abs().max() > 0
    for key, (Fv, Fs) in outs.items():
        assert torch.equal(Fv, ref[0]) and torch.equal(Fs, ref[1]), key


@pytest.mark.parametrize("l_max,prec", [(32, 1), (85, 1), (383, 1)])
def test_analysis_workgroup_sizes_give_identical_results(l_max, prec):
    """The FP32 vector and scalar Legendre analysis with 6 and 4 waves per workgroup
    (each with its own tile list) write the same coefficients bit for bit and
    leave the boundary columns untouched."""
    import torch
    from magic_amd.device import Resolution
    from magic_amd.params import Params
    N = 9
    Nb = N - 2
    p = Params(dict(_GRID_CFG, l_max=l_max, n_r_max=N, precision="mixed" if prec else "fp64"))
    res = Resolution(p, "cuda")
    fdt = torch.float32 if prec else torch.float64
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    F = torch.randn(res.fourier_buffer(9, Nb, fdt).shape, generator=gen, device="cuda", dtype=fdt)
    outs = {}
    for w in (6, 4):
        y = [torch.zeros(res.L, N, dtype=torch.complex128, device="cuda") for _ in range(8)]
        o = lambda t: t.data_ptr() + 16
        res.analysis(F, Nb, Nb, [(3, 4), (5, 6), (7, 8)], [o(y[0]), o(y[1]), o(y[2])],
                     [o(y[3]), None, o(y[4])], N, vector=True, prec=prec, waves=w)
        res.analysis(F, Nb, Nb, [0, 1, 2], [o(y[5]), o(y[6]), o(y[7])], [None, None, None], N,
                     vector=False, prec=prec, waves=w)
        torch.cuda.synchronize()
        outs[w] = y
    for a, b in zip(outs[6], outs[4]):
        assert torch.equal(a, b)
        assert not a[:, 0].any() and not a[:, N - 1].any()
    assert outs[6][0].abs().max() > 0


@pytest.mark.parametrize("l_max,n_r", [(32, 33), (127, 65), (383, 97)])
def test_row_operator_tile_shapes_give_identical_results(l_max, n_r):
    """The row operator with 32 x 64 and with 32 x 128 tiles (the tuner's
    candidates) writes the same results bit for bit, for every job table of a
    run: the S/Z/B/J and (w,p) solves with their derivatives, the flux
    derivatives and the set-up derivatives, on random operators and inputs."""
    import torch
    from magic_amd.dynamo import DynamoRun
    run = DynamoRun(dict(_GRID_CFG, l_max=l_max, n_r_max=n_r))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    for t in (run.MT4, run.MT["wp"], run.MT_d1[0], run.MT_d1r2[0], run.MT_d12[0], run.MT_d123[0]):
        t.copy_(torch.randn(t.shape, generator=gen, device="cuda", dtype=t.dtype))
    start = torch.randn(run._pool.shape, generator=gen, device="cuda", dtype=run._pool.dtype)
    for name in ("jobs1", "jobs2", "jobs_td", "jobs_setup"):
        out = []
        for wide in (0, 1):
            run._pool.copy_(start)
            run._rowop(getattr(run, name), wide)
            torch.cuda.synchronize()
            out.append(run._pool.clone())
        assert not torch.equal(out[0], start), name
        assert torch.equal(out[0], out[1]), name
    run.close()


@pytest.mark.parametrize("mixed", ["mixed", "mixed_bf16x3"])
def test_headline_configuration_mixed_tracks_fp64(mixed):
    """The headline configuration (l_max=383, n_r=97, E=1e-5, Ra=2e8, Pm=1,
    seeded noise 1e-4 and the dipole seed): 10 device-controlled steps (one HIP
    graph each) in FP64 and in mixed precision (FP32 or three-plane BF16
    Legendre transforms) on the FP64 run's step sizes; energies within 1e-6
    relative (the mixed-precision target), every field finite, and the same dt
    sequence and rebuild count."""
    import math
    import torch
    from magic_amd.dynamo import DynamoRun
    cfg = dict(l_max=383, n_r_max=97, ek=1e-5, ra=2e8, pr=1.0, prmag=1.0, radratio=0.35,
               dtmax=1e-4)
    out = {}
    sched = None
    for precision in ("fp64", mixed):
        run = DynamoRun(dict(cfg, precision=precision))
        run.dt_schedule = sched
        run.use_graphs = True
        run.initialize_fields(noise_amp=1e-4, noise_seed=20261202)
        run.setup_initial_state()
        run.initialize_dt(cfg["dtmax"])
        run.run_steps(10, run.dtMax)
        for k in ("s", "w", "z", "b", "aj"):
            assert torch.isfinite(torch.view_as_real(run.f[k])).all(), (precision, k)
        out[precision] = (run.energies(), list(run.dt_log), run.n_rebuild)
        sched = list(run.dt_log)
        run.close()
    (e64, dt64, nr64), (emx, dtmx, nrmx) = out["fp64"], out[mixed]
    assert dt64 == dtmx and nr64 == nrmx
    for a, b in zip(e64, emx):
        assert math.isfinite(b) and abs(b - a) <= 1e-6 * abs(a), (a, b)
