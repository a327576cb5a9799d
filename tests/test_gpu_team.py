"""GPU parity of the multi-wavefront integrator (mechanisms of 64..191 species,
one workgroup of 2 or 3 wavefronts per reactor; an FP32 Newton matrix
inverted in place in LDS by blocked Gauss-Jordan on FP32 MFMA, or an FP64 one
in the team's device slot on FP64 MFMA) against the FP64 oracle: the seeded
160-species / 900-reaction workload mechanism and the reference's 79-species
DME mechanism (data/mechanisms/dme/dme_24_mech.txt).

As for the one-wavefront integrators, the bar is self-calibrated on the same
inputs: GPU-vs-oracle differences in tolerance units (rtol |y| + atol) within
the oracle's own one-ulp sensitivity (the FP64 matrix with the plain method's
margins, the FP32 one with the FP32 preconditioner's), mean step counts
close, no failures, sum(Y) = 1 to 1e-9 (FP64) or 1e-8 (FP32).
"""
import numpy as np
import pytest

from conftest import mech_paths

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1.0e-6, 1.0e-12


def _units(Ya, Ta, Yb, Tb):
    eY = np.abs(Ya - Yb) / (RTOL * np.abs(Yb) + ATOL)
    eT = np.abs(Ta - Tb) / (RTOL * np.abs(Tb))
    return np.maximum(eY.max(axis=1), eT)


def _dme_states(species, n, seed):
    rng = np.random.default_rng(seed)
    idx = {s: i for i, s in enumerate(species)}
    Y = np.zeros((n, len(species)))
    phi = rng.uniform(0.5, 2.0, n)
    # DME + air: CH3OCH3 + 3 O2 -> 2 CO2 + 3 H2O (mass ratio 46.07 : 96)
    fuel = phi * 46.07 / 96.0 * 0.233
    Y[:, idx["ch3och3"]] = fuel / (1.0 + fuel)
    Y[:, idx["o2"]] = 0.233 / (1.0 + fuel)
    Y[:, idx["n2"]] = 1.0 - Y[:, idx["ch3och3"]] - Y[:, idx["o2"]]
    T = rng.uniform(900.0, 1400.0, n)
    P = rng.uniform(1.0, 20.0, n) * 101325.0
    return T, P, Y


@pytest.mark.parametrize("name,n,dt,f32", [("synth_160sp", 48, 1e-5, 1), ("ref_dme", 64, 1e-4, 1),
                                          ("synth_160sp", 48, 1e-5, 0), ("ref_dme", 64, 1e-4, 0)])
def test_team_integrator_matches_oracle(torch_gpu, oracle_mod, name, n, dt, f32):
    from zerork_hip import capi, mechgen
    torch = torch_gpu
    m = capi.Mech(*mech_paths(name))
    o = oracle_mod.Oracle(*mech_paths(name))
    if name == "synth_160sp":
        st = mechgen.workload_states("160sp", mechgen.workload_mechanism("160sp"), n, seed=160)
        T0, P0, Y0 = st.T, st.P, st.Y
    else:
        T0, P0, Y0 = _dme_states(m.species(), n, seed=79)
    nsp = m.nsp
    print("case", name, "nsp", nsp, "n", n, "fp32 preconditioner", f32, flush=True)
    dev = torch.device("cuda:0")
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)
    dT, dP, dY = t(T0), t(P0), t(Y0)
    steps = torch.zeros(n, dtype=torch.int32, device=dev)
    opts = capi.default_options(rel_tol=RTOL, abs_tol=ATOL, fp32_preconditioner=f32)
    m.integrate(n, dt, dT, dP, dY, nsp, opts, steps)
    torch.cuda.synchronize()
    Tg, Yg, sg = dT.cpu().numpy(), dY.cpu().numpy(), steps.cpu().numpy()
    oo = oracle_mod.default_opts(rtol=RTOL, atol=ATOL)
    To, Yo, ost = o.integrate(T0, P0, Y0, dt, oo)
    Tp, Yp, _ = o.integrate(np.nextafter(T0, np.inf), P0, Y0, dt, oo)
    assert np.all(ost["nsteps"] > 0)
    assert np.all(sg > 0), np.sum(sg <= 0)
    gpu, ulp = _units(Yg, Tg, Yo, To), _units(Yp, Tp, Yo, To)
    gq, uq = np.percentile(gpu, [50, 90, 100]), np.percentile(ulp, [50, 90, 100])
    print(f"{name}: GPU-oracle tolerance units p50/p90/max {gq.round(2)}; oracle 1-ulp "
          f"{uq.round(2)}; mean steps gpu {sg.mean():.1f} oracle {ost['nsteps'].mean():.1f}; "
          f"T rise max {np.max(To - T0):.1f} K", flush=True)
    if f32:
        # the FP32 preconditioner's bar (as for one wavefront): FP32 Newton
        # matrices change the iterates by more than round-off
        assert gq[0] <= 2.0 * uq[0] + 1.0 and gq[1] <= 2.0 * uq[1] + 10.0
        assert gq[2] <= 4.0 * uq[2] + 50.0
        assert abs(sg.mean() / ost["nsteps"].mean() - 1.0) < 0.05
    else:
        # FP64 throughout: the one-wavefront plain bar, except at p90, which
        # over 64 igniting DME reactors sits a few units above twice the
        # one-ulp p90: the GPU's Gauss-Jordan solve differs from the oracle's
        # pivoted LU by round-off at every Newton iteration, while the
        # one-ulp run perturbs the state once, at t = 0
        assert gq[0] <= 2.0 * uq[0] + 1.0 and gq[1] <= 2.0 * uq[1] + 5.0
        assert gq[2] <= 4.0 * uq[2] + 10.0
        assert abs(sg.mean() / ost["nsteps"].mean() - 1.0) < 0.02
    osum = max(np.abs(Yo.sum(axis=1) - 1.0).max(), np.abs(Yp.sum(axis=1) - 1.0).max())
    assert np.all(np.abs(Yg.sum(axis=1) - 1.0) <= max(1e-8 if f32 else 1e-9, 2.0 * osum))


def test_two_wave_team_on_53_species_and_autotune(torch_gpu, oracle_mod):
    """A 53-species mechanism also runs on a team of two wavefronts (FP32): same
    parity bar as the one-wavefront FP32 integrator; the autotuner times every
    team size that fits (1, 2 and 3 wavefronts) on a batch and keeps the fastest."""
    from zerork_hip import capi, mechgen
    torch = torch_gpu
    m = capi.Mech(*mech_paths("synth_53sp"))
    o = oracle_mod.Oracle(*mech_paths("synth_53sp"))
    st = mechgen.workload_states("53sp", mechgen.workload_mechanism("53sp"), 256, seed=102)
    n, nsp = st.Y.shape
    print("case 53sp two-wave team", flush=True)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda:0")
    opts = capi.default_options(rel_tol=RTOL, abs_tol=ATOL, fp32_preconditioner=1)
    m.set_team_width(1, 2)
    dT, dP, dY = t(st.T), t(st.P), t(st.Y)
    steps = torch.zeros(n, dtype=torch.int32, device="cuda:0")
    m.integrate(n, 1e-4, dT, dP, dY, nsp, opts, steps)
    torch.cuda.synchronize()
    Tg, Yg, sg = dT.cpu().numpy(), dY.cpu().numpy(), steps.cpu().numpy()
    oo = oracle_mod.default_opts(rtol=RTOL, atol=ATOL)
    To, Yo, ost = o.integrate(st.T, st.P, st.Y, 1e-4, oo)
    Tp, Yp, _ = o.integrate(np.nextafter(st.T, np.inf), st.P, st.Y, 1e-4, oo)
    gpu, ulp = _units(Yg, Tg, Yo, To), _units(Yp, Tp, Yo, To)
    gq, uq = np.percentile(gpu, [50, 90, 100]), np.percentile(ulp, [50, 90, 100])
    print(f"53sp team of 2: GPU-oracle p50/p90/max {gq.round(2)}; 1-ulp {uq.round(2)}; "
          f"mean steps {sg.mean():.1f} vs {ost['nsteps'].mean():.1f}", flush=True)
    assert np.all(sg > 0)
    assert gq[0] <= 2.0 * uq[0] + 1.0 and gq[1] <= 2.0 * uq[1] + 10.0
    assert gq[2] <= 4.0 * uq[2] + 50.0
    assert abs(sg.mean() / ost["nsteps"].mean() - 1.0) < 0.05
    # autotune on a larger batch
    m.set_team_width(1, 0)
    big = mechgen.workload_states("53sp", mechgen.workload_mechanism("53sp"), 8192, seed=5)
    choice, ms = m.autotune(8192, 1e-4, t(big.T), t(big.P), t(big.Y), nsp, opts)
    print(f"autotune: chose {choice} wavefronts per reactor; times {ms}", flush=True)
    assert 1 in ms and 2 in ms and set(ms) <= {1, 2, 3}
    assert choice in ms and ms[choice] == min(ms.values())


@pytest.mark.parametrize("f32", [1, 0])
@pytest.mark.parametrize("nsp,nrxn", [(15, 30), (16, 32), (31, 80), (47, 120), (63, 200),
                                      (64, 200), (95, 300), (112, 400), (127, 400)])
def test_team_sizes_agree_bitwise(torch_gpu, tmp_path, nsp, nrxn, f32):
    """Teams of 2 and 3 wavefronts of state hold the Newton matrix in different
    grids of 16 x 16 register tiles (2 x 2 wavefronts of 4 x 4 tiles, 4 x 2 of
    3 x 6) and split the rates over 4 and 8 wavefronts, but do the same
    operations in the same order on every element: the same bits, at the edges
    of the tiles and of the grids (nsp + 1 rows: 16, 17, 32, 48, 64, 65, 96,
    113, 128)."""
    from zerork_hip import capi, mechgen
    torch = torch_gpu
    mg = mechgen.generate(nsp, nrxn, 4000 + nsp, ("C", "H", "O", "N", "AR"), 0.25, 0.15,
                          inert=("N2", "AR"), majors=mechgen._C2_BASE, base=mechgen._C2_BASE)
    m = capi.Mech(*mg.write(str(tmp_path), "m"))
    n = 12
    st = mechgen.random_dense_states(mg, n, seed=nsp, Tlo=900.0, Thi=1600.0, Plo=1.0, Phi=20.0)
    print("case", nsp, "species, fp32 preconditioner", f32, flush=True)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda:0")
    ends = []
    for W in (2, 3):
        T, P, Y = t(st.T), t(st.P), t(st.Y)
        stats = torch.zeros(8 * n, dtype=torch.int32, device="cuda:0")
        m.set_team_width(f32, W)
        m.integrate(n, 1.0e-9, T, P, Y, nsp,
                    capi.default_options(rel_tol=RTOL, abs_tol=ATOL, fp32_preconditioner=f32),
                    None, stats)
        torch.cuda.synchronize()
        ends.append((T.cpu().numpy(), Y.cpu().numpy(), stats.cpu().numpy().reshape(n, 8)))
    m.set_team_width(f32, 0)
    a, b = ends
    assert (a[2][:, 7] == 0).all() and (a[2][:, 3] > 0).all()  # succeeded, with setups
    assert np.array_equal(a[2], b[2])
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("f32", [1, 0])
@pytest.mark.parametrize("nsp,nrxn", [(15, 30), (16, 32), (31, 80), (32, 80), (55, 160), (56, 160),
                                      (63, 200)])
def test_one_wavefront_sizes_agree_with_teams(torch_gpu, tmp_path, nsp, nrxn, f32):
    """One wavefront per reactor at the edges of its variants (up to 15 species
    everything is inlined; the FP64 inverse holds a multiple of 8 columns for
    nsp + 1 rows) against a team of two wavefronts.  With the FP32 matrix both do
    the same operations in the same order: the same bits.  With the FP64 one the
    inverses differ by round-off, and the states by no more than integration errors
    of 1e-6 a step: 100 tolerance units over the tens of steps of a nanosecond."""
    from zerork_hip import capi, mechgen
    torch = torch_gpu
    mg = mechgen.generate(nsp, nrxn, 4000 + nsp, ("C", "H", "O", "N", "AR"), 0.25, 0.15,
                          inert=("N2", "AR"), majors=mechgen._C2_BASE, base=mechgen._C2_BASE)
    m = capi.Mech(*mg.write(str(tmp_path), "m"))
    n = 12
    st = mechgen.random_dense_states(mg, n, seed=nsp, Tlo=900.0, Thi=1600.0, Plo=1.0, Phi=20.0)
    print("case", nsp, "species, fp32 preconditioner", f32, flush=True)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda:0")
    ends = []
    for W in (1, 2):
        T, P, Y = t(st.T), t(st.P), t(st.Y)
        stats = torch.zeros(8 * n, dtype=torch.int32, device="cuda:0")
        m.set_team_width(f32, W)
        m.integrate(n, 1.0e-9, T, P, Y, nsp,
                    capi.default_options(rel_tol=RTOL, abs_tol=ATOL, fp32_preconditioner=f32),
                    None, stats)
        torch.cuda.synchronize()
        ends.append((T.cpu().numpy(), Y.cpu().numpy(), stats.cpu().numpy().reshape(n, 8)))
    m.set_team_width(f32, 0)
    a, b = ends
    assert (a[2][:, 7] == 0).all() and (a[2][:, 3] > 0).all()  # succeeded, with setups
    if f32:
        assert np.array_equal(a[2], b[2])
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    else:
        assert np.max(np.abs(a[0] - b[0]) / (RTOL * np.abs(b[0]) + ATOL)) <= 100.0
        assert np.max(np.abs(a[1] - b[1]) / (RTOL * np.abs(b[1]) + ATOL)) <= 100.0


def _generated(tmp_path, nsp, nrxn, fractions=(0.25, 0.15)):
    from zerork_hip import mechgen
    mg = mechgen.generate(nsp, nrxn, 4000 + nsp, ("C", "H", "O", "N", "AR"), *fractions,
                          inert=("N2", "AR"), majors=mechgen._C2_BASE, base=mechgen._C2_BASE)
    st = mechgen.random_dense_states(mg, 12, seed=nsp, Tlo=900.0, Thi=1600.0, Plo=1.0, Phi=20.0)
    return mg.write(str(tmp_path), "m"), st


def _integrated(torch, m, st, W, f32, dt=1.0e-9, **kw):
    from zerork_hip import capi
    n = len(st.T)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda:0")
    T, P, Y = t(st.T), t(st.P), t(st.Y)
    stats = torch.zeros(8 * n, dtype=torch.int32, device="cuda:0")
    m.set_team_width(f32, W)
    m.integrate(n, dt, T, P, Y, m.nsp,
                capi.default_options(rel_tol=RTOL, abs_tol=ATOL, fp32_preconditioner=f32, **kw),
                None, stats)
    torch.cuda.synchronize()
    m.set_team_width(f32, 0)
    return T.cpu().numpy(), Y.cpu().numpy(), stats.cpu().numpy().reshape(n, 8)


@pytest.mark.parametrize("nsp,nrxn,ign", [(15, 30, 0.0), (15, 30, 400.0), (16, 32, 400.0),
                                          (31, 64, 0.0), (31, 65, 0.0), (31, 64, 400.0),
                                          (32, 64, 0.0)])
def test_small_variants_agree_with_teams(torch_gpu, tmp_path, nsp, nrxn, ign):
    """The one-wavefront FP32 variants by size: one tile (up to 15 species, with and
    without the ignition root), two tiles a side with the right-hand side inlined (up to
    31 species whose records fill one iteration of 64) or called, and the larger grid,
    against a team of two wavefronts, which has none of them: the same operations in the
    same order on every element, so the same bits."""
    from zerork_hip import capi
    files, st = _generated(tmp_path, nsp, nrxn, (0.15, 0.1))
    m = capi.Mech(*files)
    print("case", nsp, nrxn, "ignition", ign, flush=True)
    kw = dict(delta_temperature_ignition=ign) if ign else {}
    a, b = (_integrated(torch_gpu, m, st, W, 1, **kw) for W in (1, 2))
    assert (a[2][:, 7] == 0).all() and (a[2][:, 3] > 0).all()
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("nsp,nrxn,W,f32", [(15, 30, 1, 0), (16, 32, 1, 0), (23, 46, 1, 0),
                                            (24, 48, 1, 0), (31, 80, 1, 0), (39, 100, 1, 0),
                                            (40, 100, 1, 0), (47, 120, 1, 0), (48, 120, 1, 0),
                                            (55, 160, 1, 0), (63, 200, 1, 0), (63, 200, 1, 1),
                                            (127, 400, 2, 0), (128, 400, 3, 0), (143, 400, 3, 0),
                                            (144, 400, 3, 0), (175, 400, 3, 0), (176, 400, 3, 0),
                                            (191, 400, 3, 0), (143, 400, 3, 1), (191, 400, 3, 1)])
def test_inverse_sizes_match_oracle(torch_gpu, oracle_mod, tmp_path, nsp, nrxn, W, f32):
    """Newton matrices at the edges of the FP64 row inverse (8 columns more each) and of the
    team's tiles (nsp + 1 rows: full last tiles at 128, 144, 176 and 192) against the FP64
    oracle and its pivoted LU.  A wrong inverse costs Newton iterations, set-ups and
    convergence failures before it costs accuracy, so their totals are held to the bar of
    the step counts (2 % for the FP64 matrix, 5 % for the FP32 one) plus twice what one ulp
    of the initial temperatures changes in the oracle's own."""
    from zerork_hip import capi
    files, st = _generated(tmp_path, nsp, nrxn)
    m, o = capi.Mech(*files), oracle_mod.Oracle(*files)
    print("case", nsp, "species, team", W, "fp32 preconditioner", f32, flush=True)
    T, Y, stats = _integrated(torch_gpu, m, st, W, f32)
    oo = oracle_mod.default_opts(rtol=RTOL, atol=ATOL)
    To, Yo, ost = o.integrate(st.T, st.P, st.Y, 1.0e-9, oo)
    Tp, Yp, pst = o.integrate(np.nextafter(st.T, np.inf), st.P, st.Y, 1.0e-9, oo)
    assert (stats[:, 7] == 0).all() and (ost["status"] == 0).all()
    total = dict(zip(("nst", "nfe", "nje", "nsetups", "nni", "ncfn", "netf"), stats.sum(axis=0)))
    bar = 0.05 if f32 else 0.02
    for k in ("nst", "nsetups", "nni"):
        ref, ulp = float(ost[k].sum()), float(pst[k].sum())
        print(k, "gpu", total[k], "oracle", ref, "one ulp", ulp, flush=True)
        assert total[k] / ref - 1.0 <= bar + 2.0 * abs(ulp / ref - 1.0), k
    assert total["ncfn"] <= ost["ncfn"].sum() + bar * ost["nsetups"].sum()
    gpu, ulp = _units(Y, T, Yo, To), _units(Yp, Tp, Yo, To)
    assert np.median(gpu) <= 2.0 * np.median(ulp) + (10.0 if f32 else 5.0)


def test_lds_of_one_wavefront_fp32(torch_gpu, tmp_path):
    """40 species and 600 reactions: CvUni (432 bytes), the 41 x 41 FP32 matrix (6,736), the
    column factors (512) and 2 x 41 + 1,201 doubles of RHS arrays (10,264) are 17,944
    bytes and, with the flag, under a compute unit's 160 KB / 8, so 8 reactors (two a
    SIMD) are in flight on each compute unit."""
    from zerork_hip import capi
    files, _ = _generated(tmp_path, 40, 600, (0.06, 0.04))
    m = capi.Mech(*files)
    print("case LDS of 40 species, 600 reactions", flush=True)
    cus = torch_gpu.cuda.get_device_properties(0).multi_processor_count
    assert m.nstep == 1200
    assert m.resident_waves(capi.default_options(fp32_preconditioner=1)) == 8 * cus
