"""Time-fused steps of the analytic classes (nb_evolve_kernel) where its tiling can go wrong: one to
eight bands, k counts around the four-per-wave and block limits, RK4 and RK5, each decay setting, a
Fermi start, k blocks and runs split into parts. Against the oracle within 1e-10 (the bar of the
N-band paths) and the same against the separate kernels; split runs give the same bits. The grids keep
off points where two bands meet exactly (Gamma for the transition-metal and Kane-Mele classes, the line k_x = 0 with
spin-orbit, planes through Gamma for WDSM_TaAs): there the band basis, and so the dephasing and the band populations,
is the eigensolver's choice and the two paths differ with rounding / gap."""
import ctypes as C

import numpy as np
import pytest

from antelope_amd import AnalyticModel, Pulse, RunConfig, SBESolver, query_footprint, tmdc
from antelope_amd.models import synthetic_wannier
from tests.cases import rel_l2, small_config

pytestmark = pytest.mark.gpu


def _models():
    return {
        "wilson": AnalyticModel.from_reference("WilsonMass", t=0.02, delta=0.03, mu=-0.015, a0=4.0, a1=5.5),
        "mos2": tmdc("MoS2"),
        "kanemele": AnalyticModel.from_reference("KaneMele", t1=0.075, t2=0.025, tR=0.01, Mt2=1.5, phi0=0.9, a0=1.42),
        "wdsm": AnalyticModel.from_reference("WDSM_TaAs", t=0.02, delta=0.5, my=0.8, mz=0.9, a0=3.4),
        "wse2_soc": tmdc("WSe2", soc=True),
    }


def _run(cfg, m, cuts=(), **kw):
    with SBESolver(cfg, m, **kw) as s:
        for c in cuts:
            s.run(s.info.steps_done, c)
        s.run()
        out = s.series()
        out["state"] = s.state()
        return out


CASES = [
    # name, k grid, tableau, T1, T2, init
    ("wilson", (1, 1), 4, 0.0, 0.0, "uniform"),
    ("wilson", (3, 1), 5, 120.0, 90.0, "uniform"),
    ("mos2", (5, 2), 4, 0.0, 150.0, "uniform"),
    ("mos2", (17, 2), 5, 200.0, 0.0, "fermi"),
    ("kanemele", (4, 4), 5, 150.0, 150.0, "uniform"),
    ("kanemele", (9, 8), 4, 300.0, 150.0, "uniform"),
    ("wdsm", (4, 4, 2), 5, 0.0, 150.0, "uniform"),
    ("wse2_soc", (2, 1), 5, 0.0, 0.0, "uniform"),
    ("wse2_soc", (4, 2), 4, 200.0, 100.0, "fermi"),
    ("wse2_soc", (6, 1), 5, 0.0, 100.0, "uniform"),
]


@pytest.mark.parametrize("name,n,rk,T1,T2,init", CASES)
def test_evolve(oracle, monkeypatch, name, n, rk, T1, T2, init):
    m = _models()[name]
    cfg = small_config(n=n, ncycles=0.5, ellip=0.3, rk=rk, T1=T1, T2=T2, grid="mp", init=init, fermi_energy=0.02)
    print(name, n, rk, flush=True)
    ref = oracle.run(cfg, m, nthreads=8, want_state=True)
    got = _run(cfg, m)
    split = _run(cfg, m, cuts=(1, 2, 130))
    with monkeypatch.context() as mp:
        mp.setenv("ANTELOPE_NB_FUSED", "0")
        sep = _run(cfg, m)
        foot_sep = query_footprint(cfg, m)
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar", "state"):
        assert np.array_equal(got[key], split[key]), key
        if np.linalg.norm(ref[key]) == 0.0:
            continue
        e, es = rel_l2(got[key], ref[key]), rel_l2(got[key], sep[key])
        print(f"  {key}: oracle {e:.1e}, separate kernels {es:.1e}", flush=True)
        assert e < 1e-10 and es < 1e-10, key
    assert query_footprint(cfg, m) != foot_sep
    with SBESolver(cfg, m) as s:
        assert s.info.device_bytes == query_footprint(cfg, m)


def test_evolve_k_blocks(oracle):
    """Two k blocks' sums add up to the whole grid's."""
    m = _models()["kanemele"]
    cfg = small_config(n=(5, 6), ncycles=0.5, ellip=0.3, rk=5, T2=150.0, grid="mp")
    whole = _run(cfg, m)
    a, b = _run(cfg, m, k_begin=0, k_end=11), _run(cfg, m, k_begin=11, k_end=30)
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar"):
        assert rel_l2(a[key] + b[key], whole[key]) < 1e-11, key


BOX_CASES = [
    # bands, R range, k grid, tableau, T1, T2, InterIntra
    (1, (1, 1, 0), (7, 6, 1), 4, 0.0, 80.0, True),
    (2, (1, 1, 0), (512, 2, 1), 5, 150.0, 80.0, True),  # RK5 scratch in the stage-derivative slots
    (3, (2, 2, 1), (5, 4, 3), 5, 0.0, 80.0, True),
    (4, (3, 1, 0), (13, 6, 1), 4, 120.0, 60.0, True),
    (4, (1, 2, 1), (4, 7, 4), 5, 0.0, 0.0, False),
    (5, (3, 2, 0), (9, 11, 1), 5, 90.0, 90.0, True),
    (7, (2, 1, 1), (6, 5, 3), 4, 0.0, 0.0, True),
    (8, (2, 2, 0), (14, 11, 1), 5, 200.0, 80.0, True),
]


@pytest.mark.parametrize("N,nmax,npts,rk,T1,T2,ii", BOX_CASES)
def test_box_evolve(oracle, monkeypatch, N, nmax, npts, rk, T1, T2, ii):
    """Wannier models with N <= 8 (nb_box_evolve_kernel), positions not Hermitian (H~ = H + E.D is
    used as a general matrix), against the oracle, the separate kernels, split runs and k blocks."""
    m = synthetic_wannier(N, nmax=nmax, seed=70 + N)
    m.pos = m.pos * (1.0 + 0.3j)
    cfg = RunConfig(npoints=list(npts), pulses=[Pulse(E0=0.01, w0=0.05, ncycles=0.25, ellip=0.4, envelope="sin2")],
                    dt=0.5, T1=T1, T2=T2, rk_order=rk, inter_intra=ii)
    print(N, nmax, npts, rk, flush=True)
    ref = oracle.run(cfg, m, nthreads=8, want_state=True)
    got = _run(cfg, m)
    split = _run(cfg, m, cuts=(1, 2, 40))
    nk = int(np.prod(npts))
    cut = nk // 2 + 1
    blocks = [_run(cfg, m, k_begin=a, k_end=b) for a, b in ((0, cut), (cut, nk))]
    with monkeypatch.context() as mp:
        mp.setenv("ANTELOPE_NB_EVAL_STEPS", "3")
        three = _run(cfg, m)
        mp.setenv("ANTELOPE_NB_FUSED", "0")
        sep = _run(cfg, m)
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar", "state"):
        assert np.array_equal(got[key], split[key]), key
        assert np.array_equal(got[key], three[key]), key
        if np.linalg.norm(ref[key]) == 0.0:
            continue
        e, es = rel_l2(got[key], ref[key]), rel_l2(got[key], sep[key])
        print(f"  {key}: oracle {e:.1e}, separate kernels {es:.1e}", flush=True)
        assert e < 1e-10 and es < 1e-10, key
        if key != "state":
            assert rel_l2(blocks[0][key] + blocks[1][key], ref[key]) < 1e-10, key
    with SBESolver(cfg, m) as s:
        assert s.info.device_bytes == query_footprint(cfg, m)


@pytest.mark.parametrize("N,nmax,npts,T2,ii", [
    (9, (0, 1, 0), (3, 5, 1), 80.0, True),     # too few k points for the separable sums: the separate kernels
    (12, (1, 1, 0), (4, 4, 1), 80.0, False),   # (these two against the oracle)
    (9, (0, 2, 0), (5, 9, 1), 80.0, True),     # one lattice vector along a1, a block not full
    (12, (1, 1, 0), (7, 7, 1), 80.0, False),
    (13, (2, 0, 1), (5, 2, 2), 0.0, True),     # three chunks of a staged row
    (16, (3, 1, 0), (9, 3, 1), 80.0, True),    # seven lattice vectors, three blocks a column
])
def test_step_blocks(oracle, monkeypatch, N, nmax, npts, T2, ii):
    """Blocks of four k points and the staged rows of the 9..16-band step (nb16_step_kernel), against the
    oracle and the separate kernels."""
    m = synthetic_wannier(N, nmax=nmax, seed=90 + N)
    cfg = RunConfig(npoints=list(npts), pulses=[Pulse(E0=0.01, w0=0.05, ncycles=0.25, ellip=0.4, envelope="sin2")],
                    dt=0.5, T2=T2, rk_order=4, inter_intra=ii)
    print(N, nmax, npts, flush=True)
    ref = oracle.run(cfg, m, nthreads=8, want_state=True)
    got, foot = _run(cfg, m), query_footprint(cfg, m)
    with monkeypatch.context() as mp:
        mp.setenv("ANTELOPE_NB_FUSED", "0")
        sep = _run(cfg, m)
        assert (foot != query_footprint(cfg, m)) == (npts not in ((3, 5, 1), (4, 4, 1)))  # the plan that ran
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar", "state"):
        if np.linalg.norm(ref[key]) > 0.0:
            assert rel_l2(got[key], ref[key]) < 1e-10 and rel_l2(got[key], sep[key]) < 1e-10, key


@pytest.mark.parametrize("N,nmax,npts,T1,T2,ii", [
    (9, (0, 1, 0), (3, 5, 1), 0.0, 80.0, True),      # as above: the separate kernels
    (12, (1, 1, 0), (4, 4, 1), 120.0, 80.0, False),
    (9, (0, 2, 0), (5, 9, 1), 0.0, 80.0, True),
    (12, (1, 1, 0), (7, 7, 1), 120.0, 80.0, False),
    (13, (2, 0, 1), (5, 2, 2), 0.0, 0.0, True),
    (16, (3, 1, 0), (9, 3, 1), 150.0, 80.0, True),
    (16, (1, 1, 0), (64, 8, 1), 0.0, 80.0, True),  # scratch in the stage-derivative slots
])
def test_step_rk5(oracle, monkeypatch, N, nmax, npts, T1, T2, ii):
    """RK5 steps of 9 to 16 bands (nb16_step_kernel<5>), positions not Hermitian (H~ = H + E.D is used as a
    general matrix), against the oracle, the separate kernels, split runs and k blocks."""
    m = synthetic_wannier(N, nmax=nmax, seed=110 + N)
    m.pos = m.pos * (1.0 + 0.3j)
    cfg = RunConfig(npoints=list(npts), pulses=[Pulse(E0=0.01, w0=0.05, ncycles=0.125, ellip=0.4, envelope="sin2")],
                    dt=0.5, T1=T1, T2=T2, rk_order=5, inter_intra=ii)
    print(N, nmax, npts, flush=True)
    ref = oracle.run(cfg, m, nthreads=8, want_state=True)
    got = _run(cfg, m)
    split = _run(cfg, m, cuts=(1, 2, 17))
    nk = int(np.prod(npts))
    cut = nk // 2 + 1
    blocks = [_run(cfg, m, k_begin=a, k_end=b) for a, b in ((0, cut), (cut, nk))]
    with monkeypatch.context() as mp:
        mp.setenv("ANTELOPE_NB_EVAL_STEPS", "3")
        three = _run(cfg, m)
        mp.setenv("ANTELOPE_NB_FUSED", "0")
        sep = _run(cfg, m)
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar", "state"):
        assert np.array_equal(got[key], split[key]), key
        assert np.array_equal(got[key], three[key]), key
        if np.linalg.norm(ref[key]) == 0.0:
            continue
        e, es = rel_l2(got[key], ref[key]), rel_l2(got[key], sep[key])
        print(f"  {key}: oracle {e:.1e}, separate kernels {es:.1e}", flush=True)
        assert e < 1e-10 and es < 1e-10, key
        if key != "state":
            assert rel_l2(blocks[0][key] + blocks[1][key], ref[key]) < 1e-10, key
    with SBESolver(cfg, m) as s:
        assert s.info.device_bytes == query_footprint(cfg, m)


@pytest.mark.parametrize("what", ["positions", "both"])
@pytest.mark.parametrize("N,nmax,npts", [(9, (0, 2, 0), (5, 9, 1)), (12, (1, 1, 0), (7, 7, 1)), (16, (3, 1, 0), (9, 3, 1)),
                                         (17, (1, 1, 0), (4, 4, 1)), (32, (1, 1, 1), (3, 3, 3))])
def test_matrices_not_hermitian(oracle, monkeypatch, N, nmax, npts, what):
    """RK4 steps of 9 to 32 bands (nb16_step_kernel<4>, nb32_step_kernel) with matrices r(-R) != r(R)^dag, and H
    too by a thousandth (its Hermitian part has the eigenvectors, the commutator takes all of it): the oracle's and the
    separate kernels' results, as every other route gives them."""
    m = synthetic_wannier(N, nmax=nmax, seed=130 + N)
    m.pos = m.pos * (1.0 + 0.3j)
    if what == "both":
        rng = np.random.default_rng(N)
        m.ham = m.ham + 1e-3 * np.abs(m.ham).max() * rng.normal(size=m.ham.shape)
    cfg = RunConfig(npoints=list(npts), pulses=[Pulse(E0=0.01, w0=0.05, ncycles=0.25, ellip=0.4, envelope="sin2")],
                    dt=0.5, T1=150.0, T2=80.0, rk_order=4, inter_intra=True)
    print(N, nmax, npts, what, flush=True)
    got, foot = _run(cfg, m), query_footprint(cfg, m)
    with monkeypatch.context() as mp:
        mp.setenv("ANTELOPE_NB_FUSED", "0")
        sep = _run(cfg, m)
        assert foot != query_footprint(cfg, m)  # the fused step's plan was the one that ran
    ref = oracle.run(cfg, m, nthreads=8, want_state=True) if what == "positions" else sep
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar", "state"):
        if np.linalg.norm(ref[key]) > 0.0:
            print(f"  {key}: {rel_l2(got[key], ref[key]):.1e} {rel_l2(got[key], sep[key]):.1e}", flush=True)
            assert rel_l2(got[key], ref[key]) < 1e-10 and rel_l2(got[key], sep[key]) < 1e-10, key


@pytest.mark.parametrize("N,npts,nmax", [(8, (5, 5, 3), (1, 1, 1)), (16, (6, 5, 1), (2, 2, 0))])
def test_refined_eigenvectors_hold_rounding(oracle, N, npts, nmax):
    """The refinement may end only where what it leaves off the diagonal is below rounding also between
    bands whose gap is a hundredth of the largest: the intraband current, which the k sum nearly cancels and
    which is first order in the eigenvectors' error, within 200 roundings (4.5e-14; 6e-15 reached, 2e-13 where a
    round from max|K| = 1e-5 was the last)."""
    m = synthetic_wannier(N, nmax=nmax, seed=40 + N)
    cfg = RunConfig(npoints=list(npts), pulses=[Pulse(E0=0.01, w0=0.05, ncycles=0.5, ellip=0.4, envelope="sin2")],
                    dt=0.5, T2=80.0, rk_order=4, inter_intra=True)
    print(N, npts, flush=True)
    ref = oracle.run(cfg, m, nthreads=8)
    got = _run(cfg, m)
    e = {key: rel_l2(got[key], ref[key]) for key in ("j_inter", "j_intra", "band_pop", "rho_bar")}
    print({k: f"{v:.1e}" for k, v in e.items()}, flush=True)
    assert all(v < 200 * 2.0**-52 for v in e.values()), e


@pytest.mark.parametrize("N,npts,rk,T1,T2,ii", [
    (1, (5, 1, 1), 5, 0.0, 80.0, True),
    (3, (3, 3, 1), 4, 120.0, 80.0, False),
    (4, (17, 1, 1), 5, 120.0, 80.0, True),
    (5, (3, 1, 1), 4, 0.0, 0.0, True),
    (8, (3, 3, 1), 5, 0.0, 80.0, True),
    (9, (5, 1, 1), 5, 120.0, 80.0, False),
    (16, (3, 3, 1), 5, 0.0, 80.0, True),
])
def test_velocity_evolve(oracle, monkeypatch, N, npts, rk, T1, T2, ii):
    """Time-fused velocity-gauge steps (nb_vel_fused_kernel) on each tile size and tableau."""
    m = synthetic_wannier(N, nmax=(1, 1, 0), seed=50 + N)
    cfg = RunConfig(npoints=list(npts), pulses=[Pulse(E0=0.01, w0=0.05, ncycles=0.5, ellip=0.4, envelope="sin2")],
                    dt=0.5, T1=T1, T2=T2, rk_order=rk, inter_intra=ii, gauge="VelocityHamiltonian")
    print(N, npts, rk, flush=True)
    ref = oracle.run(cfg, m, nthreads=8)
    got, split = _run(cfg, m), _run(cfg, m, cuts=(1, 2, 40))
    with monkeypatch.context() as mp:
        mp.setenv("ANTELOPE_NB_FUSED", "0")
        sep = _run(cfg, m)
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar", "state"):
        assert np.array_equal(got[key], split[key]), key
        assert rel_l2(got[key], sep[key]) < 1e-12, key
        if key != "state":
            assert rel_l2(got[key], ref[key]) < 1e-10, key


@pytest.mark.parametrize("N,rk", [(9, 4), (9, 5), (16, 4), (16, 5)])
def test_velocity_eight_wave_blocks(monkeypatch, N, rk):
    """Blocks of eight waves (9 to 16 bands from 2041 k points), the last one not full, against one launch per step.
    At 16 bands they take more LDS than a kernel gets unasked."""
    npts = (409, 5, 1)  # 2045
    assert (2045 + 7) // 8 >= 256 and 2045 % 8
    m = synthetic_wannier(N, nmax=(1, 1, 0), seed=150 + N)
    cfg = RunConfig(npoints=list(npts), pulses=[Pulse(E0=0.01, w0=0.05, ncycles=0.0625, ellip=0.4, envelope="sin2")],
                    dt=0.5, T1=120.0, T2=80.0, rk_order=rk, inter_intra=True, gauge="VelocityHamiltonian")
    print(N, rk, flush=True)
    got, foot = _run(cfg, m), query_footprint(cfg, m)
    with monkeypatch.context() as mp:
        mp.setenv("ANTELOPE_NB_FUSED", "0")
        sep = _run(cfg, m)
        assert foot != query_footprint(cfg, m)
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar", "state"):
        assert rel_l2(got[key], sep[key]) < 1e-12, key


@pytest.mark.parametrize("gauge,rk", [("LengthWannier", 4), ("VelocityHamiltonian", 5)])
def test_parted_series(oracle, gauge, rk):
    """Series from 1 MiB on come parted: rho's sums straight into the caller's array, the rest beside them, through the
    buffer of the partial sums. Read half way and at the end, and without rho's sums (whole rows)."""
    m = synthetic_wannier(8, nmax=(1, 1, 0), seed=160)
    cfg = RunConfig(npoints=[3, 3, 1], pulses=[Pulse(E0=0.01, w0=0.05, ncycles=4.0, ellip=0.4, envelope="sin2")],
                    dt=0.5, T2=80.0, rk_order=rk, inter_intra=True, gauge=gauge)
    print(gauge, rk, flush=True)
    ref = oracle.run(cfg, m, nthreads=8)
    with SBESolver(cfg, m) as s:
        nt = s.nt
        assert nt * (6 + 8 + 2 * 64) * 8 >= 1 << 20
        s.run(0, nt // 2)
        half = s.series()
        s.run()
        got, again = s.series(), s.series()
        rows = {"j_inter": np.zeros((nt, 3)), "j_intra": np.zeros((nt, 3)), "band_pop": np.zeros((nt, 8))}
        p = {k: v.ctypes.data_as(C.POINTER(C.c_double)) for k, v in rows.items()}
        assert s._lib.sbe_get_series(s._ctx, p["j_inter"], p["j_intra"], None, p["band_pop"]) == 0
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar"):
        assert rel_l2(got[key], ref[key]) < 1e-10, key
        assert np.array_equal(got[key], again[key]), key
        assert np.array_equal(half[key][: nt // 2], got[key][: nt // 2]), key
    for key in rows:
        assert np.array_equal(rows[key], got[key]), key
