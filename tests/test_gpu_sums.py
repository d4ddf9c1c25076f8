"""Sums over the k points of a wave (wave_sum8) and the factored time sample of the fixed-step
2-band kernels, at k counts around a wave: one lane, one short of a wave, a wave, one more, and a
second block. Against the oracle within 1e-10 (the bar of the FP64 path); the FP32 state's
sums over whole grids have their own tests."""
import numpy as np
import pytest

from antelope_amd import Pulse, SBESolver
from tests.cases import haldane_cfg1_model, rel_l2, small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1), (9, 7), (8, 8), (13, 5), (43, 6)])
@pytest.mark.parametrize("gauge,rk,inter_intra", [
    ("LengthWannier", 4, True), ("LengthWannier", 5, False), ("VelocityHamiltonian", 4, False),
    ("VelocityHamiltonian", 5, True)])
def test_wave_sums(oracle, n, gauge, rk, inter_intra):
    # the Monkhorst-Pack grid, off Gamma
    cfg = small_config(n=n, ncycles=1.0, rk=rk, inter_intra=inter_intra, ellip=0.4,
                       grid="mp", T1=300.0, gauge=gauge)
    model = haldane_cfg1_model()
    print("case:", n, gauge, rk, inter_intra, flush=True)
    ref = oracle.run(cfg, model, nthreads=4)
    with SBESolver(cfg, model) as s:
        s.run()
        got = s.series()
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar"):
        if np.linalg.norm(ref[key]) > 0:
            assert rel_l2(got[key], ref[key]) < 1e-10, key
        else:
            assert not np.any(got[key]), key


def test_velocity_sums_by_matrix_pipe():
    """k blocks of a grid against the whole of it, the same sums to rounding. (FP64 sums by swaps at any size; the FP32
    state's change of route is tested below.)"""
    cfg = small_config(n=(520, 505), ncycles=0.02, rk=4, ellip=0.4, grid="mp", T1=300.0, gauge="VelocityHamiltonian")
    model = haldane_cfg1_model()
    nk, cut = 520 * 505, 100000

    def run(a, b):
        with SBESolver(cfg, model, a, b) as s:
            s.run()
            return s.series()

    whole, parts = run(-1, -1), [run(0, cut), run(cut, nk)]
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar"):
        assert rel_l2(parts[0][key] + parts[1][key], whole[key]) < 1e-10, key


@pytest.mark.parametrize("rk,T1", [(4, 0.0), (5, 300.0)])
@pytest.mark.parametrize("kpt", [1, 2])
def test_velocity_fp32_sums_by_matrix_pipe(monkeypatch, rk, T1, kpt):
    """With FP32 state the velocity gauge's sums take the matrix pipe from 2560 waves up: a whole grid above it against
    its k blocks below, which use swaps. Both add the same FP64 values, in another order: 1e-12 of the largest."""
    n = (500, 440) if kpt == 1 else (800, 550)
    nk, cut = n[0] * n[1], 160000 if kpt == 1 else 315000
    waves = lambda k: -(-k // (256 * kpt)) * 4  # noqa: E731  (blocks of four waves, kpt k points per lane)
    assert waves(nk) >= 2560 > max(waves(cut), waves(nk - cut))
    monkeypatch.setenv("ANTELOPE_HALDANE_KPT", str(kpt))
    cfg = small_config(n=n, ncycles=0.02, rk=rk, ellip=0.4, grid="mp", T1=T1, gauge="VelocityHamiltonian", precision="fp32")
    model = haldane_cfg1_model()
    print("fp32 velocity sums:", rk, T1, kpt, flush=True)

    def run(a, b):
        with SBESolver(cfg, model, a, b) as s:
            s.run()
            return s.series()

    whole, parts = run(-1, -1), [run(0, cut), run(cut, nk)]
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar"):
        a, b = parts[0][key] + parts[1][key], whole[key]
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max(), key


@pytest.mark.parametrize("gauge,rk,precision", [("LengthWannier", 4, "fp64"), ("LengthWannier", 5, "fp32"),
                                                ("VelocityHamiltonian", 5, "fp64"), ("VelocityHamiltonian", 4, "fp32")])
def test_nine_pulses(oracle, gauge, rk, precision):
    """More pulses than the laser-row kernel's arguments hold: the rows come from the host. FP64 against the oracle
    (1e-10), FP32 state within 6e-5 of it (the bar of the FP32 forms)."""
    cfg = small_config(n=(9, 8), ncycles=1.0, rk=rk, inter_intra=True, ellip=0.4, grid="mp", T1=300.0, gauge=gauge,
                       precision=precision)
    one = cfg.pulses[0]
    cfg.pulses = [Pulse(E0=one.E0 / (1 + i), w0=one.w0 * (1 + 0.05 * i), ncycles=1.0, ellip=0.1 * i, cep=0.2 * i, envelope="sin2")
                  for i in range(9)]
    model = haldane_cfg1_model()
    print("nine pulses:", gauge, rk, precision, flush=True)
    ref = oracle.run(cfg, model, nthreads=4)
    with SBESolver(cfg, model) as s:
        s.run()
        got = s.series()
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar"):
        assert rel_l2(got[key], ref[key]) < (1e-10 if precision == "fp64" else 6e-5), key
