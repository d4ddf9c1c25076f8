"""Sums over the k points of a wave (wave_sum8) and the factored time sample of the fixed-step
2-band kernels, at k counts around a wave: one lane, one short of a wave, a wave, one more, and a
second block. Against the oracle within 1e-10 (the bar of the FP64 path); the FP32 state's
sums over whole grids have their own tests."""
import numpy as np
import pytest

from antelope_amd import SBESolver
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
    """The velocity gauge's sums change route at 4096 waves (262144 k points): k blocks below it against the
    whole grid above, the same sums to rounding."""
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
