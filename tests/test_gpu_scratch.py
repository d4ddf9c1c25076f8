"""Device memory of the time-fused N-band routes: a serving budget that holds a solve's plan on the separate kernels
admits it (with that plan where the faster one does not fit), and the analytic classes hold no slots that
their kernel does not touch."""
import math

import numpy as np
import pytest

from antelope_amd import Pulse, RunConfig, SBESolver, tmdc
from antelope_amd.models import synthetic_wannier
from antelope_amd.serve import SBEServer, ServingRequest, run_stream
from antelope_amd.solver import query_footprint
from tests.cases import rel_l2


def _config(npoints, nt, rk, **kw):
    return RunConfig(npoints=list(npoints), dt=0.25, rk_order=rk, T2=220.0, inter_intra=True,
                     pulses=[Pulse(E0=0.0045, w0=0.05, ncycles=nt * 0.25 * 0.05 / (2 * math.pi), ellip=0.4, envelope="sin2")], **kw)


@pytest.mark.parametrize("rk", [4, 5])
@pytest.mark.parametrize("n,nt", [((1, 1), 50), ((1, 1), 20000), ((6, 6), 2000), ((30, 30), 500), ((300, 300), 2000)])
def test_analytic_footprint(monkeypatch, n, nt, rk):
    """Against the separate kernels' plan: no more than a phase table of 256 steps (1,152 bytes each) above it."""
    cfg, m = _config(n, nt, rk, grid="mp"), tmdc("MoS2")
    fused = query_footprint(cfg, m)
    monkeypatch.setenv("ANTELOPE_NB_FUSED", "0")
    assert fused <= query_footprint(cfg, m) + 257 * 1152 + 16384


@pytest.mark.gpu
@pytest.mark.parametrize("cfg,N,nmax,budget", [
    # the bytes of the separate kernels' plan
    (_config((13, 13, 1), 50, 5), 8, (2, 2, 0), 12796128),
    (_config((24, 24, 1), 2000, 5, gauge="VelocityHamiltonian"), 8, (2, 2, 0), 144903456),
])
def test_budget_of_the_separate_kernels(monkeypatch, cfg, N, nmax, budget):
    m = synthetic_wannier(N, nmax=nmax, seed=11)
    assert query_footprint(cfg, m) > budget  # or this tests nothing
    print("budget:", cfg.gauge, budget, flush=True)
    with SBEServer(hbm_budget_bytes=budget, max_active=2) as srv:
        out = run_stream(srv, [ServingRequest(0.0, cfg, m, "request", int(np.prod(cfg.npoints)))], realtime=False, keep_results=True)
    assert out["completed"] == 1 and out["failed"] == 0
    got = out["records"][0]["series"]
    with SBESolver(cfg, m) as s:
        s.run()
        ref = s.series()
    for key in ref:
        assert rel_l2(got[key], ref[key]) < 1e-10, key


@pytest.mark.gpu
@pytest.mark.parametrize("n,rk,pulses", [((3, 2), 5, 1), ((3, 2), 4, 9), ((3, 2), 5, 9)])
def test_analytic_table_per_launch(oracle, n, rk, pulses):
    """More steps than a launch's phase table covers, and more pulses than its kernel takes (A from the host)."""
    cfg, m = _config(n, 700, rk, grid="mp"), tmdc("MoS2")
    one = cfg.pulses[0]
    cfg.pulses = [Pulse(E0=one.E0 / (1 + i), w0=one.w0, ncycles=one.ncycles / (1 + 0.1 * i), ellip=0.3, cep=0.2 * i, envelope="sin2")
                  for i in range(pulses)]
    print("table:", n, rk, pulses, flush=True)
    ref = oracle.run(cfg, m, nthreads=8)
    with SBESolver(cfg, m) as s:
        assert s.info.device_bytes == query_footprint(cfg, m) and s.nt > 2 * 256
        s.run()
        got = s.series()
    for key in ("j_inter", "j_intra", "band_pop", "rho_bar"):
        assert rel_l2(got[key], ref[key]) < 1e-10, key
