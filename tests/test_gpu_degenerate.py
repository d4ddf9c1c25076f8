"""Bands that are degenerate at every k point: a model doubled by a spin that nothing couples to. The
state stays a product with the identity of the spin, so the band-diagonal part, the currents and the
populations do not depend on the basis the eigensolver takes in a pair, as long as its columns are
orthonormal eigenvectors: everything equals the single model's, which has no degeneracies. Tolerance
1e-11 (the bar of the N-band paths, 1e-10, and a tenth of it); a non-unitary basis shows above 1e-3."""
import numpy as np
import pytest

from antelope_amd import Pulse, RunConfig, SBESolver
from antelope_amd.models import synthetic_wannier
from antelope_amd.params import WannierModel
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu


def _doubled(m):
    """m with a spin, in orbitals mixed by a random unitary V (else the pairs would be separate by exact zeros):
    the model and V."""
    n, rng = 2 * m.nband, np.random.default_rng(5)
    V = np.linalg.qr(rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n)))[0]
    mix = lambda X: V @ np.kron(X, np.eye(2)) @ V.conj().T  # noqa: E731
    ham = np.array([mix(h) for h in m.ham])
    pos = np.array([[mix(p) for p in r] for r in m.pos])
    return WannierModel(lattice=m.lattice, rvec=m.rvec, rweight=m.rweight, ham=ham, pos=pos, nval=2 * m.nval), V


def _run(cfg, m):
    with SBESolver(cfg, m) as s:
        s.run()
        return s.series()


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("n,npts,rk", [(1, (9, 8, 1), 4), (2, (7, 6, 1), 5), (2, (9, 8, 1), 4), (4, (7, 6, 1), 4), (4, (7, 6, 1), 5),
                                       (5, (7, 6, 1), 5), (8, (8, 7, 1), 4), (8, (8, 7, 1), 5)])
def test_spin_doubled_wannier(monkeypatch, n, npts, rk, fused):
    single = synthetic_wannier(n, nmax=(1, 1, 0), seed=300 + n, onsite=0.3 if n > 1 else 0.0)
    cfg = RunConfig(npoints=list(npts), pulses=[Pulse(E0=0.01, w0=0.05, ncycles=0.5, ellip=0.4, envelope="sin2")],
                    dt=0.5, T1=150.0, T2=80.0, rk_order=rk, inter_intra=True)
    print("spin doubled:", n, npts, rk, fused, flush=True)
    one = _run(cfg, single)
    if not fused:
        monkeypatch.setenv("ANTELOPE_NB_FUSED", "0")
    model, V = _doubled(single)
    two = _run(cfg, model)
    for key in ("j_inter", "j_intra"):
        if np.linalg.norm(one[key]) > 0.0:
            assert rel_l2(two[key], 2.0 * one[key]) < 1e-11, key
    back = V.conj().T @ two["rho_bar"] @ V
    assert rel_l2(back, np.array([np.kron(r, np.eye(2)) for r in one["rho_bar"]])) < 1e-11
    # the populations of a pair together: which of its two columns ranks lower is rounding
    assert rel_l2(two["band_pop"].reshape(len(two["band_pop"]), n, 2).sum(-1), 2.0 * one["band_pop"]) < 1e-11
