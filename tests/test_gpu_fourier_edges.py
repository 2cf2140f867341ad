"""The FP64 Fourier product at the edges of its tiles: k-point counts, column
counts and R-vector counts that end inside, on and past a tile of 128 or a
chunk of 16, against the oracle's H(k) and dH(k) through the eigenvalues and the
cartesian velocities."""
import numpy as np
import pytest

from conftest import oracle_model, rand_kpts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,L", [(1, 0), (1, 1), (3, 1), (4, 2), (5, 1), (6, 2), (8, 1), (11, 1)])
def test_fourier_product_edges(n, L):
    from mepinterp_amd import capi, models
    import oracle as O
    m = models.make_random(seed=7 + n, n=n, L=L)
    om = oracle_model(m, do_gauge_trafo=False)
    k = rand_kpts(257, seed=n)
    with capi.Engine(m["R_frac"], m["H"], a_latt=m["a_latt"], gauge_trafo=False) as eng:
        for nk in (1, 127, 128, 129, 257):
            e, V = eng.interp(np.asfortranarray(k[:, :nk]))[:2]
            for i in {0, nk - 1, nk // 2}:
                eo, Vo = O.get_wann_interp(om, k[:, i])[:2]
                # FP64 sums of at most a few hundred terms on both sides
                assert np.max(np.abs(e[:, i] - eo)) <= 1e-12 * np.max(np.abs(eo))
                assert np.max(np.abs(V[..., i] - Vo)) <= 1e-12 * max(np.max(np.abs(Vo)), 1e-3)
