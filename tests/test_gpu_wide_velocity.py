"""The velocities above 32 bands without a position operator, at the edges of
their 16-band column tiles, element by element against the oracle: with and
without Wannier centres (whose phases go into dH before the products), an odd
and an even number of tiles (each tile pair is formed once), cartesian
velocities in the Wannier gauge, and more k-points than one round of eight."""
import numpy as np
import pytest

from conftest import oracle_model, rand_kpts

pytestmark = pytest.mark.gpu

CASES = [(n, tb, True) for n, tb in
         ((33, False), (47, True), (48, False), (49, True), (64, True), (65, False), (80, True),
          (81, False), (96, True), (97, True), (112, False), (113, False), (128, True))]
CASES += [(40, True, False), (72, False, False), (128, True, False)]


@pytest.mark.parametrize("n,tb,gauge", CASES)
def test_wide_velocities_match_oracle(n, tb, gauge):
    import oracle as O
    from mepinterp_amd import capi, models
    m = models.make_random(seed=70 + n, n=n, L=1, tb=tb)
    om = oracle_model(m, do_gauge_trafo=gauge)
    k = rand_kpts(11, seed=n)
    with capi.Engine(m["R_frac"], m["H"], wf_centers=m["wf_centers"], a_latt=m["a_latt"],
                     gauge_trafo=gauge) as eng:
        e, V = eng.interp(k)[:2]
        for ik in (0, 3, 7, 8, 10):
            eo, Vo = O.get_wann_interp(om, k[:, ik])[:2]
            # FP64 on both sides; the eigenvectors divide by gaps down to 1e-4 of
            # the spectrum
            assert np.max(np.abs(e[:, ik] - eo)) < 1e-12 * np.max(np.abs(eo))
            assert np.max(np.abs(V[..., ik] - Vo)) < 1e-10 * np.max(np.abs(Vo))
