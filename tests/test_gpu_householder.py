"""The Householder kernels above 32 bands at the edges of their ranges and of
their register tiles (chunks of four columns that end in, on and past the
matrix), with and without centres, every variant against the oracle: energies
and velocities."""
import numpy as np
import pytest

from conftest import oracle_model, rand_kpts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tb", [(33, True), (34, False), (35, False), (44, True), (45, False), (47, False),
                                  (48, True), (49, False), (61, True), (64, False), (65, False), (72, False),
                                  (73, True), (80, False), (95, False), (96, True), (113, False)])
@pytest.mark.parametrize("variant", [0, 3])
def test_householder_variants_match_oracle(n, tb, variant):
    import oracle as O
    from mepinterp_amd import capi, models
    m = models.make_random(seed=20 + n, n=n, L=1, tb=tb)
    om = oracle_model(m)
    k = rand_kpts(4, seed=n)
    with capi.Engine(m["R_frac"], m["H"], wf_centers=m["wf_centers"], a_latt=m["a_latt"]) as eng:
        eng.set_variant(capi.MEP_VAR_EIGH, variant)
        e, V = eng.interp(k)[:2]
    for ik in range(4):
        eo, Vo = O.get_wann_interp(om, k[:, ik])[:2]
        # FP64 on both sides; eigenvectors divide by gaps down to 1e-4 of the spectrum
        assert np.max(np.abs(e[:, ik] - eo)) < 1e-12 * np.max(np.abs(eo))
        assert np.max(np.abs(V[..., ik] - Vo)) < 1e-10 * np.max(np.abs(Vo))


@pytest.mark.parametrize("n,tb", [(33, True), (35, False), (48, True), (49, False), (64, True), (65, False), (128, False)])
@pytest.mark.parametrize("variant", [1, 2])
def test_householder_in_lds_matches_oracle(n, tb, variant):
    """The matrix in a workgroup's LDS (1) and in one wavefront's (2, which above
    64 bands is 1)."""
    test_householder_variants_match_oracle(n, tb, variant)
