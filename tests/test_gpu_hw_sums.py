"""The (hw, E_F) item sums of velo_ahc_tens and kubo_ohc_tens against the
oracle: one and four items a thread, fewer items than threads, more than one
pass of 1,024 items, pair counts below, at and above a chunk of 256, a
position operator (general V) and frequencies at the band gaps with a small
broadening."""
import numpy as np
import pytest

from conftest import oracle_model, rand_kpts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_hw,n_eF,pos", [
    (2, 2, 1, False), (5, 7, 1, False), (8, 8, 1, False), (12, 5, 3, False), (23, 64, 1, False),
    (24, 1, 4, False), (33, 130, 2, False), (40, 300, 4, False), (64, 3, 5, False),
    (3, 2, 1, True), (17, 6, 2, True), (23, 70, 4, True), (34, 3, 3, True), (36, 1, 1, True)])
@pytest.mark.parametrize("eta", [1e-6, 0.004])
def test_item_sums_match_oracle(n, n_hw, n_eF, pos, eta):
    import oracle as O
    from mepinterp_amd import capi, models
    m = models.make_random(seed=300 + n, n=n, L=1, with_r=pos, tb=pos)
    om = oracle_model(m)
    k = rand_kpts(4, seed=n)
    kw = dict(n_eF=n_eF, eF_min=-0.02, eF_max=0.02, n_hw=n_hw, hw_min=0.003, hw_max=0.09,
              T_kelvin=300.0, eta=eta, valence_bands=max(1, n // 2))
    with capi.Engine(m["R_frac"], m["H"], r=m["r"], wf_centers=m["wf_centers"],
                     a_latt=m["a_latt"]) as eng:
        w = np.array([0.7, 1.0, 0.25, 2.0])
        g = eng.run_kpts(k, capi.Engine.params(jobs=capi.MEP_JOB_AHC, **kw), weights=w)
    ref = None
    for i in range(4):
        o = O.accumulate(om, O.RunParams(do_ahc=True, **kw), k[:, i:i + 1])
        ref = {q: w[i] * o[q] + (ref[q] if ref else 0) for q in ("ahc_velo", "ohc")}
    for q in ("ahc_velo", "ohc"):
        # 1e-9, the sums' tolerance; a resonance 1e-6 wide amplifies the
        # eigenvalues' 1e-15 by at most 1e9 where a gap meets a frequency
        # to that width, which these few points do to 1e-4 at the nearest
        assert np.max(np.abs(g[q] - ref[q])) < 1e-9 * np.max(np.abs(ref[q])), q
