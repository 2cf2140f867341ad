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


@pytest.mark.parametrize("n,n_hw,jobs", [(4, 1, "hall"), (4, 3, "hall"), (24, 1, "hall"), (24, 1, "kubo"),
                                         (20, 300, "hall"), (40, 1, "hall"), (40, 5, "hall")])
def test_the_order_that_is_not_in_resonance(n, n_hw, jobs):
    """General V with P_ij and P_ji of different sizes, at a resonance 1e-8 wide:
    every element by itself.  One pair has a velocity, so an element holds the two
    orders of that pair and nothing else."""
    import oracle as O
    from mepinterp_amd import capi, models
    m = models.make_random(seed=n, n=n, L=1)
    e, x, y, eta = 0.25 * np.arange(n), 1, 3, 1e-8
    hw = np.linspace(0.5, 2.0, n_hw)  # the first one is the pair's gap
    V = np.zeros((3, n, n), np.complex128, order="F")
    V[:, y, x] = 1.0 + 0.3j, 1e-9 * (0.5 - 0.7j), 1e-4 * (0.2 + 1.1j)
    V[:, x, y] = 1e-9 * (0.9 + 0.2j), 0.8 - 0.5j, 1e-5 * (1.0 + 0.6j)
    fd = np.asfortranarray(np.linspace(0.9, 0.2, n)[None])
    p = capi.Engine.params(jobs=capi.MEP_JOB_AHC | (capi.MEP_JOB_KUBO if jobs == "kubo" else 0),
                           hw_lst=hw, eta=eta)
    with capi.Engine(m["R_frac"], m["H"], a_latt=m["a_latt"]) as eng:
        g = eng.bandsum(e, V[..., None], p, fd=fd)
    ref = O.kubo_ohc_tens(e, V, hw, fd, eta).reshape(g["ohc"].shape, order="F")
    assert np.all(ref != 0)
    # about 30 roundings of 1.1e-16 on the way to an element
    assert np.all(np.abs(g["ohc"] - ref) <= 4e-15 * np.abs(ref))
