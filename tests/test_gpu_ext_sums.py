"""The optical, photogalvanic and gyrotropic kernels at the edges of their
tiles and item splits against the oracle: one band to 32 bands (one and four
16 x 16 tiles), one item, a number of items that leaves threads over, more
than the 256 of one pass, many Fermi levels, with and without a position
operator, with weights."""
import numpy as np
import pytest

from conftest import oracle_model, rand_kpts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_eF,n_hw,with_r,T", [
    (1, 1, 1, True, 300.0), (2, 3, 2, True, 300.0), (15, 1, 1, True, 0.0), (16, 2, 8, True, 300.0),
    (16, 1, 300, False, 300.0), (17, 2, 130, True, 300.0), (31, 7, 3, True, 300.0),
    (32, 1, 5, True, 0.0), (32, 60, 1, True, 300.0), (72, 30, 1, False, 300.0), (33, 2, 3, True, 300.0)])
def test_ext_sums_at_tile_and_item_edges(n, n_eF, n_hw, with_r, T):
    import oracle as O
    from mepinterp_amd import capi, models
    m = models.make_random(seed=700 + n, n=n, L=1, with_r=with_r)
    k = rand_kpts(6, seed=n + n_hw)
    w = np.random.default_rng(n).uniform(0.5, 2.0, size=k.shape[1])
    kw = dict(n_eF=n_eF, eF_min=-0.02, eF_max=0.02, n_hw=n_hw, hw_min=0.01, hw_max=0.07,
              T_kelvin=T, eta=0.004, valence_bands=1)
    jobs = capi.MEP_JOB_OPT | capi.MEP_JOB_GYRO
    with capi.Engine(m["R_frac"], m["H"], r=m["r"], a_latt=m["a_latt"]) as eng:
        eng.set_kblock(64)
        g = eng.run_kpts(k, capi.Engine.params(jobs=jobs, **kw), weights=w)
    om, p = oracle_model(m), O.RunParams(do_opt=True, do_gyro=True, **kw)
    o = {}
    for q in range(k.shape[1]):
        one = O.accumulate(om, p, np.asfortranarray(k[:, q:q + 1]))
        for key in ("opt_s", "opt_a", "photo", "gyro_C", "gyro_D", "gyro_Dw"):
            o[key] = o.get(key, 0.0) + w[q] * np.asarray(one[key])
    for key, ref in o.items():
        scale = np.max(np.abs(ref))
        err = np.max(np.abs(g[key] - ref))
        # 1e-9, the sums' tolerance (n = 1 has no pairs: zero on both sides)
        assert err <= 1e-9 * scale, (key, err, scale)


@pytest.mark.parametrize("n", [40, 41, 48, 49])
def test_ext_sums_at_the_edges_of_the_register_ql(n):
    """Eigenvalues by QL in registers (two widths) and in LDS columns.  The
    frequencies lie above every gap, so no unbroadened pole is near."""
    import oracle as O
    from mepinterp_amd import capi, models
    m = models.make_random(seed=60 + n, n=n, L=1, with_r=True)
    k = rand_kpts(70, seed=n)  # more than the 64 k-points of a workgroup
    width = 2.0 * np.max(np.sum(np.abs(m["H"]), axis=(1, 2)))  # of the spectrum, at most
    kw = dict(n_eF=2, eF_min=-0.02, eF_max=0.02, n_hw=2, hw_min=width, hw_max=2.0 * width,
              T_kelvin=300.0, eta=0.004, valence_bands=1)
    with capi.Engine(m["R_frac"], m["H"], r=m["r"], a_latt=m["a_latt"]) as eng:
        g = eng.run_kpts(k, capi.Engine.params(jobs=capi.MEP_JOB_OPT, **kw))
    o = O.accumulate(oracle_model(m), O.RunParams(do_opt=True, **kw), k)
    for key in ("opt_s", "opt_a", "photo"):
        # 1e-9, the sums' tolerance
        assert np.max(np.abs(g[key] - o[key])) <= 1e-9 * np.max(np.abs(o[key])), key


@pytest.mark.parametrize("n,most", [(16, 182), (32, 81), (33, 45)])
def test_as_many_fermi_levels_as_the_tables_take(n, most):
    import oracle as O
    from mepinterp_amd import capi, models
    m = models.make_random(seed=90 + n, n=n, L=1, with_r=True)
    k = rand_kpts(2, seed=n)
    width = 2.0 * np.max(np.sum(np.abs(m["H"]), axis=(1, 2)))  # above every gap: no pole near
    kw = dict(eF_min=-0.05, eF_max=0.05, n_hw=1, hw_min=width, hw_max=width, T_kelvin=300.0,
              eta=0.004, valence_bands=1)
    jobs = capi.MEP_JOB_OPT | capi.MEP_JOB_GYRO
    with capi.Engine(m["R_frac"], m["H"], r=m["r"], a_latt=m["a_latt"]) as eng:
        g = eng.run_kpts(k, capi.Engine.params(jobs=jobs, n_eF=most, **kw))
        with pytest.raises(capi.MepError):
            eng.run_kpts(k, capi.Engine.params(jobs=jobs, n_eF=most + 1, **kw))
    o = O.accumulate(oracle_model(m), O.RunParams(do_opt=True, do_gyro=True, n_eF=most, **kw), k)
    for key in ("opt_s", "opt_a", "photo", "gyro_C", "gyro_D"):
        # 1e-9, the sums' tolerance
        assert np.max(np.abs(g[key] - o[key])) <= 1e-9 * np.max(np.abs(o[key])), key
