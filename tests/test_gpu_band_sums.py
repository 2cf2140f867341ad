"""The band sums against the oracle at the edges of their branches: k-points
whose Niu windows are all trivial (a small tolerance), some wide (the default)
and nearly everything excluded (a large one), one and four matrix tiles, the
last quarter of the band range present or not, above 32 bands odd and even
numbers of tiles, velocities formed in the kernel or read, general V, one and
several Fermi levels, and the pair sums at zero temperature, frequency and
broadening."""
import numpy as np
import pytest

from conftest import oracle_model, rand_kpts

pytestmark = pytest.mark.gpu

KEYS = ("Ne", "ahc", "ahc_velo", "ohc", "kubo_ic", "kubo_lc", "kubo_cs", "niu_ic", "niu_lc", "niu_cs")


@pytest.mark.parametrize("n,pos,tb,n_eF", [(2, False, False, 1), (9, False, True, 2), (16, False, False, 1),
                                           (17, False, False, 1), (24, False, True, 1), (25, False, False, 1),
                                           (32, False, False, 1), (32, False, False, 3), (7, True, False, 1),
                                           (24, True, True, 1), (25, True, False, 2), (32, True, False, 1),
                                           (33, False, False, 1), (48, False, True, 2), (65, False, False, 1),
                                           (100, False, False, 1), (36, True, False, 1)])
@pytest.mark.parametrize("tol", [1e-13, 1e-5, 3e-2])
def test_band_sums_match_oracle(n, pos, tb, n_eF, tol, n_val=None):
    import oracle as O
    from mepinterp_amd import capi, models
    m = models.make_random(seed=500 + n, n=n, L=1, with_r=pos, tb=tb)
    om = oracle_model(m, kubo_tol=tol)
    k = rand_kpts(5, seed=n)
    still = not pos and n_eF == 1
    kw = dict(n_eF=n_eF, eF_min=-0.01, eF_max=0.01, n_hw=1, hw_min=0.0 if still else 0.02,
              hw_max=0.0 if still else 0.02, T_kelvin=0.0 if still else 300.0,
              eta=0.0 if still else 0.002, valence_bands=n_val or max(1, n // 2))
    with capi.Engine(m["R_frac"], m["H"], r=m["r"], wf_centers=m["wf_centers"], a_latt=m["a_latt"],
                     kubo_tol=tol) as eng:
        g = eng.run_kpts(k, capi.Engine.params(
            jobs=capi.MEP_JOB_AHC | capi.MEP_JOB_KUBO | capi.MEP_JOB_MEP, **kw))
    o = O.accumulate(om, O.RunParams(do_ahc=True, do_kubo=True, do_mep=True, **kw), k)
    for q in KEYS:
        # 1e-9, the sums' tolerance (these gaps are 1e-3 and more)
        assert np.max(np.abs(g[q] - o[q])) <= 1e-9 * np.max(np.abs(o[q])), q


@pytest.mark.parametrize("n,pos,n_eF,n_hw", [
    (1, False, 1, 1), (2, True, 1, 1), (4, True, 1, 1), (8, True, 1, 1), (8, True, 2, 3), (16, True, 1, 1),
    (17, True, 1, 1), (23, True, 3, 1), (24, True, 4, 1), (24, True, 5, 1), (32, True, 1, 1), (32, True, 1, 4),
    (5, False, 1, 1), (16, False, 1, 1), (16, False, 4, 2), (20, False, 2, 1), (24, False, 1, 1)])
@pytest.mark.parametrize("T", [0.0, 300.0])
def test_hall_sums_alone_match_oracle(n, pos, n_eF, n_hw, T):
    """No magnetoelectric sums: as many k-points at a time as fill a workgroup
    (42 cannot be one k-point, 37 no multiple of any), one pair a thread or
    two rounds, up to four Fermi levels and more, weights."""
    import oracle as O
    from mepinterp_amd import capi, models
    m = models.make_random(seed=800 + n, n=n, L=1, with_r=pos)
    om = oracle_model(m)
    nk = 37
    k = rand_kpts(nk, seed=n)
    wt = np.random.default_rng(n).uniform(0.5, 2.0, size=nk)
    kw = dict(n_eF=n_eF, eF_min=-0.02, eF_max=0.02, n_hw=n_hw, hw_min=0.01, hw_max=0.05, T_kelvin=T,
              eta=0.003, valence_bands=1)
    with capi.Engine(m["R_frac"], m["H"], r=m["r"], a_latt=m["a_latt"]) as eng:
        g = eng.run_kpts(k, capi.Engine.params(jobs=capi.MEP_JOB_AHC, **kw), weights=wt)
    o = {}
    for i in range(nk):
        one = O.accumulate(om, O.RunParams(do_ahc=True, **kw), np.asfortranarray(k[:, i:i + 1]))
        for q in KEYS[:4]:
            o[q] = o.get(q, 0.0) + wt[i] * np.asarray(one[q])
    for q in KEYS[:4]:
        # 1e-9, the sums' tolerance
        assert np.max(np.abs(g[q] - o[q])) <= 1e-9 * np.max(np.abs(o[q])), q


@pytest.mark.parametrize("n,pos,n_eF", [(16, False, 1), (32, False, 1), (32, True, 3), (31, False, 2)])
def test_every_band_a_valence_band(n, pos, n_eF):
    """The largest tables of the n <= 32 kernel."""
    test_band_sums_match_oracle(n, pos, False, n_eF, 1e-5, n_val=n)


def test_no_hall_sums_with_a_long_frequency_list():
    """Without Hall sums the frequencies take no room beside the tables: the
    magnetoelectric sums are those of a single frequency, bit for bit."""
    from mepinterp_amd import capi, models
    m = models.make_random(seed=532, n=32, L=1, with_r=True)
    k = rand_kpts(3, seed=2)
    kw = dict(jobs=capi.MEP_JOB_KUBO | capi.MEP_JOB_MEP, n_eF=1, eF_min=0.0, eF_max=0.0, hw_min=0.01,
              hw_max=0.02, T_kelvin=300.0, eta=0.004, valence_bands=2)
    with capi.Engine(m["R_frac"], m["H"], r=m["r"], a_latt=m["a_latt"]) as eng:
        one = eng.run_kpts(k, capi.Engine.params(n_hw=1, **kw))
        many = eng.run_kpts(k, capi.Engine.params(n_hw=300, **kw))
    for q in KEYS[4:]:
        assert np.array_equal(one[q], many[q]), q


@pytest.mark.parametrize("n", [5, 16, 20, 32, 36, 70])
def test_given_bands_out_of_order(n):
    """A close band that is no neighbour by index: its whole row is excluded by
    the guards of the Niu terms, every other row keeps all but n0."""
    import oracle as O
    from mepinterp_amd import capi, models
    # rows of the close band: at most delta^2 0.6 n <= 1.1e-3, the others: at
    # least 0.59^2 delta = 1.7e-3
    tol, delta, nk, nv = 1.2e-3, 5e-3, 3, max(2, n // 2)
    rng = np.random.default_rng(n)
    e = np.repeat(0.6 * np.arange(n)[:, None], nk, axis=1)
    e[n - 1] = e[1] + delta
    V = rng.standard_normal((3, n, n, nk)) + 1j * rng.standard_normal((3, n, n, nk))
    m = models.make_random(seed=n, n=n, L=1)
    with capi.Engine(m["R_frac"], m["H"], a_latt=m["a_latt"], kubo_tol=tol) as eng:
        g = eng.bandsum(e, V, capi.Engine.params(jobs=capi.MEP_JOB_MEP, valence_bands=nv))
    for q, f in (("niu_ic", O.mep_niu_ic), ("niu_lc", O.mep_niu_lc)):
        ref = sum(f(np.asfortranarray(V[..., i]), np.ascontiguousarray(e[:, i]), nv, tol)
                  for i in range(nk))
        # 1e-9, the sums' tolerance
        assert np.max(np.abs(g[q] - ref)) <= 1e-9 * np.max(np.abs(ref)), q


@pytest.mark.parametrize("n", [3, 16, 24])
def test_a_band_at_zero_energy(n):
    """The padding of the band tables holds zeros too."""
    import oracle as O
    from mepinterp_amd import capi, models
    rng = np.random.default_rng(n)
    e = 0.1 * np.arange(n)
    V = np.asfortranarray(rng.standard_normal((3, n, n)) + 1j * rng.standard_normal((3, n, n)))
    fd = np.asfortranarray(np.linspace(0.9, 0.2, n)[None])
    m = models.make_random(seed=n, n=n, L=1)
    with capi.Engine(m["R_frac"], m["H"], a_latt=m["a_latt"]) as eng:
        g = eng.bandsum(e, V[..., None], capi.Engine.params(
            jobs=capi.MEP_JOB_AHC | capi.MEP_JOB_KUBO, n_hw=1, hw_min=0.03, hw_max=0.03, eta=0.01), fd=fd)
    for q, f in (("ahc_velo", O.velo_ahc_tens), ("ohc", O.kubo_ohc_tens)):
        ref = f(e, V, np.array([0.03]), fd, 0.01).reshape(g[q].shape, order="F")
        # 1e-9, the sums' tolerance
        assert np.max(np.abs(g[q] - ref)) <= 1e-9 * np.max(np.abs(ref)), q


@pytest.mark.parametrize("n", [33, 48, 70])
def test_two_bands_of_the_same_energy(n):
    """Above 32 bands: the Niu guards exclude the pair, the Kubo sums are not
    finite (1 / 0 in the reference), and nothing else notices."""
    import oracle as O
    from mepinterp_amd import capi, models
    tol, nv = 1e-5, n // 2
    rng = np.random.default_rng(n)
    e = 0.05 * np.arange(n)
    e[4] = e[3]    # valence and valence
    e[nv] = e[nv - 1]
    V = np.asfortranarray(rng.standard_normal((3, n, n)) + 1j * rng.standard_normal((3, n, n)))
    m = models.make_random(seed=n, n=n, L=1)
    with capi.Engine(m["R_frac"], m["H"], a_latt=m["a_latt"], kubo_tol=tol) as eng:
        g = eng.bandsum(e, V[..., None], capi.Engine.params(
            jobs=capi.MEP_JOB_MEP | capi.MEP_JOB_KUBO, valence_bands=nv, eF_min=0.5, eF_max=0.5))
    for q, f in (("niu_ic", O.mep_niu_ic), ("niu_lc", O.mep_niu_lc)):
        ref = f(V, e, nv, tol)
        # 1e-9, the sums' tolerance
        assert np.max(np.abs(g[q] - ref)) <= 1e-9 * np.max(np.abs(ref)), q
    assert not np.any(np.isfinite(g["kubo_ic"]))
