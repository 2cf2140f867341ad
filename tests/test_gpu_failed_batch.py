"""After a batch that ends in an error the other contexts are as they were: no
eigensolver status of the batch reaches their next call, and nothing that the
batch queued reaches its results.  (A model with a NaN in H is refused as "did
not converge", an ordinary error.)"""
import numpy as np
import pytest

from conftest import rand_kpts

pytestmark = pytest.mark.gpu

JOBS_KEYS = ("Ne", "ahc", "ahc_velo", "ohc", "kubo_ic", "kubo_lc", "niu_ic", "niu_lc")


def _engine(n, seed, nan=False):
    from mepinterp_amd import capi, models
    m = models.make_random(seed=seed, n=n, L=1)
    if nan:
        m["H"] = m["H"].copy()
        m["H"][0, 0, :] = np.nan
    return capi.Engine(m["R_frac"], m["H"], a_latt=m["a_latt"])


def _params(n):
    from mepinterp_amd import capi
    return capi.Engine.params(jobs=capi.MEP_JOB_AHC | capi.MEP_JOB_KUBO | capi.MEP_JOB_MEP,
                              n_eF=1, n_hw=1, hw_min=0.02, T_kelvin=300.0, eta=0.004,
                              valence_bands=n // 2)


@pytest.mark.parametrize("n", [8, 24, 40])
def test_band_sums_of_given_bands_after_a_failed_graph_batch(n):
    """mep_bandsum_batch solves nothing: a status is not its own."""
    from mepinterp_amd import capi
    p = _params(n)
    with _engine(n, 3) as good, _engine(n, 4, nan=True) as a, _engine(n, 5, nan=True) as b:
        e, V, _, _ = good.interp(rand_kpts(5, seed=n))
        ref = good.bandsum(e, V, p)
        with pytest.raises(capi.MepError):
            capi.run_batch([a, b], [(3, 2, 2)] * 2, [p, p], graph=True)
        for eng in (b, a):
            got = eng.bandsum(e, V, p)
            for q in JOBS_KEYS:
                assert np.array_equal(got[q], ref[q]), q


@pytest.mark.parametrize("graph", [False, True])
def test_next_calls_after_a_failed_batch(graph):
    """The first model is refused while the others, which take longer, are still
    at work: an interpolation and a run on each of them right after the error
    equal those of engines that saw no failed batch, bit for bit."""
    from mepinterp_amd import capi
    n, mesh = 40, (16, 16, 8)
    p = _params(n)
    k = rand_kpts(3, seed=1)

    def calls(eng):
        return eng.interp(k, velo=False)[0], eng.run_mesh((4, 3, 2), p), eng.interp(k)
    ref = []
    for seed in (6, 7):
        with _engine(n, seed) as eng:
            eng.run_mesh(mesh, p)  # the same workspace as below
            ref.append(calls(eng))
    with _engine(n, 6) as b, _engine(n, 7) as c, _engine(8, 4, nan=True) as a:
        for _ in range(2):
            with pytest.raises(capi.MepError):
                capi.run_batch([a, b, c], [(2, 2, 1), mesh, mesh], [_params(8), p, p],
                               graph=graph)
            for eng, (e0, s0, v0) in zip((c, b), (ref[1], ref[0])):
                e1, s1, v1 = calls(eng)
                assert np.array_equal(e1, e0)
                for q in JOBS_KEYS:
                    assert np.array_equal(s1[q], s0[q]), q
                for g, r in zip(v1[:2], v0[:2]):
                    assert np.array_equal(g, r)
