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
