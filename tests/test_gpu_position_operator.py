"""The position-operator kernels at the edges of their tiles (one 16 x 16 tile
and one wavefront up to 16 bands, four tiles up to 32, workgroup slots above)
against the oracle: every element of V, A and Omega as get_wann_interp returns
them, and the band sums, for which only V and the band diagonals (or, for the
optical sums, A) are formed.  Both conventions, the printed equations, no gauge
transformation, and a model whose H(R) and r(R) lack their partners at -R, so
that no matrix but the eigensolver's upper triangle is Hermitian."""
import numpy as np
import pytest

from conftest import oracle_model, rand_kpts

pytestmark = pytest.mark.gpu


def _model(n, tb, lone):
    from mepinterp_amd import models
    m = models.make_random(seed=900 + n, n=n, L=1, with_r=True, tb=tb)
    if lone:
        rng = np.random.default_rng(n)
        for s in (2, 20):
            m["H"][:, :, s] *= 1.0 + 0.05 * rng.normal(size=(n, n))
            m["r"][:, :, :, s] *= 1.0 + 0.05 * rng.normal(size=(3, n, n))
    return m


def _rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


CASES = [(n, tb, False, False, True) for n, tb in
         ((1, False), (2, True), (5, False), (8, True), (15, False), (16, True), (17, True), (24, False),
          (31, True), (32, False), (33, True), (49, False))]
CASES += [(n, False, True, False, True) for n in (9, 20, 36)]          # textbook
CASES += [(n, True, False, True, True) for n in (11, 27, 34)]          # no Hermitian partner
CASES += [(n, True, False, False, False) for n in (6, 18, 40)]         # no gauge transformation


@pytest.mark.parametrize("n,tb,textbook,lone,gauge", CASES)
def test_position_operator_kernels_match_oracle(n, tb, textbook, lone, gauge):
    import oracle as O
    from mepinterp_amd import capi
    m = _model(n, tb, lone)
    om = oracle_model(m, textbook=textbook, do_gauge_trafo=gauge)
    k = rand_kpts(5, seed=n)
    kw = dict(n_eF=2, eF_min=-0.01, eF_max=0.01, n_hw=2, hw_min=0.004, hw_max=0.05,
              T_kelvin=300.0, eta=0.004, valence_bands=max(1, n // 2))
    with capi.Engine(m["R_frac"], m["H"], r=m["r"], wf_centers=m["wf_centers"], a_latt=m["a_latt"],
                     textbook=textbook, gauge_trafo=gauge) as eng:
        e, V, A, Om = eng.interp(k)
        for ik in range(k.shape[1]):
            eo, Vo, Ao, Omo = O.get_wann_interp(om, k[:, ik])
            for got, ref in ((e[:, ik], eo), (V[..., ik], Vo), (A[..., ik], Ao), (Om[..., ik], Omo)):
                # FP64 on both sides; D divides by gaps down to 1e-3 of the spectrum
                assert _rel(got, ref) < 1e-10
        runs = [(capi.MEP_JOB_AHC, dict(do_ahc=True), ("ahc", "ahc_velo", "ohc")),
                (capi.MEP_JOB_KUBO | capi.MEP_JOB_MEP, dict(do_kubo=True, do_mep=True),
                 ("kubo_ic", "kubo_lc", "kubo_cs", "niu_ic", "niu_lc", "niu_cs")),
                (capi.MEP_JOB_OPT | capi.MEP_JOB_GYRO, dict(do_opt=True, do_gyro=True),
                 ("opt_s", "opt_a", "photo", "gyro_C", "gyro_D", "gyro_Dw"))]
        for bits, job, keys in runs:
            g = eng.run_kpts(k, capi.Engine.params(jobs=bits, **kw))
            o = O.accumulate(om, O.RunParams(**job, **kw), k)
            for key in keys:
                # 1e-9, the sums' tolerance; gyro_Dw and opt_a divide by
                # unbroadened poles (nearest of these few points: 1e-4 away)
                assert np.max(np.abs(o[key])) == 0 or _rel(g[key], o[key]) < 1e-9, key
