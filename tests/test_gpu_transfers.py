"""Results that go through the pinned buffer (up to 1 MiB a call) and results
that are copied directly give the same bits: interpolations on both sides of
the limit and split over k-blocks, in any order on one engine, and runs whose
record lies above it."""
import numpy as np
import pytest

from conftest import rand_kpts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pos", [False, True])
def test_interp_bits_do_not_depend_on_the_transfer(pos):
    from mepinterp_amd import capi, models
    m = models.make_random(seed=31, n=8, L=1, with_r=pos)
    per = 8 * (3 + 8) + 16 * 64 * (15 if pos else 3)  # bytes of one k-point
    edge = (1 << 20) // per
    k = rand_kpts(edge + 3, seed=5)
    with capi.Engine(m["R_frac"], m["H"], r=m["r"], a_latt=m["a_latt"]) as eng:
        one = [eng.interp(np.asfortranarray(k[:, i:i + 1])) for i in (0, edge - 1, edge + 2)]
        for nk in (edge + 3, edge - 1, 1, edge, edge + 1):
            got = eng.interp(np.asfortranarray(k[:, :nk]))
            for i, ref in zip((0, edge - 1, edge + 2), one):
                if i < nk:
                    for g, r in zip(got, ref):
                        if r is not None:
                            assert np.array_equal(g[..., i], r[..., 0])
        eng.set_kblock(16)
        got = eng.interp(k)
        for i, ref in zip((0, edge - 1, edge + 2), one):
            assert np.array_equal(got[0][:, i], ref[0][:, 0])


def test_records_above_the_buffer_equal_their_parts():
    from mepinterp_amd import capi, models
    m = models.make_random(seed=33, n=6, L=1)
    k = rand_kpts(9, seed=6)
    hw = np.linspace(0.01, 0.3, 4000)  # 36 doubles a frequency: 1.15 MB
    p = dict(jobs=capi.MEP_JOB_AHC, n_eF=1, eF_min=0.0, eF_max=0.0, T_kelvin=300.0, eta=0.004,
             valence_bands=1)
    with capi.Engine(m["R_frac"], m["H"], a_latt=m["a_latt"]) as eng:
        big = eng.run_kpts(k, capi.Engine.params(n_hw=4000, hw_min=hw[0], hw_max=hw[-1], **p))
        for lo, hi in ((0, 2000), (2000, 4000)):
            part = eng.run_kpts(k, capi.Engine.params(n_hw=hi - lo, hw_min=hw[lo], hw_max=hw[hi - 1], **p))
            for q in ("ahc_velo", "ohc"):
                a = big[q].reshape(9, -1)[:, lo:hi]
                b = part[q].reshape(9, -1)
                # the frequencies of the part are the same to rounding
                assert np.max(np.abs(a - b)) < 1e-9 * np.max(np.abs(b)), q
