"""Eigenvalues at the edges of the Sturm kernels (teams of 8, 16 and 32 lanes,
one and two wavefronts per k-point, blocks of eight and sixteen steps) against
LAPACK, for spectra that stress the brackets: random, diagonal, exactly and
nearly degenerate, clustered with tiny couplings, zero, and scaled far from
one.  A k-independent model (R = 0 only) hands each matrix to the solver."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 7, 8, 9, 15, 16, 17, 24, 25, 31, 32, 33, 48, 63, 64, 65, 96, 127, 128]


def _matrices(n):
    rng = np.random.default_rng(n)
    X = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    X = 0.5 * (X + X.conj().T)
    Q = np.linalg.qr(X)[0]

    def with_spectrum(w):
        A = (Q * w) @ Q.conj().T
        return 0.5 * (A + A.conj().T)
    lin = np.linspace(-1.0, 2.0, n)
    pairs = np.repeat(lin[: (n + 1) // 2], 2)[:n]
    cluster = np.where(np.arange(n) < n // 2, 0.3, 0.3 + 1e-9 * np.arange(n))
    T = np.diag(np.full(n, 0.25)) + np.diag(np.full(n - 1, 1e-7), 1) + np.diag(np.full(n - 1, 1e-7), -1)
    return {"random": X, "diagonal": np.diag(rng.permutation(lin)), "identity": np.eye(n),
            "pairs": with_spectrum(pairs), "close pairs": with_spectrum(pairs + 1e-11 * np.arange(n)),
            "separated": with_spectrum(lin + 1e-4 * (np.arange(n) % 2)), "cluster": with_spectrum(cluster),
            "weak chain": T, "zero": np.zeros((n, n)), "tiny": 1e-100 * X, "huge": 1e100 * X}


@pytest.mark.parametrize("n", SIZES)
def test_eigenvalues_match_lapack(n):
    from mepinterp_amd import capi
    k = np.asfortranarray(np.random.default_rng(1).uniform(-0.5, 0.5, size=(3, 5)))
    for name, A in _matrices(n).items():
        ref = np.linalg.eigvalsh(A)
        with capi.Engine(np.zeros((3, 1)), A.astype(np.complex128).reshape(n, n, 1)) as eng:
            e = eng.interp(k, velo=False)[0]
        # backward-stable reduction and eigenvalues: a small multiple of n eps |A|
        tol = 4.0 * (n + 4) * np.finfo(float).eps * np.max(np.abs(ref))
        for q in range(k.shape[1]):
            assert np.all(np.diff(e[:, q]) >= 0), (name, q)
            assert np.max(np.abs(e[:, q] - ref)) <= tol, (name, q)


@pytest.mark.parametrize("n", [5, 20, 40, 80])
def test_matrices_that_are_not_finite(n):
    """Refused as "did not converge", but for an infinite first level, which
    stays apart from the others in the reduction: it is one of the eigenvalues."""
    from mepinterp_amd import capi
    k = np.zeros((3, 1))

    def solve(pos, val):
        A = np.eye(n, dtype=np.complex128) + 0.1 * np.ones((n, n))
        A[pos] = A[pos[::-1]] = val
        with capi.Engine(np.zeros((3, 1)), A.reshape(n, n, 1)) as eng:
            return eng.interp(k, velo=False)[0]
    for pos, val in (((0, 0), np.nan), ((n // 2, n // 2), np.nan), ((n // 2, n // 2), np.inf),
                     ((1, 2), np.nan), ((0, n - 1), np.inf)):
        with pytest.raises(capi.MepError):
            solve(pos, val)
    assert np.all(np.isfinite(solve((0, 0), 2.0)))
    assert solve((0, 0), np.inf)[n - 1, 0] == np.inf
