"""Lanczos step kernels at their edges: every register-array size, bases that
span the whole space, one element to more than one per thread, a Krylov space
that closes early.

The operator is L (x) R with a known lowest pair: eigenvalue -6, the next one -3,
largest modulus 6.  The solver stops at a residual of 1e-12 |theta|, so the value
lies within 6e-12 and the vector within 6e-12 / 3, each plus rounding of 6 sqrt(n)
eps < 1e-12: bounds of 1e-11.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def hermitian(rng, eigs):
    n = len(eigs)
    q, _ = np.linalg.qr(rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n)))
    return (q * eigs) @ q.conj().T, q


@pytest.mark.parametrize("closed", [False, True])
@pytest.mark.parametrize("chiL,chiR,ncv", [(1, 2, 2), (1, 3, 5), (4, 5, 23), (16, 16, 4),
                                           (16, 17, 5), (31, 33, 8), (90, 91, 9), (64, 64, 12),
                                           (40, 41, 13), (100, 90, 16), (33, 65, 17),
                                           (257, 256, 20), (70, 130, 23)])
def test_eigensolve_edges(chiL, chiR, ncv, closed):
    from seemps2_amd import kernels as K

    rng = np.random.default_rng(chiL * 100 + chiR)
    eL = np.linspace(0.5, 1.0, chiL)
    eL[-1] = 2.0
    eR = np.linspace(-1.0, 1.0, chiR)
    eR[0] = -3.0
    L, qL = hermitian(rng, eL)
    R, qR = hermitian(rng, eR)
    want = np.outer(qL[:, -1], qR[:, 0])
    v0 = (rng.normal(size=want.shape) + 1j * rng.normal(size=want.shape))
    if closed:  # two eigenvectors: the Krylov space has dimension two
        v0 = want + np.outer(qL[:, -1], qR[:, 1])
    lam, vec, stats = K.eigensolve(
        K.as_dev(L.reshape(chiL, 1, chiL)), K.as_dev(np.eye(1) + 0j),
        K.as_dev(R.reshape(chiR, 1, chiR)), K.as_dev(v0.reshape(chiL, 1, 1, chiR)), 1, 1,
        ncv=ncv, tol=1e-12)
    vec = K.to_numpy(vec).reshape(chiL, chiR)
    assert abs(lam + 6.0) < 1e-11
    overlap = np.vdot(want, vec)
    assert abs(np.linalg.norm(vec) - 1.0) < 1e-13
    assert np.linalg.norm(vec - overlap * want) < 1e-11
    if closed:
        assert stats["restarts"] <= 2


@pytest.mark.parametrize("delta", [1e-3, 1e-7, 1e-10])
def test_nearly_converged_start(delta):
    """From an eigenvector and a little of others every Gram-Schmidt needs its second
    pass, after which the norm is |w|^2 less the squared coefficients: the basis stays
    normalised, so the value and the vector are as good as from any start."""
    from seemps2_amd import kernels as K

    chi = 40
    rng = np.random.default_rng(8)
    L, qL = hermitian(rng, np.r_[np.linspace(0.5, 1.0, chi - 1), 2.0])
    R, qR = hermitian(rng, np.r_[-3.0, np.linspace(-1.0, 1.0, chi - 1)])
    want = np.outer(qL[:, -1], qR[:, 0])
    v0 = want + delta * (rng.normal(size=want.shape) + 1j * rng.normal(size=want.shape)) / chi
    lam, vec, _ = K.eigensolve(
        K.as_dev(L.reshape(chi, 1, chi)), K.as_dev(np.eye(1) + 0j),
        K.as_dev(R.reshape(chi, 1, chi)), K.as_dev(v0.reshape(chi, 1, 1, chi)), 1, 1,
        ncv=12, tol=1e-12)
    vec = K.to_numpy(vec).reshape(chi, chi)
    assert abs(lam + 6.0) < 1e-11
    assert abs(np.linalg.norm(vec) - 1.0) < 1e-13
    assert np.linalg.norm(vec - np.vdot(want, vec) * want) < 1e-11


def test_start_that_is_no_number():
    """NaN in the start vector comes back in the value; nothing waits for it."""
    from seemps2_amd import kernels as K

    for chi in (4, 100):
        v0 = np.ones((chi, 1, 1, chi)) + 0j
        v0[1, 0, 0, 1] = np.nan
        eye = K.as_dev(np.eye(chi).reshape(chi, 1, chi) + 0j)
        lam, _, _ = K.eigensolve(eye, K.as_dev(np.eye(1) + 0j), eye, K.as_dev(v0), 1, 1, ncv=8,
                                 tol=1e-10, maxiter=3)
        assert np.isnan(lam)
