"""Edges of the SVD's own kernels: register tiles of the QR, panel widths,
row chunks, padding, both split modes.

The tolerances are the backward-error bounds of the Householder / Jacobi chain
at these sizes, as elsewhere in the suite: 1e-12 relative on reconstructions
and isometries, 5e-13 of the largest on singular values.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def K():
    from seemps2_amd import kernels

    return kernels


def crandn(rng, *shape):
    return rng.normal(size=shape) + 1j * rng.normal(size=shape)


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


# rows: 64 RPT and one more; columns: a panel and one more, the smallest QR (17)
@pytest.mark.parametrize("m,n", [(64, 17), (65, 64), (128, 65), (129, 33), (256, 32), (257, 49),
                                 (512, 17), (513, 24), (1024, 20), (1025, 33), (31, 700)])
def test_qr_edges(K, m, n):
    rng = np.random.default_rng(m * 1000 + n)
    r = min(m, n)
    A = crandn(rng, m, r) * np.exp(-0.3 * np.arange(r)) @ crandn(rng, r, n)
    U, S, VH = K.svd(K.as_dev(A))
    U, S, VH = K.to_numpy(U), S.cpu().numpy(), K.to_numpy(VH)
    assert rel((U * S) @ VH, A) < 1e-12
    assert np.abs(U.conj().T @ U - np.eye(r)).max() < 1e-12
    assert np.abs(VH @ VH.conj().T - np.eye(r)).max() < 1e-12
    s_ref = np.linalg.svd(A, compute_uv=False)
    assert np.abs(S - s_ref).max() < 5e-13 * s_ref[0]
