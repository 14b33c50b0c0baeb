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


# columns: one block pair (16, 32), an odd number of blocks (33, 48), one more
# than a tile of rows (65), padding up to 31 columns; the split's orientation
# for wide and tall matrices
@pytest.mark.parametrize("m,n", [(2, 40), (16, 16), (32, 32), (33, 40), (48, 33), (65, 65),
                                 (97, 130), (130, 97), (129, 129), (250, 193)])
@pytest.mark.parametrize("mode", [0, 1])
def test_split_edges(K, m, n, mode):
    rng = np.random.default_rng(m * 1000 + n)
    r = min(m, n)
    A = crandn(rng, m, r) * np.exp(-20.0 / r * np.arange(r)) @ crandn(rng, r, n)
    A /= np.linalg.norm(A)
    u, s, v = np.linalg.svd(A, full_matrices=False)
    for cap in (r, max(1, r // 2)):
        Ad, Bd, D, err2, sd = K.svd_split(K.as_dev(A), m, n, mode, 0 if cap == r else 2, 1e-30,
                                          cap, want_s=True)
        Ad, Bd = K.to_numpy(Ad), K.to_numpy(Bd)
        assert D == cap
        iso = Ad.conj().T @ Ad if mode == 0 else Bd @ Bd.conj().T
        assert np.abs(iso - np.eye(D)).max() < 1e-12
        # the kept subspace moves by rounding / (gap at the cut), gap >= s_D / r here
        assert rel(Ad @ Bd, (u[:, :D] * s[:D]) @ v[:D]) < 1e-12
        assert np.abs(sd.cpu().numpy() - s[:D]).max() < 5e-13 * s[0]
        assert abs(err2 - np.sum(s[D:] ** 2)) < 1e-12


@pytest.mark.parametrize("n", [1060, 1100])
def test_svd_beyond_the_register_tiles(K, n):
    """More than 1024 rows: QR panels in memory, and (35 block pairs leave seven
    workgroups each) row chunks of three LDS tiles.  A column takes n rotations
    a sweep for about ten sweeps, so the backward error is bounded by
    10 n units in the last place of 2 eps each."""
    rng = np.random.default_rng(n)
    A = crandn(rng, n, n)
    A /= np.linalg.norm(A)
    U, S, VH = K.svd(K.as_dev(A))
    U, S, VH = K.to_numpy(U), S.cpu().numpy(), K.to_numpy(VH)
    tol = 20 * n * np.finfo(float).eps
    assert rel((U * S) @ VH, A) < tol
    assert np.abs(U.conj().T @ U - np.eye(n)).max() < tol
    assert np.abs(VH @ VH.conj().T - np.eye(n)).max() < tol


# V's rows on workgroups of their own: one and more row chunks, a last partial chunk,
# the last size that has them and the first that has not; all pairs, no pair and only
# some pairs to rotate
@pytest.mark.parametrize("n", [49, 64, 65, 129, 200, 256, 257, 272])
@pytest.mark.parametrize("kind", ["full", "diagonal", "rank"])
def test_svd_v_apart(K, n, kind):
    rng = np.random.default_rng(n)
    if kind == "diagonal":
        A = np.diag(np.linspace(1.0, 2.0, n)[rng.permutation(n)]) + 0j
    else:
        r = n if kind == "full" else n // 3
        A = crandn(rng, n, r) * np.exp(-20.0 / r * np.arange(r)) @ crandn(rng, r, n)
        A /= np.linalg.norm(A)
    U, S, VH = K.svd(K.as_dev(A))
    U, S, VH = K.to_numpy(U), S.cpu().numpy(), K.to_numpy(VH)
    assert rel((U * S) @ VH, A) < 1e-12
    assert np.abs(U.conj().T @ U - np.eye(n)).max() < 1e-12
    assert np.abs(VH @ VH.conj().T - np.eye(n)).max() < 1e-12
    s_ref = np.linalg.svd(A, compute_uv=False)
    assert np.abs(S - s_ref).max() < 5e-13 * s_ref[0]


# Column norms whose squares lie near the smallest normal number (1e-152 squared times a
# few): register panels with and without trailing columns, a panel in memory, a column,
# a rank of one.  The singular values of such a matrix are not resolved (the squares of
# its Gram matrix underflow), its product is, to the bound of the chain above.
@pytest.mark.parametrize("m,n,r", [(8, 1, 1), (2, 2, 1), (40, 30, 30), (30, 40, 30), (100, 100, 100),
                                   (700, 20, 20), (1100, 20, 20)])
@pytest.mark.parametrize("mode", [0, 1])
def test_split_of_tiny_matrices(K, m, n, r, mode):
    rng = np.random.default_rng(m + n)
    A = crandn(rng, m, r) @ crandn(rng, r, n) / np.sqrt(r)
    scale = 2.0 ** -505  # exact
    Ad, Bd, D, _, _ = K.svd_split(K.as_dev(A * scale), m, n, mode, 0, 0.0, min(m, n))
    out = K.to_numpy(Ad) @ K.to_numpy(Bd) / scale
    assert D == min(m, n)
    assert rel(out, A) < 1e-12


# Columns beyond the registers: panels of one, up to four and up to eight columns and
# their remainders, the reflectors on workgroups of 256 and (from 4097 rows) of 1024
# threads; few enough columns for the norms' lanes to share a row.
@pytest.mark.parametrize("m,n", [(1025, 1), (1025, 4), (1030, 5), (1600, 8), (1601, 9),
                                 (24, 1030), (4097, 12), (5000, 40), (1100, 70)])
@pytest.mark.parametrize("mode", [0, 1])
def test_split_long_columns(K, m, n, mode):
    rng = np.random.default_rng(m * 1000 + n)
    r = min(m, n)
    A = crandn(rng, m, r) * np.exp(-20.0 / r * np.arange(r)) @ crandn(rng, r, n)
    A /= np.linalg.norm(A)
    Ad, Bd, D, _, sd = K.svd_split(K.as_dev(A), m, n, mode, 0, 0.0, r, want_s=True)
    Ad, Bd = K.to_numpy(Ad), K.to_numpy(Bd)
    assert D == r
    assert rel(Ad @ Bd, A) < 1e-12
    iso = Ad.conj().T @ Ad if mode == 0 else Bd @ Bd.conj().T
    assert np.abs(iso - np.eye(r)).max() < 1e-12
    s_ref = np.linalg.svd(A, compute_uv=False)
    assert np.abs(sd.cpu().numpy() - s_ref).max() < 5e-13 * s_ref[0]


@pytest.mark.parametrize("c", [0.1, 0.3, 0.5, 0.7, 1.0, 1.6])
def test_one_rotation_is_exact(K, c):
    """Columns that are orthogonal but for one pair: a sweep meets that pair once, and
    a rotation whose angle is good to rounding leaves it orthogonal to far below the
    1e-9 from which the next sweep is the last.  An angle off by 1e-8 takes three."""
    import ctypes

    from seemps2_amd._lib import check, lib, ptr, stream, workspace

    n, a, b = 64, 3, 40
    rng = np.random.default_rng(11)
    R = np.diag(np.linspace(3.0, 1.0, n)) + 0j
    R[a, b] = c
    A = K.as_dev(np.linalg.qr(crandn(rng, n, n))[0] @ R)
    U, VH = K.empty(n, n), K.empty(n, n)
    S = torch.empty(n, dtype=torch.float64, device=A.device)
    wp, wn = workspace.get(lib.seemps_svd_workspace(n, n))
    info = (ctypes.c_int32 * 2)()
    check(lib.seemps_zgesvd(n, n, ptr(A), n, ptr(U), ptr(S), ptr(VH), wp, wn, info, stream()))
    assert list(info) == [2, 1]
    s_ref = np.linalg.svd(R, compute_uv=False)
    assert np.abs(S.cpu().numpy() - s_ref).max() < 5e-13 * s_ref[0]


@pytest.mark.parametrize("n", [4090, 4100])
def test_split_long_spectrum(K, n):
    """The sort and the truncation on spectra that just fit LDS and that do not."""
    d = torch.linspace(2.0, 1.0, n, dtype=torch.float64, device="cuda")
    p = torch.from_numpy(np.random.default_rng(n).permutation(n)).cuda()
    A = torch.diag(d[p]).to(torch.complex128)
    Ad, Bd, D, err2, s = K.svd_split(A, n, n, 0, 2, 0.0, 2000, want_s=True)
    assert D == 2000
    assert float((s - d[:2000]).abs().max()) < 1e-14
    assert abs(err2 - float((d[2000:] ** 2).sum())) < 1e-11 * err2
    # entries at most 2, each off by a few ulp
    assert float((Ad.mH @ Ad - torch.eye(D, device="cuda")).abs().max()) < 1e-14
    assert float(((Ad @ Bd) - torch.diag(torch.where(d[p] >= d[1999], d[p], 0.0))).abs().max()) < 1e-14


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("m,n", [(3, 2), (16, 16), (40, 30), (70, 90), (1100, 9)])
def test_split_spreads_nan(K, m, n, bad):
    """A value that is no number ends in an error or in the result, in every mode and
    rule, never in factors that look right."""
    from scipy.linalg import LinAlgError

    A = crandn(np.random.default_rng(m), m, n)
    A[m // 2, n // 2] = bad
    for mode in (0, 1):
        for method in range(4):
            try:
                Ad, Bd, D, err2, _ = K.svd_split(K.as_dev(A), m, n, mode, method, 1e-10, 7)
            except LinAlgError:
                continue
            assert 1 <= D <= min(m, n)
            finite = np.isfinite(K.to_numpy(Ad)).all() and np.isfinite(K.to_numpy(Bd)).all()
            assert not (finite and np.isfinite(err2)), (mode, method)
