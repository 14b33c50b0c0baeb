"""Edges of the direct GEMM and the local-operator kernels: tiles of 16 and 32, K remainders of every
wavefront's run, leading dimensions beyond the rows, all sixteen operand forms.

Gaussian integers: every partial sum is an exact integer in any order, so the
result equals the exact one bit for bit.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

OPS = {0: lambda x: x, 1: lambda x: x.T, 2: lambda x: x.conj().T, 3: lambda x: x.conj()}


# one tile and its edges; four waves' runs with none, one or part of a step; a
# tile for each CU (512 x 512), for each SIMD (1024 x 1023), and neither (320 tiles)
@pytest.mark.parametrize("M,N,K_", [(1, 1, 1), (16, 16, 3), (17, 33, 5), (31, 15, 67), (2, 40, 64),
                                    (49, 16, 129), (512, 511, 71), (630, 509, 18),
                                    (1024, 1023, 129)])
def test_direct_gemm_edges(M, N, K_):
    from seemps2_amd import kernels as K
    from seemps2_amd._lib import check, lib

    rng = np.random.default_rng(M * 7 + N)

    def ints(r, c):
        return rng.integers(-3, 4, (r, c)) + 1j * rng.integers(-3, 4, (r, c))

    def padded(x, extra):  # rows followed by NaN that nothing may read into a result
        p = np.full((x.shape[0], x.shape[1] + extra), np.nan + 1j * np.nan)
        p[:, :x.shape[1]] = x
        return K.as_dev(p)

    alpha, beta = 1 + 2j, 2 - 1j
    for opA in range(4):
        for opB in range(4):
            A = ints(*((K_, M) if opA in (1, 2) else (M, K_)))
            B = ints(*((N, K_) if opB in (1, 2) else (K_, N)))
            C = ints(M, N)
            ref = alpha * (OPS[opA](A) @ OPS[opB](B)) + beta * C
            a, b, c = padded(A, 3), padded(B, 1), padded(C, 2)
            check(lib.seemps_zgemm(opA, opB, M, N, K_, alpha.real, alpha.imag, a.data_ptr(),
                                   a.shape[1], 0, b.data_ptr(), b.shape[1], 0, beta.real,
                                   beta.imag, c.data_ptr(), c.shape[1], 0, 1,
                                   torch.cuda.current_stream().cuda_stream))
            out = K.to_numpy(c)
            assert np.array_equal(out[:, :N], ref), (opA, opB)
            assert np.isnan(out[:, N:]).all()


# remainders of the eight loads ahead, one and two stages of operator rows (64), outputs
# short of a group of four, runs that end inside a workgroup and inside a q range, J2 > 1,
# ten outputs a thread (the last three)
@pytest.mark.parametrize("P,I,Q,J1,J2", [(1, 1, 1, 1, 1), (3, 8, 5, 2, 1), (7, 9, 37, 3, 2),
                                         (5, 16, 51, 5, 1), (2, 17, 129, 1, 7), (3, 64, 85, 9, 1),
                                         (4, 65, 63, 2, 3), (1, 150, 300, 13, 1),
                                         (511, 20, 129, 20, 1), (300, 3, 437, 7, 3),
                                         (257, 81, 512, 1, 11)])
def test_local_edges(P, I, Q, J1, J2):
    from seemps2_amd import kernels as K

    rng = np.random.default_rng(P + 10 * I)

    def ints(*shape):
        return rng.integers(-3, 4, shape) + 1j * rng.integers(-3, 4, shape)

    x, op = ints(P, I, Q), ints(I, J1, J2)
    ref = np.tensordot(x, op, axes=(1, 0)).transpose(0, 2, 1, 3)
    out = K.local(K.as_dev(x), K.as_dev(op), P, I, Q, J1, J2)
    assert np.array_equal(K.to_numpy(out).reshape(ref.shape), ref)
    out = K.local(K.as_dev(x), K.as_dev(op), P, I, Q, J1, J2, out=out, accumulate=True)
    assert np.array_equal(K.to_numpy(out).reshape(ref.shape), 2 * ref)


# two 32 x 32 tiles a CU or more (whole tiles), fewer (quarters), and 64 x 64 tiles
@pytest.mark.parametrize("tile,count", [(1, 130), (1, 6), (0, 6)])
@pytest.mark.parametrize("opA,opB", [(0, 0), (2, 0), (0, 1), (1, 0), (3, 0), (0, 2)])
def test_grouped_gemm_edges(tile, count, opA, opB):
    from seemps2_amd import batch, kernels as K

    rng = np.random.default_rng(count)
    edges = [1, 15, 16, 17, 33, 64, 65, 80, 97]
    probs, refs, outs, keep = [], [], [], []
    for p in range(count):
        M, N, Kd = edges[p % 9], edges[(p // 2) % 9], int(rng.integers(1, 90))
        A = rng.integers(-3, 4, (Kd, M) if opA in (1, 2) else (M, Kd)) + 1j * 0
        A = A + 1j * rng.integers(-3, 4, A.shape)
        B = rng.integers(-3, 4, (N, Kd) if opB in (1, 2) else (Kd, N)) + 1j * 0
        B = B + 1j * rng.integers(-3, 4, B.shape)
        Ad, Bd, Cd = K.as_dev(A), K.as_dev(B), K.empty(M, N)
        keep += [Ad, Bd]
        probs.append((M, N, Kd, Ad, A.shape[1], Bd, B.shape[1], Cd, N))
        refs.append(OPS[opA](A) @ OPS[opB](B))
        outs.append(Cd)
    gg = batch.GroupedGemm(opA, opB, probs, tile)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert (gg.ntiles >= 2 * cus) == (count == 130)
    gg.launch()
    for Cd, ref in zip(outs, refs):
        assert np.array_equal(K.to_numpy(Cd), ref)


# Both sides of the lines between the direct and the staged kernel (256 CUs): few tiles
# and a long K, aligned and past an edge; whole and part-empty rounds of the CUs and of
# the SIMDs; a K too short for many tiles; both operands along K,
# their rows whole cache lines apart or not.
@pytest.mark.parametrize("opA,opB,M,N,K_,direct", [
    (0, 0, 64, 64, 1024, True), (0, 0, 64, 64, 8192, False), (2, 0, 64, 64, 2048, True),
    (0, 0, 33, 40, 8192, False), (2, 0, 33, 40, 8192, True), (0, 1, 128, 128, 512, True),
    (0, 1, 128, 128, 768, False), (0, 1, 512, 512, 512, True), (0, 1, 512, 512, 768, False),
    (0, 1, 272, 1000, 256, False), (0, 1, 272, 1000, 768, False), (3, 2, 700, 700, 768, True),
    (2, 0, 640, 512, 256, True), (0, 0, 900, 900, 16, False), (0, 0, 900, 900, 256, True),
    (1, 1, 1024, 1000, 300, True), (1, 0, 1100, 1000, 60, False), (1, 0, 1100, 1000, 333, False),
    (1, 0, 700, 640, 333, True), (0, 1, 144, 134, 804, True), (0, 1, 144, 134, 800, False),
    (0, 1, 512, 160, 636, True), (0, 1, 512, 160, 640, False)])
def test_gemm_route(opA, opB, M, N, K_, direct):
    from seemps2_amd import _lib, kernels as K

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are drawn for 256 CUs")
    rng = np.random.default_rng(M + N + K_)

    def ints(r, c):
        return rng.integers(-3, 4, (r, c)) + 1j * rng.integers(-3, 4, (r, c))

    A = ints(*((K_, M) if opA in (1, 2) else (M, K_)))
    B = ints(*((N, K_) if opB in (1, 2) else (K_, N)))
    a, b = K.as_dev(A), K.as_dev(B)
    _lib.timing_enable("zgemm_kernel,zgemm_direct")
    try:
        out = K.to_numpy(K.gemm(a, b, opA, opB))
        ran = [k for k, r in _lib.timing_records().items() if r["launches"]]
    finally:
        _lib.timing_enable(None)
    assert ran == ["zgemm_direct" if direct else "zgemm_kernel"]
    assert np.array_equal(out, OPS[opA](A) @ OPS[opB](B))
