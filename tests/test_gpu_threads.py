"""Several host threads, each on a stream and a workspace of its own: the splits and
the eigensolver wait for a flag that their kernels set in pinned memory of the calling
thread, and hand tiles between workgroups on the device.  Every result equals the one
that the call gives alone, bit for bit (fixed orders of summation)."""

import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def split(lib, check, A, mode, stream):
    m, n = A.shape
    r = min(m, n)
    out = [torch.empty(m * r, dtype=torch.complex128, device="cuda"),
           torch.empty(r * n, dtype=torch.complex128, device="cuda"),
           torch.empty(r, dtype=torch.float64, device="cuda")]
    bytes_ = lib.seemps_svd_split_workspace(m, n)
    work = torch.empty(bytes_, dtype=torch.uint8, device="cuda")
    D, err, info = ctypes.c_int64(0), ctypes.c_double(0.0), (ctypes.c_int32 * 2)()
    check(lib.seemps_svd_split(m, n, A.data_ptr(), mode, 2, 1e-20, r, out[0].data_ptr(),
                               out[1].data_ptr(), out[2].data_ptr(), ctypes.byref(D),
                               ctypes.byref(err), work.data_ptr(), bytes_, info, stream))
    torch.cuda.current_stream().synchronize()
    D = D.value
    return [D, err.value, out[0][:m * D].cpu(), out[1][:D * n].cpu(), out[2].cpu()]


def solve(lib, check, H, v0, stream):
    chi = v0.shape[0]
    L, Hm, R = H
    evec = torch.empty_like(v0)
    stats = (ctypes.c_double * 5)()
    bytes_ = lib.seemps_eigensolve_workspace(chi, 1, 1, 1, 1, chi, 12)
    work = torch.empty(bytes_, dtype=torch.uint8, device="cuda")
    check(lib.seemps_two_site_eigensolve_prec(0, chi, 1, 1, 1, 1, chi, L.data_ptr(),
                                              Hm.data_ptr(), R.data_ptr(), v0.data_ptr(),
                                              evec.data_ptr(), 12, 1e-10, 50, stats,
                                              work.data_ptr(), bytes_, stream))
    return [stats[0], stats[2], evec.cpu()]


def test_threads_and_streams():
    from seemps2_amd._lib import check, lib

    rng = np.random.default_rng(3)

    def dev(*shape):
        return torch.from_numpy(rng.normal(size=shape) + 1j * rng.normal(size=shape)).cuda()

    def hermitian(n):
        x = dev(n, n)
        return ((x + x.mH) / 2).contiguous()

    jobs = []
    for i, (m, n) in enumerate([(64, 64), (40, 100), (12, 9), (90, 70)]):
        jobs.append((split, dev(m, n), i % 2))
    one = torch.ones(1, dtype=torch.complex128, device="cuda")
    for chi in (32, 100):  # the larger one waits for its residual every second step
        eye = torch.eye(chi, dtype=torch.complex128, device="cuda")
        jobs.append((solve, (hermitian(chi), one, eye + 0.1 * hermitian(chi)), dev(chi, chi)))
    torch.cuda.synchronize()

    def run(job):
        return job[0](lib, check, job[1], job[2], torch.cuda.current_stream().cuda_stream)

    alone = [run(j) for j in jobs]
    failures = []

    def worker(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for rep in range(6):
                    j = (k + rep) % len(jobs)
                    for x, y in zip(run(jobs[j]), alone[j]):
                        same = torch.equal(x, y) if isinstance(x, torch.Tensor) else x == y
                        assert same, (k, rep, j)
        except Exception as e:  # noqa: BLE001 - reported by the main thread
            failures.append(e)

    threads = [threading.Thread(target=worker, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
