"""Host decisions around the block Jacobi, on the CPU.

Its status from the control block: a wait that ran out in any workgroup is an
error, also when the workgroup that records the sweeps had already left with
"converged" (the workgroups that rotate V are not counted in the last barrier).
Its form: each one is launched only as far as that form's own workgroups are
resident."""

import ctypes
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parents[1] / "seemps2_amd" / "libseemps_hip.so"


class Ctrl(ctypes.Structure):  # svd_work.h
    _fields_ = [("barrier", ctypes.c_uint32), ("abort", ctypes.c_uint32),
                ("off", ctypes.c_uint64 * 3), ("info", ctypes.c_int32 * 4),
                ("prof", ctypes.c_int64 * 8), ("frob2", ctypes.c_double),
                ("tiny2", ctypes.c_double), ("offhist", ctypes.c_double * 64)]


OK, NOCONVERGE, RUNTIME = 0, 2, 3


@pytest.mark.skipif(not LIB.exists(), reason="libseemps_hip.so not built")
@pytest.mark.parametrize("abort,sweeps,converged,want", [
    (0, 7, 1, OK), (0, 60, 0, NOCONVERGE), (1, 7, 1, RUNTIME), (1, 0, 0, RUNTIME)])
def test_jacobi_status(abort, sweeps, converged, want):
    # seemps::ctrl_status(seemps::Ctrl const&, int*)
    status = ctypes.CDLL(str(LIB))._ZN6seemps11ctrl_statusERKNS_4CtrlEPi
    c = Ctrl(abort=abort)
    c.info[0], c.info[1] = sweeps, converged
    info = (ctypes.c_int32 * 2)()
    assert status(ctypes.byref(c), info) == want
    assert list(info) == [sweeps, converged]


APART, LOCAL, STRIDED = 0, 1, 2


@pytest.mark.skipif(not LIB.exists(), reason="libseemps_hip.so not built")
@pytest.mark.parametrize("P,R,VS,lim,want", [
    (4, 2, 2, (256, 256, 256), (APART, 16)), (4, 2, 2, (15, 256, 256), (LOCAL, 8)),
    (4, 2, 2, (256, 15, 256), (APART, 16)), (4, 2, 0, (256, 8, 256), (LOCAL, 8)),
    (4, 2, 0, (256, 7, 256), (STRIDED, 8)), (4, 2, 2, (15, 7, 3), (STRIDED, 3)),
    (1, 1, 0, (0, 1, 0), (LOCAL, 1)), (4, 2, 2, (0, 0, 0), None)])
def test_jacobi_form(P, R, VS, lim, want):
    # bool seemps::jacobi_plan(long, long, long, long const*, int*, int*)
    plan = ctypes.CDLL(str(LIB))._ZN6seemps11jacobi_planElllPKlPiS2_
    plan.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_void_p] * 3
    plan.restype = ctypes.c_bool
    variant, grid = ctypes.c_int(-1), ctypes.c_int(-1)
    ok = plan(P, R, VS, (ctypes.c_int64 * 3)(*lim), ctypes.byref(variant), ctypes.byref(grid))
    assert ((variant.value, grid.value) if ok else None) == want
