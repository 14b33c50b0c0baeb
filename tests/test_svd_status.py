"""Status of a finished block Jacobi from its control block, on the CPU: a wait
that ran out in any workgroup is an error, also when the workgroup that records
the sweeps had already left with "converged" (the workgroups that rotate V are
not counted in the last barrier)."""

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
