"""Which panels of the direct solver exchange pivots between workgroups: those
whose workgroups of 256 rows the device holds at once, at most 64."""
import ctypes as C
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_route(tmp_path):
    from mstm_amd.build import HIPCC

    so = str(tmp_path / "lu_route_host.so")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-fPIC", "-shared",
                    os.path.join(HERE, "native", "lu_route_host.cpp"), "-o", so], check=True)
    exchanges = C.CDLL(so).lu_route_host
    assert exchanges(16384, 256) and not exchanges(16385, 256)
    assert exchanges(8192, 32) and not exchanges(8193, 32)  # a partition of 32 CUs
    assert exchanges(1, 1) and exchanges(256, 1) and not exchanges(257, 1)
    assert not exchanges(1, 0)  # not known, or refused
