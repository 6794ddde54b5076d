"""The fib decode's table of partial sums as the host half keeps it, on the CPU
with the HIP runtime replaced by tests/host_hip.cpp: a profile whose table cannot
be allocated is created all the same and decodes by the kernel without one, and
profiles with equal constants share a table; a bounded decode walks any number of
tiles a segment table may have."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
TABLE = 32 ** 3 * 64 * 4   # bytes


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host_hip") / "libhost_hip.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "host_hip.cpp"), "-o", so], check=True)
    return so


def _child(stub, name):
    """Runs child_<name> of this file in a process of its own."""
    r = subprocess.run([sys.executable, os.path.abspath(__file__), stub, name], capture_output=True, text=True,
                       timeout=120, env={**os.environ, "PYTHONPATH": os.path.dirname(HERE)})
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("name", ["no_memory", "with_memory", "equal_constants", "many_tiles"])
def test_profile_creation(stub, name):
    _child(stub, name)


class Host:
    def __init__(self, stub):
        self.hip = C.CDLL(stub, mode=C.RTLD_GLOBAL)   # found ahead of the runtime's own
        self.hip.host_hip_live.argtypes = [C.c_size_t]
        self.hip.host_hip_fail_from.argtypes = [C.c_size_t]
        self.hip.host_hip_launched.restype = C.c_char_p
        from provekv_amd import _lib
        self.L = _lib.lib()
        self.ctx = C.c_void_p()
        assert self.L.pkv_ctx_create(0, C.byref(self.ctx)) == 0

    def tables(self):
        return self.hip.host_hip_live(TABLE)

    def profile(self, seed=0):
        rng = np.random.RandomState(seed)
        cb, rot, p = rng.randn(32, 4).astype(np.float32), np.eye(64), C.c_void_p()
        rc = self.L.pkv_fib_profile_create_with_constants(self.ctx, 64, 4, 32, cb.ctypes.data, rot.ctypes.data,
                                                          C.byref(p))
        assert rc == 0, rc
        return p

    def decode(self, prof, fanout):
        """The kernel a decode of 5 vectors into `fanout` f32 copies launches."""
        from provekv_amd.device import SEG_DTYPE
        segs = np.array([(0, 0, 64, 0, 5, 5)], dtype=SEG_DTYPE)
        wire, status = np.zeros(19 + 5 * 12 + 16, np.uint8), np.zeros(4, np.uint32)
        out = np.zeros(fanout * 5 * 64 + 4, np.float32)
        ptr = out.ctypes.data + -out.ctypes.data % 16
        rc = self.L.pkv_decode_segments_ex(self.ctx, prof, 0, wire.ctypes.data, wire.size, segs.ctypes.data, 1, ptr,
                                           0, fanout * 5 * 64, fanout, 5 * 64, status.ctypes.data, None)
        assert rc == 0, rc
        return self.hip.host_hip_launched().decode().split()[-1]


STAGED_NO_TABLE = "fib_decode_mfma_kernelILi64ELb1ELb0E"


def child_no_memory(h):
    h.hip.host_hip_fail_from(TABLE)
    prof = h.profile()
    assert h.tables() == 0
    for fanout in (1, 2, 4):
        assert STAGED_NO_TABLE in h.decode(prof, fanout)
    h.L.pkv_profile_destroy(prof)


def child_with_memory(h):
    prof = h.profile()
    assert h.tables() == 1
    assert "fib_decode_mfma_kernelILi64ELb0ELb1E" in h.decode(prof, 1)
    assert "fib_decode_mfma_kernelILi64ELb1ELb1E" in h.decode(prof, 2)
    assert STAGED_NO_TABLE in h.decode(prof, 4)
    h.L.pkv_profile_destroy(prof)
    assert h.tables() == 0


def child_equal_constants(h):
    a, b, other = h.profile(), h.profile(), h.profile(seed=1)
    assert h.tables() == 2
    h.L.pkv_profile_destroy(a)
    assert h.tables() == 2   # b's
    assert "fib_decode_mfma_kernelILi64ELb0ELb1E" in h.decode(b, 1)
    h.L.pkv_profile_destroy(b)
    assert h.tables() == 1
    b = h.profile()          # built again
    assert h.tables() == 2
    h.L.pkv_profile_destroy(b)
    h.L.pkv_profile_destroy(other)
    assert h.tables() == 0


def child_many_tiles(h):
    """More than 2^30 tiles of 256 vectors (one blob decoded again and again)."""
    from provekv_amd.device import SEG_DTYPE
    n, per = 1 << 24, 1 << 16   # vectors and tiles of a segment
    segs = np.array([(0, 0, 0, 0, n, n)] * ((1 << 30) // per + 1), dtype=SEG_DTYPE)
    status, buf = np.zeros(2 * len(segs), np.uint32), np.zeros(64, np.float32)
    ptr = buf.ctypes.data + -buf.ctypes.data % 16
    rc = h.L.pkv_decode_segments_bounded(h.ctx, h.profile(), 0, ptr, 19 + 12 * n, segs.ctypes.data, len(segs), ptr, 0,
                                         64, 1, 0, 640, status.ctypes.data, None)
    assert rc == 0, rc
    assert "fib_decode_mfma_kernel" in h.hip.host_hip_launched().decode().split()[-1]


if __name__ == "__main__":
    globals()[f"child_{sys.argv[2]}"](Host(sys.argv[1]))
