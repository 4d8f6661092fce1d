"""GPU: the B^T B engine on a work buffer of the caller's allocates no device
memory while it runs."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# a process of its own: the library's buffers are as a first call finds them
CODE = """
import ctypes as C, sys
import numpy as np
from ca3dmm_amd import device as hip, engine as E
n, k, force = int(sys.argv[1]), int(sys.argv[2]), sys.argv[3]
rt = C.CDLL("libamdhip64.so.7")
B = np.random.default_rng(5).integers(-3, 4, (k, n)).astype(float)
dB, dC = hip.DeviceArray.from_numpy(B), hip.DeviceArray.filled((n, n), 0xFF)
eng, bytes_ = E.CA3P(), C.c_size_t()
E.lib.ca3dmm_engine_init_BTB(n, k, 0, k, 0, n, 0, n, 0, n, None, E.comm_self(), E.DEV_TYPE_HIP, C.byref(eng),
                             C.byref(bytes_))
work = hip.DeviceArray.zeros((bytes_.value // 8 + 1,))
E.lib.ca3dmm_engine_attach_workbuf(eng, None, work.ptr)
hip.copy_matrix_block(8, 1, 1, dB.ptr, 1, work.ptr, 1)             # the runtime's own start-up
def free():
    a, b = C.c_size_t(), C.c_size_t()
    assert rt.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value
hip.sync()
before = free()
E.lib.ca3dmm_engine_exec(eng, None, 0, dB.ptr, k, dC.ptr, n)
hip.sync()
after = free()
assert np.array_equal(dC.numpy(), B.T @ B)
assert before - after < 16 << 20, (before, after)
print("fine")
"""


@pytest.mark.parametrize("n,k,force", [(1000, 20000, "0"), (512, 30001, "1"), (3968, 3000, "0")])
def test_exec_allocates_nothing(hip, n, k, force):
    env = dict(os.environ, CA3DMM_FORCE_REDIST=force)
    out = subprocess.run([sys.executable, "-c", CODE, str(n), str(k), force], cwd=ROOT, env=env, capture_output=True,
                         text=True, timeout=100)
    assert out.returncode == 0 and "fine" in out.stdout, out.stdout + out.stderr
