"""The host side of nt_attention_schedule where it ends before any launch."""
import subprocess
import sys

OUT_OF_MEMORY = """
import ctypes, resource
import numpy as np
from nestedtensor_amd import _C
B = 1 << 23
lens = np.full(B, 3, dtype=np.int64)
p = lens.ctypes.data_as(ctypes.c_void_p)
n = _C.lib.nt_attention_schedule_items(p, B, 128)
assert n == B
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (64 << 20), resource.RLIM_INFINITY))
rc = _C.lib.nt_attention_schedule(p, p, B, 128, p, n, None)     # 20 bytes a sequence: 160 MiB
print("rc", rc, _C.lib.nt_last_error())
"""


def test_out_of_host_memory_is_an_error_code():
    # no C++ exception may leave a C entry point
    got = subprocess.run([sys.executable, "-c", OUT_OF_MEMORY], capture_output=True, text=True, timeout=300)
    assert got.returncode == 0, got.stderr[-500:]
    assert "rc 2" in got.stdout and "no host memory" in got.stdout
