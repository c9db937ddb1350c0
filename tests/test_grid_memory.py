"""wx_grid_create without host memory for its check: an error code, not an exception through
the C interface (which would end the process)."""
import subprocess
import sys

PROGRAM = """
import ctypes as C, resource
import numpy as np
import woxel_amd as wx

root = np.zeros(4, np.int32)
n5 = np.zeros(16384, np.uint32)
n4 = np.zeros((1 << 20) * 1024, np.uint32)  # never touched: pages of the zero page
d = wx.GridDesc()
d.n5, d.n4, d.n3, d.bound = 1, 1 << 20, 0, 4096.0
d.root = root.ctypes.data_as(C.POINTER(C.c_int32))
d.n5_records, d.n4_records = [a.ctypes.data_as(C.POINTER(C.c_uint32)) for a in (n5, n4)]
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
old = resource.getrlimit(resource.RLIMIT_AS)
resource.setrlimit(resource.RLIMIT_AS, (used + (8 << 20), old[1]))
hold = []
try:
    while True:
        hold.append(bytearray(1 << 20))
except MemoryError:
    pass
h = C.c_void_p()
rc = wx.lib.wx_grid_create(C.byref(d), C.byref(h))
resource.setrlimit(resource.RLIMIT_AS, old)
print("code", rc, wx.lib.wx_last_error().decode())
"""


def test_no_host_memory_is_an_error_code():
    r = subprocess.run([sys.executable, "-c", PROGRAM], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stderr[-500:])
    assert "host allocation failed" in r.stdout, r.stdout
