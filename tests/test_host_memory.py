"""Calls whose lists do not fit in host memory return an error: no C++ exception leaves libkvx's C functions."""

import subprocess
import sys

import pytest

from conftest import ROOT

# The limit on the address space leaves no room for the copies that the calls make of their lists. They are refused
# before any device work, so no device is needed.
SCRIPT = """
import ctypes, resource, sys
sys.path[:0] = [{package!r}]
import numpy as np
from kvx import _lib

n = 4 << 20
layout = _lib.BlockLayout(n * 8, 8, 1, 1, 8, n, 2, 0)
ids = np.arange(n, dtype=np.int32)
entries = (np.arange(n, dtype=np.uint64) + 1) * 256
handle = _lib.lib()
ids_p = ids.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))
entries_p = entries.ctypes.data_as(ctypes.POINTER(ctypes.c_uint64))
out = ctypes.c_void_p()
pages = int(open("/proc/self/statm").read().split()[0])
limit = pages * resource.getpagesize() + (4 << 20)
resource.setrlimit(resource.RLIMIT_AS, (limit, limit))
print(handle.{call})
print(handle.kvx_last_error().decode())
"""

CALLS = {
    "save": "kvx_save_blocks(4096, ctypes.byref(layout), 1, ids_p, entries_p, n, 8, None)",
    "restore": "kvx_restore_blocks(4096, ctypes.byref(layout), 1, ids_p, entries_p, n, 8, None)",
    "scatter": "kvx_scatter_tokens(4096, ctypes.byref(layout), ids_p, n, n, 1 << 32, None)",
    "scatter_fp8": "kvx_scatter_tokens_fp8(4096, ctypes.byref(layout), ids_p, n, n, 1 << 32, 1 << 36, None)",
    "cache_create": "kvx_cache_create(4096, ctypes.byref(layout), 1, 16, 32, 0, ctypes.byref(out))",
}


@pytest.mark.parametrize("call", CALLS)
def test_lists_beyond_host_memory_are_refused(call):
    script = SCRIPT.format(package=str(ROOT / "kv-cache-offloading_amd"), call=CALLS[call])
    run = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, (run.returncode, run.stderr[-2000:])
    status, message = run.stdout.strip().splitlines()
    assert status == "-3" and "out of host memory" in message, run.stdout
