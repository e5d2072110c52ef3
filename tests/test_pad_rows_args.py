"""lucid_pad_rows rejects null arrays and null tensors before anything is launched (on the CPU)."""
import os
import subprocess
import sys

CALLS = """
import ctypes
from lucid_amd import _lib
lib = _lib.load()
for which, inner in ((0, False), (1, False), (2, False), (3, False), (0, True), (3, True)):
    args = [(ctypes.c_void_p * 1)(1 << 20), (ctypes.c_int64 * 3)(64, 64, 64), (ctypes.c_int * 1)(1),
            (ctypes.c_void_p * 1)(1 << 20)]
    if inner:
        args[which][0] = None
    else:
        args[which] = None
    print(which, inner, flush=True)
    rc = lib.lucid_pad_rows(1, *args, 1, 1, 128, 64, 64, 0, None)
    assert rc == _lib.LUCID_EINVAL, rc
    assert b"null" in lib.lucid_last_error(), lib.lucid_last_error()
"""


def test_null_arguments():
    # in a process of its own: a null that is read ends it
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CALLS], capture_output=True, text=True, timeout=120, cwd=root)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr[-500:])
