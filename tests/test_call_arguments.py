"""What the collective calls from Python take for a stream and for a table of device addresses:
all that ctypes converts to a c_void_p.  Null contexts, so that nothing reaches a device."""
import ctypes as C

import pytest

import gpu_ipc_example_amd as vr
from gpu_ipc_example_amd import binding


def call(stream, ptrs=(8, 16)):
    vr.lib()
    return binding._call.allreduce(0, C.c_uint32(1), "simple", vr.TRANSPORT_DIRECT, ptrs, None, 16, stream)


class Holder:
    def __init__(self, p):
        self._as_parameter_ = p


def test_streams_that_ctypes_takes():
    want = call(None)
    assert want != 0        # no context
    for stream in (0, 64, C.c_void_p(), C.c_void_p(64), Holder(C.c_void_p(64)), Holder(C.c_void_p()), Holder(64),
                   Holder(None)):
        assert call(stream) == want
    for stream in ("x", 1.5, object(), [], Holder("x")):
        with pytest.raises((TypeError, AttributeError)):
            call(stream)


def test_tables():
    want = call(None)
    for ptrs in ((8, 16), [8, 16], (8, 16.0), [8] * 17, []):
        assert call(None, ptrs) == want
    for ptrs in ([None, 8], 5, [[]]):
        with pytest.raises(TypeError):
            call(None, ptrs)


class Shrinks:
    """An address whose conversion empties the list it came from."""

    def __init__(self, table):
        self.table = table

    def __int__(self):
        self.table.clear()
        return 8


def test_tables_that_change_while_they_are_read():
    """In a process of its own: a table read beyond its end would end that process."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = ("from tests.test_call_arguments import Shrinks, call\n"
            "for n in (1, 2, 16):\n"
            "    table = []\n"
            "    table.extend([Shrinks(table)] + [8] * (n - 1))\n"
            "    assert call(None, table) == call(None)\n"
            "print('read whole')\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "read whole" in r.stdout, (r.returncode, r.stderr)
