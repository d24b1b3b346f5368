"""What the collective calls from Python take for a stream, a count and a table of device
addresses: all that ctypes converts in a call of the C ABI, and nothing that it refuses.  Null
contexts, so that nothing reaches a device."""
import ctypes as C

import numpy as np
import pytest

import gpu_ipc_example_amd as vr
from gpu_ipc_example_amd import binding


def call(stream, ptrs=(8, 16), nelems=16, transport=vr.TRANSPORT_DIRECT):
    vr.lib()
    return binding._call.allreduce(0, C.c_uint32(1), "simple", transport, ptrs, None, nelems, stream)


def call_ctypes(stream, nelems=16, transport=vr.TRANSPORT_DIRECT):
    return vr.lib().vr_allreduce(None, stream, vr.algo_id("simple"), transport, (C.c_void_p * 2)(8, 16), None, nelems,
                                 C.byref(C.c_uint32(1)))


class Holder:
    def __init__(self, p):
        self._as_parameter_ = p


def same_as_ctypes(**where):
    """Taken or refused as ctypes does."""
    try:
        want = call_ctypes(**where)
    except C.ArgumentError as e:
        with pytest.raises(type(e)):
            call(**where)
        return False
    assert call(**where) == want != 0        # no context
    return True


def test_streams_that_ctypes_takes():
    for stream in (None, 0, 64, True, -1, 1 << 70, C.c_void_p(), C.c_void_p(64), Holder(C.c_void_p(64)),
                   Holder(C.c_void_p()), Holder(64), Holder(None), Holder(Holder(8)), C.pointer(C.c_int(3)),
                   C.byref(C.c_int(3)), (C.c_char * 8)(), C.c_char_p(b"x"), b"x", "x", Holder("x")):
        assert same_as_ctypes(stream=stream), stream
    for stream in (1.5, object(), [], C.c_int(4), C.c_size_t(4), Holder(1.5), Holder(C.c_int(4))):
        assert not same_as_ctypes(stream=stream), stream


@pytest.mark.parametrize("where", ["nelems", "transport"])
def test_numbers_that_ctypes_takes(where):
    exact = C.c_size_t if where == "nelems" else C.c_int
    for number in (1, True, np.int64(1), np.uint8(1), exact(1), Holder(1), Holder(exact(1)), Holder(Holder(1)), -1, 1 << 70):
        assert same_as_ctypes(stream=None, **{where: number}), number
    for number in (16.0, None, "16", b"16", object(), C.c_short(16), Holder(16.0)):
        assert not same_as_ctypes(stream=None, **{where: number}), number


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


def test_the_module_is_built_for_one_interpreter_where_its_headers_are():
    """Its name carries the interpreter's tag; without Python's headers the library and the CLI
    are built all the same."""
    import os
    import subprocess
    import sys
    import sysconfig
    headers = os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h"))
    if headers:
        assert binding._call.__file__.endswith("_call" + sysconfig.get_config_var("EXT_SUFFIX"))
    csrc = os.path.join(os.path.dirname(binding.__file__), "csrc")
    for include, built in ((sysconfig.get_paths()["include"], headers), ("/nonexistent", False)):
        r = subprocess.run(["make", "-n", "-B", "-C", csrc, "PYTHON=" + sys.executable, "PYINC=" + include], capture_output=True,
                           text=True, timeout=120)
        assert r.returncode == 0 and "libvrank_allreduce.so" in r.stdout and "vr_main" in r.stdout
        assert ("vr_pycall.c" in r.stdout) == built


def test_the_calls_through_ctypes():
    """What stands in for the module where it was not built: the same results of the same calls."""
    vr.lib()
    for outs in (None, (24, 32)):
        for algo, n in (("simple", 16), ("allgather_simple", 16), ("simple", 1 << 41)):
            a, b = C.c_uint32(3), C.c_uint32(3)
            args = (algo, vr.TRANSPORT_DIRECT, [8, 16], outs, n, None)
            assert binding._call.allreduce(0, a, *args) == binding._CtypesCalls.allreduce(0, b, *args) != 0
            assert binding._call.allgather(0, a, *args) == binding._CtypesCalls.allgather(0, b, *args) != 0
            assert a.value == b.value == 3
            args = (algo, [8, 16], outs, n, None)
            assert binding._call.allreduce_static(0, *args) == binding._CtypesCalls.allreduce_static(0, *args) != 0
