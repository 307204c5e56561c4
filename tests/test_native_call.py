"""lib/hk_call.so and lib/ht_call.so: what an argument may be, and that what is no such thing is refused before the entry point runs."""
import importlib
import os
import subprocess
import sys
import sysconfig

import pytest
import torch


@pytest.fixture(scope="module")
def call():
    return importlib.import_module("hotspa-ae_amd.capi").native()


def test_operands_are_asked_for_their_layout(call):
    x = torch.zeros(3, 4, 5)
    assert call.rows_cols(x) == (12, 5) and call.rows_cols(x[:, :0]) == (0, 5) and call.rows_cols(x[..., :0]) == (0, 0)
    assert call.rows_cols(torch.zeros(7)) == (1, 7)
    assert call.dense(x, None, x[1]) is True and call.dense(x, x.transpose(0, 1)) is False
    with pytest.raises(IndexError):
        call.rows_cols(torch.zeros(()))
    with pytest.raises(AttributeError):
        call.dense([1, 2])


def test_values_are_refused_before_the_call(hk, call):
    ops = importlib.import_module("hotspa-ae_amd.hetu_ops")
    x, out = torch.ones(2, 3), torch.zeros(2)
    with pytest.raises(AttributeError):
        hk.sce_sparse_fwd(x, [0, 1], out, -100, stream=0)          # labels lie on the device
    with pytest.raises(TypeError):
        ops.native().ht_reduce(x, out, torch.tensor([1]), 1, 0, 1)         # axes do not
    with pytest.raises(TypeError):
        call.hk_unary(0, 6, x, x)
    with pytest.raises(AssertionError):
        ops.softmax(torch.ones([1] * 9), torch.ones([1] * 9), 0)
    with pytest.raises(KeyError):
        ops.softmax(torch.ones(2, 3, dtype=torch.complex64), x, 1)
    with pytest.raises(hk.HkError):
        hk.check(call.hk_unary(99, 6, x, x, 6, 0))


def test_numbers_convert_like_c(call):
    ops = importlib.import_module("hotspa-ae_amd.hetu_ops")
    import numpy as np
    x, out = torch.randn(4, 6), torch.empty(4, 6)
    for dim in (1, True, np.int64(1), 1.0):
        out.zero_()
        ops.softmax(x, out, dim)
        assert torch.allclose(out, torch.softmax(x, 1), atol=1e-6)
    s = torch.empty(1, 6)
    for axes in ((0,), [0], range(1)):
        ops.ndarray_reduce(x, "sum", axes, np.bool_(True), s)
        assert torch.allclose(s[0], x.sum(0), atol=1e-5)
    ops.ndarray_binary("add", x[:, ::2], x[:, ::2], out[:, :3].contiguous())   # strided operands are described as they are


def test_a_long_or_changing_list_of_integers(call):
    ops = importlib.import_module("hotspa-ae_amd.hetu_ops")
    x, s = torch.randn(4, 6), torch.empty(6)
    ops.ndarray_reduce(x, "sum", [0] * 40, False, s)     # more of them than the fixed array holds; duplicates are one axis
    assert torch.allclose(s, x.sum(0), atol=1e-5)

    class Shrinks:
        def __int__(self):
            axes.clear()
            return 0
    axes = [Shrinks(), 1]
    with pytest.raises(ValueError):
        ops.native().ht_reduce(x, s, axes, 2, 0, 1)


def test_an_exception_of_an_entry_point_is_raised_with_the_lock_held(tmp_path):
    """In a process of its own: what leaves an entry point without the interpreter's lock ends the program."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    lib = os.path.join(root, "hotspa-ae_amd", "lib")
    out = str(tmp_path / "throwing_entries.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-I" + os.path.join(root, "include"),
                    "-I" + sysconfig.get_paths()["include"], os.path.join(root, "tests", "cpp", "throwing_entries.cc"), "-o", out,
                    "-L" + lib, "-lhk_rowwise", "-Wl,-rpath," + lib], check=True)
    code = """
import importlib.util, threading
spec = importlib.util.spec_from_file_location("throwing_entries", %r)
m = importlib.util.module_from_spec(spec)
spec.loader.exec_module(m)
def raised(what, *args):
    try:
        return m.throws(what, *args)
    except Exception as e:
        return type(e).__name__, str(e)
def check():
    for _ in range(100):
        assert raised(0, [7]) == 7
        assert raised(1, None)[0] == "MemoryError"
        assert raised(2, list(range(40))) == ("RuntimeError", "a list too long")
        assert raised(3, None)[0] == "RuntimeError"
threads = [threading.Thread(target=check) for _ in range(4)]
[t.start() for t in threads]
[t.join() for t in threads]
check()
print("done")
""" % out
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0 and done.stdout == "done\n" and "Error" not in done.stderr, (done.returncode, done.stderr)
