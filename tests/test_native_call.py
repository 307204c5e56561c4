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
        def __index__(self):
            axes.clear()
            return 0
    axes = [Shrinks(), 1]
    with pytest.raises(ValueError):
        ops.native().ht_reduce(x, s, axes, 2, 0, 1)


def test_what_is_no_integer_is_refused(hk, call):
    """Axes, flags, streams, the numbers that ctypes took as they are: an integer of any type and nothing else.  Where
    the wrappers call int() or float() themselves (dim, eps, the truth values), what these take goes through."""
    import numpy as np
    ops = importlib.import_module("hotspa-ae_amd.hetu_ops")
    x, out = torch.randn(4, 6), torch.full((4,), 5.0)

    class One:
        def __index__(self):
            return 1
    for no in (1.9, 1.0, "1", np.float32(1), None, torch.tensor(1.5)):
        for refused in (lambda: ops.reduce(x, out, [no], "sum"), lambda: ops.reduce(x, out, [1], "sum", stream=no),
                        lambda: ops.ndarray_reduce(x, "sum", [no], False, out),
                        lambda: ops.reduce_gradient(out, x.clone(), "sum", [no], [False]),
                        lambda: ops.broadcast_shape(out, x.clone(), [no]),
                        lambda: ops.ndarray_layernorm(x, x[0], x[0], no, 1e-5, True, x.clone()),
                        lambda: call.hk_unary(0, 6, x, x, no, 0)):
            with pytest.raises(TypeError):
                refused()
        with pytest.raises((TypeError, AttributeError)):
            hk.unary("exp", x[:0], x[:0], stream=1.5)
    assert (out == 5.0).all()
    for yes in (1, True, np.int8(1), np.uint64(1), One(), torch.tensor(1), -1):
        ops.reduce(x, out.fill_(0), [yes], "sum")
        assert torch.allclose(out, x.sum(1), atol=1e-5)
    y, want = torch.empty(4, 6), torch.softmax(x, 1)
    for dim in (1, 1.0, "1", np.float32(1.0)):
        ops.softmax(x, y.fill_(0), dim)
        assert torch.allclose(y, want, atol=1e-6)
    mean, var = torch.empty(4), torch.empty(4)
    for eps in (1e-5, "1e-5", np.float64(1e-5), 0):
        ops.layer_norm(x, x[0].contiguous(), x[1].contiguous(), mean, var, y, 1, eps)
        assert torch.allclose(y, torch.nn.functional.layer_norm(x, (6,), x[0], x[1], float(eps)), atol=1e-5)


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


def test_a_forked_child_asks_for_the_stream_anew():
    """A child of fork() cannot use its parent's device: torch's current_stream() refuses there, so it has to be asked, as
    before the first call.  With stand-ins for torch's functions, in a process of its own, without a device."""
    code = """
import importlib, os
capi = importlib.import_module("hotspa-ae_amd.capi")
call, parent, asked = capi.native(), os.getpid(), []
def current_stream():
    if os.getpid() != parent:
        raise RuntimeError("a forked child")
    asked.append(1)
    return 0
call.setup(capi._dtype_codes(), current_stream, lambda: 0, lambda device: 0)
for _ in range(3):
    assert call.hk_unary(0, 6, None, None, 0, None) == 0     # no elements: nothing is launched
assert asked == [1]
pid = os.fork()
if pid == 0:
    try:
        call.hk_unary(0, 6, None, None, 0, None)
    except RuntimeError as e:
        os._exit(7 if "a forked child" in str(e) else 1)
    os._exit(0)
assert os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1]) == 7
assert call.hk_unary(0, 6, None, None, 0, None) == 0 and asked == [1]
print("done")
"""
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120,
                          cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert done.returncode == 0 and done.stdout == "done\n", done.stderr
