"""Bindings of include/hetu_ops_c.h: the C++ operator layer (libhetu_rowwise.so)
called, through lib/ht_call.so, with torch tensors as borrowed arrays.

Errors of the C++ layer come back as Python exceptions named after the C++
ones (AssertionError_, NotImplemented_, ValueError_, RuntimeError_).
"""
import ctypes
import os

from . import capi

_HERE = os.path.dirname(os.path.abspath(__file__))
_LIB = os.path.join(_HERE, "lib", "libhetu_rowwise.so")
_lib = None

RED = {"sum": 0, "mean": 1, "max": 2, "min": 3, "prod": 4, "none": 5}
MAX_NDIM = 8
DEFAULT_STREAM = 1   # hetu::kComputingStream


class HetuError(RuntimeError):
    kind = "other"


class AssertionError_(HetuError):
    kind = "assertion_error"


class NotImplemented_(HetuError):
    kind = "not_implemented"


class ValueError_(HetuError):
    kind = "value_error"


class RuntimeError_(HetuError):
    kind = "runtime_error"


class BadAlloc_(HetuError):
    kind = "bad_alloc"


_KINDS = {1: AssertionError_, 2: NotImplemented_, 3: ValueError_, 4: RuntimeError_, 5: BadAlloc_}


class HtArray(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p), ("dtype", ctypes.c_int32), ("ndim", ctypes.c_int32),
                ("shape", ctypes.c_int64 * MAX_NDIM), ("stride", ctypes.c_int64 * MAX_NDIM),
                ("device_type", ctypes.c_int32), ("device_index", ctypes.c_int32)]


def lib_path():
    return _LIB


def lib():
    """Loads libhetu_rowwise.so; raises if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(_LIB):
            raise HetuError("native library %s is missing: run __graft_entry__.build() first" % _LIB)
        capi.lib()   # libhk_rowwise.so first, so the dependency resolves from the same folder
        _lib = ctypes.CDLL(_LIB)
        _lib.ht_last_error.restype = ctypes.c_char_p
    return _lib


def check(rc):
    if rc != 0:
        raise _KINDS.get(rc, HetuError)(lib().ht_last_error().decode("utf-8", "replace"))


def desc(t):
    """HtArray borrowing a torch tensor (None -> NULL = undefined NDArray), for calls through lib()."""
    if t is None:
        return None
    assert t.dim() <= MAX_NDIM
    a = HtArray()
    a.data = t.data_ptr()
    a.dtype = capi.dtype_code(t)
    a.ndim = t.dim()
    for i in range(t.dim()):
        a.shape[i] = t.shape[i]
        a.stride[i] = t.stride(i)
    a.device_type = 1 if t.is_cuda else 0
    a.device_index = t.device.index or 0 if t.is_cuda else 0
    a._keep = t
    return a


_CALL = os.path.join(_HERE, "lib", "ht_call.so")
_native = None


def native():
    """ht_call.so; raises if it has not been built."""
    global _native
    if _native is None:
        lib()
        _native = capi.load_binding(_CALL, HetuError("native library %s is missing: run __graft_entry__.build() first" % _CALL))
    return _native


def _call(name, *args):
    check(getattr(_native or native(), name)(*args))


def stream_sync(stream=DEFAULT_STREAM, device=0):
    check(lib().ht_stream_sync(ctypes.c_int(device), ctypes.c_int(stream)))


def host_stream_sync(stream=DEFAULT_STREAM):
    """Waits for the host stream of that index and raises what a host kernel on it failed with."""
    check(lib().ht_host_stream_sync(ctypes.c_int(stream)))


def set_host_async(on):
    """Host calls return once their work is on its stream (True) or once it has finished (False, the default);
    returns the previous setting.  While on, the caller keeps the arrays alive until host_stream_sync."""
    return bool(lib().ht_set_host_async(ctypes.c_int(int(bool(on)))))


def set_host_threads(n):
    """OpenMP team size of the host twins; returns the size now in force (n <= 0 only asks)."""
    return int(lib().ht_set_host_threads(ctypes.c_int(int(n))))


def synchronize_all():
    check(lib().ht_synchronize_all())


# ---- kernel entry points --------------------------------------------------
def layer_norm(x, scale, bias, mean, var, out, reduce_dims, eps, stream=DEFAULT_STREAM):
    _call("ht_layer_norm", x, scale, bias, mean, var, out, int(reduce_dims),
          float(eps), stream)


def layer_norm_gradient(dy, x, scale, dx, dscale, dbias, mean, var, reduce_dims, eps, stream=DEFAULT_STREAM):
    _call("ht_layer_norm_gradient", dy, x, scale, dx, dscale, dbias, mean,
          var, int(reduce_dims), float(eps), stream)


def fused_layer_norm(x, scale, bias, mean, invvar, out, reduce_dims, eps, stream=DEFAULT_STREAM):
    _call("ht_fused_layer_norm", x, scale, bias, mean, invvar, out,
          int(reduce_dims), float(eps), stream)


def fused_layer_norm_gradient(dy, x_or_y, scale, bias, dx, dscale, dbias, mean, invvar, reduce_dims, eps, inplace,
                              stream=DEFAULT_STREAM):
    _call("ht_fused_layer_norm_gradient", dy, x_or_y, scale, bias, dx, dscale,
          dbias, mean, invvar, int(reduce_dims), float(eps), int(inplace),
          stream)


def dropout_add_ln_fwd(x0, residual, gamma, beta, z, x, mu, rsigma, eps, is_rms_norm, dropout_p=0.0,
                       rowscale=None, colscale=None, residual_in_fp32=False, x0_subset=None, z_subset=None,
                       dmask=None, rowscale_const=1.0, z_numrows=0, stream=DEFAULT_STREAM):
    _call("ht_dropout_add_ln_fwd", x0, residual, gamma, beta, rowscale,
          colscale, x0_subset, z_subset, z, x, dmask, mu, rsigma,
          float(dropout_p), float(eps), float(rowscale_const), int(z_numrows), int(residual_in_fp32),
          int(is_rms_norm), stream)


def dropout_add_ln_bwd(dz, dx, x, mu, rsigma, gamma, dx0, dresidual, dgamma, dbeta, has_residual, is_rms_norm,
                       dropout_p=0.0, rowscale=None, colscale=None, x0=None, dmask=None, x0_subset=None,
                       z_subset=None, dcolscale=None, rowscale_const=1.0, x0_numrows=0, stream=DEFAULT_STREAM):
    _call("ht_dropout_add_ln_bwd", dz, dx, x, x0, dmask, mu, rsigma,
          gamma, rowscale, colscale, x0_subset, z_subset, dx0,
          dresidual, dgamma, dbeta, dcolscale, float(dropout_p), float(rowscale_const),
          int(x0_numrows), int(has_residual), int(is_rms_norm), stream)


def dropout_add_ln_parallel_residual_fwd(x0, x1, residual, gamma0, beta0, gamma1, beta1, z0, z1, x, dmask0, dmask1,
                                         mu, rsigma, dropout_p, eps, residual_in_fp32=False, is_rms_norm=False,
                                         stream=DEFAULT_STREAM):
    _call("ht_dropout_add_ln_parallel_residual_fwd", x0, x1, residual, gamma0, beta0,
          gamma1, beta1, z0, z1, x, dmask0, dmask1, mu,
          rsigma, float(dropout_p), float(eps), int(residual_in_fp32),
          int(is_rms_norm), stream)


def dropout_add_ln_parallel_residual_bwd(dz0, dz1, dx, x, dmask0, dmask1, mu, rsigma, gamma0, gamma1, dx0, dx1,
                                         dresidual, dgamma0, dbeta0, dgamma1, dbeta1, dropout_p, has_x1,
                                         has_residual, is_rms_norm=False, stream=DEFAULT_STREAM):
    _call("ht_dropout_add_ln_parallel_residual_bwd", dz0, dz1, dx, x, dmask0,
          dmask1, mu, rsigma, gamma0, gamma1, dx0, dx1, dresidual,
          dgamma0, dbeta0, dgamma1, dbeta1, float(dropout_p), int(has_x1),
          int(has_residual), int(is_rms_norm), stream)


BINARY_OPS = {"add": 0, "sub": 1, "mul": 2, "div": 3}
UNARY_OPS = {"exp": 0, "log": 1, "neg": 2, "sqrt": 3}


def binary(op, a, b, out, stream=DEFAULT_STREAM):
    _call("ht_binary", BINARY_OPS[op], a, b, out, stream)


def binary_const(op, x, value, out, stream=DEFAULT_STREAM):
    """AddConst / SubConst (value - x) / MulConst / DivConst (value / x)."""
    _call("ht_binary_const", BINARY_OPS[op], x, value, out,
          stream)


def unary(op, x, out, stream=DEFAULT_STREAM):
    _call("ht_unary", UNARY_OPS[op], x, out, stream)


def ndarray_binary(op, a, b, out=None, in_place=False, stream=DEFAULT_STREAM):
    _call("ht_ndarray_binary", BINARY_OPS[op], a, b, out,
          int(in_place), stream)


def ndarray_unary(op, x, out=None, in_place=False, stream=DEFAULT_STREAM):
    _call("ht_ndarray_unary", UNARY_OPS[op], x, out, int(in_place),
          stream)


def vocab_parallel_cross_entropy(logits, labels, vocab_start, vocab_end, ignored_index, picked, lse,
                                 stream=DEFAULT_STREAM):
    _call("ht_vocab_parallel_cross_entropy", logits, labels, int(vocab_start), int(vocab_end),
          int(ignored_index), picked, lse, stream)


def vocab_parallel_cross_entropy_gradient(softmax, labels, vocab_start, vocab_end, ignored_index, grad_loss, out,
                                          stream=DEFAULT_STREAM):
    _call("ht_vocab_parallel_cross_entropy_gradient", softmax, labels, int(vocab_start),
          int(vocab_end), int(ignored_index), grad_loss, out, stream)


def norm(x, out, dim, p, stream=DEFAULT_STREAM):
    _call("ht_norm", x, out, int(dim), int(p), stream)


def norm_gradient(x, norm_out, grad, dx, dim, p, stream=DEFAULT_STREAM):
    _call("ht_norm_gradient", x, norm_out, grad, dx, int(dim), int(p), stream)


def ndarray_norm(x, p, dim, keepdim, out, stream=DEFAULT_STREAM):
    _call("ht_ndarray_norm", x, int(p), int(dim), int(keepdim), out, stream)


def batch_norm(x, scale, bias, y, momentum, eps, running_mean, running_var, save_mean, save_var,
               stream=DEFAULT_STREAM):
    _call("ht_batch_norm", x, scale, bias, y, momentum, eps,
          running_mean, running_var, save_mean, save_var, stream)


def batch_norm_gradient(dy, x, scale, dx, dscale, dbias, eps, save_mean, save_var, stream=DEFAULT_STREAM):
    _call("ht_batch_norm_gradient", dy, x, scale, dx, dscale, dbias,
          eps, save_mean, save_var, stream)


def set_random_seed(seed):
    _call("ht_set_random_seed", seed)


def instance_norm(x, mean, var, out, eps, stream=DEFAULT_STREAM):
    _call("ht_instance_norm", x, mean, var, out, float(eps), stream)


def instance_norm_gradient(dy, x, dx, mean, var, eps, stream=DEFAULT_STREAM):
    _call("ht_instance_norm_gradient", dy, x, dx, mean, var, float(eps),
          stream)


def softmax(x, out, dim, stream=DEFAULT_STREAM):
    _call("ht_softmax", x, out, int(dim), stream)


def softmax_gradient(y, dy, dx, dim, stream=DEFAULT_STREAM):
    _call("ht_softmax_gradient", y, dy, dx, int(dim), stream)


def softmax_cross_entropy(pred, label, loss, stream=DEFAULT_STREAM):
    _call("ht_softmax_cross_entropy", pred, label, loss, stream)


def softmax_cross_entropy_gradient(pred, label, grad_loss, out, stream=DEFAULT_STREAM):
    _call("ht_softmax_cross_entropy_gradient", pred, label, grad_loss, out,
          stream)


def softmax_cross_entropy_sparse(pred, label, loss, ignored_index, stream=DEFAULT_STREAM):
    _call("ht_softmax_cross_entropy_sparse", pred, label, loss, int(ignored_index),
          stream)


def softmax_cross_entropy_sparse_gradient(pred, label, grad_loss, out, ignored_index, stream=DEFAULT_STREAM):
    _call("ht_softmax_cross_entropy_sparse_gradient", pred, label, grad_loss, out,
          int(ignored_index), stream)


def nll_loss(pred, label, loss, stream=DEFAULT_STREAM):
    _call("ht_nll_loss", pred, label, loss, stream)


def nll_loss_gradient(pred, label, grad_loss, out, stream=DEFAULT_STREAM):
    _call("ht_nll_loss_gradient", pred, label, grad_loss, out, stream)


def reduce(x, out, axes, red_type, stream=DEFAULT_STREAM):
    ax = list(axes)
    _call("ht_reduce", x, out, ax, len(ax), RED[red_type], stream)


# ---- NDArray statics ------------------------------------------------------
def ndarray_reduce(x, red_type, axes, keepdims, out, stream=DEFAULT_STREAM):
    ax = list(axes)
    _call("ht_ndarray_reduce", x, RED[red_type], ax, len(ax), int(keepdims), out,
          stream)


def ndarray_softmax(x, dim, out, stream=DEFAULT_STREAM):
    _call("ht_ndarray_softmax", x, int(dim), out, stream)


def ndarray_layernorm(x, scale, bias, normalized_ndim, eps, fused, out, mean=None, var=None,
                      stream=DEFAULT_STREAM):
    _call("ht_ndarray_layernorm", x, scale, bias, normalized_ndim,
          eps, int(fused), out, mean, var, stream)


def ndarray_sceloss(preds, labels, out, reduction="mean", ignored_index=None, stream=DEFAULT_STREAM):
    sparse = ignored_index is not None
    _call("ht_ndarray_sceloss", preds, labels, int(sparse),
          int(ignored_index) if sparse else 0, RED[reduction], out, stream)


# ---- gradients of the reductions and of the reduced losses ----------------
def broadcast_shape(x, out, add_axes=(), const_value=None, stream=DEFAULT_STREAM):
    """BroadcastShapeCuda, or BroadcastShapeMulCuda when const_value is given."""
    ax = list(add_axes)
    _call("ht_broadcast_shape", x, int(const_value is not None),
          0.0 if const_value is None else const_value, out, ax, len(ax), stream)


def reduce_gradient(grad_output, out, reduction, axes, keepdims, stream=DEFAULT_STREAM):
    ax = list(axes)
    keep = [keepdims] if isinstance(keepdims, bool) else list(keepdims)
    _call("ht_reduce_gradient", grad_output, RED[reduction], ax, len(ax), [int(k) for k in keep],
          len(keep), out, stream)


def sceloss_gradient(preds, labels, grad_output, out, reduction="mean", ignored_index=None, fused=True,
                     stream=DEFAULT_STREAM):
    sparse = ignored_index is not None
    _call("ht_sceloss_gradient", preds, labels, grad_output, int(sparse),
          int(ignored_index) if sparse else 0, RED[reduction], int(fused), out,
          stream)


# ---- device memory pool ---------------------------------------------------
class PoolBlock:
    def __init__(self, ptr, ident, size, device):
        self.ptr, self.id, self.size, self.device = ptr, ident, size, device


def pool_alloc(nbytes, stream=DEFAULT_STREAM, device=0):
    ptr, ident, granted = ctypes.c_void_p(), ctypes.c_uint64(), ctypes.c_size_t()
    check(lib().ht_pool_alloc(ctypes.c_int(device), ctypes.c_size_t(nbytes), ctypes.c_int(stream),
                              ctypes.byref(ptr), ctypes.byref(ident), ctypes.byref(granted)))
    return PoolBlock(ptr.value or 0, ident.value, granted.value, device)


def pool_free(block):
    check(lib().ht_pool_free(ctypes.c_int(block.device), ctypes.c_void_p(block.ptr), ctypes.c_uint64(block.id),
                             ctypes.c_size_t(block.size)))


def pool_mark_used(block, stream):
    check(lib().ht_pool_mark_used(ctypes.c_int(block.device), ctypes.c_void_p(block.ptr), ctypes.c_uint64(block.id),
                                  ctypes.c_size_t(block.size), ctypes.c_int(stream)))


def pool_empty_cache(device=0):
    check(lib().ht_pool_empty_cache(ctypes.c_int(device)))


_STAT_NAMES = ["allocated", "peak_allocated", "reserved", "peak_reserved", "alloc_cnt", "free_cnt", "mark_cnt",
               "segment_allocs", "segment_frees", "cache_hits", "cross_stream_takes", "parked", "splits", "merges"]


def pool_stats(device=0):
    vals = (ctypes.c_uint64 * len(_STAT_NAMES))()
    check(lib().ht_pool_stats(ctypes.c_int(device), vals, ctypes.c_int(len(_STAT_NAMES))))
    return dict(zip(_STAT_NAMES, [int(v) for v in vals]))
