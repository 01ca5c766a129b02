"""ctypes bindings of liborion_kernels.so (the hand-written gfx950 kernels).

torch is used only as the owner of device memory and streams; the arithmetic
runs in the HIP kernels behind the C ABI declared in ``include/orion_kernels.h``
(the co-location kernels) and ``include/orion_model_kernels.h`` (the kernels of the
Transformer-XL client: ``transformer_xl.py`` asks here which calls they take).
"""

import atexit
import ctypes
import os
import warnings

import torch
from torch.autograd import forward_ad

from . import _lib

try:
    from . import kernel_calls as _calls       # csrc/calls: the same calls for plain tensors
except ImportError as error:
    _calls = None
    if os.path.exists(_lib.KERNEL_CALLS):      # built, for another PyTorch or Python perhaps
        warnings.warn(f"{_lib.KERNEL_CALLS} does not load, so small kernels are called at up to "
                      f"1.6 times the time: {error}", RuntimeWarning, stacklevel=2)

STATUS = {0: "ok", 1: "bad argument", 2: "shape not a multiple of the tile",
          3: "pointer not 16-byte aligned", 4: "launch rejected"}


class _TxlDims(ctypes.Structure):
    _fields_ = [(name, ctypes.c_int) for name in
                ("layers", "heads", "inner", "q_len", "m_len", "batch")] + [("eps", ctypes.c_float)]


class _Nll(ctypes.Structure):
    _fields_ = [(name, ctypes.c_void_p) for name in
                ("hidden", "weight", "bias", "tail_weight", "tail_bias", "target")] + [
                    ("rows", ctypes.c_int), ("tails", ctypes.c_int), ("edges", ctypes.c_int * 9)]


class KernelError(RuntimeError):
    def __init__(self, name, code):
        super().__init__(f"{name}: {STATUS.get(code, code)}")
        self.code = code


def lib():
    handle = _lib.load(_lib.KERNELS_LIB)
    if not getattr(handle, "_orion_typed", False):
        handle.orion_triad_f32.argtypes = [
            ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_float,
            ctypes.c_size_t, ctypes.c_int, ctypes.c_void_p]
        handle.orion_triad_f32.restype = ctypes.c_int
        handle.orion_gemm_bf16_nt.argtypes = [
            ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int,
            ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
        handle.orion_gemm_bf16_nt.restype = ctypes.c_int
        handle.orion_lamb_workspace_bytes.argtypes = [ctypes.c_void_p, ctypes.c_int]
        handle.orion_lamb_workspace_bytes.restype = ctypes.c_size_t
        handle.orion_lamb_step.argtypes = [
            ctypes.c_void_p, ctypes.c_int, ctypes.c_double, ctypes.c_double, ctypes.c_double,
            ctypes.c_double, ctypes.c_double, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]
        handle.orion_lamb_step.restype = ctypes.c_int
        ptr, size = ctypes.c_void_p, ctypes.c_size_t
        handle.orion_txl_workspace_bytes.argtypes = [ptr]
        handle.orion_txl_workspace_bytes.restype = size
        handle.orion_txl_hidden.argtypes = [ptr, ptr, ptr, ptr, ptr, ptr, size, ptr, size,
                                            ctypes.c_int, ptr, ptr, size, ptr]
        handle.orion_txl_hidden.restype = ctypes.c_int
        handle.orion_nll_workspace_bytes.argtypes = [ptr]
        handle.orion_nll_workspace_bytes.restype = size
        handle.orion_nll_bf16.argtypes = [ptr, ptr, ptr, size, ptr]
        handle.orion_nll_bf16.restype = ctypes.c_int
        handle.orion_stream_create.argtypes = [ctypes.c_int, ctypes.POINTER(ctypes.c_void_p)]
        handle.orion_stream_create.restype = ctypes.c_int
        handle.orion_stream_destroy.argtypes = [ctypes.c_void_p]
        handle.orion_stream_destroy.restype = ctypes.c_int
        handle._orion_typed = True
        if _calls is not None:
            _calls.entries(*(ctypes.cast(entry, ctypes.c_void_p).value for entry in (
                handle.orion_triad_f32, handle.orion_gemm_bf16_nt)))
    return handle


_streams = []          # raw handles of the streams made here, destroyed at exit


def cu_masked_stream(cu_count, device=0):
    """A ``torch.cuda.ExternalStream`` over a stream limited to ``cu_count``
    compute units (the whole GPU for ``cu_count <= 0``)."""
    out = ctypes.c_void_p()
    rc = lib().orion_stream_create(int(cu_count), ctypes.byref(out))
    if rc != 0:
        raise KernelError("orion_stream_create", rc)
    _streams.append(out.value)
    return torch.cuda.ExternalStream(out.value, device=device)


def _profiler_attached():
    """True when a rocprofiler *tool* library is in this process: rocprofv3
    names it in ROCP_TOOL_LIBRARIES and LD_PRELOAD and it shows in the process's
    maps.  (``librocprofiler-register.so`` does not count: the HIP runtime maps
    it in every process, profiled or not.)"""
    named = os.environ.get("ROCP_TOOL_LIBRARIES", "") + ":" + os.environ.get("LD_PRELOAD", "")
    if "rocprofiler-sdk-tool" in named:
        return True
    try:
        with open("/proc/self/maps") as f:
            return any("rocprofiler-sdk-tool" in line for line in f)
    except OSError:
        return False


@atexit.register
def _shutdown():
    """Gives back what this module took from the HIP runtime while the runtime
    is still up: waits for the device and destroys the streams made here.  Under
    a profiler the kernel library is unloaded as well (which un-registers its
    code object): left to process exit, the library's own finaliser then runs
    after the interpreter and the profiler's hooks have shut down, and the
    process dies in it.  Without a profiler the library stays mapped until the
    process ends, so that whoever lists the process's libraries at exit sees it."""
    handle = _lib.loaded(_lib.KERNELS_LIB)
    if handle is None:
        return
    if torch.cuda.is_initialized():
        torch.cuda.synchronize()
    while _streams:
        handle.orion_stream_destroy(ctypes.c_void_p(_streams.pop()))
    if _profiler_attached():
        if _calls is not None:
            _calls.entries(0, 0)
        _lib.unload(_lib.KERNELS_LIB)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_current_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream_ptr(stream):
    """The handle of ``stream``, or of the current device's current stream.  Callers hold
    device tensors, so the runtime is up; a ``torch.cuda.Stream`` made only to be asked
    for its handle costs more than half as much as the launch itself."""
    if stream is not None:
        return stream.cuda_stream
    if _raw_stream is None or _current_device is None:     # private: not in every torch
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_current_device())


def _check_device(*tensors):
    for t in tensors:
        if not t.is_cuda:
            raise ValueError("orion_amd kernels take device tensors only")
        if not t.is_contiguous():
            raise ValueError("orion_amd kernels take contiguous tensors only")


_TENSOR_TYPES = (torch.Tensor, torch.nn.Parameter)


def triad(a, b, c, s, grid_blocks=0, stream=None):
    """a = b + s * c (fp32, one FMA per element), in place into ``a``."""
    done = _calls and _calls.triad(a, b, c, s, grid_blocks, stream)
    if done is not None:
        return done
    _check_device(a, b, c)
    if not (a.dtype == b.dtype == c.dtype == torch.float32):
        raise ValueError("triad is fp32")
    n = a.numel()
    if not n == b.numel() == c.numel():
        raise ValueError("triad operands differ in length")
    rc = lib().orion_triad_f32(a.data_ptr(), b.data_ptr(), c.data_ptr(),
                               ctypes.c_float(s), n, grid_blocks,
                               _stream_ptr(stream))
    if rc != 0:
        raise KernelError("orion_triad_f32", rc)
    return a


def gemm_bf16_nt(a, b, out=None, out_dtype=torch.bfloat16, stream=None):
    """out[M,N] = a[M,K] @ b[N,K].T with bf16 inputs and fp32 accumulation."""
    done = _calls and _calls.gemm(a, b, out, out_dtype, stream)
    if done is not None:
        return done
    _check_device(a, b)
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16:
        raise ValueError("gemm_bf16_nt takes bf16 operands")
    if a.dim() != 2 or b.dim() != 2 or a.shape[1] != b.shape[1]:
        raise ValueError("gemm_bf16_nt wants a[M,K] and b[N,K]")
    m, k = a.shape
    n = b.shape[0]
    if out is None:
        # the same tensor either way (``new_empty`` refuses named dimensions); parsing a
        # device takes as long as the kernel of a small product
        out = (a.new_empty((m, n), dtype=out_dtype)
               if type(a) in _TENSOR_TYPES and not a.has_names()
               else torch.empty((m, n), dtype=out_dtype, device=a.device))
        fits = True
    else:
        _check_device(out)
        fits = out.shape == (m, n)
    if not fits or out.dtype not in (torch.bfloat16, torch.float32):
        raise ValueError("gemm_bf16_nt output must be [M,N] bf16 or fp32")
    rc = lib().orion_gemm_bf16_nt(a.data_ptr(), b.data_ptr(), out.data_ptr(),
                                  m, n, k, int(out.dtype == torch.float32),
                                  _stream_ptr(stream))
    if rc != 0:
        raise KernelError("orion_gemm_bf16_nt", rc)
    return out


def plain_eager():
    """False while something has to see every operation: a transform or a mode
    that rewrites them, a tracer, or forward-mode derivatives, which ``no_grad``
    leaves on and whose dual tensors have no type of their own."""
    return (forward_ad._current_level < 0
            and torch._C._functorch.peek_interpreter_stack() is None
            and torch._C._len_torch_dispatch_stack() == 0
            and torch._C._len_torch_function_stack() == 0
            and not torch.jit.is_tracing()
            and not torch.compiler.is_compiling())


def plain_tensors(tensors, dtype, index):
    """Whether these are ordinary contiguous tensors of GPU ``index`` (-1: of the CPU),
    their values as they lie in memory: what a kernel that takes addresses can work on."""
    types, strided = _TENSOR_TYPES, torch.strided    # looked up once: lists are long
    for t in tensors:
        if (type(t) not in types or t.dtype is not dtype or t.get_device() != index
                or t.layout is not strided or t.is_neg() or not t.is_contiguous()):
            return False
    return True


def lamb_takes(params, grads, ms, vs):
    """Whether ``lamb_step`` takes these lists: contiguous fp32 tensors of one
    GPU, of equal shapes item by item."""
    if not params[0].is_cuda or not plain_eager():
        return False
    index = params[0].get_device()
    if not all(plain_tensors(ts, torch.float32, index) for ts in (params, grads, ms, vs)):
        return False
    return all(p.shape == g.shape == m.shape == v.shape
               for p, g, m, v in zip(params, grads, ms, vs))


def lamb_step(params, grads, ms, vs, lr, betas, eps, weight_decay):
    """One LAMB step in place over lists that ``lamb_takes`` accepts, on the
    current stream of their device."""
    device = params[0].device
    table = []
    for p, g, m, v in zip(params, grads, ms, vs):
        table += (p.data_ptr(), g.data_ptr(), m.data_ptr(), v.data_ptr(), p.numel())
    table = (ctypes.c_uint64 * len(table))(*table)
    handle = lib()
    with torch.cuda.device(device):
        size = handle.orion_lamb_workspace_bytes(table, len(params))
        # in stream order: the allocator hands it on only behind these kernels
        work = torch.empty(size, dtype=torch.uint8, device=device)
        rc = handle.orion_lamb_step(table, len(params), lr, betas[0], betas[1], eps,
                                    weight_decay, work.data_ptr(), size, _stream_ptr(None))
    if rc != 0:
        raise KernelError("orion_lamb_step", rc)
    for ts in (params, ms, vs):          # written behind autograd's back
        torch.autograd.graph.increment_version(ts)


TXL_WIDTH, TXL_HEAD, TXL_TAILS = 512, 64, 7     # what the Transformer-XL kernels are built for


def _bf16_addresses(tensors, shapes, index):
    """Addresses of tensors that are what the bf16 kernels read: plain, contiguous, of
    these shapes, on GPU ``index`` and 16-byte aligned; None if one is not.  (Lazily
    negated tensors are imaginary parts of conjugates: of no 16-bit brain float.)"""
    types, bf16, strided = _TENSOR_TYPES, torch.bfloat16, torch.strided
    out = []
    for t, shape in zip(tensors, shapes):
        if (type(t) not in types or t.dtype is not bf16 or t.shape != shape
                or t.get_device() != index or t.layout is not strided
                or not t.is_contiguous()):
            return None
        at = t.data_ptr()
        if at & 15:
            return None
        out.append(at)
    return out


def _bf16_operand(t, shape, index):
    return _bf16_addresses((t,), (shape,), index) is not None


def inference_only():
    """No gradients to record, no tracing or rewriting, no autocast."""
    return (not torch.is_grad_enabled() and plain_eager()
            and not torch.is_autocast_enabled("cuda"))


def txl_hidden(x, mems, u, v, layers, inner, eps, keep):
    """Hidden states [q, batch, 512] of the embedded tokens ``x`` behind the memory
    ``mems`` [layers, m, batch, 512] (or None), and the last ``keep`` positions of
    the layers' inputs, memory included (None for ``keep`` 0).  ``layers`` holds,
    per layer, the eleven tensors of ``orion_txl_layer``.  None where the kernels
    do not take these tensors."""
    index = x.get_device()
    if index < 0 or not _bf16_operand(x, x.shape, index) or x.dim() != 3 or not x.numel():
        return None
    q_len, batch, width = x.shape
    heads = u.shape[0]
    proj = heads * TXL_HEAD
    if width != TXL_WIDTH or not (_bf16_operand(u, (heads, TXL_HEAD), index)
                                  and _bf16_operand(v, (heads, TXL_HEAD), index)):
        return None
    row = (width,)
    shapes = ((3 * proj, width), (proj, width), (width, proj), row, row,
              (inner, width), (inner,), (width, inner), row, row, row)
    table = []
    for tensors in layers:
        addresses = _bf16_addresses(tensors, shapes, index)
        if addresses is None:
            return None
        table += addresses
    m_len = 0
    if mems is not None:
        if (type(mems) is not torch.Tensor or mems.dtype is not torch.bfloat16
                or mems.dim() != 4 or mems.get_device() != index
                or mems.shape[0] != len(layers) or mems.shape[2:] != (batch, width)):
            return None
        m_len = mems.shape[1]
        if m_len and (mems.stride()[1:] != (batch * width, width, 1) or mems.stride(0) % 8
                      or mems.data_ptr() & 15):
            return None
    dims = _TxlDims(len(layers), heads, inner, q_len, m_len, batch, eps)
    handle = lib()
    size = handle.orion_txl_workspace_bytes(ctypes.byref(dims))
    if not size:
        return None
    table = (ctypes.c_void_p * len(table))(*table)
    with torch.cuda.device(index):
        hidden = torch.empty_like(x)
        work = torch.empty(size, dtype=torch.uint8, device=x.device)
        new, new_at, new_stride, from_x = None, None, 0, 0
        if keep:
            keep = min(keep, m_len + q_len)
            from_x = min(keep, q_len)
            new = torch.empty((len(layers), keep, batch, width), dtype=x.dtype, device=x.device)
            if keep > q_len:
                new[:, :keep - q_len].copy_(mems[:, m_len - (keep - q_len):])
            new_at, new_stride = new[0, keep - from_x].data_ptr(), new.stride(0)
        rc = handle.orion_txl_hidden(
            ctypes.byref(dims), table, u.data_ptr(), v.data_ptr(), x.data_ptr(),
            mems.data_ptr() if m_len else None, mems.stride(0) if m_len else 0,
            new_at, new_stride, from_x, hidden.data_ptr(), work.data_ptr(), size,
            _stream_ptr(None))
    if rc != 0:
        raise KernelError("orion_txl_hidden", rc)
    return hidden, new


def adaptive_nll(hidden, target, weight, bias, tail_weight, tail_bias, edges):
    """Losses [n] of ``target`` [n] under an adaptive softmax over ``hidden``
    [n, 512]; None where the kernels do not take these tensors."""
    index = hidden.get_device()
    tails = len(edges) - 2
    if index < 0 or hidden.dim() != 2 or not 0 <= tails <= TXL_TAILS or not edges[-1] < 1 << 31:
        return None
    n, width = hidden.shape
    if width != TXL_WIDTH or not n or any(lo >= hi for lo, hi in zip(edges, edges[1:])):
        return None
    for t, shape in ((hidden, (n, width)), (weight, (edges[-1], width)), (bias, (edges[-1],)),
                     (tail_weight, (tails, width)), (tail_bias, (tails,))):
        if not _bf16_operand(t, shape, index):
            return None
    if (type(target) is not torch.Tensor or target.dtype is not torch.int64
            or target.shape != (n,) or target.get_device() != index
            or not target.is_contiguous()):
        return None
    args = _Nll(hidden.data_ptr(), weight.data_ptr(), bias.data_ptr(), tail_weight.data_ptr(),
                tail_bias.data_ptr(), target.data_ptr(), n, tails,
                (ctypes.c_int * 9)(*edges))
    handle = lib()
    size = handle.orion_nll_workspace_bytes(ctypes.byref(args))
    if not size:
        return None
    with torch.cuda.device(index):
        nll = torch.empty(n, dtype=hidden.dtype, device=hidden.device)
        work = torch.empty(size, dtype=torch.uint8, device=hidden.device)
        rc = handle.orion_nll_bf16(ctypes.byref(args), nll.data_ptr(), work.data_ptr(), size,
                                   _stream_ptr(None))
    if rc != 0:
        raise KernelError("orion_nll_bf16", rc)
    return nll
