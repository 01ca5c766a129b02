"""Calls that go to the kernels without Python in between against the same calls made in
Python: which ones are taken, what they give, and how the others are refused."""

import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from orion_amd import _lib, kernels

DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "orion_amd", "csrc")


class Sub(torch.Tensor):
    pass


class SeesFunctions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class SeesOperations(TorchDispatchMode):
    seen = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        SeesOperations.seen += 1
        return func(*args, **(kwargs or {}))


def test_module_is_built_and_leaves_host_tensors_to_python():
    calls = kernels._calls
    assert calls is not None
    x = torch.ones(4)
    bf = torch.ones(256, 64, dtype=torch.bfloat16)
    assert calls.triad(x, x, x, 1.0, 0, None) is None
    assert calls.gemm(bf, bf, None, torch.bfloat16, None) is None
    for bad in ((x,), (None,) * 6, (1, 2, 3, 4, 5, 6)):
        assert calls.triad(*bad) is None and calls.gemm(*bad) is None
    with pytest.raises(TypeError):
        calls.entries(1)
    with pytest.raises(ValueError, match="device tensors"):
        kernels.triad(x, x, x, 1.0)
    with pytest.raises(ValueError, match="device tensors"):
        kernels.gemm_bf16_nt(bf, bf)


# Entry points that answer with a code, and tensors "on the GPU" over addresses that nothing
# reads: in a process of its own, since torch then takes the GPU runtime for initialised.
STUBS = """
import ctypes, json, sys, types
import torch
torch.cuda._lazy_init = lambda: None
from orion_amd import kernels
P, I, F, Z = ctypes.c_void_p, ctypes.c_int, ctypes.c_float, ctypes.c_size_t

class DLTensor(ctypes.Structure):
    _fields_ = [("data", P), ("device_type", I), ("device_id", I), ("ndim", I),
                ("type", ctypes.c_uint8 * 4), ("shape", P), ("strides", P),
                ("offset", ctypes.c_uint64), ("context", P), ("deleter", P)]

capsule = ctypes.pythonapi.PyCapsule_New
capsule.restype, capsule.argtypes = ctypes.py_object, [P, ctypes.c_char_p, P]
held = []

def tensor(shape, code, bits):
    sizes = (ctypes.c_int64 * len(shape))(*shape)
    managed = DLTensor(1 << 40, 10, 0, len(shape), (code, bits, 1, 0), ctypes.addressof(sizes))
    held.extend((sizes, managed))
    return torch.utils.dlpack.from_dlpack(capsule(ctypes.addressof(managed), b"dltensor", None))

made, answer = [], 0
def native(*args):
    made.append("native")
    return answer
def in_python(*args):
    made.append("python")
    return answer
stubs = (ctypes.CFUNCTYPE(I, P, P, P, F, Z, I, P)(native),
         ctypes.CFUNCTYPE(I, P, P, P, I, I, I, I, P)(native))
kernels.lib = lambda: types.SimpleNamespace(orion_triad_f32=in_python,
                                            orion_gemm_bf16_nt=in_python)
kernels._calls.entries(*(ctypes.cast(s, P).value for s in stubs))
stream = types.SimpleNamespace(cuda_stream=0)
x, m, out = tensor((1003,), 2, 32), tensor((256, 64), 4, 16), tensor((256, 256), 2, 32)
seen = []
for answer in range(6):
    for call, result in ((lambda: kernels.triad(x, x, x, 2.0, stream=stream), x),
                         (lambda: kernels.gemm_bf16_nt(m, m, out=out, stream=stream), out)):
        del made[:]
        try:
            got = call() is result
        except kernels.KernelError as e:
            got = (e.code, str(e))
        seen.append((answer, got, list(made)))
kernels._calls.entries(0, 0)
print(json.dumps(seen))
"""


def test_the_runtimes_error_is_raised_and_the_kernel_not_launched_again():
    out = subprocess.run([sys.executable, "-c", STUBS], cwd=ROOT, check=True, timeout=120,
                         capture_output=True, text=True).stdout
    for answer, got, made in json.loads(out):
        if answer == 0:
            assert got is True and made == ["native"]
            continue
        code, text = got
        assert code == answer and text.startswith("orion_")
        # 1 to 3 come before the launch and are said again by the Python code
        assert made == (["native"] if answer >= 4 else ["native", "python"])


def test_the_calls_follow_the_headers_of_the_entry_points(tmp_path):
    plan = subprocess.run(["make", "-C", CSRC, "-n", "-B", _lib.KERNEL_CALLS], check=True,
                          capture_output=True, text=True).stdout
    (command,) = [line.split() for line in plan.split("\n") if "kernel_calls.cpp" in line]
    with open(os.path.join(ROOT, "include", "orion_kernels.h")) as f:
        header = f.read()
    for was, becomes, compiles in (("", "", True),
                                   ("size_t n, int grid_blocks", "size_t n, int* grid_blocks", False),
                                   ("int K, int out_is_f32", "int K, int* out_is_f32", False)):
        changed = header.replace(was, becomes) if was else header
        assert compiles or changed != header
        # first among the folders of headers
        (tmp_path / "orion_kernels.h").write_text(changed)
        done = subprocess.run([command[0], "-fsyntax-only", f"-I{tmp_path}", *command[1:]],
                              cwd=CSRC, capture_output=True, text=True, timeout=300)
        assert (done.returncode == 0) == compiles, done.stderr[-2000:]


def test_without_python_or_torch_headers_the_rest_is_built():
    def plan(*settings):
        return subprocess.run(["make", "-C", CSRC, "-n", "-B", *settings, "all"], check=True,
                              capture_output=True, text=True)
    assert "kernel_calls.cpp" in plan().stdout
    for settings in (("PYTHON=false",), ("PYTHON=echo",), ("PYINC=/nowhere",), ("TORCH=/nowhere",)):
        made = plan(*settings)
        assert "kernel_calls.cpp" not in made.stdout and "kernel_calls.so is left out" in made.stdout
        assert all(lib in made.stdout for lib in ("liborion_kernels.so", "scheduler_eval.so"))
        assert "Traceback" not in made.stderr


BROKEN = """
import sys, warnings
from orion_amd import _lib
_lib.KERNEL_CALLS = sys.argv[1]
sys.modules["orion_amd.kernel_calls"] = None       # importing it is an ImportError
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    from orion_amd import kernels
assert kernels._calls is None
print(sum("does not load" in str(w.message) for w in seen))
"""


@pytest.mark.parametrize("path,warned", [(_lib.KERNEL_CALLS, 1), ("/nowhere/kernel_calls.so", 0)])
def test_a_module_that_does_not_load_is_named(path, warned):
    out = subprocess.run([sys.executable, "-c", BROKEN, path], cwd=ROOT, check=True, timeout=120,
                         capture_output=True, text=True).stdout
    assert int(out) == warned


def _outcome(call):
    try:
        got = call()
    except Exception as e:                 # noqa: BLE001
        return type(e), str(e).split("\n")[0]
    return type(got), got.dtype, tuple(got.shape), got.detach().double().cpu().numpy().tobytes()


@pytest.mark.gpu
def test_the_same_as_in_python_whatever_the_arguments(monkeypatch):
    kernels.lib()
    n = 1003
    b, c = torch.randn(n, device=DEV), torch.randn(n, device=DEV)
    m1, m2 = (torch.randn(256, 128, device=DEV).bfloat16() for _ in range(2))
    stream = kernels.cu_masked_stream(32)
    torch.cuda.synchronize()

    def new(like=b):
        return torch.empty_like(like)

    def triad(*args, **kw):
        return lambda: kernels.triad(*args, **kw)

    def gemm(*args, **kw):
        return lambda: kernels.gemm_bf16_nt(*args, **kw)

    taken = [
        triad(new(), b, c, 1.7), triad(new(), b, c, 2), triad(new(), b, c, 1e40),
        triad(new(), b, c, float("nan")), triad(new(), b, c, 1.7, 70), triad(new(), b, b, -0.5),
        triad(b.clone().view(17, 59), b, c, 1.7), triad(new()[:0], b[:0], c[:0], 1.0),
        triad(torch.nn.Parameter(new()), b, c, 1.7),
        triad(new(), b, c, 1.7, stream=stream),
        triad(new(), b, c, 1.7, stream=torch.cuda.current_stream()),
        gemm(m1, m2), gemm(m1, m2, out_dtype=torch.float32), gemm(torch.nn.Parameter(m1), m2),
        gemm(m1, m2, torch.empty(256, 256, device=DEV)), gemm(m1, m2, stream=stream),
        gemm(m1, m2, out=torch.empty(256, 256, device=DEV, dtype=torch.bfloat16))]
    left = [
        triad(new()[1:], b[1:], c[1:], 1.7),       # not aligned to 16 bytes: refused
        triad(new(), b, c, np.float32(1.7)), triad(new(), b, c, True), triad(new(), b, c, "1"),
        triad(new(), b, c, None), triad(new(), b, c, 1.7, 1 << 40), triad(new(), b, c, 1.7, -3),
        triad(new(), b[:-1], c, 1.7), triad(new(), b.double(), c, 1.7), triad(new(), b, 3, 1.7),
        triad(new(), b.cpu(), c, 1.7), triad(new()[::2], b[::2], c[::2], 1.7),
        triad(new().as_subclass(Sub), b, c, 1.7), triad(new(), b, c, 1.7, stream=7),
        triad(new().rename("x"), b, c, 1.7), triad(new(), b.to_sparse(), c, 1.7),
        gemm(m1, m2[:, :64]), gemm(m1.t(), m2), gemm(m1.float(), m2), gemm(m1[0], m2),
        gemm(m1[:100], m2), gemm(m1[:0], m2), gemm(m1, m2, out_dtype=torch.float16),
        gemm(m1, m2, out_dtype="f32"), gemm(m1, m2, out=torch.empty(256, 255, device=DEV)),
        gemm(m1, m2, out=torch.empty(256, 256, device=DEV, dtype=torch.float16)),
        gemm(m1, m2, out=torch.empty(256, 256, device=DEV).t()),
        gemm(m1, m2, out=torch.empty(1, 256, 256, device=DEV)), gemm(m1.as_subclass(Sub), m2),
        gemm(m1.rename("r", "k"), m2)]
    native = []
    real = kernels._calls

    class Counted:
        entries = staticmethod(real.entries)

        @staticmethod
        def triad(*args):
            native.append(real.triad(*args))
            return native[-1]

        @staticmethod
        def gemm(*args):
            native.append(real.gemm(*args))
            return native[-1]

    for i, call in enumerate(taken + left):
        monkeypatch.setattr(kernels, "_calls", Counted)
        del native[:]
        got = _outcome(call)
        # the second list: refusals, and what only the Python code converts or allocates
        if i < len(taken):
            assert native[0] is not None, i
        torch.cuda.synchronize()
        monkeypatch.setattr(kernels, "_calls", None)
        want = _outcome(call)
        torch.cuda.synchronize()
        assert got == want, (i, got[:3], want[:3])


@pytest.mark.gpu
def test_what_sees_operations_keeps_the_python_calls():
    kernels.lib()
    b = torch.randn(100, device=DEV)
    m = torch.randn(256, 64, device=DEV).bfloat16()
    calls = kernels._calls
    assert calls.triad(b.clone(), b, b, 1.0, 0, None) is not None
    with SeesFunctions():
        assert calls.triad(b.clone(), b, b, 1.0, 0, None) is None
    with SeesOperations():
        assert calls.gemm(m, m, None, torch.bfloat16, None) is None
        before = SeesOperations.seen
        kernels.gemm_bf16_nt(m, m)
        assert SeesOperations.seen > before
    taken = []
    torch.vmap(lambda x: taken.append(calls.gemm(m, m, None, torch.bfloat16, None)) or x)(b)
    torch.jit.trace(lambda x: taken.append(calls.gemm(m, m, None, torch.bfloat16, None)) or x + 1, b,
                    check_trace=False)
    assert taken == [None, None]


@pytest.mark.gpu
def test_current_stream_and_captures():
    b, c = torch.randn(5000, device=DEV), torch.randn(5000, device=DEV)
    m = torch.randn(256, 128, device=DEV).bfloat16()
    kernels.lib()
    want = torch.empty_like(b)
    kernels.triad(want, b, c, 1.5)
    product = kernels.gemm_bf16_nt(m, m)
    torch.cuda.synchronize()
    a = torch.zeros_like(b)
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        kernels.triad(a, b, c, 1.5)
        out = kernels.gemm_bf16_nt(m, m)
    for _ in range(3):
        a.zero_()
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(a, want) and torch.equal(out, product)
