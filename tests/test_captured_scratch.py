"""Kernels whose plan wants scratch but does not need it (16-bit Matmul split
over K, attention of a few rows, attention in runs of key steps), recorded in a
HIP graph: with any allocator that gives scratch, warm or cold, the graph holds
the kernels of the plan, and its replays equal the eager call; and the errors
of an allocator."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    from gpu_util import gpu_env

    return gpu_env()


def _hip(name, *args):
    from popcorn_amd import runtime as R

    f = getattr(R.lib(), name)  # a symbol of the HIP runtime that the library links
    f.restype = C.c_int
    assert f(*args) == 0, name


def _record(stream, work, mode):
    """The executable graph of work() recorded on the stream, and its kernel count."""
    s, g, e, n = C.c_void_p(stream.handle), C.c_void_p(), C.c_void_p(), C.c_size_t(0)
    _hip("hipStreamBeginCapture", s, C.c_int(mode))
    try:
        work()
    finally:
        _hip("hipStreamEndCapture", s, C.byref(g))
    _hip("hipGraphGetNodes", g, None, C.byref(n))
    _hip("hipGraphInstantiate", C.byref(e), g, None, None, C.c_size_t(0))
    _hip("hipGraphDestroy", g)
    return e, n.value


def _matmul(pa, M, K, N, t):
    import oracle as O
    from gpu_util import rounded, upload

    a, b = (upload(pa, rounded(O.normal(i, s, std=0.1), t), t) for i, s in ((1, (M, K)), (2, (N, K))))
    c = pa.Tensor.empty([M, N], t)
    return pa.Kernels.Matmul(a, b, c, True), c


def _attention(pa, Nq, Nkv, Sq, Sk, Hd, t):
    import oracle as O
    from gpu_util import rounded, upload

    q, k, v = (upload(pa, rounded(O.normal(i, s), t), t) for i, s in ((1, (1, Nq, Sq, Hd)), (2, (1, Nkv, Sk, Hd)), (3, (1, Nkv, Sk, Hd))))
    out = pa.Tensor.empty([1, Nq, Sq, Hd], t)
    return pa.Kernels.FlashAttention(q, k, v, out=out, scale=Hd ** -0.5, batch=1, query_heads=Nq, kv_heads=Nkv, query_len=Sq,
                                     key_len=Sk, head_dim=Hd, key_capacity=Sk), out


CALLS = {"small_grid": lambda pa: _matmul(pa, 137, 9216, 2304, "bf16"),
         "long_k": lambda pa: _matmul(pa, 2048, 24576, 3072, "f16"),
         "few_rows": lambda pa: _attention(pa, 8, 4, 8, 4104, 256, "bf16"),
         "runs": lambda pa: _attention(pa, 8, 4, 300, 3000, 256, "bf16"),
         "runs_or_pairs": lambda pa: _attention(pa, 8, 8, 1000, 1000, 256, "bf16")}


def _allocator(pa, kind):
    if kind == "pool":
        return pa.ScratchPool()
    if kind != "python":
        return None  # the encoder's own pool

    class Python(pa.KernelScratchAllocator):
        free, held = [], {}

        def borrow(self, length):
            for p in self.free:
                if self.held[p].nbytes >= length:
                    self.free.remove(p)
                    return p, True
            t = pa.Tensor.empty([length], "u8")  # allocates, also inside the capture
            self.held[t.ptr] = t
            return t.ptr, False

        def release(self, ptr):
            self.free.append(ptr)

    return Python()


@pytest.mark.parametrize("call", CALLS)
@pytest.mark.parametrize("kind", ["own", "pool", "python"])
@pytest.mark.parametrize("warm", [False, True])
@pytest.mark.parametrize("mode", [0, 1])  # global, thread-local
def test_graph_holds_the_plan(env, call, kind, warm, mode):
    pa, lib, _, _ = env
    stream = pa.Stream()
    eager = pa.KernelCommandEncoder(lib, stream)
    kern, out = CALLS[call](pa)
    eager.encode(kern)
    stream.synchronize()
    want = out.numpy(stream)
    alloc = _allocator(pa, kind)
    enc = pa.KernelCommandEncoder(lib, stream, scratch=alloc)
    if warm:
        enc.encode(kern)
        stream.synchronize()
    graph, kernels = _record(stream, lambda: enc.encode(kern), mode)
    assert kernels == len(kern.function_names) == 2
    for _ in range(3):
        out.copy_from(np.zeros(want.shape, want.dtype), stream)
        eager.encode(kern)  # the program's own work between replays
        stream.synchronize()
        out.copy_from(np.zeros(want.shape, want.dtype), stream)
        _hip("hipGraphLaunch", graph, C.c_void_p(stream.handle))
        stream.synchronize()
        np.testing.assert_array_equal(out.numpy(stream), want)
    _hip("hipGraphExecDestroy", graph)


@pytest.mark.parametrize("call,eager", [("small_grid", False), ("few_rows", False), ("runs", False), ("runs_or_pairs", False),
                                        ("runs_or_pairs", True)])
def test_graph_without_scratch(env, call, eager):
    # nothing to borrow while recording: one kernel that needs none, and right.
    # Attention whose plan without runs is pairs records whole tiles where the
    # stream has no exchange for them yet, pairs where an eager call made it.
    pa, lib, _, _ = env
    stream = pa.Stream()

    class Empty(pa.KernelScratchAllocator):
        def borrow(self, length):
            raise MemoryError

    kern, out = CALLS[call](pa)
    pa.KernelCommandEncoder(lib, stream).encode(kern)
    stream.synchronize()
    want = out.numpy(stream).view(np.uint16)
    enc = pa.KernelCommandEncoder(lib, stream, scratch=Empty())
    if eager:
        enc.encode(kern)
        stream.synchronize()
    graph, kernels = _record(stream, lambda: enc.encode(kern), 1)
    assert kernels == 1
    import oracle as O

    ref = O.from_bits(want, O.BF16)
    for _ in range(3):
        out.copy_from(np.zeros(want.shape, want.dtype), stream)
        _hip("hipGraphLaunch", graph, C.c_void_p(stream.handle))
        stream.synchronize()
        got = O.from_bits(out.numpy(stream).view(np.uint16), O.BF16)
        # the same sums in another order: a bf16 unit in the last place apart at most, or under the smallest normal result
        np.testing.assert_allclose(got, ref, rtol=2.0 ** -7, atol=1e-4)
    _hip("hipGraphExecDestroy", graph)


def test_allocator_errors(env):
    # no memory: the kernels that can do without it run; any other error of the
    # allocator reaches the caller, with what it raised
    import torch

    pa, lib, stream, _ = env

    class Failing(pa.KernelScratchAllocator):
        def borrow(self, length):
            raise self.exc

    alloc = Failing()
    enc = pa.KernelCommandEncoder(lib, stream, scratch=alloc)
    token, _ = _attention(pa, 8, 4, 1, 1000, 256, "bf16")  # needs its partials
    for call in ("small_grid", "few_rows", "runs"):
        kern, _ = CALLS[call](pa)
        for exc in (MemoryError(), torch.OutOfMemoryError(), pa.PopcornError(pa.PopcornError.GPU_OUT_OF_MEMORY, "none")):
            alloc.exc = exc
            before = enc.stats()["dispatches"]
            enc.encode(kern)
            assert enc.stats()["dispatches"] == before + 1
            with pytest.raises(pa.PopcornError) as e:
                enc.encode(token)
            assert e.value.__cause__ is exc and e.value.code == getattr(exc, "code", pa.PopcornError.TENSOR_ALLOCATION_FAILED)
        alloc.exc = RuntimeError("lost track of a buffer")
        with pytest.raises(pa.PopcornError) as e:
            enc.encode(kern)
        assert e.value.__cause__ is alloc.exc and e.value.code == pa.PopcornError.GPU_INTERNAL
    stream.synchronize()
