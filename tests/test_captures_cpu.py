"""What the GPU tests of stream capture leave behind, seen on the CPU.

A torch CUDAGraph waits for the device when it is destroyed, and a device that is waited for while a stream is being
captured is an error: out of a destructor, the end of the process.  torch collects no garbage before a capture, so a graph
that an earlier test left in a reference cycle may be destroyed at any moment of a later test's capture."""
import contextlib
import gc
import types
import weakref

import numpy as np
import pytest

import oracle
import test_gpu_graph
import test_gpu_reentrant
import test_zz_no_alloc


class Graph:
    """stands in for torch.cuda.CUDAGraph"""
    made = []

    def __init__(self):
        Graph.made.append(weakref.ref(self))

    def replay(self):
        pass


@contextlib.contextmanager
def stand_in_for_the_device(monkeypatch, pkg, m, n, k):
    """the torch calls and the entry points of the padded-plan test, on host memory"""
    import torch
    on_cpu = lambda make: lambda *a, **kw: make(*a, **{**kw, "device": "cpu"})
    monkeypatch.setattr(torch.Tensor, "cuda", lambda t: t)
    for name in ("empty", "zeros"):
        monkeypatch.setattr(torch, name, on_cpu(getattr(torch, name)))
    # nothing is written over between the replays, which do nothing
    monkeypatch.setattr(torch.Tensor, "fill_", lambda t, value: t)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", Graph)
    monkeypatch.setattr(torch.cuda, "graph", lambda graph: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=0))

    def gemm_ex(a, b, sa, sb, c, m, n, k, options, workspace, nbytes, stream):
        if nbytes <= 1024:
            raise pkg.Fp8GemmError(-4, "fp8_block_gemm_ex")
        ref = oracle.ref_gemm(a.numpy(), b.numpy(), sa.numpy(), sb.numpy(), m, n, k)
        c.copy_(torch.from_numpy(np.asarray(ref).reshape(m, n).view(np.int16)))

    yield types.SimpleNamespace(gemm_ex=gemm_ex, workspace_bytes_ex=lambda *a: 4096, last_kernel=lambda: "padded_stand_in",
                                Fp8GemmError=pkg.Fp8GemmError)


def test_padded_plan_test_leaves_no_graph_behind(pkg, monkeypatch):
    m, n, k = 24, 40, 128
    Graph.made.clear()
    gc.collect()
    gc.disable()
    try:
        with stand_in_for_the_device(monkeypatch, pkg, m, n, k) as fake:
            test_gpu_reentrant.test_padded_plan_with_callers_workspace_eager_and_in_a_graph(fake, m, n, k, 3)
        assert len(Graph.made) == 1 and Graph.made[0]() is None
    finally:
        gc.enable()


@pytest.mark.parametrize("module", [test_gpu_graph, test_gpu_reentrant, test_zz_no_alloc], ids=lambda m: m.__name__)
def test_modules_that_capture_collect_garbage_before_each_test(module):
    marks = module.pytestmark if isinstance(module.pytestmark, list) else [module.pytestmark]
    assert any(mark.name == "usefixtures" and "garbage_collected" in mark.args for mark in marks)


left_behind = []


def test_garbage_collected_leaves_none(request):
    class Node:
        pass
    gc.disable()
    try:
        node = Node()
        node.itself = node
        left_behind.append(weakref.ref(node))
        del node
        assert left_behind[-1]() is not None
        request.getfixturevalue("garbage_collected")
        assert left_behind[-1]() is None
    finally:
        gc.enable()
