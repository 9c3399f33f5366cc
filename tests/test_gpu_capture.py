"""What a layer call allocates, and what it records into a graph.  A call whose shape needs no
workspace must stay one kernel; a workspace would be one array shared by
unordered streams (the no-allocation entry point) or an allocation inside the
graph (the others).  The recorded nodes are counted before any replay; then
every replay, with eager work between, must equal the eager call."""
import ctypes as C

import numpy as np
import pytest
import torch

from neuroflow_amd import _lib
from neuroflow_amd import quant as Q
from neuroflow_amd import workloads as WL
from oracle import oracle as O
from tests.test_gpu_one_pass import _cu, _int8

pytestmark = pytest.mark.gpu

KERNEL = 0   # hipGraphNodeTypeKernel


def _hip():
    return C.CDLL("libamdhip64.so.7")   # the runtime the library is linked to, already loaded


def _node_types(graph):
    hip, h = _hip(), C.c_void_p(graph.raw_cuda_graph())
    n = C.c_size_t(0)
    assert hip.hipGraphGetNodes(h, None, C.byref(n)) == 0
    nodes = (C.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(h, nodes, C.byref(n)) == 0
    out = []
    for node in nodes:
        t = C.c_int(-1)
        assert hip.hipGraphNodeGetType(C.c_void_p(node), C.byref(t)) == 0
        out.append(t.value)
    return out


def _captured(call, out):
    """The graph of call() writing out."""
    g = torch.cuda.CUDAGraph(keep_graph=True)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        call(out)
    return g


def _replays_equal(g, out, want, between):
    for r in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int32), want.view(torch.int32)), f"replay {r}"
        between()
        torch.cuda.synchronize()


def _stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("M,K,N", [(8192, 512, 1024), (20000, 512, 576), (6000, 512, 768), (65536, 512, 576), (9000, 256, 512)])
def test_noalloc_shapes_without_scratch_are_one_kernel(gpu, M, K, N):
    """K = 128, 256, 512 with N a multiple of 64 never touch the no-allocation
    entry point's one array, at any row count: calls on them are independent
    on any streams."""
    q, s, _, _, b = _int8(N, K, 600)
    p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), None, _cu(b, 0))
    ps = p.c_struct()
    fn = _lib.lib().nflow_int8_linear_forward_per_token_noalloc
    x = torch.from_numpy(WL.normal(603, (M, K))).cuda()

    def call(out):
        _lib.check(fn(C.byref(ps), M, x.data_ptr(), out.data_ptr(), None, 1, _stream()), "noalloc")

    want = Q.linear_forward_per_token(p, x, "relu")
    out = torch.empty_like(want)
    g = _captured(call, out)
    assert _node_types(g) == [KERNEL]
    other = torch.empty_like(want)
    _replays_equal(g, out, want, lambda: call(other))


# Shapes that run as quantise + GEMM outside a capture.
@pytest.mark.parametrize("kind,M,K,N", [("int8", 8192, 512, 1024), ("int8", 4096, 1024, 1024), ("int8", 3000, 960, 300),
                                        ("fp8", 4096, 1024, 1024), ("fp8", 20000, 512, 2048), ("rows", 8192, 512, 2048),
                                        ("rows", 4096, 1024, 256), ("batched", 2000, 640, 512)])
def test_layers_up_to_1024_allocate_nothing_in_a_graph(gpu, kind, M, K, N):
    """Layers of K <= 1024 record one kernel: no workspace inside the graph.
    The replays equal the eager one-pass kernel (no_gemm keeps it off the
    GEMM), and INT8 the eager call as it runs by itself."""
    L = _lib.lib()
    if kind == "fp8":
        qw, sw = O.quantise_weight_fp8(WL.uniform(610, (N, K), -0.125, 0.125))
        p = Q.Fp8LinearParams(_cu(qw, 0), _cu(sw, 0))
    else:
        q, s, zps, sw, b = _int8(N, K, 611)
        fixed = kind != "int8"
        p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), _cu(zps, 0) if fixed else None, _cu(b, 0), 0.02, 3,
                               _cu(sw, 0) if fixed else None)
    fn, args = {"int8": (L.nflow_int8_linear_forward_per_token, (None, 1)),
                "fp8": (L.nflow_fp8_linear_forward_per_token, (None, 1)),
                "rows": (L.nflow_int8_linear_forward_rows, ()),
                "batched": (L.nflow_int8_linear_forward_batched, ())}[kind]
    ps = p.c_struct()
    x = torch.from_numpy(WL.normal(614, (M, K)).astype(np.float32)).cuda()

    def call(out):
        _lib.check(fn(C.byref(ps), M, x.data_ptr(), out.data_ptr(), *args, _stream()), kind)

    eager, want, out = (torch.empty(M, N, device="cuda") for _ in range(3))
    call(eager)
    prev = C.c_int(0)
    _lib.check(L.nflow_debug_set_kernel_path(b"no_gemm", 1, C.byref(prev)), "path")
    try:
        call(want)
    finally:
        _lib.check(L.nflow_debug_set_kernel_path(b"no_gemm", prev.value, None), "path")
    if kind != "fp8":
        assert torch.equal(eager.view(torch.int32), want.view(torch.int32))
    g = _captured(call, out)
    assert _node_types(g) == [KERNEL]
    _replays_equal(g, out, want, lambda: call(eager))


def _pool_used_high(reset=False):
    """High-water mark of the device's default pool of stream-ordered allocations."""
    hip, pool, v = _hip(), C.c_void_p(), C.c_uint64(0)
    assert hip.hipDeviceGetDefaultMemPool(C.byref(pool), torch.cuda.current_device()) == 0
    USED_CURRENT, USED_HIGH = 7, 8   # hipMemPoolAttrUsedMemCurrent, hipMemPoolAttrUsedMemHigh
    if reset:
        assert hip.hipMemPoolSetAttribute(pool, USED_HIGH, C.byref(v)) == 0
        assert hip.hipMemPoolGetAttribute(pool, USED_CURRENT, C.byref(v)) == 0
    else:
        assert hip.hipMemPoolGetAttribute(pool, USED_HIGH, C.byref(v)) == 0
    return v.value


@pytest.mark.parametrize("M,K,N,allocates", [(8192, 512, 1024, False), (9000, 256, 512, False), (4096, 1024, 256, True)])
def test_per_thread_stream_keeps_workspace_free_shapes(gpu, M, K, N, allocates):
    """The per-thread default stream keeps no workspace (a call that takes one
    allocates and frees it): shapes that need none take none there.  The
    K = 1024 row shows that the mark moves when a call does allocate."""
    PER_THREAD = 2   # hipStreamPerThread
    q, s, _, _, b = _int8(N, K, 620)
    p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), None, _cu(b, 0))
    ps = p.c_struct()
    x = torch.from_numpy(WL.normal(623, (M, K))).cuda()
    want, out = Q.linear_forward_per_token(p, x, "relu"), torch.empty(M, N, device="cuda")
    torch.cuda.synchronize()
    before = _pool_used_high(reset=True)
    _lib.check(_lib.lib().nflow_int8_linear_forward_per_token(C.byref(ps), M, x.data_ptr(), out.data_ptr(), None, 1,
                                                              PER_THREAD), "per token")
    torch.cuda.synchronize()
    assert (_pool_used_high() > before) == allocates
    assert torch.equal(out.view(torch.int32), want.view(torch.int32))
