"""What a layer call records into a graph.  A call whose shape needs no
workspace must stay one kernel; a workspace would be one array shared by
unordered streams (the no-allocation entry point) or an allocation inside the
graph (the others).  The recorded nodes are counted before any replay; then
every replay, with eager work between, must equal the eager call."""
import ctypes as C

import pytest
import torch

from neuroflow_amd import _lib
from neuroflow_amd import quant as Q
from neuroflow_amd import workloads as WL
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
