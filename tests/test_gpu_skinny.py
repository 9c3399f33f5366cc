"""The few-row kernel (K split over a block's waves) where it can go wrong,
against the oracle: each wave count and K-blocks-per-wave form at its edges,
K off 4, 16 and 64 (with the row form's dropped tail), N off 16, row counts
around its 16-row blocks, 4-byte-aligned buffers; and the fixed-scale split
(quantise with row sums, then the tiled GEMM with zero points on both
sides).  INT8 bit for bit; FP8 to its fp32 accumulation bound."""
import ctypes

import numpy as np
import pytest

from neuroflow_amd import _lib
from neuroflow_amd import quant as Q
from neuroflow_amd import workloads as WL
from oracle import oracle as O
from tests.test_gpu_one_pass import _cu, _guarded, _guards_kept, _int8

pytestmark = pytest.mark.gpu

SHAPES = [(1, 4, 4), (1, 64, 64), (2, 65, 17), (16, 255, 33), (17, 256, 16), (1, 257, 40), (15, 1000, 100), (33, 1023, 31),
          (1, 1024, 1024), (3, 1025, 20), (16, 2047, 48), (1, 2048, 512), (2, 2049, 19), (5, 4095, 35), (1, 4096, 64)]


@pytest.fixture
def skinny():
    prev = ctypes.c_int(0)
    L = _lib.lib()
    _lib.check(L.nflow_debug_set_kernel_path(b"skinny", 1, ctypes.byref(prev)), "path")
    yield
    _lib.check(L.nflow_debug_set_kernel_path(b"skinny", prev.value, None), "path")


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("zp", [False, True])
def test_skinny_int8(gpu, skinny, M, K, N, zp):
    off = (M + K + N) % 3
    q, s, zps, sw, b = _int8(N, K, 840)
    A = WL.normal(843, (M, K))
    p = Q.Int8LinearParams(_cu(q, off), _cu(s, 0), _cu(zps, 0) if zp else None, _cu(b, 0), 0.02, 5,
                           sum_W_per_row=_cu(sw, 0) if zp else None)
    buf, out = _guarded(M, N, off)
    y, sc = Q.linear_forward_per_token(p, _cu(A, off), "relu", out=out, return_scales=True)
    want, s_want = O.layer_per_token_i8(A, q, s, zps if zp else None, b, sw if zp else None, 1)
    assert np.array_equal(sc.cpu().numpy().view(np.uint32), s_want.view(np.uint32))
    assert np.array_equal(y.cpu().numpy().view(np.uint32), want.view(np.uint32))
    assert _guards_kept(buf, M, N, off)
    if not zp:
        return
    for fn, ref in ((Q.linear_forward_batched, O.linear_forward_batched), (Q.linear_forward, O.linear_forward_rows)):
        rc, want = ref(A, q, s, zps, b, 0.02, 5, sw)
        assert rc == 0
        assert np.array_equal(fn(p, _cu(A, off)).cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_skinny_fp8(gpu, skinny, M, K, N):
    off = (M + K + N) % 3
    A = (2.0 * WL.normal(850, (M, K))).astype(np.float32)
    if M > 4:
        A[1] = 0.0
        A[2, -1] = np.nan
        A[3] = 1e-40
    W = WL.uniform(851, (N, K), -0.125, 0.125)
    b = WL.uniform(852, (N,), -0.125, 0.125)
    qw, sw = O.quantise_weight_fp8(W)
    p = Q.Fp8LinearParams(_cu(qw, off), _cu(sw, 0), _cu(b, 0))
    buf, out = _guarded(M, N, off)
    got, sc = Q.fp8_linear_forward_per_token(p, _cu(A, off), "none", out=out, return_scales=True)
    qa, sa = O.quantise_per_token_fp8(A)
    assert np.array_equal(sc.cpu().numpy().view(np.uint32), sa.view(np.uint32))
    got, want = got.cpu().numpy(), O.layer_fp8_exact(qa, sa, qw, sw, b, 0)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fin = np.isfinite(want).all(axis=1)
    terms = (np.abs(O.e4m3_decode(qa[fin])) * sa[fin, None]).astype(np.float64) @ \
        (np.abs(O.e4m3_decode(qw)) * sw[:, None]).astype(np.float64).T
    bound = (K + 3) * 2.0 ** -24 * (terms + np.abs(b)[None, :]) + 1e-38
    assert np.all(np.abs(got[fin].astype(np.float64) - want[fin]) <= bound)
    assert _guards_kept(buf, M, N, off)


# Zero points whose product with K passes 2^31 make the 64-bit integer term.
@pytest.mark.parametrize("M,K,N,zp_a,zp_w", [(300, 576, 68, 5, 6), (1025, 1024, 132, -7, 6), (4000, 512, 512, 3, 6),
                                             (200, 4160, 64, 100, 6), (130, 2048, 60, 100000, 30000),
                                             (700, 1024, 260, -1024, 1 << 24), (700, 1024, 260, 1025, 1 << 24),
                                             (9000, 512, 1000, 0, 6), (66000, 512, 520, 7, 1 << 24)])
@pytest.mark.parametrize("form", ["rows", "rows_sum", "batched"])
def test_fixed_split(gpu, M, K, N, zp_a, zp_w, form):
    W = WL.uniform(860, (N, K), -0.125, 0.125)
    s = O.per_channel_scales(W, 127.0)
    zps = WL.uniform(861, (N,), -zp_w, zp_w).astype(np.int32)
    q, sw = O.quantise_weight_2d(W, s, zps)
    b = WL.uniform(862, (N,), -0.1, 0.1)
    A = WL.normal(863, (M, K))
    sum_w = None if form == "rows" else sw
    p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), _cu(zps, 0), _cu(b, 0), 0.02, zp_a,
                           None if sum_w is None else _cu(sum_w, 0))
    fn, ref = ((Q.linear_forward_batched, O.linear_forward_batched) if form == "batched"
               else (Q.linear_forward, O.linear_forward_rows))
    y = fn(p, _cu(A, 0)).cpu().numpy()
    rows = np.arange(M) if M <= 512 else np.unique(np.concatenate([np.arange(130), np.arange(M - 130, M)]))
    rc, want = ref(A[rows], q, s, zps, b, 0.02, zp_a, sum_w)
    assert rc == 0
    assert np.array_equal(y[rows].view(np.uint32), want.view(np.uint32))
