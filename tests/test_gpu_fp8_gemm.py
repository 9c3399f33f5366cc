"""The tiled GEMM on E4M3 codes at its edges (row and column tiles of 64 and
128, K steps around its three stages, N off 16 and 64), through the raw
product, the quantised-input layer and the per-token layer, against the
exact-product oracle.  Bound: fp32 accumulation of exact products, K * 2^-24
* sum|terms|, and the three roundings of the dequantise."""
import ctypes

import numpy as np
import pytest
import torch

from neuroflow_amd import _lib
from neuroflow_amd import quant as Q
from neuroflow_amd import workloads as WL
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 128, 4), (63, 192, 60), (64, 256, 64), (65, 320, 68), (127, 512, 132), (129, 576, 128), (300, 1024, 200),
          (257, 2048, 96), (200, 1088, 260), (5000, 512, 2060)]


@pytest.fixture(params=[0, 22, 44], ids=["auto", "64x64", "128x128"])
def tile(request):
    prev = ctypes.c_int(0)
    L = _lib.lib()
    _lib.check(L.nflow_debug_set_kernel_path(b"gemm_tile", request.param, ctypes.byref(prev)), "path")
    yield request.param
    _lib.check(L.nflow_debug_set_kernel_path(b"gemm_tile", prev.value, None), "path")


def _cu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_fp8_tiled_gemm(gpu, tile, M, K, N):
    x = (2.0 * WL.normal(930, (M, K))).astype(np.float32)
    x[M // 2] = 0.0
    if M > 4:
        x[3, 5] = np.nan
    W = WL.uniform(931, (N, K), -0.125, 0.125)
    b = WL.uniform(932, (N,), -0.125, 0.125)
    qw, sw = O.quantise_weight_fp8(W)
    rows = np.arange(M) if M <= 512 else np.unique(np.concatenate([np.arange(130), np.arange(M - 130, M)]))
    qa_all, sa_all = O.quantise_per_token_fp8(x)
    qa, sa = qa_all[rows], sa_all[rows]
    raw = Q.fp8_gemm_f32(_cu(qa_all), _cu(qw)).cpu().numpy()[rows].astype(np.float64)
    want_raw = O.gemm_fp8_exact(qa, qw)
    assert np.array_equal(np.isnan(raw), np.isnan(want_raw))
    fin = np.isfinite(want_raw).all(axis=1)
    mag = np.abs(O.e4m3_decode(qa[fin])).astype(np.float64) @ np.abs(O.e4m3_decode(qw)).astype(np.float64).T
    assert np.all(np.abs(raw[fin] - want_raw[fin]) <= K * 2.0 ** -24 * mag + 1e-30)
    p = Q.Fp8LinearParams(_cu(qw), _cu(sw), _cu(b))
    want = O.layer_fp8_exact(qa, sa, qw, sw, b, 1)
    bound = (K + 3) * 2.0 ** -24 * (mag * sa[fin, None] * sw[None, :] + np.abs(b)[None, :]) + 1e-38
    y_q = Q.fp8_linear_forward_quantised(p, _cu(qa_all), _cu(sa_all), "relu").cpu().numpy()[rows]
    y_t, s_t = Q.fp8_linear_forward_per_token(p, _cu(x), "relu", return_scales=True)
    assert np.array_equal(s_t.cpu().numpy()[rows].view(np.uint32), sa.view(np.uint32))
    for y in (y_q, y_t.cpu().numpy()[rows]):
        assert np.array_equal(np.isnan(y), np.isnan(want))
        assert np.all(np.abs(y[fin].astype(np.float64) - want[fin]) <= bound)
