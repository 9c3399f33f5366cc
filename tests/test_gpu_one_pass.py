"""The one-pass layer kernel (quantise into LDS, then the whole N range) at the
sizes where it can go wrong, against the oracle: K and N off every tile
(K % 64, K % 4, N % 64, N % 4, K below a wave's float4s), row counts around
the 16- and 64-row tiles, buffers aligned to 4 bytes only, the column chunks
shared over blocks, per-token INT8, fixed-scale INT8 (both formulas, with the
row form's dropped K tail) and FP8, on either tile height.

INT8 outputs must equal the oracle's bits (codes, accumulators and dequantise
are exact); FP8 is held to K * 2^-24 * sum|terms| (fp32 accumulation of exact
products) plus the three roundings of the dequantise."""
import ctypes

import numpy as np
import pytest
import torch

from neuroflow_amd import _lib
from neuroflow_amd import quant as Q
from neuroflow_amd import workloads as WL
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (M, K, N): tile edges and remainders of the 16 / 64-row tiles, the 64-wide
# K blocks (template sizes 64, 128, 256, 512, 1024) and the 128 / 256-column
# chunks; the last ones cross the 16-row line and share chunks over blocks.
SHAPES = [(1, 4, 4), (3, 5, 7), (17, 64, 65), (63, 67, 127), (64, 128, 128), (65, 130, 129), (16, 192, 256),
          (129, 255, 300), (40, 257, 64), (70, 320, 200), (33, 511, 96), (15, 512, 257), (48, 513, 66),
          (31, 1000, 130), (18, 1023, 33), (20000, 101, 128), (9000, 256, 513), (300, 100, 1030)]


@pytest.fixture(params=[0, 16, 64], ids=["auto", "rows16", "rows64"])
def tile_rows(request):
    prev = ctypes.c_int(0)
    L = _lib.lib()
    _lib.check(L.nflow_debug_set_kernel_path(b"token_rows", request.param, ctypes.byref(prev)), "path")
    yield request.param
    _lib.check(L.nflow_debug_set_kernel_path(b"token_rows", prev.value, None), "path")


def _cu(a, off):
    """A device copy that starts `off` elements past a 256-byte boundary."""
    a = np.ascontiguousarray(a)
    buf = torch.empty(a.size + off, dtype=torch.from_numpy(a[:0].reshape(-1)).dtype, device="cuda")
    out = buf[off:].view(a.shape)
    out.copy_(torch.from_numpy(a))
    return out


def _guarded(M, N, off):
    """An (M, N) output `off` floats past a boundary, with guards around it."""
    buf = torch.full((M * N + 64 + off,), 7.0, dtype=torch.float32, device="cuda")
    return buf, buf[off:off + M * N].view(M, N)


def _guards_kept(buf, M, N, off):
    return bool((buf[:off] == 7.0).all()) and bool((buf[off + M * N:] == 7.0).all())


def _rows(M):
    return np.arange(M) if M <= 512 else np.unique(np.concatenate([np.arange(70), np.arange(M - 70, M),
                                                                   np.arange(0, M, 89)]))


def _int8(N, K, sid):
    W = WL.uniform(sid, (N, K), -0.125, 0.125)
    s = O.per_channel_scales(W, 127.0)
    zps = WL.uniform(sid + 1, (N,), -6, 6).astype(np.int32)
    q, sw = O.quantise_weight_2d(W, s, zps)
    return q, s, zps, sw, WL.uniform(sid + 2, (N,), -0.1, 0.1)


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("zp", [False, True])
def test_per_token_int8(gpu, tile_rows, M, K, N, zp):
    off = (M + K + N) % 3
    q, s, zps, sw, b = _int8(N, K, 800)
    A = WL.normal(803, (M, K))
    A[M // 2] = 0.0
    p = Q.Int8LinearParams(_cu(q, off), _cu(s, 0), _cu(zps, 0) if zp else None, _cu(b, 0),
                           sum_W_per_row=_cu(sw, 0) if zp else None)
    buf, out = _guarded(M, N, off)
    y, sc = Q.linear_forward_per_token(p, _cu(A, off), "relu", out=out, return_scales=True)
    rows = _rows(M)
    want, s_want = O.layer_per_token_i8(A[rows], q, s, zps if zp else None, b, sw if zp else None, 1)
    assert np.array_equal(sc.cpu().numpy()[rows].view(np.uint32), s_want.view(np.uint32))
    assert np.array_equal(y.cpu().numpy()[rows].view(np.uint32), want.view(np.uint32))
    assert _guards_kept(buf, M, N, off)


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("form", ["rows", "batched"])
def test_fixed_int8(gpu, tile_rows, M, K, N, form):
    off = (M + K + N) % 3
    q, s, zps, sw, b = _int8(N, K, 810)
    A = WL.normal(813, (M, K))
    A.reshape(-1)[:min(M * K, 8)] = np.array([np.nan, np.inf, -np.inf, 3e9, -3e9, 1e-40, -0.0, 0.05],
                                             np.float32)[:min(M * K, 8)]
    p = Q.Int8LinearParams(_cu(q, off), _cu(s, 0), _cu(zps, 0), _cu(b, 0), 0.02, 5,
                           _cu(sw, 0) if form == "batched" else None)
    fn, ref = ((Q.linear_forward_batched, O.linear_forward_batched) if form == "batched"
               else (Q.linear_forward, O.linear_forward_rows))
    y = fn(p, _cu(A, off)).cpu().numpy()
    rows = _rows(M)
    rc, want = ref(A[rows], q, s, zps, b, 0.02, 5, sw if form == "batched" else None)
    assert rc == 0
    assert np.array_equal(y[rows].view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_fp8(gpu, tile_rows, M, K, N):
    off = (M + K + N) % 3
    A = (2.0 * WL.normal(820, (M, K))).astype(np.float32)
    A = np.where(WL.uniform(821, (M, K)) < 0.02, 20.0 * A, A).astype(np.float32)
    A[M // 2] = 0.0
    if M > 8:
        A[1, -1] = np.nan
        A[2, 0] = np.inf
        A[3] = 1e-40          # a subnormal row scale: its reciprocal is infinite
        A[3, 0] = 0.0
        A[4, :] = (np.arange(K) % 64 - 32) * 2.0 ** -9     # around the subnormal cap of the format
        A[4, 0] = 448.0
    W = WL.uniform(822, (N, K), -0.125, 0.125)
    b = WL.uniform(823, (N,), -0.125, 0.125)
    qw, sw = O.quantise_weight_fp8(W)
    p = Q.Fp8LinearParams(_cu(qw, off), _cu(sw, 0), _cu(b, 0))
    buf, out = _guarded(M, N, off)
    y, sc = Q.fp8_linear_forward_per_token(p, _cu(A, off), "none", out=out, return_scales=True)
    rows = _rows(M)
    qa, sa = O.quantise_per_token_fp8(A[rows])
    got = y.cpu().numpy()[rows]
    assert np.array_equal(sc.cpu().numpy()[rows].view(np.uint32), sa.view(np.uint32))
    want = O.layer_fp8_exact(qa, sa, qw, sw, b, 0)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fin = np.isfinite(want).all(axis=1)
    terms = (np.abs(O.e4m3_decode(qa[fin])) * sa[fin, None]).astype(np.float64) @ \
        (np.abs(O.e4m3_decode(qw)) * sw[:, None]).astype(np.float64).T
    bound = (K + 3) * 2.0 ** -24 * (terms + np.abs(b)[None, :]) + 1e-38
    assert np.all(np.abs(got[fin].astype(np.float64) - want[fin]) <= bound)
    assert _guards_kept(buf, M, N, off)


def test_noalloc_large_codes_keep_the_one_pass_kernel(gpu):
    """K = 512 with a wide N takes quantise + GEMM where that is faster, but the
    no-allocation entry point, whose scratch cannot hold 160000 rows of codes,
    serves it all the same (it never needed scratch at K = 512)."""
    M, K, N = 160000, 512, 576
    q, s, _, _, b = _int8(N, K, 870)
    x = torch.from_numpy(WL.normal(873, (1000, K))).cuda().repeat(M // 1000, 1)
    p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), None, _cu(b, 0))
    ps = p.c_struct()
    out = torch.empty(M, N, device="cuda")
    rc = _lib.lib().nflow_int8_linear_forward_per_token_noalloc(ctypes.byref(ps), M, x.data_ptr(), out.data_ptr(), None,
                                                                0, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "noalloc")
    want = Q.linear_forward_per_token(p, x, "none")
    assert torch.equal(out.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("M,K", [(1, 64), (8, 200), (16, 1024), (300, 200), (300, 512), (5000, 256), (70, 1024), (33, 96)])
@pytest.mark.parametrize("fmt", ["int8", "fp8", "fixed"])
def test_square_layer_in_place(gpu, M, K, fmt):
    """out = the input tensor: the same bits as out of place (a tile's columns
    are then not shared over blocks, and rows not over the few-row kernel's)."""
    A = WL.normal(880, (M, K))
    if fmt == "fp8":
        qw, sw = O.quantise_weight_fp8(WL.uniform(881, (K, K), -0.125, 0.125))
        p = Q.Fp8LinearParams(_cu(qw, 0), _cu(sw, 0))
        fn, args = _lib.lib().nflow_fp8_linear_forward_per_token, (None, 1)
    else:
        q, s, zps, sw, b = _int8(K, K, 882)
        p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), _cu(zps, 0), _cu(b, 0), 0.02, 3)
        fn, args = ((_lib.lib().nflow_int8_linear_forward_per_token, (None, 1)) if fmt == "int8"
                    else (_lib.lib().nflow_int8_linear_forward_rows, ()))
    ps, st = p.c_struct(), torch.cuda.current_stream().cuda_stream
    x = _cu(A, 0)
    out = torch.empty(M, K, device="cuda")
    _lib.check(fn(ctypes.byref(ps), M, x.data_ptr(), out.data_ptr(), *args, st), "layer")
    for _ in range(3):
        y = _cu(A, 0)
        _lib.check(fn(ctypes.byref(ps), M, y.data_ptr(), y.data_ptr(), *args, st), "in place")
        if fmt == "fp8":     # another kernel may sum in another order
            assert torch.allclose(y, out, rtol=1e-5, atol=1e-5)
        else:
            assert torch.equal(y.view(torch.int32), out.view(torch.int32))


# Zero points within 8 bits (the 32-bit epilogue), at the edge of 24 bits and
# beyond, where its products and the 64-bit term need the general form.
@pytest.mark.parametrize("zp_w,zp_a", [(127, -128), (1 << 21, 3), ((1 << 22) + 1, 3), (1 << 24, 100000), (1 << 30, 0)])
@pytest.mark.parametrize("M,K,N", [(70, 100, 65), (33, 512, 128), (20, 1000, 36), (65, 60, 260)])
def test_zero_point_range(gpu, tile_rows, zp_w, zp_a, M, K, N):
    W = WL.uniform(890, (N, K), -0.125, 0.125)
    s = O.per_channel_scales(W, 127.0)
    zps = WL.uniform(891, (N,), -zp_w, zp_w).astype(np.int32)
    zps[:2] = zp_w, -zp_w
    q, sw = O.quantise_weight_2d(W, s, zps)
    b = WL.uniform(892, (N,), -0.1, 0.1)
    A = WL.normal(893, (M, K))
    p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), _cu(zps, 0), _cu(b, 0), 0.02, zp_a, _cu(sw, 0))
    want, _ = O.layer_per_token_i8(A, q, s, zps, b, sw, 0)
    got = Q.linear_forward_per_token(p, _cu(A, 0), "none").cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    for fn, ref in ((Q.linear_forward_batched, O.linear_forward_batched), (Q.linear_forward, O.linear_forward_rows)):
        rc, want = ref(A, q, s, zps, b, 0.02, zp_a, sw)
        assert rc == 0
        assert np.array_equal(fn(p, _cu(A, 0)).cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("M", [1, 63, 64, 65, 200, 6000])
@pytest.mark.parametrize("K,N", [(128, 64), (256, 128), (512, 64), (512, 128), (256, 192)])
def test_whole_shapes(gpu, tile_rows, M, K, N):
    """Whole K blocks and column strips at aligned buffers, the narrow (N <= 128)
    and the wide form, in the three formats."""
    q, s, zps, sw, b = _int8(N, K, 895)
    A = WL.normal(898, (M, K))
    rows = _rows(M)
    p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), _cu(zps, 0), _cu(b, 0), 0.02, 5, _cu(sw, 0))
    buf, out = _guarded(M, N, 0)
    y = Q.linear_forward_per_token(p, _cu(A, 0), "relu", out=out).cpu().numpy()[rows]
    want, _ = O.layer_per_token_i8(A[rows], q, s, zps, b, sw, 1)
    assert np.array_equal(y.view(np.uint32), want.view(np.uint32))
    assert _guards_kept(buf, M, N, 0)
    y = Q.linear_forward_batched(p, _cu(A, 0)).cpu().numpy()[rows]
    rc, want = O.linear_forward_batched(A[rows], q, s, zps, b, 0.02, 5, sw)
    assert rc == 0 and np.array_equal(y.view(np.uint32), want.view(np.uint32))
    qw, s8 = O.quantise_weight_fp8(WL.uniform(899, (N, K), -0.125, 0.125))
    buf, out = _guarded(M, N, 0)
    y = Q.fp8_linear_forward_per_token(Q.Fp8LinearParams(_cu(qw, 0), _cu(s8, 0), _cu(b, 0)), _cu(A, 0), "none", out=out)
    assert _guards_kept(buf, M, N, 0)
    qa, sa = O.quantise_per_token_fp8(A[rows])
    want = O.layer_fp8_exact(qa, sa, qw, s8, b, 0)
    terms = (np.abs(O.e4m3_decode(qa)) * sa[:, None]).astype(np.float64) @ \
        (np.abs(O.e4m3_decode(qw)) * s8[:, None]).astype(np.float64).T
    bound = (K + 3) * 2.0 ** -24 * (terms + np.abs(b)[None, :]) + 1e-38
    assert np.all(np.abs(y.cpu().numpy()[rows].astype(np.float64) - want) <= bound)


# Many rows of small layers: the row-tile kernel's share (per-token INT8 of K < 64
# into 65 to 160 columns, two K blocks into a few), a thread per output (K N <=
# 48), and their neighbours on the one-pass kernel.
@pytest.mark.parametrize("kind,M,K,N", [("int8", 65537, 8, 132), ("int8", 65600, 60, 68), ("int8", 65536, 4, 160),
                                        ("int8", 65536, 64, 132), ("int8", 65537, 8, 164), ("fp8", 100003, 100, 8),
                                        ("fp8", 100000, 128, 16), ("fp8", 100000, 68, 20), ("fp8", 24577, 84, 4),
                                        ("int8", 49153, 100, 40), ("int8", 49152, 128, 20), ("int8", 49153, 68, 4),
                                        ("int8", 49160, 72, 48), ("int8", 49160, 72, 52), ("fixed", 100003, 100, 8),
                                        ("fixed", 100000, 128, 16), ("fixed", 49153, 124, 40), ("fixed", 49153, 128, 24), ("fixed", 32769, 4, 5), ("fixed", 40001, 16, 3),
                                        ("fixed", 32769, 7, 7)])
def test_many_rows_of_small_layers(gpu, kind, M, K, N):
    base = 1009
    A = WL.normal(900, (base, K))
    idx = torch.arange(M, device="cuda") % base
    x = torch.from_numpy(A).cuda()[idx].contiguous()
    q, s, zps, sw, b = _int8(N, K, 901)
    buf, out = _guarded(M, N, 0)
    st = torch.cuda.current_stream().cuda_stream
    if kind == "fp8":
        qw, s8 = O.quantise_weight_fp8(WL.uniform(902, (N, K), -0.125, 0.125))
        Q.fp8_linear_forward_per_token(Q.Fp8LinearParams(_cu(qw, 0), _cu(s8, 0), _cu(b, 0)), x, "none", out=out)
        qa, sa = O.quantise_per_token_fp8(A)
        want = O.layer_fp8_exact(qa, sa, qw, s8, b, 0)
        terms = (np.abs(O.e4m3_decode(qa)) * sa[:, None]).astype(np.float64) @ \
            (np.abs(O.e4m3_decode(qw)) * s8[:, None]).astype(np.float64).T
        bound = (K + 3) * 2.0 ** -24 * (terms + np.abs(b)[None, :]) + 1e-38
        assert np.all(np.abs(out[:base].cpu().numpy().astype(np.float64) - want) <= bound)
        assert torch.equal(out.view(torch.int32), out[:base][idx].view(torch.int32))
    elif kind == "int8":
        p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), _cu(zps, 0), _cu(b, 0), sum_W_per_row=_cu(sw, 0))
        Q.linear_forward_per_token(p, x, "relu", out=out)
        want, _ = O.layer_per_token_i8(A, q, s, zps, b, sw, 1)
        assert torch.equal(out.view(torch.int32), torch.from_numpy(want).cuda()[idx].view(torch.int32))
    else:
        ps = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), _cu(zps, 0), _cu(b, 0), 0.02, 5, _cu(sw, 0))
        for fn, ref in ((_lib.lib().nflow_int8_linear_forward_batched, O.linear_forward_batched),
                        (_lib.lib().nflow_int8_linear_forward_rows, O.linear_forward_rows)):
            out.fill_(7.0)
            _lib.check(fn(ctypes.byref(ps.c_struct()), M, x.data_ptr(), out.data_ptr(), st), "fixed")
            rc, want = ref(A, q, s, zps, b, 0.02, 5, sw)
            assert rc == 0
            assert torch.equal(out.view(torch.int32), torch.from_numpy(want).cuda()[idx].view(torch.int32))
    assert _guards_kept(buf, M, N, 0)


# Sizes on both sides of the rules that choose between the one-pass kernel and
# quantise + GEMM, and among the GEMM's tiles; whichever runs, the same bits.
@pytest.mark.parametrize("M,K,N", [(3000, 128, 800), (1000, 128, 800), (3000, 256, 1000), (1500, 256, 1000), (6000, 192, 640),
                                   (12500, 192, 640), (2000, 384, 1000), (1000, 384, 1000), (4096, 512, 500), (16385, 320, 300),
                                   (4096, 640, 768), (9000, 1536, 384), (2100, 960, 516), (300, 3072, 512)])
def test_same_bits_in_either_form(gpu, M, K, N):
    base = 997
    q, s, zps, sw, b = _int8(N, K, 920)
    A = WL.normal(923, (base, K))
    idx = torch.arange(M, device="cuda") % base
    x = torch.from_numpy(A).cuda()[idx].contiguous()
    p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), _cu(zps, 0), _cu(b, 0), sum_W_per_row=_cu(sw, 0))
    want, _ = O.layer_per_token_i8(A[:min(M, base)], q, s, zps, b, sw, 1)
    want = torch.from_numpy(want).cuda()[idx]
    L = _lib.lib()
    for path in (None, b"no_gemm", b"no_token_gemm"):
        if path == b"no_gemm" and K > 1024:
            continue     # that leaves the generic kernel
        prev = ctypes.c_int(0)
        if path:
            _lib.check(L.nflow_debug_set_kernel_path(path, 1, ctypes.byref(prev)), "path")
        try:
            y = Q.linear_forward_per_token(p, x, "relu")
        finally:
            if path:
                _lib.check(L.nflow_debug_set_kernel_path(path, prev.value, None), "path")
        assert torch.equal(y.view(torch.int32), want.view(torch.int32)), path


@pytest.mark.parametrize("M,K,N,path", [(70, 100, 65, None), (70, 60, 260, None), (33, 1000, 36, None), (40, 20, 36, None),
                                        (5, 100, 48, "skinny"), (3, 1000, 20, "skinny")])
def test_rows_of_vanishing_scale(gpu, M, K, N, path):
    """Rows so small that absmax / 127 rounds to 0: every code is -128 and the
    output is the bias plus a zero whose sign is the integer result's, so a
    code past K in the row's sum shows under a bias of -0."""
    q, s, zps, sw, _ = _int8(N, K, 910)
    b = np.full(N, -0.0, np.float32)
    A = np.full((M, K), 1e-44, np.float32)
    A[1::2, ::3] = -7e-45
    L = _lib.lib()
    prev = ctypes.c_int(0)
    if path:
        _lib.check(L.nflow_debug_set_kernel_path(path.encode(), 1, ctypes.byref(prev)), "path")
    p = Q.Int8LinearParams(_cu(q, 0), _cu(s, 0), _cu(zps, 0), _cu(b, 0), sum_W_per_row=_cu(sw, 0))
    got = Q.linear_forward_per_token(p, _cu(A, 0), "none").cpu().numpy()
    if path:
        _lib.check(L.nflow_debug_set_kernel_path(path.encode(), prev.value, None), "path")
    want, sc = O.layer_per_token_i8(A, q, s, zps, b, sw, 0)
    assert (sc == 0.0).all() and np.signbit(want).any() and not np.signbit(want).all()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
