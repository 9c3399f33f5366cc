"""The elementwise kernels (codec, QuantiseActivation) where their 16-byte
groups can go wrong: element counts around 4, 1024 and several passes, and
buffers 4 bytes (floats) or 1 byte (codes) off a boundary, against the
oracle bit for bit, with the special values in every position of a group."""
import numpy as np
import pytest
import torch

from neuroflow_amd import _lib
from neuroflow_amd import quant as Q
from neuroflow_amd import workloads as WL
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SPECIAL = np.array([np.nan, -np.nan, np.inf, -np.inf, 448.0, 448.1, -455.0, 464.0, 464.1, -480.0, 496.0, 1e30, 0.0, -0.0,
                    1e-10, -1e-10, 0.0146, -0.0149, 0.015625, 1e-40], np.float32)
SIZES = [1, 3, 4, 5, 1023, 1024, 1025, 4099, 4 * 256 * 4 * 3 + 2, 2_000_003]


def _dev(a, off):
    buf = torch.empty(a.size + off, dtype=torch.from_numpy(a[:0]).dtype, device="cuda")
    buf[off:].copy_(torch.from_numpy(a))
    return buf[off:]


def _call(fn, n, in_t, out_dtype, off, *scalars):
    """fn over n elements into a guarded output `off` elements past a boundary."""
    buf = torch.full((n + 64 + off,), 7, dtype=out_dtype, device="cuda")
    _lib.check(fn(in_t.data_ptr(), *scalars[:1], buf[off:].data_ptr(), n, torch.cuda.current_stream().cuda_stream)
               if scalars else fn(in_t.data_ptr(), buf[off:].data_ptr(), n, torch.cuda.current_stream().cuda_stream),
               "call")
    torch.cuda.synchronize()
    out = buf.cpu().numpy()
    assert (out[:off] == 7).all() and (out[off + n:] == 7).all()
    return out[off:off + n]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("off", [0, 1])
def test_codec(gpu, n, off):
    L = _lib.lib()
    x = (WL.normal(900, (n,)) * 3.0).astype(np.float32)
    k = min(n, SPECIAL.size)
    x[n - k:] = SPECIAL[:k]
    x[:k] = SPECIAL[-k:]
    t = _dev(x, off)
    bits = _call(L.nflow_fp8_e4m3_to_bits, n, t, torch.uint8, off)
    assert np.array_equal(bits, O.e4m3_encode(x))
    b = np.resize(np.arange(256, dtype=np.uint8), n)
    vals = _call(L.nflow_fp8_e4m3_from_bits, n, _dev(b, off), torch.float32, off)
    assert np.array_equal(vals.view(np.uint32), O.e4m3_decode(b).view(np.uint32))
    for scale in (0.75, 0.0):
        fq = _call(L.nflow_fp8_e4m3_fake_quant, n, t, torch.float32, off, scale)
        assert np.array_equal(fq.view(np.uint32), O.fp8_fake_quant(x, scale).view(np.uint32))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("scale,zp", [(0.02, 5), (0.25, -3), (0.0, 1), (1e-38, 2)])
def test_quantise_activation(gpu, n, off, scale, zp):
    x = WL.normal(901, (n,)).astype(np.float32)
    k = min(n, SPECIAL.size)
    x[n - k:] = SPECIAL[:k]
    if n > 100:
        x[40:80] = (np.arange(40) - 20 + 0.5) * 0.25      # ties at 0.25
    q = Q.quantise_activation(_dev(x, off).view(1, n), scale, zp)
    assert np.array_equal(q.cpu().numpy().reshape(-1), O.quantise_activation(x.reshape(1, n), scale, zp).reshape(-1))


# From 2^21 elements a thread takes four groups instead of one: the line, a
# ragged end, and several passes of the grid.
@pytest.mark.parametrize("n", [(1 << 21) - 4, 1 << 21, (1 << 21) + 4, 2_500_003, 17_000_001])
def test_large_tensors(gpu, n):
    L = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(n)
    t = torch.randn(n, device="cuda", generator=g) * 3.0
    x = t.cpu().numpy()
    bits = _call(L.nflow_fp8_e4m3_to_bits, n, t, torch.uint8, 0)
    assert np.array_equal(bits, O.e4m3_encode(x))
    vals = _call(L.nflow_fp8_e4m3_from_bits, n, _dev(bits, 0), torch.float32, 0)
    assert np.array_equal(vals.view(np.uint32), O.e4m3_decode(bits).view(np.uint32))
    fq = _call(L.nflow_fp8_e4m3_fake_quant, n, t, torch.float32, 0, 0.75)
    assert np.array_equal(fq.view(np.uint32), O.fp8_fake_quant(x, 0.75).view(np.uint32))
    q = Q.quantise_activation(t.view(1, n), 0.02, 5)
    assert np.array_equal(q.cpu().numpy().reshape(-1), O.quantise_activation(x.reshape(1, n), 0.02, 5).reshape(-1))
