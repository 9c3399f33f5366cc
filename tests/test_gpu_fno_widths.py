"""The FNO runtime's one-launch local linear + tail and projection head at the
widths other than 64, and the blocked fp32 Linear at widths that have
neither, bit for bit against the oracle (and the fused forms against the
separate launches, kernel path no_layer_tail): every instantiated width,
with and without the last k % 8 fused terms, thread counts the width does
not divide (20, 24, 40, 48), every x2 fake-quant the fused form takes, ReLU
and GELU; blocked Linear: one column block and several, k off 4 and 8, rows
that do not fill a block, padded rows."""
import ctypes as C

import numpy as np
import pytest

from neuroflow_amd import _lib
from neuroflow_amd.runtime import load
from oracle import fno1d as OF
from oracle import fno2d as OF2
from tests import test_gpu_runtime as T1
from tests import test_gpu_runtime_2d as T2

pytestmark = pytest.mark.gpu


def _run(tmp_path, ir, x, out_ch, flag=0, int8=False):
    path = tmp_path / "m.nneuroir"
    path.write_bytes(ir)
    prev = C.c_int(0)
    L = _lib.lib()
    _lib.check(L.nflow_debug_set_kernel_path(b"no_layer_tail", flag, C.byref(prev)), "path")
    try:
        rt = load().InferenceRuntime(str(path))
        if int8:
            rt.enable_int8_gemm()
        y = np.zeros(x.shape[:-1] + (out_ch,), np.float32)
        rt.run(x, y)
        return y
    finally:
        _lib.check(L.nflow_debug_set_kernel_path(b"no_layer_tail", prev.value, None), "path")


# 512 whole 32-token tiles (several per block), then one and a few tiles.
FUSED = [(1, 32, 1, 1, 64, 6, 2, 1, False, ["tensor"], True), (2, 64, 1, 1, 64, 6, 2, 1, True, ["token", "tensor"], False),
         (16, 1024, 1, 1, 32, 6, 3, 1, False, ["tensor"], True), (3, 64, 1, 1, 48, 6, 3, 1, True, ["tensor", "fp8", "tensor"], True),
         (2, 32, 1, 1, 20, 6, 3, 1, False, ["fp8", "tensor"], True), (5, 32, 1, 1, 16, 6, 2, 1, False, ["tensor"], True),
         (2, 64, 1, 1, 24, 6, 2, 1, False, ["tensor"], True), (2, 64, 1, 1, 40, 6, 2, 1, False, ["tensor"], True),
         (1, 32, 1, 1, 20, 6, 2, 1, False, ["tensor"], False), (3, 32, 1, 1, 48, 6, 2, 1, False, ["fp8"], False)] + \
        [(16, 1024, 1, 1, w, 6, 2, 1, relu, kinds, False)
         for w, relu, kinds in [(16, False, ["tensor"]), (20, True, None), (20, False, ["fp8"]), (24, False, ["tensor"]),
                                (32, True, ["fp8", "tensor"]), (32, False, None), (40, False, ["tensor", "fp8"]),
                                (48, False, ["tensor"]), (48, True, ["fp8"])]]


@pytest.mark.parametrize("case", FUSED, ids=T1._ids)
def test_fused_widths_fno1d(gpu, tmp_path, case):
    ir, x, m = T1._model(case)
    want = OF.forward(m, x)
    for flag in (0, 1):
        y = _run(tmp_path, ir, x, 1, flag, case[10])
        assert np.array_equal(T1._bits(y), T1._bits(want)), (flag, int((T1._bits(y) != T1._bits(want)).sum()))


@pytest.mark.parametrize("case", [(4, 64, 64, 1, 1, w, 5, 5, 2, 1, relu, kinds) for w, relu, kinds in
                                  [(16, True, ["fp8"]), (20, False, ["tensor", "fp8"]), (32, False, ["fp8"]),
                                   (48, False, ["tensor"])]], ids=T2._ids)
def test_fused_widths_fno2d(gpu, tmp_path, case):
    ir, x, m = T2._model(case)
    want = OF2.forward(m, x)
    for flag in (0, 1):
        y = _run(tmp_path, ir, x, 1, flag)
        assert np.array_equal(T2._bits(y), T2._bits(want)), flag


@pytest.mark.parametrize("case", [(3, 32, 2, 1, 17, 6, 2, 1, False, None, False),    # k and n off 4, 2 input channels
                                  (1, 8, 3, 2, 33, 4, 1, 1, True, ["tensor"], False),  # two column blocks, part-filled rows
                                  (2, 16, 1, 1, 70, 4, 1, 1, False, ["fp8"], False),
                                  (1, 4, 3, 1, 20, 2, 2, 8, False, ["tensor"], False),  # padded rows
                                  (2, 256, 1, 1, 100, 4, 1, 1, False, None, False)], ids=T1._ids)
def test_blocked_linear(gpu, tmp_path, case):
    ir, x, m = T1._model(case)
    y = _run(tmp_path, ir, x, case[3])
    want = OF.forward(m, x)
    assert np.array_equal(T1._bits(y), T1._bits(want))


# The same forms at the row counts the blocked Linear serves (1536 and more;
# the cases above run one thread per output).
@pytest.mark.parametrize("case", [(48, 32, 2, 1, 17, 6, 2, 1, False, None, False),
                                  (201, 8, 3, 2, 33, 4, 1, 1, True, ["tensor"], False),
                                  (99, 16, 1, 1, 70, 4, 1, 1, False, ["fp8"], False),
                                  (400, 4, 3, 1, 20, 2, 2, 8, False, ["tensor"], False),
                                  (8, 256, 1, 1, 100, 4, 1, 1, False, None, False),
                                  (6, 256, 1, 1, 28, 4, 2, 1, False, None, False)], ids=T1._ids)
def test_blocked_linear_many_rows(gpu, tmp_path, case):
    ir, x, m = T1._model(case)
    y = _run(tmp_path, ir, x, case[3])
    want = OF.forward(m, x)
    assert np.array_equal(T1._bits(y), T1._bits(want))
