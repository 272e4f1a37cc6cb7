"""The streaming GEMV beyond four two-row chunks per wave: its outputs equal the
pair-walking kernel's bit for bit (they share the quantizer and the pair
product) at chunk counts around whole passes of the 2048 waves, odd rows and
one and two block pairs per lane, and on both sides of the widths from which
such matrices stream (3584 columns, past 20480 rows 3072); and the float64 evaluation within
1e-5 sum |terms| + 1e-6."""
import numpy as np
import pytest

import oracle
from test_gpu_gemv import _launch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(16385, 2048), (16387, 2048), (20480, 2048), (20482, 2304), (36863, 2048),
                                       (24577, 4352), (16385, 256), (16385, 1792),
                                       (16385, 3584), (16387, 3840), (20480, 3584), (20482, 3072), (36863, 3072),
                                       (16385, 3328), (20480, 3072)])
def test_stream_equals_pair_walk(gpu, rows, cols):
    w = oracle.quantize_q4_0(oracle.normal(rows + cols, rows * cols)).view(np.uint8).copy()
    x = oracle.normal(17 + cols, cols)
    a = _launch(gpu, w, 0, x, rows, cols)
    b = _launch(gpu, w, 4, x, rows, cols)  # off the 16-byte grid: the pair-walking kernel
    assert np.all(np.isfinite(a))
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    ref, tabs = oracle.gemv_q4_0_q8_1_f64(w.view(oracle.BLOCK_DTYPE), oracle.quantize_q8_1(x), rows, cols)
    assert np.all(np.abs(a - ref) <= 1e-5 * tabs + 1e-6)
