"""The rule that gives a decode call its workgroup shape, on the host."""
import pytest

import test_gpu_decode_shapes
import test_gpu_parity
from _shapes import decode_shapes

FORCED = sorted(set(test_gpu_parity.SHAPES) | set(test_gpu_decode_shapes.SHAPES))


@pytest.mark.parametrize("forced", FORCED)
def test_a_forced_shape_is_the_shape(forced):
    """The shapes that the GPU tests force are compiled, so that none of those
    tests runs the fallback in their place."""
    want = (tuple(map(int, forced.split(","))) + (1,))[:3]
    (got,) = decode_shapes([(24, 1, 32, 2 * want[2], True)], forced)
    assert got[:3] == want


def test_a_shape_without_a_kernel_falls_back():
    for forced, per in (("3,1", 1), ("1,2,4", 2), ("1,2,0", 1), ("16,2", 1)):
        assert decode_shapes([(24, 1, 32, per, True)], forced)[0][:3] == (1, 1, 1)


def test_no_launch_of_too_many_threads():
    """Every call that one wave per unit can serve (fewer than 2^32 threads)
    keeps below 2^32 with the shape it takes."""
    units = sorted({1, 2048, 2049, 1 << 20} | {(1 << e) + i for e in range(21, 26) for i in (-1, 0, 1)} | {(1 << 26) - 1})
    calls = [(u, layers, n, per, fused) for u in units for layers in (1, 3) for n in (1, 2, 31, 32, 64, 65, 200)
             for per in (1, 2, 3, 4, 6, 16) for fused in (False, True)]
    for call, (nw, _, r, threads) in zip(calls, decode_shapes(calls)):
        assert threads == call[0] * 64 * nw < 2**32 and call[3] % r == 0, (call, nw, r)
