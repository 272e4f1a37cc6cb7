"""The rule that gives a decode call its workgroup shape, on the host."""
import pytest

import test_gpu_decode_shapes
import test_gpu_parity
from _shapes import decode_shapes

FORCED = sorted(set(test_gpu_parity.SHAPES) | set(test_gpu_decode_shapes.SHAPES) | {"1,2,4"})


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


@pytest.mark.parametrize("fused,groups,per,low,low_shape,high_shape", [
    (True, 32, 1, 127, (8, 1, 1), (4, 2, 1)), (False, 32, 1, 127, (8, 2, 1), (4, 2, 1)),
    (True, 64, 1, 256, (8, 2, 1), (4, 2, 1)), (False, 64, 2, 256, (8, 2, 1), (4, 2, 2)),
    (True, 32, 3, 768, (4, 2, 1), (2, 2, 1)), (False, 32, 3, 768, (4, 2, 1), (1, 2, 1)),
    (True, 64, 1, 1536, (2, 2, 1), (1, 2, 1)), (False, 32, 1, 2048, (1, 2, 1), (4, 2, 1)),
    (True, 32, 2, 512, (4, 2, 2), (2, 2, 2)), (False, 32, 4, 1536, (2, 2, 2), (1, 2, 4)),
    (True, 31, 2, 1536, (2, 2, 2), (1, 2, 2)),
    (True, 1, 1, 256, (2, 1, 1), (1, 1, 1)), (True, 3, 1, 511, (2, 1, 1), (1, 2, 1)),
    (False, 6, 1, 512, (4, 2, 1), (2, 2, 1)), (True, 2, 4, 512, (2, 2, 2), (1, 2, 1)),
])
def test_lines_of_units(fused, groups, per, low, low_shape, high_shape):
    got = decode_shapes([(low, 1, groups, per, fused), (low + 1, 1, groups, per, fused)])
    assert [g[:3] for g in got] == [low_shape, high_shape]


@pytest.mark.parametrize("fused,waves", [
    # 1, 2, ... groups: no more waves on short windows than pay there
    (True, [1, 1, 1, 2, 1, 2, 2, 1, 2, 2, 1, 2, 2, 4, 4]),
    (False, [1, 1, 2, 2, 1, 2, 2, 1, 2, 2, 2, 2, 2, 2, 2])])
@pytest.mark.parametrize("units", [513, 640, 768])
def test_waves_of_short_windows(units, fused, waves):
    got = decode_shapes([(units, 1, n + 1, 1, fused) for n in range(len(waves))])
    assert [g[0] for g in got] == waves


@pytest.mark.parametrize("groups", [1, 2, 7, 8, 32, 63, 64, 188])
def test_a_launch_of_several_layers_splits_as_one(groups):
    """The same waves a unit, and for fewer than eight the same groups in flight
    (they decide how often V's code offset is settled)."""
    calls = [(u, layers, groups, per, True) for u in (16, 32, 127, 128, 300, 1000) for per in (1, 2, 4)
             for layers in (1, 2, 32)]
    got = decode_shapes(calls)
    for i in range(0, len(calls), 3):
        for other in got[i + 1:i + 3]:
            assert (other[0], other[2]) == (got[i][0], got[i][2])
            assert other[1] == got[i][1] or got[i][0] == 8
