"""The rule that gives a decode call its workgroup shape, on the host."""
from _shapes import decode_shapes


def test_no_launch_of_too_many_threads():
    """Every call that one wave per unit can serve (fewer than 2^32 threads)
    keeps below 2^32 with the shape it takes."""
    units = sorted({1, 2048, 2049, 1 << 20} | {(1 << e) + i for e in range(21, 26) for i in (-1, 0, 1)} | {(1 << 26) - 1})
    calls = [(u, layers, n, per, fused) for u in units for layers in (1, 3) for n in (1, 2, 31, 32, 64, 65, 200)
             for per in (1, 2, 3, 4, 6, 16) for fused in (False, True)]
    for call, (nw, _, r, threads) in zip(calls, decode_shapes(calls)):
        assert threads == call[0] * 64 * nw < 2**32 and call[3] % r == 0, (call, nw, r)
