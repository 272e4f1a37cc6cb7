"""The rule that gives a staged prefill call its workgroup shapes, on the host."""
import test_gpu_prefill_shapes
from _shapes import staged_shapes

QUERIES = {(16, 1): 256, (16, 2): 128, (8, 1): 128, (8, 2): 64}


def test_the_gpu_tests_meet_every_shape():
    cases = test_gpu_prefill_shapes.STAGED
    got = staged_shapes([(c[0] * c[1], c[5], c[3]) for c in cases])
    assert got == [c[6] for c in cases]
    assert {g[1:] for g in got} == set(QUERIES) and any(g[0] for g in got)


def test_no_call_takes_more_threads_than_with_one_shape():
    """Past one round of the chip the shapes hold no more threads in all than
    16 waves x 16 queries do, so that no call passes a launch's 2^32."""
    calls = [(units, tokens, slots) for units in (1 << 20, (1 << 21) + 7, 3999999) for tokens in range(1, 700, 3)
             for slots in (512, 2048)]
    for (units, tokens, _), (full, qw, ks) in zip(calls, staged_shapes(calls)):
        whole = -(-tokens // 256) * 1024
        rest = -(-tokens // QUERIES[qw, ks]) * 64 * qw
        assert 0 <= full < units and full * whole + (units - full) * rest <= units * whole


def test_short_chunks_on_short_rings_split_no_block():
    """Up to 128 tokens 16 waves with two on a block serve only rings of more
    than 512 slots: on empty ones they take longer than 16 waves x 16 queries."""
    for tokens in (65, 100, 128):
        assert staged_shapes([(192, tokens, 512), (192, tokens, 513)]) == [(0, 8, 1), (0, 16, 2)]
    assert staged_shapes([(96, 129, 512)]) == [(0, 16, 2)]
