"""Staged prefill in each of its workgroup shapes against the float64 oracle
(|gpu - ref| <= 2e-3 + 1e-3 |ref|): 16 or 8 waves, one or two on each block
of 16 queries, picked by the number of units and the chunk's length (asserted), at chunks
around a workgroup's queries, rings on and off the 32-slot grid, and queries
that see keys in only one half of the tiles.  The committed ring is exact."""
import numpy as np
import pytest

import oracle
from _ringsim import Mirror, check_close
from _shapes import staged_shapes

pytestmark = pytest.mark.gpu


# entries, heads, kv heads, slots, position, tokens, and the shape: units in full
# rounds of 16 waves x 16 queries, waves per workgroup and per block of queries
# of the rest
STAGED = [
    (1, 4, 2, 128, 200, 63, (0, 8, 2)), (1, 4, 2, 128, 200, 65, (0, 8, 2)),  # 64-query workgroups, an edge and past it
    (1, 4, 2, 96, 0, 1, (0, 8, 2)),                # one key: the second wave of a block sees none
    (1, 4, 2, 100, 40, 33, (0, 8, 2)),             # off the 32-slot grid
    (1, 2, 2, 300, 500, 300, (0, 8, 2)),           # more than 256 tokens, one head a kv head
    (3, 32, 2, 96, 130, 90, (0, 8, 2)),            # 96 units
    (9, 32, 1, 40, 70, 33, (0, 8, 2)),             # 288 units: past one round of lone workgroups
    (8, 32, 4, 64, 90, 17, (0, 8, 2)),             # 256 units
    (20, 32, 1, 40, 50, 20, (0, 8, 2)),            # 640 units: past a round of two workgroups a CU
    (4, 32, 2, 160, 200, 129, (0, 16, 2)),         # 128-query workgroups, an edge and past it
    (3, 32, 2, 300, 280, 200, (0, 16, 2)),         # off the grid
    (3, 32, 2, 256, 0, 256, (0, 16, 2)),           # empty history: half the tiles at most
    (6, 32, 2, 544, 600, 100, (0, 16, 2)), (6, 32, 2, 512, 600, 100, (0, 8, 1)),  # past | up to 512 slots
    (16, 32, 1, 96, 70, 70, (0, 8, 1)),            # 8 waves, 128 queries
    (16, 32, 1, 160, 100, 128, (0, 8, 1)), (9, 32, 2, 100, 130, 100, (0, 8, 1)),
    (5, 32, 2, 160, 100, 130, (0, 16, 1)),         # 160 units, 130 tokens
    (5, 32, 2, 512, 100, 500, (128, 8, 2)),        # 128 units in a full round, 32 apart
]


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n_batch,heads,kv,n_ctx,pos0,n_tok,shape", STAGED)
def test_staged_shapes(gpu, d, n_batch, heads, kv, n_ctx, pos0, n_tok, shape):
    assert staged_shapes([(n_batch * heads, n_tok, n_ctx)]) == [shape]
    m = Mirror(gpu, 1, n_batch, kv, d, n_ctx)
    pos = [max(0, pos0 - 7 * (b % 3)) for b in range(n_batch)]
    for b in range(n_batch):
        m.fill_range(0, b, 0, pos[b], seed=300 + 2 * b)
    q, k, v = (oracle.round_bf16(oracle.normal(20 + i, n_batch * n_tok * h * d)).reshape(n_batch, n_tok, h, d)
               for i, h in enumerate((heads, kv, kv)))
    out = gpu.full(q.shape, float("nan"), device="cuda")
    m.ring.prefill(0, gpu.tensor(pos, dtype=gpu.int32, device="cuda"), m.dev(q, gpu.bfloat16),
                   m.dev(k, gpu.bfloat16), m.dev(v, gpu.bfloat16), out, heads, stream=m.stream)
    gpu.cuda.synchronize()
    got = out.cpu().numpy()
    for b in range(0, n_batch, max(1, n_batch // 3)):
        kc, vc = m.orc[(0, b)]
        check_close(got[b], oracle.ring_prefill_f64(kc, vc, pos[b], q[b], k[b], v[b], heads), f"entry {b}")
        m.assert_ring_equal(0, b)
    assert np.all(np.isfinite(got))


def test_not_a_number_stays_in_its_row(gpu):
    """Two waves on a block of queries: a NaN or an infinity in q makes its own
    row's output NaN and no other's."""
    heads, kv, d, n_ctx, n_tok = 4, 2, 128, 64, 40
    m = Mirror(gpu, 1, 1, kv, d, n_ctx)
    m.fill_range(0, 0, 0, 50, seed=9)
    q, k, v = (oracle.round_bf16(oracle.normal(50 + i, n_tok * h * d)).reshape(1, n_tok, h, d)
               for i, h in enumerate((heads, kv, kv)))
    q[0, 5, 1, 7] = np.nan
    q[0, 20, 3, 90] = np.inf
    out = gpu.zeros(q.shape, dtype=gpu.float32, device="cuda")
    m.ring.prefill(0, gpu.tensor([50], dtype=gpu.int32, device="cuda"), m.dev(q, gpu.bfloat16),
                   m.dev(k, gpu.bfloat16), m.dev(v, gpu.bfloat16), out, heads, stream=m.stream)
    gpu.cuda.synchronize()
    bad = np.zeros((n_tok, heads), dtype=bool)
    bad[5, 1] = bad[20, 3] = True
    assert np.array_equal(np.isnan(out.cpu().numpy()[0]).all(axis=-1), bad)
    assert np.array_equal(np.isnan(out.cpu().numpy()[0]).any(axis=-1), bad)
