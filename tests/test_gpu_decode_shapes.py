"""Waves per unit and groups in flight of the decode kernel against the float64
oracle (|gpu - ref| <= 2e-3 + 1e-3 |ref|): the default rule on both sides of
each of its lines, and the shapes that it chooses, forced, at runs of no, one
and few groups per wave."""
import numpy as np
import pytest

import oracle
from _ringsim import Mirror, check_close

pytestmark = pytest.mark.gpu

SHAPES = ["2,1", "2,2", "4,2", "8,2", "1,2,2", "2,2,2", "4,2,2"]


def _check(gpu, n_batch, heads, kv, d, n_ctx, positions, fused, what):
    m = Mirror(gpu, 1, n_batch, kv, d, n_ctx)
    for s in range(n_batch):
        m.fill_range(0, s, 0, positions[s] + (0 if fused else 1), seed=40 + 2 * s)
    q, k, v = (oracle.normal(7 + i, n_batch * h * d).reshape(n_batch, h, d) for i, h in enumerate((heads, kv, kv)))
    out = gpu.full(q.shape, float("nan"), device="cuda")
    pos = gpu.tensor(positions, dtype=gpu.int32, device="cuda")
    if fused:
        m.ring.append_decode(0, pos, m.dev(q), m.dev(k), m.dev(v), out, heads, stream=m.stream)
        for s in range(n_batch):
            m.oracle_append(0, s, positions[s], k[s], v[s])
    else:
        m.ring.decode(0, pos, m.dev(q), out, heads, stream=m.stream)
    gpu.cuda.synchronize()
    got = out.cpu().numpy()
    for s in range(n_batch):
        check_close(got[s], m.oracle_decode(0, s, positions[s], q[s], heads), f"{what} entry {s}")
    for s in range(0, n_batch, max(1, n_batch // 8)):
        m.assert_ring_equal(0, s)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("n_batch,heads,n_ctx", [
    (127, 1, 40), (2, 64, 40), (2, 128, 40), (257, 1, 40), (3, 256, 40), (769, 1, 40),      # 127 | 128, 256 | 257, 768 | 769
    (3, 512, 40), (1537, 1, 33), (8, 256, 40), (683, 3, 40),     # 1536 | 1537, 2048 | 2049 units
    (4, 512, 1024), (9, 228, 1024),                              # 2048 | 2052 units of 32 groups
    (2, 4, 2016), (2, 4, 2048), (2, 80, 2016), (2, 80, 2048),    # 63 | 64 groups, few units
    (2, 512, 2048), (2, 512, 2080),                              # 64 | 65 groups, 1024 units
])
def test_default_shapes(gpu, n_batch, heads, n_ctx, fused):
    """One kv head, head_dim 64 (32 slots a group), entries with full and
    partly filled windows."""
    pos = [(n_ctx + 5 * s) if s % 3 else (7 * s) % n_ctx for s in range(n_batch)]
    _check(gpu, n_batch, heads, 1, 64, n_ctx, pos, fused, f"{n_batch * heads} units, {n_ctx} slots")


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("heads,kv", [(8, 4), (12, 3), (16, 2), (12, 2), (9, 3)])
@pytest.mark.parametrize("d,n_ctx,n_batch", [(64, 40, 33), (128, 40, 70), (64, 8, 70), (128, 600, 200),
                                             (64, 500, 200)])
def test_grouped_queries(gpu, heads, kv, d, n_ctx, n_batch, fused):
    """2, 4, 8, 6 and 3 query heads a kv head on both sides of the grouped
    shapes' lines (256, 512 and 1536 units, 32 groups)."""
    pos = [(n_ctx + 5 * s) if s % 3 else (7 * s) % n_ctx for s in range(n_batch)]
    _check(gpu, n_batch, heads, kv, d, n_ctx, pos, fused, f"{heads}/{kv} heads, {n_batch} entries")


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("d,n_ctx,pos", [(128, 512, 700), (128, 512, 20), (128, 3000, 3100), (64, 8, 5),
                                         (128, 100, 95), (64, 200, 450)])
def test_forced_shapes(gpu, monkeypatch, shape, d, n_ctx, pos, fused):
    monkeypatch.setenv("BMO_ATTN_SHAPE", shape)
    _check(gpu, 2, 4, 2, d, n_ctx, [pos, max(0, pos - 19)], fused, f"shape {shape}")
