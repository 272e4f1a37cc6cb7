"""Waves per unit and groups in flight of the decode kernel against the float64
oracle (|gpu - ref| <= 2e-3 + 1e-3 |ref|): the default rule near both sides of
each of its lines (tests/test_decode_shapes.py has the lines themselves), and
the shapes that it chooses, forced, at runs of no, one and few groups per
wave."""
import numpy as np
import pytest

import oracle
from _ringsim import Mirror, check_close
from _shapes import decode_shapes

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


# (entries, heads, slots), one kv head, head_dim 64 (32 slots a group): the shapes
# (waves per unit, groups in flight, heads per workgroup) of the plain and the
# fused call.  Neighbouring rows are the two sides of a line.
DEFAULT = [
    # heads odd: one head a workgroup
    (1, 127, 288, (8, 2, 1), (8, 1, 1)), (3, 43, 288, (4, 2, 1), (4, 2, 1)),         # 127 | 129 units
    (5, 51, 2048, (8, 2, 1), (8, 2, 1)), (1, 257, 2048, (4, 2, 1), (4, 2, 1)),       # 255 | 257 of 64 groups
    (5, 51, 2016, (4, 2, 1), (4, 2, 1)),                                             # ... 63 groups
    (3, 3, 2016, (8, 2, 1), (8, 1, 1)), (3, 3, 2048, (8, 2, 1), (8, 2, 1)),          # 63 | 64 groups, few units
    (13, 59, 288, (2, 2, 1), (2, 2, 1)), (1, 769, 288, (1, 2, 1), (2, 2, 1)),        # 767 | 769
    (5, 307, 288, (1, 2, 1), (2, 2, 1)), (29, 53, 288, (1, 2, 1), (1, 2, 1)),        # 1535 | 1537
    (3, 341, 2048, (1, 2, 1), (2, 2, 1)), (3, 341, 2080, (1, 2, 1), (1, 2, 1)),      # 64 | 65 groups, 1023 units
    (2, 1023, 1024, (1, 2, 1), (1, 2, 1)), (3, 683, 1024, (4, 2, 1), (1, 2, 1)),     # 2046 | 2049 of 32 groups
    (3, 683, 992, (1, 2, 1), (1, 2, 1)),                                             # ... 31 groups
    (1, 255, 32, (1, 1, 1), (2, 1, 1)), (1, 257, 32, (1, 1, 1), (1, 1, 1)),          # 255 | 257 of 1 group
    (1, 127, 64, (2, 1, 1), (2, 1, 1)),                                              # fewer groups than waves
    (7, 73, 96, (2, 1, 1), (2, 1, 1)), (512, 1, 96, (2, 1, 1), (1, 2, 1)),           # 511 | 512 of 3 groups
    (512, 1, 128, (4, 1, 1), (4, 2, 1)), (3, 171, 96, (2, 2, 1), (1, 2, 1)),         # 512 of 4 | 513 of 3
    (3, 171, 256, (1, 2, 1), (1, 2, 1)), (3, 171, 288, (2, 2, 1), (2, 2, 1)),        # 513 units, 8 | 9 groups
    (3, 171, 352, (2, 2, 1), (1, 2, 1)),                                             # ... 11
    (3, 171, 416, (2, 2, 1), (2, 2, 1)), (3, 171, 448, (2, 2, 1), (4, 2, 1)),        # ... 13 | 14
    (3, 171, 992, (2, 2, 1), (4, 2, 1)), (3, 171, 1024, (4, 2, 1), (4, 2, 1)),       # ... 31 | 32
    (3, 341, 64, (1, 2, 1), (1, 2, 1)), (3, 341, 96, (1, 2, 1), (2, 2, 1)),          # 2 | 3 groups, 1023 units
    # heads even: grouped
    (4, 64, 288, (4, 2, 1), (4, 2, 1)), (3, 86, 288, (4, 2, 2), (4, 2, 2)),          # 256 | 258 units
    (4, 128, 288, (4, 2, 2), (4, 2, 2)), (2, 258, 288, (2, 2, 2), (2, 2, 2)),        # 512 | 516
    (3, 512, 288, (2, 2, 2), (2, 2, 2)), (4, 388, 288, (1, 2, 4), (1, 2, 4)),        # 1536 | 1552, four heads
    (4, 386, 992, (1, 2, 2), (1, 2, 2)), (4, 386, 1024, (2, 2, 2), (2, 2, 2)),       # 31 | 32 groups, two heads
    (4, 128, 32, (1, 1, 1), (1, 1, 1)), (4, 128, 64, (2, 2, 2), (2, 2, 2)),          # 1 | 2 groups
    (3, 172, 64, (1, 2, 1), (1, 2, 1)), (4, 388, 64, (1, 2, 4), (1, 2, 4)),          # 2 groups, 516 | 1552
]


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("n_batch,heads,n_ctx,plain_shape,fused_shape", DEFAULT)
def test_default_shapes(gpu, n_batch, heads, n_ctx, plain_shape, fused_shape, fused):
    """Entries with full and partly filled windows; the shape is the one named."""
    units = n_batch * heads
    (shape,) = decode_shapes([(units, 1, (n_ctx + 31) // 32, heads, fused)])
    assert shape[:3] == (fused_shape if fused else plain_shape)
    pos = [(n_ctx + 5 * s) if s % 3 != 1 else (7 * s) % n_ctx for s in range(n_batch)]
    _check(gpu, n_batch, heads, 1, 64, n_ctx, pos, fused, f"{units} units, {n_ctx} slots")


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("heads,kv", [(8, 4), (12, 3), (16, 2), (12, 2), (9, 3)])
@pytest.mark.parametrize("d,n_ctx,n_batch", [(64, 40, 33), (128, 40, 70), (64, 8, 70), (128, 600, 200),
                                             (64, 500, 200)])
def test_grouped_queries(gpu, heads, kv, d, n_ctx, n_batch, fused):
    """2, 4, 8, 6 and 3 query heads a kv head, both head dims, several kv heads."""
    pos = [(n_ctx + 5 * s) if s % 3 else (7 * s) % n_ctx for s in range(n_batch)]
    _check(gpu, n_batch, heads, kv, d, n_ctx, pos, fused, f"{heads}/{kv} heads, {n_batch} entries")


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("d,n_ctx,pos", [(128, 512, 700), (128, 3000, 3100), (64, 8, 5), (64, 200, 450)])
def test_forced_four_heads(gpu, monkeypatch, d, n_ctx, pos, fused):
    monkeypatch.setenv("BMO_ATTN_SHAPE", "1,2,4")
    _check(gpu, 2, 8, 2, d, n_ctx, [pos, max(0, pos - 19)], fused, "shape 1,2,4")


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("d,n_ctx,pos", [(128, 512, 700), (128, 512, 20), (128, 3000, 3100), (64, 8, 5),
                                         (128, 100, 95), (64, 200, 450)])
def test_forced_shapes(gpu, monkeypatch, shape, d, n_ctx, pos, fused):
    monkeypatch.setenv("BMO_ATTN_SHAPE", shape)
    _check(gpu, 2, 4, 2, d, n_ctx, [pos, max(0, pos - 19)], fused, f"shape {shape}")
