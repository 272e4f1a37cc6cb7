"""GPU tests of the handle's whole-step calls, which run every layer of a step
in one launch: many layers at the edges of the launch's shapes, and buffers
that overlap, where the layers still run one after another."""
import numpy as np
import pytest

import oracle
from _ringsim import Mirror, check_close
from bmo_jetson_amd import Session

pytestmark = pytest.mark.gpu

THETA = 10000.0


def _step(m, layers, heads, pos, q, k, v):
    """The oracle's step (RoPE), layer by layer."""
    out = []
    for layer in range(layers):
        m.oracle_append(layer, 0, pos, oracle.rope_interleaved(k[layer], pos, THETA), v[layer])
        out.append(m.oracle_decode(layer, 0, pos, oracle.rope_interleaved(q[layer], pos, THETA), heads))
    return np.stack(out)


@pytest.mark.parametrize("layers,heads,kv,d,n_ctx,pos", [
    (1, 1, 1, 64, 8, 0),        # one unit, one key
    (7, 4, 4, 64, 40, 90),      # a ring off the group size
    (19, 32, 8, 128, 72, 71),   # 608 units, a window one short of the ring's end
    (33, 16, 16, 128, 16, 500),
])
def test_step_of_many_layers(gpu, layers, heads, kv, d, n_ctx, pos):
    m = Mirror(gpu, layers, 2, kv, d, n_ctx)
    for layer in range(layers):
        m.fill_range(layer, 0, 0, pos, seed=10 + layer)
    q = oracle.normal(1, layers * heads * d).reshape(layers, heads, d)
    k = oracle.normal(2, layers * kv * d).reshape(layers, kv, d)
    v = oracle.normal(3, layers * kv * d).reshape(layers, kv, d)
    bufs = [m.dev(x) for x in (q, k, v)] + [gpu.full(q.shape, float("nan"), device="cuda")]
    gpu.cuda.synchronize()
    sess = Session(m.ring, 0, heads, rope_theta=THETA)
    sess.capture(*bufs)
    for i in range(3):  # eager, then captured, then a layer at a time
        if i == 0:
            sess.forward(pos, *bufs)
        elif i == 1:
            sess.replay(pos + i)
        else:
            for layer in range(layers):  # at the position the step before left
                sess.layer(layer, *(b[layer] for b in bufs))
            sess.end_step()
            sess.sync()
        assert sess.pos == pos + i + 1
        check_close(bufs[3].cpu().numpy(), _step(m, layers, heads, pos + i, q, k, v), f"step {i}")
    for layer in range(layers):
        m.assert_ring_equal(layer, 0)
        m.assert_ring_equal(layer, 1)
    sess.close()


def test_overlapping_buffers_run_in_layer_order(gpu):
    """out one layer behind q in one buffer: layer l + 1's query is layer l's
    output, as in a step whose layers run one after another."""
    layers, heads, d, n_ctx, pos = 4, 4, 128, 32, 50
    m = Mirror(gpu, layers, 1, heads, d, n_ctx)
    for layer in range(layers):
        m.fill_range(layer, 0, 0, pos, seed=30 + layer)
    rows = gpu.zeros((layers + 1, heads, d), dtype=gpu.float32, device="cuda")
    q0 = oracle.normal(4, heads * d).reshape(heads, d)
    k = oracle.normal(5, layers * heads * d).reshape(layers, heads, d)
    v = oracle.normal(6, layers * heads * d).reshape(layers, heads, d)
    rows[0] = m.dev(q0)
    kd, vd = m.dev(k), m.dev(v)
    gpu.cuda.synchronize()
    sess = Session(m.ring, 0, heads, rope_theta=THETA)
    sess.forward(pos, rows[:layers], kd, vd, rows[1:])
    got = rows.cpu().numpy()
    for layer in range(layers):
        m.oracle_append(layer, 0, pos, oracle.rope_interleaved(k[layer], pos, THETA), v[layer])
        ref = m.oracle_decode(layer, 0, pos, oracle.rope_interleaved(got[layer], pos, THETA), heads)
        check_close(got[layer + 1], ref, f"layer {layer}")
        m.assert_ring_equal(layer, 0)
    sess.close()
