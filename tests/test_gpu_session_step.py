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


@pytest.mark.parametrize("layers,heads,kv,d,n_ctx,pos,rope", [
    (20, 32, 32, 128, 128, 300, True),   # runs of few groups
    (64, 32, 32, 128, 512, 700, True),   # 2048 units in the launch
    (32, 32, 8, 128, 512, 90, False),    # grouped queries, a partly filled window
    (8, 16, 16, 64, 8, 40, True),        # one group
    (6, 16, 4, 64, 200, 450, True),
    (2, 32, 32, 128, 1100, 2300, False),  # 69 groups
    (3, 160, 32, 64, 300, 900, True),    # 160 units a layer: four waves
    (2, 520, 4, 64, 300, 900, True),     # 520: grouped
])
def test_a_step_is_its_layers_bit_for_bit(gpu, layers, heads, kv, d, n_ctx, pos, rope):
    """The layers of a step in one launch give each output, rounding included,
    as the layer's call by itself."""
    m = Mirror(gpu, layers, 1, kv, d, n_ctx)
    g = gpu.Generator(device="cuda")
    g.manual_seed(5)
    n = min(pos, n_ctx)
    for layer in range(layers):
        rows = gpu.randn(2, n, kv, d, generator=g, device="cuda")
        m.ring.write(layer, 0, pos - n, rows[0], rows[1], n_tok=n, stream=m.stream)
    q, k, v = (gpu.randn(layers, h, d, generator=g, device="cuda") for h in (heads, kv, kv))
    out = gpu.full(q.shape, float("nan"), device="cuda")
    gpu.cuda.synchronize()
    sess = Session(m.ring, 0, heads, rope_theta=THETA if rope else 0.0)
    sess.begin_step(pos)
    for layer in range(layers):
        sess.layer(layer, q[layer], k[layer], v[layer], out[layer])
    sess.end_step()
    sess.sync()
    want = out.cpu().numpy().view(np.uint32)
    sess.capture(q, k, v, out)
    for step in (lambda: sess.forward(pos, q, k, v, out), lambda: sess.replay(pos)):
        out.fill_(float("nan"))
        gpu.cuda.synchronize()
        step()
        assert np.array_equal(out.cpu().numpy().view(np.uint32), want)
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


@pytest.mark.parametrize("resets", ["first", "between", "never"])
def test_captured_steps_take_their_positions(gpu, resets):
    """A recorded graph of five steps, with a reset before them, after the
    second or not at all: each step's layers attend and rotate at the position
    that the replay's beginning and the steps before them give, and the device
    position is where an eager step then goes on."""
    layers, heads, d, n_ctx, steps = 2, 4, 64, 20, 5
    m = Mirror(gpu, layers, 2, heads, d, n_ctx)
    for layer in range(layers):
        m.fill_range(layer, 1, 0, 30, seed=70 + layer)
    shape = (steps + 1, layers, heads, d)
    q, k, v = (oracle.normal(80 + i, int(np.prod(shape))).reshape(shape) for i in range(3))
    qd, kd, vd = m.dev(q), m.dev(k), m.dev(v)
    out = gpu.full(shape, float("nan"), device="cuda")
    gpu.cuda.synchronize()
    sess = Session(m.ring, 1, heads, rope_theta=THETA)
    reset_at = {"first": 0, "between": 2, "never": None}[resets]
    sess.capture_begin()
    for t in range(steps):
        if t == reset_at:
            sess.reset_async()
        for layer in range(layers):
            sess.layer(layer, qd[t, layer], kd[t, layer], vd[t, layer], out[t, layer])
        sess.end_step()
    sess.capture_end()

    def step(t, pos):
        for layer in range(layers):
            m.oracle_append(layer, 1, pos, oracle.rope_interleaved(k[t, layer], pos, THETA), v[t, layer])
            ref = m.oracle_decode(layer, 1, pos, oracle.rope_interleaved(q[t, layer], pos, THETA), heads)
            check_close(out[t, layer].cpu().numpy(), ref, f"step {t} at {pos}, layer {layer}")

    for start in (30, 41):
        # a graph with a reset takes no position: its steps before the reset
        # are at the handle's
        pos = start if resets == "never" else sess.pos
        sess.replay(start)
        for t in range(steps):
            if t == reset_at:
                for layer in range(layers):
                    m.orc[(layer, 1)] = oracle.new_ring(heads, n_ctx, d)
                pos = 0
            step(t, pos)
            pos += 1
        assert sess.pos == pos
        for layer in range(layers):  # at the device position the graph left
            sess.layer(layer, qd[steps, layer], kd[steps, layer], vd[steps, layer], out[steps, layer])
        sess.end_step()
        sess.sync()
        step(steps, pos)
        assert sess.pos == pos + 1
    for layer in range(layers):
        m.assert_ring_equal(layer, 0)
        m.assert_ring_equal(layer, 1)
    sess.close()


def test_the_latest_capture_is_what_replay_runs(gpu):
    """A captured step and a recorded graph replace each other, either way
    round; a failed recording replaces nothing."""
    layers, heads, d, n_ctx = 2, 4, 64, 20
    m = Mirror(gpu, layers, 1, heads, d, n_ctx)
    shape = (2, layers, heads, d)
    q, k, v = (oracle.normal(90 + i, int(np.prod(shape))).reshape(shape) for i in range(3))
    qd, kd, vd = m.dev(q), m.dev(k), m.dev(v)
    out = gpu.full(shape, float("nan"), device="cuda")
    gpu.cuda.synchronize()
    sess = Session(m.ring, 0, heads, rope_theta=THETA)

    def record(t):
        sess.capture_begin()
        for layer in range(layers):
            sess.layer(layer, qd[t, layer], kd[t, layer], vd[t, layer], out[t, layer])
        sess.end_step()
        sess.capture_end()

    def fail_to_record():
        sess.capture_begin()
        with pytest.raises(RuntimeError):
            sess.layer(layers, qd[0, 0], kd[0, 0], vd[0, 0], out[0, 0])
        with pytest.raises(RuntimeError):
            sess.capture_end()

    pos = 0
    for t, take in [(0, lambda: sess.capture(qd[0], kd[0], vd[0], out[0])),
                    (0, fail_to_record),
                    (1, lambda: record(1)),
                    (1, fail_to_record),
                    (0, lambda: sess.capture(qd[0], kd[0], vd[0], out[0]))]:
        take()
        assert sess.has_graph
        out.fill_(float("nan"))
        gpu.cuda.synchronize()
        sess.replay(pos)
        check_close(out[t].cpu().numpy(), _step(m, layers, heads, pos, q[t], k[t], v[t]), f"replay at {pos}")
        assert gpu.isnan(out[1 - t]).all()
        pos += 1
        assert sess.pos == pos
    for layer in range(layers):
        m.assert_ring_equal(layer, 0)
    sess.close()
