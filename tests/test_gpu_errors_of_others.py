"""A HIP error that another call of the program left on the thread (here an
invalid device number, refused on the host).  A handle's call may report it,
and then neither its position nor where the device goes on has moved; the end
of a recording does not fail for it, and a readout neither fails for it nor
takes it from the thread."""
import ctypes

import numpy as np
import pytest

import oracle
from _ringsim import Mirror, check_close
from bmo_jetson_amd import RingError, Session
from bmo_jetson_amd._lib import lib

pytestmark = pytest.mark.gpu

THETA = 10000.0


def _hip():
    lib()  # its libamdhip64, already loaded
    return ctypes.CDLL("libamdhip64.so.7")


def _leave_error():
    error = _hip().hipSetDevice(9999)
    assert error != 0
    return error


@pytest.mark.parametrize("call", ["forward", "replay", "replay graph", "begin_step", "end_step", "reset_async"])
def test_a_failed_call_leaves_the_position(gpu, call):
    layers, heads, d, n_ctx, pos = 3, 4, 64, 40, 25
    m = Mirror(gpu, layers, 1, heads, d, n_ctx)
    for layer in range(layers):
        m.fill_range(layer, 0, 0, pos, seed=110 + layer)
    shape = (layers, heads, d)
    q, k, v = (oracle.normal(120 + i, int(np.prod(shape))).reshape(shape) for i in range(3))
    qd, kd, vd = m.dev(q), m.dev(k), m.dev(v)
    out = gpu.full(shape, float("nan"), device="cuda")
    gpu.cuda.synchronize()
    sess = Session(m.ring, 0, heads, rope_theta=THETA)
    sess.begin_step(pos)
    if call == "replay graph":
        sess.capture_begin()
        for layer in range(layers):
            sess.layer(layer, qd[layer], kd[layer], vd[layer], out[layer])
        sess.end_step()
        sess.capture_end()
    else:
        sess.capture(qd, kd, vd, out)
    _leave_error()
    try:
        {"forward": lambda: sess.forward(pos, qd, kd, vd, out),
         "replay": lambda: sess.replay(pos),
         "replay graph": lambda: sess.replay(pos),
         "begin_step": lambda: sess.begin_step(7),
         "end_step": sess.end_step,
         "reset_async": sess.reset_async}[call]()
    except RingError:
        if call == "reset_async":  # (the ring may be cleared, the position is not)
            for layer in range(layers):
                m.ring.reset(0, stream=m.stream)
                m.orc[(layer, 0)] = oracle.new_ring(heads, n_ctx, d)
            gpu.cuda.synchronize()
        assert sess.pos == pos
    else:
        pytest.skip("the runtime keeps no error of a refused call")
    # the same token again, layer by layer at the device position
    for layer in range(layers):
        sess.layer(layer, qd[layer], kd[layer], vd[layer], out[layer])
    sess.end_step()
    sess.sync()
    assert sess.pos == pos + 1
    for layer in range(layers):
        m.oracle_append(layer, 0, pos, oracle.rope_interleaved(k[layer], pos, THETA), v[layer])
        ref = m.oracle_decode(layer, 0, pos, oracle.rope_interleaved(q[layer], pos, THETA), heads)
        check_close(out[layer].cpu().numpy(), ref, f"{call}, layer {layer}")
        m.assert_ring_equal(layer, 0)
    sess.close()


@pytest.mark.parametrize("reset", [False, True])
def test_a_recording_ends_whatever_others_left(gpu, reset):
    heads, d, n_ctx = 4, 64, 40
    m = Mirror(gpu, 1, 1, heads, d, n_ctx)
    q, k, v = (oracle.normal(140 + i, heads * d).reshape(heads, d) for i in range(3))
    qd, kd, vd = m.dev(q), m.dev(k), m.dev(v)
    out = gpu.full((heads, d), float("nan"), device="cuda")
    gpu.cuda.synchronize()
    sess = Session(m.ring, 0, heads, rope_theta=THETA)
    sess.capture_begin()
    if reset:
        sess.reset_async()
    sess.layer(0, qd, kd, vd, out)
    sess.end_step()
    _leave_error()
    sess.capture_end()
    assert sess.has_graph
    _hip().hipGetLastError()
    sess.replay(0)
    m.oracle_append(0, 0, 0, oracle.rope_interleaved(k, 0, THETA), v)
    check_close(out.cpu().numpy(), m.oracle_decode(0, 0, 0, oracle.rope_interleaved(q, 0, THETA), heads))
    assert sess.pos == 1
    sess.close()


@pytest.mark.parametrize("n", [5, 40])
def test_readouts_keep_to_their_own_errors(gpu, n):
    kv, d, n_ctx = 3, 128, 40
    m = Mirror(gpu, 1, 2, kv, d, n_ctx)
    for s in range(2):
        m.fill_range(0, s, 0, n_ctx, seed=130 + s)
    gpu.cuda.synchronize()
    error = _leave_error()
    blocks = [m.ring.export_q4_0(0, 0, which, 0, n) for which in (0, 1)]
    k = m.ring.get_k_cache_f32(0, 0, n)
    for which in (0, 1):
        m.ring.import_q4_0(0, 1, which, 0, blocks[which])
        assert np.array_equal(m.ring.export_q4_0(0, 1, which, 0, n), blocks[which])
        want = m.orc[(0, 0)][which].transpose(1, 0, 2)[:n]
        assert np.array_equal(blocks[which].reshape(-1), np.ascontiguousarray(want).view(np.uint8).reshape(-1))
    assert np.array_equal(k, m.ring.get_k_cache_f32(0, 0, n, session=1))
    assert _hip().hipGetLastError() in (error, 0)  # (0: a runtime that forgets it at the next good call)
