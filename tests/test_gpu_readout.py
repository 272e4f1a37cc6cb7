"""Readout and import of ring slots as ggml blocks at the sizes where the kernels
that move them can go wrong: block counts around a workgroup's 256, more
blocks than the pinned buffer holds at once, slot ranges inside a group, both
head dims.  Exports equal the oracle's blocks byte for byte, fp32 K its
dequantized values, and an import changes the named slots and nothing else."""
import numpy as np
import pytest

import oracle
from _ringsim import Mirror

pytestmark = pytest.mark.gpu


def _blocks(m, layer, session, which):
    """The oracle's blocks of a session's K or V, [slot][head][block][18]."""
    c = m.orc[(layer, session)][which]
    return np.ascontiguousarray(c.transpose(1, 0, 2)).view(np.uint8).reshape(m.n_ctx, m.n_kv, m.d // 32, 18)


@pytest.mark.parametrize("kv,d,n_ctx,t0,n", [
    (1, 64, 8, 0, 1),          # 2 blocks
    (2, 128, 40, 3, 31),       # 248 blocks, within and across groups
    (2, 128, 40, 4, 32),       # 256
    (1, 128, 80, 9, 65),       # 260
    (3, 64, 70, 33, 37),       # 222 of 32-slot groups
    (32, 128, 1100, 50, 1000),  # 128000 blocks: the buffer twice
])
def test_export_import_ranges(gpu, kv, d, n_ctx, t0, n):
    m = Mirror(gpu, 2, 2, kv, d, n_ctx)
    for s in (0, 1):
        m.fill_range(1, s, 0, n_ctx + 5, seed=60 + s)
    for which in (0, 1):
        want = _blocks(m, 1, 0, which)
        got = m.ring.export_q4_0(1, 0, which, t0, n)
        assert np.array_equal(got, want[t0:t0 + n])
        m.ring.import_q4_0(1, 1, which, t0, got)
        after = _blocks(m, 1, 1, which).copy()
        after[t0:t0 + n] = got
        assert np.array_equal(m.ring.export_q4_0(1, 1, which, 0, n_ctx), after)
        assert np.array_equal(m.ring.export_q4_0(1, 0, which, 0, n_ctx), want)
    k = m.ring.get_k_cache_f32(1, t0, n)
    ref = oracle.dequantize_q4_0(_blocks(m, 1, 0, 0)[t0:t0 + n].reshape(-1, 18).copy().view(oracle.BLOCK_DTYPE).reshape(-1))
    assert np.array_equal(k.reshape(-1).view(np.uint32), np.asarray(ref, np.float32).reshape(-1).view(np.uint32))
