"""Test helper: the decode calls' workgroup shapes, from the rule that the
library is compiled with (bmo_jetson_amd/csrc/decode_shape.hpp)."""
import os
import subprocess

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "build", "decode_shape_check")


def decode_shapes(calls, forced="-"):
    """(waves per unit, groups in flight, heads per workgroup, threads) of each
    (units, layers, groups, query heads per kv head, fused), with the shape
    that BMO_ATTN_SHAPE forces."""
    assert os.path.exists(EXE), "tests/build/decode_shape_check is not built (run __graft_entry__.build())"
    text = "".join("%d %d %d %d %d %s\n" % (u, layers, n, per, bool(f), forced) for u, layers, n, per, f in calls)
    res = subprocess.run([EXE], input=text, capture_output=True, text=True, timeout=60, check=True)
    out = [tuple(map(int, line.split())) for line in res.stdout.splitlines()]
    assert len(out) == len(calls)
    return out
