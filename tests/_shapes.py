"""Test helper: the workgroup shapes of decode and staged prefill calls, from the
rules that the library is compiled with (bmo_jetson_amd/csrc/decode_shape.hpp
and prefill_shape.hpp)."""
import os
import subprocess

BUILD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "build")


def _ask(program, lines):
    exe = os.path.join(BUILD, program)
    assert os.path.exists(exe), f"tests/build/{program} is not built (run __graft_entry__.build())"
    res = subprocess.run([exe], input="".join(l + "\n" for l in lines), capture_output=True, text=True,
                         timeout=60, check=True)
    out = [tuple(map(int, line.split())) for line in res.stdout.splitlines()]
    assert len(out) == len(lines)
    return out


def decode_shapes(calls, forced="-"):
    """(waves per unit, groups in flight, heads per workgroup, threads) of each
    (units, layers, groups, query heads per kv head, fused), with the shape
    that BMO_ATTN_SHAPE forces."""
    return _ask("decode_shape_check",
                ["%d %d %d %d %d %s" % (u, layers, n, per, bool(f), forced) for u, layers, n, per, f in calls])


def staged_shapes(calls):
    """(units in full rounds of 16 waves x 16 queries, waves per workgroup and
    per block of queries of the rest) of each (units, tokens, slots)."""
    return _ask("prefill_shape_check", ["%d %d %d" % c for c in calls])
