"""The work that users of this library have it do, as cases to be timed and
compared: each kind of call over the range of sizes it is used at.

A case names its kind (`kind`) and its sizes:

  step      one token of one session through every layer, replayed from the
            session handle's captured graph (fused append + attention, RoPE
            or not): the single-user voice loop
  frame     the depformer's frame from a handle's captured graph: a reset,
            then `steps` positions through every layer of a small ring
  layers    a model's layer loop on a handle, captured: QKV projection,
            RoPE + append + attention, output projection, layer after layer
  append    one token of many sessions through `layers` layers, the calls
            captured in a HIP graph that ends by advancing the positions: a
            server's token step
  decode    the same without the append (the token is in the ring already)
  prefill   a chunk of a prompt for several sessions, one layer
  project   the Q4_0 projections of a layer or a head, one after another,
            captured in a graph (a projection never runs alone in a model)
  snapshot  a session's ring read out as ggml blocks and written back into
            another session: a session that moves or is kept

Every ring holds as much history as the position says, K and V ~N(0, 1) with
one element in a hundred 8 times as large, and every run returns the outputs
with the ring's bytes (or, in `snapshot`, the blocks that were read).
"""
import math

import numpy as np
import torch

from bmo_jetson_amd import KVRing, Session, gemv_q4_0_q8_1, positions_advance

THETA = 10000.0


def listed():
    return [
        # one user's token through the 32-layer temporal stack, 512-slot ring
        {"name": "step", "kind": "step", "layers": 32, "heads": 32, "kv": 32, "dim": 128, "ctx": 512,
         "pos": 700, "rope": True},
        # the same at the model's native context of 3000 positions
        {"name": "step, long context", "kind": "step", "layers": 32, "heads": 32, "kv": 32, "dim": 128,
         "ctx": 3000, "pos": 4100, "rope": True},
        # the depformer: 8 codebook steps through 6 layers after a reset; the
        # smallest calls there are
        {"name": "depformer frame", "kind": "frame", "layers": 6, "heads": 16, "kv": 16, "dim": 64, "ctx": 8,
         "steps": 8},
        # projections and attention of four temporal layers, one token
        {"name": "layers with projections", "kind": "layers", "layers": 4, "heads": 32, "dim": 128, "ctx": 512,
         "pos": 1500},
        # a server's step with a dozen sessions
        {"name": "append, 12 sessions", "kind": "append", "sessions": 12, "layers": 16, "heads": 32, "kv": 32,
         "dim": 128, "ctx": 512, "rope": True},
        # and with 256 sessions, the largest
        {"name": "append, 256 sessions", "kind": "append", "sessions": 256, "layers": 2, "heads": 32, "kv": 32,
         "dim": 128, "ctx": 512, "rope": True},
        # attention alone over 64 sessions, the headline workload
        {"name": "decode, 64 sessions", "kind": "decode", "sessions": 64, "layers": 4, "heads": 32, "kv": 32,
         "dim": 128, "ctx": 512},
        # grouped queries: 4 query heads read each kv head
        {"name": "decode, grouped queries", "kind": "decode", "sessions": 40, "layers": 4, "heads": 32, "kv": 8,
         "dim": 128, "ctx": 1024},
        # a 256-token chunk of 16 prompts into rings with a full history
        {"name": "prefill", "kind": "prefill", "sessions": 16, "tokens": 256, "heads": 32, "kv": 32, "dim": 128,
         "ctx": 512, "pos": 1024},
        # a longer chunk, grouped queries, ragged sizes
        {"name": "prefill, long chunk", "kind": "prefill", "sessions": 5, "tokens": 500, "heads": 32, "kv": 8,
         "dim": 128, "ctx": 1000, "pos": 611},
        # QKV, output and both gating projections of a temporal layer, twice,
        # and the text head
        {"name": "projections", "kind": "project", "rows": "12288 4096 11264 4096 12288 4096 11264 4096 32000",
         "cols": "4096 4096 4096 5632 4096 4096 4096 5632 4096"},
        # two layers of a session's 512-slot ring out and back in
        {"name": "snapshot", "kind": "snapshot", "layers": 2, "kv": 32, "dim": 128, "ctx": 512, "pos": 900},
    ]


def _log_int(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng):
    """(query heads, kv heads): mostly one query head per kv head."""
    kv = rng.choice([4, 8, 12, 16, 20, 24, 32])
    per = rng.choice([1, 1, 1, 2, 4, 8])
    while kv * per > 32:
        per //= 2
    return kv * max(1, per), kv


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        # no more than the largest listed cases (and not a case of nothing)
        if w["bytes"] <= 1.0e9 and w["flops"] <= 3.0e10:
            return c


def _draw(rng):
    kind = rng.choice(["step", "step", "frame", "layers", "append", "append", "decode", "decode", "prefill",
                       "prefill", "project", "snapshot"])
    heads, kv = _heads(rng)
    dim = rng.choice([64, 128, 128])
    if kind == "step":
        ctx = _log_int(rng, 100, 4096)
        return {"kind": kind, "layers": rng.randint(4, 32), "heads": heads, "kv": kv, "dim": dim, "ctx": ctx,
                "pos": _log_int(rng, 8, 4 * ctx), "rope": rng.random() < 0.7}
    if kind == "frame":
        steps = rng.randint(4, 32)
        return {"kind": kind, "layers": rng.randint(2, 8), "heads": heads, "kv": kv, "dim": 64,
                "ctx": rng.randint(steps, 32), "steps": steps}
    if kind == "layers":
        return {"kind": kind, "layers": rng.randint(1, 4), "heads": rng.choice([8, 16, 20, 24, 32, 40]), "dim": 128,
                "ctx": _log_int(rng, 128, 3000), "pos": _log_int(rng, 16, 6000)}
    if kind in ("append", "decode"):
        c = {"kind": kind, "sessions": _log_int(rng, 2, 256), "layers": rng.randint(2, 16), "heads": heads,
             "kv": kv, "dim": dim, "ctx": _log_int(rng, 128, 3000)}
        if kind == "append":
            c["rope"] = rng.random() < 0.6
        return c
    if kind == "prefill":
        ctx = rng.choice([256, 512, 512, 768, 1000, 1024, 2048, 3000])
        return {"kind": kind, "sessions": _log_int(rng, 1, 24), "tokens": min(ctx, _log_int(rng, 16, 600)),
                "heads": heads, "kv": kv, "dim": dim, "ctx": ctx, "pos": rng.choice([0, rng.randint(1, 3 * ctx)])}
    if kind == "project":
        n = rng.randint(2, 6)
        cols = [rng.choice([64, 256, 512]) * rng.randint(1, 32) for _ in range(n)]
        rows = [_log_int(rng, 64, 32768) for _ in range(n)]
        return {"kind": kind, "rows": " ".join(map(str, rows)), "cols": " ".join(map(str, cols))}
    return {"kind": kind, "layers": 1, "kv": rng.choice([4, 8, 16, 32]), "dim": dim, "ctx": _log_int(rng, 64, 1024),
            "pos": _log_int(rng, 8, 4000)}


# ---- what the cases share --------------------------------------------------


class _Memory:
    """A ring's allocation as torch sees it, without a copy."""

    def __init__(self, ring):
        self.ring = ring  # the memory is the ring's
        self.__cuda_array_interface__ = {"shape": (ring.nbytes,), "typestr": "|u1",
                                         "data": (ring.k_base, False), "version": 2}


def _bytes_of(ring):
    t = torch.as_tensor(_Memory(ring), device="cuda")
    t.ring = ring  # an output can outlive its state
    return t


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed & (2**62 - 1))
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _kv(g, *shape):
    """K or V rows: N(0, 1), one element in a hundred 8 times as large."""
    x = torch.randn(*shape, generator=g, device="cuda")
    return torch.where(torch.rand(*shape, generator=g, device="cuda") < 0.01, x * 8, x)


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def _positions(c, seed):
    """A batch's positions: most sessions past a full window, some younger."""
    r = np.random.default_rng([seed, 3])
    pos = r.integers(c["ctx"], 8 * c["ctx"], c["sessions"])
    young = r.random(c["sessions"]) < 0.125
    return [int(p) for p in np.where(young, r.integers(c["ctx"] // 8, c["ctx"], c["sessions"]), pos)]


def _expected_window(c):
    """A batch's mean window: 7 in 8 are full, the others uniform from ctx / 8."""
    return c["ctx"] * (0.875 + 0.125 * 0.5625)


def _history(c, layer, session, end, seed):
    """K and V of the positions lo .. end - 1 that the ring still holds, in
    one layer of one session: (lo, k, v), [end - lo][kv][dim]."""
    lo = max(0, end - c["ctx"])
    g = _generator(seed * 1000003 + layer * 4099 + session * 17 + 1)
    return lo, _kv(g, end - lo, c["kv"], c["dim"]), _kv(g, end - lo, c["kv"], c["dim"])


def _fill(ring, c, ends, seed):
    """Writes the history before position ends[s] into every layer."""
    for layer in range(ring.n_layers):
        for s, end in enumerate(ends):
            if end > 0:
                lo, k, v = _history(c, layer, s, end, seed)
                ring.write(layer, s, lo, k, v, stream=torch.cuda.current_stream())


def _graph(calls):
    """The calls, captured."""
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        calls(torch.cuda.current_stream())
    torch.cuda.current_stream().wait_stream(side)
    return graph


def _q4_0_weights(g, rows, cols):
    """A ggml Q4_0 matrix: random codes, scales of weights of variance 1 / cols."""
    blocks = torch.randint(0, 256, (rows * cols // 32, 18), generator=g, dtype=torch.uint8, device="cuda")
    d = (torch.rand(rows * cols // 32, generator=g, device="cuda") + 0.5) * (0.21 / math.sqrt(cols))
    blocks[:, :2] = d.to(torch.float16).view(torch.uint8).view(-1, 2)
    return blocks


def _shapes(c):
    return list(zip(map(int, c["rows"].split()), map(int, c["cols"].split())))


# ---- prepare ---------------------------------------------------------------


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _qkv(c, seed, *lead):
    g = _generator(seed * 7 + 5)
    q = _normal(g, *lead, c["heads"], c["dim"])
    return q, _kv(g, *lead, c["kv"], c["dim"]), _kv(g, *lead, c["kv"], c["dim"])


def _prepare_step(c, seed):
    ring = KVRing(c["layers"], 1, c["kv"], c["dim"], c["ctx"])
    _fill(ring, c, [c["pos"]], seed)
    q, k, v = _qkv(c, seed, c["layers"])
    out = torch.zeros_like(q)
    torch.cuda.synchronize()  # the handle has a stream of its own
    s = Session(ring, 0, c["heads"], rope_theta=THETA if c["rope"] else 0.0)
    s.capture(q, k, v, out)
    return {"kind": "step", "ring": ring, "session": s, "pos": c["pos"], "keep": (q, k, v), "out": out,
            "bytes": _bytes_of(ring)}


def _prepare_frame(c, seed):
    ring = KVRing(c["layers"], 1, c["kv"], c["dim"], c["ctx"])
    q, k, v = _qkv(c, seed, c["steps"], c["layers"])
    out = torch.zeros_like(q)
    torch.cuda.synchronize()
    s = Session(ring, 0, c["heads"])
    s.capture_begin()
    s.reset_async()
    for t in range(c["steps"]):
        for layer in range(c["layers"]):
            s.layer(layer, q[t, layer], k[t, layer], v[t, layer], out[t, layer])
        s.end_step()
    s.capture_end()
    return {"kind": "frame", "ring": ring, "session": s, "keep": (q, k, v), "out": out, "bytes": _bytes_of(ring)}


def _model(c, seed):
    """The weights and the input row of `layers`."""
    e = c["heads"] * c["dim"]
    g = _generator(seed * 11 + 2)
    w = [(_q4_0_weights(g, 3 * e, e), _q4_0_weights(g, e, e)) for _ in range(c["layers"])]
    return e, w, _normal(g, e)


def _prepare_layers(c, seed):
    c = dict(c, kv=c["heads"])
    ring = KVRing(c["layers"], 1, c["kv"], c["dim"], c["ctx"])
    _fill(ring, c, [c["pos"]], seed)
    e, w, x = _model(c, seed)
    qkv = torch.zeros(c["layers"], 3 * e, device="cuda")
    att = torch.zeros(c["layers"], e, device="cuda")
    y = torch.zeros(c["layers"], e, device="cuda")
    torch.cuda.synchronize()
    s = Session(ring, 0, c["heads"], rope_theta=THETA)
    s.capture_begin()
    for n, (wi, wo) in enumerate(w):
        gemv_q4_0_q8_1(wi, x if n == 0 else y[n - 1], qkv[n], 3 * e, e, stream=s.stream)
        s.layer(n, qkv[n, :e], qkv[n, e:2 * e], qkv[n, 2 * e:], att[n])
        gemv_q4_0_q8_1(wo, att[n], y[n], e, e, stream=s.stream)
    s.end_step()
    s.capture_end()
    return {"kind": "layers", "ring": ring, "session": s, "pos": c["pos"], "keep": (w, x), "qkv": qkv, "att": att,
            "y": y, "bytes": _bytes_of(ring)}


def _prepare_append(c, seed):
    ring = KVRing(c["layers"], c["sessions"], c["kv"], c["dim"], c["ctx"])
    ends = _positions(c, seed)
    _fill(ring, c, ends, seed)
    q, k, v = _qkv(c, seed, c["layers"], c["sessions"])
    out = torch.zeros_like(q)
    pos = _i32(ends)

    def step(stream):
        for n in range(c["layers"]):
            ring.append_decode(n, pos, q[n], k[n], v[n], out[n], c["heads"], stream=stream,
                               rope_theta=THETA if c["rope"] else None)
        positions_advance(pos, c["sessions"], 1, stream=stream)

    return {"kind": "append", "ring": ring, "graph": _graph(step), "keep": (q, k, v), "pos": pos, "out": out,
            "bytes": _bytes_of(ring)}


def _prepare_decode(c, seed):
    ring = KVRing(c["layers"], c["sessions"], c["kv"], c["dim"], c["ctx"])
    ends = _positions(c, seed)
    _fill(ring, c, ends, seed)
    q, _, _ = _qkv(c, seed, c["layers"], c["sessions"])
    out = torch.zeros_like(q)
    pos = _i32([e - 1 for e in ends])

    def step(stream):
        for n in range(c["layers"]):
            ring.decode(n, pos, q[n], out[n], c["heads"], stream=stream)

    return {"kind": "decode", "ring": ring, "graph": _graph(step), "keep": (q, pos), "out": out}


def _prepare_prefill(c, seed):
    ring = KVRing(1, c["sessions"], c["kv"], c["dim"], c["ctx"])
    _fill(ring, c, [c["pos"]] * c["sessions"], seed)
    q, k, v = (x.to(torch.bfloat16) for x in _qkv(c, seed, c["sessions"], c["tokens"]))
    return {"kind": "prefill", "ring": ring, "qkv": (q, k, v), "pos": _i32([c["pos"]] * c["sessions"]),
            "heads": c["heads"], "out": torch.zeros(q.shape, device="cuda"), "bytes": _bytes_of(ring)}


def _prepare_project(c, seed):
    g = _generator(seed * 13 + 4)
    w = [_q4_0_weights(g, r, n) for r, n in _shapes(c)]
    x = [_kv(g, n) for _, n in _shapes(c)]
    y = [torch.zeros(r, device="cuda") for r, _ in _shapes(c)]

    def layer(stream):
        for i, (r, n) in enumerate(_shapes(c)):
            gemv_q4_0_q8_1(w[i], x[i], y[i], r, n, stream=stream)

    return {"kind": "project", "graph": _graph(layer), "keep": (w, x), "y": y}


def _prepare_snapshot(c, seed):
    ring = KVRing(c["layers"], 2, c["kv"], c["dim"], c["ctx"])
    _fill(ring, c, [c["pos"]], seed)
    return {"kind": "snapshot", "ring": ring, "slots": min(c["pos"], c["ctx"]), "bytes": _bytes_of(ring)}


# ---- run -------------------------------------------------------------------


def run(state):
    return globals()["_run_" + state["kind"]](state)


def _run_step(s):
    s["session"].replay(s["pos"])
    s["pos"] += 1
    return {"out": s["out"], "ring": s["bytes"]}


def _run_frame(s):
    s["session"].replay(0)
    return {"out": s["out"], "ring": s["bytes"]}


def _run_layers(s):
    s["session"].replay(s["pos"])
    s["pos"] += 1
    return {"qkv": s["qkv"], "att": s["att"], "y": s["y"], "ring": s["bytes"]}


def _run_append(s):
    s["graph"].replay()
    return {"out": s["out"], "pos": s["pos"], "ring": s["bytes"]}


def _run_decode(s):
    s["graph"].replay()
    return {"out": s["out"]}


def _run_prefill(s):
    s["ring"].prefill(0, s["pos"], *s["qkv"], s["out"], s["heads"], stream=torch.cuda.current_stream())
    return {"out": s["out"], "ring": s["bytes"]}


def _run_project(s):
    s["graph"].replay()
    return s["y"]


def _run_snapshot(s):
    ring, n, blocks = s["ring"], s["slots"], []
    for layer in range(ring.n_layers):
        for which in (0, 1):
            blocks.append(ring.export_q4_0(layer, 0, which, 0, n))
            ring.import_q4_0(layer, 1, which, 0, blocks[-1])
    return {"blocks": blocks, "ring": s["bytes"]}


# ---- work ------------------------------------------------------------------


def _attention(units_q, units_kv, window, dim, fused):
    """Bytes and operations of decode attention: the windows' Q4_0 K and V, q
    and out in 32 bits; fused, the new rows and their blocks."""
    row = dim // 32 * 18
    b = 2 * units_kv * window * row + 8 * units_q * dim
    if fused:
        b += 2 * units_kv * (4 * dim + row)
    return b, 4 * units_q * window * dim


def work(c):
    kind = c["kind"]
    if kind in ("step", "layers"):
        kv = c.get("kv", c["heads"])
        b, f = _attention(c["heads"], kv, min(c["pos"] + 1, c["ctx"]), c["dim"], True)
        b, f = b * c["layers"], f * c["layers"]
        if kind == "layers":
            e = c["heads"] * c["dim"]
            b += c["layers"] * (4 * e * e * 18 // 32 + 4 * (e + 3 * e + e + e))
            f += c["layers"] * 8 * e * e
    elif kind == "frame":
        b = f = 0
        for t in range(c["steps"]):
            x = _attention(c["heads"], c["kv"], t + 1, c["dim"], True)
            b, f = b + c["layers"] * x[0], f + c["layers"] * x[1]
    elif kind in ("append", "decode"):
        b, f = _attention(c["heads"], c["kv"], _expected_window(c), c["dim"], kind == "append")
        b, f = b * c["sessions"] * c["layers"], f * c["sessions"] * c["layers"]
    elif kind == "prefill":
        keys = sum(min(c["pos"] + i + 1, c["ctx"]) for i in range(c["tokens"]))
        f = 4 * c["dim"] * keys * c["heads"] * c["sessions"]
        row = c["dim"] // 32 * 18
        old = min(c["pos"], c["ctx"] - 1)
        b = c["sessions"] * (c["tokens"] * c["dim"] * (6 * c["heads"] + 4 * c["kv"])
                             + 2 * c["kv"] * row * (old + c["tokens"]))
    elif kind == "project":
        b = sum(r * n // 32 * 18 + 4 * (r + n) for r, n in _shapes(c))
        f = sum(2 * r * n for r, n in _shapes(c))
    else:
        b = 4 * c["layers"] * 2 * min(c["pos"], c["ctx"]) * c["kv"] * (c["dim"] // 32) * 18
        f = 0
    return {"bytes": float(b), "flops": float(f)}


# ---- how far off another implementation may be -----------------------------


def tolerance(case):
    """About four times what the paths show against `exact`: 32-bit sums give
    8e-8 (projections) to 8e-7, prefill's 16-bit weights and V values 2e-4.
    In `layers` a rounding can move an activation's 8-bit code, or a 4-bit
    code of K or V, by one (2.4e-3 seen)."""
    kind = case["kind"]
    if kind == "snapshot":
        return "exact"
    if kind == "project":
        return {"rel": 1e-6}
    if kind == "prefill":
        return {"rel": 8e-4}
    if kind == "layers":
        return {"rel": 1e-2, "max": 0.2, "differ": 1e-4}
    return {"rel": 4e-6}


# ---- in 64 bits ------------------------------------------------------------


def _q4_0(x):
    """The values that x (last axis whole blocks of 32) has as Q4_0, in 64
    bits: ggml's steps, each rounded to 32 bits on its own."""
    b = x.reshape(-1, 32)
    at = b.abs().max(dim=1, keepdim=True)
    first = (b.abs() == at.values).to(torch.uint8).argmax(dim=1, keepdim=True)
    d = b.gather(1, first) / -8.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    code = torch.clamp((b * inv + 8.5).to(torch.int32), max=15)
    return ((code - 8).double() * d.to(torch.float16).double()).reshape(x.shape)


def _rope(x, pos):
    """Pairs (2i, 2i + 1) of the last axis turned by pos THETA^(-2i / dim):
    the angle in 64 bits, the products in 32 as the ring receives them."""
    dim = x.shape[-1]
    f = torch.pow(torch.tensor(THETA, dtype=torch.float64, device=x.device),
                  -2.0 * torch.arange(dim // 2, device=x.device, dtype=torch.float64) / dim)
    a = torch.as_tensor(pos, dtype=torch.float64, device=x.device)[..., None, None] * f
    c, s = a.cos().float(), a.sin().float()
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack((u * c - v * s, u * s + v * c), dim=-1).reshape(x.shape)


def _attend(q, k, v, hide=None):
    """softmax(q k / sqrt(dim)) v in 64 bits: q [tokens][heads][dim], k and v
    [keys][kv][dim]; hide [tokens][keys]: keys that a token does not see."""
    n, heads, dim = q.shape
    keys, kv = k.shape[:2]
    q = q.double().reshape(n, kv, heads // kv, dim).permute(1, 2, 0, 3).reshape(kv, heads // kv * n, dim)
    s = torch.matmul(q, k.permute(1, 2, 0).contiguous()) / math.sqrt(dim)
    if hide is not None:
        s = s.reshape(kv, heads // kv, n, keys).masked_fill(hide, -math.inf).reshape(s.shape)
    o = torch.matmul(torch.softmax(s, dim=-1), v.permute(1, 0, 2).contiguous())
    return o.reshape(kv, heads // kv, n, dim).permute(2, 0, 1, 3).reshape(n, heads, dim)


def _token(c, layer, session, end, seed, q, k, v):
    """One token's attention at position `end`, its own K and V with it."""
    _, hk, hv = _history(c, layer, session, end, seed)
    hk, hv = torch.cat((hk, k[None]))[-c["ctx"]:], torch.cat((hv, v[None]))[-c["ctx"]:]
    return _attend(q[None], _q4_0(hk), _q4_0(hv))[0]


def _project(w, x, rows, cols):
    """W x with x as the library's Q8_1: codes and scales as defined there in
    32 and 16 bits, the products in 64."""
    b = x.float().reshape(-1, 32)
    d = b.abs().amax(dim=1) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    p = b * inv[:, None]
    t = p.trunc()
    code = torch.where((p - t).abs() >= 0.5, t + torch.copysign(torch.ones_like(p), p), t).clamp(-128, 127)
    total = torch.zeros_like(d)
    for j in range(32):
        total = total + b[:, j]
    d8, s8 = d.to(torch.float16).double(), total.to(torch.float16).double()
    out = []
    step = max(1, (1 << 27) // cols)
    blocks = w.reshape(rows, cols // 32, 18)
    for r in range(0, rows, step):
        part = blocks[r:r + step]
        d4 = part[:, :, :2].contiguous().view(torch.float16)[:, :, 0].double()
        qs = part[:, :, 2:]
        c = torch.cat((qs & 15, qs >> 4), dim=2).double()
        out.append((d4 * ((c * code.double()).sum(dim=2) * d8 - 8.0 * s8)).sum(dim=1))
    return torch.cat(out)


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


def _exact_step(c, seed):
    q, k, v = _qkv(c, seed, c["layers"])
    if c["rope"]:
        q, k = _rope(q, float(c["pos"])), _rope(k, float(c["pos"]))
    out = [_token(c, n, 0, c["pos"], seed, q[n], k[n], v[n]) for n in range(c["layers"])]
    return {"out": torch.stack(out), "ring": None}


def _exact_frame(c, seed):
    q, k, v = _qkv(c, seed, c["steps"], c["layers"])
    out = [[_attend(q[t, n][None], _q4_0(k[:t + 1, n]), _q4_0(v[:t + 1, n]))[0] for n in range(c["layers"])]
           for t in range(c["steps"])]
    return {"out": torch.stack([torch.stack(o) for o in out]), "ring": None}


def _exact_layers(c, seed):
    c = dict(c, kv=c["heads"])
    e, w, x = _model(c, seed)
    qkv, att, y = [], [], []
    for n, (wi, wo) in enumerate(w):
        qkv.append(_project(wi, x, 3 * e, e))
        q, k, v = (t.reshape(c["heads"], c["dim"]) for t in qkv[-1].float().split(e))
        q, k = _rope(q, float(c["pos"])), _rope(k, float(c["pos"]))
        att.append(_token(c, n, 0, c["pos"], seed, q, k, v).reshape(e))
        y.append(_project(wo, att[-1], e, e))
        x = y[-1]
    return {"qkv": torch.stack(qkv), "att": torch.stack(att), "y": torch.stack(y), "ring": None}


def _exact_append(c, seed):
    ends = _positions(c, seed)
    q, k, v = _qkv(c, seed, c["layers"], c["sessions"])
    if c["rope"]:
        q, k = _rope(q, ends), _rope(k, ends)
    out = [[_token(c, n, s, ends[s], seed, q[n, s], k[n, s], v[n, s]) for s in range(c["sessions"])]
           for n in range(c["layers"])]
    return {"out": torch.stack([torch.stack(o) for o in out]), "pos": None, "ring": None}


def _exact_decode(c, seed):
    ends = _positions(c, seed)
    q, _, _ = _qkv(c, seed, c["layers"], c["sessions"])
    out = []
    for n in range(c["layers"]):
        for s, end in enumerate(ends):
            _, k, v = _history(c, n, s, end, seed)
            out.append(_attend(q[n, s][None], _q4_0(k), _q4_0(v))[0])
    return {"out": torch.stack(out).reshape(q.shape)}


def _exact_prefill(c, seed):
    q, k, v = (x.to(torch.bfloat16).float() for x in _qkv(c, seed, c["sessions"], c["tokens"]))
    out = []
    for s in range(c["sessions"]):
        _, hk, hv = _history(c, 0, s, c["pos"], seed)
        key = torch.arange(hk.shape[0] + c["tokens"], device="cuda")[None, :]
        own = torch.arange(c["tokens"], device="cuda")[:, None] + hk.shape[0]  # a token's own key
        out.append(_attend(q[s], _q4_0(torch.cat((hk, k[s]))), _q4_0(torch.cat((hv, v[s]))),
                           (key > own) | (key <= own - c["ctx"])))
    return {"out": torch.stack(out), "ring": None}


def _exact_project(c, seed):
    g = _generator(seed * 13 + 4)
    w = [_q4_0_weights(g, r, n) for r, n in _shapes(c)]
    x = [_kv(g, n) for _, n in _shapes(c)]
    return [_project(w[i], x[i], r, n) for i, (r, n) in enumerate(_shapes(c))]


def _exact_snapshot(c, seed):
    return None
