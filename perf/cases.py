"""Performance cases: the calls that programs make of this package, over the sizes they make them at.

Kinds of case (``kind``) and what each stands for:

* ``stream``: one tick of the slot-stream engine (``SlotStreamEngine.step_packed``) on live sessions with full
  attention windows. One session receiving one token is the smallest call and a latency; 352 sessions with the mixed
  chunk sizes of ``MixedServingLoad`` are the serving load the package is built for.
* ``context``: new sessions sent their initial contexts (``reset`` of their slots, then ``step``, which cuts them into
  64-token ticks).
* ``score``: a complete message scored in one forward (``WholeSequenceScorer.forward``): a chat turn, a document.
* ``gdn_step`` / ``gdn_prefill``: one gated-delta layer's state update, token by token for decode ticks
  (``gdn_slot_v8``) and in chunks for contexts (``gdn_chunk_prefill``).
* ``ring_decode`` / ``ring_tick``: one attention layer over the slots' 512-token rings, for one new token a slot (with
  the ring write) and for chunks of up to 64 (``ring_attention_v8``).
* ``mlp_glue`` / ``qk_rope``: the element-wise ops around the products, composed from the kernel-contract functions as
  an engine built on them does: residual add, RMSNorm and SiLU-mul; per-head norms and rotary embedding of q and k.

Whole calls run the full 24 layers or (``layers`` 4) one period of the hybrid stack, three gated-delta layers and one
attention layer. Geometries: 16 query / 4 kv heads and the released 8 / 2 (``q_heads``).
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hs-guard_amd"))

from hs_guard.engine import kernels  # noqa: E402
from hs_guard.engine.slot_engine import ROLES, SlotStreamEngine  # noqa: E402
from hs_guard.engine.whole import WholeSequenceScorer  # noqa: E402
from hs_guard.model import GuardConfig, GuardModel  # noqa: E402

BF16, F32, F64, I64 = torch.bfloat16, torch.float32, torch.float64, torch.long
DEV = "cuda"
HEADS, KD = 16, 128            # gated-delta heads and their key / value width
HD, W = 256, 512               # attention head width and window
HID, MLP, ROT = 1024, 3584, 64
EPS = 1e-6
STD = 0.0025                   # weight scale at which 24 random layers do not amplify a rounding into the outputs


def listed():
    return [
        # one live session, one token: the latency a single chat sees
        {"name": "stream_1", "kind": "stream", "rows": 1, "slots": 16, "mixed": False, "layers": 24, "q_heads": 16,
         "state": "float32"},
        # the serving load: 352 sessions, chunks of 1 (p 0.8), 2-16 (0.15) and 17-64 (0.05) tokens
        {"name": "stream_mixed_352", "kind": "stream", "rows": 352, "slots": 352, "mixed": True, "layers": 24,
         "q_heads": 16, "state": "float32"},
        # three sessions join with contexts of ~900 tokens
        {"name": "context_3x900", "kind": "context", "rows": 3, "tokens": 900, "layers": 4, "q_heads": 16},
        # an ordinary chat turn, and a long document, scored at once
        {"name": "score_311", "kind": "score", "tokens": 311, "layers": 4, "q_heads": 8},
        {"name": "score_8000", "kind": "score", "tokens": 8000, "layers": 4, "q_heads": 16},
        # a gated-delta layer's decode step: a few sessions (launch and latency), and a full engine (memory)
        {"name": "gdn_step_16", "kind": "gdn_step", "rows": 16, "length": 1, "state": "float32"},
        {"name": "gdn_step_352", "kind": "gdn_step", "rows": 352, "length": 1, "state": "float32"},
        # a gated-delta layer over 16 initial contexts of 512, 2048 and 8000 tokens
        {"name": "gdn_prefill_16x8000", "kind": "gdn_prefill", "rows": 16, "longest": 8000, "state": "float32"},
        # an attention layer's decode step of 64 sessions, rings partly filled
        {"name": "ring_decode_64", "kind": "ring_decode", "rows": 64, "q_heads": 16},
        # an attention layer for the multi-token rows of a mixed tick
        {"name": "ring_tick_72", "kind": "ring_tick", "rows": 72, "length": 64, "q_heads": 16},
        # the element-wise ops around one layer's products, at the token count of a mixed tick
        {"name": "mlp_glue_1473", "kind": "mlp_glue", "tokens": 1473},
        {"name": "qk_rope_1473", "kind": "qk_rope", "rows": 491, "length": 3, "q_heads": 16},
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["stream", "context", "score", "gdn_step", "gdn_prefill", "ring_decode", "ring_tick", "mlp_glue",
                       "qk_rope"])
    q_heads, state = rng.choice([16, 8]), rng.choice(["float32", "float16"])
    if kind == "stream":
        rows = spread(1, 352)
        return {"kind": kind, "rows": rows, "slots": max(rows, 4), "mixed": rng.random() < 0.6, "layers": 4,
                "q_heads": q_heads, "state": state}
    if kind == "context":
        return {"kind": kind, "rows": rng.randint(1, 8), "tokens": spread(40, 1600), "layers": 4, "q_heads": q_heads}
    if kind == "score":
        return {"kind": kind, "tokens": spread(20, 8000), "layers": 4, "q_heads": q_heads}
    if kind == "gdn_step":
        return {"kind": kind, "rows": spread(1, 352), "length": rng.choice([1, 1, 2, 5, 16]), "state": state}
    if kind == "gdn_prefill":
        return {"kind": kind, "rows": rng.randint(1, 16), "longest": spread(64, 8000), "state": state}
    if kind == "ring_decode":
        return {"kind": kind, "rows": spread(1, 352), "q_heads": q_heads}
    if kind == "ring_tick":
        return {"kind": kind, "rows": spread(1, 96), "length": spread(2, 64), "q_heads": q_heads}
    if kind == "mlp_glue":
        return {"kind": kind, "tokens": spread(1, 8000)}
    return {"kind": kind, "rows": spread(1, 1000), "length": rng.randint(1, 8), "q_heads": q_heads}


# ---------------------------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, scale=1.0, dtype=BF16):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


def _lens(case, seed):
    """The rows' lengths: one multiset a case (so every seed is the same work), in the seed's order."""
    kind, rows = case["kind"], case["rows"]
    rng = random.Random("%s %d" % (kind, rows))
    if kind == "stream":
        def size():
            u = rng.random()
            return 1 if u < 0.8 else rng.randint(2, 16) if u < 0.95 else rng.randint(17, 64)
        lens = [size() if case["mixed"] else 1 for _ in range(rows)]
    elif kind == "context":
        lens = [max(1, round(case["tokens"] * rng.uniform(0.9, 1.1))) for _ in range(rows)]
    elif kind == "gdn_step":
        lens = [case["length"] if n == 0 else rng.randint(1, case["length"]) for n in range(rows)]
    elif kind == "gdn_prefill":
        full = case["longest"]
        cycle = (8000, 512, 2048)
        lens = [max(1, full * cycle[n % 3] // 8000) for n in range(rows)]
    elif kind == "ring_tick":
        top = case["length"]
        lens = [top if n == 0 else min(top, rng.randint(2, 16) if rng.random() < 0.75 else rng.randint(17, 64))
                for n in range(rows)]
    else:
        lens = [1] * rows
    if kind != "context":           # its outputs come row by row: their shapes stay the case's
        random.Random(int(seed)).shuffle(lens)
    return lens


def _decay(g, heads):
    """A_log and dt_bias as gated-delta layers are initialised: A in [1, 16], time steps in [1e-3, 1e-1]."""
    a_log = torch.log(torch.rand(heads, generator=g, device=DEV) * 15 + 1)
    dt = torch.exp(torch.rand(heads, generator=g, device=DEV) * (math.log(0.1) - math.log(0.001)) + math.log(0.001))
    return a_log.to(BF16), torch.log(torch.expm1(dt)).to(BF16)


def _gdn_inputs(case, seed):
    g = _gen(seed)
    lens = _lens(case, seed)
    n = case["rows"]
    dtype = torch.float32 if case["state"] == "float32" else torch.float16
    lens_d = torch.tensor(lens, dtype=I64, device=DEV)
    if case["kind"] == "gdn_step":
        shape = (n, case["length"])
    else:
        shape = (sum(lens),)
    # the layer's conv ends in SiLU: q, k, v are SiLU outputs
    packed = torch.nn.functional.silu(_randn(g, *shape, 3 * HEADS * KD, dtype=F32)).to(BF16)
    a_log, dt_bias = _decay(g, HEADS)
    return {"packed": packed, "a": _randn(g, *shape, HEADS), "b": _randn(g, *shape, HEADS), "A_log": a_log,
            "dt_bias": dt_bias, "lens": lens_d, "offsets": torch.cumsum(lens_d, 0) - lens_d,
            "slots": torch.randperm(n, generator=g, device=DEV),
            "pool": _randn(g, n + 1, HEADS, KD, KD, scale=0.02, dtype=dtype)}


def _ring_positions(starts):
    """ring_pos [N, W + 1] of rings whose next position is starts [N]: column c holds the last p < start, p = c mod W."""
    c = torch.arange(W, device=DEV)[None]
    p = starts[:, None] - W + torch.remainder(c - starts[:, None], W)
    pos = torch.full((len(starts), W + 1), -1, dtype=I64, device=DEV)
    pos[:, :W] = torch.where(p >= 0, p, torch.full_like(p, -1))
    return pos


def _ring_inputs(case, seed):
    g = _gen(seed)
    n, hq = case["rows"], case["q_heads"]
    hkv = hq // 4
    lens = _lens(case, seed)
    lb = case.get("length", 1)
    # one row in four is in its first window, the others past it
    starts = torch.randint(1, 8000, (n,), generator=g, device=DEV)
    starts = torch.where(torch.rand(n, generator=g, device=DEV) < 0.25, starts % W, starts + W)
    slots = torch.randperm(n, generator=g, device=DEV)
    ring_pos = torch.full((n + 1, W + 1), -1, dtype=I64, device=DEV)
    ring_pos[slots] = _ring_positions(starts)
    return {"q": _randn(g, n, hkv, 4 * lb, HD), "ring_k": _randn(g, n + 1, hkv, W + 1, HD),
            "ring_v": _randn(g, n + 1, hkv, W + 1, HD), "new_k": _randn(g, n, hkv, lb, HD),
            "value": _randn(g, n, lb, hkv * HD), "gate": _randn(g, n, lb, hq * 2 * HD), "ring_pos": ring_pos,
            "slots": slots, "starts": starts, "lens": torch.tensor(lens, dtype=I64, device=DEV)}


def _model(case):
    make = GuardConfig.baseline if case["q_heads"] == 16 else GuardConfig.v10
    cfg = make(num_hidden_layers=case["layers"])
    model = GuardModel.random(cfg, seed=1, device=DEV, std=STD, gen_device=DEV)
    g = _gen(2)
    for name in sorted(model.weights):
        if name.endswith("A_log"):
            model.weights[name], model.weights[name[:-len("A_log")] + "dt_bias"] = _decay(g, HEADS)
    return model


def _sessions(case, seed, cfg):
    """(slot, snapshot) of every live session, in slot order: as a stream of `start` tokens has left it."""
    g = _gen(seed)
    n_att = cfg.layer_types.count("full_attention")
    n_gdn = len(cfg.layer_types) - n_att
    hkv = cfg.num_key_value_heads
    starts = torch.randint(W, 8000, (case["rows"],), generator=g, device=DEV)
    ring_pos = _ring_positions(starts)
    for s, start in enumerate(starts.tolist()):
        yield s, {"rec": _randn(g, n_gdn, HEADS, KD, KD, scale=0.02, dtype=F32),
                  "conv": _randn(g, n_gdn, 3, cfg.conv_dim, scale=0.08),
                  "ring_k": _randn(g, n_att, hkv, W + 1, HD), "ring_v": _randn(g, n_att, hkv, W + 1, HD, scale=0.08),
                  "ring_pos": ring_pos[s], "length": start}


def _ids(lens, seed, vocab):
    rng = np.random.default_rng(int(seed))
    return [rng.integers(0, vocab, k).tolist() for k in lens]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("gdn_step", "gdn_prefill"):
        s = _gdn_inputs(case, seed)
        if kind == "gdn_prefill":
            from hs_guard._lib import lib
            bytes_ = lib().hsg_gdn_chunk_workspace_bytes(case["rows"], case["longest"], HEADS)
            s["workspace"] = torch.empty(max(int(bytes_), 256), dtype=torch.uint8, device=DEV)
    elif kind in ("ring_decode", "ring_tick"):
        s = _ring_inputs(case, seed)
    elif kind == "mlp_glue":
        g, t = _gen(seed), case["tokens"]
        s = {"hidden": _randn(g, t, HID), "mix": _randn(g, t, HID), "w1": 1 + _randn(g, HID, scale=0.02, dtype=F32),
             "gate": _randn(g, t, MLP), "up": _randn(g, t, MLP)}
    elif kind == "qk_rope":
        g, n, lb, hq = _gen(seed), case["rows"], case["length"], case["q_heads"]
        pos = torch.randint(0, 8000, (n, 1), generator=g, device=DEV) + torch.arange(lb, device=DEV)[None]
        inv = 1.0 / 10000.0 ** (torch.arange(0, ROT, 2, dtype=F64, device=DEV) / ROT)
        ang = (pos[..., None] * inv).repeat(1, 1, 2)
        s = {"q": _randn(g, n, lb, hq * 2 * HD), "k": _randn(g, n, lb, hq // 4 * HD), "cos": ang.cos().to(BF16),
             "sin": ang.sin().to(BF16), "q_w1": 1 + _randn(g, HD, scale=0.02, dtype=F32),
             "k_w1": 1 + _randn(g, HD, scale=0.02, dtype=F32)}
    else:
        model = _model(case)
        vocab = model.config.vocab_size
        if kind == "score":
            s = {"scorer": WholeSequenceScorer(model), "ids": _ids([case["tokens"]], seed, vocab)[0]}
            s["scorer"].forward(s["ids"][:64])
        else:
            lens = _lens(case, seed)
            requests = list(enumerate(_ids(lens, seed, vocab)))
            eng = SlotStreamEngine(model, case.get("slots", case["rows"]), state_dtype=case.get("state", "float32"))
            if kind == "stream":
                for slot, snap in _sessions(case, seed, model.config):
                    eng.restore(slot, snap)
                eng.prepare(case["rows"], [sum(lens)])
            else:
                eng.step(requests)      # captures the ticks' graphs, as a server's warm-up does
            s = {"engine": eng, "requests": requests}
    s["case"] = case
    return s


# ---------------------------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "stream":
        eng = s["engine"]
        probs, _ = eng.step_packed(s["requests"])
        return {"probs": probs, "rec": eng.rec, "conv": eng.conv, "ring_k": eng.ring_k, "ring_v": eng.ring_v,
                "ring_pos": eng.ring_pos}
    if kind == "context":
        eng = s["engine"]
        eng.reset([slot for slot, _ in s["requests"]])
        probs = eng.step(s["requests"])
        return {"probs": probs, "rec": eng.rec, "conv": eng.conv, "ring_k": eng.ring_k, "ring_v": eng.ring_v,
                "ring_pos": eng.ring_pos}
    if kind == "score":
        return s["scorer"].forward(s["ids"])
    if kind == "gdn_step":
        o, sq = kernels.gdn_slot_v8(s["packed"], HEADS * KD, HEADS, KD, HEADS, KD, s["a"], s["b"], s["A_log"],
                                    s["dt_bias"], s["pool"], s["slots"], s["lens"])
        return {"o": o, "sq": sq, "state": s["pool"]}
    if kind == "gdn_prefill":
        o, _ = kernels.gdn_chunk_prefill(s["packed"], HEADS * KD, HEADS, KD, HEADS, KD, s["a"], s["b"], s["A_log"],
                                         s["dt_bias"], s["pool"], s["slots"], s["lens"], offsets=s["offsets"],
                                         max_len=case["longest"], workspace=s["workspace"])
        return {"o": o, "state": s["pool"]}
    if kind in ("ring_decode", "ring_tick"):
        out = kernels.ring_attention_v8(s["q"], s["ring_k"], s["ring_v"], s["new_k"], s["value"], s["gate"],
                                        s["ring_pos"], s["slots"], s["starts"], s["lens"], HD ** -0.5, W,
                                        kind == "ring_decode")
        return {"out": out, "ring_k": s["ring_k"], "ring_v": s["ring_v"]} if kind == "ring_decode" else out
    if kind == "mlp_glue":
        hidden, sq = kernels.add_square(s["hidden"], s["mix"])
        normed = kernels.rms_finish(hidden, sq.mean(-1, keepdim=True), s["w1"], EPS)
        return {"hidden": hidden, "normed": normed, "act": kernels.silu_mul(s["gate"], s["up"])}
    n, lb, hq = case["rows"], case["length"], case["q_heads"]
    hkv = hq // 4
    var = kernels.square_rows(s["q"], n * lb, hq, hq * 2 * HD, 2 * HD, HD).mean(-1)
    q = kernels.norm_rope(s["q"], var.reshape(-1), s["q_w1"], s["cos"], s["sin"], EPS, n, lb, hq, 4, hq * 2 * HD,
                          2 * HD, HD)
    var = kernels.square_rows(s["k"], n * lb, hkv, hkv * HD, HD, HD).mean(-1)
    k = kernels.norm_rope(s["k"], var.reshape(-1), s["k_w1"], s["cos"], s["sin"], EPS, n, lb, hkv, 1, hkv * HD, HD, HD)
    return {"q": q, "k": k}


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------
def _network_work(case, tokens, rows, ring_keys):
    """Bytes and flops of `tokens` tokens through the layers, `rows` sessions' state and `ring_keys` ring keys apart."""
    hq, layers = case["q_heads"], case["layers"]
    n_att = layers // 4
    n_gdn = layers - n_att
    gdn_w = HID * (3 * HEADS * KD + HEADS * KD + 2 * HEADS) + HEADS * KD * HID
    att_w = HID * (hq * 2 * HD + hq // 4 * 2 * HD) + hq * HD * HID
    weights = n_gdn * gdn_w + n_att * att_w + layers * 3 * HID * MLP + 2 * 512 * HID
    state = 4 if case.get("state", "float32") == "float32" else 2
    bytes_ = 2 * weights + tokens * (2 * HID + 8 + 24)
    bytes_ += rows * n_gdn * (2 * state * HEADS * KD * KD + 2 * 2 * 3 * 3 * HEADS * KD)
    bytes_ += n_att * hq // 4 * HD * 2 * 2 * (ring_keys + tokens * (rows > 0))
    flops = 2 * weights * tokens + n_gdn * tokens * HEADS * 6 * KD * KD + n_att * tokens * hq * 4 * HD * min(W, max(tokens, W))
    return {"bytes": bytes_, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "stream":
        return _network_work(case, sum(_lens(case, 0)), case["rows"], case["rows"] * W)
    if kind == "context":
        return _network_work(case, sum(_lens(case, 0)), case["rows"], 0)
    if kind == "score":
        return _network_work(case, case["tokens"], 0, 0)
    if kind in ("gdn_step", "gdn_prefill"):
        tokens, n = sum(_lens(case, 0)), case["rows"]
        state = 4 if case["state"] == "float32" else 2
        out = n * case["length"] * 6 if kind == "gdn_step" else tokens * 2
        return {"bytes": n * HEADS * 2 * state * KD * KD + tokens * HEADS * (6 * KD + 4) + out * HEADS * KD,
                "flops": tokens * HEADS * 6 * KD * KD}
    if kind in ("ring_decode", "ring_tick"):
        n, hq = case["rows"], case["q_heads"]
        lens = _lens(case, 0)
        keys = n * W * 7 // 8        # one row in four holds half a window on average
        lb = case.get("length", 1)
        bytes_ = (keys * 2 + sum(lens) * 2) * (hq // 4) * HD * 2 + n * W * 8
        bytes_ += (sum(lens) * 2 + n * lb) * hq * HD * 2
        bytes_ += 2 * n * (hq // 4) * HD * 2 if kind == "ring_decode" else 0
        return {"bytes": bytes_, "flops": sum(k * (W * 7 // 8 + k // 2 + 1) for k in lens) * hq * 4 * HD}
    if kind == "mlp_glue":
        return {"bytes": case["tokens"] * (4 * HID * 2 + 3 * MLP * 2), "flops": case["tokens"] * (6 * HID + 6 * MLP)}
    heads = case["q_heads"] * 5 // 4
    tokens = case["rows"] * case["length"]
    return {"bytes": tokens * (heads * HD * 2 * 2 + 2 * ROT * 2), "flops": tokens * heads * HD * 6}


def tolerance(case):
    """About four times the error against 64 bits: bf16 outputs of single layers 2e-3 to 3.6e-3 (the squares of bf16
    values); the probabilities of a scored message 2e-4; of engine ticks the bf16 conv histories, which carry the
    roundings of all layers before, 3e-3 over 4 layers and 9e-3 over 24."""
    kind = case["kind"]
    if kind == "score":
        return {"rel": 0.001}
    if kind in ("stream", "context") and case["layers"] > 4:
        return {"rel": 0.03}
    return {"rel": 0.012}


# ---------------------------------------------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------------------------------------------
def _recurrence(qkv, a, b, a_log, dt_bias, state, lens):
    """qkv [N, L, 3 * HEADS * KD], a, b [N, L, HEADS], state [N, HEADS, KD, KD] (updated), all in 64 bits: outputs
    [N, L, HEADS, KD], zero past a row's length."""
    n, length = qkv.shape[:2]
    order = sorted(range(n), key=lambda r: -lens[r])
    at = torch.tensor(order, device=DEV)
    q, k, v = (x.reshape(n, length, HEADS, KD)[at] for x in qkv.split(HEADS * KD, -1))
    q = q * (q.square().sum(-1, keepdim=True) + 1e-6).rsqrt() * KD ** -0.5
    k = k * (k.square().sum(-1, keepdim=True) + 1e-6).rsqrt()
    decay = torch.exp(-a_log.double().exp() * torch.nn.functional.softplus(a[at] + dt_bias.double()))
    beta = torch.sigmoid(b[at])
    s = state[at]
    out = torch.zeros_like(v)
    for t in range(max(lens)):
        r = sum(1 for x in lens if x > t)
        s_r = s[:r]
        s_r.mul_(decay[:r, t, :, None, None])
        read = torch.matmul(k[:r, t, :, None, :], s_r)
        s_r.add_(k[:r, t, :, :, None] * (beta[:r, t, :, None, None] * (v[:r, t, :, None, :] - read)))
        out[:r, t] = torch.matmul(q[:r, t, :, None, :], s_r)[:, :, 0]
    state[at] = s
    back = torch.empty_like(out)
    back[at] = out
    return back


def _window(q, ring_k, ring_v, ring_pos, new_k, new_v, starts, lens, scale):
    """q [N, hq, L, HD], ring_k / ring_v [N, hkv, W, HD], ring_pos [N, W], new_k / new_v [N, hkv, L, HD]: [N, hq, L, HD],
    zero past a row's length."""
    n, hq, length, _ = q.shape
    steps = torch.arange(length, device=DEV)
    lens_d = torch.tensor(lens, device=DEV)
    qpos = starts[:, None] + steps
    live = steps < lens_d[:, None]
    kpos = torch.cat([ring_pos, torch.where(live, qpos, -1)], 1)
    out = torch.zeros_like(q)
    for r0 in range(0, n, 32):
        r = slice(r0, r0 + 32)
        ok = (kpos[r, None] >= 0) & (kpos[r, None] <= qpos[r, :, None]) & (kpos[r, None] > qpos[r, :, None] - W)
        ok = ok & live[r, :, None]
        for h in range(ring_k.shape[1]):
            keys = torch.cat([ring_k[r, h], new_k[r, h]], 1).double()
            values = torch.cat([ring_v[r, h], new_v[r, h]], 1).double()
            for g in range(hq // ring_k.shape[1]):
                j = h * (hq // ring_k.shape[1]) + g
                p = torch.matmul(q[r, j], keys.transpose(1, 2)) * scale
                p = torch.softmax(p.masked_fill(~ok, -math.inf), -1).nan_to_num(0.0)
                out[r, j] = torch.matmul(p, values)
    return out


def _rms(x, w):
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * (1 + w.double())


def _rope(x, ang):
    c, s = ang.cos(), ang.sin()
    r = x[..., :ROT]
    turned = torch.cat([-r[..., ROT // 2:], r[..., :ROT // 2]], -1)
    return torch.cat([r * c + turned * s, x[..., ROT:]], -1)


def _network(model, ids, lens, starts, pools):
    """The model in 64 bits over rows ids [N, L] (lens valid): probabilities [roles, N, L, 3]. pools: rec, conv, ring_k,
    ring_v [layer, N, ...] of the rows before (updated)."""
    w, cfg = model.weights, model.config
    n, length = ids.shape
    hq, hkv = cfg.num_attention_heads, cfg.num_key_value_heads
    lens_d = torch.tensor(lens, device=DEV)
    steps = torch.arange(length, device=DEV)
    pos = starts[:, None] + steps
    ang = (pos[..., None] * (1.0 / cfg.rope_theta ** (torch.arange(0, ROT, 2, dtype=F64, device=DEV) / ROT)))
    ang = ang.repeat(1, 1, 2)[:, :, None]
    ring_pos = _ring_positions(starts)[:, :W]
    rows = torch.arange(n, device=DEV)[:, None]
    x = w["backbone.embed_tokens.weight"][ids].double()
    done = {"linear_attention": 0, "full_attention": 0}
    for i, kind in enumerate(cfg.layer_types):
        p, idx = "backbone.layers.%d." % i, done[kind]
        done[kind] += 1
        h = _rms(x, w[p + "input_layernorm.weight"])
        if kind == "linear_attention":
            m = {k: w[p + "linear_attn." + k] for k in ("A_log", "dt_bias")}
            m.update({k: w[p + "linear_attn." + k + ".weight"].double()
                      for k in ("in_proj_qkv", "in_proj_z", "in_proj_b", "in_proj_a", "conv1d", "norm", "out_proj")})
            ext = torch.cat([pools["conv"][idx], h @ m["in_proj_qkv"].T], 1)
            conv = sum(ext[:, t:t + length] * m["conv1d"][:, 0, t] for t in range(4))
            pools["conv"][idx] = ext[rows, lens_d[:, None] + torch.arange(3, device=DEV)]
            o = _recurrence(torch.nn.functional.silu(conv), h @ m["in_proj_a"].T, h @ m["in_proj_b"].T, m["A_log"],
                            m["dt_bias"], pools["rec"][idx], lens)
            z = (h @ m["in_proj_z"].T).reshape(o.shape)
            o = o * (o.square().mean(-1, keepdim=True) + EPS).rsqrt() * m["norm"] * torch.nn.functional.silu(z)
            x = x + o.reshape(n, length, -1) @ m["out_proj"].T
        else:
            a = p + "self_attn."
            qg = (h @ w[a + "q_proj.weight"].double().T).reshape(n, length, hq, 2, HD)
            k = (h @ w[a + "k_proj.weight"].double().T).reshape(n, length, hkv, HD)
            v = (h @ w[a + "v_proj.weight"].double().T).reshape(n, length, hkv, HD).transpose(1, 2)
            q = _rope(_rms(qg[:, :, :, 0], w[a + "q_norm.weight"]), ang).transpose(1, 2)
            k = _rope(_rms(k, w[a + "k_norm.weight"]), ang).transpose(1, 2)
            rk, rv = pools["ring_k"][idx], pools["ring_v"][idx]
            o = _window(q, rk[:, :, :W], rv[:, :, :W], ring_pos, k, v, starts, lens, HD ** -0.5)
            o = o.transpose(1, 2) * torch.sigmoid(qg[:, :, :, 1])
            for t in range(length):     # the last W of each row's new keys stay in its ring
                r = torch.nonzero((t < lens_d) & (t >= lens_d - W)).flatten()
                if len(r):
                    rk[r, :, pos[r, t] % W], rv[r, :, pos[r, t] % W] = k[r, :, t], v[r, :, t]
            x = x + o.reshape(n, length, -1) @ w[a + "o_proj.weight"].double().T
        h = _rms(x, w[p + "post_attention_layernorm.weight"])
        h = torch.nn.functional.silu(h @ w[p + "mlp.gate_proj.weight"].double().T) * (
            h @ w[p + "mlp.up_proj.weight"].double().T)
        x = x + h @ w[p + "mlp.down_proj.weight"].double().T
    x = _rms(x, w["backbone.norm.weight"])
    probs = []
    for r in ROLES:
        m = {k: w["heads.%s.%s" % (r, k)].double() for k in (
            "projection.0.weight", "projection.0.bias", "projection.1.weight", "projection.1.bias", "risk.weight",
            "risk.bias")}
        y = x @ m["projection.0.weight"].T + m["projection.0.bias"]
        y = torch.nn.functional.layer_norm(y, y.shape[-1:], m["projection.1.weight"], m["projection.1.bias"],
                                           cfg.layer_norm_eps)
        probs.append(torch.softmax(torch.nn.functional.silu(y) @ m["risk.weight"].T + m["risk.bias"], -1))
    return torch.stack(probs)


def _padded(ids):
    out = torch.zeros(len(ids), max(map(len, ids)), dtype=I64, device=DEV)
    for r, row in enumerate(ids):
        out[r, :len(row)] = torch.tensor(row, device=DEV)
    return out


def _exact_whole(case, seed):
    kind = case["kind"]
    model = _model(case)
    cfg = model.config
    n_att = cfg.layer_types.count("full_attention")
    n_gdn, hkv = len(cfg.layer_types) - n_att, cfg.num_key_value_heads
    lens = [case["tokens"]] if kind == "score" else _lens(case, seed)
    n, slots = len(lens), case.get("slots", len(lens))
    ids = _ids(lens, seed, cfg.vocab_size)
    pools = {"rec": torch.zeros(n_gdn, n, HEADS, KD, KD, dtype=F64, device=DEV),
             "conv": torch.zeros(n_gdn, n, 3, cfg.conv_dim, dtype=F64, device=DEV),
             "ring_k": torch.zeros(n_att, n, hkv, W + 1, HD, dtype=F64, device=DEV)}
    pools["ring_v"] = torch.zeros_like(pools["ring_k"])
    starts = torch.zeros(n, dtype=I64, device=DEV)
    if kind == "stream":
        for slot, snap in _sessions(case, seed, cfg):
            rec = snap["rec"].to(torch.float16) if case["state"] == "float16" else snap["rec"]
            pools["rec"][:, slot] = rec.double()
            for name in ("conv", "ring_k", "ring_v"):
                pools[name][:, slot] = snap[name].double()
            starts[slot] = snap["length"]
    probs = _network(model, _padded(ids), lens, starts, pools)
    if kind == "score":
        return probs[:, 0]
    out = {k: torch.cat([v, torch.zeros_like(v[:, :1]).expand(-1, slots + 1 - n, *v.shape[2:])], 1)
           for k, v in pools.items()}
    if kind == "context":
        out["probs"] = {r: [probs[i, j, :lens[j]] for j in range(n)] for i, r in enumerate(ROLES)}
        return out
    # a single session's tick has six probabilities: too few for the size of their error to say anything
    if sum(lens) < 64:
        out["probs"] = None
        return out
    lb = next(b for b in (1, 2, 4, 8, 16, 32, 64) if b >= max(lens))
    out["probs"] = torch.zeros(len(ROLES), n, lb, 3, dtype=F64, device=DEV)
    for j, k in enumerate(lens):
        out["probs"][:, j, :k] = probs[:, j, :k]
    return out


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind in ("stream", "context", "score"):
        return _exact_whole(case, seed)
    if kind in ("gdn_step", "gdn_prefill"):
        s = _gdn_inputs(case, seed)
        lens, n = _lens(case, seed), case["rows"]
        if kind == "gdn_step":
            packed, a, b = (s[k].double() for k in ("packed", "a", "b"))
        else:
            packed, a, b = (torch.zeros(n, max(lens), s[k].shape[-1], dtype=F64, device=DEV) for k in ("packed", "a", "b"))
            for r, (o, k) in enumerate(zip(s["offsets"].tolist(), lens)):
                for to, name in ((packed, "packed"), (a, "a"), (b, "b")):
                    to[r, :k] = s[name][o:o + k].double()
        state = s["pool"].double()
        live = state[s["slots"]]
        o = _recurrence(packed, a, b, s["A_log"], s["dt_bias"], live, lens)
        state[s["slots"]] = live
        if kind == "gdn_step":
            return {"o": o, "sq": o.square(), "state": state}
        return {"o": torch.cat([o[r, :k] for r, k in enumerate(lens)]), "state": state}
    if kind in ("ring_decode", "ring_tick"):
        s = _ring_inputs(case, seed)
        n, hq, lb = case["rows"], case["q_heads"], case.get("length", 1)
        hkv, at = hq // 4, s["slots"]
        value = s["value"].double().reshape(n, lb, hkv, HD).transpose(1, 2)
        o = _window(s["q"].double().reshape(n, hq, lb, HD), s["ring_k"][at][:, :, :W], s["ring_v"][at][:, :, :W],
                    s["ring_pos"][at][:, :W], s["new_k"], value, s["starts"], _lens(case, seed), HD ** -0.5)
        o = o.transpose(1, 2) * torch.sigmoid(s["gate"].double().reshape(n, lb, hq, 2, HD)[:, :, :, 1])
        o = o.reshape(n, lb, hq * HD)
        if kind == "ring_tick":
            return o
        ring_k, ring_v = s["ring_k"].double(), s["ring_v"].double()
        col = s["starts"] % W
        ring_k[at, :, col], ring_v[at, :, col] = s["new_k"][:, :, 0].double(), value[:, :, 0]
        return {"out": o, "ring_k": ring_k, "ring_v": ring_v}
    s = prepare(case, seed)
    if kind == "mlp_glue":
        h = s["hidden"].double() + s["mix"].double()
        normed = h * (h.square().mean(-1, keepdim=True) + EPS).rsqrt() * s["w1"].double()
        return {"hidden": h, "normed": normed, "act": torch.nn.functional.silu(s["gate"].double()) * s["up"].double()}
    n, lb, hq = case["rows"], case["length"], case["q_heads"]
    hkv = hq // 4

    def turn(x, w1):
        x = x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * w1.double()
        c, sn = s["cos"].double()[:, :, None], s["sin"].double()[:, :, None]
        r = x[..., :ROT]
        r = r * c + torch.cat([-r[..., ROT // 2:], r[..., :ROT // 2]], -1) * sn
        return torch.cat([r, x[..., ROT:]], -1).transpose(1, 2)

    q = turn(s["q"].double().reshape(n, lb, hq, 2, HD)[:, :, :, 0], s["q_w1"])
    k = turn(s["k"].double().reshape(n, lb, hkv, HD), s["k_w1"])
    return {"q": q.reshape(n, hkv, 4 * lb, HD), "k": k}
