"""GPU parity of the whole streaming step (SlotStreamEngine on libhsg.so) against the CPU oracle.

Geometry: the kernels' fixed sizes (hidden 1024, GDN heads 128 wide, attention head_dim 256) with few
layers and heads, GQA in both mixers, and a 32-token window so that ring wraparound, masking of stale
columns and multi-tick appends are all exercised in a few hundred tokens.

Two comparisons:
* Matched GEMMs, on a 2-layer net (one GDN and one attention layer): the oracle's
  projections go through the product the engine runs at its packed shape (hipBLASLt, or the skinny kernel in
  ticks of at most 8 tokens), so they are bitwise the engine's; everything else (conv, recurrence, norms, RoPE, ring attention, heads, bookkeeping) is the CPU
  restatement. Per-token class probabilities (so 1 - p(safe)) within 2e-3 absolute; a planted mistake in
  the oracle (dropped attention gate) must exceed it several times.
* Independent GEMMs (numpy fp32 products), on a 4-layer net: hipBLASLt and the CPU round 0.02% of bf16
  products differently (one ulp, measured), and random-init weights amplify such flips with depth
  (flipping 0.02% of the oracle's own products by one ulp moves its probabilities by 2.6e-3 at 4 layers and
  6.9e-3 at the 24-layer benchmark geometry), so that comparison uses 1e-2.
ring_pos and length are bit-exact in both; the recurrent state within 2e-2 relative end to end (the
kernel alone is held to 1e-3 in test_gdn_gpu.py).
"""
import numpy as np
import pytest
import torch
from parity_helpers import LONG_PIECES, POOL_BARS, long_piece_case, pool_errors
from parity_helpers import matched_gemm as _matched_gemm
from parity_helpers import max_diff as _max_diff

pytestmark = pytest.mark.gpu

PROB_TOL = 2e-3
PROB_TOL_INDEPENDENT = 1e-2


def _cfg():
    from hs_guard.model import GuardConfig
    return GuardConfig(vocab_size=1000, hidden_size=1024, num_hidden_layers=4, intermediate_size=1024,
                       linear_num_key_heads=2, linear_num_value_heads=4, num_attention_heads=8,
                       num_key_value_heads=2, window_tokens=32)


def _schedule(rng, vocab):
    """Ticks as (slot, ids) lists: appends of 1..70 tokens over 4 slots, past the 32-token window."""
    ticks = [[(0, rng.integers(0, vocab, 20).tolist()), (3, rng.integers(0, vocab, 7).tolist())],
             [(3, [5]), (1, rng.integers(0, vocab, 40).tolist()), (0, [7])],
             [(2, rng.integers(0, vocab, 70).tolist())]]
    for _ in range(6):
        ticks.append([(s, rng.integers(0, vocab, int(rng.choice([1, 1, 1, 3, 9]))).tolist()) for s in (0, 1, 3)])
    ticks.append([(1, [1]), (2, rng.integers(0, vocab, 33).tolist())])
    return ticks


@pytest.fixture(scope="module")
def setup():
    from hs_guard.model import GuardModel
    cfg = _cfg()
    model_cpu = GuardModel.random(cfg, seed=0, device="cpu")
    weights = {k: v.float().numpy() for k, v in model_cpu.weights.items()}
    return cfg, model_cpu.to("cuda:0"), weights


@pytest.fixture(scope="module")
def setup2():
    from hs_guard.model import GuardConfig, GuardModel
    cfg = GuardConfig(vocab_size=1000, hidden_size=1024, num_hidden_layers=2,
                      layer_types=["linear_attention", "full_attention"], intermediate_size=1024,
                      linear_num_key_heads=2, linear_num_value_heads=4, num_attention_heads=8,
                      num_key_value_heads=2, window_tokens=32)
    model_cpu = GuardModel.random(cfg, seed=0, device="cpu")
    weights = {k: v.float().numpy() for k, v in model_cpu.weights.items()}
    return cfg, model_cpu.to("cuda:0"), weights


@pytest.fixture(scope="module")
def setup_small():
    """The 2-layer net of setup2 at weight scale N(0, 0.005) and seed 1: here the oracle's own fp32-level noise floor
    is 5e-4 (tests/test_oracle_backbone.py::test_noise_floor_scales_with_weights), so the 2e-3 bar has about four
    times its margin; at setup2's N(0, 0.02) that floor is 2.7-3.0e-3 on other schedules."""
    from hs_guard.model import GuardConfig, GuardModel
    cfg = GuardConfig(vocab_size=1000, hidden_size=1024, num_hidden_layers=2,
                      layer_types=["linear_attention", "full_attention"], intermediate_size=1024,
                      linear_num_key_heads=2, linear_num_value_heads=4, num_attention_heads=8,
                      num_key_value_heads=2, window_tokens=32)
    model_cpu = GuardModel.random(cfg, seed=1, device="cpu", std=0.005)
    weights = {k: v.float().numpy() for k, v in model_cpu.weights.items()}
    return cfg, model_cpu.to("cuda:0"), weights


def _schedule_b(rng, vocab):
    """A second schedule: other slots first, a 64-token row (two window-sized ticks), a 50-token row beside short
    ones, rows of 2-16 tokens across all four slots, and a 40-token row at the end."""
    ticks = [[(1, rng.integers(0, vocab, 50).tolist()), (2, rng.integers(0, vocab, 3).tolist())],
             [(0, rng.integers(0, vocab, 64).tolist())],
             [(3, rng.integers(0, vocab, 12).tolist()), (1, [9]), (2, rng.integers(0, vocab, 33).tolist())]]
    for _ in range(6):
        ticks.append([(s, rng.integers(0, vocab, int(rng.choice([1, 1, 2, 5, 16]))).tolist()) for s in range(4)])
    ticks.append([(0, [3]), (3, rng.integers(0, vocab, 40).tolist())])
    return ticks


@pytest.mark.parametrize("chunk_min_tokens", [0, 2], ids=["slot_step", "chunk_route"])
def test_engine_second_seed_and_schedule(setup_small, chunk_min_tokens):
    """Matched GEMMs at the 2e-3 bar on a second seed, weight scale and schedule, for the slot-step route and the
    chunk route (every row of two or more tokens in a prefill-like tick through hsg_gdn_chunk_prefill_gated)."""
    from hs_guard.engine.slot_engine import SlotStreamEngine
    from oracle.backbone import StreamOracle
    cfg, model, weights = setup_small
    print(f"[engine] seed 1, N(0, 0.005), second schedule, chunk_min_tokens {chunk_min_tokens}", flush=True)
    eng = SlotStreamEngine(model, 4, use_graphs=False, chunk_min_tokens=chunk_min_tokens)
    orc = StreamOracle(weights, cfg, 4)
    gemm = _matched_gemm(eng)
    worst = 0.0
    for t, tick in enumerate(_schedule_b(np.random.default_rng(1), cfg.vocab_size)):
        diff = _max_diff(eng.step(tick), orc.step(tick, gemm=gemm))
        worst = max(worst, diff)
        assert diff <= PROB_TOL, f"tick {t}: prob diff {diff:.2e}"
    print(f"[engine] second schedule worst prob diff {worst:.2e}", flush=True)
    np.testing.assert_array_equal(eng.length, orc.length)
    np.testing.assert_array_equal(eng.ring_pos.cpu().numpy(), orc.ring_pos)
    rec = eng.rec.double().cpu().numpy()
    for s in range(4):
        rel = np.linalg.norm(rec[:, s] - orc.rec[:, s]) / np.linalg.norm(orc.rec[:, s])
        assert rel < 1e-3, f"slot {s} state rel err {rel:.2e}"


@pytest.mark.parametrize("chunk_min_tokens", [0, 2], ids=["slot_step", "chunk_route"])
def test_engine_fp16_state_matches_oracle(setup_small, chunk_min_tokens):
    """The reference StreamingGuard's storage (state_dtype='float16', src/hs_guard/runtime.py:157) through the whole
    engine: per-token cut scores within 2e-3 of the oracle storing its state in fp16 at the same points (the end of
    each tick), matched GEMMs; state within 4e-3 relative (fp16 storage: one rounding of 2^-11 per tick, more where
    values fall below fp16's normal range, as the kernel test's bar); ring_pos and length bit-exact."""
    from hs_guard.engine.slot_engine import SlotStreamEngine
    from oracle.backbone import StreamOracle
    cfg, model, weights = setup_small
    print(f"[engine] fp16 state, chunk_min_tokens {chunk_min_tokens}", flush=True)
    eng = SlotStreamEngine(model, 4, state_dtype="float16", use_graphs=False, chunk_min_tokens=chunk_min_tokens)
    assert eng.rec.dtype == torch.float16
    orc = StreamOracle(weights, cfg, 4, state_dtype="float16")
    gemm = _matched_gemm(eng)
    worst = 0.0
    for t, tick in enumerate(_schedule(np.random.default_rng(3), cfg.vocab_size)):
        diff = _max_diff(eng.step(tick), orc.step(tick, gemm=gemm))
        worst = max(worst, diff)
        assert diff <= PROB_TOL, f"tick {t}: prob diff {diff:.2e}"
    print(f"[engine] fp16 state worst prob diff {worst:.2e}", flush=True)
    np.testing.assert_array_equal(eng.length, orc.length)
    np.testing.assert_array_equal(eng.ring_pos.cpu().numpy(), orc.ring_pos)
    rec = eng.rec.double().cpu().numpy()
    for s in range(4):
        rel = np.linalg.norm(rec[:, s] - orc.rec[:, s]) / np.linalg.norm(orc.rec[:, s])
        print(f"[engine] fp16 state slot {s} rel err {rel:.2e}", flush=True)
        assert rel < 4e-3, f"slot {s} state rel err {rel:.2e}"


def test_single_token_ticks_match_oracle(setup_small):
    """The single-slot single-token path (ticks of one token in graphs, as the serving loop replays them): every
    product on the skinny kernels with the residual add + RMSNorm and the SiLU gate inside them, the attention's
    q / k norm and RoPE inside the split-K decode (hsg_ring_decode_rope), the final norm with the heads' first
    Linear in one launch. Rings run past the 32-token window first; a tick of two one-token rows takes the skinny
    products with the separate norm + RoPE. Matched GEMMs (the oracle's biased head product is torch.addmm, which
    the engine's one-launch norm + Linear may differ from by one bf16 step in a few outputs), cut scores within
    2e-3 of the oracle, ring_pos and length bit-exact, state within 1e-3 relative."""
    from hs_guard.engine.slot_engine import SlotStreamEngine
    from oracle.backbone import StreamOracle
    cfg, model, weights = setup_small
    assert cfg.rotary_dim == 64 and cfg.head_dim == 256 and cfg.hidden_size == 1024   # the fused routes' geometry
    print("[engine] one-token ticks vs oracle, matched GEMMs", flush=True)
    eng = SlotStreamEngine(model, 4)
    assert eng.gemm_skinny_rows >= 2
    orc = StreamOracle(weights, cfg, 4)
    gemm = _matched_gemm(eng)
    rng = np.random.default_rng(4)
    V = cfg.vocab_size
    ticks = [[(0, rng.integers(0, V, 40).tolist()), (1, rng.integers(0, V, 36).tolist())],
             [(2, rng.integers(0, V, 33).tolist())]]
    ticks += [[(t % 3, [int(rng.integers(0, V))])] for t in range(14)]
    ticks.append([(0, [int(rng.integers(0, V))]), (3, [int(rng.integers(0, V))])])
    ticks += [[(3, [int(rng.integers(0, V))])], [(1, [int(rng.integers(0, V))])]]
    worst = 0.0
    for t, tick in enumerate(ticks):
        diff = _max_diff(eng.step(tick), orc.step(tick, gemm=gemm))
        worst = max(worst, diff)
        assert diff <= PROB_TOL, f"tick {t}: prob diff {diff:.2e}"
    print(f"[engine] one-token ticks worst prob diff {worst:.2e}", flush=True)
    assert (orc.length[:3] > cfg.window_tokens).all()
    np.testing.assert_array_equal(eng.length, orc.length)
    np.testing.assert_array_equal(eng.ring_pos.cpu().numpy(), orc.ring_pos)
    rec = eng.rec.double().cpu().numpy()
    for s in range(4):
        rel = np.linalg.norm(rec[:, s] - orc.rec[:, s]) / np.linalg.norm(orc.rec[:, s])
        assert rel < 1e-3, f"slot {s} state rel err {rel:.2e}"


def test_engine_matches_oracle_matched_gemms(setup2):
    from hs_guard.engine.slot_engine import SlotStreamEngine
    from oracle.backbone import StreamOracle
    cfg, model, weights = setup2
    print("[engine] eager vs oracle, matched GEMMs", flush=True)
    eng = SlotStreamEngine(model, 4, use_graphs=False)
    orc = StreamOracle(weights, cfg, 4)
    gemm = _matched_gemm(eng)
    rng = np.random.default_rng(0)
    worst = 0.0
    for t, tick in enumerate(_schedule(rng, cfg.vocab_size)):
        got = eng.step(tick)
        ref = orc.step(tick, gemm=gemm)
        diff = _max_diff(got, ref)
        worst = max(worst, diff)
        assert diff <= PROB_TOL, f"tick {t}: prob diff {diff:.2e}"
    print(f"[engine] matched-GEMM worst prob diff {worst:.2e}", flush=True)
    np.testing.assert_array_equal(eng.length, orc.length)
    np.testing.assert_array_equal(eng.ring_pos.cpu().numpy(), orc.ring_pos)
    rec = eng.rec.double().cpu().numpy()
    for s in range(4):
        rel = np.linalg.norm(rec[:, s] - orc.rec[:, s]) / np.linalg.norm(orc.rec[:, s])
        assert rel < 1e-3, f"slot {s} state rel err {rel:.2e}"
    # a planted mistake in the oracle (attention gate dropped) is far outside the tolerance
    import oracle.ring as oring
    orig = oring.ring_attention_v8
    oring.ring_attention_v8 = lambda q, rk, rv, nk, value, gate, *a, **k: orig(q, rk, rv, nk, value,
                                                                               np.full_like(gate, 30.0), *a, **k)
    try:
        eng2 = SlotStreamEngine(model, 4, use_graphs=False)
        orc2 = StreamOracle(weights, cfg, 4)
        tick = _schedule(np.random.default_rng(0), cfg.vocab_size)[0]
        assert _max_diff(eng2.step(tick), orc2.step(tick, gemm=_matched_gemm(eng2))) > 5 * PROB_TOL
    finally:
        oring.ring_attention_v8 = orig


def test_engine_chunk_route_matches_oracle_matched_gemms(setup2):
    """The engine with the chunked GDN kernels on (chunk_min_tokens 2: in the schedule's prefill-like ticks every
    row of two or more tokens goes through hsg_gdn_chunk_prefill_gated, single tokens and the mixed ticks through
    the slot step) against the oracle with matched GEMMs, at the same 2e-3 bar as the slot-step route."""
    from hs_guard.engine.slot_engine import SlotStreamEngine
    from oracle.backbone import StreamOracle
    cfg, model, weights = setup2
    print("[engine] chunk route vs oracle, matched GEMMs", flush=True)
    eng = SlotStreamEngine(model, 4, use_graphs=False, chunk_min_tokens=2)
    orc = StreamOracle(weights, cfg, 4)
    gemm = _matched_gemm(eng)
    worst = 0.0
    for t, tick in enumerate(_schedule(np.random.default_rng(0), cfg.vocab_size)):
        diff = _max_diff(eng.step(tick), orc.step(tick, gemm=gemm))
        worst = max(worst, diff)
        assert diff <= PROB_TOL, f"tick {t}: prob diff {diff:.2e}"
    print(f"[engine] chunk route worst prob diff {worst:.2e}", flush=True)
    np.testing.assert_array_equal(eng.length, orc.length)
    np.testing.assert_array_equal(eng.ring_pos.cpu().numpy(), orc.ring_pos)
    rec = eng.rec.double().cpu().numpy()
    for s in range(4):
        rel = np.linalg.norm(rec[:, s] - orc.rec[:, s]) / np.linalg.norm(orc.rec[:, s])
        assert rel < 1e-3, f"slot {s} state rel err {rel:.2e}"


def test_engine_matches_oracle(setup):
    from hs_guard.engine.slot_engine import SlotStreamEngine
    from oracle.backbone import StreamOracle
    cfg, model, weights = setup
    print("[engine] eager vs oracle, independent GEMMs", flush=True)
    eng = SlotStreamEngine(model, 4, use_graphs=False)
    orc = StreamOracle(weights, cfg, 4)
    rng = np.random.default_rng(0)
    for t, tick in enumerate(_schedule(rng, cfg.vocab_size)):
        got = eng.step(tick)
        ref = orc.step(tick)
        diff = _max_diff(got, ref)
        assert diff <= PROB_TOL_INDEPENDENT, f"tick {t}: prob diff {diff:.2e}"
    np.testing.assert_array_equal(eng.length, orc.length)
    np.testing.assert_array_equal(eng.ring_pos.cpu().numpy(), orc.ring_pos)
    rec = eng.rec.double().cpu().numpy()
    for s in range(4):
        rel = np.linalg.norm(rec[:, s] - orc.rec[:, s]) / np.linalg.norm(orc.rec[:, s])
        assert rel < 2e-2, f"slot {s} state rel err {rel:.2e}"
    assert np.count_nonzero(rec[:, 4]) == 0        # scratch slot untouched
    W = cfg.window_tokens
    rk = eng.ring_k[:, :, :, :W].float().cpu().numpy()
    valid = orc.ring_pos[:4, :W] >= 0
    for s in range(4):
        got_k, ref_k = rk[:, s][..., valid[s], :], orc.ring_k[:, s, :, :W][..., valid[s], :]
        rel = np.linalg.norm(got_k - ref_k) / np.linalg.norm(ref_k)
        assert rel < 2e-2, f"ring_k slot {s} rel diff {rel:.2e}"


def test_graph_replays_match_eager(setup):
    """Every replay of every captured bucket equals the eager program bit for bit, with eager work and
    synchronizations between the replays."""
    from hs_guard.engine.slot_engine import SlotStreamEngine
    cfg, model, _ = setup
    print("[engine] graph vs eager", flush=True)
    eg = SlotStreamEngine(model, 4, use_graphs=True)
    ee = SlotStreamEngine(model, 4, use_graphs=False)
    rng = np.random.default_rng(1)
    for t, tick in enumerate(_schedule(rng, cfg.vocab_size) * 2):
        a = eg.step(tick)
        torch.cuda.synchronize()
        b = ee.step(tick)
        _ = torch.ones(1024, device="cuda").sum().item()   # unrelated eager work between replays
        for role in a:
            for x, y in zip(a[role], b[role]):
                np.testing.assert_array_equal(x.numpy(), y.numpy(), err_msg=f"tick {t}")
    assert eg.stats["graph_replays"] > 0 and eg.stats["captures"] >= 3
    for name in ("rec", "conv", "ring_k", "ring_v", "ring_pos"):
        assert torch.equal(getattr(eg, name), getattr(ee, name)), name


def test_step_packed_matches_step(setup):
    """step_packed (the serving scheduler's call, src/hs_guard/engine/slot_engine_v7.py:138-145) returns, for
    the same ticks on an identical engine, exactly step's per-request probabilities in its [R, n, lb, 3]
    layout (lb = the token bucket of the tick's longest request), zeros past each request's length, and
    leaves the same pools and lengths."""
    from hs_guard.engine.slot_engine import SlotStreamEngine, bucket
    cfg, model, _ = setup
    print("[engine] step_packed vs step", flush=True)
    ea = SlotStreamEngine(model, 4)
    eb = SlotStreamEngine(model, 4)
    rng = np.random.default_rng(4)
    for t, tick in enumerate(_schedule(rng, cfg.vocab_size)):
        tick = [(s, ids[:ea.max_tick_tokens]) for s, ids in tick]   # step_packed takes one tick
        a = ea.step(tick)
        packed, lens = eb.step_packed(tick)
        lb = bucket(max(len(ids) for _, ids in tick), (1, 2, 4, 8, 16, 32, 64))
        assert packed.shape == (len(ea.roles), len(tick), lb, 3) and list(lens) == [len(ids) for _, ids in tick]
        for r_i, role in enumerate(ea.roles):
            for n, (_, ids) in enumerate(tick):
                np.testing.assert_array_equal(packed[r_i, n, :len(ids)], a[role][n].numpy(), err_msg=f"tick {t}")
                assert not packed[r_i, n, len(ids):].any()
    for name in ("rec", "conv", "ring_k", "ring_v", "ring_pos"):
        assert torch.equal(getattr(ea, name), getattr(eb, name)), name
    assert np.array_equal(ea.length, eb.length)


def test_fused_conv_engine_equals_separate_conv():
    """With one value head per key head the engine runs the GDN conv inside the slot step; over several ticks it
    gives exactly the probabilities and pools of the engine that runs the conv as its own kernel."""
    from hs_guard.engine.slot_engine import SlotStreamEngine
    from hs_guard.model import GuardConfig, GuardModel
    print("[engine] fused conv vs separate conv", flush=True)
    cfg = GuardConfig(vocab_size=1000, hidden_size=1024, num_hidden_layers=4, intermediate_size=1024,
                      linear_num_key_heads=2, linear_num_value_heads=2, num_attention_heads=8,
                      num_key_value_heads=2, window_tokens=32)
    model = GuardModel.random(cfg, seed=3, device="cuda:0")
    ef = SlotStreamEngine(model, 4)
    es = SlotStreamEngine(model, 4, fuse_conv=False)
    assert ef.fuse_conv and not es.fuse_conv
    rng = np.random.default_rng(9)
    for t, tick in enumerate(_schedule(rng, cfg.vocab_size)):
        a = ef.step(tick)
        b = es.step(tick)
        for role in a:
            for x, y in zip(a[role], b[role]):
                np.testing.assert_array_equal(x.numpy(), y.numpy(), err_msg=f"tick {t}")
    for name in ("rec", "conv", "ring_k", "ring_v", "ring_pos"):
        assert torch.equal(getattr(ef, name), getattr(es, name)), name


def test_streaming_guard_api(setup):
    """Drop-in API: cut scores = 1 - p(safe) of the chosen role, reset clears every slot, snapshots restore."""
    from hs_guard.runtime import StreamingGuard, random_metadata
    cfg, model, weights = setup
    print("[engine] StreamingGuard", flush=True)
    guard = StreamingGuard(model, random_metadata(), max_slots=3)
    ids = np.random.default_rng(2).integers(0, cfg.vocab_size, 12).tolist()
    first = guard.step([(1, ids[:5]), (0, ids[:3])], role="user")
    assert [r["slot"] for r in first] == [1, 0]
    assert len(first[0]["cut_scores"]) == 5 and first[0]["threshold"] == pytest.approx(0.0761368871)
    snap = guard.engine.snapshot(1)
    more = guard.step([(1, ids[5:])])
    guard.engine.restore(1, snap)
    again = guard.step([(1, ids[5:])])
    np.testing.assert_array_equal(more[0]["cut_scores"], again[0]["cut_scores"])
    guard.reset()
    assert guard.engine.length.sum() == 0 and int((guard.engine.ring_pos >= 0).sum()) == 0
    fresh = guard.step([(1, ids[:5])], role="user")
    np.testing.assert_allclose(fresh[0]["cut_scores"], first[0]["cut_scores"], rtol=0, atol=0)
    with pytest.raises(ValueError):
        guard.step([(3, [1])])
    with pytest.raises(ValueError):
        guard.step([(0, [cfg.vocab_size])])
    # a tick shape first captured by step_packed (under inference mode), then stepped through the guard
    guard.engine.step_packed([(2, ids[:2])])
    rec = guard.step([(2, ids[2:4])])
    assert len(rec) == 1 and len(rec[0]["cut_scores"]) == 2
    # the engine's own entry points (step_packed is the serving backend's call) refuse out-of-vocabulary ids too,
    # before anything runs: lengths, rings and state stay as they were
    eng = guard.engine
    before = (eng.length.copy(), eng.rec.clone(), eng.ring_pos.clone())
    for bad in ([(0, [1, cfg.vocab_size])], [(2, [3]), (1, [-1])], [(0, [2.0])], [(0, list(range(70)) + [10 ** 9])]):
        for call in (eng.step, eng.step_packed):
            with pytest.raises(ValueError, match="in-vocabulary"):
                call(bad)
    assert np.array_equal(eng.length, before[0]) and torch.equal(eng.rec, before[1])
    assert torch.equal(eng.ring_pos, before[2])


def test_reset_slots_neighbours_untouched_and_fresh(setup2):
    """reset(slots) (the per-slot reset config 5's sessions and the demo's scheduler rely on,
    examples/demo/runtime_v10.py:98-111): the reset slots' pools return to the empty state, every other slot's
    pools stay bit for bit, later ticks match the oracle reset the same way (matched GEMMs, 2e-3), and the
    reset slot's outputs equal bit for bit those of a fresh engine that never saw the slot's earlier tokens
    but runs the same later ticks."""
    from hs_guard.engine.slot_engine import SlotStreamEngine
    from oracle.backbone import StreamOracle
    cfg, model, weights = setup2
    print("[engine] reset(slots)", flush=True)
    sched = _schedule(np.random.default_rng(5), cfg.vocab_size)
    first, later = sched[:5], sched[5:]
    eng = SlotStreamEngine(model, 4, use_graphs=False)
    fresh = SlotStreamEngine(model, 4, use_graphs=False)
    orc = StreamOracle(weights, cfg, 4)
    gemm = _matched_gemm(eng)
    reset = [1, 3]
    for tick in first:
        eng.step(tick)
        orc.step(tick, gemm=gemm)
        rest = [(s, ids) for s, ids in tick if s not in reset]
        if rest:
            fresh.step(rest)
    before = {n: getattr(eng, n).clone() for n in ("rec", "conv", "ring_k", "ring_v", "ring_pos")}
    length = eng.length.copy()
    eng.reset(reset)
    orc.reset(reset)
    keep = [0, 2, 4]                       # the other slots and the scratch slot
    for n, t in before.items():
        now = getattr(eng, n)
        if n == "ring_pos":
            assert torch.equal(now[keep], t[keep]) and bool((now[reset] == -1).all())
        else:
            assert torch.equal(now[:, keep], t[:, keep]), n
            assert int(torch.count_nonzero(now[:, reset])) == 0, n
    assert list(eng.length[reset]) == [0, 0] and list(eng.length[[0, 2]]) == list(length[[0, 2]])
    worst = 0.0
    for t, tick in enumerate(later):
        got = eng.step(tick)
        ref = orc.step(tick, gemm=gemm)
        alone = fresh.step(tick)
        worst = max(worst, _max_diff(got, ref))
        assert worst <= PROB_TOL, f"tick {t}: {worst:.2e}"
        for i, (s, _) in enumerate(tick):
            if s in reset:
                for role in got:
                    np.testing.assert_array_equal(got[role][i].numpy(), alone[role][i].numpy(), err_msg=f"tick {t}")
    print(f"[engine] after reset: worst prob diff {worst:.2e}", flush=True)
    np.testing.assert_array_equal(eng.length, orc.length)
    np.testing.assert_array_equal(eng.ring_pos.cpu().numpy(), orc.ring_pos)
    for n in ("rec", "conv", "ring_k", "ring_v"):
        assert torch.equal(getattr(eng, n)[:, reset], getattr(fresh, n)[:, reset]), n


def test_matched_engine_pools_match_oracle(setup2):
    """With matched GEMMs the pools the engine leaves behind match the oracle's: the GDN layer's conv history
    (raw projections of the embedding's RMSNorm, identical inputs) bit for bit; the attention layer's ring keys
    and values, whose inputs have passed the GDN layer (fp32 against float64 arithmetic, so a few bf16 roundings
    of its output go the other way), within 5e-3 relative; state within 1e-3 relative."""
    from hs_guard.engine.slot_engine import SlotStreamEngine
    from oracle.backbone import StreamOracle
    cfg, model, weights = setup2
    print("[engine] pools vs oracle, matched GEMMs", flush=True)
    eng = SlotStreamEngine(model, 4, use_graphs=False)
    orc = StreamOracle(weights, cfg, 4)
    gemm = _matched_gemm(eng)
    for tick in _schedule(np.random.default_rng(0), cfg.vocab_size):
        eng.step(tick)
        orc.step(tick, gemm=gemm)
    W = cfg.window_tokens
    conv = eng.conv[:, :4].float().cpu().numpy()
    np.testing.assert_array_equal(conv, orc.conv[:, :4])
    for name in ("ring_k", "ring_v"):
        got = getattr(eng, name)[:, :4, :, :W].float().cpu().numpy()
        ref = getattr(orc, name)[:, :4, :, :W]
        rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        print(f"[engine] {name}: {np.mean(got != ref):.1e} of values differ, rel {rel:.1e}", flush=True)
        assert rel <= 5e-3, f"{name} rel {rel:.2e}"
    rec = eng.rec.double().cpu().numpy()
    for s in range(4):
        rel = np.linalg.norm(rec[:, s] - orc.rec[:, s]) / np.linalg.norm(orc.rec[:, s])
        assert rel < 1e-3, f"slot {s} state rel err {rel:.2e}"


@pytest.mark.parametrize("sizes", LONG_PIECES)
def test_long_pieces_match_ticks(sizes):
    """Contexts in long pieces against the same engine cut into 64-token ticks, past the window, then one more tick and
    a second context on the live sessions. The two paths round their products and softmax blocks differently, so the
    probabilities agree to PROB_TOL at the weight scale where rounding alone moves them by 5e-4 (setup_small); lengths
    and ring positions are equal. After every step the sessions' pools agree within POOL_BARS, which a dropped row, a wrong
    conv history, segment state or GDN output exceeds many times (tests/test_oracle_backbone.py), where the probabilities
    move by less than PROB_TOL."""
    from hs_guard.engine.slot_engine import SlotStreamEngine
    cfg, model, steps = long_piece_case(sizes)
    model = model.to("cuda:0")
    long, ticks = SlotStreamEngine(model, len(sizes) + 1), SlotStreamEngine(model, len(sizes) + 1)
    ticks._long_scratch = lambda rows, piece: None      # as on a card without room for the scratch
    slots = range(len(sizes))
    for reqs in steps:
        lens = [len(ids) for _, ids in reqs]
        before = long.stats["eager_steps"]
        a, b = long.step(reqs), ticks.step(reqs)
        assert (long.stats["eager_steps"] > before) == (max(lens) > 64)
        for role in a:
            for x, y, n in zip(a[role], b[role], lens):
                assert x.shape == y.shape == (n, 3)
                assert float((x - y).abs().max()) <= PROB_TOL
        errs = pool_errors(long, ticks, slots, cfg.window_tokens)
        print("[engine] long piece pools", {k: f"{v:.1e}" for k, v in errs.items()}, flush=True)
        assert all(errs[k] <= bar for k, bar in POOL_BARS.items()), errs
    assert ticks.stats["eager_steps"] == 0
    np.testing.assert_array_equal(long.length, ticks.length)
    assert torch.equal(long.ring_pos[:len(sizes)], ticks.ring_pos[:len(sizes)])


@pytest.mark.parametrize("chunk_min_tokens,routes", [(16, {("slot", 16), ("chunk", 16)}), (1, {("chunk", 1)}),
                                                     (65, set())])
def test_long_pieces_keep_the_chunk_rule(monkeypatch, chunk_min_tokens, routes):
    """A long piece's rows of fewer than chunk_min_tokens tokens run the slot step, as in ticks, and an engine whose
    chunk_min_tokens no tick's row reaches runs no long piece."""
    from hs_guard.engine import slot_engine
    from hs_guard.model import GuardConfig, GuardModel
    cfg = GuardConfig(vocab_size=1000, hidden_size=1024, num_hidden_layers=2,
                      layer_types=["linear_attention", "full_attention"], intermediate_size=1024,
                      linear_num_key_heads=2, linear_num_value_heads=4, num_attention_heads=8,
                      num_key_value_heads=2, window_tokens=96)
    model = GuardModel.random(cfg, seed=1, device="cpu", std=0.005).to("cuda:0")
    eng = slot_engine.SlotStreamEngine(model, 3, use_graphs=False, chunk_min_tokens=chunk_min_tokens)
    native, seen = slot_engine.calls(), set()

    class Recorded:
        def __getattr__(self, name):
            fn = getattr(native, name)
            if name == "hsg_gdn_slot_step_gated":        # skip_min_len: third from last of its arguments
                return lambda *args: seen.add(("slot", args[-3])) or fn(*args)
            if name == "hsg_gdn_chunk_prefill_gated":    # min_len: fourth from last
                return lambda *args: seen.add(("chunk", args[-4])) or fn(*args)
            return fn

    long_piece, pieces = eng._run_long, []

    def run_long(*args):
        with monkeypatch.context() as m:
            m.setattr(slot_engine, "calls", Recorded)
            pieces.append(len(args[0]))
            return long_piece(*args)

    eng._run_long = run_long
    out = eng.step([(0, list(range(100))), (1, [1, 2, 3]), (2, list(range(17)))])
    for role in out:
        assert all(torch.isfinite(p).all() for p in out[role])
    assert pieces == ([3] if routes else []) and seen == routes
