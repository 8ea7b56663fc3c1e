"""One LFM2 decode step on the GPU (GGUF file -> model handle -> forward) against the oracle's restatement
of the reference's aarch64 CPU model (wick/src/model/lfm2.rs:1020-1124, 2258-2289) on seeded random models."""
import numpy as np
import pytest

import lfm2_synth
import wick_amd as W
from conftest import rel_l2
from oracle import lfm2_oracle as L
from wick_amd import gguf as G
from wick_amd.lfm2 import RocmLfm2Model

pytestmark = pytest.mark.gpu

# f32 tolerance of a whole step: every operation is within a few ulp of the oracle's and the residual
# stream keeps that near 1e-7; 1e-5 rel-L2 is the bar of the matmul path itself.
LOGITS_REL_L2 = 1e-5
# The step re-quantizes f32 activations to Q8_0 before every GEMV, and that quantizer is discontinuous:
# when some x/d sits within the f32 noise of a rounding tie, two correct pipelines that differ in the last
# bit of one activation differ by a whole quant step afterwards (about 1e-3 of a GEMV output per flipped
# quant), and the KV cache / conv state carry it to later positions.  The oracle reports how close every
# GEMV input came to such a tie (quantizer_margin); positions are held to the strict bar until the first
# near-tie, to the loose one (what one flipped quant can do) from there on.
NEAR_TIE = 3e-5  # in quant steps; the GPU's activations differ from the oracle's by <= ~1e-5 of a step
LOOSE_REL_L2 = 5e-2
LOOSE_COSINE = 0.999


def cosine(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(a @ b / (np.linalg.norm(a) * np.linalg.norm(b)))


def check_step(logits, want, margin, what):
    """Returns True when the step was held to the strict bar."""
    assert np.isfinite(logits).all(), what
    if margin >= NEAR_TIE:
        assert rel_l2(logits, want) <= LOGITS_REL_L2, f"{what}: rel-L2 {rel_l2(logits, want):.2e} (margin {margin:.1e})"
        assert int(np.argmax(logits)) == int(np.argmax(want)), what
        return True
    assert rel_l2(logits, want) <= LOOSE_REL_L2 and cosine(logits, want) >= LOOSE_COSINE, f"{what}: rel-L2 {rel_l2(logits, want):.2e} after a near-tie"
    return False


def load(ctx, oracle, tmp_path, context=64, **kw):
    img, cfg, tensors = lfm2_synth.build(oracle, **kw)
    path = tmp_path / "lfm2_synth.gguf"
    path.write_bytes(img)
    with G.GgufFile.open(str(path)) as g:
        model = RocmLfm2Model(ctx, g, context)
    return model, L.Lfm2Oracle(cfg, tensors), cfg


# Small models and seeds picked so that the whole token sequence stays clear of quantizer ties (the search ran
# on the oracle alone; the test re-checks the margin, so a change of the generator cannot go unnoticed).
CLEAR = {
    "q4_0+q6k": dict(hidden=256, inter=256, vocab=256, seed=16),                      # Q4_0 body, Q6_K embedding: a shipped Q4_0 file
    "q8_0": dict(hidden=256, inter=256, vocab=256, wtype=W.Q8_0, embd_type=W.Q8_0, seed=25),
    "kernel4": dict(hidden=256, inter=256, vocab=256, kernel=4, kv_heads=(2, 0, 0, 4), rope_theta=10000.0, eps=1e-6, seed=20),
    "mixed-qkv": dict(hidden=256, inter=256, vocab=256, mixed_qkv=True, seed=27),      # Q/K Q4_0, V Q8_0: separate launches
    "3-layer-q4embd": dict(n_layers=3, hidden=512, inter=512, n_heads=8, kv_heads=(0, 4, 8), vocab=512, embd_type=W.Q4_0, seed=1),
}


@pytest.mark.parametrize("name", list(CLEAR))
def test_forward_matches_the_oracle_step_by_step(ctx, oracle, tmp_path, name):
    kw = CLEAR[name]
    model, ref, cfg = load(ctx, oracle, tmp_path, **kw)
    assert model.kv_heads_per_layer == cfg["kv_heads_per_layer"]
    assert model.config["max_seq_len"] == 64 and model.config["n_kv_heads"] == max(cfg["kv_heads_per_layer"])
    state = ref.new_state()
    tokens = np.random.default_rng(100 + kw["seed"]).integers(0, cfg["vocab_size"], 6)
    for pos, tok in enumerate(tokens):
        logits = model.forward(int(tok), pos)
        want = ref.forward(int(tok), pos, state)
        assert ref.min_margin >= NEAR_TIE, "this seed no longer stays clear of quantizer ties: search another"
        assert check_step(logits, want, ref.min_margin, f"{name} pos {pos}")
    model.free()


@pytest.mark.parametrize("hidden,wtype", [(256, W.Q4_0), (512, W.Q8_0), (1024, W.Q4_0), (1024, W.Q8_0), (2048, W.Q4_0)])
def test_step_at_positions_around_the_split_edges(ctx, oracle, tmp_path, hidden, wtype):
    """One record per head, a second split's first key, a partial last group of splits, both sides of the position up to which
    the output projection merges the records itself (1024) -- for head counts 4 to 32, on a restored random state."""
    model, ref, cfg = load(ctx, oracle, tmp_path, context=1100, n_layers=1, hidden=hidden, inter=256, n_heads=hidden // 64, kv_heads=(hidden // 128,),
                           vocab=256, wtype=wtype, embd_type=W.Q8_0, seed=7)
    kvd, rng = hidden // 2, np.random.default_rng(hidden)
    for pos in (0, 1, 63, 64, 300, 1022, 1023, 1024):
        k, v = rng.standard_normal((2, pos, kvd)).astype(np.float32)
        if pos:
            model.restore_state(np.concatenate([k.ravel(), v.ravel()]).view(np.uint8), pos)
        state = {"seq_len": pos, "layers": [{"k": list(k), "v": list(v)}]}
        check_step(model.forward(pos % 256, pos), ref.forward(pos % 256, pos, state), ref.min_margin, f"hidden {hidden} pos {pos}")
    model.free()


def test_larger_model_longer_sequence(ctx, oracle, tmp_path):
    """Six layers, 24 positions: strict until the oracle reports the first near-tie, bounded afterwards."""
    model, ref, cfg = load(ctx, oracle, tmp_path, n_layers=6, hidden=512, inter=1024, n_heads=8, kv_heads=(0, 0, 4, 0, 8, 2), vocab=1000,
                           embd_type=W.Q4_0, seed=3)
    state = ref.new_state()
    tokens = np.random.default_rng(11).integers(0, cfg["vocab_size"], 24)
    strict = sum(check_step(model.forward(int(t), p), ref.forward(int(t), p, state), ref.min_margin, f"pos {p}") for p, t in enumerate(tokens))
    assert strict >= 1
    model.free()


def test_a_quantizer_tie_is_the_only_thing_that_loosens_the_bar(ctx, oracle, tmp_path):
    """Token 42 of this model puts an FFN input at x/d = 61.499996: the oracle flags it, the GPU step stays
    within what one flipped quant can do, and the very same model is strict on tokens that stay clear of ties."""
    model, ref, cfg = load(ctx, oracle, tmp_path, wtype=W.Q8_0, embd_type=W.Q8_0, seed=2)
    state = ref.new_state()
    want = ref.forward(42, 0, state)
    assert ref.min_margin < 1e-5
    assert check_step(model.forward(42, 0), want, ref.min_margin, "token 42") is False
    model.reset()
    ref2 = L.Lfm2Oracle(cfg, ref.t)
    state = ref2.new_state()
    want = ref2.forward(3, 0, state)
    assert ref2.min_margin >= NEAR_TIE
    assert check_step(model.forward(3, 0), want, ref2.min_margin, "clear token 3") is True
    model.free()


def test_reset_starts_a_fresh_state(ctx, oracle, tmp_path):
    model, ref, cfg = load(ctx, oracle, tmp_path)
    first = [model.forward(t, p) for p, t in enumerate([5, 9, 200])]
    model.reset()
    again = [model.forward(t, p) for p, t in enumerate([5, 9, 200])]
    for a, b in zip(first, again):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    model.free()


def test_greedy_generation_stays_on_the_device(ctx, oracle, tmp_path):
    """forward_greedy == argmax(forward) with the reference's tie rule; n steps without a host round trip
    give the same tokens as n single steps."""
    model, ref, cfg = load(ctx, oracle, tmp_path, hidden=256, inter=256, vocab=256, seed=26)
    state, tok, want = ref.new_state(), 17, []
    for pos in range(10):
        tok = L.argmax(ref.forward(tok, pos, state))
        want.append(tok)
    assert ref.min_margin >= NEAR_TIE, "this seed walks into a quantizer tie: pick another"
    got = model.generate_greedy(17, 0, 10)
    assert got.tolist() == want
    model.reset()
    tok, single = 17, []
    for pos in range(10):
        tok = model.forward_greedy(tok, pos)
        single.append(tok)
    assert single == want
    # the two kinds of step interleave on one state: logits of the next position follow the greedy prefix
    logits = model.forward(want[-1], 10)
    expect = ref.forward(want[-1], 10, state)
    check_step(logits, expect, ref.min_margin, "logits after the greedy prefix")
    model.free()


def test_graph_replay_and_plain_launches_agree(ctx, oracle, tmp_path):
    model, ref, cfg = load(ctx, oracle, tmp_path, seed=9)
    replayed = [model.forward(t, p) for p, t in enumerate([4, 8, 15, 16])]
    picks = model.generate_greedy(23, 4, 5)
    model.reset()
    model.set_graph_replay(False)
    plain = [model.forward(t, p) for p, t in enumerate([4, 8, 15, 16])]
    for a, b in zip(replayed, plain):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert model.generate_greedy(23, 4, 5).tolist() == picks.tolist()
    model.free()


def test_per_dispatch_timing_sees_the_step(ctx, oracle, tmp_path):
    """While per-dispatch timing is on, a step is enqueued launch by launch (a graph hides its kernels from
    the timer) and still gives the replayed step's logits."""
    model, ref, cfg = load(ctx, oracle, tmp_path, seed=9)
    replayed = [model.forward(4, 0), model.forward(8, 1)]
    model.reset()
    ctx.kernel_timing_begin()
    timed = model.forward(4, 0)
    fams = ctx.kernel_timing_end()
    assert np.array_equal(replayed[0].view(np.uint32), timed.view(np.uint32))
    assert sum(n for _, n in fams.values()) >= 4 * cfg["n_layers"], fams
    # the state the timed step left carries the next replayed one
    assert np.array_equal(replayed[1].view(np.uint32), model.forward(8, 1).view(np.uint32))
    model.free()


def test_load_and_step_errors(ctx, oracle, tmp_path):
    model, ref, cfg = load(ctx, oracle, tmp_path, context=8, context_length=6)
    assert model.config["max_seq_len"] == 6  # min(context_size, lfm2.context_length), wick/src/model/lfm2.rs:121-125
    assert model.gpu_memory_bytes() > 0
    with pytest.raises(W.RocmError, match="token_id out of range"):
        model.forward(cfg["vocab_size"], 0)
    with pytest.raises(W.RocmError, match="beyond the context"):
        model.forward(1, 6)
    with pytest.raises(W.RocmError, match="beyond the context"):
        model.generate_greedy(1, 4, 3)
    model.free()
    img, _, _ = lfm2_synth.build(oracle)
    with G.GgufFile.from_bytes(img) as g:
        with pytest.raises(W.RocmError, match="context_size"):
            RocmLfm2Model(ctx, g, 0)
    # a file without the LFM2 metadata / tensors is refused with the missing name
    import gguf_writer as GW
    with G.GgufFile.from_bytes(GW.build([("general.architecture", GW.T_STRING, "llama")])[0]) as g:
        with pytest.raises(W.RocmError, match="missing lfm2.block_count"):
            RocmLfm2Model(ctx, g, 16)


# ---- prompts (batched prefill) -------------------------------------------------------------------------------
# The reference's prefill computes what n single steps compute, with the projections batched into GEMMs
# (prefill_layers_and_logits, wick/src/model/lfm2.rs:1139-2109; its own tests compare prefill against sequential
# decode by cosine / top-1, wick/tests/blas_parity.rs:71-152).  The oracle for a prompt is therefore the oracle's
# sequential decode; the same quantizer-tie rule applies.

def oracle_prompt(ref, tokens, state, start=0):
    logits = None
    for j, t in enumerate(tokens):
        logits = ref.forward(int(t), start + j, state)
    return logits


@pytest.mark.parametrize("name,n", [("q4_0+q6k", 1), ("q8_0", 3), ("q4_0+q6k", 5), ("q4_0+q6k", 11), ("q4_0+q6k", 24), ("q8_0", 17), ("kernel4", 33), ("kernel4", 2), ("mixed-qkv", 16), ("3-layer-q4embd", 40)])
def test_prefill_matches_the_oracle(ctx, oracle, tmp_path, name, n):
    """One or two tokens run as single steps, up to eight with the projections as multi-token GEMVs, longer prompts on the
    int8-MFMA GEMM."""
    kw = CLEAR[name]
    model, ref, cfg = load(ctx, oracle, tmp_path, **kw)
    tokens = np.random.default_rng(7 + n).integers(0, cfg["vocab_size"], n)
    state = ref.new_state()
    want = oracle_prompt(ref, tokens, state)
    got = model.forward_prefill(tokens, 0)
    check_step(got, want, ref.min_margin, f"{name}: prompt of {n}")
    assert cosine(got, want) >= 0.9999
    # the state the prompt left behind (KV rows, conv state) carries the next single steps
    for pos, tok in enumerate([3, 11], start=n):
        check_step(model.forward(tok, pos), ref.forward(tok, pos, state), ref.min_margin, f"{name}: step after the prompt")
    model.free()


def test_model_without_the_gemm_copies(ctx, oracle, tmp_path):
    """A model loaded with wick_rocm_set_gemm_packing(0) keeps the raw blocks only: its prompt pass runs the projections as
    multi-token GEMVs (and the unfused gate / up + SiLU path) and still meets the oracle; it holds less device memory."""
    kw = CLEAR["q4_0+q6k"]
    packed, ref, cfg = load(ctx, oracle, tmp_path, context=256, **kw)
    ctx.set_gemm_packing(False)
    try:
        plain, _, _ = load(ctx, oracle, tmp_path, context=256, **kw)
    finally:
        ctx.set_gemm_packing(True)
    assert plain.gpu_memory_bytes() < packed.gpu_memory_bytes()
    for n in (24, 150):
        tokens = np.random.default_rng(70 + n).integers(0, cfg["vocab_size"], n)
        state = ref.new_state()
        want = oracle_prompt(ref, tokens, state)
        for model in (packed, plain):
            model.reset()
            got = model.forward_prefill(tokens, 0)
            check_step(got, want, ref.min_margin, f"prompt of {n}")
            assert cosine(got, want) >= 0.9999
            check_step(model.forward(3, n), ref.forward(3, n, ref_copy(ref, state)), ref.min_margin, "step after the prompt")
    packed.free(), plain.free()


def ref_copy(ref, state):
    """A copy of an oracle state (the same position is stepped from twice above)."""
    import copy
    return copy.deepcopy(state)


def test_prefill_in_pieces_and_against_single_steps(ctx, oracle, tmp_path):
    model, ref, cfg = load(ctx, oracle, tmp_path, **CLEAR["q4_0+q6k"])
    tokens = np.random.default_rng(3).integers(0, cfg["vocab_size"], 30)
    whole = model.forward_prefill(tokens, 0)
    model.reset()
    model.forward_prefill(tokens[:18], 0)
    pieces = model.forward_prefill(tokens[18:], 18)
    model.reset()
    single = None
    for pos, t in enumerate(tokens):
        single = model.forward(int(t), pos)
    # same arithmetic up to GEMM-vs-GEMV summation order (and what a quantizer tie may do to it)
    assert cosine(whole, pieces) >= 0.9999 and cosine(whole, single) >= 0.9999
    assert int(np.argmax(whole)) == int(np.argmax(single))
    with pytest.raises(W.RocmError, match="beyond the context"):
        model.forward_prefill(tokens, 40)
    with pytest.raises(W.RocmError, match="token_id out of range"):
        model.forward_prefill([1, cfg["vocab_size"]], 0)
    with pytest.raises(W.RocmError, match="empty prompt"):
        model.forward_prefill([], 0)
    model.free()


def test_long_prompt_runs_in_passes(ctx, oracle, tmp_path):
    """2100 tokens = one pass of 2048 + one of 52, attention over up to 2100 cached positions."""
    model, ref, cfg = load(ctx, oracle, tmp_path, context=2200, **CLEAR["q4_0+q6k"])
    tokens = np.random.default_rng(5).integers(0, cfg["vocab_size"], 2100)
    state = ref.new_state()
    want = oracle_prompt(ref, tokens, state)
    got = model.forward_prefill(tokens, 0)
    check_step(got, want, ref.min_margin, "long prompt")
    check_step(model.forward(9, 2100), ref.forward(9, 2100, state), ref.min_margin, "step after the long prompt")
    model.free()


def test_prefill_chunked_and_cancel(ctx, oracle, tmp_path):
    """Model::forward_prefill_chunked (wick/src/model/mod.rs:111-140): chunks of `ubatch` tokens, the cancel flag looked at
    after each chunk (so one chunk always runs), consumed tokens and the last chunk's logits reported."""
    import ctypes as C

    model, ref, cfg = load(ctx, oracle, tmp_path, **CLEAR["q4_0+q6k"])
    tokens = np.random.default_rng(13).integers(0, cfg["vocab_size"], 30)
    consumed, chunked = model.forward_prefill_chunked(tokens, 0, 8)
    assert consumed == 30
    model.reset()
    for lo in range(0, 30, 8):
        piecewise = model.forward_prefill(tokens[lo:lo + 8], lo)
    assert np.array_equal(chunked.view(np.uint32), piecewise.view(np.uint32))  # the same calls, so the same bits
    model.reset()
    consumed, whole = model.forward_prefill_chunked(tokens, 0, 0)  # ubatch 0: one chunk
    assert consumed == 30 and cosine(whole, chunked) >= 0.9999
    # a flag that is already set stops the call after the first chunk
    model.reset()
    flag = C.c_int32(1)
    consumed, first = model.forward_prefill_chunked(tokens, 0, 8, cancel=flag)
    assert consumed == 8
    model.reset()
    assert np.array_equal(first.view(np.uint32), model.forward_prefill(tokens[:8], 0).view(np.uint32))
    # ... and the state holds exactly those 8 tokens: the next step continues from position 8
    state = ref.new_state()
    for j, t in enumerate(tokens[:8]):
        ref.forward(int(t), j, state)
    check_step(model.forward(5, 8), ref.forward(5, 8, state), ref.min_margin, "step after a cancelled prompt")
    consumed, none = model.forward_prefill_chunked([], 0, 8)
    assert consumed == 0 and none is None
    model.free()


def test_step_graph_survives_a_scratch_regrow(ctx, oracle, tmp_path):
    """The step graphs of a model whose LM head is Q6_K go through the context's quantization scratch.  A later, wider
    matmul on the same context frees and reallocates that scratch: the model notices the stale graph and captures it
    again instead of replaying launches that hold freed addresses."""
    model, ref, cfg = load(ctx, oracle, tmp_path, **CLEAR["q4_0+q6k"])
    before = model.forward(7, 0)  # captures the logits graph
    # grow the context's scratch well past anything used so far (n x k quantized activations)
    k, n, m = 8192, 6000, 32  # more columns than any other test asks for, so the scratch really is reallocated here
    w = ctx.upload_weight(oracle.synth_weight(W.Q8_0, m, k, 3), W.Q8_0, m, k)
    d_x, d_y = ctx.to_device(oracle.fill_normal(1, 1.0, n * k)), ctx.alloc(n * m * 4)
    ctx.encode_gemm(w, d_x, 0, d_y, 0, n, k, m)
    ctx.sync()
    # something else takes the addresses the old scratch had
    junk = [ctx.to_device(np.full(4096, np.nan, np.float32)) for _ in range(8)]
    model.reset()
    after = model.forward(7, 0)
    assert np.array_equal(before.view(np.uint32), after.view(np.uint32))
    for b in junk + [d_x, d_y]:
        b.free()
    w.free()
    model.free()


LFM2_350M = dict(n_layers=16, hidden=1024, inter=4608, n_heads=16, kv_heads=(0, 0, 8, 0, 0, 8, 0, 0, 8, 0, 8, 0, 8, 0, 8, 0), vocab=65536,
                 sigma=0.02, seed=7)


def _oracle_spread(cfg, tensors, run, seeds):
    """Per-step rel-L2 spread of the oracle's own logits when the f32 summation order of its GEMVs is jittered
    (Lfm2Oracle(jitter_seed=...)): `run(ref)` returns a list of logits."""
    base = run(L.Lfm2Oracle(cfg, tensors))
    spread = np.zeros(len(base))
    for sd in seeds:
        spread = np.maximum(spread, [rel_l2(a, b) for a, b in zip(run(L.Lfm2Oracle(cfg, tensors, jitter_seed=sd)), base)])
    return base, spread


def test_lfm2_350m_shaped_model(ctx, oracle, tmp_path):
    """The model the decode benchmark times (hidden 1024, FFN 4608, 16 / 8 heads of 64, attention at layers 2, 5, 8, 10,
    12, 14, vocabulary 65536, Q4_0 body + Q6_K tied embedding): the shapes the toy models never reach as a composition
    (k = 4608 takes two lane chunks per row, the gated gate / up kernel at k = 1024, the 65536-row Q6_K head inside the
    step graph, 16-token-tile GEMMs in the prompt pass).  Five decode steps, then a 512-token prompt and a step after it.

    At this width every step has some of its ~120 000 re-quantized activations within 3e-5 quant steps of a rounding tie,
    and a randomly initialised model amplifies a flipped quant: the ORACLE's own logits move by 1e-2 .. 3e-2 when the f32
    sums of its GEMVs are jittered by two ulp (measured below, per step).  The device is held to that spread: it may sit no
    further from the oracle than twice what the oracle does to itself, and the oracle's pick must be in the device's top two."""
    model, ref, cfg = load(ctx, oracle, tmp_path, context=1024, **LFM2_350M)
    steps = [5, 77, 1000, 65535, 31337]

    def decode(r):
        st = r.new_state()
        return [r.forward(t, p, st) for p, t in enumerate(steps)]

    want, spread = _oracle_spread(cfg, ref.t, decode, seeds=(1, 2, 3))
    allowed = np.maximum.accumulate(spread)  # the state carries a flip to every later step
    for pos, tok in enumerate(steps):
        got = model.forward(tok, pos)
        err = rel_l2(got, want[pos])
        assert np.isfinite(got).all()
        assert err <= max(LOGITS_REL_L2, 2.0 * allowed[pos]), f"pos {pos}: rel-L2 {err:.2e}, the oracle's own spread is {allowed[pos]:.2e}"
        assert cosine(got, want[pos]) >= LOOSE_COSINE
        assert int(np.argmax(want[pos])) in np.argsort(got)[-2:].tolist()
    assert spread.max() <= LOOSE_REL_L2, "the jittered oracle itself leaves the loose bar: pick another model seed"
    # prompt of 512 tokens in one batched pass against the oracle's 512 single steps, and the step after it
    tokens = np.random.default_rng(350).integers(0, cfg["vocab_size"], 512)

    def prompt(r):
        st = r.new_state()
        for j, t in enumerate(tokens[:-1]):
            r.hidden_after_layers(int(t), j, st)
        return [r.forward(int(tokens[-1]), 511, st), r.forward(123, 512, st)]

    want, spread = _oracle_spread(cfg, ref.t, prompt, seeds=(4,))
    model.reset()
    got = [model.forward_prefill(tokens, 0), model.forward(123, 512)]
    for what, g, w, sp in zip(("prompt of 512", "step after the prompt"), got, want, np.maximum.accumulate(spread)):
        assert np.isfinite(g).all()
        assert rel_l2(g, w) <= max(LOGITS_REL_L2, 3.0 * sp), f"{what}: rel-L2 {rel_l2(g, w):.2e}, the oracle's own spread is {sp:.2e}"
        assert cosine(g, w) >= LOOSE_COSINE
        assert int(np.argmax(w)) in np.argsort(g)[-2:].tolist()
    model.free()


def test_lfm2_1p2b_wide_layers(ctx, oracle, tmp_path):
    """Three layers (gated conv, attention, gated conv) of the LFM2-1.2B's widths -- hidden 2048, FFN 6912, 32 / 8 heads of 64 --
    over a 4096-entry vocabulary: what the 350M shape does not reach as a composition (the conv fused into its out projection
    at the widest hidden size that kernel takes, the gated gate / up kernel at k = 2048, the down projection's 108 block pairs
    per row, 32-head attention, the prompt pass's K split at k = 6912).  Four decode steps, a 200-token prompt, a step after it;
    held to the oracle's own spread under a two-ulp jitter of its f32 sums, like the 350M-shaped model."""
    model, ref, cfg = load(ctx, oracle, tmp_path, context=512, n_layers=3, hidden=2048, inter=6912, n_heads=32, kv_heads=(0, 8, 0), vocab=4096,
                           sigma=0.02, seed=12)
    steps = [5, 77, 1000, 4095]

    def decode(r):
        st = r.new_state()
        return [r.forward(t, p, st) for p, t in enumerate(steps)]

    want, spread = _oracle_spread(cfg, ref.t, decode, seeds=(1, 2, 3))
    allowed = np.maximum.accumulate(spread)
    for pos, tok in enumerate(steps):
        got = model.forward(tok, pos)
        err = rel_l2(got, want[pos])
        assert np.isfinite(got).all()
        assert err <= max(LOGITS_REL_L2, 2.0 * allowed[pos]), f"pos {pos}: rel-L2 {err:.2e}, the oracle's own spread is {allowed[pos]:.2e}"
        assert cosine(got, want[pos]) >= LOOSE_COSINE
    assert spread.max() <= LOOSE_REL_L2, "the jittered oracle itself leaves the loose bar: pick another model seed"
    tokens = np.random.default_rng(12).integers(0, cfg["vocab_size"], 200)

    def prompt(r):
        st = r.new_state()
        for j, t in enumerate(tokens[:-1]):
            r.hidden_after_layers(int(t), j, st)
        return [r.forward(int(tokens[-1]), 199, st), r.forward(123, 200, st)]

    want, spread = _oracle_spread(cfg, ref.t, prompt, seeds=(4,))
    model.reset()
    got = [model.forward_prefill(tokens, 0), model.forward(123, 200)]
    for what, g, w, sp in zip(("prompt of 200", "step after the prompt"), got, want, np.maximum.accumulate(spread)):
        assert np.isfinite(g).all()
        assert rel_l2(g, w) <= max(LOGITS_REL_L2, 3.0 * sp), f"{what}: rel-L2 {rel_l2(g, w):.2e}, the oracle's own spread is {sp:.2e}"
        assert cosine(g, w) >= LOOSE_COSINE
    model.free()


def test_cpp_host_mirror_runs_the_model(ctx, oracle, tmp_path):
    """The C++ mirror's RocmLfm2Model (statically linked selftest binary) and this binding drive the same library:
    same greedy tokens from the same GGUF file, and they are the oracle's."""
    import os
    import subprocess

    from conftest import ROOT

    exe = os.path.join(ROOT, "wick_amd", "lib", "host_selftest")
    assert os.path.exists(exe), "host_selftest has not been built (make -C wick_amd/csrc)"
    kw = dict(hidden=256, inter=256, vocab=256, seed=26)
    img, cfg, tensors = lfm2_synth.build(oracle, **kw)
    path = tmp_path / "model.gguf"
    path.write_bytes(img)
    out = subprocess.run([exe, str(path)], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and "selftest OK" in out.stdout, out.stdout + out.stderr
    lines = dict(l.split(":", 1) for l in out.stdout.splitlines() if ":" in l)
    got = [int(t) for t in lines["tokens"].split()]
    ref, state, tok, want = L.Lfm2Oracle(cfg, tensors), None, 17, []
    state = ref.new_state()
    for pos in range(10):
        tok = L.argmax(ref.forward(tok, pos, state))
        want.append(tok)
    assert got == want
    a, b = lines["prefill"].split()
    assert a == b


def test_greedy_run_across_the_change_of_step_graphs(ctx, oracle, tmp_path):
    """A run that passes the position from which the merge of the attention partials is a launch of its own: the second graph of the
    step is captured between two of its tokens (first run) or is there already (second), and the picks are those of steps
    enqueued launch by launch."""
    model, _, cfg = load(ctx, oracle, tmp_path, context=1100, n_layers=2, hidden=512, inter=512, n_heads=8, kv_heads=(4, 0), vocab=320, seed=8)
    start = np.random.default_rng(3).standard_normal(model.snapshot_state(1018).size // 4).astype(np.float32).view(np.uint8)
    picks = []
    for graphs in (True, True, False):
        model.set_graph_replay(graphs)
        model.restore_state(start, 1018)
        picks.append(model.generate_greedy(7, 1018, 12))
    assert np.array_equal(picks[0], picks[2]) and np.array_equal(picks[1], picks[2])
    model.free()


@pytest.mark.parametrize("wtype", [W.Q4_0, W.Q8_0])
def test_a_prompt_is_the_same_on_either_block_loop(ctx, oracle, tmp_path, wtype):
    """Prompts on both sides of the token counts at which a pass takes other launches (gate | up with the gate in its epilogue, one granule
    per workgroup or on tiles; K shares side by side, on one granule per workgroup, 64-row or 128-row tiles): logits and state are bit for
    bit those of the 16x16x32 kernels, which take the separate launches throughout."""
    model, _, _ = load(ctx, oracle, tmp_path, context=320, n_layers=2, hidden=512, inter=2304, n_heads=8, kv_heads=(0, 2), vocab=256, wtype=wtype, embd_type=W.Q8_0)
    tokens = np.random.default_rng(3).integers(0, 256, 300).astype(np.uint32)
    try:
        for n in (9, 16, 17, 32, 33, 48, 49, 64, 65, 129, 300):
            got = []
            for shape in (32, 16):
                ctx.set_gemm_mfma_shape(shape)
                model.reset()
                got.append((model.forward_prefill(tokens[:n], 0), model.snapshot_state(n)))
            assert np.array_equal(got[0][0].view(np.uint32), got[1][0].view(np.uint32)), f"{n} tokens: logits"
            assert np.array_equal(got[0][1], got[1][1]), f"{n} tokens: state"
    finally:
        ctx.set_gemm_mfma_shape(32)
        model.free()


@pytest.mark.parametrize("hidden,inter", [(128, 1152), (640, 128), (1152, 640), (128, 1952), (1152, 1152)])
def test_short_prompts_at_the_edges_of_their_tiles(ctx, oracle, tmp_path, hidden, inter):
    """The few-token launches on both sides of their 16-token tiles, gate | up in one launch among them, over 1, 5 and 9 slabs of K (fewer than
    their ring of stages holds, one more, and twice round), and over several tiles of 32 and 64 tokens: bit for bit the 16x16x32 kernels, which take
    none of them."""
    model, _, _ = load(ctx, oracle, tmp_path, context=512, n_layers=2, hidden=hidden, inter=inter, n_heads=hidden // 64, kv_heads=(0, 2), vocab=256, embd_type=W.Q8_0)
    tokens = np.random.default_rng(5).integers(0, 256, 449).astype(np.uint32)
    try:
        for n in (10, 15, 31, 34, 47, 63, 65, 97, 130, 449):
            got = []
            for shape in (32, 16):
                ctx.set_gemm_mfma_shape(shape)
                model.reset()
                got.append(model.forward_prefill(tokens[:n], 0).view(np.uint32))
            assert np.array_equal(*got), f"{n} tokens"
    finally:
        ctx.set_gemm_mfma_shape(32)
        model.free()


def on_either_block_loop(ctx, model, tokens):
    """The logits and the state behind a prompt, bit for bit the same on the 16x16x32 kernels, which run every layer for all tokens, the gate in a
    launch of its own."""
    got = []
    try:
        for shape in (32, 16):
            ctx.set_gemm_mfma_shape(shape)
            model.reset()
            got.append((model.forward_prefill(tokens, 0).view(np.uint32), model.snapshot_state(tokens.size)))
    finally:
        ctx.set_gemm_mfma_shape(32)
    assert all(np.array_equal(a, b) for a, b in zip(*got)), f"{tokens.size} tokens"
    return got[0][0].view(np.float32)


@pytest.mark.parametrize("gate_sigma", [0.08, 0.45, 8.0])
def test_gates_of_all_sizes_on_the_tile_of_eight_waves(ctx, oracle, tmp_path, gate_sigma):
    """Gate | up of 1952 rows over 449 tokens and five slabs of K, gates of 25 gate_sigma: a launch whose silu takes gates below 41 in a shorter way, for a
    wave's 1024 of them together; all of them inside, a few outside in some waves, most outside in all."""
    model, _, _ = load(ctx, oracle, tmp_path, context=512, n_layers=2, hidden=640, inter=1952, n_heads=10, kv_heads=(0, 2), vocab=256, embd_type=W.Q8_0, gate_sigma=gate_sigma)
    try:
        assert np.isfinite(on_either_block_loop(ctx, model, np.random.default_rng(11).integers(0, 256, 449).astype(np.uint32))).all()
    finally:
        model.free()


@pytest.mark.parametrize("kv_heads", [(2, 0), (0, 2)])
def test_the_last_token_alone_is_the_whole_layer(ctx, oracle, tmp_path, kv_heads):
    """The last layer's feed-forward block as products of one token, behind a convolution and behind attention, with the K shares of the products over
    all tokens: none of 4 slabs, eight of 32 (up to 128 tokens), four of 32 from 64 tiles of 128 x 128 on."""
    model, _, _ = load(ctx, oracle, tmp_path, context=2048, n_layers=2, hidden=512, inter=4096, n_heads=8, kv_heads=kv_heads, vocab=256, embd_type=W.Q8_0)
    tokens = np.random.default_rng(13).integers(0, 256, 2000).astype(np.uint32)
    try:
        for n in (65, 128, 2000):
            on_either_block_loop(ctx, model, tokens[:n])
    finally:
        model.free()


@pytest.mark.parametrize("embd_type,hidden", [(W.Q6_K, 1280), (W.Q4_0, 1152), (W.Q8_0, 1152)])
def test_a_prompts_rows_are_the_embeddings(ctx, oracle, tmp_path, embd_type, hidden):
    """Rows past the lookup's 1024 elements, tokens past its groups of four: bit for bit the prompt given as the oracle's rows."""
    kw = dict(n_layers=1, hidden=hidden, inter=256, n_heads=hidden // 64, kv_heads=(2,), vocab=256, embd_type=embd_type)
    model, _, _ = load(ctx, oracle, tmp_path, **kw)
    dtype, _, wb = lfm2_synth.build(oracle, **kw)[2]["token_embd.weight"]
    tokens = np.random.default_rng(7).integers(0, 256, 21).astype(np.uint32)
    tokens[[0, -1]] = 255, 0
    try:
        for n in (3, 4, 21):
            rows = np.stack([L.embed_row(dtype, wb, int(t), hidden) for t in tokens[:n]])
            got = [model.forward_prefill(tokens[:n], 0).view(np.uint32)]
            model.reset()
            got.append(model.forward_prefill_from_embeddings(rows, 0).view(np.uint32))
            model.reset()
            assert np.array_equal(*got), f"{n} tokens"
    finally:
        model.free()


@pytest.mark.parametrize("kv_heads", [(2, 0), (0, 2)])
def test_a_prompt_of_two_passes_is_the_two_prompts(ctx, oracle, tmp_path, kv_heads):
    """A pass that is not the last stops at the last layer's state: the same state and logits as the two passes as prompts of their own."""
    model, _, _ = load(ctx, oracle, tmp_path, context=2200, n_layers=2, hidden=128, inter=128, n_heads=2, kv_heads=kv_heads, vocab=256, embd_type=W.Q8_0)
    tokens = np.random.default_rng(9).integers(0, 256, 2048 + 77).astype(np.uint32)
    try:
        got = [(model.forward_prefill(tokens, 0).view(np.uint32), model.snapshot_state(tokens.size))]
        model.reset()
        model.forward_prefill(tokens[:2048], 0)
        got.append((model.forward_prefill(tokens[2048:], 2048).view(np.uint32), model.snapshot_state(tokens.size)))
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        model.free()
