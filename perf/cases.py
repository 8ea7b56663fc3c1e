"""What a program built on this backend spends its time on, as cases that can be timed: single projections over one f32
activation (a decode step's GEMVs, the LM head), batched projections (a prompt's GEMMs), and the LFM2 model handle at work --
prompts, greedy and sampled decoding, the session state -- over the sizes, weight types and cache types it is used with."""
import math

import numpy as np
import torch

import wick_amd as W
from wick_amd import gguf as G
from wick_amd.lfm2 import RocmLfm2Model

TYPES = {"q4_0": W.Q4_0, "q8_0": W.Q8_0, "q6_k": W.Q6_K}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q6_k": (256, 210)}
HEAD_DIM, VOCAB = 64, 65536

# The two sizes of the LFM2 family that bench.py runs: hidden size, FFN size, width of a key row, layers, which of them are
# attention layers (the others are gated convolutions).  The larger one is cut to its first six layers, so that making it stays short.
MODELS = {
    "350m": {"hs": 1024, "inter": 4608, "kv": 512, "layers": 16, "attn": (2, 5, 8, 10, 12, 14)},
    "1p2b": {"hs": 2048, "inter": 6912, "kv": 512, "layers": 6, "attn": (2, 5)},
}
BODIES = {"q4_0": "q6_k", "q8_0": "q8_0"}  # body type -> type of the tied embedding, as shipped files pair them


def listed():
    return [
        # the smaller model's Q, K and V projections in one call: about the smallest there is, all launch and latency
        {"name": "gemv_q4_0_qkv_1024", "kind": "gemv", "type": "q4_0", "m": 1024, "k": 1024, "kv": 512},
        # the larger model's LM head over one token: the largest single read of a step
        {"name": "gemv_q8_0_65536x2048", "kind": "gemv", "type": "q8_0", "m": 65536, "k": 2048, "kv": 0},
        # a down projection over a short prompt: few tokens, long rows
        {"name": "gemm_q4_0_2048x6912_n37", "kind": "gemm", "type": "q4_0", "m": 2048, "k": 6912, "n": 37},
        # an FFN projection over a whole prompt, the benchmark's GEMM
        {"name": "gemm_q4_0_6912x2048_n2002", "kind": "gemm", "type": "q4_0", "m": 6912, "k": 2048, "n": 2002},
        # greedy generation right behind a short prompt
        {"name": "greedy_350m_pos30", "kind": "decode", "model": "350m", "body": "q4_0", "f16": False, "pos": 30, "n": 24, "greedy": True},
        # sampled generation: every step's logits go to the host, where the sampler is
        {"name": "sampled_350m_pos1500", "kind": "decode", "model": "350m", "body": "q4_0", "f16": False, "pos": 1500, "n": 8, "greedy": False},
        # greedy generation far into a long context, on half-precision caches
        {"name": "greedy_350m_f16_pos20000", "kind": "decode", "model": "350m", "body": "q4_0", "f16": True, "pos": 20000, "n": 12, "greedy": True},
        # a chat turn: a few tokens onto an existing context
        {"name": "prompt_350m_n23_at700", "kind": "prompt", "model": "350m", "body": "q4_0", "f16": False, "pos": 700, "n": 23},
        # an ordinary prompt
        {"name": "prompt_350m_n555", "kind": "prompt", "model": "350m", "body": "q4_0", "f16": False, "pos": 0, "n": 555},
        # a long prompt through the larger model on 8-bit weights
        {"name": "prompt_1p2b_q8_0_n2002", "kind": "prompt", "model": "1p2b", "body": "q8_0", "f16": False, "pos": 0, "n": 2002},
        # a document: several passes, attention over everything before
        {"name": "prompt_350m_f16_n9000", "kind": "prompt", "model": "350m", "body": "q4_0", "f16": True, "pos": 0, "n": 9000},
        # a session taken up from its stored state, shifted to make room, and stored again
        {"name": "state_350m_n3000", "kind": "state", "model": "350m", "body": "q4_0", "f16": False, "n": 3000, "keep": 64, "shift": 800},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemm", "decode", "decode", "prompt", "prompt", "state"])
    if kind in ("gemv", "gemm"):
        t = rng.choice(["q4_0", "q8_0", "q6_k"] if kind == "gemv" else ["q4_0", "q8_0"])
        step = {"gemv": BLOCK[t][0], "gemm": 128}[kind]
        k = max(step, _log(rng, 256, 8192) // step * step)
        if kind == "gemv":
            m = min(_log(rng, 64, 65536), (140 << 20) * BLOCK[t][0] // BLOCK[t][1] // k)
            return {"kind": kind, "type": t, "m": m, "k": k, "kv": m // 4 if m < 8192 and rng.random() < 0.4 else 0}
        n = _log(rng, 2, 4096)
        return {"kind": kind, "type": t, "m": min(_log(rng, 64, 16384), int(1.2e11 / (2 * n * k))), "k": k, "n": n}
    c = {"kind": kind, "model": rng.choice(["350m", "350m", "1p2b"]), "body": rng.choice(["q4_0", "q4_0", "q8_0"]), "f16": rng.random() < 0.5}
    if kind == "decode":
        c.update(pos=_log(rng, 8, 20000), n=rng.randint(4, 24), greedy=rng.random() < 0.5)
    elif kind == "prompt":
        pos = 0 if rng.random() < 0.6 else _log(rng, 16, 2000)
        c.update(pos=pos, n=_log(rng, 3, (9000 if c["model"] == "350m" else 6000) - pos))
    else:
        n = _log(rng, 100, 4000)
        shift = rng.randint(1, n // 2)
        c.update(n=n, keep=rng.randint(0, n - shift - 1), shift=shift)
    return c


# ---- inputs ----------------------------------------------------------------------------------

_CTX = []


def _context():
    if not _CTX:  # one context per program, as the host has it
        _CTX.append(W.RocmContext(0))
    return _CTX[0]


def _blocks(gen, t, m, k, sigma):
    """m x k weights ~ N(0, sigma^2) (Q6_K: uniform quants of that spread) as quantized blocks, host bytes."""
    n = m * k // BLOCK[t][0]
    if t == "q6_k":
        b = torch.randint(0, 256, (n, 210), generator=gen, device="cuda", dtype=torch.uint8)
        b[:, 192:208] = torch.randint(24, 56, (n, 16), generator=gen, device="cuda", dtype=torch.uint8)  # sub-block scales
        b[:, 208:] = torch.full((n, 1), sigma / (18.5 * 40.0), device="cuda", dtype=torch.float16).view(torch.uint8)
        return b.cpu().numpy()
    x = torch.randn(n, 32, generator=gen, device="cuda") * sigma
    at = x.abs().argmax(1, keepdim=True)
    top = x.gather(1, at)
    if t == "q4_0":
        d = (top / -8.0).half()
        q = torch.clamp(x / d.float() + 8.5, 0, 15).to(torch.uint8)
        q = q[:, :16] | (q[:, 16:] << 4)
    else:
        d = (top.abs() / 127.0).half()
        q = torch.clamp(torch.round(x / d.float()), -127, 127).to(torch.int8).view(torch.uint8)
    return torch.cat([d.view(torch.uint8).reshape(n, 2), q], 1).cpu().numpy()


def _image(gen, c):
    """A randomly initialised model as a GGUF image: projections of unit gain, embedding rows a tenth of what the layers add."""
    s = MODELS[c["model"]]
    hs, inter, kv, hd = s["hs"], s["inter"], s["kv"], HEAD_DIM
    body, embd, tensors = c["body"], BODIES[c["body"]], []

    def quant(name, t, m, k, sigma):
        tensors.append((name, [k, m], TYPES[t], _blocks(gen, t, m, k, sigma)))

    def f32(name, dims, center, spread):
        v = center + spread * torch.randn(int(np.prod(dims)), generator=gen, device="cuda")
        tensors.append((name, list(dims), 0, v.cpu().numpy()))

    quant("token_embd.weight", embd, VOCAB, hs, 0.3)
    f32("token_embd_norm.weight", [hs], 1.0, 0.1)
    for i in range(s["layers"]):
        p, unit = "blk.%d." % i, hs ** -0.5
        f32(p + "attn_norm.weight", [hs], 1.0, 0.1)
        f32(p + "ffn_norm.weight", [hs], 1.0, 0.1)
        if i in s["attn"]:
            for name, m in (("attn_q", hs), ("attn_k", kv), ("attn_v", kv), ("attn_output", hs)):
                quant(p + name + ".weight", body, m, hs, unit)
            f32(p + "attn_q_norm.weight", [hd], 1.0, 0.1)
            f32(p + "attn_k_norm.weight", [hd], 1.0, 0.1)
        else:
            quant(p + "shortconv.in_proj.weight", body, 3 * hs, hs, unit)
            quant(p + "shortconv.out_proj.weight", body, hs, hs, unit)
            f32(p + "shortconv.conv.weight", [3, hs], 0.0, 0.5)
        quant(p + "ffn_gate.weight", body, inter, hs, unit)
        quant(p + "ffn_up.weight", body, inter, hs, unit)
        quant(p + "ffn_down.weight", body, hs, inter, inter ** -0.5)
    meta = [("general.architecture", G.T_STRING, "lfm2"), ("lfm2.block_count", G.T_U32, s["layers"]), ("lfm2.embedding_length", G.T_U32, hs),
            ("lfm2.feed_forward_length", G.T_U32, inter), ("lfm2.attention.head_count", G.T_U32, hs // hd), ("lfm2.vocab_size", G.T_U32, VOCAB),
            ("lfm2.rope.freq_base", G.T_F32, 1000000.0), ("lfm2.attention.layer_norm_rms_epsilon", G.T_F32, 1e-5), ("lfm2.shortconv.l_cache", G.T_U32, 3),
            ("lfm2.attention.head_count_kv", G.T_ARRAY, (G.T_I32, [kv // hd if i in s["attn"] else 0 for i in range(s["layers"])]))]
    return G.build_image(meta, tensors)


def _stored(gen, model, n):
    """A stored session state of n positions: normed keys and values of unit spread, conv inputs."""
    parts = []
    for i, kv in enumerate(model.kv_heads_per_layer):
        size = model.layer_state_bytes(i, n)
        half = kv and model.kv_f16
        v = torch.randn(size // (2 if half else 4), generator=gen, device="cuda")
        parts.append((v.half() if half else v).cpu().numpy().view(np.uint8))
    return np.concatenate(parts)


class _State:
    """What one program has in hand; gives its device memory back when it goes."""

    def __init__(self, case):
        self.case, self.ctx, self.model, self.weights = case, _context(), None, []

    def __del__(self):
        if self.model is not None:
            self.model.free()
        for w in self.weights:
            w.free()


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    st = _State(case)
    if case["kind"] in ("gemv", "gemm"):
        m, k, n = case["m"], case["k"], case.get("n", 1)
        kv = case.get("kv", 0)
        for rows in (m, kv, kv) if kv else (m,):
            st.weights.append(st.ctx.upload_weight(_blocks(gen, case["type"], rows, k, k ** -0.5), TYPES[case["type"]], rows, k))
        st.x = torch.randn(n, k, generator=gen, device="cuda")
        st.ys = [torch.zeros(n, w.m, device="cuda") for w in st.weights]
        torch.cuda.synchronize()
        return st
    pos, n = case.get("pos", 0), case["n"]
    with G.GgufFile.from_bytes(_image(gen, case)) as g:
        st.model = RocmLfm2Model(st.ctx, g, (pos + n + 255) // 256 * 256, kv_f16=case["f16"])
    st.tokens = torch.randint(0, VOCAB, (n,), generator=gen, device="cuda").cpu().numpy().astype(np.uint32)
    if case["kind"] == "state":
        st.stored = _stored(gen, st.model, n)
    elif pos:
        st.model.restore_state(_stored(gen, st.model, pos), pos)
    if case["kind"] == "prompt":  # a program serves more than one prompt: the handle's prompt buffers exist
        st.model.forward_prefill(st.tokens[:3], pos)
    torch.cuda.synchronize()
    return st


def run(st):
    c = st.case
    if c["kind"] == "gemv":
        if c["kv"]:
            st.ctx.encode_gemv_fused(st.weights, st.x.data_ptr(), 0, [y.data_ptr() for y in st.ys])
        else:
            st.ctx.encode_gemv(st.weights[0], st.x.data_ptr(), 0, st.ys[0].data_ptr(), 0)
        return st.ys
    if c["kind"] == "gemm":
        st.ctx.encode_gemm(st.weights[0], st.x.data_ptr(), 0, st.ys[0].data_ptr(), 0, c["n"], c["k"], c["m"])
        return st.ys
    model = st.model
    if c["kind"] == "decode":
        if c["greedy"]:
            return model.generate_greedy(int(st.tokens[0]), c["pos"], c["n"])
        return [model.forward(int(t), c["pos"] + i) for i, t in enumerate(st.tokens)]
    if c["kind"] == "prompt":
        if c["pos"] == 0:
            model.reset()
        return model.forward_prefill(st.tokens, c["pos"])
    model.restore_state(st.stored, c["n"])
    return model.snapshot_state(model.shift_kv(c["n"], c["keep"], c["shift"]))


# ---- what a pass cannot do without -------------------------------------------------------------

def work(case):
    if case["kind"] in ("gemv", "gemm"):
        per, size = BLOCK[case["type"]]
        m, k, n = case["m"] + 2 * case.get("kv", 0), case["k"], case.get("n", 1)
        return {"bytes": m * k // per * size + 4 * n * k + 4 * n * m, "flops": 2 * m * k * n}
    s = MODELS[case["model"]]
    hs, inter, kv = s["hs"], s["inter"], s["kv"]
    n_attn = len(s["attn"])
    n_conv = s["layers"] - n_attn
    row = 2 * kv * (2 if case["f16"] else 4) * n_attn  # one position's keys and values, all layers
    n, pos = case["n"], case.get("pos", 0)
    if case["kind"] == "state":
        stored = n * row + n_conv * 2 * hs * 4
        moved = (n - case["keep"] - case["shift"]) * row
        return {"bytes": 2 * stored + 2 * moved + 2 * (stored - case["shift"] * row), "flops": 0}
    body = n_conv * 4 * hs * hs + n_attn * (2 * hs * hs + 2 * kv * hs) + s["layers"] * 3 * hs * inter
    head = hs * VOCAB
    per, size = BLOCK[case["body"]]
    hper, hsize = BLOCK[BODIES[case["body"]]]
    weights, seen = body // per * size, n * pos + n * (n + 1) // 2
    attn = 4 * hs * n_attn * seen
    if case["kind"] == "decode":
        return {"bytes": n * (weights + head // hper * hsize + (0 if case["greedy"] else 8 * VOCAB)) + row * seen, "flops": 2 * n * (body + head) + attn}
    return {"bytes": weights + head // hper * hsize + row * (pos + 2 * n) + 4 * VOCAB, "flops": 2 * n * body + 2 * head + attn}


def tolerance(case):
    if case["kind"] in ("gemv", "gemm"):
        return {"rel": 1e-5, "max": 1e-4}  # exact integer dots per block, f32 sums
    if case["kind"] == "state" or case.get("greedy"):
        return "exact"
    # Logits behind a model whose activations are rounded to 8 bits in front of every projection: a sum that differs in its last
    # bit now and then lands on the other side of a rounding step, which moves that projection's result by 1e-3 of itself.
    return {"rel": 1e-2, "max": 0.1}
