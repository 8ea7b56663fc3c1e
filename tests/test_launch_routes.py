"""Which kernel a call runs on, at sizes on both sides of the rules that choose it: the library's host code against a pretended HIP
runtime (tests/host/fake_hip.cpp), so that it is seen on the CPU."""
import os
import re

import numpy as np
import pytest

import lfm2_synth
import test_gpu_gemm as gemm
from conftest import ROOT
from lfm2_synth import Q4_0, Q8_0


@pytest.fixture(scope="session")
def routes(host_faults):
    """(calls) -> the kernels of each, e.g. "gemm_tile_kernel<2, false, false, TileX>"; with grids=True, the kernels' grids."""
    def run(*calls, grids=False):
        out = host_faults("routes", *calls)
        out = re.sub(r"wick_rocm::|\(anonymous namespace\)::", "", out)
        kernels = []
        for line in out.splitlines():
            if line.startswith("\t"):
                kernels[-1].append(tuple(map(int, re.search(r" \((\d+) x (\d+)\)$", line).groups())) if grids else re.sub(r"^void |\(.*$", "", line.strip()))
            else:
                kernels.append([])
        assert len(kernels) == len(calls), out
        return kernels

    return run


def short(kernels):
    """The same as test_gpu_gemm.py names them."""
    names = []
    for k in kernels:
        name, args = re.match(r"gemm_(\w+)_kernel<(.*)>$", k).groups()
        args = args.split(", ")
        names.append({"few": f"few {' '.join(args[3:])}", "narrow": f"narrow {args[-1]}", "tile": args[-1], "splitk_reduce": f"in {args[0]}"}[name])
    return ", ".join(names)


def test_the_sides_of_every_launch_rule_are_on_their_kernels(routes):
    calls = [f"gemm {m} {n} {k} {splits}" for m, n, k in gemm.EDGES for splits in (0, 1)]
    got = [short(k) for k in routes(*calls)]
    assert dict(zip(gemm.EDGES, zip(got[::2], got[1::2]))) == gemm.EDGES


def test_the_ragged_launches_are_on_every_tile(routes):
    for tiles in (gemm.PROMPT_TILES, gemm.RAGGED_TILES):
        for splits in (0, 1):
            assert {s: short(k) for s, k in zip(tiles, routes(*(f"gemm {m} {n} {k} {splits}" for m, n, k in tiles)))} == tiles
    gated = gemm.RAGGED_GATED_TILES
    kernels = routes(*(f"gate_up {m} {n} {k}" for m, n, k in gated))
    assert {s: short(k) for s, k in zip(gated, kernels)} == gated and all("<2, false, true, " in k for k, in kernels)
    with open(os.path.join(ROOT, "wick_amd", "csrc", "gemm.hip")) as f:
        plain, with_gate = (set(t.split(", ")) for t in re.findall(r"cheapest_tile<(Tile\w, [^>]*)>", f.read()))
    # (TileN with the gate is for fewer workgroups than the public launch takes: prompts reach it, see below)
    assert plain == set(gemm.RAGGED_TILES.values()) and with_gate == set(gated.values()) | {"TileN"}


def test_prompts_on_the_few_token_kernel(routes):
    calls = [f"gemm {m} {n} {k} {splits}" for m, n, k in gemm.FEW_TILES for splits in (0, 1)]
    got = [short(k) for k in routes(*calls)]
    assert dict(zip(gemm.FEW_TILES, zip(got[::2], got[1::2]))) == gemm.FEW_TILES


@pytest.mark.parametrize("m,n,k,even", [(1056, 832, 1024, False), (1312, 768, 1024, False), (1568, 300, 2048, False), (5408, 130, 2688, False),
                                        (1024, 832, 384, True), (2208, 200, 1024, True), (544, 300, 1024, True), (7712, 128, 1024, True)])
def test_few_token_tiles_are_even_over_the_xcds(routes, m, n, k, even):
    """Workgroup i of a launch goes to XCD i % 8.  A granule's token tiles share an XCD unless that takes one of its 32 CUs another workgroup."""
    (x, y), = routes(f"gemm {m} {n} {k} 1", grids=True)[0]
    granules = -(-m // 32)
    on = [sum(i + x * j & 7 == xcd for i in range(granules) for j in range(y)) for xcd in range(8)]
    assert x in (granules, -(-granules // 8) * 8) and (x % 8 == 0) == even
    assert -(-max(on) // 32) == -(-(-(-granules * y // 8)) // 32)


@pytest.mark.parametrize("m,n,k,shares", [(1344, 163, 7040, 4), (192, 635, 3968, 8), (32, 100, 2048, 8), (512, 200, 4608, 8)])
def test_shares_leave_no_granules_of_workgroups_without_work(routes, m, n, k, shares):
    call = f"gemm {m} {n} {k} 8"
    assert routes(call) == [["gemm_few_kernel<2, false, false, %s>" % ("1, 4" if m == 32 else "2, 8"), f"gemm_splitk_reduce_kernel<{shares}>"]]
    assert routes(call, grids=True)[0][0][0] == -(-(-(-m // 32) * shares) // 8) * 8


@pytest.mark.parametrize("dim,quads", [(32, 1), (1024, 1), (1056, 2), (2048, 2), (2080, 0), (2304, 0), (4096, 0), (8192, 0), (8224, 0)])
def test_the_norm_keeps_short_rows_only(routes, dim, quads):
    """Rows past 2048 elements are read a second time: kept, they would leave the CU four workgroups."""
    assert routes(f"norm 30 {dim}") == [[f"rmsnorm_quantize_kernel<0, {quads}>"]]


class Zeros:
    """Weights for a model whose kernels do not run."""

    @staticmethod
    def synth_weight(ggml_type, m, k, seed, sigma):
        per, size = {Q4_0: (32, 18), Q8_0: (32, 34)}[ggml_type]
        return np.zeros(m * k // per * size, np.uint8)


@pytest.mark.parametrize("inter,hidden,tokens,gated", [
    (1024, 1024, 23, True), (1024, 1152, 23, True),
    (2048, 1280, 32, True), (3040, 2816, 32, True), (3040, 2944, 32, False),  # 22 slabs of K
    (3072, 2944, 24, True), (4096, 4096, 9, True), (4096, 4224, 9, False),    # 32 from 3072 rows on
    (4128, 4224, 24, True), (4128, 2944, 25, True),    # past 256 granules of both
    (8192, 3200, 32, True),                            # 512
    (8224, 1024, 23, False),                           # 257 granules
    (4608, 1024, 32, True), (4608, 1024, 33, True),    # 32 tokens
    (2048, 1408, 33, True), (2048, 1536, 33, False),   # 11 slabs above them
    (4096, 1408, 64, True), (4096, 1536, 64, False),
    (4128, 1536, 64, True),                            # past 256 granules of both
])
def test_few_tokens_take_the_gate_into_the_launch_while_k_is_short(routes, tmp_path, inter, hidden, tokens, gated):
    """A prompt's gate | up over up to 64 tokens: one launch, or the projections and the gate behind them."""
    path = tmp_path / "model.gguf"
    path.write_bytes(bytes(lfm2_synth.build(Zeros, n_layers=1, hidden=hidden, inter=inter, n_heads=hidden // 64, kv_heads=(0,), embd_type=Q8_0)[0]))
    kernels, = routes(f"prompt {path} {tokens}")
    assert (f"gemm_few_kernel<2, false, true, {1 if tokens <= 32 else 2}, 8>" in kernels) == gated
    assert ("silu_mul_quantize_kernel" not in kernels) == gated


@pytest.mark.parametrize("tokens,kernel", [(200, "few_kernel<2, false, false, 2, 8>"),  # 512 tiles of 64 tokens, four shares
                                           (255, "few_kernel<2, false, false, 2, 8>"), (257, "few_kernel<2, false, false, 1, 4>"),  # 8 slabs, 256 x 1024 outputs
                                           (512, "few_kernel<2, false, false, 2, 8>"), (513, "tile_kernel<2, false, false, TileH>"), (1000, "tile_kernel<2, false, false, TileN>")])
def test_residual_projections_of_a_prompt(routes, tokens, kernel):
    """Shares of K that the norm behind adds up: side by side on the few-token kernel, walked by it, on the tiles."""
    assert routes(f"residual 1024 {tokens} 1024 8")[0][0] == f"gemm_{kernel}"


@pytest.mark.parametrize("hidden,inter,tokens,kernel", [
    (1024, 3584, 65, "few_kernel<2, false, true, 1, 8>"), (1024, 3584, 128, "few_kernel<2, false, true, 1, 8>"),  # 448 tiles of 32 tokens
    (1024, 2048, 280, "few_kernel<2, false, true, 2, 8>"), (1024, 2048, 281, "tile_kernel<2, false, true, TileN>"),  # 256 of 64
    (1024, 4096, 256, "tile_kernel<2, false, true, TileN>"), (1024, 4096, 257, "tile_kernel<2, false, true, TileS>"),  # 256 tiles of 64 rows
    (640, 1952, 449, "tile_kernel<2, false, true, TileN>"),  # 5 slabs
    (2048, 4096, 160, "few_kernel<2, false, true, 2, 8>"), (2048, 4096, 161, "tile_kernel<2, false, true, TileN>"),  # 1280 of 16 tokens
])
def test_prompts_take_the_gate_into_the_few_token_kernel(routes, tmp_path, hidden, inter, tokens, kernel):
    path = tmp_path / "model.gguf"
    path.write_bytes(bytes(lfm2_synth.build(Zeros, n_layers=2, hidden=hidden, inter=inter, n_heads=hidden // 64, kv_heads=(0, 0), embd_type=Q8_0)[0]))
    kernels, = routes(f"prompt {path} {tokens}")
    assert f"gemm_{kernel}" in kernels and "silu_mul_quantize_kernel" not in kernels


def test_the_last_layer_is_for_the_last_token(routes, tmp_path):
    """Past 64 tokens its feed-forward block is a product of one token, and a pass that is not the last one does without."""
    path = tmp_path / "model.gguf"
    path.write_bytes(bytes(lfm2_synth.build(Zeros, n_layers=1, hidden=1024, inter=1024, n_heads=16, kv_heads=(0,), embd_type=Q8_0)[0]))
    short, long, passes = routes(f"prompt {path} 64", f"prompt {path} 65", f"prompt {path} 2113")
    gated, one = "gemm_few_kernel<2, false, true, 2, 8>", "gemm_few_kernel<2, false, true, 1, 8>"
    assert gated in short and one not in short and gated not in long and one in long
    assert passes[-len(long) + 3:] == long[3:] and len(passes) < 2 * len(long) and passes.count(one) == 1


def test_the_last_token_has_room_for_its_norm(routes, tmp_path):
    """A row of hidden elements longer than all gated rows of the prompt together: the norm in front of the last token's feed-forward block
    stays in its buffers (the pretended runtime looks)."""
    path = tmp_path / "model.gguf"
    path.write_bytes(bytes(lfm2_synth.build(Zeros, n_layers=1, hidden=8448, inter=128, n_heads=132, kv_heads=(2,), embd_type=Q8_0)[0]))
    kernels, = routes(f"prompt {path} 65")
    assert "gemm_few_kernel<2, false, true, 1, 8>" in kernels


def test_arguments_in_front_of_a_struct_are_no_pointers(host_faults, tmp_path):
    """The fields that a kernel takes once more, to have them in registers when it starts: numbers, which the runtime does not look up at every launch."""
    path = tmp_path / "model.gguf"
    path.write_bytes(bytes(lfm2_synth.build(Zeros, n_layers=2, hidden=1024, inter=4608, n_heads=16, kv_heads=(0, 2), embd_type=Q8_0)[0]))
    out = host_faults("routes", *(f"prompt {path} {n}" for n in (23, 128, 555)))
    found = re.findall(r"(gemm_few|gemm_tile|qk_norm_rope_tokens64|attention_prefill_f16x3)_kernel<.*>\((.*?)(?:wick_rocm::\(anonymous namespace\)::)?\w+Args", out)
    assert {name for name, _ in found} == {"gemm_few", "gemm_tile", "qk_norm_rope_tokens64", "attention_prefill_f16x3"}
    assert [(name, args) for name, args in found if "*" in args or "unsigned int" not in args] == []
