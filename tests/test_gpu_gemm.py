"""Batched prefill GEMM on the GPU against the oracle, both output layouts, both
kernel paths (multi-token GEMV below the hand-off n or when k % 128 != 0; int8 MFMA
otherwise).  Block dots BIT-EXACT, f32 within rel-L2 1e-5 / max-abs 1e-4 x RMS."""
import numpy as np
import pytest

import wick_amd as W
from conftest import assert_f32_parity, rel_l2
from gpu_util import Problem, fetch_gemm
from test_oracle_matmul import ref_inputs, ref_weights

pytestmark = pytest.mark.gpu

# (m, n, k)
SHAPES = [
    (8, 1, 64), (8, 5, 64), (8, 7, 64), (8, 8, 64), (8, 11, 64), (8, 16, 64),  # the reference's own test shapes
    (4, 1, 32), (64, 4, 32), (64, 20, 96), (33, 3, 2080),                        # generic path
    (64, 2, 256), (100, 15, 512),                                                # multi-token GEMV
    (128, 16, 256), (128, 128, 256), (1, 16, 256), (130, 129, 512), (200, 50, 512), (256, 300, 1024),
    (512, 100, 2048), (1000, 257, 4608), (300, 64, 6912),                        # MFMA, ragged tiles
    (129, 17, 128), (16, 33, 256), (250, 63, 384), (131, 64, 1024), (257, 65, 512),  # narrow kernel (n <= 64) and its hand-off
]


@pytest.mark.parametrize("dtype", [W.Q4_0, W.Q8_0])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_parity(ctx, oracle, dtype, m, n, k):
    with Problem(ctx, oracle, dtype, m, k, n, seed=m + 5 * n + 11 * k + dtype) as p:
        ref = oracle.gemm_q8(dtype, p.wb, p.s, p.q, m, n, k)
        for layout, stride in ((W.LAYOUT_ROW_MAJOR, n), (W.LAYOUT_TOKEN_MAJOR, m), (W.LAYOUT_ROW_MAJOR, n + 3), (W.LAYOUT_TOKEN_MAJOR, m + 5)):
            rows = m if layout == W.LAYOUT_ROW_MAJOR else n
            d_y = p.to_device(np.full(rows * stride, -7.0, np.float32))
            ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, y_stride=stride, layout=layout)
            assert_f32_parity(fetch_gemm(d_y, m, n, stride, layout), ref, f"gemm {dtype} {m}x{n}x{k} layout {layout}")
            # padding between rows is left untouched
            full = d_y.download(np.float32, rows * stride).reshape(rows, stride)
            used = n if layout == W.LAYOUT_ROW_MAJOR else m
            assert np.all(full[:, used:] == -7.0)
        d_d = p.alloc(n * m * (k // 32) * 4)
        ctx.block_dots_i32(p.w, p.d_q, n, d_d)
        dots = d_d.download(np.int32, n * m * (k // 32)).reshape(n, m, k // 32)
        assert np.array_equal(dots, oracle.block_dots_i32(dtype, p.wb, p.q, m, n, k))


# more than 256 wide tiles (fewer run on the narrow tile), ragged in rows and tokens; the fourth is cut over K on the wide tile;
# the last two take the narrow tile (n > 48: both of its block loops exist), the very last one cut over K
WIDE_SHAPES = [(2100, 2010, 128, True), (2100, 1990, 256, False), (4700, 1100, 384, False), (1024, 2002, 4608, False),
               (300, 64, 512, True), (1000, 700, 1024, False)]


@pytest.mark.parametrize("dtype", [W.Q4_0, W.Q8_0])
@pytest.mark.parametrize("m,n,k,with_dots", WIDE_SHAPES)
def test_wide_tile_on_either_mfma_shape(ctx, oracle, dtype, m, n, k, with_dots):
    """The two block loops of the wide tile and of the full narrow tile (32x32x32, the default, and 16x16x32): each against the oracle (two row bands over all
    tokens) in both layouts with ragged strides and with the accumulate flag, block dots bit-exact through either, and the
    two within 1e-6 of each other everywhere."""
    rb = (k // 32) * (18 if dtype == W.Q4_0 else 34)
    bands = [(0, 96), (m - 70, m)]
    with Problem(ctx, oracle, dtype, m, k, n, seed=3 * m + 7 * n + k + dtype) as p:
        refs = [oracle.gemm_q8(dtype, p.wb[r0 * rb:r1 * rb], p.s, p.q, r1 - r0, n, k) for r0, r1 in bands]
        outs = {}
        try:
            for shape in (32, 16):
                ctx.set_gemm_mfma_shape(shape)
                for layout, stride in ((W.LAYOUT_TOKEN_MAJOR, m), (W.LAYOUT_ROW_MAJOR, n + 3), (W.LAYOUT_TOKEN_MAJOR, m + 5)):
                    rows = m if layout == W.LAYOUT_ROW_MAJOR else n
                    d_y = ctx.to_device(np.full(rows * stride, -7.0, np.float32))
                    ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, y_stride=stride, layout=layout)
                    got = fetch_gemm(d_y, m, n, stride, layout)
                    for (r0, r1), ref in zip(bands, refs):
                        assert_f32_parity(got[r0:r1], ref, f"gemm {dtype} {m}x{n}x{k} layout {layout} mfma {shape} rows {r0}..{r1}")
                    full = d_y.download(np.float32, rows * stride).reshape(rows, stride)
                    assert np.all(full[:, (n if layout == W.LAYOUT_ROW_MAJOR else m):] == -7.0)
                    if layout == W.LAYOUT_TOKEN_MAJOR and stride == m:
                        outs[shape] = got
                        ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, y_stride=stride, layout=layout, accumulate=True)  # y += W x
                        twice = fetch_gemm(d_y, m, n, stride, layout)
                        for (r0, r1), ref in zip(bands, refs):
                            assert_f32_parity(twice[r0:r1], 2.0 * ref, f"accumulate, mfma {shape}")
                    d_y.free()
                if with_dots:
                    d_d = p.alloc(n * m * (k // 32) * 4)
                    ctx.block_dots_i32(p.w, p.d_q, n, d_d)
                    dots = d_d.download(np.int32, n * m * (k // 32)).reshape(n, m, k // 32)
                    assert np.array_equal(dots, oracle.block_dots_i32(dtype, p.wb, p.q, m, n, k))
        finally:
            ctx.set_gemm_mfma_shape(0)
        assert rel_l2(outs[16], outs[32]) < 1e-6


def test_mfma_shape_knob_rejects_other_values(ctx):
    with pytest.raises(W.RocmError):
        ctx.set_gemm_mfma_shape(8)
    ctx.set_gemm_mfma_shape(0)


@pytest.mark.parametrize("dtype,n", [(W.Q4_0, 7), (W.Q8_0, 5), (W.Q4_0, 8), (W.Q4_0, 11), (W.Q4_0, 16)])
def test_reference_gemm_vs_gemv_inputs(ctx, oracle, dtype, n):
    """The reference's GEMM == sequential GEMV tests (simd.rs:1440-1623) on their own
    weights/inputs: GPU GEMM column j vs GPU GEMV of column j within the reference's 1e-4."""
    m, k = 8, 64
    wb = oracle.build_matrix(dtype, ref_weights(m, k), m, k)
    s, q = oracle.quantize_q8_0_batch(ref_inputs(n, k), n, k)
    w = ctx.upload_weight(wb, dtype, m, k)
    d_q, d_s = ctx.to_device(q), ctx.to_device(s)
    d_c, d_y = ctx.alloc(m * n * 4), ctx.alloc(m * 4)
    ctx.gemm_preq(w, d_s, d_q, n, d_c, layout=W.LAYOUT_ROW_MAJOR)
    c = d_c.download(np.float32, m * n).reshape(m, n)
    assert_f32_parity(c, oracle.gemm_q8(dtype, wb, s, q, m, n, k), "reference inputs")
    for j in range(n):
        ctx.gemv_with_preq(w, d_s.ptr + j * (k // 32) * 4, d_q.ptr + j * k, d_y)
        assert np.abs(c[:, j] - d_y.download(np.float32, m)).max() < 1e-4
    w.free()
    for b in (d_q, d_s, d_c, d_y):
        b.free()


def test_q8_0_closed_form(ctx, oracle):
    """test_q8_0_gemm_standalone (wick/tests/bench_perf.rs:852-971): m=64, k=32, n=4,
    scale 1/(row+1), quants -16..15, x == 1, x_stride = k, y_stride = m, through the
    f32 call-site entry point."""
    m, k, n = 64, 32, 4
    rows = []
    for r in range(m):
        h = int(np.float16(1.0 / (r + 1.0)).view(np.uint16))
        rows.append(np.concatenate([np.array([h & 0xFF, h >> 8], np.uint8), (np.arange(32) - 16).astype(np.int8).view(np.uint8)]))
    w = ctx.upload_weight(np.concatenate(rows), W.Q8_0, m, k)
    d_x = ctx.to_device(np.ones(n * k, np.float32))
    d_y = ctx.alloc(m * n * 4)
    ctx.encode_gemm(w, d_x, 0, d_y, 0, n, k, m)
    y = d_y.download(np.float32, m * n).reshape(n, m)
    expect = np.array([-16.0 * float(np.float16(1.0 / (r + 1.0))) for r in range(m)]) * 127.0 * float(np.float16(1.0 / 127.0))
    for col in range(n):
        assert np.abs(y[col] - (-16.0 / (np.arange(m) + 1.0))).max() < 1.0  # the reference's bound
        assert np.allclose(y[col], expect, rtol=1e-6)
    w.free(), d_x.free(), d_y.free()


@pytest.mark.parametrize("dtype", [W.Q4_0, W.Q8_0])
@pytest.mark.parametrize("n", [3, 40])
def test_accumulate(ctx, oracle, dtype, n):
    m, k = 256, 512
    with Problem(ctx, oracle, dtype, m, k, n, seed=8) as p:
        y0 = oracle.fill_normal(4, 1.0, n * m)
        d_y = p.to_device(y0)
        ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, layout=W.LAYOUT_TOKEN_MAJOR, accumulate=True)
        ref = y0.reshape(n, m).T.astype(np.float64) + oracle.gemm_q8(dtype, p.wb, p.s, p.q, m, n, k, f64=True)
        assert_f32_parity(fetch_gemm(d_y, m, n, m, W.LAYOUT_TOKEN_MAJOR), ref, "gemm accumulate")


def test_weight_free_releases_both_copies(ctx, oracle):
    """Uploading and freeing a weight over and over leaves the device's free memory where it was: the raw blocks and the
    GEMM's copy both go (read through hipMemGetInfo of the HIP runtime the library itself is linked against)."""
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def free_bytes():
        ctx.sync()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    m, k = 16384, 2048  # 36 MB of Q8_0 blocks + 42 MB of slabs
    wb = np.tile(oracle.synth_weight(W.Q8_0, 256, k, 9, 0.02), m // 256)
    ctx.upload_weight(wb, W.Q8_0, m, k).free()  # the runtime's own pools settle on the first round
    before = free_bytes()
    for _ in range(12):
        w = ctx.upload_weight(wb, W.Q8_0, m, k)
        assert w.device_bytes > 2 * 36_000_000
        w.free()
    assert abs(before - free_bytes()) <= 8 << 20


def test_weights_without_the_gemm_copy_take_the_gemv_route(ctx, oracle):
    """wick_rocm_set_gemm_packing(0): weights uploaded from then on hold the raw blocks only (no second layout for the
    matrix-core kernel) and run as multi-token GEMVs for any n -- same block dots bit for bit, f32 results to the bar."""
    m, n, k = 200, 70, 512
    for dtype, raw_per_block in ((W.Q4_0, 18), (W.Q8_0, 34)):
        wb = oracle.synth_weight(dtype, m, k, 5, 0.02)
        s, q = oracle.quantize_q8_0_batch(oracle.fill_normal(6, 1.0, n * k), n, k)
        packed = ctx.upload_weight(wb, dtype, m, k)
        ctx.set_gemm_packing(False)
        try:
            plain = ctx.upload_weight(wb, dtype, m, k)
        finally:
            ctx.set_gemm_packing(True)
        raw = m * (k // 32) * raw_per_block
        assert plain.device_bytes == raw
        # whole pairs of 32-row granules, 5 KB per granule and 128 K-elements
        assert packed.device_bytes == raw + 2 * ((m + 63) // 64) * (k // 128) * 5120
        d_q, d_s = ctx.to_device(q), ctx.to_device(s)
        ref = oracle.gemm_q8(dtype, wb, s, q, m, n, k)
        outs, dots = [], []
        for w in (packed, plain):
            d_y, d_d = ctx.alloc(n * m * 4), ctx.alloc(n * m * (k // 32) * 4)
            ctx.gemm_preq(w, d_s, d_q, n, d_y, y_stride=m, layout=W.LAYOUT_TOKEN_MAJOR)
            ctx.block_dots_i32(w, d_q, n, d_d)
            outs.append(fetch_gemm(d_y, m, n, m, W.LAYOUT_TOKEN_MAJOR))
            dots.append(d_d.download(np.int32, n * m * (k // 32)))
            d_y.free(), d_d.free()
        assert_f32_parity(outs[0], ref, "packed weight")
        assert_f32_parity(outs[1], ref, "raw-only weight")
        assert np.array_equal(dots[0], dots[1])
        assert np.array_equal(dots[0].reshape(n, m, k // 32), oracle.block_dots_i32(dtype, wb, q, m, n, k))
        # a launch over several weights falls back to one call per weight when one of them has no copy
        d_a, d_b = ctx.alloc(n * 2 * m * 4), ctx.alloc(n * 2 * m * 4)
        ctx.gemm_preq_multi([packed, plain], d_s, d_q, n, [d_a.ptr, d_a.ptr + m * 4], 2 * m)
        ctx.gemm_preq(packed, d_s, d_q, n, d_b.ptr, y_stride=2 * m, layout=W.LAYOUT_TOKEN_MAJOR)
        ctx.gemm_preq(plain, d_s, d_q, n, d_b.ptr + m * 4, y_stride=2 * m, layout=W.LAYOUT_TOKEN_MAJOR)
        assert np.array_equal(d_a.download(np.uint32, n * 2 * m), d_b.download(np.uint32, n * 2 * m))
        for b in (d_q, d_s, d_a, d_b):
            b.free()
        packed.free(), plain.free()


@pytest.mark.parametrize("dtype", [W.Q4_0, W.Q8_0])
@pytest.mark.parametrize("ms,n,k,layout,acc", [
    ((256, 128, 128), 200, 512, W.LAYOUT_TOKEN_MAJOR, False),   # Q / K / V into one [n][q|k|v] row
    ((300, 300), 130, 1024, W.LAYOUT_TOKEN_MAJOR, True),         # gate / up, ragged row tiles, accumulate
    ((129, 1, 257), 40, 256, W.LAYOUT_TOKEN_MAJOR, False),       # narrow tile
    ((128, 64), 17, 128, W.LAYOUT_ROW_MAJOR, False),
    ((64, 96), 5, 256, W.LAYOUT_TOKEN_MAJOR, False),             # below the MFMA hand-off: one call per weight
])
def test_gemm_multi_equals_one_launch_per_weight(ctx, oracle, dtype, ms, n, k, layout, acc):
    """Up to three weights over the same activations in one launch: bit-identical to one launch per weight (each taken unsplit:
    a single weight's launch with few tiles may otherwise walk K in shares, which moves its sums by a few 1e-7)."""
    with Problem(ctx, oracle, dtype, ms[0], k, n, seed=sum(ms) + n) as p:
        ws = [p.w] + [ctx.upload_weight(oracle.synth_weight(dtype, m, k, 50 + i, 0.02), dtype, m, k) for i, m in enumerate(ms[1:])]
        tm = layout == W.LAYOUT_TOKEN_MAJOR
        stride = sum(ms) + 3 if tm else n + 1
        y0 = oracle.fill_normal(9, 1.0, (n if tm else sum(ms)) * stride)
        d_a, d_b = p.to_device(y0), p.to_device(y0)
        offs = np.concatenate([[0], np.cumsum(ms)[:-1]])
        elem = lambda o: int(o) * 4 if tm else int(o) * stride * 4  # byte offset of a weight's first output
        ya = [d_a.ptr + elem(o) for o in offs]
        yb = [d_b.ptr + elem(o) for o in offs]
        ctx.gemm_preq_multi(ws, p.d_s, p.d_q, n, ya, stride, layout=layout, accumulate=acc)
        ctx.set_gemm_max_k_splits(1)
        try:
            for w, y in zip(ws, yb):
                ctx.gemm_preq(w, p.d_s, p.d_q, n, y, y_stride=stride, layout=layout, accumulate=acc)
        finally:
            ctx.set_gemm_max_k_splits(0)
        a, b = d_a.download(np.float32, y0.size), d_b.download(np.float32, y0.size)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        assert not np.array_equal(a, y0)
        d_c = p.to_device(y0)  # the same launches as the library routes them by default: equal to the f32 bar
        for w, o in zip(ws, offs):
            ctx.gemm_preq(w, p.d_s, p.d_q, n, d_c.ptr + elem(o), y_stride=stride, layout=layout, accumulate=acc)
        c = d_c.download(np.float32, y0.size)
        assert np.linalg.norm(c.astype(np.float64) - a) <= 1e-6 * np.linalg.norm(a)
        with pytest.raises(W.RocmError, match="share k and dtype"):
            other = ctx.upload_weight(oracle.synth_weight(dtype, 32, k + 128, 3, 0.02), dtype, 32, k + 128)
            ws.append(other)
            ctx.gemm_preq_multi([ws[0], other], p.d_s, p.d_q, n, ya[:2], stride, layout=layout)
        for w in ws[1:]:
            w.free()


@pytest.mark.parametrize("dtype", [W.Q4_0, W.Q8_0])
def test_full_size_prefill_shape(ctx, oracle, dtype):
    """m=6912, n=2002, k=2048 (the LFM2-1.2B ffn_up prefill shape).  The oracle checks a
    band of rows across ALL tokens plus scattered rows; size-independent properties cover
    the rest: column j of the GEMM equals the GEMV of column j, and both layouts agree."""
    m, n, k = 6912, 2002, 2048
    with Problem(ctx, oracle, dtype, m, k, n, seed=2026) as p:
        d_y = p.alloc(m * n * 4)
        ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, layout=W.LAYOUT_TOKEN_MAJOR)
        y = fetch_gemm(d_y, m, n, m, W.LAYOUT_TOKEN_MAJOR)
        assert np.isfinite(y).all()
        bb = 18 if dtype == W.Q4_0 else 34
        rows = np.concatenate([np.arange(0, 40), np.arange(6890, 6912), np.arange(100, 6800, 397)])
        sub = np.concatenate([p.wb.reshape(m, -1)[r] for r in rows])
        assert sub.size == len(rows) * (k // 32) * bb
        assert_f32_parity(y[rows], oracle.gemm_q8(dtype, sub, p.s, p.q, len(rows), n, k), "C3 row band")
        d_v = p.alloc(m * 4)
        for j in (0, 1, 127, 128, 1000, 1983, 1984, 2001):
            ctx.gemv_with_preq(p.w, p.d_s.ptr + j * (k // 32) * 4, p.d_q.ptr + j * k, d_v)
            assert rel_l2(y[:, j], d_v.download(np.float32, m)) < 1e-6
        ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, layout=W.LAYOUT_ROW_MAJOR)
        y2 = fetch_gemm(d_y, m, n, n, W.LAYOUT_ROW_MAJOR)
        assert np.array_equal(y, y2)


def test_argument_errors(ctx, oracle):
    with Problem(ctx, oracle, W.Q4_0, 64, 256, 20) as p:
        d_y = p.alloc(64 * 20 * 4)
        with pytest.raises(W.RocmError) as e:
            ctx.gemm_preq(p.w, p.d_s, p.d_q, 20, d_y, y_stride=10, layout=W.LAYOUT_ROW_MAJOR)
        assert e.value.status == -1
        with pytest.raises(W.RocmError) as e:
            ctx.gemm_preq(p.w, p.d_s, p.d_q, 20, d_y, y_stride=63, layout=W.LAYOUT_TOKEN_MAJOR)
        assert e.value.status == -1
        with pytest.raises(W.RocmError) as e:
            ctx.gemm_preq(p.w, p.d_s, p.d_q, 20, d_y, y_stride=64, layout=5)
        assert e.value.status == -1
        ctx.gemm_preq(p.w, p.d_s, p.d_q, 0, d_y, y_stride=64, layout=W.LAYOUT_TOKEN_MAJOR)  # n = 0: no-op


@pytest.mark.parametrize("dtype,m,n,k,layout,accumulate", [
    (W.Q4_0, 1024, 512, 4608, "token", True),    # the down projection of a 512-token prompt: 64 tiles, 4 shares
    (W.Q8_0, 1024, 100, 2048, "token", False),   # 16 tiles, 4 shares of 4 stages
    (W.Q4_0, 300, 70, 4608, "row", True),        # ragged rows and tokens, 8 shares, row-major output
    (W.Q8_0, 2048, 640, 6912, "token", False),   # 160 narrow tiles (80 wide): 4 shares on the wide tile
    (W.Q4_0, 1024, 2002, 4608, "token", False),  # 256 narrow tiles = 128 wide ones with a long K: 4 shares on the wide tile
    (W.Q8_0, 2048, 700, 4224, "row", True),      # 96 wide tiles, 33 stages: 4 shares of 8 or 9 on the wide tile, ragged tokens
    (W.Q8_0, 1024, 2002, 2048, "token", False),  # 16 stages: too short for the wide split, too many tiles for the narrow one
    (W.Q4_0, 256, 300, 1024, "row", False),      # 10 tiles (not a multiple of the 8 slots the tile map deals out), 4 shares of 2 stages
    (W.Q8_0, 640, 200, 2048, "token", True),     # 20 tiles, 4 shares
    (W.Q4_0, 384, 130, 1152, "token", False),    # 9 stages in 4 shares: 2, 2, 2, 3
    (W.Q8_0, 200, 40, 4224, "row", True),        # 33 stages in 8 shares: 4 or 5 each
    (W.Q4_0, 3072, 128, 1024, "token", False),   # the in projection of a short prompt: 48 tiles, 4 shares
])
def test_gemm_split_over_k(ctx, oracle, dtype, m, n, k, layout, accumulate):
    """GEMM launches with few tiles and a long K walk K in shares (one workgroup per tile and share, a second launch adds the
    shares in a fixed order): held against the oracle like every other launch, equal to the unsplit launch to a few 1e-7,
    and the same bits on every run."""
    wb = oracle.synth_weight(dtype, m, k, seed=77)
    w = ctx.upload_weight(wb, dtype, m, k)
    s, q = oracle.quantize_q8_0_batch(oracle.fill_normal(5, 1.0, n * k), n, k)
    d_q, d_s = ctx.to_device(q), ctx.to_device(s)
    lay = W.LAYOUT_TOKEN_MAJOR if layout == "token" else W.LAYOUT_ROW_MAJOR
    stride = (m + 8) if layout == "token" else (n + 4)
    size = n * stride if layout == "token" else m * stride
    y0 = oracle.fill_normal(6, 1.0, size)
    outs = []
    for splits in (0, 0, 1):  # default twice, then switched off
        ctx.set_gemm_max_k_splits(splits)
        d_y = ctx.to_device(y0)
        ctx.gemm_preq(w, d_s, d_q, n, d_y, y_stride=stride, layout=lay, accumulate=accumulate)
        y = d_y.download(np.float32, size)
        outs.append((y.reshape(n, stride)[:, :m].T if layout == "token" else y.reshape(m, stride)[:, :n]).copy())
        pad = y.reshape(n, stride)[:, m:] if layout == "token" else y.reshape(m, stride)[:, n:]
        assert np.array_equal(pad, (y0.reshape(n, stride)[:, m:] if layout == "token" else y0.reshape(m, stride)[:, n:]))
        d_y.free()
    ctx.set_gemm_max_k_splits(0)
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    ref = oracle.gemm_q8(dtype, wb, s, q, m, n, k, f64=True)
    if accumulate:
        ref = ref + (y0.reshape(n, stride)[:, :m].T if layout == "token" else y0.reshape(m, stride)[:, :n])
    assert_f32_parity(outs[0], ref, "split GEMM")
    assert_f32_parity(outs[2], ref, "unsplit GEMM")
    assert np.linalg.norm(outs[0].astype(np.float64) - outs[2]) <= 1e-6 * np.linalg.norm(outs[2])
    w.free(), d_q.free(), d_s.free()


@pytest.mark.parametrize("shape", [32, 16])
@pytest.mark.parametrize("dtype,m,n,k,pad", [
    (W.Q4_0, 1024, 512, 4608, 0),   # the down projection of a 512-token prompt: split, the norm's kernel adds the shares up
    (W.Q8_0, 1024, 100, 1024, 8),   # an out projection of a short prompt: split in 4, padded rows
    (W.Q4_0, 256, 300, 1024, 0),    # 10 tiles
    (W.Q4_0, 1024, 2002, 4608, 0),  # 256 tiles: unsplit, the plain norm kernel
    (W.Q8_0, 512, 7, 256, 4),       # below the MFMA hand-off: multi-token GEMV, then the norm
    (W.Q4_0, 1024, 23, 1024, 0),    # few tokens, split in 4: the shares walked inside the launch (by the norm on the 16x16x32 loop)
    (W.Q8_0, 768, 32, 1024, 4), (W.Q8_0, 736, 32, 1024, 4),   # 24 granules: inside the launch; fewer: the norm adds them up
    (W.Q4_0, 2304, 20, 1536, 0), (W.Q4_0, 2272, 20, 1536, 0),  # 72 granules, 12 slabs: the same
    (W.Q4_0, 3840, 33, 1024, 0), (W.Q4_0, 3808, 64, 1024, 0),  # 120 granules, 33 tokens and more: the same
    (W.Q8_0, 512, 64, 1024, 4),     # the norm adds them up; the plain call walks them inside the launch
    (W.Q4_0, 1024, 40, 4608, 0),    # K too long for that: shares side by side either way
])
def test_residual_projection_with_norm_and_quantizer(ctx, oracle, dtype, m, n, k, pad, shape):
    """x += W a, then Q8_0(rmsnorm(x)): one call == wick_rocm_gemm_q8 (accumulate) + wick_rocm_rmsnorm_quantize_q8_0, bit for bit -- the
    residual rows, the quants and the scales -- whether or not the projection is split over K, on either block loop; and x against
    the oracle."""
    ctx.set_gemm_mfma_shape(shape)
    try:
        residual_projection_with_norm_and_quantizer(ctx, oracle, dtype, m, n, k, pad)
    finally:
        ctx.set_gemm_mfma_shape(0)


@pytest.mark.parametrize("m,n,k,pad", [(1056, 150, 1024, 4), (2048, 40, 2048, 0), (2016, 100, 4608, 0)])
def test_residual_projection_over_row_lengths(ctx, oracle, m, n, k, pad):
    """Rows of 1025 .. 2048 elements, whose shares the norm's kernel adds up with eight elements per thread on their way."""
    residual_projection_with_norm_and_quantizer(ctx, oracle, W.Q4_0, m, n, k, pad)


def residual_projection_with_norm_and_quantizer(ctx, oracle, dtype, m, n, k, pad):
    from wick_amd.lfm2 import Lfm2Ops
    ops, eps, stride = Lfm2Ops(ctx), 1e-5, m + pad
    wb = oracle.synth_weight(dtype, m, k, seed=31)
    w = ctx.upload_weight(wb, dtype, m, k)
    s, q = oracle.quantize_q8_0_batch(oracle.fill_normal(5, 1.0, n * k), n, k)
    d_q, d_s = ctx.to_device(q), ctx.to_device(s)
    x0 = oracle.fill_normal(6, 1.0, n * stride)
    nw = (1 + 0.3 * oracle.fill_normal(7, 1.0, m)).astype(np.float32)
    d_nw = ctx.to_device(nw)
    res = []
    for fused in (True, False):
        d_x, d_oq, d_os = ctx.to_device(x0), ctx.alloc(n * m), ctx.alloc(n * (m // 32) * 4)
        if fused:
            ctx.gemm_preq_residual_rmsnorm_quantize(w, d_s, d_q, n, d_x, stride, d_nw, eps, d_oq, d_os)
        else:
            ctx.gemm_preq(w, d_s, d_q, n, d_x, y_stride=stride, layout=W.LAYOUT_TOKEN_MAJOR, accumulate=True)
            ops.rmsnorm_quantize(d_x, d_nw, n, m, eps, d_oq, d_os, x_stride=stride)
        res.append((d_x.download(np.float32, n * stride), d_oq.download(np.int8, n * m), d_os.download(np.float32, n * (m // 32))))
        for b in (d_x, d_oq, d_os):
            b.free()
    for a, b in zip(*res):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    x = res[0][0].reshape(n, stride)
    assert np.array_equal(x[:, m:], x0.reshape(n, stride)[:, m:])  # padding untouched
    ref = oracle.gemm_q8(dtype, wb, s, q, m, n, k, f64=True).T + x0.reshape(n, stride)[:, :m]
    assert_f32_parity(x[:, :m], ref, "residual projection")
    # quantizing the input in place of the projection's own input buffers is what the prompt pass does
    if m == k:
        d_x, d_q2, d_s2 = ctx.to_device(x0), ctx.to_device(q), ctx.to_device(s)
        ctx.gemm_preq_residual_rmsnorm_quantize(w, d_s2, d_q2, n, d_x, stride, d_nw, eps, d_q2, d_s2)
        assert np.array_equal(d_q2.download(np.int8, n * m), res[0][1]) and np.array_equal(d_s2.download(np.float32, n * (m // 32)).view(np.uint32), res[0][2].view(np.uint32))
        for b in (d_x, d_q2, d_s2):
            b.free()
    with pytest.raises(W.RocmError, match="multiple of 32"):
        w2 = ctx.upload_weight(oracle.synth_weight(dtype, 48, 256, seed=1), dtype, 48, 256)
        ctx.gemm_preq_residual_rmsnorm_quantize(w2, d_s, d_q, 1, d_nw, 48, d_nw, eps, d_q, d_s)
    w.free(), w2.free(), d_q.free(), d_s.free(), d_nw.free()


# ragged in rows and tokens, and the tile that their costs choose
PROMPT_TILES = {(8150, 2021, 2048): "TileL", (3001, 1500, 256): "TileH", (2050, 1990, 1024): "TileH", (1000, 1999, 384): "TileN"}


@pytest.mark.parametrize("m,n,k", list(PROMPT_TILES))
def test_prompt_tiles_against_the_gemv_route(ctx, oracle, m, n, k):
    """Every element of a prompt-sized projection on the tile its size selects: both layouts and the accumulate flag bit-equal to each
    other, and within the f32 bar of the multi-token GEMV."""
    with Problem(ctx, oracle, W.Q4_0, m, k, n, seed=m + n + k) as p:
        d_y = p.alloc((n + 4) * (m + 4) * 4)
        old = oracle.fill_normal(3, 1.0, (n + 4) * (m + 4))
        out = {}
        for layout, stride in ((W.LAYOUT_TOKEN_MAJOR, m + 4), (W.LAYOUT_ROW_MAJOR, n + 4)):
            for acc in (False, True):
                d_y.upload(old)
                ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, y_stride=stride, layout=layout, accumulate=acc)
                out[layout, acc] = fetch_gemm(d_y, m, n, stride, layout).copy()
            was = old[:(n if layout == W.LAYOUT_TOKEN_MAJOR else m) * stride].reshape(-1, stride)
            was = was[:, :m].T if layout == W.LAYOUT_TOKEN_MAJOR else was[:, :n]
            assert np.array_equal(out[layout, True], was + out[layout, False])
        assert np.array_equal(out[W.LAYOUT_TOKEN_MAJOR, False], out[W.LAYOUT_ROW_MAJOR, False])
        ctx.set_gemm_min_n(n + 1)
        try:
            ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, y_stride=m, layout=W.LAYOUT_TOKEN_MAJOR)
        finally:
            ctx.set_gemm_min_n(0)
        assert rel_l2(out[W.LAYOUT_TOKEN_MAJOR, False], fetch_gemm(d_y, m, n, m, W.LAYOUT_TOKEN_MAJOR)) < 1e-6


@pytest.mark.parametrize("dtype", [W.Q4_0, W.Q8_0])
@pytest.mark.parametrize("m,n,k", [(33, 9, 128), (32, 32, 1024), (100, 33, 1152), (64, 64, 4608), (1000, 31, 6912), (2080, 37, 1664)])
def test_few_token_launches(ctx, oracle, dtype, m, n, k):
    """Granule-per-workgroup launches at their edges: one row past a granule, one / two token groups full and one short, fewer slabs
    than waves, slabs that do not deal out evenly over waves and shares; split over K with the shares walked and added up by one
    workgroup (repeated: the same bits every time) and unsplit; both layouts, accumulate, block dots."""
    with Problem(ctx, oracle, dtype, m, k, n, seed=m + 3 * n + k + dtype) as p:
        ref = oracle.gemm_q8(dtype, p.wb, p.s, p.q, m, n, k)
        first = {}
        for splits in (0, 1, 0, 2, 8, 0):
            ctx.set_gemm_max_k_splits(splits)
            try:
                for layout, stride in ((W.LAYOUT_ROW_MAJOR, n + 3), (W.LAYOUT_TOKEN_MAJOR, m + 5)):
                    rows = m if layout == W.LAYOUT_ROW_MAJOR else n
                    d_y = p.to_device(np.full(rows * stride, 2.5, np.float32))
                    ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, y_stride=stride, layout=layout)
                    y = fetch_gemm(d_y, m, n, stride, layout).copy()
                    assert_f32_parity(y, ref, f"few {dtype} {m}x{n}x{k} splits {splits} layout {layout}")
                    assert np.array_equal(y, first.setdefault(splits, y))  # same bits in either layout and every time
                    full = d_y.download(np.float32, rows * stride).reshape(rows, stride)
                    assert np.all(full[:, n if layout == W.LAYOUT_ROW_MAJOR else m:] == 2.5)
                    ctx.gemm_preq(p.w, p.d_s, p.d_q, n, d_y, y_stride=stride, layout=layout, accumulate=True)
                    assert np.array_equal(fetch_gemm(d_y, m, n, stride, layout), y + y)
            finally:
                ctx.set_gemm_max_k_splits(0)
        d_d = p.alloc(n * m * (k // 32) * 4)
        ctx.block_dots_i32(p.w, p.d_q, n, d_d)
        assert np.array_equal(d_d.download(np.int32, n * m * (k // 32)).reshape(n, m, k // 32), oracle.block_dots_i32(dtype, p.wb, p.q, m, n, k))


@pytest.mark.parametrize("dtype", [W.Q4_0, W.Q8_0])
@pytest.mark.parametrize("layout", [W.LAYOUT_ROW_MAJOR, W.LAYOUT_TOKEN_MAJOR])
@pytest.mark.parametrize("ms,k", [
    ((100, 33, 7), 512),       # ragged rows, per-lane loads
    ((1500, 500, 12), 1024),   # span loads
    ((70, 64, 1), 4608),       # two chunks of pairs per row
    ((140001, 3, 1), 64),      # several passes per wave
    ((65, 40, 2), 96),         # odd block count: the generic kernel
])
def test_one_token_accumulates_into_a_column(ctx, oracle, dtype, layout, ms, k):
    """y += W x of ONE token into a column of a [rows][N] matrix (row-major, a stride that is no extent) and into a strided
    token-major row, by wick_rocm_gemm_q8 per weight and by wick_rocm_gemm_q8_multi: every other element stays."""
    rm = layout == W.LAYOUT_ROW_MAJOR
    col, stride = 2, 5 if rm else sum(ms) + 9
    with Problem(ctx, oracle, dtype, ms[0], k, 1, seed=ms[0] + k + dtype) as p:
        wbs = [p.wb] + [oracle.synth_weight(dtype, m, k, 50 + i, 0.02) for i, m in enumerate(ms[1:])]
        ws = [p.w] + [ctx.upload_weight(wb, dtype, m, k) for wb, m in zip(wbs[1:], ms[1:])]
        offs = np.concatenate([[0], np.cumsum(ms)[:-1]])
        elem = [int(o) * stride + col if rm else int(o) for o in offs]
        y0 = oracle.fill_normal(21, 1.0, sum(ms) * stride if rm else stride)
        step, want, touched = stride if rm else 1, y0.copy(), np.zeros(y0.size, bool)
        for wb, m, e in zip(wbs, ms, elem):
            at = slice(e, e + (m - 1) * step + 1, step)
            want[at] += oracle.gemv_q8(dtype, wb, p.s[0], p.q[0], m, k)
            touched[at] = True
        for multi in (False, True):
            d_y = ctx.to_device(y0)
            ys = [d_y.ptr + 4 * e for e in elem]
            if multi:
                ctx.gemm_preq_multi(ws, p.d_s, p.d_q, 1, ys, stride, layout=layout, accumulate=True)
            else:
                for w, y in zip(ws, ys):
                    ctx.gemm_preq(w, p.d_s, p.d_q, 1, y, y_stride=stride, layout=layout, accumulate=True)
            y = d_y.download(np.float32, y0.size)
            assert np.array_equal(y[~touched], y0[~touched])
            assert_f32_parity(y[touched], want[touched], f"one token, {'multi' if multi else 'single'}")
            d_y.free()
        for w in ws[1:]:
            w.free()


# Pairs of launches on the two sides of each rule that chooses a GEMM kernel, a tile or a number of shares: (m, n, k), the rule's
# quantity at its limit and one step past it; and the kernels that the rules send them to (test_launch_routes.py), as the library
# splits K and unsplit: "few" token groups and waves, "narrow" 16-token columns, a tile; "in" shares that a second launch adds up.
EDGES = {
    # 512 granules of rows: one workgroup per granule
    (16384, 9, 128): ("few 1 4", "few 1 4"),
    (16416, 9, 128): ("few 1 4", "few 1 4"),
    # 1024 granules, up to 32 tokens; 768 past 16 slabs of K
    (32768, 9, 128): ("few 1 4", "few 1 4"),
    (32800, 9, 128): ("narrow 1", "narrow 1"),
    (32800, 32, 128): ("narrow 2", "narrow 2"),
    (24608, 17, 2048): ("few 1 4", "few 1 4"),
    (24576, 17, 2176): ("few 1 4", "few 1 4"),
    (24608, 17, 2176): ("narrow 2", "narrow 2"),
    # two shares of 512 granules, up to 32 tokens
    (16384, 32, 3072): ("few 1 4, in 2", "few 1 4"),
    (16384, 32, 3200): ("few 1 4, in 2", "few 1 4"),
    # 8 slabs of 512 granules walked, 9 in shares, 33 tokens and more
    (16384, 33, 1024): ("few 2 8", "few 2 8"),
    (16384, 33, 1152): ("TileN, in 2", "few 2 8"),
    # 64 tokens
    (512, 64, 512): ("few 2 8", "few 2 8"),
    (512, 65, 512): ("few 1 4", "few 1 4"),
    (512, 2049, 512): ("TileN", "TileN"),
    # 15 slabs of a split launch, up to 32 tokens and under 96 granules
    (256, 32, 1920): ("few 1 8", "few 1 8"),
    (256, 32, 2048): ("few 1 8, in 8", "few 1 8"),
    # 16 slabs from 96 granules on
    (3040, 9, 2048): ("few 1 4, in 8", "few 1 8"),
    (3072, 9, 2048): ("few 1 8", "few 1 8"),
    (3072, 9, 2176): ("few 1 4, in 8", "few 1 8"),
    # shares past two workgroups a CU: up to 32 tokens
    (4096, 32, 4096): ("few 1 4, in 8", "few 1 8"),
    (4096, 33, 4096): ("TileN, in 8", "few 2 8"),
    # 8 slabs, 33 tokens and more
    (256, 33, 1024): ("few 2 8", "few 2 8"),
    (256, 33, 1152): ("few 2 8, in 4", "few 2 8"),
    # 256 granules, up to 32 tokens: eight waves or four
    (8192, 9, 128): ("few 1 8", "few 1 8"),
    (8224, 9, 128): ("few 1 4", "few 1 4"),
    # 256 granules, 33 tokens and more: one workgroup a CU, or two; 512 below
    (8192, 33, 256): ("few 2 8", "few 2 8"),
    (8224, 33, 256): ("few 2 8", "few 2 8"),
    # 48 tokens on the 128-row tiles; 49 .. 64 on the 32x32x32 loop
    (16416, 48, 128): ("narrow 3", "narrow 3"),
    (16416, 49, 128): ("TileS", "TileS"),
    # 8 stages: split over K (one launch either way)
    (64, 40, 896): ("few 2 8", "few 2 8"),
    (64, 40, 1024): ("few 2 8", "few 2 8"),
    # 256 tiles of 128 x 128
    (4096, 1024, 128): ("TileX", "TileX"),
    (4096, 1025, 128): ("TileL", "TileL"),
    # 256 tiles of 128 x 64
    (2048, 1024, 128): ("TileS", "TileS"),
    (2048, 1025, 128): ("TileX", "TileX"),
    # 64 wide tiles, 32 stages: shares on the wide tile
    (1024, 1024, 4096): ("TileN, in 4", "few 2 8"),
    (1024, 896, 4096): ("TileN, in 2", "few 2 8"),
    (1024, 1024, 3968): ("TileN, in 2", "few 2 8"),
    # 256 wide tiles
    (4096, 1024, 4096): ("TileX, in 2", "TileN"),
    (4096, 1025, 4096): ("TileH", "TileH"),
}


@pytest.mark.parametrize("m,n,k", list(EDGES))
def test_both_sides_of_every_launch_rule(ctx, oracle, m, n, k):
    """Either side of a rule gives the multi-token GEMV's result (another kernel, other sums: within 1e-6), in both layouts, added to
    what is there, and leaves the padding alone; split over K as the library does it, and unsplit."""
    dtype = W.Q4_0 if (m + n + k) % 2 == 0 else W.Q8_0
    rows = 256 if m % 256 == 0 else 32  # of the weight, repeated: making 16384 of them takes the oracle seconds
    wb = np.tile(oracle.synth_weight(dtype, rows, k, 7, 0.02).reshape(rows, -1), (-(-m // rows), 1))[:m]
    s, q = oracle.quantize_q8_0_batch(oracle.fill_normal(5, 1.0, n * k), n, k)
    w, d_q, d_s = ctx.upload_weight(wb, dtype, m, k), ctx.to_device(q), ctx.to_device(s)
    old = oracle.fill_normal(6, 1.0, (n + 3) * (m + 5))
    d_ref = ctx.alloc(n * m * 4)
    ctx.set_gemm_min_n(n + 1)
    try:
        ctx.gemm_preq(w, d_s, d_q, n, d_ref, y_stride=m, layout=W.LAYOUT_TOKEN_MAJOR)
    finally:
        ctx.set_gemm_min_n(0)
    ref = fetch_gemm(d_ref, m, n, m, W.LAYOUT_TOKEN_MAJOR)
    for splits in (0, 1):  # (a limit on unsplit launches is met by launches over several weights, or with the split switched off)
        got = {}
        ctx.set_gemm_max_k_splits(splits)
        try:
            for layout, stride in ((W.LAYOUT_TOKEN_MAJOR, m + 5), (W.LAYOUT_ROW_MAJOR, n + 3)):
                outer, inner = (n, m) if layout == W.LAYOUT_TOKEN_MAJOR else (m, n)
                d_y = ctx.to_device(old)
                ctx.gemm_preq(w, d_s, d_q, n, d_y, y_stride=stride, layout=layout)
                got[layout] = fetch_gemm(d_y, m, n, stride, layout).copy()
                assert rel_l2(got[layout], ref) < 1e-6
                d_y.upload(old)
                ctx.gemm_preq(w, d_s, d_q, n, d_y, y_stride=stride, layout=layout, accumulate=True)
                y, was = d_y.download(np.float32, outer * stride).reshape(outer, stride), old[:outer * stride].reshape(outer, stride)
                assert np.array_equal(y[:, inner:], was[:, inner:])
                assert np.array_equal(y[:, :inner], was[:, :inner] + (got[layout].T if layout == W.LAYOUT_TOKEN_MAJOR else got[layout]))
                d_y.free()
        finally:
            ctx.set_gemm_max_k_splits(0)
        assert np.array_equal(got[W.LAYOUT_TOKEN_MAJOR], got[W.LAYOUT_ROW_MAJOR])
    w.free(), d_q.free(), d_s.free(), d_ref.free()


@pytest.mark.parametrize("m,n,k", [(2048, 1025, 128), (2080, 1024, 128), (2048, 1024, 128), (8224, 65, 128), (8224, 64, 128), (96, 64, 256)])
def test_the_gated_launch_starts_past_256_tiles(ctx, oracle, m, n, k):
    """Where the gate | up launch with the gate in its epilogue applies: more than 256 tiles of 64 rows x 128 tokens and more than 64
    tokens; on the first shapes it takes, the same bits as the separate launches."""
    from wick_amd.lfm2 import Lfm2Ops

    ops = Lfm2Ops(ctx)
    ws = [ctx.upload_weight(oracle.synth_weight(W.Q4_0, m, k, seed=41 + i), W.Q4_0, m, k) for i in range(2)]
    tiles = (m + 63) // 64 * ((n + 127) // 128)
    assert ops.ffn_gate_up_silu_quantize_applies(ws[0], ws[1], n) == (tiles > 256 and n > 64)
    if tiles > 256 and n > 64:
        s, q = oracle.quantize_q8_0_batch(oracle.fill_normal(9, 1.0, n * k), n, k)
        d_q, d_s, out = ctx.to_device(q), ctx.to_device(s), []
        d_g, d_u, d_oq, d_os = ctx.alloc(n * m * 4), ctx.alloc(n * m * 4), ctx.alloc(n * m), ctx.alloc(n * (m // 32) * 4)
        for gated in (True, False):
            if gated:
                ops.encode_ffn_gate_up_silu_quantize(ws[0], ws[1], d_s, d_q, n, d_oq, d_os)
            else:
                ctx.gemm_preq_multi(ws, d_s, d_q, n, [d_g, d_u], m)
                ops.silu_mul_quantize(d_g, d_u, n, m, d_oq, d_os)
            out.append((d_oq.download(np.uint8, n * m), d_os.download(np.uint32, n * (m // 32))))
        assert all(np.array_equal(a, b) for a, b in zip(*out))
        for b in (d_q, d_s, d_g, d_u, d_oq, d_os):
            b.free()
    ws[0].free(), ws[1].free()


# A launch with a last tile of 32 rows and of few tokens on each of the tiles that launch costs choose from, plain and with the gate.
RAGGED_TILES = {(31, 2081, 384): "TileH", (65, 2111, 128): "TileH", (96, 2051, 256): "TileH", (5472, 131, 1024): "TileN", (5408, 643, 128): "TileS", (4832, 1027, 512): "TileQ", (6176, 451, 128): "TileX",
                (6944, 1669, 128): "TileL"}
RAGGED_GATED_TILES = {(5472, 259, 128): "TileS", (6560, 259, 128): "TileQ", (6176, 451, 512): "TileX", (6752, 1031, 1024): "TileL"}


@pytest.mark.parametrize("m,n,k", list(RAGGED_TILES))
def test_ragged_launches_on_every_tile(ctx, oracle, m, n, k):
    """Partly filled tiles give the multi-token GEMV's result, in both layouts, added to what is there, and leave the padding alone."""
    test_both_sides_of_every_launch_rule(ctx, oracle, m, n, k)


@pytest.mark.parametrize("m,n,k", list(RAGGED_GATED_TILES))
def test_ragged_gated_launches_on_every_tile(ctx, oracle, m, n, k):
    """The same of the launches with the gate in the epilogue, against the separate ones, bit for bit."""
    from wick_amd.lfm2 import Lfm2Ops

    ops = Lfm2Ops(ctx)
    wb = [np.tile(oracle.synth_weight(W.Q4_0, 32, k, seed=61 + i).reshape(32, -1), (m // 32, 1)) for i in range(2)]
    ws = [ctx.upload_weight(b, W.Q4_0, m, k) for b in wb]
    assert ops.ffn_gate_up_silu_quantize_applies(ws[0], ws[1], n)
    s, q = oracle.quantize_q8_0_batch(oracle.fill_normal(12, 1.0, n * k), n, k)
    d_q, d_s, out = ctx.to_device(q), ctx.to_device(s), []
    d_g, d_u = ctx.alloc(n * m * 4), ctx.alloc(n * m * 4)
    d_oq, d_os = ctx.to_device(np.full(n * m + 64, 77, np.int8)), ctx.to_device(np.full(n * (m // 32) + 16, 77.0, np.float32))
    for gated in (True, False):
        if gated:
            ops.encode_ffn_gate_up_silu_quantize(ws[0], ws[1], d_s, d_q, n, d_oq, d_os)
        else:
            ctx.gemm_preq_multi(ws, d_s, d_q, n, [d_g, d_u], m)
            ops.silu_mul_quantize(d_g, d_u, n, m, d_oq, d_os)
        out.append((d_oq.download(np.uint8, n * m + 64), d_os.download(np.uint32, n * (m // 32) + 16)))
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    assert (out[0][0][n * m:] == 77).all() and (out[0][1][n * (m // 32):].view(np.float32) == 77.0).all()
    for b in (d_q, d_s, d_g, d_u, d_oq, d_os, *ws):
        b.free()


@pytest.mark.parametrize("dtype", [W.Q4_0, W.Q8_0])
def test_the_gate_in_the_launch_over_all_magnitudes(ctx, oracle, dtype):
    """The launch's own silu takes gates of 2^-60 .. 41 in a shorter way than the others: groups of 32 tokens whose gates lie inside, across
    either end and outside (tiny, subnormal, zero, huge, infinite), the same bits as the separate launches."""
    from wick_amd.lfm2 import Lfm2Ops

    m, n, k = 2112, 1030, 128
    ops = Lfm2Ops(ctx)
    ws = [ctx.upload_weight(oracle.synth_weight(dtype, m, k, seed=51 + i), dtype, m, k) for i in range(2)]
    assert ops.ffn_gate_up_silu_quantize_applies(ws[0], ws[1], n)
    s, q = oracle.quantize_q8_0_batch(oracle.fill_normal(10, 1.0, n * k), n, k)
    unit = oracle.gemm_q8(dtype, oracle.synth_weight(dtype, m, k, seed=51), s, q, m, n, k).std()  # a gate of factor 1 is one of this size
    factors = np.array([1, 3, 9, 13, 20, 45, 1e3, 1e-2, 1e-6, 1e-12, 1e-17, 1e-18, 1e-19, 1e-22, 1e-30, 1e-38, 0, 1e20, 1e30, 3e38], np.float32)
    s = np.minimum(s.reshape(n, -1) * (factors[np.arange(n) // 32 % factors.size].astype(np.float64) / unit)[:, None], 3e38).astype(np.float32)
    d_q, d_s, out = ctx.to_device(q), ctx.to_device(s), []
    d_g, d_u, d_oq, d_os = ctx.alloc(n * m * 4), ctx.alloc(n * m * 4), ctx.alloc(n * m), ctx.alloc(n * (m // 32) * 4)
    for gated in (True, False):
        if gated:
            ops.encode_ffn_gate_up_silu_quantize(ws[0], ws[1], d_s, d_q, n, d_oq, d_os)
        else:
            ctx.gemm_preq_multi(ws, d_s, d_q, n, [d_g, d_u], m)
            ops.silu_mul_quantize(d_g, d_u, n, m, d_oq, d_os)
        out.append((d_oq.download(np.uint8, n * m), d_os.download(np.uint32, n * (m // 32))))
    g = np.abs(d_g.download(np.float32, n * m).reshape(n, m))
    assert (g[:32] < 41).all() and (g == 0).any() and np.isinf(g[~np.isnan(g)]).any()
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    for b in (d_q, d_s, d_g, d_u, d_oq, d_os, *ws):
        b.free()


# m, n, k -> the kernels of a projection, split over K as the library does it and unsplit: several tiles of 32 or 64 tokens on the few-token kernel
FEW_TILES = {
    (1056, 97, 640): ("few 1 4", "few 1 4"),           # one token and one granule over
    (2080, 81, 128): ("few 1 4", "few 1 4"),           # one slab
    (544, 65, 512): ("few 1 4", "few 1 4"),            # 512 x 512 and a granule
    (96, 67, 256): ("few 1 4", "few 1 4"),
    (31, 832, 128): ("few 1 4", "few 1 4"),            # less than a granule, one slab
    (33, 200, 4096): ("few 1 4, in 8", "few 1 4"),     # few rows in shares
    (3584, 128, 256): ("few 1 4", "few 1 4"),          # 448 tiles of 32 tokens
    (3584, 129, 256): ("few 2 8", "few 2 8"),
    (8192, 128, 128): ("few 2 8", "few 2 8"),          # 512 of 64
    (8224, 128, 128): ("TileS", "TileS"),
    (1056, 831, 384): ("few 2 8", "few 2 8"),          # 33 granules, not rounded up
    (160, 635, 3968): ("few 2 8, in 8", "few 1 4"),    # 40 workgroups of shares, all with work
    (1024, 832, 384): ("few 2 8", "few 2 8"),          # 832 tokens
    (1024, 833, 384): ("few 2 8", "few 2 8"),
    (512, 2048, 384): ("few 2 8", "few 2 8"), (480, 2049, 384): ("TileN", "TileN"),
    (512, 1024, 2304): ("few 2 8", "few 2 8"), (512, 1025, 2304): ("TileH, in 2", "few 2 8"),  # 18 slabs walked up to 1024 tokens
    (1024, 768, 4608): ("few 2 8", "few 2 8"), (1024, 769, 4608): ("TileN, in 2", "few 2 8"),  # 36 up to 768
    (1024, 76, 2048): ("few 1 4", "few 1 4"),          # 16 slabs in shares: in the launch
    (1024, 74, 2048): ("few 2 8, in 8", "few 1 4"),    # or 512 side by side
    (1024, 334, 3328): ("few 1 4", "few 1 4"), (1024, 334, 3456): ("TileH, in 4", "few 1 4"),  # 26 slabs walked in tiles of 32
    (1600, 448, 5376): ("few 2 8", "few 2 8"), (1600, 448, 5504): ("TileH, in 2", "few 2 8"),  # 42 in tiles of 64
    (3072, 96, 3840): ("few 1 4", "few 1 4"), (3072, 97, 3840): ("TileH, in 4", "few 1 4"),    # or over 96 tokens
    (256, 330, 2048): ("few 1 4", "few 1 4"), (256, 300, 2048): ("few 2 8, in 8", "few 1 4"),  # 16 slabs, 256 x 301 results
}


@pytest.mark.parametrize("m,n,k", list(FEW_TILES))
def test_few_token_tiles_side_by_side(ctx, oracle, m, n, k):
    """More than 64 tokens on the few-token kernel give the multi-token GEMV's result, in both layouts, added to what is there, and leave the padding alone."""
    test_both_sides_of_every_launch_rule(ctx, oracle, m, n, k)
