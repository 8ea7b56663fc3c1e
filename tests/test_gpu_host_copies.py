"""Copies between device and host memory through the pinned slots (wick_rocm_upload / wick_rocm_download): sizes on either side of a
slot, of the single-wait path and of the 16-byte pieces of the copy kernel, at aligned and unaligned offsets."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SLOT = 2 << 20


@pytest.mark.parametrize("nbytes", [1, 15, 4096, SLOT, 2 * SLOT, 2 * SLOT + 1, 2 * SLOT + 16, 13 * SLOT + 48, 27 * SLOT - 7])
@pytest.mark.parametrize("off", [0, 3, 16])
def test_round_trip(ctx, nbytes, off):
    src = np.random.default_rng(nbytes + off).integers(0, 256, nbytes, dtype=np.uint8)
    buf = ctx.to_device(np.full(nbytes + off + 32, 7, np.uint8))
    buf.upload(src, off)
    whole = buf.download(np.uint8, nbytes + off + 32)
    assert np.array_equal(whole[off:off + nbytes], src) and np.all(whole[:off] == 7) and np.all(whole[off + nbytes:] == 7)
    assert np.array_equal(buf.download(np.uint8, nbytes, off), src)
    buf.free()


@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("n,keep,shift", [(64, 0, 63), (64, 3, 1), (64, 5, 4), (64, 10, 17), (61, 0, 30)])
def test_model_shift_in_place_equals_the_staged_one(ctx, oracle, n, keep, shift, kv_f16):
    """shift_kv of a model (rows moved in place where that takes at most 16 launches, staged otherwise) against the staged
    per-layer operation on the same caches."""
    import lfm2_synth
    from wick_amd import gguf as G
    from wick_amd.lfm2 import Lfm2Ops, RocmLfm2Model, rope_theta_scale

    img, cfg, _ = lfm2_synth.build(oracle, seed=5)
    with G.GgufFile.from_bytes(img) as g:
        model = RocmLfm2Model(ctx, g, 64, kv_f16=kv_f16)
    rng = np.random.default_rng(n + shift)
    dt = np.float16 if kv_f16 else np.float32
    state = [rng.standard_normal(model.layer_state_bytes(i, n) // (np.dtype(dt).itemsize if kv else 4)).astype(dt if kv else np.float32)
             for i, kv in enumerate(model.kv_heads_per_layer)]
    model.restore_state(np.concatenate([s.view(np.uint8) for s in state]), n)
    got = model.snapshot_state(model.shift_kv(n, keep, shift))
    model.free()
    hd = cfg["hidden_size"] // cfg["n_heads"]
    scale, ops, at = rope_theta_scale(hd, cfg["rope_theta"]), Lfm2Ops(ctx), 0
    for kv, s in zip(model.kv_heads_per_layer, state):
        if kv:
            rows = s.astype(np.float32).reshape(2, n, kv * hd)
            d_k, d_v = ctx.to_device(rows[0]), ctx.to_device(rows[1])
            stage = ctx.alloc(4 * max(1, ops.kv_shift_scratch_floats(n, keep, shift, kv, hd)))
            ops.encode_kv_shift(d_k, d_v, stage, n, keep, shift, kv, hd, scale)
            s = np.concatenate([d.download(np.float32, n * kv * hd)[:(n - shift) * kv * hd] for d in (d_k, d_v)]).astype(dt)
            for b in (d_k, d_v, stage):
                b.free()
        want = s.view(np.uint8)
        assert np.array_equal(got[at:at + want.size], want)
        at += want.size
    assert at == got.size


@pytest.mark.parametrize("nbytes", [8192 + 16, 3 * SLOT])
def test_a_range_past_its_allocation_is_refused(ctx, nbytes):
    """The library's own check, in front of the copy kernel (what it does with other addresses: tests/test_host_faults.py)."""
    import wick_amd as W

    buf, host = ctx.alloc(8192), np.zeros(nbytes, np.uint8)
    for off in (0, 16):
        for call in (lambda: ctx._lib.wick_rocm_upload(ctx._h, buf.ptr + off, host.ctypes.data, nbytes),
                     lambda: ctx._lib.wick_rocm_download(ctx._h, host.ctypes.data, buf.ptr + off, nbytes)):
            with pytest.raises(W.RocmError, match="range"):
                ctx._check(call())
    buf.free()


@pytest.mark.parametrize("pinned", [False, True])
def test_memory_of_other_allocators(ctx, pinned):
    """A pointer into the middle of an allocation that the caller made, on the device or (pinned) on the host."""
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so")
    src, p = np.random.default_rng(3).integers(0, 256, 100_000, dtype=np.uint8), ctypes.c_void_p()
    assert (hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(150_000), 0) if pinned else hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(150_000))) == 0
    for off in (4096, 4099):
        back = np.empty_like(src)
        ctx._check(ctx._lib.wick_rocm_upload(ctx._h, p.value + off, src.ctypes.data, src.nbytes))
        ctx._check(ctx._lib.wick_rocm_download(ctx._h, back.ctypes.data, p.value + off, src.nbytes))
        assert np.array_equal(back, src)
    assert (hip.hipHostFree(p) if pinned else hip.hipFree(p)) == 0
