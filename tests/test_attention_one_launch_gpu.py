"""Decode steps whose window fits the LDS of a CU: scores and class chains in one launch give the fused kernels' logits, keys and values bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def f16_bits(rng, shape, scale):
    return rng.normal(0, scale, shape).astype(np.float16).view(np.uint16)


# the largest window that fits, one past it (the forms for windows up to 512), a window of no whole four, a tiny one
@pytest.mark.parametrize("window", [496, 497, 131, 5])
@pytest.mark.parametrize("heads,grp", [(8, 4), (8, 2), (32, 4)])
def test_one_launch_is_the_fused_kernels_bit_for_bit(gpu, monkeypatch, heads, grp, window):
    """positions with empty classes (0 .. 3), classes that fill sixteens or spill by one (63 .. 65, 255 .. 257), the last ones; an infinite and a NaN value behind the context"""
    hp = gpu.LlmHParams(2, 128 * heads, heads, heads // grp, 128, 1024, 512, 1e-5, 10000.0, 0, 0, 0, 0, 1)
    model = gpu.LlmModel(hp).fill_synthetic(4)
    hp = model.hparams
    at = [c for c in (window - 1, window - 2, 320, 257, 256, 255, 66, 65, 64, 63, 17, 16, 15, 4, 3, 2, 1, 0) if c < window]
    cases = [(rows, c) for c in at for rows in (1, 2)]
    rng = np.random.default_rng(heads + grp)
    kv = []
    for _ in range(4):
        k, v = f16_bits(rng, (window, hp.n_kv_head, 128), 0.6), f16_bits(rng, (window, hp.n_kv_head, 128), 1.0)
        if window > 300:
            v[321:], v[330:340] = 0x7E00, 0x7C00  # read by no case that comes behind (they go downwards), and by the first two as what they are
        kv.append((k, v))
    runs = {}
    for off in ("0", "1"):
        monkeypatch.setenv("TK_MI355X_NO_LONG_ATT", off)
        sess = gpu.LlmSession(model, 2, window)
        for layer in range(2):
            for s in range(2):
                sess.kv_write(layer, s, 0, *kv[2 * layer + s])
        if off == "0" and gpu.lib().tk_mi355x_device_cu_count(0) == 256 and window <= 496:
            assert all(gpu.attention_plan(rows, hp.n_head, hp.n_kv_head, 128, window, True, top_position=0)[0] == 3 for rows in (1, 2))
        for rows, ctx in cases:
            tok = (np.arange(rows) + ctx % 400 + 3).astype(np.int32)
            logits, ids = sess.forward(np.arange(rows, dtype=np.int32), np.full(rows, ctx, np.int32), tok)
            runs[off, rows, ctx] = logits.copy(), ids.copy(), [sess.kv_read(layer, 0, ctx, 1) for layer in range(2)]
        sess.close()
    for off, rows, ctx in [k for k in runs if k[0] == "0"]:
        a, b = runs["0", rows, ctx], runs["1", rows, ctx]
        same = np.array_equal(a[0], b[0], equal_nan=True) if ctx > 320 else np.array_equal(a[0].view(np.uint32), b[0].view(np.uint32)) and np.isfinite(a[0]).all()
        assert same, (rows, ctx)
        assert all(np.array_equal(x, y) for u, v in zip(a[2], b[2]) for x, y in zip(u, v)) or ctx > 320, (rows, ctx)
    model.close()
