"""Whole prompts (prefill) against the same rows through passes of at most 256 rows (forward, which other tests hold to the oracle): the sampled ids, and the logits of the
position behind each prompt, which read every key and value the prompt left, bit for bit.  Totals at the edges of the wide kernel's parts (96 and 128 rows) and of a pass (2048)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def models(gpu):
    made = {}

    def get(name):
        if name not in made:
            hp = {"tiny": gpu.TINY(), "tiny-f16": gpu.TINY(),
                  "wide": gpu.LlmHParams(2, 1024, 8, 2, 128, 2048, 512, 1e-5, 10000.0, 0, 0, 0, 0, 1),
                  "wide-f16": gpu.LlmHParams(2, 1024, 8, 2, 128, 2048, 512, 1e-5, 10000.0, 0, 0, 0, 0, 1)}[name]
            made[name] = gpu.LlmModel(hp).fill_synthetic(4, f16=name.endswith("f16"))
        return made[name]
    return get


@pytest.mark.parametrize("model", ["tiny", "tiny-f16", "wide", "wide-f16"])
@pytest.mark.parametrize("nseq,n_prompt", [(1, 1), (1, 2), (2, 1), (3, 1), (5, 2), (1, 33), (3, 65), (1, 257), (3, 96), (9, 32), (1, 385), (256, 2), (2, 300), (7, 130), (32, 32), (41, 25), (3, 683), (64, 33), (1, 2100)])
def test_prefill_equals_passes_of_256_rows(gpu, models, model, nseq, n_prompt):
    m = models(model)
    vocab = m.hparams.vocab
    rng = np.random.default_rng(nseq * 1000 + n_prompt)
    toks = rng.integers(3, vocab, (nseq, n_prompt)).astype(np.int32)
    follow = rng.integers(3, vocab, nseq).astype(np.int32)
    seq, pos = np.repeat(np.arange(nseq, dtype=np.int32), n_prompt), np.tile(np.arange(n_prompt, dtype=np.int32), nseq)
    one, other = gpu.LlmSession(m, nseq, n_prompt + 4), gpu.LlmSession(m, nseq, n_prompt + 4)
    for _ in range(2):  # a second call finds the first one's caches and buffers
        first = one.prefill(toks)
    ids, _ = one.decode(nseq, 1)
    got, got_ids = one.forward(np.arange(nseq, dtype=np.int32), np.full(nseq, n_prompt, np.int32), follow)
    flat, picked = toks.ravel(), np.zeros(nseq * n_prompt, np.int32)
    for r in range(0, flat.size, 256):
        _, picked[r:r + 256] = other.forward(seq[r:r + 256], pos[r:r + 256], flat[r:r + 256])
    want_first = picked[n_prompt - 1::n_prompt]
    _, want_ids = other.forward(np.arange(nseq, dtype=np.int32), np.full(nseq, n_prompt, np.int32), want_first)
    want, _ = other.forward(np.arange(nseq, dtype=np.int32), np.full(nseq, n_prompt, np.int32), follow)
    assert np.array_equal(first, want_first)
    assert np.array_equal(ids[0], want_ids)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.abs(got - want).max()


@pytest.mark.parametrize("model", ["wide", "wide-f16"])
@pytest.mark.parametrize("rows", [1, 2, 3, 40])
def test_passes_without_a_head_leave_every_layers_keys_and_values(gpu, models, monkeypatch, model, rows):
    """one position of each sequence whose logits nobody wants, as plain launches and as a graph, at row counts of either kind of product: what the next position reads is the same,
    and what a pass with a head leaves"""
    m = models(model)
    toks = np.random.default_rng(rows).integers(3, m.hparams.vocab, (2, rows)).astype(np.int32)
    got = {}
    for name, graphs, head in (("head", "0", True), ("graph", "0", False), ("plain", "1", False)):
        monkeypatch.setenv("TK_MI355X_NO_GRAPH", graphs)
        s = gpu.LlmSession(m, rows, 8)
        s.forward_rows(range(rows), [0] * rows, toks[0], range(rows) if head else [], want_logits=head)
        got[name] = s.forward(np.arange(rows), np.ones(rows), toks[1])[0].view(np.uint32)
    assert np.array_equal(got["graph"], got["head"]) and np.array_equal(got["plain"], got["head"])


@pytest.mark.parametrize("ctx,rows", [(64, 256), (2100, 2048)])
def test_memory_of_a_session(gpu, ctx, rows):
    """what a pass of `rows` rows writes once: its K-split slabs, the residual stream, queries, activation images (their sums are 0.4 of their bytes), the logits of 256 rows and the caches;
    a tenth and 48 MB for tables, what is kept of 256 sampled rows and the allocator's pages"""
    import gc

    import torch
    m = gpu.LlmModel(gpu.LlmHParams(1, 4096, 32, 8, 128, 14336, 32000, 1e-5, 10000.0, 0, 0, 0, 0, 1)).fill_synthetic(4)
    h = m.hparams
    slabs = max(h.ks_qkv * 6144, h.ks_o * 4096, h.ks_gateup * 2 * 14336, h.ks_down * 4096)
    need = 4 * rows * (slabs + 2 * 4096) + 1.4 * rows * (2 * 4096 + 14336) + 4 * 256 * 32000 + 4 * ctx * 1024
    gc.collect()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info(0)[0]
    s = gpu.LlmSession(m, 1, ctx)
    used = before - torch.cuda.mem_get_info(0)[0]
    s.close()
    assert used < 1.1 * need + (48 << 20), (used >> 20, int(need) >> 20)
