"""Wide prompt passes whose o and down projections add the first K ranges up in the workgroups that make them: every row's logits are, bit for bit, those
of passes that leave each range in a slab of its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WIDTH, FF, VOCAB = 4096, 14336, 512


@pytest.fixture(scope="module")
def model(gpu):
    # four layers: Q6_K and Q4_K down projections
    return gpu.LlmModel(gpu.LlmHParams(4, WIDTH, 32, 8, 128, FF, VOCAB, 1e-5, 10000.0, 0, 0, 0, 0, 1)).fill_synthetic(9)


# rows of the whole pass: parts of 96 (two ranges of down in one workgroup), of 128 with a ragged last part (two of down), four of down and two of o, all of both
@pytest.mark.parametrize("seqs,prompt", [(9, 32), (19, 23), (16, 64), (31, 65), (64, 32)])
def test_rows_of_a_wide_pass_equal_rows_of_narrow_passes(gpu, model, seqs, prompt):
    rng = np.random.default_rng(seqs)
    toks = rng.integers(3, VOCAB, (seqs, prompt)).astype(np.int32)
    wide, narrow = gpu.LlmSession(model, seqs, prompt + 8), gpu.LlmSession(model, seqs, prompt + 8)
    first = wide.prefill(toks)
    rows, per = np.arange(seqs, dtype=np.int32), max(1, 190 // prompt)  # 190 rows: not the wide kernel
    want = []
    for at in range(0, seqs, per):
        some = rows[at:at + per]
        pos = np.tile(np.arange(prompt, dtype=np.int32), len(some))
        last = narrow.forward(np.repeat(some, prompt), pos, toks[some].reshape(-1))
        want.append(last[1].reshape(len(some), prompt)[:, -1])
    assert np.array_equal(first, np.concatenate(want))
    at = np.full(seqs, prompt, np.int32)
    for s in range(0, seqs, 16):  # the next position reads every key and value that the passes left
        a = wide.forward(rows[s:s + 16], at[s:s + 16], first[s:s + 16])[0]
        b = narrow.forward(rows[s:s + 16], at[s:s + 16], first[s:s + 16])[0]
        assert np.isfinite(a).all() and np.array_equal(a.view(np.uint32), b.view(np.uint32))
