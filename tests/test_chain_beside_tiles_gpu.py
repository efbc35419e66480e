"""The chain of the delta rule's chunks with the attention tiles beside it in one launch (up to 256 workgroups of chains, heads of 64 or 128 in both branches), and the two as launches of
their own: the same sequences in passes on either side of that line, against the plain numpy restatement.  Float32 models take the second form always."""
import numpy as np
import pytest

import layered_util as U
from layered_util import BF16, Case, attention, close, config, delta, dense, layer, tokens_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,runs,length", [(64, 1, 72), (64, 1, 300), (64, 5, 90), (128, 1, 129), (128, 4, 90), (128, 5, 90), (128, 2, 200)])
def test_chain_and_tiles(gpu, tmp_path, dim, runs, length):
    heads = 8  # 4 or 8 workgroups of 16 columns a head: 5 runs of 128 are 320
    cfg = config(96, 64, [layer(attention(4, 2, dim, dim, 32, 70, 2), delta(heads, 4, dim, dim, 4), dense(96))] * 2)
    c = Case(gpu, tmp_path, cfg)
    toks = [tokens_for(cfg, length - 3 * i, i) for i in range(runs)]
    ns = [len(t) for t in toks]
    s = c.session("bfloat16", max_seq=8)
    seq, pos = np.repeat(np.arange(runs + 1), ns + [1]), np.concatenate([np.arange(n) for n in ns] + [np.zeros(1, int)])  # and a single row, which goes token by token
    flat = np.concatenate(toks + [[5]])
    for _ in range(2):
        got, _ = s.forward_rows(seq, pos, flat, range(len(flat)))
        at = 0
        for t in toks:
            assert close(got[at:at + len(t)], c.want(t)[0], BF16)
            at += len(t)
        assert U.rel_rms(got[at:], c.want([5])[0]) < BF16
