"""Layer-list decoders: the rows whose logits are wanted, which alone go through the last layer behind its mixers, against the same rows of a pass that wants them all; and a pass
that wants none, whose keys, values and states the next one reads.  Float32 against the error of sums in another order, bf16 against that of its roundings (the tolerances that the
other tests of these decoders state)."""
import numpy as np
import pytest

import layered_util as U
from layered_util import attention, chunked, config, delta, dense, kaparax, layer, moe, retention, serial, tokens_for

pytestmark = pytest.mark.gpu

TOL = {"float32": 1e-5, "bfloat16": 0.03}
CONFIGS = {
    "delta": config(128, 96, [layer(attention(4, 2, 64, 64, 32, 70, 2), delta(4, 2, 64, 64, 4), dense(192))] * 2),
    "odd": config(93, 131, [layer(attention(4, 2, 24, 40, 12, 33, 3), delta(3, 3, 20, 36, 3), dense(70))] * 2),
    "experts": config(128, 96, [layer(attention(4, 2, 64, 64, 32, 70, 2), delta(4, 2, 64, 64, 4), moe(48, 4, 4))] * 2),  # all of them: no call of a router is close
    "attention last": kaparax(93, 96, [serial(retention(2, 33, 21, 12, [0.7, 0.97]), (50, 1.5)), serial(chunked(4, 2, 24, 40, 12, 33, 3, 4.0))]),
    "retention last": kaparax(96, 96, [serial(chunked(4, 2, 64, 64, 32, 48, 4, 15.0), (64, 2.0)), serial(retention(2, 64, 64, 64, [0.9, 0.99]), (64, 2.0))]),
}
LENGTHS = {"one": [40], "few": [65, 1, 30, 130], "many": [2] * 128, "most": [3] * 60 + [1] * 20, "long": [700]}


def wanted(name, lengths, n):
    ends = np.cumsum(lengths) - 1
    if name == "most":
        return list(range(0, n, 2)) + [n - 1] * (n % 2 == 0)  # more than half of the rows: all go on
    if name == "many":
        return list(ends)  # half of them, exactly
    if name == "long":
        return [0, 63, 64, 127, 350, 699]
    return list(ends)


@pytest.mark.parametrize("dtype", sorted(TOL))
@pytest.mark.parametrize("lengths", sorted(LENGTHS))
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_wanted_rows_of_the_last_layer(gpu, name, lengths, dtype):
    cfg, ns = CONFIGS[name], LENGTHS[lengths]
    m = gpu.LlmModel(config=cfg, dtype=dtype, seed=9)
    n = sum(ns)
    seq, pos = np.repeat(np.arange(len(ns)), ns), np.concatenate([np.arange(k) for k in ns])
    toks = tokens_for(cfg, n + len(ns))
    s, t, u = (gpu.LlmSession(m, len(ns), max(ns) + 8) for _ in range(3))
    out = wanted(lengths, ns, n)
    whole, _ = s.forward_rows(seq, pos, toks[:n], range(n))
    some, ids = t.forward_rows(seq, pos, toks[:n], out, want_ids=True)
    assert U.rel_rms(some, whole[out]) < TOL[dtype] and np.array_equal(ids, some.argmax(1))
    none, _ = u.forward_rows(seq, pos, toks[:n], [], want_logits=False)
    assert none is None
    nxt = [x.forward_rows(range(len(ns)), ns, toks[n:], range(len(ns)))[0] for x in (s, t, u)]
    assert U.rel_rms(nxt[1], nxt[0]) < TOL[dtype] and U.rel_rms(nxt[2], nxt[0]) < TOL[dtype]


# 32 wide: products over the width are one chain in every kernel, so that the head's sums don't depend on how many rows it takes; those of the last layer's other products do
NARROW = {
    "delta": config(32, 96, [layer(attention(4, 2, 64, 64, 32, 70, 2), delta(4, 2, 64, 64, 4), dense(576))] * 2),
    "deep": config(32, 96, [layer(attention(4, 2, 64, 64, 32, 70, 2), delta(4, 2, 64, 64, 4), dense(4096))]),
    "odd": config(31, 131, [layer(attention(4, 2, 24, 40, 12, 33, 3), delta(3, 3, 20, 36, 3), dense(1070))] * 2),
    "experts": config(32, 96, [layer(attention(4, 2, 64, 64, 32, 70, 2), delta(4, 2, 64, 64, 4), moe(448, 8, 2))] * 2),
    "retention last": kaparax(32, 96, [serial(chunked(4, 2, 64, 64, 32, 48, 4, 15.0), (64, 2.0)), serial(retention(4, 64, 64, 64, [0.9, 0.99, 0.5, 0.8]), (640, 2.0))]),
}


@pytest.mark.parametrize("dtype", sorted(TOL))
@pytest.mark.parametrize("lengths", ["one", "few", "many", "long"])
@pytest.mark.parametrize("name", sorted(NARROW))
def test_a_rows_logits_do_not_depend_on_which_others_are_wanted(gpu, name, lengths, dtype):
    """bit for bit those of a pass that wants all"""
    cfg, ns = NARROW[name], LENGTHS[lengths]
    m = gpu.LlmModel(config=cfg, dtype=dtype, seed=9)
    n = sum(ns)
    seq, pos, toks, out = np.repeat(np.arange(len(ns)), ns), np.concatenate([np.arange(k) for k in ns]), tokens_for(cfg, n + len(ns)), wanted(lengths, ns, n)
    s, t = (gpu.LlmSession(m, len(ns), max(ns) + 8) for _ in range(2))
    whole, _ = s.forward_rows(seq, pos, toks[:n], range(n))
    some, _ = t.forward_rows(seq, pos, toks[:n], out)
    assert np.array_equal(some.view(np.uint32), whole[out].view(np.uint32))
    nxt = [x.forward_rows(range(len(ns)), ns, toks[n:], range(len(ns)))[0] for x in (s, t)]
    assert np.array_equal(nxt[0].view(np.uint32), nxt[1].view(np.uint32))
