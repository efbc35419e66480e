"""The gated activation on its way into a bf16 product, with gates from zero over tiny ones to thousands (where e^-z overflows, and where it vanishes): against the plain numpy
restatement within the bf16 tolerance of the other layer-list tests."""
import numpy as np
import pytest

import layered_util as U
from layered_util import BF16, Case, attention, chunked, close, config, delta, dense, kaparax, layer, retention, serial, tokens_for

pytestmark = pytest.mark.gpu

CONFIGS = {
    "silu": config(96, 64, [layer(attention(4, 2, 24, 24, 12, 40, 2), delta(2, 2, 24, 24, 3), dense(192))]),
    "clamped": kaparax(96, 64, [serial(retention(2, 32, 32, 16, [0.9, 0.99]), (192, 7.0)), serial(chunked(4, 2, 24, 24, 12, 64, 3, 8.0), (160, 2.0))]),
}
GAINS = [0.0, 1e-30, 1e-3, 1.0, 8.0, 100.0, 4000.0]


@pytest.mark.parametrize("rows", [1, 17, 70, 300])
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_gates_of_every_size(gpu, tmp_path, name, rows):
    cfg = CONFIGS[name]
    w = (U.kaparax_weights if name == "clamped" else U.random_weights)(cfg, 11)
    for i, L in enumerate(cfg["layers"]):
        g = np.resize(GAINS, L["mlp"]["ff"])[:, None]
        w["l%d.mlp.gate" % i] = U.bf16_round(w["l%d.mlp.gate" % i] * g)
        w["l%d.mlp.up" % i] = U.bf16_round(w["l%d.mlp.up" % i] / np.maximum(g, 1.0))  # products of one size
    c = Case(gpu, tmp_path, cfg, w=w)
    toks = tokens_for(cfg, rows)
    want = c.want(toks)[0]
    got = U.feed(c.session("bfloat16"), 0, toks, [rows])
    assert np.isfinite(got).all() and close(got, want, BF16)


def test_activations_are_float32_ones_rounded_once(gpu, tmp_path):
    """a bf16 model's activations, one by one: a token's stream holds a single 1, so that gates and ups are weights; each activation has a channel of the stream for itself behind the norm
    of the layer's output, whose factor is known from a gate of 64 (silu(64) = 64).  Each is the rounding of the 64-bit value up to 8 units of 2^-24: expf 2, its sum and
    the division 1 each, the product 1, and room for double that."""
    n_in, ff, f32 = 128, 512, np.float32
    cfg = config(n_in + ff, n_in, [layer(attention(2, 2, 16, 16, 8, 40, 2), delta(2, 2, 16, 16, 2), dense(ff))])
    w, rng = U.random_weights(cfg, 5), np.random.default_rng(6)
    w["embed"] = np.eye(n_in, n_in + ff)
    gate, up = np.where(rng.random((ff, n_in)) < 0.7, rng.uniform(-80, -8, (ff, n_in)), rng.uniform(-8, 20, (ff, n_in))), rng.uniform(1, 2, (ff, n_in))
    gate[0], up[0] = 64.0, 1.0
    gate, up = U.bf16_round(gate), U.bf16_round(up)
    w["l0.norm1"], w["l0.norm2"] = np.zeros(n_in + ff), np.ones(n_in + ff)  # nothing of the mixers; the output as it is, over its root mean square
    w["l0.mlp.gate"], w["l0.mlp.up"] = (np.concatenate([t, np.zeros((ff, ff), f32)], 1) for t in (gate, up))
    w["l0.mlp.down"] = np.concatenate([np.zeros((n_in, ff)), np.eye(ff)])
    s = Case(gpu, tmp_path, cfg, w={k: U.bf16_round(v) for k, v in w.items()}).session("bfloat16")
    out = s.forward_streams([0] * n_in, range(n_in), range(n_in))[0]
    got = U.bf16_round((out[:, n_in:].astype(np.float64) * (64.0 / out[:, n_in:n_in + 1])).astype(f32)).T
    z = gate.astype(np.float64)
    want = z / (1 + np.exp(-z)) * up
    lo, hi = (U.bf16_round((np.abs(want) * (1 + d * 8 * 2.0 ** -24)).astype(f32)) for d in (-1, 1))
    assert np.all((lo <= np.abs(got)) & (np.abs(got) <= hi) & (np.sign(got) == np.sign(want))), np.sum((lo > np.abs(got)) | (np.abs(got) > hi))
