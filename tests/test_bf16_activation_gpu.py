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
