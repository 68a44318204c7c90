"""GPU tier: the plain feed-forward's activation as the end of the product that forms its columns (rows, split sums, tiles) or behind it (large bf16 prompts), against
the float64 restatement of tests/layer_list_oracle.py: beside the mixer's columns (Fonapel) and of its own matrices with a bias (Vabuzen); widths that come in
fours and widths that do not.  The whole list's logits, tolerances of the families' own tests."""

import pytest
import torch

import layer_list_oracle as O
from layer_list_engine_helpers import TOL, make_engine, rel_err, tokens_for, whole

pytestmark = pytest.mark.gpu


def _fonapel(ff):
    return O.fonapel_config([O.attention_layer(heads=2, kv_heads=1, dim=32, vdim=32, ff=ff), O.delta_layer(heads=2, kv_heads=1, dim=32, vdim=32, ff=ff)], width=128)


def _vabuzen(ff):
    return O.vabuzen_config([O.vabuzen_attention_layer(mlp={"kind": "dense", "ff": ff})], width=128)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 16, 17, 191, 192, 260])
@pytest.mark.parametrize("ff", [256, 130, 77])
@pytest.mark.parametrize("family", ["Fonapel", "Vabuzen"])
def test_activation_behind_the_product(family, ff, n, dtype):
    config = _fonapel(ff) if family == "Fonapel" else _vabuzen(ff)
    make, forward = (O.make_fonapel_weights, O.fonapel_forward) if family == "Fonapel" else (O.make_vabuzen_weights, O.vabuzen_forward)
    W = make(config, seed=31)
    toks = tokens_for(config, n, seed=32)
    engine = make_engine(config, W, dtype)
    try:
        assert rel_err(whole(engine, toks), forward(config, W, toks)) < TOL[dtype]
    finally:
        engine.close()
