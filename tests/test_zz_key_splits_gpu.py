"""GPU tier: single-token steps of the layer-list engine around the borders of their key splits (64 keys a split, four splits at least): splits without keys,
the last split's first key, value widths the merge takes four columns at a time and others, every tile kernel (bf16 pairs, float32, latent rows).
Against the float64 restatement, tolerances of the layer-list tests."""

import pytest
import torch

import layer_list_oracle as O
from layer_list_engine_helpers import TOL, make_engine, rel_err, tokens_for

pytestmark = pytest.mark.gpu

LAYERS = {
    "attention": (O.fonapel_config([O.attention_layer(heads=4, kv_heads=2, dim=32, vdim=32)]), O.make_fonapel_weights, O.fonapel_forward),
    "attention_wide": (O.fonapel_config([O.attention_layer(heads=4, kv_heads=1, dim=128, vdim=120)]), O.make_fonapel_weights, O.fonapel_forward),
    "attention_odd_values": (O.fonapel_config([O.attention_layer(heads=3, kv_heads=1, dim=24, vdim=18)]), O.make_fonapel_weights, O.fonapel_forward),
    "latent": (O.zefapel_config([O.latent_layer(heads=4, kv_rank=40)]), O.make_zefapel_weights, O.zefapel_forward),
    "latent_odd_rank": (O.zefapel_config([O.latent_layer(heads=3, rot_dim=6, kv_rank=26)]), O.make_zefapel_weights, O.zefapel_forward),
}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("layer", sorted(LAYERS))
def test_single_token_steps_across_split_borders(layer, dtype):
    config, make, forward = LAYERS[layer]
    W = make(config, seed=11)
    toks = tokens_for(config, 262, seed=12)
    want = forward(config, W, toks)
    engine = make_engine(config, W, dtype)
    try:
        engine.begin(0)
        at = 0
        for border in (1, 64, 128, 192, 256):  # a portion up to three tokens ahead of the border (two at the start), then single tokens across it
            if border - 3 > at:
                engine.step([(0, toks[at:border - 3], [])])
                at = border - 3
            while at < border + 3:
                got = engine.logits_host(engine.step([(0, [toks[at]], [0])]))
                assert rel_err(got, want[at:at + 1]) < TOL[dtype], f"token {at}"
                at += 1
        engine.release(0)
    finally:
        engine.close()
