"""GPU tier: many decode steps in one call (tl_hybrid_decode_ids) against as many calls of one step: the ids, through pages that fill on the way, and
where the pool runs dry in the middle."""

import pytest

import layer_list_oracle as O
from layer_list_engine_helpers import make_engine, tokens_for

pytestmark = pytest.mark.gpu

CONFIG = O.fonapel_config([O.delta_layer(heads=2, kv_heads=1, dim=32, vdim=16, conv=4), O.attention_layer(heads=4, kv_heads=2, dim=32, vdim=32, rot_dims=16)])


def _start(engine, prompts):
    for s, p in enumerate(prompts):
        engine.begin(s)
        engine.prefill(s, p)


@pytest.mark.parametrize("steps", [1, 37, 256, 300])
def test_steps_of_one_call(steps):
    W = O.make_fonapel_weights(CONFIG, seed=8)
    prompts = [tokens_for(CONFIG, n, seed=n) for n in (5, 31, 16)]
    one, many = (make_engine(CONFIG, W, num_pages=80, max_pages_per_seq=24) for _ in range(2))
    try:
        _start(one, prompts)
        _start(many, prompts)
        for _ in range(steps):
            one.decode(1, slots=[2, 0, 1])
        many.decode(steps, slots=[2, 0, 1])
        for s in range(3):
            assert many.read_tokens(s, steps + 1) == one.read_tokens(s, steps + 1)
            assert many.context_len(s) == one.context_len(s)
        assert many.read_pending_slots([0, 1, 2]) == one.read_pending_slots([0, 1, 2])
    finally:
        one.close()
        many.close()


def test_pool_that_runs_dry_keeps_the_steps_before():
    W = O.make_fonapel_weights(CONFIG, seed=8)
    engine = make_engine(CONFIG, W, num_pages=3, max_pages_per_seq=8, max_batch=1)
    try:
        engine.begin(0)
        engine.prefill(0, tokens_for(CONFIG, 20, seed=1))
        with pytest.raises(RuntimeError, match="pool exhausted"):
            engine.decode(60, slots=[0])
        n = engine.context_len(0)
        assert n == 3 * 16 and len(engine.read_tokens(0, n - 20 + 1)) == n - 20 + 1
        assert engine.read_pending_slots([0]) == engine.read_tokens(0, 1)
    finally:
        engine.close()
