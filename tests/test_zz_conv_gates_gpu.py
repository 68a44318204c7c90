"""GPU tier: the short convolutions ahead of the delta rule (four columns and eight rows a thread; steps of single tokens in one launch with their
state) and the scan of exponential gates over several waves, against the float64 restatement of tests/layer_list_oracle.py, where they can go wrong:
filters of one tap, of the templates' taps, one more (the general kernel); columns that do not come in fours; portions shorter than a filter;
sequences of unequal length in one step; prompts of a pass of the scan, one token more, several passes.

The residual stream behind the layer is compared row by row, float32: 1e-5 of the row (the token loop's tolerance; a convolution adds at most 9 terms,
and the scan's sums are those of a single wave)."""

import pytest

import layer_list_oracle as O
from layer_list_engine_helpers import TOL, make_engine, rel_err, tokens_for

import torch

pytestmark = pytest.mark.gpu

CONV = {
    "one_tap": dict(heads=2, kv_heads=1, dim=32, vdim=16, conv=1),
    "two_taps": dict(heads=2, kv_heads=2, dim=20, vdim=12, conv=2),
    "four_taps": dict(heads=4, kv_heads=2, dim=64, vdim=24, conv=4),
    "five_taps": dict(heads=4, kv_heads=2, dim=32, vdim=16, conv=5),
    "eight_taps": dict(heads=2, kv_heads=1, dim=16, vdim=8, conv=8),
    "nine_taps": dict(heads=2, kv_heads=1, dim=16, vdim=8, conv=9),
    "odd_columns": dict(heads=1, kv_heads=1, dim=24, vdim=33, conv=4),
}


def _run(config, W, forward, seqs, steps):
    """seqs: the whole token sequences; steps: per step the number of tokens of every sequence (0: it does not take part)."""
    streams = []
    want = []
    for toks in seqs:
        s = []
        want.append(forward(config, W, toks, s))
        streams.append(s[0])
    engine = make_engine(config, W, num_pages=160, max_prefill_rows=2304)
    try:
        engine.set_trace(True)
        for slot in range(len(seqs)):
            engine.begin(slot)
        at = [0] * len(seqs)
        for step in steps:
            parts = [(slot, seqs[slot][at[slot]:at[slot] + n], list(range(n))) for slot, n in enumerate(step) if n]
            got = engine.logits_host(engine.step(parts))
            rows = engine.read_trace(0, sum(step))
            r = 0
            for slot, n in enumerate(step):
                if not n:
                    continue
                a = at[slot]
                assert rel_err(rows[r:r + n], streams[slot][a:a + n]) < 1e-5, f"slot {slot}, tokens {a} .. {a + n}"
                assert rel_err(got[r:r + n], want[slot][a:a + n]) < TOL[torch.float32]
                at[slot] += n
                r += n
    finally:
        engine.close()


@pytest.mark.parametrize("case", sorted(CONV))
def test_convolutions(case):
    config = O.fonapel_config([O.delta_layer(ff=0, **CONV[case])])
    W = O.make_fonapel_weights(config, seed=5)
    seqs = [tokens_for(config, n, seed=20 + n) for n in (43, 26, 12)]
    steps = [(1, 2, 1), (1, 1, 1), (17, 1, 2), (7, 3, 0), (1, 1, 1), (16, 18, 7)]
    _run(config, W, O.fonapel_forward, seqs, steps)


@pytest.mark.parametrize("portions", [(64,), (65, 1, 1), (1023, 2), (1024, 1), (1025, 64), (2049,)])
def test_gate_scan(portions):
    config = O.zefapel_config([O.mlstm_layer(heads=3, dim=16, vdim=12)])
    W = O.make_zefapel_weights(config, seed=6)
    _run(config, W, O.zefapel_forward, [tokens_for(config, sum(portions), seed=7)], [(n,) for n in portions])
