"""GPU tier: the recurrences of prompts in chunks of 64 tokens (csrc/recur_chunk.h) against the float64 restatement of tests/layer_list_oracle.py, at
the sizes where they can go wrong: a chunk not full, full, one token more; state columns that end inside a block of 16; both key widths; grouped heads;
several sequences of unequal length in one step; a prompt that goes on from a state; decays that underflow inside a block.

The residual stream behind the layer is compared row by row, float32: sums of up to 128 + 64 float32 terms a token and what the stream around them
rounds, 1e-5 of the row (the tolerance of the token loop's own tests); 2e-4 on the logits as everywhere."""

import numpy as np
import pytest

import layer_list_oracle as O
from layer_list_engine_helpers import TOL, make_engine, rel_err, tokens_for

import torch

pytestmark = pytest.mark.gpu

RETENTION = [0.5, 0.97, 1.0]


def _fonapel(**kw):
    return O.fonapel_config([O.delta_layer(ff=0, **kw)]), O.make_fonapel_weights, O.fonapel_forward


def _zefapel(layer):
    return O.zefapel_config([layer]), O.make_zefapel_weights, O.zefapel_forward


CASES = {
    "delta": lambda: _fonapel(heads=4, kv_heads=2, dim=64, vdim=24, conv=3),
    "delta_wide": lambda: _fonapel(heads=3, kv_heads=3, dim=128, vdim=128, conv=4),
    "delta_odd_columns": lambda: _fonapel(heads=2, kv_heads=1, dim=128, vdim=37, conv=1),
    "mlstm": lambda: _zefapel(O.mlstm_layer(heads=2, dim=128, vdim=64)),     # the normaliser's column starts a block
    "mlstm_odd_columns": lambda: _zefapel(O.mlstm_layer(heads=3, dim=64, vdim=19)),
    "gla": lambda: _zefapel(O.gla_layer(heads=2, dim=128, vdim=48, a_rank=8)),
    "gla_odd_columns": lambda: _zefapel(O.gla_layer(heads=3, dim=64, vdim=21, a_rank=4)),
    "retention": lambda: (O.muduvik_config([O.muduvik_retention(heads=3, dim=64, vdim=40, rot_dims=16, decay=RETENTION)]), O.make_muduvik_weights, O.muduvik_forward),
}


def _check(config, W, forward, toks, portions, start=0):
    streams = []
    want = forward(config, W, toks, streams)
    engine = make_engine(config, W)
    try:
        engine.set_trace(True)
        engine.begin(0)
        at = 0
        for n in portions:
            part = toks[at:at + n]
            got = engine.logits_host(engine.step([(0, part, list(range(n)))]))
            assert rel_err(engine.read_trace(0, n), streams[0][at:at + n]) < 1e-5, f"rows {at} .. {at + n}"
            assert rel_err(got, want[at:at + n]) < TOL[torch.float32]
            at += n
        engine.release(0)
    finally:
        engine.close()


@pytest.mark.parametrize("n", [48, 63, 64, 65, 128, 201])
@pytest.mark.parametrize("case", sorted(CASES))
def test_prompt_lengths(case, n):
    config, make, forward = CASES[case]()
    _check(config, make(config, seed=1), forward, tokens_for(config, n, seed=n), [n])


@pytest.mark.parametrize("case", sorted(CASES))
def test_prompt_in_portions(case):
    """The state a chunked portion leaves feeds the token loop and the next chunks, and the other way round."""
    config, make, forward = CASES[case]()
    _check(config, make(config, seed=2), forward, tokens_for(config, 260, seed=3), [70, 1, 64, 5, 120])


@pytest.mark.parametrize("case", ["delta", "mlstm", "gla"])
def test_unequal_sequences_in_one_step(case):
    config, make, forward = CASES[case]()
    W = make(config, seed=4)
    seqs = [tokens_for(config, n, seed=10 + n) for n in (1, 130, 64, 17)]
    engine = make_engine(config, W)
    try:
        for s in range(len(seqs)):
            engine.begin(s)
        got = engine.logits_host(engine.step([(s, t, list(range(len(t)))) for s, t in enumerate(seqs)]))
        at = 0
        for t in seqs:
            assert rel_err(got[at:at + len(t)], forward(config, W, t)) < TOL[torch.float32]
            at += len(t)
        more = engine.logits_host(engine.step([(s, [7], [0]) for s in range(len(seqs))]))
        for s, t in enumerate(seqs):
            assert rel_err(more[s:s + 1], forward(config, W, t + [7])[-1:]) < TOL[torch.float32]
    finally:
        engine.close()


@pytest.mark.parametrize("case", ["delta_wide", "mlstm", "gla", "gla_odd_columns"])
@pytest.mark.parametrize("strength", ["vanishing", "some_channels", "none"])
def test_decays_at_their_limits(case, strength):
    """Decays whose products leave float32's range inside a block of 16 tokens (all, or those of a few heads or channels), and decays of 1."""
    config, make, forward = CASES[case]()
    W = make(config, seed=5)
    m = "l0.mix."
    far = {"vanishing": 1.0, "some_channels": 1.0, "none": -1.0}[strength]
    if case.startswith("delta"):
        b = W[m + "dt_bias"].copy()
        b[:] = -30.0 if far < 0 else b
        b[: 1 if strength == "some_channels" else len(b)] += 25.0 * far if far > 0 else 0.0
        W[m + "dt_bias"] = b
    elif case.startswith("mlstm"):
        b = W[m + "f.b"].copy()
        b[: 1 if strength == "some_channels" else len(b)] = -40.0 * far  # capped at the layer's gate cap
        W[m + "f.b"] = b
    else:
        b = W[m + "a2.b"].copy()
        b[: 3 if strength == "some_channels" else len(b)] = -120.0 * far
        W[m + "a2.b"] = b
    toks = tokens_for(config, 150, seed=6)
    streams = []
    forward(config, W, toks, streams)
    engine = make_engine(config, W)
    try:
        engine.set_trace(True)
        engine.begin(0)
        engine.step([(0, toks, [])])
        got = engine.read_trace(0, len(toks))
        assert np.isfinite(got).all()
        assert rel_err(got, streams[0]) < 1e-5
    finally:
        engine.close()
