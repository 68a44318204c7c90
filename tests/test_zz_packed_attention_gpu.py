"""GPU tier: a packed prefill pass, whose sequences share one launch of the head preparation and one of the FlashAttention kernel, at lengths around the
kernels' blocks (8 tokens: the decode kernel's rows; 32-row query blocks, 64-token stages, items of 8 and 4 waves), over pages the kernel's forms treat apart
(16: no stage lies in one page; 64, 128: one does), going on from earlier context, bf16 and FP8 pages.

bf16: held against the float64 truth like every model-level test.  FP8: a packed and a solo prefill differ by what their projections round; the bound is three
times the solo run's own distance from the truth (two rounded paths, each at most 1.5 times the oracle's distance)."""

import numpy as np
import pytest

from helpers import TINY_CFG, check_against_truth, to_mlx_shaped
from oracle import tiny_oracle as O

pytestmark = [pytest.mark.gpu]

FIRST = [9, 1, 8, 33, 64, 65, 130]
SECOND = [70, 9, 1, 8, 64, 31, 3]


def _ids(n, seed):
    return [int(t) for t in np.random.default_rng(seed).integers(1, TINY_CFG["vocab_size"], size=n)]


def _packed(engine, prompts):
    for s in range(len(prompts)):
        engine.begin(s)
    engine.prefill_packed([(s, p[:n], False) for s, (p, n) in enumerate(zip(prompts, FIRST))])
    engine.prefill_packed([(s, p[n:], True) for s, (p, n) in enumerate(zip(prompts, FIRST))])
    got = engine.logits(len(prompts)).float().cpu().numpy()
    for s in range(len(prompts)):
        engine.release(s)
    return got


@pytest.mark.parametrize("page_size", [16, 64, 128])
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
def test_unequal_sequences_share_the_launches(page_size, kv):
    from tiny_llm_hip.engine import DecodeEngine

    w = O.make_qwen3_weights(TINY_CFG, seed=3, sigma=0.05)
    prompts = [_ids(a + b, 40 + i) for i, (a, b) in enumerate(zip(FIRST, SECOND))]
    engine = DecodeEngine(to_mlx_shaped(TINY_CFG, w), page_size=page_size, num_pages=48 if page_size > 16 else 96, max_batch=len(prompts), max_prefill_rows=512, kv_format=kv)
    try:
        got = _packed(engine, prompts)
        truth = np.stack([O.TruthQwen3(TINY_CFG, w).forward(p)[0, -1] for p in prompts])
        if kv == "bf16":
            oracle = np.stack([O.OracleQwen3(TINY_CFG, w).forward(p)[0, -1] for p in prompts])
            check_against_truth(got, oracle, truth, what=f"packed prefill, pages of {page_size}")
        else:
            solo = []
            for p, n in zip(prompts, FIRST):
                engine.begin(0)
                engine.prefill(0, p[:n], want_logits=False)
                engine.prefill(0, p[n:])
                solo.append(engine.logits(1)[0].float().cpu().numpy())
                engine.release(0)
            solo = np.stack(solo)
            assert np.abs(got - solo).max() <= 3.0 * np.abs(solo - truth).max()
        assert engine.stats()["pages_in_use"] == 0
    finally:
        engine.close()
