"""GPU tier: the bf16 tile GEMM (csrc/gemm8.h) on 128-row tiles with three and four LDS stages, against float64: reductions of exactly the stages, one step
more, fewer (the two-stage tiles take those); ragged rows and columns; and workgroups that walk several tiles, whose first step after a tile's stores
waits for all of them.

Tolerance per element as in test_zz_rows_product_gpu: sqrt(K) * 2^-22 of sum |a w|."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (192, 64, 128), (200, 132, 192), (129, 128, 256), (257, 260, 320), (130, 1000, 448),     # 128 x 128: stages, remainders
    (1900, 4096, 192), (1900, 4096, 256),                                                      # 128 x 256
    (2000, 2560, 256), (1985, 2556, 320),                                                      # 128 x 160, one tile a workgroup
    (100, 81916, 256), (100, 81920, 384),                                                      # ... two tiles
    (100, 98300, 256), (128, 98304, 320),                                                      # 128 x 128, three tiles
])
def test_tile_stages(M, N, K):
    import tiny_llm_ext_hybrid as ext

    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randn((M, K), generator=gen, device="cuda").to(torch.bfloat16)
    w = torch.randn((N, K), generator=gen, device="cuda").to(torch.bfloat16)
    out = torch.full((M + 1, N), 7.0, device="cuda")
    ext.check(ext.lib().tl_hybrid_linear(ext.HY_BF16, a.data_ptr(), K, w.data_ptr(), out.data_ptr(), N, M, N, K, 3, None))
    torch.cuda.synchronize()
    assert bool((out[M] == 7.0).all()), "a row behind M was written"
    for c in range(0, N, 16384):  # (float64 products of a piece of the columns at a time)
        y = w[c:c + 16384].double()
        want, bound = a.double() @ y.T, (a.double().abs() @ y.abs().T) * (K ** 0.5 * 2.0 ** -22)
        assert bool(((out[:M, c:c + 16384].double() - want).abs() <= bound).all())


@pytest.mark.parametrize("n", [191, 192, 700])
def test_chunks_whose_projections_take_either_gemm(n):
    """Chunks far below the engine's largest: every projection on the GEMM its estimate names (below 192 rows always the 4-bit one), against the float64
    truth with the band every model-level test uses."""
    import numpy as np

    from helpers import TINY_CFG, check_against_truth, to_mlx_shaped
    from oracle import tiny_oracle as O
    from tiny_llm_hip.engine import DecodeEngine

    weights = O.make_qwen3_weights(TINY_CFG, seed=12, sigma=0.05)
    prompt = [int(t) for t in np.random.default_rng(n).integers(1, TINY_CFG["vocab_size"], size=n)]
    eng = DecodeEngine(to_mlx_shaped(TINY_CFG, weights), page_size=128, num_pages=9, max_batch=1, max_prefill_rows=2048)
    try:
        eng.begin(0)
        eng.prefill(0, prompt)
        got = eng.logits(1)[0].float().cpu().numpy()
    finally:
        eng.close()
    ref, truth = O.OracleQwen3(TINY_CFG, weights), O.TruthQwen3(TINY_CFG, weights)
    check_against_truth(got[None], ref.forward(prompt)[0, -1][None], truth.forward(prompt)[0, -1][None], what=f"engine prefill of {n} rows")
