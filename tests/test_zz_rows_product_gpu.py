"""GPU tier: the layer-list engine's products for up to 16 rows (csrc/hybrid_kernels.h gemm_rows_kernel and its any-layout twin) and for 17 .. 191 rows
(gemm_mid_kernel) against float64, at the borders of their forms: 4, 8 and 16 columns a block; K of a piece, a chunk, several batches of chunks and remainders; one wave to four sharing a block's K; rows behind M and
columns behind N.

Tolerance per element: float32 sums of K products, each rounded at most twice, in any order: K * 2^-23 of sum |a w| is a bound; sqrt(K) * 2^-22 is what
independent roundings give with a factor of 4 to spare."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _product(dtype, M, N, K, lda=None, offset=0):
    import tiny_llm_ext_hybrid as ext

    gen = torch.Generator(device="cuda").manual_seed(1000 * M + N + K)
    td = torch.bfloat16 if dtype == "bf16" else torch.float32
    lda = lda or K
    a = torch.randn((M, lda), generator=gen, device="cuda").to(td)
    flat = torch.randn(N * K + offset, generator=gen, device="cuda").to(td)
    w = flat[offset:]
    out = torch.full((M + 1, N), 7.0, device="cuda")
    ext.check(ext.lib().tl_hybrid_linear(ext.HY_BF16 if dtype == "bf16" else ext.HY_F32, a.data_ptr(), lda, w.data_ptr(), out.data_ptr(), N, M, N, K, 0, None))
    torch.cuda.synchronize()
    x, y = a[:, :K].double(), w.reshape(N, K).double()
    want, bound = x @ y.T, (x.abs() @ y.abs().T) * (max(16.0, K) ** 0.5 * 2.0 ** -22)
    assert bool(((out[:M].double() - want).abs() <= bound + 1e-30).all()), float(((out[:M].double() - want).abs() / bound).max())
    assert bool((out[M] == 7.0).all()), "a row behind M was written"


@pytest.mark.parametrize("dtype", ["bf16", "float32"])
@pytest.mark.parametrize("M", [1, 3, 4, 5, 8, 9, 15, 16])
@pytest.mark.parametrize("N,K", [(1, 8), (3, 24), (4, 32), (5, 128), (17, 136), (64, 1024), (66, 1032), (130, 4096), (1024, 2056), (4100, 512)])
def test_rows_product(dtype, M, N, K):
    _product(dtype, M, N, K)


@pytest.mark.parametrize("dtype", ["bf16", "float32"])
@pytest.mark.parametrize("M", [1, 7, 8])
@pytest.mark.parametrize("K,lda,offset", [(100, 100, 0), (96, 100, 0), (96, 96, 3), (13, 21, 1)])
def test_rows_product_any_layout(dtype, M, K, lda, offset):
    """K, row strides and alignments that 16-byte loads do not fit."""
    _product(dtype, M, 37, K, lda, offset)


@pytest.mark.parametrize("dtype", ["bf16", "float32"])
@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64, 65, 129, 191])
@pytest.mark.parametrize("N,K", [(1, 8), (5, 72), (31, 64), (33, 256), (64, 520), (100, 2056), (1030, 136)])
def test_mid_product(dtype, M, N, K):
    _product(dtype, M, N, K)


@pytest.mark.parametrize("M,N,K", [(192, 33, 256), (250, 64, 520), (1000, 130, 72), (1000, 1984, 136), (1000, 2047, 136)])  # (the last: 512 tiles of 64 x 64)
def test_mid_product_of_many_rows(M, N, K):
    _product("float32", M, N, K)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [17, 40, 70])
def test_products_that_split_their_sums_over_workgroups(n, dtype):
    """Few columns of a long K (the feed-forward's way back): partial sums of several workgroups, in every epilogue form a layer's sums take."""
    import layer_list_oracle as O
    from layer_list_engine_helpers import TOL, make_engine, rel_err, tokens_for, whole

    for config, make, forward in ((O.fonapel_config([O.attention_layer(ff=4096)]), O.make_fonapel_weights, O.fonapel_forward),
                                  (O.zefapel_config([O.latent_layer(mlp=O.dense_ff(4096)), O.gla_layer(mlp=O.dense_ff(4096))]), O.make_zefapel_weights, O.zefapel_forward)):
        W = make(config, seed=21)
        toks = tokens_for(config, n, seed=22)
        engine = make_engine(config, W, dtype)
        try:
            assert rel_err(whole(engine, toks), forward(config, W, toks)) < TOL[dtype]
        finally:
            engine.close()
