"""GPU tier: q and k normed and rotated in one launch, K and V written to a page in one launch, against the operators they stand for -- the same bits -- and
the forms the kernels do not take, which go operator by operator."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(shape, dtype, seed):
    return torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,Hq,Hk,D", [(1, 1, 32, 8, 128), (1, 1, 1, 1, 128), (2, 3, 5, 2, 128), (3, 17, 16, 8, 128), (1, 130, 7, 3, 128), (1, 5, 4, 2, 64)])
@pytest.mark.parametrize("offset", [0, 29999, "list", "tensor", "scalar"])
def test_norm_and_rotate(dtype, B, L, Hq, Hk, D, offset):
    from tiny_llm_hip.week2_kernels import FastRMSNorm, FastRoPE, norm_and_rotate

    per_row = [7 * b + 3 for b in range(B)]
    offset = {"list": per_row, "tensor": torch.tensor(per_row, dtype=torch.int64, device=DEV), "scalar": torch.tensor(11, device=DEV)}.get(offset, offset)
    q, k = _rand((B, L, Hq, D), dtype, 1), _rand((B, L, Hk, D), dtype, 2)
    nq, nk = FastRMSNorm(D, _rand((D,), torch.float32, 3), eps=1e-6), FastRMSNorm(D, _rand((D,), dtype, 4), eps=1e-5)
    rope = FastRoPE(D, 32768, 1000000)
    got = norm_and_rotate(q, k, nq, nk, rope, offset)
    for x, norm, out in ((q, nq, got[0]), (k, nk, got[1])):
        want = rope(norm(x), offset=offset).transpose(1, 2)
        assert out.shape == want.shape and torch.equal(out, want)


def test_norm_and_rotate_of_other_forms():
    from tiny_llm_hip.week2_kernels import FastRMSNorm, FastRoPE, norm_and_rotate

    base = _rand((1, 9, 6, 136), torch.bfloat16, 5)
    w = _rand((128,), torch.bfloat16, 6)
    for rope, x in ((FastRoPE(64, 4096, 10000), base[..., :128].contiguous()), (FastRoPE(128, 4096, 10000, traditional=True), base[..., :128].contiguous()),
                    (FastRoPE(128, 4096, 10000), base[..., 1:129])):
        norm = FastRMSNorm(128, w)
        for got in norm_and_rotate(x, x, norm, norm, rope, 5):
            assert torch.equal(got, rope(norm(x), offset=5).transpose(1, 2))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,D,page,length,start", [(8, 128, 128, 128, 0), (8, 128, 128, 1, 127), (3, 128, 16, 7, 4), (2, 24, 8, 3, 1), (2, 20, 8, 3, 1), (1, 8, 4, 4, 0)])
@pytest.mark.parametrize("form", ["whole", "tokens_first", "shifted", "strided_rows"])
def test_paged_cache_write(dtype, H, D, page, length, start, form):
    import tiny_llm_ext_hip as ext

    if form == "tokens_first":
        make = lambda s: _rand((1, length + 2, H, D), dtype, s).transpose(1, 2)[:, :, 1:1 + length]
    elif form == "shifted":
        make = lambda s: _rand((1, H, length, D + 8), dtype, s)[..., 1:D + 1]  # not on 16 bytes
    elif form == "strided_rows":
        make = lambda s: _rand((1, H, length, 2 * D), dtype, s)[..., ::2]
    else:
        make = lambda s: _rand((1, H, length, D), dtype, s)
    k, v = make(1), make(2)
    kp, vp = _rand((5, H, page, D), dtype, 3), _rand((5, H, page, D), dtype, 4)
    want = [ext.paged_cache_update(p.clone(), x.contiguous(), 3, start) for p, x in ((kp, k), (vp, v))]
    before = kp.clone(), vp.clone()
    took = ext.paged_cache_write(kp, vp, k, v, 3, start)
    assert took == (form in ("whole", "tokens_first") and D * k.element_size() % 16 == 0)
    assert torch.equal(kp, want[0] if took else before[0]) and torch.equal(vp, want[1] if took else before[1])
    assert not ext.paged_cache_write(kp, vp, k, v, 5, 0) and not ext.paged_cache_write(kp, vp, k, v, 0, page - length + 1)
