"""fp32 LM head of few rows (the weight-streaming kernel and the tile kernel around it) against
float64: every row bucket, column and k-tile remainders, gathered and inactive rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("M,N,H", [(1, 64, 128), (16, 65, 256), (17, 1000, 512), (32, 63, 384), (33, 4096, 128),
                                   (64, 130, 1408), (65, 70, 128), (8, 100, 192), (5, 1, 128)])
def test_f32_rows_match_float64(M, N, H):
    from flashgrpo_amd import kernels as K

    g = torch.Generator(device=DEV).manual_seed(M + N + H)
    x = torch.randn(M + 3, H, device=DEV, generator=g)
    w = torch.randn(N, H, device=DEV, generator=g)
    rows = torch.randperm(M + 3, device=DEV, generator=g)[:M].to(torch.int32)
    want = x[rows.long()].double() @ w.double().t().contiguous()
    # any order of H fused multiply-adds: at most H roundings of 2^-24 of the sum of magnitudes
    bound = H * 2.0 ** -24 * (x[rows.long()].double().abs() @ w.double().abs().t().contiguous())
    got = K.lm_head(x, w, row_index=rows)
    assert bool(((got.double() - want).abs() <= bound).all())
    direct = K.lm_head(x[rows.long()].contiguous(), w)
    assert torch.equal(direct, got)
    half = K.lm_head(x, w, row_index=rows, out_dtype=torch.bfloat16)
    assert torch.equal(half, got.to(torch.bfloat16))
    # nothing is computed when no row is active; otherwise the active rows are written
    out = torch.full((M, N), 7.0, device=DEV)
    K.lm_head(x, w, row_index=rows, row_active=torch.zeros(M, dtype=torch.int32, device=DEV), out=out)
    assert bool((out == 7.0).all())
    act = torch.zeros(M, dtype=torch.int32, device=DEV)
    act[M - 1] = 1
    K.lm_head(x, w, row_index=rows, row_active=act, out=out)
    assert torch.equal(out[M - 1], got[M - 1])
