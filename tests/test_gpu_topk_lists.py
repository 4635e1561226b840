"""fg_medusa_topk where its candidate list can go wrong: rows shorter than a pass, chunk and group
remainders, more equal maxima than a list holds, runs of -inf."""
import numpy as np
import pytest
import torch

from oracle import tree as OT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("V", [16, 2047, 2049, 10240, 10241, 20489])
@pytest.mark.parametrize("kmax", [1, 2, 3, 7, 16])
def test_lists_match_oracle(dtype, V, kmax):
    from flashgrpo_amd import kernels as K

    g = torch.Generator(device="cpu").manual_seed(V + kmax)
    x = torch.randn(8, V, generator=g)
    x[1] = torch.round(x[1])                     # long ties
    x[2, V // 2:] = x[2].max() + 1               # half the row shares the maximum
    x[3, 3:] = float("-inf")                     # fewer finite values than candidates, at times
    x[4, : V // 2] = float("-inf")
    x[5] = torch.arange(V).float() / 7           # ascending: the last elements win
    x[6] = -torch.arange(V).float() / 7
    x = x.to(dtype)
    for sanitize in (False, True):
        tok, sc, st = K.medusa_topk(x.cuda(), kmax, stats=True, sanitize=sanitize)
        xs = x.float().numpy()
        xs = OT.nan_to_num_logits(xs) if sanitize else xs
        for r in range(8):
            ids, vals = OT.topk_canonical(xs[r], kmax)
            assert tok[r].tolist() == ids.tolist(), (r, sanitize)
            assert np.array_equal(sc[r].cpu().numpy(), vals.astype(np.float32) + 0.0), (r, sanitize)
            m = float(xs[r].max())
            lse = np.log(np.sum(np.exp(xs[r].astype(np.float64) - m))) + m
            assert float(st[r, 0]) == m and abs(float(st[r, 1]) - lse) < 1e-4 * max(1.0, abs(lse)), (r, sanitize)
