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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("V", [2049, 4097, 30001, 152065])
def test_nan_reaches_the_log_sum_exp(dtype, V):
    """One NaN anywhere makes the row's log-sum-exp NaN when the logits are ranked as they are, also
    where a thread holds nothing finite beside it; runs of -inf alone do not."""
    from flashgrpo_amd import kernels as K

    x = torch.randn(6, V + 7, generator=torch.Generator().manual_seed(V))[:, :V].clone()
    x[0, V - 1] = float("nan")                  # alone in its thread (V % 8 == 1)
    x[1, 8:16] = float("nan")                   # all eight of one thread
    x[2, 16:24] = float("-inf")
    x[2, 19] = float("nan")
    x[3, 1: V // 2] = float("-inf")
    x[4, :] = float("-inf")
    x[4, V // 2] = float("nan")                 # nothing finite in the row
    x = x.to(dtype)
    _, _, st = K.medusa_topk(x.cuda(), 2, stats=True, sanitize=False)
    st = st.cpu()
    assert torch.isnan(st[[0, 1, 2, 4], 1]).all(), st
    for r in (3, 5):
        want = float(torch.logsumexp(x[r].double(), 0))
        assert abs(float(st[r, 1]) - want) < 1e-4 * max(1.0, abs(want)), (r, st[r], want)


@pytest.mark.parametrize("M", [3, 40])
def test_nan_reaches_the_lm_head_log_sum_exp(M):
    """The same for the statistics of the LM head's epilogue: weight rows that give NaN or -inf logits."""
    from flashgrpo_amd import kernels as K

    V, H = 4096, 64
    w = torch.randn(V, H, generator=torch.Generator().manual_seed(3)) * 0.1
    x = torch.ones(M, H)
    x[1] = -1.0
    w[64:72] = float("-inf")                    # row 1: +inf; the others: a run of -inf logits
    for nan in (False, True):
        if nan:
            w[128:136, 0] = float("nan")        # all eight columns of one thread
        xd, wd = x.to(torch.bfloat16).cuda(), w.to(torch.bfloat16).cuda()
        _, tok, sc, st = K.lm_head_topk(xd, wd, 2, stats=True)
        st = st.cpu()
        if nan:
            assert torch.isnan(st[:, 1]).all(), st
        else:
            lg = (xd.double().cpu()[0] @ wd.double().cpu().t()).float().to(torch.bfloat16).double()
            assert abs(float(st[0, 1]) - float(torch.logsumexp(lg, 0))) < 2e-2, st
