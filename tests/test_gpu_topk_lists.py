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


def _check(x, rows, kmax, sanitize):
    """Candidates and statistics of the given rows of x (on the device) against the oracle."""
    from flashgrpo_amd import kernels as K

    tok, sc, st = (t.cpu() for t in K.medusa_topk(x, kmax, stats=True, sanitize=sanitize))
    for r in rows:
        xs = x[r].float().cpu().numpy()
        xs = OT.nan_to_num_logits(xs) if sanitize else xs
        ids, vals = OT.topk_canonical(xs, kmax)
        assert tok[r].tolist() == ids.tolist(), (r, sanitize)
        assert np.array_equal(sc[r].numpy(), vals.astype(np.float32) + 0.0), (r, sanitize)
        m = float(xs.max())
        lse = np.log(np.sum(np.exp(xs.astype(np.float64) - m))) + m
        assert float(st[r, 0]) == m and abs(float(st[r, 1]) - lse) < 1e-4 * max(1.0, abs(lse)), (r, sanitize)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
# 2,048 rows leave one chunk a row up to 10,240 logits: the ends of what keeps sorted lists for the
# different kmax, and chunks of one to five load groups with their remainders
@pytest.mark.parametrize("V", [1536, 1537, 1793, 1920, 1921, 2048, 2049, 4104, 6145, 8200, 10239, 10240, 10241])
@pytest.mark.parametrize("kmax", [1, 2, 4, 8, 16])
def test_chunks_of_every_length_match_oracle(dtype, V, kmax):
    g = torch.Generator(device="cuda").manual_seed(V + kmax)
    x = torch.randn(2048, V, device="cuda", generator=g)
    x[1] = torch.round(x[1])                               # long ties
    x[2, V // 2:] = x[2].max() + 1                         # half the row shares the maximum
    x[3] = torch.arange(V, device="cuda").float() / 7      # the last elements win
    x[4] = -x[3]
    x[5, -min(V, 9):] = 9.0                                # the winners in the last, padded group
    x[6, ::8] += 3                                         # spread over all groups
    x[2047, V // 3:] = float("-inf")
    x = x.to(dtype)
    for sanitize in (False, True):
        _check(x, [0, 1, 2, 3, 4, 5, 6, 1000, 2047], kmax, sanitize)


@pytest.mark.parametrize("kmax", [1, 2, 5, 16])
def test_chunks_of_two_passes_match_oracle(kmax):
    """Vocabularies whose 64 chunks are longer than a pass: the list carries over."""
    V = 700_001                                            # chunks of 10,944
    g = torch.Generator(device="cuda").manual_seed(kmax)
    x = torch.randn(4, V, device="cuda", generator=g)
    x[0, 10_944 * 3 + 10_240: 10_944 * 4] += 5             # winners in a second pass
    x[1, 10_944 * 2 + 10_230: 10_944 * 2 + 10_250] = 8.0   # a tie across the two passes
    x[2] = torch.round(x[2] * 2)
    x[3, V - 3:] = 7.0                                     # the short last chunk
    for dtype in (torch.float32, torch.bfloat16):
        for sanitize in (False, True):
            _check(x.to(dtype), range(4), kmax, sanitize)
