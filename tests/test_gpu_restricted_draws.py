"""Top-k and top-p draws against the CPU oracle, at the edges of the launch paths: one
workgroup's row, lists that overflow, cuts inside long ties, NaN and infinite logits."""
import numpy as np
import pytest
import torch

from oracle import sampling as OS

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(V, seed):
    """Rows whose cuts fall in different places."""
    g = np.random.default_rng(seed)
    x = g.standard_normal((12, V)).astype(np.float32) * 2
    x[1] += (g.random(V) < 0.002) * 10.0            # a few tokens hold the mass
    x[2] = 0.25                                     # one tie over the whole row
    x[3] = np.round(x[3] * 4) / 4                   # long ties
    x[4] = x[4] * 0.05                              # nearly flat: the list overflows on long rows
    x[5, ::3] = -np.inf
    x[6, : min(V, 7)] = np.nan                      # NaN takes the first top-k slots
    x[7] = -60.0
    x[7, V // 2] = 3.0                              # one element of weight, the rest 40 octaves down
    x[7, V - 1] = 2.5
    x[8] = -np.inf
    x[8, V - 1] = 1.0
    x[9, V // 3] = np.inf                           # total weight 0: the first maximum
    x[10] = np.nan
    x[11] = np.where(g.random(V) < 0.5, 0.0, -0.0)  # -0 ranks as +0
    return torch.from_numpy(x)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [64, 1000, 2055, 32000, 32768, 32776, 65536, 65545, 152064])
def test_restricted_draws_match_oracle(dtype, V):
    from flashgrpo_amd import kernels as K

    x = _rows(V, V).to(dtype)
    xd = x.to(DEV)
    xs = x.float().numpy()
    noise = np.random.default_rng(1).integers(0, 2 ** 32, (12, 1), dtype=np.uint32)
    nd = torch.from_numpy(noise.view(np.int32)).to(DEV)
    for kw in (dict(top_p=0.95), dict(top_p=0.3, temperature=0.7), dict(top_k=1), dict(top_k=5),
               dict(top_k=50, temperature=0.6), dict(top_k=50, top_p=0.9), dict(top_k=4096, top_p=0.5),
               dict(top_k=4097), dict(top_p=1e-9)):
        got = K.sample_tokens(xd, noise=nd, **kw).cpu().numpy()
        want = OS.sample_rows(xs, noise, do_sample=True, temperature=kw.get("temperature", 1.0),
                              top_p=kw.get("top_p", 1.0), top_k=kw.get("top_k"))
        assert np.array_equal(got, want), (V, dtype, kw, got, want)


@pytest.mark.parametrize("kw", [dict(top_p=0.9), dict(top_k=9), dict(top_k=9, top_p=0.6)])
def test_restricted_walk_step_with_given_maxima(kw):
    """A walk step whose row maxima come with the logits equals one that forms them, and the
    single-workgroup draw, on active and inactive rows."""
    from flashgrpo_amd import kernels as K

    B, N, V, H = 9, 5, 40000, 64
    g = torch.Generator(device="cpu").manual_seed(7)
    w = (torch.randn(V, H, generator=g) * 0.3).to(torch.bfloat16).to(DEV)
    h = torch.randn(B, H, generator=g).to(torch.bfloat16).to(DEV)
    P = K.lm_head_parts(V)
    parts = (torch.empty(B, P, dtype=torch.float32, device=DEV), torch.empty(B, P, dtype=torch.int64, device=DEV))
    lg = K.lm_head_topk(h, w, 0, parts=parts)[0]
    toks = torch.randint(0, V, (B, N), generator=g, dtype=torch.int32)
    toks[:, 1] = lg.float().argmax(-1).cpu().to(torch.int32)
    par = torch.tensor([[-1, 0, 0, 1, 1]] * B, dtype=torch.int32)
    nn = torch.full((B,), N, dtype=torch.int32)
    nn[::4] = 1                                     # a root alone: nothing to walk
    toks, par, nn = toks.to(DEV), par.to(DEV), nn.to(DEV)
    res = []
    for split, pt in ((True, parts), (True, None), (False, None)):
        wk = K.walk_begin(toks, par, nn, acc_stride=3)
        K.walk_rows(wk, N)
        K.walk_step(wk, lg, toks, par, nn, walk_step=0, seed=5, split=split, parts=pt, next_rows=True, **kw)
        res.append([wk[k].cpu().numpy() for k in ("acc_tokens", "acc_nodes", "acc_len", "correction", "state",
                                                  "row_active")])
    for other in res[1:]:
        for a, b in zip(res[0], other):
            assert np.array_equal(a, b)
