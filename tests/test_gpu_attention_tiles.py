"""Tree attention at the edges of its row tiles and key ranges, against float64."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _want(q, k, v, seq, see):
    """float64 attention; see [N, N] or per row [B, N, N]: the new keys a new token attends."""
    B, N, Hq, d = q.shape
    Hkv, cap = k.shape[1], k.shape[2]
    out = torch.zeros(B, N, Hq, d, dtype=torch.float64, device=q.device)
    for b in range(B):
        L = int(seq[b])
        S = min(L + N, cap)  # slots past the capacity hold nothing
        s = see if see.dim() == 2 else see[b]
        allow = torch.cat([torch.ones(N, L, dtype=torch.bool, device=q.device), s], 1)[:, :S]
        for h in range(Hq):
            kk, vv = k[b, h * Hkv // Hq, :S].double(), v[b, h * Hkv // Hq, :S].double()
            sc = (q[b, :, h].double() @ kk.t().contiguous() / math.sqrt(d)).masked_fill(~allow, float("-inf"))
            out[b, :, h] = torch.softmax(sc, -1) @ vv
    return out


def _close(got, want):
    # bf16 probabilities and output: 2^-8 each, relative to the largest value of a row
    err = (got.double() - want).abs().amax(-1) / want.abs().amax(-1).clamp_min(1e-3)
    assert float(err.max()) < 2e-2, float(err.max())


@pytest.mark.parametrize("B,Hq,Hkv,N", [(2, 8, 2, 65), (3, 4, 4, 257), (1, 28, 4, 200), (40, 16, 8, 129), (2, 8, 8, 1)])
def test_chain_rows_stop_at_their_own_key(B, Hq, Hkv, N):
    """A causal chunk after ragged prefixes: every row tile ends at its last row's key, whatever
    lies in the slots behind it."""
    from flashgrpo_amd import kernels as K

    g = torch.Generator(device=DEV).manual_seed(N + B)
    cap, d = 700, 128
    seq = torch.tensor([(37 * b) % 400 for b in range(B)], dtype=torch.int32, device=DEV)
    q = torch.randn(B, N, Hq, d, device=DEV, generator=g).bfloat16()
    k = torch.randn(B, Hkv, cap, d, device=DEV, generator=g).bfloat16()
    v = torch.randn(B, Hkv, cap, d, device=DEV, generator=g).bfloat16()
    for b in range(B):
        k[b, :, int(seq[b]) + N:] = 40.0  # never attended
        v[b, :, int(seq[b]) + N:] = 1e4
    got = K.tree_attention(q, k, v, seq_len=seq, anc=None, num_nodes=N, q_heads=Hq, kv_heads=Hkv, head_dim=d)
    _close(got, _want(q, k, v, seq, torch.tril(torch.ones(N, N, dtype=torch.bool, device=DEV))))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("prefix", [0, 1, 30, 63, 127, 260])
@pytest.mark.parametrize("chain", [True, False])
def test_fp32_key_groups(d, prefix, chain):
    """Key counts around the steps of the four waves, from one key to several rounds; q and V only
    dword-aligned; slots behind a row's keys hold what no sum survives."""
    from flashgrpo_amd import kernels as K

    g = torch.Generator(device=DEV).manual_seed(prefix + d)
    B, N, Hq, Hkv, cap = 2, 5, 4, 2, 300
    seq = torch.tensor([prefix, prefix // 2], dtype=torch.int32, device=DEV)
    n = lambda *s: torch.randn(math.prod(s) + 1, device=DEV, generator=g)[1:].view(*s)
    q, k, v = n(B, N, Hq, d), n(B, Hkv, cap, d).clone(), n(B, Hkv, cap, d)
    for b in range(B):
        k[b, :, int(seq[b]) + N:], v[b, :, int(seq[b]) + N:] = 3e38, float("nan")
    see = torch.tril(torch.ones(N, N, dtype=torch.bool, device=DEV))
    anc = None
    if not chain:  # two branches below node 0
        see[2, 1] = see[4, 3] = False
        anc = (see.long() << torch.arange(N, device=DEV)).sum(1).expand(B, N).contiguous()
    got = K.tree_attention(q, k, v, seq_len=seq, anc=anc, num_nodes=N, q_heads=Hq, kv_heads=Hkv, head_dim=d)
    want = _want(q, k, v, seq, see)
    # fp32 scores of d terms and sums of at most 265 keys, each rounded to 2^-24
    err = (got.double() - want).abs().amax(-1) / want.abs().amax(-1)
    assert float(err.max()) < (d + 265) * 2.0 ** -24, float(err.max())


@pytest.mark.parametrize("B,Hq,Hkv,N,cap", [(9, 16, 8, 129, 700),      # 72 units: groups of 32, 32 and 8
                                            (9, 16, 8, 129, 2400),     # groups of 24
                                            (9, 8, 8, 300, 9000),      # groups of 8
                                            (63, 2, 1, 200, 500),      # 63 units: one group
                                            (65, 2, 1, 200, 500)])     # 65 units padded to 72
def test_chain_tile_orders(B, Hq, Hkv, N, cap):
    """Every row tile of every (sequence, kv head) is computed once, however they are grouped."""
    from flashgrpo_amd import kernels as K

    g = torch.Generator(device=DEV).manual_seed(cap)
    d = 128
    seq = torch.tensor([(41 * b) % 190 for b in range(B)], dtype=torch.int32, device=DEV)
    q = torch.randn(B, N, Hq, d, device=DEV, generator=g).bfloat16()
    k = torch.randn(B, Hkv, cap, d, device=DEV, generator=g, dtype=torch.bfloat16)
    v = torch.randn(B, Hkv, cap, d, device=DEV, generator=g, dtype=torch.bfloat16)
    got = K.tree_attention(q, k, v, seq_len=seq, anc=None, num_nodes=N, q_heads=Hq, kv_heads=Hkv, head_dim=d,
                           out=torch.full_like(q, float("nan")))
    _close(got, _want(q, k, v, seq, torch.tril(torch.ones(N, N, dtype=torch.bool, device=DEV))))
