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


def _oracle(xs, noise, kw):
    return OS.sample_rows(xs, noise, do_sample=not kw.get("greedy", False), temperature=kw.get("temperature", 1.0),
                          top_p=kw.get("top_p", 1.0), top_k=kw.get("top_k"))


def _flat_rows(V, seed):
    """Rows whose logits crowd a few bins of the exponent, or one."""
    g = np.random.default_rng(seed)
    z = g.standard_normal((10, V)).astype(np.float32)
    x = z * np.float32(0.3)
    x[1] = z[1] * 0.05
    x[2] = z[2] * 1e-3
    x[3] = z[3] * 1e-6
    x[4] = 7.25                                                            # one value
    x[5] = np.where(g.random(V) < 0.7, 1.0, 1.5)                           # two
    x[6] = torch.from_numpy(z[6] * 0.3 + 20).to(torch.bfloat16).float().numpy()  # a few values far from zero
    x[7] = z[7] * 0.01
    x[7, V // 5: V // 4] = -np.inf
    x[8] = 0.5
    x[8, :3] = np.nan
    x[8, 5] = 9.0                                                          # one logit above long ties
    x[9] = z[9] * 0.02
    x[9, ::7] = -30.0                                                      # a crowd far below another
    return torch.from_numpy(x)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [8200, 9000, 16384, 20003, 32768, 50304, 152064, 163848])
def test_flat_rows_match_oracle(dtype, V):
    """Cuts in bins with more logits than a list: sampled, and as walk steps that form the row maxima,
    are given them, or have one workgroup per row."""
    from flashgrpo_amd import kernels as K

    x = _flat_rows(V, V).to(dtype)
    R = x.shape[0]
    xd, xs = x.to(DEV), x.float().numpy()
    noise = np.random.default_rng(2).integers(0, 2 ** 32, (R, 1), dtype=np.uint32)
    nd = torch.from_numpy(noise.view(np.int32)).to(DEV)
    big = torch.nan_to_num(x.float(), nan=float("-inf"), neginf=float("-inf")).amax(1, keepdim=True).to(DEV)
    parts = (big.contiguous(), torch.zeros(R, 1, dtype=torch.int64, device=DEV))  # a cut needs the maxima alone
    tt = torch.full((R, 2), -5, dtype=torch.int32, device=DEV)
    par = torch.tensor([[-1, 0]] * R, dtype=torch.int32, device=DEV)
    nn = torch.full((R,), 2, dtype=torch.int32, device=DEV)
    for kw in (dict(top_p=0.9), dict(top_p=0.4, temperature=0.8), dict(top_k=50), dict(top_k=1000, top_p=0.7),
               dict(top_k=4096)):
        want = _oracle(xs, noise, kw)
        assert np.array_equal(K.sample_tokens(xd, noise=nd, **kw).cpu().numpy(), want), (V, dtype, kw)
        for split, pt in ((True, None), (True, parts), (False, None)):
            wk = K.walk_begin(tt, par, nn, acc_stride=2)
            K.walk_rows(wk, 2)
            K.walk_step(wk, xd, tt, par, nn, walk_step=0, noise=nd, split=split, parts=pt, **kw)
            assert np.array_equal(wk["correction"].cpu().numpy(), want), (V, dtype, kw, split, pt is not None)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [163848, 200008])
def test_chunks_of_two_passes_match_oracle(dtype, V):
    """Rows whose 16 chunks are longer than a workgroup's pass (10,240 logits), with cuts and ties in the
    second pass."""
    from flashgrpo_amd import kernels as K

    x = _rows(V, V)
    chunk = (-(-V // 16) + 7) // 8 * 8
    x[0, 10_240: chunk] += 8.0                      # the mass in the first chunk's second pass
    x[1, 2 * chunk + 10_240: 3 * chunk] = 12.0      # a tie there
    x[3, 5 * chunk + 10_000: 5 * chunk + 10_250] = 9.0   # a tie across the two passes
    x = x.to(dtype)
    noise = np.random.default_rng(3).integers(0, 2 ** 32, (12, 1), dtype=np.uint32)
    nd = torch.from_numpy(noise.view(np.int32)).to(DEV)
    for kw in (dict(top_p=0.95), dict(top_p=0.3), dict(top_k=5), dict(top_k=50, top_p=0.9), dict(top_k=256),
               dict(top_k=1500)):
        got = K.sample_tokens(x.to(DEV), noise=nd, **kw).cpu().numpy()
        assert np.array_equal(got, _oracle(x.float().numpy(), noise, kw)), (V, dtype, kw)


@pytest.mark.parametrize("rows", [3, 15, 16, 130])
@pytest.mark.parametrize("V", [8192, 8200, 16384, 16392, 32768, 32776, 65536, 65544])
def test_draws_at_the_path_lines(V, rows):
    """Every kind of draw on both sides of the sizes and row counts at which its path changes."""
    from flashgrpo_amd import kernels as K

    base = _rows(V, V)[[0, 1, 3, 6, 9]]
    x = base[torch.arange(rows) % 5].to(torch.bfloat16)
    n5 = np.random.default_rng(4).integers(0, 2 ** 32, (5, 1), dtype=np.uint32)
    noise = n5[np.arange(rows) % 5]
    nd = torch.from_numpy(noise.view(np.int32)).to(DEV)
    xd, xs = x.to(DEV), base.to(torch.bfloat16).float().numpy()
    for kw in (dict(), dict(temperature=0.6), dict(greedy=True), dict(top_p=0.9), dict(top_k=20)):
        want = _oracle(xs, n5, kw)[np.arange(rows) % 5]
        for split in (True, False):
            got = K.sample_tokens(xd, noise=nd, split=split, **kw).cpu().numpy()
            assert np.array_equal(got, want), (V, rows, kw, split)


@pytest.mark.parametrize("V", [64, 8192, 32000, 65536, 70000])
def test_greedy_walk_step_with_given_maxima_reads_no_logits(V):
    """The first maxima that come with the logits are the greedy draw: the logits are not read again."""
    from flashgrpo_amd import kernels as K

    B = 6
    tt = torch.full((B, 2), -5, dtype=torch.int32, device=DEV)
    par = torch.tensor([[-1, 0]] * B, dtype=torch.int32, device=DEV)
    nn = torch.full((B,), 2, dtype=torch.int32, device=DEV)
    first = torch.arange(B, device=DEV) * 9 + 1
    key = (torch.full((B,), 0xC0000000, dtype=torch.int64, device=DEV) << 32) | (0xffffffff - first)  # the value 2.0
    parts = (torch.full((B, 1), 2.0, device=DEV), key[:, None].contiguous())
    wk = K.walk_begin(tt, par, nn, acc_stride=2)
    K.walk_rows(wk, 2)
    K.walk_step(wk, torch.zeros(B, V, device=DEV), tt, par, nn, walk_step=0, greedy=True, parts=parts)
    assert torch.equal(wk["correction"].long(), first)


@pytest.mark.parametrize("kw", [dict(top_p=0.9), dict(top_k=1000)])
def test_flat_rows_take_no_more_than_others(kw):
    """A flat row costs about what any other does: it once went to a draw of many passes by one
    workgroup (top-p 5.8 times as long, top-k 1,000 4.9)."""
    from flashgrpo_amd import kernels as K

    g = torch.Generator(device=DEV).manual_seed(1)
    z = torch.randn(64, 152064, device=DEV, generator=g)

    def best_us(x):
        t = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                K.sample_tokens(x, seed=1, **kw)
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b) * 50)
        return min(t)

    broad = best_us((z * 2).to(torch.bfloat16))
    for spread in (0.3, 0.05):
        flat = best_us((z * spread).to(torch.bfloat16))
        assert flat < 2.5 * broad, (spread, flat, broad)
