"""The fp32 chain cell in one call and the fp32 Medusa block, at the remainders of their 64 x 64
tiles and 32-wide K steps, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows", [1, 63, 65, 300])
@pytest.mark.parametrize("H,bott", [(8, 4), (40, 64), (512, 64), (1536, 192), (1000, 68)])
def test_chain_cell_step_matches_float64(rows, H, bott):
    from flashgrpo_amd import kernels as K

    g = torch.Generator(device=DEV).manual_seed(rows + H)
    n = lambda *s: torch.randn(*s, device=DEV, generator=g)
    st, tk = n(rows, H) * 2 + 1, n(rows, H)
    sw, sb, tw, tb = 1 + 0.1 * n(H), 0.1 * n(H), 1 + 0.1 * n(H), 0.1 * n(H)
    pw, ow, ob, gate = n(bott, 2 * H) * 0.05, n(H, bott) * 0.1, n(H) * 0.1, torch.tensor(0.4, device=DEV)
    args = (st, tk, sw, sb, tw, tb, pw[:, :H].contiguous(), pw[:, H:].contiguous(), ow, ob, gate, 1e-5)
    got = K.chain_cell_step(*args)
    ln = lambda x, w, b: torch.nn.functional.layer_norm(x.double(), (H,), w.double(), b.double(), 1e-5)
    x = torch.cat([ln(st, sw, sb), ln(tk, tw, tb)], 1)
    mix = x @ pw.double().t().contiguous()
    mid = torch.nn.functional.silu(mix)
    want = st.double() + gate.double() * (mid @ ow.double().t().contiguous() + ob.double())
    # fp32 products of 2H and bott terms (2^-24 a term, as a sum of magnitudes), SiLU' <= 1.1, the norms'
    # relative 2^-18 as test_gpu_chain_cell takes it, and the last roundings
    e_mix = 2.0 ** -17 * (x.abs() @ pw.double().abs().t().contiguous()) + 2 * H * 2.0 ** -24 * (x.abs() @ pw.double().abs().t().contiguous())
    e_out = (1.1 * e_mix + bott * 2.0 ** -24 * mid.abs() + 2.0 ** -22 * mid.abs()) @ ow.double().abs().t().contiguous()
    bound = gate.double() * e_out + 2.0 ** -22 * (want.abs() + st.double().abs()) + 1e-6
    assert bool(((got.double() - want).abs() <= bound).all())
    assert torch.equal(got, K.chain_cell_step(*args))
    # bf16 token rows (embeddings): the same as their widened copy
    assert torch.equal(K.chain_cell_step(st, tk.bfloat16(), *args[2:]),
                       K.chain_cell_step(st, tk.bfloat16().float(), *args[2:]))


@pytest.mark.parametrize("B,H,heads", [(1, 64, 1), (65, 132, 2), (96, 1000, 3), (7, 4096, 1)])
def test_f32_medusa_block_matches_float64(B, H, heads):
    from flashgrpo_amd import kernels as K

    g = torch.Generator(device=DEV).manual_seed(B + H)
    n = lambda *s: torch.randn(*s, device=DEV, generator=g)
    h, lw, lb = n(B, H), 1 + 0.1 * n(heads, H), 0.1 * n(heads, H)
    fw, fb = n(heads, H, H) * 0.02, n(heads, H) * 0.1
    got = K.medusa_heads(h, lw, lb, fw, fb).view(heads, B, H)
    for i in range(heads):
        x = torch.nn.functional.layer_norm(h.double(), (H,), lw[i].double(), lb[i].double(), 1e-5)
        fc = x @ fw[i].double().t().contiguous()
        want = h.double() + torch.nn.functional.silu(fc + fb[i].double())
        bound = 1.1 * (H * 2.0 ** -24 + 2.0 ** -17) * (x.abs() @ fw[i].double().abs().t().contiguous()) + 2.0 ** -21 * (
            want.abs() + h.double().abs()) + 1e-6
        assert bool(((got[i].double() - want).abs() <= bound).all())
