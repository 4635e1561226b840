"""Several small arrays in one launch, and the torch copy of what that launch does not take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_array_copies():
    from flashgrpo_amd import kernels as K

    g = torch.Generator(device="cuda").manual_seed(1)
    shapes = [(1,), (64, 29), (3, 5), (20000,), (7,)]
    types = [torch.int32, torch.int32, torch.int64, torch.int32, torch.int64]
    make = lambda: [torch.randint(-1000, 1000, s, device="cuda", generator=g).to(t) for s, t in zip(shapes, types)]
    dst = make()
    fill = K.ArrayCopies(dst)
    for _ in range(3):
        src = make()
        fill(src)
        assert all(torch.equal(d, s) for d, s in zip(dst, src))
    # a transposed view, another dtype, a broadcast row, a host tensor: as torch copies them
    src = make()
    odd = [src[0], src[1].t().contiguous().t(), src[2].to(torch.int32), src[3], src[4].cpu()]
    fill(odd)
    assert all(torch.equal(d, s) for d, s in zip(dst, src))
    fill([dst[0], src[1][:1], *src[2:]])
    assert torch.equal(dst[1], src[1][:1].expand(64, 29))
