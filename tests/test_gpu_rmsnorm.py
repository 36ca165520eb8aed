"""RMSNorm kernel (``kernels/rmsnorm.py``) against the same in 64 bits.

Bound per element: one fp16 rounding (2^-11, or half of the smallest
subnormal) and 1e-6 of the value for the fp32 sum of at most 16384 squares.
"""
import math

import pytest
import torch

from kernels.rmsnorm import MAX_H, rmsnorm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [0, 1, 3, 700])
@pytest.mark.parametrize("h", [8, 256, 3584, 4088, 4096, 4104, 8192, MAX_H])
def test_rmsnorm(gpu, m, h):
    print(f"rmsnorm m={m} h={h}", flush=True)
    g = torch.Generator().manual_seed(m + h)
    x = (torch.randn((m, h), generator=g) * 10.0 ** torch.randint(-3, 4, (m, 1), generator=g)).half()
    w = (1 + 0.1 * torch.randn(h, generator=g)).half()
    y = rmsnorm(x.to(gpu), w.to(gpu), 1e-6).double().cpu()
    x64 = x.double()
    ref = x64 * torch.rsqrt(x64.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
    assert y.shape == ref.shape and ((y - ref).abs() <= ref.abs() * (2.0**-11 + 1e-6) + 2.0**-25).all()


def test_rmsnorm_views_and_refusals(gpu):
    x = torch.randn((4, 528), device=gpu).half()
    w = torch.randn(513, device=gpu).half()
    want = rmsnorm(x[:, 1:513].clone(), w[1:].clone(), 1e-5)
    assert torch.equal(rmsnorm(x[:, 1:513], w[1:], 1e-5), want)       # strided rows, odd offsets
    assert torch.equal(rmsnorm(x[:, 1:513].unsqueeze(0), w[1:], 1e-5)[0], want)
    for a, b in ((x.float(), w[:528]), (x, w[:8]), (x[:, :12], w[:12]), (x.cpu(), w[:512].cpu())):
        with pytest.raises(ValueError):
            rmsnorm(a, b, 1e-5)


@pytest.mark.parametrize("h", [256, 3584, 8192])
def test_rmsnorm_rounds_as_seldom_as_fp32(gpu, h):
    """The fp32 work errs no more than the same formula in plain torch fp32:
    as few outputs land on another fp16 value than the 64-bit result's.  (Two
    counts of about b differ by 2 sqrt(2 b) by chance: two standard deviations.)"""
    other = [0, 0]
    for seed in range(4):
        g = torch.Generator(device=gpu).manual_seed(seed)
        x = (torch.randn((4096, h), generator=g, device=gpu) * 3).half()
        w = (1 + 0.1 * torch.randn(h, generator=g, device=gpu)).half()
        exact, plain = ((v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-6) * w.to(v.dtype)).half()
                        for v in (x.double(), x.float()))
        other[0] += int((rmsnorm(x, w, 1e-6) != exact).sum())
        other[1] += int((plain != exact).sum())
    print(f"rmsnorm rounding h={h}: {other}", flush=True)
    assert other[0] <= other[1] + 2 * math.sqrt(2 * other[1])
