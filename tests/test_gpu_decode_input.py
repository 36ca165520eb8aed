"""The decode GEMVs that make their row of x in the prologue
(``awq_gemm_decode``).  SiLU * up: the row is rounded to fp16 by the same
formula as in the kernel of its own, so the results agree bit for bit.
RMSNorm (another order of the fp32 sum) against 64 bits: 2^-11 of sum |x w|
for the row's rounding to fp16 (a bound that holds if every rounding adds up),
and 2^-11 of the value at each rounding of the result.
"""
import numpy as np
import pytest
import torch

from kernels import _native
from kernels.awq_gemm import awq_gemm_decode, awq_gemm_forward_ex, decode_linear_served
from kernels.rmsnorm import rmsnorm
from kernels.silu_mul import silu_mul_gate_up
from oracle import awq_oracle as O

pytestmark = pytest.mark.gpu

# quads, pairs and singles; one group; ragged strips; many splits
SHAPES = [(3584, 4608), (3584, 3584), (3584, 37888), (18944, 3584), (3584, 18944), (3584, 512), (128, 32), (256, 512),
          (512, 1024), (512, 96), (1152, 4640), (3968, 9504)]


def _operands(k, n, gpu):
    _, qw, qz, s = O.make_inputs(1, k, n, seed=k + n)
    g = torch.Generator().manual_seed(n)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    return (t(qw), t(qz), t(s)), O.dequant_awq(qw, qz, s).astype(np.float64), g


@pytest.mark.parametrize("k,n", SHAPES)
def test_decode_rmsnorm(gpu, k, n):
    if not decode_linear_served(n, k, _native.INPUT_RMSNORM):
        assert k > 4096       # longer than the threads hold
        return
    print(f"decode rmsnorm K={k} N={n}", flush=True)
    op, w64, g = _operands(k, n, gpu)
    x = (torch.randn((1, k), generator=g) * 3).half().to(gpu)
    nw = (1 + 0.1 * torch.randn(k, generator=g)).half().to(gpu)
    bias, res = torch.randn(n, generator=g).half().to(gpu), torch.randn((1, n), generator=g).half().to(gpu)
    x64 = x.double().cpu().numpy()
    row64 = x64 / np.sqrt((x64**2).mean() + 1e-6) * nw.double().cpu().numpy()
    y64, scale = row64 @ w64, np.abs(row64) @ np.abs(w64)
    for kw in ({}, {"bias": bias}, {"residual": res}, {"bias": bias, "residual": res}):
        got = awq_gemm_decode(_native.INPUT_RMSNORM, x, *op, norm_w=nw, eps=1e-6, **kw).double().cpu().numpy()
        want, rounded = y64, np.abs(y64)               # each add rounds once more
        for t in kw.values():
            want = want + t.double().cpu().numpy()
            rounded = rounded + np.abs(want)
        assert (np.abs(got - want) <= 2.0**-11 * (1.01 * scale + rounded) + 2.0**-24).all()


@pytest.mark.parametrize("k,n", [(3584, 4608), (3584, 37888), (128, 32), (1152, 4640)])
def test_decode_rmsnorm_eps(gpu, k, n):
    """eps as large as the row's mean square (the factor is off by 1.4 without
    it), against 64 bits and against the norm's own kernel.  The two factors
    differ by the order of the fp32 sum, so that about one in a thousand of the
    row's values rounds to another fp16 value: 2^-10 of it, and all that do
    together are less than a 32nd of sum |x w|."""
    print(f"decode rmsnorm eps K={k} N={n}", flush=True)
    op, w64, g = _operands(k, n, gpu)
    x = (torch.randn((1, k), generator=g) * 1e-3).half().to(gpu)
    nw = (1 + 0.1 * torch.randn(k, generator=g)).half().to(gpu)
    x64 = x.double().cpu().numpy()
    row64 = x64 / np.sqrt((x64**2).mean() + 1e-6) * nw.double().cpu().numpy()
    y64, scale = row64 @ w64, np.abs(row64) @ np.abs(w64)
    got = awq_gemm_decode(_native.INPUT_RMSNORM, x, *op, norm_w=nw, eps=1e-6)
    two = awq_gemm_forward_ex(rmsnorm(x, nw, 1e-6), *op).double().cpu().numpy()
    got = got.double().cpu().numpy()
    assert (np.abs(got - y64) <= 2.0**-11 * (1.01 * scale + np.abs(y64)) + 2.0**-24).all()
    assert (np.abs(got - two) <= (2.0**-10 * (scale / 32 + np.abs(y64)) + 2.0**-24)).all()


@pytest.mark.parametrize("k,n", SHAPES)
def test_decode_silu_mul(gpu, k, n):
    assert decode_linear_served(n, k, _native.INPUT_SILU_MUL)
    print(f"decode silu_mul K={k} N={n}", flush=True)
    op, _, g = _operands(k, n, gpu)
    gu = (torch.randn((1, 2 * k), generator=g) * 4).half().to(gpu)
    res = torch.randn((1, n), generator=g).half().to(gpu)
    row = silu_mul_gate_up(gu)
    for kw in ({}, {"residual": res}):
        got = awq_gemm_decode(_native.INPUT_SILU_MUL, gu, *op, **kw)
        assert torch.equal(got, awq_gemm_forward_ex(row, *op, **kw))


def test_decode_input_refuses(gpu):
    op, _, _ = _operands(256, 512, gpu)
    x, w = torch.zeros((1, 256), dtype=torch.float16, device=gpu), torch.ones(256, dtype=torch.float16, device=gpu)
    for args in ((_native.INPUT_RMSNORM, x, *op), (_native.INPUT_RMSNORM, x, *op, w[:8]),
                 (_native.INPUT_RMSNORM, x.float(), *op, w), (_native.INPUT_RMSNORM, x.expand(2, 256), *op, w),
                 (_native.INPUT_SILU_MUL, x, *op), (3, x, *op)):
        with pytest.raises(ValueError):
            awq_gemm_decode(*args)
    assert not decode_linear_served(24, 256, _native.INPUT_RMSNORM)        # N % 32 != 0: another kernel
