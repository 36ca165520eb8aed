"""The engine's attention kernels (``kernels/attention.py``) against the same
attention in 64 bits, in plain torch on the CPU.

Bound per element: one fp16 rounding of the result (2^-11 of it, or half of
the smallest subnormal), and for the fp32 work before it 2e-5 of the largest
value: a dot product of d terms and a sum over T positions err by a few of
their square roots times 2^-24 (d = 128, T = 2000: about 3e-6), and an error e
of a score moves its probability by e, scores being up to about 20.
"""
import math

import pytest
import torch

from kernels import _native
from kernels.attention import attention_decode, attention_prefill, attention_served

pytestmark = pytest.mark.gpu


def _tables(max_seq, hd, dev):
    inv = 1.0 / (1e6 ** (torch.arange(0, hd, 2, dtype=torch.float32) / hd))
    f = torch.outer(torch.arange(max_seq, dtype=torch.float32), inv)
    f = torch.cat((f, f), -1)
    return f.cos().to(dev), f.sin().to(dev)


def _rope64(t, cos, sin):
    """t [S, heads, hd] in 64 bits; cos, sin [S, hd]."""
    h = t.shape[-1] // 2
    return t * cos.unsqueeze(1) + torch.cat((-t[..., h:], t[..., :h]), -1) * sin.unsqueeze(1)


def _attend64(q, k, v, first):
    """q [S, nh, hd] of positions first .., k and v [kvh, T, hd]: [S, nh * hd]."""
    S, nh, hd = q.shape
    out = torch.empty((S, nh, hd), dtype=torch.float64)
    mask = torch.arange(k.shape[1]).unsqueeze(0) > torch.arange(first, first + S).unsqueeze(1)
    for h in range(nh):
        g = h // (nh // k.shape[0])
        s = (q[:, h] @ k[g].t().contiguous() / math.sqrt(hd)).masked_fill(mask, float("-inf"))
        out[:, h] = torch.softmax(s, -1) @ v[g]
    return out.view(S, nh * hd)


def _close(y, ref, what):
    y = y.double().cpu()
    bound = ref.abs() * 2.0**-11 + 2.0**-25 + 2e-5 * ref.abs().max()
    worst = ((y - ref).abs() / bound).max().item()
    assert torch.isfinite(y).all() and worst <= 1.0, f"{what}: {worst:.2f} of the bound"


@pytest.mark.parametrize("nh,kvh,hd,max_seq,positions", [
    (28, 4, 128, 1152, (0, 1, 15, 16, 63, 64, 65, 1023, 1151)),
    (28, 4, 128, 5000, (127, 128, 4095, 4999)),
    (4, 2, 64, 20000, (383, 384, 511, 512, 19999)),    # ranges of several passes
    (4, 2, 64, 64, (0, 7, 63)),
    (6, 2, 64, 130, (128, 129)),
    (18, 1, 64, 300, (99, 271)),                       # more query heads than one workgroup takes
    (3, 3, 128, 1, (0,)),
    (34, 2, 128, 70, (64, 69)),
])
def test_attention_decode(gpu, nh, kvh, hd, max_seq, positions):
    g = torch.Generator().manual_seed(max_seq)
    cos, sin = _tables(max_seq, hd, gpu)
    k0 = torch.randn((kvh, max_seq, hd), generator=g).half()
    v0 = torch.randn((kvh, max_seq, hd), generator=g).half()
    for pos in positions:
        print(f"attention_decode nh={nh} kvh={kvh} hd={hd} max_seq={max_seq} pos={pos}", flush=True)
        qkv = (torch.randn((1, (nh + 2 * kvh) * hd), generator=g) * 2).half()
        kc, vc = k0.to(gpu), v0.to(gpu)
        kc[:, pos + 1:] = float("nan")                 # rows past the position are never used
        vc[:, pos + 1:] = float("nan")
        keep_k, keep_v = kc.clone(), vc.clone()
        out = attention_decode(qkv.to(gpu), kc, vc, cos, sin, torch.tensor([pos], device=gpu), nh)
        c, s = cos[pos:pos + 1].cpu().double(), sin[pos:pos + 1].cpu().double()
        heads = qkv.double().view(1, nh + 2 * kvh, hd)
        q, knew = _rope64(heads[:, :nh], c, s), _rope64(heads[:, nh:nh + kvh], c, s)
        k, v = k0[:, :pos + 1].double(), v0[:, :pos + 1].double()
        v[:, pos] = heads[0, nh + kvh:]
        _close(kc[:, pos], knew[0], "new key")
        k[:, pos] = kc[:, pos].double().cpu()          # the cache holds fp16 keys
        assert torch.equal(vc[:, pos].cpu(), v[:, pos].half())
        keep_k[:, pos], keep_v[:, pos] = kc[:, pos], vc[:, pos]
        assert torch.equal(kc.view(torch.int16), keep_k.view(torch.int16))
        assert torch.equal(vc.view(torch.int16), keep_v.view(torch.int16))
        _close(out, _attend64(q, k, v, pos), "attention")


@pytest.mark.parametrize("nh,kvh,hd,max_seq,lengths", [
    (28, 4, 128, 1200, (1, 2, 15, 17, 63, 64, 65, 127, 129, 700, 1153)),
    (4, 2, 64, 700, (1, 33, 64, 200, 700)),
    (128, 2, 64, 840, (833,)),                          # 128 queries per workgroup
    (128, 2, 128, 790, (769,)),
    (3, 3, 128, 70, (70,)),
])
def test_attention_prefill(gpu, nh, kvh, hd, max_seq, lengths):
    g = torch.Generator().manual_seed(max_seq + 1)
    cos, sin = _tables(max_seq, hd, gpu)
    for S in lengths:
        print(f"attention_prefill nh={nh} kvh={kvh} hd={hd} max_seq={max_seq} S={S}", flush=True)
        qkv = (torch.randn((S, (nh + 2 * kvh) * hd), generator=g) * 2).half()
        kc = torch.full((kvh, max_seq, hd), float("nan"), dtype=torch.float16, device=gpu)
        vc = kc.clone()
        out = attention_prefill(qkv.to(gpu), kc, vc, cos, sin, nh)
        c, s = cos[:S].cpu().double(), sin[:S].cpu().double()
        heads = qkv.double().view(S, nh + 2 * kvh, hd)
        q, knew = _rope64(heads[:, :nh], c, s), _rope64(heads[:, nh:nh + kvh], c, s)
        _close(kc[:, :S], knew.transpose(0, 1), "keys")
        v = heads[:, nh + kvh:].transpose(0, 1)
        assert torch.equal(vc[:, :S].cpu().double(), v)
        assert kc[:, S:].isnan().all() and vc[:, S:].isnan().all()
        _close(out, _attend64(q, kc[:, :S].double().cpu(), v, 0), "attention")


def test_attention_prefill_and_decode_agree_on_extremes(gpu):
    """Values from 1e-4 to 2, queries of one sign: the split operands keep
    their bits, and a position's attention is the same from both kernels."""
    nh, kvh, hd, S = 8, 2, 128, 190
    cos, sin = _tables(S, hd, gpu)
    g = torch.Generator().manual_seed(5)
    for scale in (1e-4, 1e-2, 1.0, 2.0):
        print(f"attention extremes: scale {scale}", flush=True)
        qkv = (torch.randn((S, (nh + 2 * kvh) * hd), generator=g) * scale).half()
        qkv[:, :nh * hd] += torch.tensor(scale).half()
        kc = torch.zeros((kvh, S, hd), dtype=torch.float16, device=gpu)
        vc = kc.clone()
        out = attention_prefill(qkv.to(gpu), kc, vc, cos, sin, nh)
        c, s = cos.cpu().double(), sin.cpu().double()
        heads = qkv.double().view(S, nh + 2 * kvh, hd)
        ref = _attend64(_rope64(heads[:, :nh], c, s), kc.double().cpu(), heads[:, nh + kvh:].transpose(0, 1), 0)
        _close(out, ref, "prefill")
        one = attention_decode(qkv[-1:].contiguous().to(gpu), kc, vc, cos, sin, torch.tensor([S - 1], device=gpu), nh)
        _close(one, ref[-1:], "decode")


def test_attention_decode_refuses(gpu):
    cos, sin = _tables(8, 64, gpu)
    c = torch.zeros((2, 8, 64), dtype=torch.float16, device=gpu)
    qkv = torch.zeros((1, 8 * 64), dtype=torch.float16, device=gpu)
    pos = torch.zeros(1, dtype=torch.int64, device=gpu)
    attention_decode(qkv, c, c.clone(), cos, sin, pos, 4)
    for bad in (dict(qkv=qkv.float()), dict(qkv=qkv[:, :-64]), dict(pos=pos.int()), dict(cos=cos[:4]),
                dict(k_cache=c.transpose(0, 1)), dict(k_cache=c[:1])):
        args = dict(qkv=qkv, k_cache=c, v_cache=c.clone(), cos=cos, sin=sin, pos=pos) | bad
        with pytest.raises(ValueError):
            attention_decode(num_heads=4, **args)
    with pytest.raises(_native.AwqNativeError):        # head counts that do not divide
        attention_decode(torch.zeros((1, 7 * 64), dtype=torch.float16, device=gpu), c, c.clone(), cos, sin, pos, 3)
    assert attention_served(28, 4, 128, 2048) and not attention_served(4, 2, 32, 64)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("size", [65504.0, 1.0, 2.0**-10])
def test_attention_queries_of_any_size(gpu, hd, size):
    """Queries at fp16's limit, which RoPE takes past it (both halves of a
    rotated pair at 65504, a rotation of 45 degrees: 92636), and small ones
    against keys as much larger.  Scores of about 1 throughout."""
    nh, kvh, S = 4, 2, 70
    cos = torch.full((S, hd), math.sqrt(0.5), device=gpu)
    g = torch.Generator().manual_seed(hd)
    sign = torch.where(torch.rand((S, nh + 2 * kvh, hd // 2), generator=g) < 0.5, -1.0, 1.0)
    qkv = torch.cat((sign, -sign), -1) * size                  # rotated: sqrt(2) size in the lower half
    qkv[:, nh:nh + kvh] = torch.randn((S, kvh, hd), generator=g) / size
    qkv[:, nh + kvh:] = torch.randn((S, kvh, hd), generator=g)
    qkv = qkv.reshape(S, -1).half()
    kc = torch.zeros((kvh, S, hd), dtype=torch.float16, device=gpu)
    vc = kc.clone()
    print(f"attention queries hd={hd} size={size}", flush=True)
    out = attention_prefill(qkv.to(gpu), kc, vc, cos, cos, nh)
    heads, c = qkv.double().view(S, -1, hd), cos.double().cpu()
    ref = _attend64(_rope64(heads[:, :nh], c, c), kc.double().cpu(), heads[:, nh + kvh:].transpose(0, 1), 0)
    _close(out, ref, "prefill")
    one = attention_decode(qkv[-1:].contiguous().to(gpu), kc, vc, cos, cos, torch.tensor([S - 1], device=gpu), nh)
    _close(one, ref[-1:], "decode")


@pytest.mark.parametrize("hd", [64, 128])
def test_attention_scores_of_any_size(gpu, hd):
    """Scores of up to 3e10, as far as fp16 queries and keys go: a difference of
    two is exact to 2^-24 of itself where each is only known to some
    thousands.  The largest wins, whether it comes first or last."""
    nh, kvh, S = 4, 2, 150
    cos = torch.full((S, hd), math.sqrt(0.5), device=gpu)
    g = torch.Generator().manual_seed(hd)
    sign = torch.where(torch.rand((1, 1, hd // 2), generator=g) < 0.5, -1.0, 1.0)
    qkv = torch.empty((S, nh + 2 * kvh, hd))
    qkv[:, :nh] = torch.cat((sign, -sign), -1) * 65504
    rising = torch.arange(1, S + 1) / S
    qkv[:, nh] = torch.cat((sign, -sign), -1)[0] * 46000 * rising.unsqueeze(1)
    qkv[:, nh + 1] = torch.cat((sign, -sign), -1)[0] * 46000 * rising.flip(0).unsqueeze(1)
    qkv[:, nh + kvh:] = torch.randn((S, kvh, hd), generator=g)
    qkv = qkv.reshape(S, -1).half()
    kc = torch.zeros((kvh, S, hd), dtype=torch.float16, device=gpu)
    vc = kc.clone()
    print(f"attention scores hd={hd}", flush=True)
    out = attention_prefill(qkv.to(gpu), kc, vc, cos, cos, nh)
    heads, c = qkv.double().view(S, -1, hd), cos.double().cpu()
    ref = _attend64(_rope64(heads[:, :nh], c, c), kc.double().cpu(), heads[:, nh + kvh:].transpose(0, 1), 0)
    _close(out, ref, "prefill")
    one = attention_decode(qkv[-1:].contiguous().to(gpu), kc, vc, cos, cos, torch.tensor([S - 1], device=gpu), nh)
    _close(one, ref[-1:], "decode")


def test_attention_rounds_as_seldom_as_fp32(gpu):
    """The fp32 work before the output's rounding to fp16 errs no more than
    plain fp32 attention does: as few outputs land on another fp16 value than
    the 64-bit result's.  Flat softmaxes, where the probabilities' own error
    decides, and steep ones, where the scores' does."""
    nh, kvh, hd, S = 28, 4, 128, 100
    cos, sin = _tables(S, hd, gpu)
    c, s = cos.cpu(), sin.cpu()
    g = torch.Generator().manual_seed(1)
    for std in (0.3, 1.0, 2.0):
        other = {"prefill": [0, 0], "decode": [0, 0]}
        for _ in range(2):
            qkv = (torch.randn((S, (nh + 2 * kvh) * hd), generator=g) * std).half()
            kc = torch.zeros((kvh, S, hd), dtype=torch.float16, device=gpu)
            vc = kc.clone()
            out = {"prefill": attention_prefill(qkv.to(gpu), kc, vc, cos, sin, nh)}
            # the same rows one by one: the caches' rows before each are in place
            out["decode"] = torch.cat([attention_decode(qkv[i:i + 1].to(gpu), kc, vc, cos, sin,
                                                        torch.tensor([i], device=gpu), nh) for i in range(S)])
            heads = qkv.view(S, -1, hd)
            exact, plain = (_attend64(_rope64(heads[:, :nh].to(t), c.to(t), s.to(t)), kc.cpu().to(t),
                                      heads[:, nh + kvh:].transpose(0, 1).to(t), 0).half()
                            for t in (torch.float64, torch.float32))
            for name, got in out.items():
                other[name][0] += int((got.cpu() != exact).sum())
                other[name][1] += int((plain != exact).sum())
        print(f"attention rounding std={std}: {other} of {2 * S * nh * hd}", flush=True)
        assert all(a <= b for a, b in other.values())


@pytest.mark.parametrize("max_seq", [70, 5000])      # ranges of one pass and of several
def test_attention_decode_outside_the_cache(gpu, max_seq):
    nh, kvh, hd = 4, 2, 64
    cos, sin = _tables(max_seq, hd, gpu)
    kc = torch.ones((kvh, max_seq, hd), dtype=torch.float16, device=gpu)
    vc = kc.clone()
    qkv = torch.full((1, (nh + 2 * kvh) * hd), 2.0, dtype=torch.float16, device=gpu)
    for pos in (-1, max_seq, 1 << 40):
        print(f"attention_decode max_seq={max_seq} pos={pos}", flush=True)
        assert attention_decode(qkv, kc, vc, cos, sin, torch.tensor([pos], device=gpu), nh).isnan().all()
        assert (kc == 1).all() and (vc == 1).all()
