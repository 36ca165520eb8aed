"""A decoder layer in one native call (``qwen2_layer``) against the engine's own
sequence of calls, which models the kernels do not serve take: other head
sizes, fp32 norm weights, a subclass with its own projections.

Both round the same values to fp16 and differ by the order of fp32 sums, so a
few fp16 roundings (2^-11 each) over two layers: 4e-3 of the largest value,
for the logits and for each layer's caches on its own.
"""
import pytest
import torch

from engine.qwen2_decode import Qwen2AwqDecoder, Qwen2Shape

pytestmark = pytest.mark.gpu

TINY = dict(vocab_size=512, hidden_size=256, intermediate_size=512, num_layers=2)


def _run(m, prompt, forced):
    m.k_cache.zero_()
    m.v_cache.zero_()
    outs = [m.prefill(prompt)]
    outs += [m.decode_logits(t, len(prompt) + i) for i, t in enumerate(forced)]
    return [torch.stack(outs), *m.k_cache.clone(), *m.v_cache.clone()]


def _close(got, want):
    return all((a.float() - b.float()).abs().max() <= 4e-3 * b.float().abs().max() for a, b in zip(got, want, strict=True))


@pytest.mark.parametrize("heads,kv_heads", [(4, 2), (2, 1), (4, 4)])     # head sizes 64, 128, 64
def test_native_layer_matches_calls(gpu, heads, kv_heads):
    m = Qwen2AwqDecoder(Qwen2Shape(num_heads=heads, num_kv_heads=kv_heads, **TINY), max_seq_len=80, seed=heads,
                        device=gpu)
    assert m._native_layers
    g = torch.Generator().manual_seed(3)
    for length in (1, 2, 65):
        prompt, forced = torch.randint(0, 512, (length,), generator=g), torch.randint(0, 512, (4,), generator=g)
        print(f"native layer heads={heads} prompt={length}", flush=True)
        native = _run(m, prompt, forced)
        m._native_layers = False
        calls = _run(m, prompt, forced)
        m._native_layers = True
        assert _close(native, calls)


def test_other_models_take_the_calls(gpu):
    class Own(Qwen2AwqDecoder):
        calls = 0

        def linear(self, *a, **kw):
            self.calls += 1
            return super().linear(*a, **kw)

    shape = Qwen2Shape(num_heads=4, num_kv_heads=2, **TINY)
    ref = Qwen2AwqDecoder(shape, max_seq_len=40, seed=1, device=gpu)
    prompt, forced = torch.arange(20), torch.arange(3)
    want = _run(ref, prompt, forced)
    own = Own(shape, max_seq_len=40, seed=1, device=gpu)
    assert _close(_run(own, prompt, forced), want) and own.calls == 4 * 2 * 4
    wide = Qwen2AwqDecoder(shape, max_seq_len=40, seed=1, device=gpu)
    for p in wide.layers:
        p["ln1"], p["ln2"] = p["ln1"].float(), p["ln2"].float()
    assert _close(_run(wide, prompt, forced), want)
    small = Qwen2AwqDecoder(Qwen2Shape(num_heads=8, num_kv_heads=2, **TINY), max_seq_len=40, seed=1, device=gpu)
    assert not small._native_layers and all(t.isfinite().all() for t in _run(small, prompt, forced))


def test_positions_outside_the_cache_are_refused(gpu):
    m = Qwen2AwqDecoder(Qwen2Shape(num_heads=4, num_kv_heads=2, **TINY), max_seq_len=8, seed=1, device=gpu)
    for pos in (-1, 8, 1 << 40):
        with pytest.raises(ValueError):
            m.decode_logits(torch.tensor(3), pos)
    with pytest.raises(ValueError):
        m.prefill(torch.zeros(9, dtype=torch.int64))
    m.prefill(torch.zeros(8, dtype=torch.int64))
    assert torch.equal(m.decode_logits(torch.tensor(3), torch.tensor(7)), m.decode_logits(torch.tensor(3), 7))


def test_replaced_projections_are_called(gpu, monkeypatch):
    """Projections set on the object or on the class after construction."""
    m = Qwen2AwqDecoder(Qwen2Shape(num_heads=4, num_kv_heads=2, **TINY), max_seq_len=40, seed=1, device=gpu)
    prompt, forced = torch.arange(20), torch.arange(3)
    want, own, calls = _run(m, prompt, forced), Qwen2AwqDecoder.linear, []

    def linear(self, *a, **kw):
        calls.append(1)
        return own(self, *a, **kw)

    m.linear = linear.__get__(m)
    assert _close(_run(m, prompt, forced), want) and len(calls) == 4 * 2 * 4
    del m.linear
    assert all(map(torch.equal, _run(m, prompt, forced), want)) and len(calls) == 4 * 2 * 4
    monkeypatch.setattr(Qwen2AwqDecoder, "linear", linear)
    assert _close(_run(m, prompt, forced), want) and len(calls) == 2 * 4 * 2 * 4
