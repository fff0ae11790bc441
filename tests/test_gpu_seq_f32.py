"""The float32 sequence layer in one host call each way (moc_seq_layer_f32_*) against the per-op
autograd functions, over the forms it accepts, and the calls that stay with those functions."""

import pytest
import torch

from helpers import gen

pytestmark = pytest.mark.gpu


def _layer(dev, d, H, HK, C, S, k, norm, strategy="sequence", wr_dtype=torch.float32):
    from memory_amd.model import RoutedMemoryLayer
    layer = RoutedMemoryLayer(d, H, C, 64, k, num_shared_chapters=S, num_kv_heads=HK, wo_init_zero=False,
                              normalize_shared_routed_before_mixing=norm != "none",
                              shared_routed_norm_type="rms" if norm == "none" else norm, routing_strategy=strategy,
                              routing_window_size=7)
    g = gen(d + C + k)
    with torch.no_grad():
        for p in layer.parameters():
            p.copy_(torch.randn(p.shape, generator=g) * 0.05)
    layer = layer.to(dev)
    layer.router.to(wr_dtype) if wr_dtype != torch.float32 else None
    return layer


def _step(layer, h, bank, up, fused, frozen=(), losses=True):
    layer.fused = fused
    for p in layer.parameters():
        p.grad = None
    h = h.detach().clone().requires_grad_("h" not in frozen)
    bank = bank.detach().clone().requires_grad_("bank" not in frozen)
    out, ls = layer(h, bank, return_losses=losses)
    loss = (out * up).sum() + sum(v for v in ls.values())
    loss.backward()
    grads = {n: p.grad for n, p in layer.named_parameters()}
    grads.update(h=h.grad, bank=bank.grad)
    return out.detach(), {n: v.detach() for n, v in ls.items()}, grads


def _same(a, b, name):
    assert (a is None) == (b is None), name
    if a is None:
        return
    # the two paths differ in the products' summation order only: a few roundings of 2^-24 per
    # product of up to ~1,000 terms, carried through the chain's four products
    err = ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-12)).item()
    assert err < 2e-5, (name, err)


CASES = [
    # B, L, d, H, HK, C, S, k, norm, strategy
    (1, 1, 64, 1, 1, 3, 1, 2, "none", "sequence"),
    (2, 128, 256, 4, 4, 33, 1, 4, "none", "sequence"),
    (3, 251, 256, 4, 2, 257, 1, 16, "rms", "sequence"),
    (2, 33, 128, 2, 1, 9, 3, 6, "layernorm", "sequence-rolling"),
    (1, 130, 320, 5, 5, 40, 2, 1, "rms", "sequence"),
]


@pytest.mark.parametrize("case", CASES)
def test_f32_layer_equals_per_op(gpu_device, case, monkeypatch):
    from memory_amd import _lib as lib
    from memory_amd import seq_layer
    B, L, d, H, HK, C, S, k, norm, strategy = case
    dev = gpu_device
    layer = _layer(dev, d, H, HK, C, S, k, norm, strategy)
    g = gen(B * L)
    h, up = torch.randn(B, L, d, generator=g).to(dev), torch.randn(B, L, d, generator=g).to(dev)
    bank = (torch.randn(C * 64, d, generator=g) * 0.1).to(dev)
    called = []
    real = seq_layer.call
    monkeypatch.setattr(seq_layer, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    for frozen in ((), ("h",), ("bank",)):
        got = _step(layer, h, bank, up, True, frozen)
        assert called == ["moc_seq_layer_f32_fwd", "moc_seq_layer_f32_bwd"]
        called.clear()
        want = _step(layer, h, bank, up, False, frozen)
        assert not called
        _same(got[0], want[0], "out")
        for n in want[1]:
            _same(got[1][n], want[1][n], n)
        for n in want[2]:
            _same(got[2][n], want[2][n], n)
    layer.fused = True
    with torch.no_grad():
        assert torch.equal(layer(h, bank, return_losses=False)[0], got[0])
    for p in (layer.memory_attn.k_proj.weight, layer.memory_attn.o_proj.weight, layer.router.router.bias):
        p.requires_grad_(False)
    got, want = _step(layer, h, bank, up, True, losses=False), _step(layer, h, bank, up, False, losses=False)
    for n in want[2]:
        _same(got[2][n], want[2][n], n)


def test_f32_layer_stays_per_op(gpu_device, monkeypatch):
    """Unpacked or unaligned inputs, other sizes and types, hooks and autocast keep the per-op functions."""
    from memory_amd import seq_layer
    dev = gpu_device
    layer = _layer(dev, 128, 2, 2, 9, 1, 3, "none")
    g = gen(5)
    h, bank = torch.randn(2, 40, 128, generator=g).to(dev), (torch.randn(9 * 64, 128, generator=g) * 0.1).to(dev)
    up = torch.randn(2, 40, 128, generator=g).to(dev)
    called = []
    real = seq_layer.call
    monkeypatch.setattr(seq_layer, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    want = layer(h, bank)[0]
    assert called.pop() == "moc_seq_layer_f32_fwd"
    flat = torch.empty(h.numel() + 1, device=dev)
    flat[1:] = h.reshape(-1)
    for x in (flat[1:].view(h.shape), h.transpose(0, 1).contiguous().transpose(0, 1)):
        _same(layer(x, bank)[0], want, "layout")
    hits = []
    handle = layer.memory_attn.register_forward_hook(lambda *a: hits.append(1))
    _same(layer(h, bank)[0], want, "hook")
    handle.remove()
    assert hits == [1]
    with torch.autocast("cuda", torch.bfloat16):
        layer(h, bank)
    assert not called
    # an unaligned or absent upstream gradient reaches the same backward
    x = h.clone().requires_grad_()
    out, losses = layer(x, bank)
    flat[1:] = up.reshape(-1)
    out.backward(flat[1:].view(h.shape))
    y = h.clone().requires_grad_()
    layer.fused = False
    layer(y, bank)[0].backward(up)
    _same(x.grad, y.grad, "unaligned upstream")
    layer.fused = True
    x.grad = y.grad = None
    sum(layer(x, bank)[1].values()).backward()
    layer.fused = False
    sum(layer(y, bank)[1].values()).backward()
    _same(x.grad, y.grad, "losses alone")


@pytest.mark.parametrize("norm", ["none", "rms"])
def test_f32_layer_recorded_backward(gpu_device, norm):
    """A penalty on o_proj's weight gradient (create_graph), alone and added to another loss, against float64
    autograd: the gradient is a recorded product of the attention's output, whose own derivative is the
    attention's backward.  Gradients to 1e-4 of their largest value: two float32 chains of sums of up to 330
    keys (2^-24 each, square-root growth below 1e-5) and the penalty's squares."""
    import oracle as O
    from memory_amd import seq_layer
    dev = gpu_device
    B, L, d, H, C, S, k = 2, 40, 128, 2, 9, 1, 4
    layer = _layer(dev, d, H, H, C, S, k, norm)
    g = gen(77)
    h, up = torch.randn(B, L, d, generator=g), torch.randn(B, L, d, generator=g)
    bank = torch.randn(C * 64, d, generator=g)
    attn, r = layer.memory_attn, layer.router.router
    params = [r.weight, r.bias, attn.q_proj.weight, attn.k_proj.weight, attn.v_proj.weight, attn.o_proj.weight]
    leaves = [t.detach().double().cpu().requires_grad_() for t in (h, bank, *params)]
    ref = O.sequence_memory_layer(*leaves, H=H, HK=H, C=C, T=64, S=S, top_k=k, routed_scale=2.5, normalize=norm != "none")
    hd, bd = h.to(dev).requires_grad_(), bank.to(dev).requires_grad_()
    assert seq_layer.supported_f32(hd, bd, *params, num_chapters=C, tokens_per_chapter=64, num_shared=S, top_k=k,
                                   num_heads=H, num_kv_heads=H)
    out = layer(hd, bd, return_losses=False)[0]
    got_leaves = [hd, bd, *params]
    for extra in (0.0, 0.5):
        def penalty(out, up, wo):
            gw, = torch.autograd.grad((out * up).sum(), wo, create_graph=True)
            return (gw ** 2).sum() * 0.01 + extra * (out ** 2).sum()

        want = torch.autograd.grad(penalty(ref, up.double(), leaves[-1]), leaves, retain_graph=True, allow_unused=True)
        got = torch.autograd.grad(penalty(out, up.to(dev), params[-1]), got_leaves, retain_graph=True, allow_unused=True)
        for n, a, b in zip(("h", "bank", "wr", "br", "wq", "wk", "wv", "wo"), got, want):
            if n == "wo" and extra == 0.0:      # the weight's gradient does not depend on the weight
                assert a is None or a.abs().max().item() <= 1e-6
                continue
            err = ((a.double().cpu() - b).abs().max() / b.abs().max()).item()
            assert err <= 1e-4, (extra, n, err)


def test_f32_layer_recorded_gradients_are_the_gradients(gpu_device):
    """create_graph changes no first-order gradient, frozen inputs keep none, and one input may depend on
    another."""
    dev = gpu_device
    layer = _layer(dev, 128, 2, 1, 9, 1, 3, "layernorm")
    g = gen(6)
    h = torch.randn(2, 33, 128, generator=g).to(dev)
    bank = (torch.randn(9 * 64, 128, generator=g) * 0.1).to(dev)
    layer.memory_attn.k_proj.weight.requires_grad_(False)

    def grads(create_graph):
        x = h.clone().requires_grad_()
        b = (bank + x.mean() * 0.1)
        out, losses = layer(x, b)
        leaves = [x] + [p for p in layer.parameters() if p.requires_grad]
        return torch.autograd.grad((out ** 2).sum() + sum(losses.values()), leaves, create_graph=create_graph)

    for a, b in zip(grads(True), grads(False)):
        _same(a, b, "gradient")


def test_f32_layer_asks_the_callers_router(gpu_device):
    """A router subclass, and router or attention methods replaced on the instance, are used as the per-op
    path uses them."""
    from memory_amd.router import ChapterRouter
    dev = gpu_device
    g = gen(8)
    h, bank = torch.randn(2, 40, 128, generator=g).to(dev), (torch.randn(9 * 64, 128, generator=g) * 0.1).to(dev)

    class Noisy(ChapterRouter):
        def sequence_logits(self, *a, **kw):
            return -super().sequence_logits(*a, **kw)

    def results(change):
        layer = _layer(dev, 128, 2, 2, 9, 1, 3, "none")
        plain = layer(h, bank)[0]
        change(layer)
        a = layer(h, bank)[0]
        layer.fused = False
        return plain, a, layer(h, bank)[0]

    def subclass(layer):
        other = Noisy(128, 9, 3).to(dev)
        other.load_state_dict(layer.router.state_dict())
        layer.router = other

    def replaced(layer):
        real = layer.router.sequence_logits
        layer.router.sequence_logits = lambda *a, **kw: -real(*a, **kw)

    def queries(layer):
        real = layer.memory_attn._queries
        layer.memory_attn._queries = lambda *a, **kw: real(*a, **kw) * 2

    for change in (subclass, replaced, queries):
        plain, a, per_op = results(change)
        _same(a, per_op, change.__name__)
        assert not torch.allclose(a, plain, rtol=1e-3)


@pytest.mark.parametrize("B,L,C,k,one_call", [(1, 8192, 5, 2, True), (1, 8193, 5, 2, False), (43, 3, 128, 2, True),
                                              (44, 3, 129, 2, False)])
def test_f32_training_step_long_reductions(gpu_device, monkeypatch, B, L, C, k, one_call):
    """Training steps whose weight gradients reduce over more than 8,192 tokens or bank rows keep the per-op
    functions, their forwards alone do not; both give the same."""
    from memory_amd import seq_layer
    dev = gpu_device
    layer = _layer(dev, 64, 1, 1, C, 1, k, "none")
    g = gen(B + L)
    h, up = torch.randn(B, L, 64, generator=g).to(dev), torch.randn(B, L, 64, generator=g).to(dev)
    bank = (torch.randn(C * 64, 64, generator=g) * 0.1).to(dev)
    called = []
    real = seq_layer.call
    monkeypatch.setattr(seq_layer, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    got = _step(layer, h, bank, up, True)
    assert called == (["moc_seq_layer_f32_fwd", "moc_seq_layer_f32_bwd"] if one_call else [])
    called.clear()
    with torch.no_grad():
        _same(layer(h, bank, return_losses=False)[0], got[0], "forward alone")
    assert called == ["moc_seq_layer_f32_fwd"]
    want = _step(layer, h, bank, up, False)
    for n in want[2]:
        _same(got[2][n], want[2][n], n)
