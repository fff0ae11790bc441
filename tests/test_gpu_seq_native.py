"""The native sequence layer with a normalised bank and without a backward: against the per-op
functions (both within the bf16 gate), a no-grad call against the training forward bit for bit, and
the one-pass normalised rows against the two kernels they replace."""

import pytest
import torch

from helpers import assert_parity, gen

pytestmark = pytest.mark.gpu


def _layer(dev, d, H, HK, C, k, norm, strategy):
    from memory_amd.model import RoutedMemoryLayer
    torch.manual_seed(5)
    layer = RoutedMemoryLayer(d, H, C, 64, k, num_kv_heads=HK, wo_init_zero=False, routing_strategy=strategy,
                              routing_window_size=16 if "rolling" in strategy else None,
                              normalize_shared_routed_before_mixing=norm is not None,
                              shared_routed_norm_type=norm or "rms").to(dev)
    with torch.no_grad():
        for n in "qkvo":
            lin = getattr(layer.memory_attn, n + "_proj")
            lin.weight.normal_(0, 0.08)
            lin.to(torch.bfloat16)
        layer.router.router.weight.normal_(0, 0.08)
    return layer


@pytest.mark.parametrize("norm", [None, "rms", "layernorm"])
@pytest.mark.parametrize("B,L,d,H,HK,C,k,strategy", [(2, 96, 256, 4, 4, 33, 4, "sequence"),
                                                     (3, 200, 768, 12, 4, 70, 20, "sequence-rolling"),
                                                     (1, 33, 1024, 16, 2, 40, 8, "sequence")])
def test_native_against_per_op(gpu_device, norm, B, L, d, H, HK, C, k, strategy):
    from memory_amd import seq_layer
    from memory_amd.router import compute_total_router_loss
    dev = gpu_device
    g = gen(B + L)
    h0 = torch.randn(B, L, d, generator=g).to(dev, torch.bfloat16)
    bank0 = (torch.randn(C * 64, d, generator=g) * 0.5).to(dev, torch.bfloat16)
    bank0[70] = 0                     # a zero row: rstd = 1 / sqrt(eps)
    dout = torch.randn(B, L, d, generator=g).to(dev, torch.bfloat16)
    layer = _layer(dev, d, H, HK, C, k, norm, strategy)
    assert seq_layer._native_sizes(h0, bank0, layer.router.router.bias, *(getattr(layer.memory_attn, n + "_proj").weight
                                                                          for n in "qkvo"),
                                   (C, 64, 1, k, 2.5, H, HK, {None: 0, "rms": 1, "layernorm": 2}[norm], 1e-6, True))

    def step(fused):
        layer.fused = fused
        for p in layer.parameters():
            p.grad = None
        h, bank = h0.clone().requires_grad_(True), bank0.clone().requires_grad_(True)
        out, losses = layer(h, bank)
        total = compute_total_router_loss(losses, 0.01, 0.0, 0.001)
        torch.autograd.backward([out, total], [dout, None])
        return {"out": out.detach(), "loss": total.detach(), "dh": h.grad, "dbank": bank.grad,
                **{n: p.grad for n, p in layer.named_parameters()}}

    a, b = step(True), step(False)
    for n in b:
        assert_parity(a[n], b[n], torch.bfloat16, n)
    layer.fused = True
    with torch.no_grad():
        out, _ = layer(h0, bank0, return_losses=False)
    assert torch.equal(out, a["out"])
    for p in layer.parameters():      # grad mode on, nothing to differentiate: the same forward
        p.requires_grad_(False)
    out, _ = layer(h0, bank0, return_losses=False)
    assert torch.equal(out, a["out"]) and not out.requires_grad


@pytest.mark.parametrize("norm", ["rms", "layernorm"])
@pytest.mark.parametrize("d", [8, 512, 520, 768, 1032, 2048, 2056, 4096])
def test_norm_gather_rows(gpu_device, norm, d):
    from memory_amd import _lib as lib
    from memory_amd import ops
    dev = gpu_device
    g = gen(d)
    C = 9
    bank = (torch.randn(C * 64, d, generator=g) * 3 + 1).to(dev, torch.bfloat16)
    plan = ops.chapter_plan(torch.tensor([7, 2, 2, 5, -1], dtype=torch.int32, device=dev), C)
    code = ops.norm_code(norm)
    mean, rstd = ops.row_stats(bank, plan, 64, code, 1e-6)
    n = 3 * 64
    mean2, rstd2 = torch.empty_like(mean), torch.empty_like(rstd)
    out = torch.empty(plan.max_u * 64, d, device=dev, dtype=torch.bfloat16)
    lib.call("moc_norm_gather_rows", bank.data_ptr(), d, plan.uniq.data_ptr(), plan.n_uniq.data_ptr(), plan.max_u, code,
             1e-6, mean2.data_ptr(), rstd2.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert_parity(mean2[:n], mean[:n], torch.float32, "mean")
    assert_parity(rstd2[:n], rstd[:n], torch.float32, "rstd")
    rows = torch.cat([torch.arange(c * 64, c * 64 + 64) for c in (2, 5, 7)])
    x = bank[rows.to(dev)].double()
    want = (x - mean[:n, None].double()) * rstd[:n, None].double()
    assert_parity(out[:n], want, torch.bfloat16, "rows")
