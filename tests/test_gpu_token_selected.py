"""Token-routed branch over the selected chapters only, against the same branch over the whole bank:
every mode, ids outside the bank, chapters nobody selects, and no valid selection at all."""

import pytest
import torch

from helpers import gen

pytestmark = pytest.mark.gpu


def _run(dev, B, Lq, H, HK, C, k, version, weighted, factor, monkeypatch, idx, tail=True, wdt=torch.bfloat16):
    from memory_amd import sparse_attention as sa
    from memory_amd.model import split_rows
    monkeypatch.setattr(sa, "SELECT_FACTOR", factor)
    g = gen(C * 100 + Lq)
    d = 64 * H
    bf = torch.bfloat16
    q = torch.randn(B, Lq, H, 64, generator=g).to(dev, bf).requires_grad_()
    bank = (torch.randn((C + 1) * 64, d, generator=g) * 0.3).to(dev, bf).requires_grad_()
    wk = (torch.randn(HK * 64, d, generator=g) * 0.05).to(dev, wdt).requires_grad_()
    wv = (torch.randn(HK * 64, d, generator=g) * 0.05).to(dev, wdt).requires_grad_()
    w = torch.rand(B, Lq, k, generator=g).to(dev).requires_grad_() if weighted else None
    up = torch.randn(B, Lq, H, 64, generator=g).to(dev, bf)
    routed = split_rows(bank, 64)[1] if tail else bank[64:].clone()
    out = sa.token_routed_attention(q, routed, wk, wv, idx.to(dev), w, tokens_per_chapter=64, version=version,
                                    num_kv_heads=HK)
    sel = out.grad_fn.sel if hasattr(out.grad_fn, "sel") else None
    out.backward(up)
    return [out.detach(), q.grad, bank.grad, wk.grad, wv.grad, None if w is None else w.grad], sel is not None


@pytest.mark.parametrize("B,Lq,H,HK,C,k,version,weighted,wdt", [
    (1, 1, 4, 4, 40, 1, "v4", True, torch.bfloat16),
    (1, 37, 4, 4, 40, 3, "v4", True, torch.bfloat16),
    (2, 65, 12, 4, 200, 4, "v5", True, torch.float32),
    (1, 300, 8, 2, 61, 2, "v2", False, torch.bfloat16),
    (1, 17, 4, 4, 40, 3, "none", True, torch.bfloat16),
    (3, 90, 12, 12, 30, 8, "v4", True, torch.bfloat16),
])
def test_selected_equals_whole_bank(gpu_device, monkeypatch, B, Lq, H, HK, C, k, version, weighted, wdt):
    dev = gpu_device
    g = gen(Lq + k)
    # distinct ids per token out of the lower half of the bank (the upper half is never selected),
    # with ids outside the bank among them; "none": no valid id at all
    pool = max(k, C // 2)
    idx = torch.stack([torch.randperm(pool, generator=g)[:k] for _ in range(B * Lq)]).view(B, Lq, k).to(torch.int32)
    if Lq > 1:
        idx[:, ::5, 0] = -1
        idx[:, 3::7, 0] = C
    if version == "none":
        idx, version = torch.full_like(idx, -1), "v4"
    args = (dev, B, Lq, H, HK, C, k, version, weighted)
    got, sel = _run(*args, 1 << 30, monkeypatch, idx, wdt=wdt)
    want, whole = _run(*args, 0, monkeypatch, idx, wdt=wdt)
    assert sel and not whole
    for name, a, b in zip(("out", "dq", "dbank", "dwk", "dwv", "dw"), got, want):
        assert (a is None) == (b is None), name
        if a is None:
            continue
        assert a.dtype == b.dtype and a.shape == b.shape
        # the same products of the same rounded operands; the bank rows' products and the weight
        # gradient add up in another order, one bf16 rounding (2^-9) apart at the output at most
        err = ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-9)).item()
        assert err <= 2.0 ** -8, (name, err)
    # bank rows: the shared chapter, `pool` chapters that may be selected, chapters that nobody selects
    rest = got[2][(1 + pool) * 64:]
    assert rest.shape[0] == (C - pool) * 64 > 0 and bool((rest == 0).all())
    again, _ = _run(*args, 1 << 30, monkeypatch, idx, tail=False, wdt=wdt)
    assert torch.equal(again[2], got[2]) and torch.equal(again[0], got[0])


def test_other_forms_take_the_whole_bank(gpu_device, monkeypatch):
    from memory_amd import sparse_attention as sa
    dev = gpu_device
    bf = torch.bfloat16
    bank, wkv = torch.zeros(640, 256, device=dev, dtype=bf), torch.zeros(512, 256, device=dev, dtype=bf)
    idx = torch.zeros(1, 4, 2, dtype=torch.int32, device=dev)
    assert sa._selected_only(bank, wkv, idx, 10)
    flat = torch.zeros(640 * 256 + 1, device=dev, dtype=bf)
    for b, w, i in ((bank.float(), wkv, idx), (bank, wkv.float(), idx), (bank[:, :192], wkv[:, :192], idx),
                    (bank, wkv[:128], idx), (bank, wkv, idx.unsqueeze(2)), (bank, wkv, idx[:, :0]),
                    (flat[1:].view(640, 256), wkv, idx)):
        assert not sa._selected_only(b, w, i, 10)
    assert not sa._selected_only(bank, wkv, idx, 2)
