"""The attention forward and dQ with the slots split over workgroups (small grids) against the
unsplit kernels on the same operands: split counts from two to one slot each, ragged query rows,
grouped heads, skipped slots (a whole split of them, and a row of only skipped slots), zero and tiny
weights."""

import pytest
import torch

from helpers import assert_parity, gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,L,H,HK,NS", [(1, 1, 4, 4, 33), (2, 130, 4, 2, 9), (1, 509, 12, 12, 65), (4, 100, 4, 1, 20),
                                         (3, 257, 12, 4, 24)])
def test_split_against_unsplit(gpu_device, dtype, B, L, H, HK, NS):
    from memory_amd import _lib as lib
    dev = gpu_device
    g = gen(3 * B + L + NS)
    U = NS + 3
    kv = torch.randn(U * 64, 2 * HK * 64, generator=g).to(dev, dtype)
    q, dout = (torch.randn(B, L, H, 64, generator=g).to(dev, dtype) for _ in range(2))
    slot = torch.stack([torch.randperm(U, generator=g)[:NS] for _ in range(B)]).to(torch.int32)
    slot[0, : max(1, NS // 3)] = -1          # the first splits of sequence 0 hold skipped slots only
    if B > 2:
        slot[1, :] = -1                      # a sequence without any slot
    om = torch.rand(B, NS, generator=g) * 2 / NS
    om[-1, NS // 2:] = 0.0
    om[-1, 0] = 1e-30
    slot, om = slot.to(dev), om.to(dev)
    KV, row, es = HK * 64, 2 * HK * 64, kv.element_size()
    Lp = (L + 127) // 128 * 128
    dt = lib.dtype_code(dtype)
    nbytes = lib.query("moc_xattn_split_workspace", dt, B, L, H, NS)
    assert nbytes > 0, "these sizes are split"
    kvl = (kv.numel() - KV, 64 * row, 64, row)
    s = torch.cuda.current_stream().cuda_stream

    def run(ws):
        out = torch.empty_like(q)
        lse = torch.empty(B, H, Lp, device=dev)
        p, n = (None, 0) if ws is None else (ws.data_ptr(), ws.numel())
        lib.call("moc_xattn_fwd_split", dt, q.data_ptr(), kv.data_ptr(), kv.data_ptr() + KV * es, *kvl, slot.data_ptr(),
                 om.data_ptr(), B, L, H, HK, 64, 64, NS, 0.125, out.data_ptr(), lse.data_ptr(), p, n, s)
        delta, dq = torch.empty(B, H, Lp, device=dev), torch.empty_like(q)
        lib.call("moc_xattn_bwd_dq_delta_split", dt, q.data_ptr(), kv.data_ptr(), kv.data_ptr() + KV * es, *kvl,
                 slot.data_ptr(), om.data_ptr(), out.data_ptr(), dout.data_ptr(), lse.data_ptr(), delta.data_ptr(), B, L,
                 H, HK, 64, 64, NS, 0.125, dq.data_ptr(), p, n, s)
        return out, lse, delta, dq

    a = run(None)
    b = run(torch.full((nbytes,), 255, device=dev, dtype=torch.uint8))   # NaN patterns: every read was written
    assert torch.equal(torch.isinf(a[1]), torch.isinf(b[1])) and not torch.isnan(b[1]).any()
    assert_parity(b[0], a[0], dtype, "out")
    assert_parity(torch.where(torch.isinf(b[1]), 0.0, b[1]), torch.where(torch.isinf(a[1]), 0.0, a[1]), torch.float32,
                  "lse")
    assert_parity(b[2], a[2], torch.float32 if dtype == torch.float32 else dtype, "delta")
    assert_parity(b[3], a[3], dtype, "dq")
    if dtype == torch.bfloat16:
        # one reference maximum per row, so every P~ has the unsplit kernel's bf16 rounding and the outputs
        # are apart by float32 sums: below 2^-16 of a value, which moves its rounding to 2^-9 once in 64
        # times at most, and never by more than one step (2^-8 of the value, and of the row for sums
        # that cancel)
        x, y = a[0].double(), b[0].double()
        assert (x != y).double().mean().item() <= 1 / 64
        assert bool(((x - y).abs() <= 2.0 ** -7 * y.abs() + 2.0 ** -16 * y.abs().amax()).all())
