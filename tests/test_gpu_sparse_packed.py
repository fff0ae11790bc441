"""The packed form of the FSA entry points (per-head block choices as one plan) against a float64
reference, at the sizes where its kernels can go wrong: units of 64 and 128 keys, a half last block,
one to 16 query rows per edge, row counts around the 32- / 64-row steps, units split over several
workgroups, ids out of range in either id type; and the segments it replaces on the same inputs."""

import pytest
import torch

from helpers import assert_parity, gen

pytestmark = pytest.mark.gpu


def _reference(q, k, v, idx, w, mode, BS, scale):
    """sum over the chosen blocks in float64; a block past the keys keeps the keys inside."""
    B, Tq, HQ, _ = q.shape
    Tk, HK = k.shape[1], k.shape[2]
    S, G = idx.shape[-1], HQ // HK
    rows = idx.unsqueeze(-1) * BS + torch.arange(BS)                     # (B, Tq, HK, S, BS)
    ok = (idx >= 0).unsqueeze(-1) & (rows < Tk) & (rows >= 0)
    rows = torch.where(ok, rows, torch.zeros_like(rows))
    out = []
    for b in range(B):
        kb = k[b].permute(1, 0, 2)                                       # (HK, Tk, 64)
        vb = v[b].permute(1, 0, 2)
        h = torch.arange(HK).view(1, HK, 1, 1)
        kk, vv = kb[h, rows[b]], vb[h, rows[b]]                          # (Tq, HK, S, BS, 64)
        s = torch.einsum("thgd,thsjd->thgsj", q[b].view(Tq, HK, G, 64), kk) * scale
        s = s.masked_fill(~ok[b].unsqueeze(2), float("-inf"))
        wb = None if w is None else (w[b] if w.dim() == 4 else w[b].unsqueeze(1).expand(Tq, HK, S))
        if mode == 0:
            p = torch.softmax(s, -1).nan_to_num(0.0) * wb.view(Tq, HK, 1, S, 1)
        else:
            if mode == 3:
                s = s + torch.log(wb.clamp_min(1e-20)).view(Tq, HK, 1, S, 1)
            e = torch.exp(s - s.amax((-1, -2), keepdim=True).clamp_min(-1e30))
            if mode == 2:
                e = e * wb.clamp_min(0).view(Tq, HK, 1, S, 1)
            p = e / e.sum((-1, -2), keepdim=True).clamp_min(1e-300)
        out.append(torch.einsum("thgsj,thsjd->thgd", p, vv).reshape(Tq, HQ, 64))
    return torch.stack(out)


# (B, Tq, HQ, HK, Tk, S, BS): a few rows per unit; G = 16 on 1.5 blocks of 128 (units split over
# workgroups, a half last block); G = 1, 33 rows past a step; G = 3, three 64-key blocks of 192; a
# batch of shared keys is covered by Bk = 1 below
CASES = [(1, 33, 3, 1, 320, 2, 64), (2, 150, 16, 1, 192, 2, 128), (1, 129, 4, 4, 192, 3, 64),
         (2, 65, 6, 2, 576, 2, 192), (1, 400, 8, 2, 384, 2, 128), (1, 300, 12, 12, 256, 4, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_packed_against_float64(gpu_device, dtype, mode, case):
    from memory_amd import sparse_attention as SA
    B, Tq, HQ, HK, Tk, S, BS = CASES[case]
    print(f"packed {CASES[case]} mode={mode} {dtype}", flush=True)
    dev = gpu_device
    g = gen(500 + 10 * case + mode)
    M = -(-Tk // BS)
    q, dO = (torch.randn(B, Tq, HQ, 64, generator=g) for _ in range(2))
    Bk = 1 if case == 4 else B
    k, v = (torch.randn(Bk, Tk, HK, 64, generator=g) for _ in range(2))
    idx = torch.rand(B, Tq, HK, M, generator=g).argsort(-1)[..., :S]
    if idx.shape[-1] < S:
        S = idx.shape[-1]
    if mode != 0 and S > 1:     # skipped slots: below, past the end, and far past 32 bits
        idx[:, ::5, :, 0] = -1
        idx[:, 1::7, :, 1] = M
    wide = case % 2 == 1
    dev_idx = idx.clone()
    if wide and mode != 0 and S > 1:
        dev_idx[:, 1::7, :, 1] = 2 ** 40
    w = None
    if mode == 2:
        w = torch.rand(B, Tq, HK, S, generator=g) + 0.05
    elif mode in (0, 3):
        w = torch.softmax(torch.randn(B, Tq, S, generator=g), -1)
    scale = 0.2
    r = [t.to(dtype).double().requires_grad_(True) for t in (q, k, v)]
    rw = None if w is None else w.double().requires_grad_(True)
    ref = _reference(r[0], r[1].expand(B, -1, -1, -1), r[2].expand(B, -1, -1, -1), idx, rw, mode, BS, scale)
    (ref * dO.to(dtype).double()).sum().backward()

    def run():
        t = [x.to(dev, dtype).requires_grad_(True) for x in (q, k, v)]
        tw = None if w is None else w.to(dev).requires_grad_(True)
        di = dev_idx.to(dev, torch.int64 if wide else torch.int32)
        kw = dict(softmax_scale=scale, disable_causal_mask=True)
        if mode == 0:
            out = SA.FSA_topk_sparse_attention_weighted_bthd(*t, di, tw, BS, **kw)
        elif mode == 3:
            out = SA.FSA_topk_sparse_attention_weighted_joint_bias_bthd(*t, di, tw, BS, **kw)
        else:
            out = SA.FSA_topk_sparse_attention_bthd(*t, di, BS, block_weights_bths=tw, **kw)
        out.backward(dO.to(dev, dtype))
        return [out.detach()] + [x.grad for x in t] + ([] if tw is None else [tw.grad])

    got = run()
    names = ["out", "dq", "dk", "dv", "dw"]
    want = [ref.detach()] + [x.grad for x in r] + ([] if rw is None else [rw.grad])
    for n, a, b in zip(names, got, want):
        assert_parity(a, b, dtype, n)
    for n, a, b in zip(names, got, run()):      # fixed-order sums: the same bits again
        assert torch.equal(a, b), n


@pytest.mark.parametrize("scale", [0.125, 0.0, -0.125])
def test_packed_scale_signs(gpu_device, scale):
    """A softmax scale of any sign gives what the segments give (the pipelined kernels take a
    positive one; the others stay on the one-wave-per-unit kernels)."""
    from memory_amd import sparse_attention as SA
    dev = gpu_device
    g = gen(77)
    q, k, v = (torch.randn(1, n, h, 64, generator=g).to(dev, torch.bfloat16) for n, h in ((256, 8), (256, 2), (256, 2)))
    idx = torch.rand(1, 256, 2, 2, generator=g).argsort(-1).to(dev, torch.int32)
    out = SA.FSA_topk_sparse_attention_bthd(q, k, v, idx, 128, softmax_scale=scale, disable_causal_mask=True)
    seg = SA._FSAFunction.apply(q, k, v, None, (idx.unsqueeze(-1) * 2 + torch.arange(2, device=dev)).flatten(-2).int(), 1,
                                scale)
    assert_parity(out, seg, torch.bfloat16, f"scale {scale}")


@pytest.mark.parametrize("S,Tk", [(8, 2048), (3, 1088)])
def test_128_key_units_round_as_64_key_ones(gpu_device, S, Tk):
    """Outputs of 128-key units are no further from float64 than those of the same blocks as 64-key units
    (the segments): one maximum, and so one exact P, per 64 keys.  The ratio of the two errors over N =
    65,536 rows is a ratio of mean squares of at least 4 N independent terms (the roundings of a row's P
    and partial rows): 1 within 4 sqrt(2 / 4 N) / 2 = 0.0055; one maximum per 128 keys puts it at 1.018."""
    from memory_amd import sparse_attention as SA
    dev = gpu_device
    g = gen(S)
    Tq, HQ = 4096, 16
    q, k, v = (torch.randn(1, n, h, 64, generator=g).to(dev, torch.bfloat16) for n, h in ((Tq, HQ), (Tk, 1), (Tk, 1)))
    idx = torch.rand(1, Tq, 1, -(-Tk // 128), generator=g).argsort(-1)[..., :S]
    assert SA._packed_block(q, k, v, None, idx.to(dev), 1, 0.125, 128) == 128
    out = SA.FSA_topk_sparse_attention_bthd(q, k, v, idx.to(dev, torch.int32), 128, disable_causal_mask=True)
    sub = (idx.unsqueeze(-1) * 2 + torch.arange(2)).flatten(-2).to(dev, torch.int32)
    seg = SA._FSAFunction.apply(q, k, v, None, sub, 1, 0.125)
    ref = torch.cat([_reference(q[:, a:a + 256].double().cpu(), k.double().cpu(), v.double().cpu(), idx[:, a:a + 256], None,
                                1, 128, 0.125) for a in range(0, Tq, 256)], 1)
    err, base = ((t.double().cpu() - ref).norm().item() for t in (out, seg))
    print(f"S={S} Tk={Tk}: error ratio {err / base:.4f}", flush=True)
    assert err <= 1.0055 * base


@pytest.mark.parametrize("mode", [2, 3])
def test_128_key_units_block_weight_gradient(gpu_device, mode):
    """The block weights' gradient of 128-key units is free of the output's bf16 rounding: products of exact
    bf16 operands and float32 sums over 128 keys of 64 dims, P and lse to a few units of 2^-23, divided by
    the weight: below 1e-5 of the largest value here (2^-23 times the ~30 for the cancelling sum of a
    token's slots), against 1e-2 with the error of dO . out left in."""
    from memory_amd import sparse_attention as SA
    dev = gpu_device
    g = gen(90 + mode)
    Tq, HQ, Tk, S = 400, 8, 448, 3
    q, dO = (torch.randn(1, Tq, HQ, 64, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(1, Tk, 2, 64, generator=g).bfloat16() for _ in range(2))
    idx = torch.rand(1, Tq, 2, 4, generator=g).argsort(-1)[..., :S]
    idx[:, ::5, :, 0] = -1
    idx[:, ::10, :, 1] = 4                        # one valid block: no gradient at all
    idx[:, 7] = -1                                # none
    w = torch.softmax(torch.randn(1, Tq, 2, S, generator=g), -1)
    if mode == 2:
        w[:, 11, :, 0] = 0.0
    rw = w.double().requires_grad_(True)
    ref = _reference(q.double(), k.double(), v.double(), idx, rw, mode, 128, 0.125)
    (ref * dO.double()).sum().backward()
    fn = (SA.FSA_topk_sparse_attention_weighted_joint_bias_bthd if mode == 3 else
          lambda a, b, c, i, x, n, **kw: SA.FSA_topk_sparse_attention_bthd(a, b, c, i, n, block_weights_bths=x, **kw))
    tw = w.to(dev).requires_grad_(True)
    assert SA._packed_block(q.to(dev), k.to(dev), v.to(dev), tw, idx.to(dev), mode, 0.125, 128) == 128
    fn(q.to(dev), k.to(dev), v.to(dev), idx.to(dev, torch.int32), tw, 128, disable_causal_mask=True).backward(dO.to(dev))
    got, want = tw.grad.double().cpu(), rw.grad
    if mode == 2:                                 # the gradient at a weight of zero is the clamp's: none here
        got, want = (torch.where(w > 0, t, 0.0) for t in (got, want))
    assert ((got - want).abs().max() / want.abs().max()).item() <= 1e-5


def test_128_key_unit_with_a_half_of_infinite_scores(gpu_device):
    """Keys whose scores are -inf (here a whole half of a block) take no part, as in a softmax over the
    block."""
    from memory_amd import sparse_attention as SA
    dev = gpu_device
    g = gen(5)
    q = (torch.rand(1, 200, 4, 64, generator=g) + 0.1).to(dev, torch.bfloat16)
    k, v = (torch.randn(1, 256, 1, 64, generator=g).to(dev, torch.bfloat16) for _ in range(2))
    k[:, 64:128, :, 0] = -float("inf")
    k[:, 128:192, :, 0] = -float("inf")
    idx = torch.zeros(1, 200, 1, 2, dtype=torch.int32, device=dev)
    idx[..., 1] = 1
    out = SA.FSA_topk_sparse_attention_bthd(q, k, v, idx, 128, disable_causal_mask=True)
    s = torch.einsum("thd,jd->thj", q[0].double(), k[0, :, 0].double().nan_to_num(neginf=-1e300)) * 0.125
    assert_parity(out[0], torch.softmax(s, -1) @ v[0, :, 0].double(), torch.bfloat16, "out")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("S", [1, 4, 5, 7, 8])
def test_few_slot_combine_order(gpu_device, dtype, mode, S):
    """The combines for at most 8 slots against the one-wave-per-row kernels, which take the same rows with
    skipped slots up to 9: float32 adds in their order, to the same bits, and bf16 is apart by the order of
    float32 sums (8 roundings of 2^-24: 2^-20 of the largest value, and in log2 for lse) and then one
    rounding of its own (a step of at most 2^-7 of the value)."""
    from memory_amd import _lib as lib
    dev = gpu_device
    g = gen(10 * S + mode)
    ntok, rpe, S9 = 301, 3, 9
    dt, st = lib.dtype_code(dtype), torch.cuda.current_stream().cuda_stream
    part = torch.randn(ntok, S9, rpe, 64, generator=g).to(dtype)
    lse = torch.randn(ntok, S9, rpe, generator=g) * 3
    w = torch.rand(ntok, S9, generator=g)
    edge = torch.zeros(ntok, S9, dtype=torch.int32)
    edge[:, S:] = -1
    edge[::5, 0] = -1
    edge[7] = -1
    part[edge.eq(-1).unsqueeze(-1).expand(ntok, S9, rpe)] = float("nan")     # never written by the kernels

    def run(n):
        p, l, ww, e = (t[:, :n].contiguous().to(dev) for t in (part, lse, w, edge))
        out, dq = (torch.empty(ntok, rpe, 64, device=dev, dtype=dtype) for _ in range(2))
        lj = torch.empty(ntok, rpe, device=dev)
        lib.call("moc_sparse_combine", dt, p.data_ptr(), l.data_ptr(), e.data_ptr(), None if mode == 1 else ww.data_ptr(),
                 mode, n, rpe, ntok, rpe, 0, out.data_ptr(), None if mode == 0 else lj.data_ptr(), st)
        lib.call("moc_sparse_dq_combine", dt, p.data_ptr(), e.data_ptr(), n, rpe, ntok, rpe, 0, dq.data_ptr(), st)
        return [out, dq] + ([] if mode == 0 else [lj])

    for a, b in zip(run(S), run(S9)):
        assert not torch.isnan(a).any()
        if dtype == torch.float32:
            assert torch.equal(a, b)
            continue
        a, b, step = a.double(), b.double(), 2.0 ** -7 if a.dtype == dtype else 0.0
        a, b = (torch.where(torch.isinf(t), 1e9, t) for t in (a, b))
        ok = torch.where(b < 1e9, b, 0.0).abs().max()
        assert bool(((a - b).abs() <= step * b.abs() + 2.0 ** -20 * ok).all())


@pytest.mark.parametrize("HK,per_head", [(1, False), (2, True)])
def test_mixture_recorded_backward(gpu_device, HK, per_head):
    """A penalty on the block weights' gradient (create_graph) at 128-key blocks: the weights' gradient is a
    recorded product of the slots' outputs, whose own derivative is the attention's backward; against float64
    autograd, bf16 gate."""
    from memory_amd import sparse_attention as SA
    dev = gpu_device
    g = gen(40 + HK)
    B, Tq, HQ, Tk, S = 1, 130, 4, 512, 3
    q, dO = (torch.randn(B, Tq, HQ, 64, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(B, Tk, HK, 64, generator=g).bfloat16() for _ in range(2))
    idx = torch.rand(B, Tq, HK, 4, generator=g).argsort(-1)[..., :S]
    w = torch.rand(B, Tq, HK, S, generator=g) if per_head else torch.rand(B, Tq, S, generator=g)
    t = [x.to(dev).requires_grad_() for x in (q, k, v, w)]
    r = [x.double().requires_grad_() for x in (q, k, v, w)]
    assert SA._packed_block(*t[:3], t[3], idx.to(dev), 0, 0.125, 128) == 128
    out = SA.FSA_topk_sparse_attention_weighted_bthd(*t[:3], idx.to(dev, torch.int32), t[3], 128, disable_causal_mask=True)
    ref = _reference(*r[:3], idx, r[3], 0, 128, 0.125)
    first = torch.autograd.grad(out, t, dO.to(dev), retain_graph=True)
    recorded = torch.autograd.grad(out, t, dO.to(dev), create_graph=True)
    for n, a, b in zip("qkvw", recorded, first):
        assert_parity(a, b, torch.bfloat16, f"d{n} recorded")
    gw, = torch.autograd.grad((ref * dO.double()).sum(), r[3], create_graph=True)
    want = torch.autograd.grad((gw ** 2).sum() * 0.01, r[:3])
    got = torch.autograd.grad((recorded[3].float() ** 2).sum() * 0.01, t[:3])
    for n, a, b in zip("qkv", got, want):
        assert_parity(a, b, torch.bfloat16, f"penalty d{n}")


@pytest.mark.parametrize("mode", [0, 1])
def test_packed_float32_at_any_offset(gpu_device, mode):
    """Contiguous float32 views one element into a buffer (4-byte boundary), upstream gradient too, give what
    aligned operands give; bf16 ones are refused, as the segments refuse them."""
    from memory_amd import sparse_attention as SA
    dev = gpu_device
    g = gen(60 + mode)
    B, Tq, HQ, HK, Tk, S = 2, 37, 4, 2, 320, 2
    q, dO = (torch.randn(B, Tq, HQ, 64, generator=g) for _ in range(2))
    k, v = (torch.randn(B, Tk, HK, 64, generator=g) for _ in range(2))
    idx = torch.rand(B, Tq, HK, 5, generator=g).argsort(-1)[..., :S].to(dev, torch.int32)
    w = torch.rand(B, Tq, S, generator=g).to(dev)

    def run(place, dtype=torch.float32):
        t = [place(x.to(dev, dtype)).requires_grad_() for x in (q, k, v)]
        if mode == 0:
            out = SA.FSA_topk_sparse_attention_weighted_bthd(*t, idx, w, 64, disable_causal_mask=True)
        else:
            out = SA.FSA_topk_sparse_attention_bthd(*t, idx, 64, disable_causal_mask=True)
        out.backward(place(dO.to(dev, dtype)))
        return [out.detach()] + [x.grad for x in t]

    def off(x):
        flat = torch.empty(x.numel() + 1, device=dev, dtype=x.dtype)
        flat[1:] = x.reshape(-1)
        return flat[1:].view(x.shape)

    for a, b in zip(run(off), run(lambda x: x)):
        assert torch.equal(a, b)
    with pytest.raises(ValueError, match="aligned"):
        run(off, torch.bfloat16)
