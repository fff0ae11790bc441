"""The one-call decode step, its routing and its rolling window against the separate entry points (equal
bits), and the single-workgroup chapter plan at the edges of its blocks of 1,024 edges."""

import numpy as np
import pytest
import torch

from helpers import gen

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("E,C", [(1023, 700), (1024, 33), (1025, 1), (2048, 8192), (2049, 300), (4095, 4097), (4096, 8),
                                 (4097, 50), (8191, 8192), (8192, 900), (8193, 60), (6144, 64), (6145, 64), (8192, 65)])
def test_small_plan(gpu_device, E, C):
    from memory_amd import ops
    ids = torch.randint(0, C, (E,), generator=gen(E + C), dtype=torch.int32)
    ids[::7] = -1
    ids[3::11] = C
    ids[E // 2:E // 2 + 40] = C // 2
    if E % 1024 != 1:
        ids[E // 3:E - 5:2] = C // 3      # one chapter with most of several blocks
    a = ids.numpy()
    ok = (a >= 0) & (a < C)
    uniq = np.unique(a[ok])
    want_u = np.where(ok, np.searchsorted(uniq, a), -1)
    order = np.array([e for e in np.argsort(a, kind="stable") if ok[e]], dtype=np.int64)
    p = ops.chapter_plan(ids.to(gpu_device), C)
    n = len(uniq)
    assert p.n_uniq.tolist() == [n, int((~ok).sum())]
    assert p.uniq[:n].tolist() == uniq.tolist() and p.edge_u.tolist() == want_u.tolist()
    assert p.csr_off[:n + 1].tolist() == np.concatenate([[0], np.cumsum(np.bincount(want_u[ok], minlength=n))]).tolist()
    assert p.csr_edge[:len(order)].tolist() == order.tolist()


@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("B,n_old,n_new,window,d,sliced", [(1, 1, 1, 1, 8, False), (2, 15, 1, 16, 768, True),
                                                           (3, 16, 1, 128, 256, False), (2, 128, 1, 128, 1032, True),
                                                           (2, 33, 40, 19, 64, True), (16, 127, 3, 128, 768, False)])
def test_window_pool(gpu_device, dtype, B, n_old, n_new, window, d, sliced):
    from memory_amd import ops
    from memory_amd.decode import DecodeRouter, _window_native
    dev = gpu_device
    g = gen(B + n_old + d)
    full = torch.randn(B, n_old + 5, d, generator=g).to(dev, dtype)
    old = full[:, 5:] if sliced else full[:, 5:].contiguous()
    h = torch.randn(B, n_new, d, generator=g).to(dev, dtype)
    assert _window_native(old, h)
    r = DecodeRouter(None, num_chapters=9, strategy="rolling", window_size=window)
    r.cache = old
    got = r._window(h, None)
    want = torch.cat([old, h], 1)[:, -window:]
    assert torch.equal(r.cache, want) and torch.equal(got, ops.router_pool(want))
    odd = torch.zeros(B, n_old, d + 1, device=dev, dtype=dtype)
    for o, x in ((odd[:, :, 1:], h), (odd, torch.zeros(B, 1, d + 1, device=dev, dtype=dtype)), (old.half(), h),
                 (old, h.transpose(1, 2))):
        assert not _window_native(o, x)


@pytest.mark.parametrize("B,d,H,HK,C,S,k,bias,wdt", [(1, 256, 4, 4, 33, 1, 3, True, BF), (16, 768, 12, 4, 700, 1, 64, True, BF),
                                                     (5, 128, 2, 1, 40, 4, 36, False, torch.float32),
                                                     (64, 256, 4, 2, 500, 1, 63, True, torch.float32)])
def test_step_equals_separate_calls(gpu_device, monkeypatch, B, d, H, HK, C, S, k, bias, wdt):
    from memory_amd import _lib as lib
    from memory_amd import decode
    from memory_amd.model import RoutedMemoryLayer
    dev = gpu_device
    g = gen(B + C)
    layer = RoutedMemoryLayer(d, H, C, 64, k, num_shared_chapters=S, num_kv_heads=HK, wo_init_zero=False)
    with torch.no_grad():
        for p in layer.parameters():
            p.copy_(torch.randn(p.shape, generator=g) * 0.05)
    layer = layer.to(dev, BF)
    layer.router.to(wdt)
    if not bias:
        layer.router.router.bias = None
    attn = layer.memory_attn
    bank = (torch.randn(C * 64, d, generator=g) * 0.3).to(dev, BF)
    cache = decode.MemoryDecodeCache(bank, attn.k_proj.weight, attn.v_proj.weight, num_chapters=C, tokens_per_chapter=64,
                                     num_kv_heads=HK)
    prompt = torch.randn(B, 20, d, generator=g).to(dev, BF)
    steps = [torch.randn(B, 1, d, generator=g).to(dev, BF) for _ in range(3)]
    runs = []
    for separate in (False, True):
        called = []
        real = lib.call
        monkeypatch.setattr(decode, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
        monkeypatch.setattr(lib, "KERNEL_EVENTS", {} if separate else None)
        r = decode.DecodeRouter(layer.router, num_chapters=C, num_shared_chapters=S, strategy="rolling", window_size=16)
        r.prefill(prompt)
        res = []
        for h in steps:
            routing = r.step(h)
            out = decode.memory_decode_step(attn, h, cache, routing)
            n = int(routing.plan.n_uniq[0])
            res.append((out, r.last_logits, routing.idx, routing.omega, routing.plan.uniq[:n], routing.plan.edge_u,
                        routing.plan.csr_off[:n + 1], routing.plan.csr_edge, routing.row_tab))
            assert routing.unique_chapters() == n and routing.max_units == min(B * (S + k), C)
        assert ("moc_decode_step" in called and "moc_decode_route" in called) != separate
        runs.append(res)
    for a, b in zip(*runs):
        for x, y in zip(a, b):
            assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y)


@pytest.mark.parametrize("n,B,H,HK,C,k,grouped", [(2, 1, 4, 4, 90, 64, True), (9, 3, 4, 2, 40, 8, True),
                                                  (3, 17, 12, 12, 120, 67, True), (2, 2, 4, 4, 40, 7, False),
                                                  (2, 2, 4, 4, 90, 68, False), (1, 2, 4, 4, 40, 20, False)])
def test_graph_groups_layers(gpu_device, monkeypatch, n, B, H, HK, C, k, grouped):
    """Layers of one shape captured as one launch per kernel: every replay equals the layers' own steps;
    other slot counts, single layers and layers of different shapes keep a chain each."""
    from memory_amd import decode
    from memory_amd.memory_attention import MemoryCrossAttention
    dev = gpu_device
    d = 64 * H
    g = gen(n * 100 + k)
    layers = []
    for i in range(n):
        attn = MemoryCrossAttention(d, H, HK, wo_init_zero=False).to(dev, BF)
        bank = torch.randn(C * 64, d, generator=g).to(dev, BF)
        cache = decode.MemoryDecodeCache(bank, attn.k_proj.weight, attn.v_proj.weight, num_chapters=C,
                                         tokens_per_chapter=64, num_kv_heads=HK)
        idx = torch.stack([torch.randperm(C, generator=g)[:k + 1] for _ in range(B)])
        if i == 1:
            idx[:] = idx[0]                 # one set of chapters for every sequence: fewer units
        w = torch.rand(B, k + 1, generator=g) + 0.1
        layers.append((attn, cache, decode.DecodeRouting(idx.to(dev), w.to(dev), C, sync=i != 0)))
    called = []
    real = decode.call
    monkeypatch.setattr(decode, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    xs = [torch.randn(B, 1, d, generator=g).to(dev, BF) for _ in range(n)]
    graph = decode.DecodeStepGraph(layers, xs)
    assert ("moc_decode_step_group" in called) == grouped
    for rep in range(3):
        inputs = [torch.randn(B, 1, d, generator=g).to(dev, BF) for _ in range(n)]
        outs = [o.clone() for o in graph.run(inputs)]
        junk = torch.randn(1000, device=dev).sum()
        torch.cuda.synchronize()
        for i, ((a, c, r), x) in enumerate(zip(layers, inputs)):
            assert torch.equal(outs[i], decode.memory_decode_step(a, x, c, r)), (rep, i)
        graph.static_in[0].copy_(inputs[-1])      # inputs written straight into the captured buffers
        outs = graph.run(graph.static_in)
        assert torch.equal(outs[0], decode.memory_decode_step(layers[0][0], inputs[-1], *layers[0][1:]))
    if grouped:
        other = MemoryCrossAttention(d, H, 1, wo_init_zero=False).to(dev, BF)
        cache = decode.MemoryDecodeCache(bank, other.k_proj.weight, other.v_proj.weight, num_chapters=C,
                                         tokens_per_chapter=64, num_kv_heads=1)
        assert not decode._group_native(layers + [(other, cache, layers[0][2])], xs + xs[:1])


def test_stream_ptr(gpu_device):
    from memory_amd._lib import stream_ptr
    side = torch.cuda.Stream()
    for st in (torch.cuda.current_stream(), side):
        with torch.cuda.stream(st):
            for dev in (None, torch.device("cuda"), torch.device("cuda", torch.cuda.current_device())):
                assert stream_ptr(dev) == st.cuda_stream
