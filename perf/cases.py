"""The framework's work in real use, as cases that can be timed and checked one by one.

Each kind of case is one public entry point, called as a user's program calls it:

  sequence   RoutedMemoryLayer: training step (forward, router losses where the recipe has them,
             backward) or the forward of a prompt
  token      TokenRoutedMemoryLayer: training step or the forward of a prompt
  sparse     the FSA entry points (top-k block-sparse attention), forward and backward
  sublayer   MemorySublayer over a dense memory: norm, cross-attention, residual; forward and backward
  decode     memory_decode_step through several layers, routing fixed by the prompt, called
             directly or replayed from a DecodeStepGraph
  reroute    DecodeRouter.step and memory_decode_step: the routing decided again at every token

Distributions: hidden states and upstream gradients N(0, 1), bank and weights N(0, 0.02), router
bias 0, routed scaling 2.5, one shared chapter of 64 rows.  Router weights hold values that bf16
represents, as a bf16-trained checkpoint does.
"""

import math
import random

import torch
import torch.nn.functional as F

T = 64          # rows of a chapter
SCALE = 2.5     # routed scaling factor
LB, ZL = 0.01, 0.001    # router loss coefficients of the training recipe


def listed():
    return [
        # one user's generation: four memory layers per token from one captured graph, batch 1;
        # the smallest call, launches and latency
        dict(name="decode_one", kind="decode", B=1, d=768, H=12, HK=12, C=4097, k=64, layers=4, graph=True),
        # a serving batch at the paper's bank: reads the selected chapters of 64 sequences
        dict(name="decode_batch", kind="decode", B=64, d=768, H=12, HK=12, C=4097, k=64, layers=4, graph=False),
        # generation with the rolling inference strategy: router, plan and decode at each token
        dict(name="decode_rolling", kind="reroute", B=16, d=768, H=12, HK=12, C=4097, k=64, window=128, prompt=512),
        # the prompt of one sequence through a memory layer (inference, batch 1, odd length)
        dict(name="prefill_prompt", kind="sequence", train=False, dtype="bf16", B=1, L=509, d=768, H=12, HK=12,
             C=4097, k=64, norm="none", rolling=0, losses=False),
        # the reference's small configuration in float32, trained: the whole step is small launches
        dict(name="train_small_f32", kind="sequence", train=True, dtype="f32", B=2, L=128, d=256, H=4, HK=4,
             C=33, k=4, norm="none", rolling=0, losses=False),
        # the headline: the paper's layer, a training step of 8 x 1,024 tokens
        dict(name="train_sequence", kind="sequence", train=True, dtype="bf16", B=8, L=1024, d=768, H=12, HK=12,
             C=4097, k=64, norm="none", rolling=0, losses=False),
        # the paper's recipe: rows normalised before mixing and the router losses, ragged length
        dict(name="train_recipe", kind="sequence", train=True, dtype="bf16", B=8, L=1000, d=768, H=12, HK=12,
             C=4097, k=64, norm="rms", rolling=0, losses=True),
        # per-token routing, trained: every chapter of the bank projected (the largest)
        dict(name="train_token", kind="token", train=True, B=4, L=2048, d=768, H=12, HK=12, C=4097, k=16,
             version="v4", weighted=True, losses=False),
        # per-token routing of one short prompt (inference)
        dict(name="prefill_token", kind="token", train=False, B=1, L=301, d=768, H=12, HK=12, C=4097, k=16,
             version="v4", weighted=True, losses=False),
        # the sparse-attention kernels on their own at the published harness' head layout:
        # 16 query heads on one kv head, blocks of 128, top-8 of 65,536 keys
        dict(name="sparse_mqa", kind="sparse", entry="joint", dtype="bf16", B=2, Tq=8192, Tk=65536, HQ=16, HK=1,
             block=128, S=8),
        # grouped kv heads that choose their blocks separately, per-block weights, a ragged length
        dict(name="sparse_gqa", kind="sparse", entry="moe", dtype="bf16", B=2, Tq=1500, Tk=8192, HQ=16, HK=4,
             block=64, S=8),
        # a block's memory sublayer over a dense learned memory (no routing), grouped kv heads
        dict(name="sublayer_dense", kind="sublayer", dtype="bf16", B=4, L=1024, N=4096, d=1024, H=16, HK=4,
             rms=True, batched=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["sequence", "sequence", "sequence", "token", "sparse", "sparse", "sublayer", "decode", "reroute"])
    d, H, HK = rng.choice([(768, 12, 12), (768, 12, 12), (768, 12, 4), (512, 8, 8), (1024, 16, 4), (256, 4, 4),
                           (256, 4, 2)])
    C = _log(rng, 33, 4097)
    k = min(_log(rng, 4, 64), C - 1)
    if kind == "sequence":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        train = rng.random() < 0.7
        if dtype == "f32":      # float32 is the reference's small parity setting
            return dict(kind=kind, train=train, dtype=dtype, B=rng.randint(1, 3), L=_log(rng, 16, 256), d=256, H=4,
                        HK=rng.choice([4, 2]), C=min(C, 257), k=min(k, 16, min(C, 257) - 1),
                        norm=rng.choice(["none", "rms"]), rolling=0, losses=False)
        return dict(kind=kind, train=train, dtype=dtype, B=rng.randint(1, 8), L=_log(rng, 24, 1024), d=d, H=H, HK=HK,
                    C=C, k=k, norm=rng.choice(["none", "rms", "rms", "layernorm"]), rolling=rng.choice([0, 0, 128]),
                    losses=train and rng.random() < 0.5)
    if kind == "token":
        version, weighted = rng.choice([("v4", True), ("v4", True), ("v5", True), ("v2", False)])
        train = rng.random() < 0.6
        return dict(kind=kind, train=train, B=rng.randint(1, 4), L=_log(rng, 40, 2048), d=d, H=H, HK=HK, C=C,
                    k=min(k, 16), version=version, weighted=weighted, losses=train and rng.random() < 0.5)
    if kind == "sparse":
        HQ, HKs = rng.choice([(16, 1), (16, 4), (8, 1), (12, 12), (8, 2)])
        block = rng.choice([64, 64, 128])
        entry = rng.choice(["joint", "joint", "moe", "bias", "block"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        Tq = _log(rng, 48, 512 if dtype == "f32" else 1024 if entry == "moe" and block > 64 else 8192)
        Tk = block * _log(rng, 32, 16384 // block)
        S = rng.randint(2, 8)
        if HKs * Tq > 16384:
            Tq = 16384 // HKs
        return dict(kind=kind, entry=entry, dtype=dtype, B=rng.randint(1, 2), Tq=Tq, Tk=Tk, HQ=HQ, HK=HKs, block=block,
                    S=S)
    if kind == "sublayer":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        if dtype == "f32":
            return dict(kind=kind, dtype=dtype, B=rng.randint(1, 2), L=_log(rng, 16, 200), N=64 * rng.randint(1, 12),
                        d=256, H=4, HK=rng.choice([4, 2]), rms=rng.random() < 0.5, batched=rng.random() < 0.5)
        return dict(kind=kind, dtype=dtype, B=rng.randint(1, 4), L=_log(rng, 16, 1024), N=64 * _log(rng, 2, 64), d=d,
                    H=H, HK=HK, rms=rng.random() < 0.7, batched=rng.random() < 0.3)
    if kind == "decode":
        return dict(kind=kind, B=_log(rng, 1, 64), d=d, H=H, HK=HK, C=C, k=k, layers=rng.choice([1, 2, 4]),
                    graph=rng.random() < 0.5)
    return dict(kind=kind, B=_log(rng, 1, 64), d=d, H=H, HK=HK, C=C, k=k, window=rng.choice([32, 128]),
                prompt=_log(rng, 16, 512))


# --------------------------------------------------------------------------------- inputs

def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _dtype(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.bfloat16


def _inputs(case, seed):
    """Every tensor of a case, from the seed alone."""
    dev, dt = _device(), _dtype(case)
    g = torch.Generator(device=dev).manual_seed(int(seed))

    def normal(*shape, std=1.0, dtype=dt):
        return torch.randn(*shape, device=dev, generator=g).mul_(std).to(dtype)

    kind = case["kind"]
    x = {}
    if kind == "sparse":
        B, Tq, Tk, HQ, HK, S = (case[n] for n in ("B", "Tq", "Tk", "HQ", "HK", "S"))
        M = Tk // case["block"]
        x["q"], x["k"], x["v"] = normal(B, Tq, HQ, 64), normal(B, Tk, HK, 64), normal(B, Tk, HK, 64)
        x["idx"] = torch.rand(B, Tq, HK, M, device=dev, generator=g).topk(S, dim=-1).indices.to(torch.int32)
        if case["entry"] == "block":
            x["w"] = torch.rand(B, Tq, HK, S, device=dev, generator=g) + 0.05
        elif case["entry"] in ("moe", "bias"):
            x["w"] = torch.softmax(torch.randn(B, Tq, S, device=dev, generator=g), -1)
        x["dout"] = normal(B, Tq, HQ, 64)
        return x
    d, H, HK = case["d"], case["H"], case["HK"]
    KV = HK * 64
    nlayers = case.get("layers", 1)
    x["layers"] = []
    for _ in range(nlayers):
        w = {"wq": normal(d, d, std=0.02), "wk": normal(KV, d, std=0.02), "wv": normal(KV, d, std=0.02),
             "wo": normal(d, d, std=0.02)}
        if kind != "sublayer":
            w["wr"] = normal(case["C"], d, std=0.02, dtype=torch.bfloat16).float()
        x["layers"].append(w)
    if kind == "sublayer":
        B, L, N = case["B"], case["L"], case["N"]
        x["h"] = normal(B, L, d)
        x["mem"] = normal(B, N, d) if case["batched"] else normal(N, d)
        x["g"] = (1 + 0.1 * torch.randn(d, device=dev, generator=g)).to(dt)
        x["b"] = None if case["rms"] else normal(d, std=0.1)
        x["dout"] = normal(B, L, d)
        return x
    x["bank"] = normal(case["C"] * T, d, std=0.02)
    if kind in ("sequence", "token"):
        x["h"] = normal(case["B"], case["L"], d)
        if case["train"]:
            x["dout"] = normal(case["B"], case["L"], d)
    else:
        x["prompt"] = normal(case["B"], case.get("prompt", 256), d)
        x["h"] = [normal(case["B"], 1, d) for _ in range(nlayers)]
    return x


# ------------------------------------------------------------------------ the user's program

def _load(attn, w):
    with torch.no_grad():
        for name in ("q", "k", "v", "o"):
            lin = getattr(attn, name + "_proj")
            lin.to(w["w" + name].dtype)
            lin.weight.copy_(w["w" + name])


def _layer(case, w):
    from memory_amd.model import RoutedMemoryLayer, TokenRoutedMemoryLayer
    C, k, norm = case["C"], case["k"], case.get("norm", "none")
    kw = dict(num_shared_chapters=1, routed_scaling_factor=SCALE, num_kv_heads=case["HK"], wo_init_zero=False,
              normalize_shared_routed_before_mixing=norm != "none",
              shared_routed_norm_type=norm if norm != "none" else "rms")
    if case["kind"] == "token":
        layer = TokenRoutedMemoryLayer(case["d"], case["H"], C, T, k, weighted=case["weighted"],
                                       kernel_version=case["version"], **kw)
    else:
        roll = case.get("rolling", 0)
        layer = RoutedMemoryLayer(case["d"], case["H"], C, T, k,
                                  routing_strategy="sequence-rolling" if roll else "sequence",
                                  routing_window_size=roll or None, **kw)
    layer = layer.to(_device())
    _load(layer.memory_attn, w)
    with torch.no_grad():
        layer.router.router.weight.copy_(w["wr"])
        layer.router.router.bias.zero_()
    return layer


def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "sparse":
        for n in ("q", "k", "v", "w"):
            s[n] = x[n].requires_grad_(True) if n in x else None
        s["idx"], s["dout"] = x["idx"], x["dout"]
        return s
    if kind == "sublayer":
        from memory_amd.memory_block import MemorySublayer
        sub = MemorySublayer(case["d"], case["H"], case["HK"], use_rms_norm=case["rms"], norm_eps=1e-5,
                             wo_init_zero=False).to(_device(), _dtype(case))
        _load(sub.memory_attn, x["layers"][0])
        with torch.no_grad():
            sub.memory_layernorm.weight.copy_(x["g"])
            if x["b"] is not None:
                sub.memory_layernorm.bias.copy_(x["b"])
        s.update(layer=sub, h=x["h"].requires_grad_(True), mem=x["mem"].requires_grad_(True), dout=x["dout"])
        return s
    if kind in ("sequence", "token"):
        s.update(layer=_layer(case, x["layers"][0]), h=x["h"], bank=x["bank"])
        if case["train"]:
            s["h"].requires_grad_(True)
            s["bank"].requires_grad_(True)
            s["dout"] = x["dout"]
        return s
    from memory_amd.decode import DecodeRouter, DecodeRouting, DecodeStepGraph, MemoryDecodeCache
    s["h"], s["layers"] = x["h"], []
    with torch.no_grad():
        for w in x["layers"]:
            layer = _layer(case, w)
            attn = layer.memory_attn
            cache = MemoryDecodeCache(x["bank"], attn.k_proj.weight, attn.v_proj.weight, num_chapters=case["C"],
                                      tokens_per_chapter=T, num_kv_heads=case["HK"])
            if kind == "reroute":
                router = DecodeRouter(layer.router, num_chapters=case["C"], num_shared_chapters=1,
                                      routed_scaling_factor=SCALE, strategy="rolling", window_size=case["window"])
                router.prefill(x["prompt"])
                s.update(attn=attn, cache=cache, router=router)
            else:
                idx, omega, _ = layer.route(x["prompt"], return_losses=False)
                s["layers"].append((attn, cache, DecodeRouting(idx, omega, case["C"])))
        if case.get("graph"):
            s["graph"] = DecodeStepGraph(s["layers"], s["h"])
    return s


def _gradients(leaves):
    return [t.grad for t in leaves]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        from memory_amd.decode import memory_decode_step
        if "graph" in s:
            return s["graph"].run(s["h"])
        return [memory_decode_step(attn, h, cache, routing) for (attn, cache, routing), h in zip(s["layers"], s["h"])]
    if kind == "reroute":
        from memory_amd.decode import memory_decode_step
        routing = s["router"].step(s["h"][0])
        return {"out": memory_decode_step(s["attn"], s["h"][0], s["cache"], routing), "logits": s["router"].last_logits}
    if kind == "sparse":
        from memory_amd import sparse_attention as sa
        leaves = [s[n] for n in ("q", "k", "v", "w") if s[n] is not None]
        for t in leaves:
            t.grad = None
        kw = dict(disable_causal_mask=True)
        if case["entry"] == "moe":
            out = sa.FSA_topk_sparse_attention_weighted_bthd(s["q"], s["k"], s["v"], s["idx"], s["w"], case["block"], **kw)
        elif case["entry"] == "bias":
            out = sa.FSA_topk_sparse_attention_weighted_joint_bias_bthd(s["q"], s["k"], s["v"], s["idx"], s["w"],
                                                                        case["block"], **kw)
        else:
            out = sa.FSA_topk_sparse_attention_bthd(s["q"], s["k"], s["v"], s["idx"], case["block"],
                                                    block_weights_bths=s["w"], **kw)
        out.backward(s["dout"])
        return {"out": out.detach(), "grads": _gradients(leaves)}
    layer = s["layer"]
    if kind == "sublayer":
        params = list(layer.parameters())
        leaves = [s["h"], s["mem"]] + params
        for t in leaves:
            t.grad = None
        out = layer(s["h"], s["mem"])
        out.backward(s["dout"])
        return {"out": out.detach(), "grads": _gradients(leaves)}
    if not case["train"]:
        with torch.no_grad():
            return layer(s["h"], s["bank"], return_losses=False)[0]
    leaves = [s["h"], s["bank"]] + list(layer.parameters())
    for t in leaves:
        t.grad = None
    out, losses = layer(s["h"], s["bank"], return_losses=case["losses"])
    if case["losses"]:
        from memory_amd.router import compute_total_router_loss
        total = compute_total_router_loss(losses, LB, 0.0, ZL)
        torch.autograd.backward([out, total], [s["dout"], None])
        return {"out": out.detach(), "loss": total.detach(), "grads": _gradients(leaves)}
    out.backward(s["dout"])
    return {"out": out.detach(), "grads": _gradients(leaves)}


# ------------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    e = 4 if case.get("dtype") == "f32" else 2
    if kind == "sparse":
        B, Tq, Tk, HQ, HK, S = (case[n] for n in ("B", "Tq", "Tk", "HQ", "HK", "S"))
        flops = 3 * 4 * B * Tq * HQ * S * case["block"] * 64
        used = min(Tk, Tq * S * case["block"])
        nbytes = B * (Tq * HQ * 64 * 4 * e + (used * 2 + Tk * 2) * HK * 64 * e + Tq * HK * S * 4)
        return {"bytes": nbytes, "flops": flops}
    d, H, HK, B = case["d"], case["H"], case["HK"], case["B"]
    KV = HK * 64
    weights = (2 * d * d + 2 * KV * d) * e
    if kind == "sublayer":
        L, N = case["L"], case["N"]
        nb = B if case["batched"] else 1
        fwd = 4 * B * L * d * d + 4 * nb * N * d * KV + 4 * B * L * H * N * 64
        return {"bytes": (B * L * d * 4 + 2 * nb * N * d) * e + 2 * weights, "flops": 3 * fwd}
    C, k = case["C"], case["k"]
    Cr = C - 1
    if kind in ("decode", "reroute"):
        unique = 1 + Cr * (1 - (1 - k / Cr) ** B)
        nbytes = case.get("layers", 1) * (unique * T * 2 * KV * 2 + 2 * d * d * 2 + 2 * B * d * 2)
        flops = case.get("layers", 1) * (4 * B * d * d + 4 * B * H * (k + 1) * T * 64)
        if kind == "reroute":
            nbytes += C * d * 4 + B * case["window"] * d * 2 + B * C * 4
            flops += 2 * B * C * d
        return {"bytes": nbytes, "flops": flops}
    L = case["L"]
    ntok = B * L
    if kind == "sequence":
        unique = 1 + Cr * (1 - (1 - k / Cr) ** B)
        fwd = 4 * ntok * d * d + 4 * unique * T * d * KV + 4 * ntok * H * (k + 1) * T * 64 + 2 * B * C * d
        router = C * d * 4
    else:
        unique = 1 + Cr * (1 - (1 - k / Cr) ** ntok)
        fwd = 4 * ntok * d * d + 4 * unique * T * d * KV + 4 * ntok * H * (k + 1) * T * 64 + 2 * ntok * C * d
        router = C * d * 4
    nbytes = 2 * ntok * d * e + unique * T * d * e + weights + router
    if case["train"]:
        return {"bytes": nbytes + 2 * ntok * d * e + C * T * d * e + weights + router, "flops": 3 * fwd}
    return {"bytes": nbytes, "flops": fwd}


def tolerance(case):
    # about four times the distance from the 64-bit results: float32 up to 2e-6, bf16 (one rounding
    # of each intermediate to 8 bits) up to 5e-3.  Per-token routing over thousands of tokens holds
    # a near-tie now and then: one token's other choice moves single values by their own size.
    if case.get("dtype") == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 0.02, "max": 0.99 if case["kind"] == "token" else 0.3}


# ----------------------------------------------------------------------- the same in 64 bits

def _route(logits, k):
    """(chapter ids, weights) of the router: softmax, shared prefix masked, top-k, renormalised."""
    p = torch.softmax(logits, -1).clone()
    mask = torch.ones_like(p)
    mask[..., 0] = 0
    p = p * mask
    p = p / p.sum(-1, keepdim=True).clamp_min(1e-12)
    z = logits.detach().clone()
    z[..., 0] = -math.inf
    idx = torch.sort(z, dim=-1, descending=True, stable=True)[1][..., :k]
    w = torch.gather(p, -1, idx)
    return idx, w / w.sum(-1, keepdim=True).clamp_min(1e-12)


def _prepend(idx, w):
    B = idx.shape[0]
    idx = torch.cat([idx.new_zeros(B, 1), idx], -1)
    w = torch.cat([w.new_ones(B, 1), w * SCALE], -1)
    return idx, w / w.sum(-1, keepdim=True).clamp_min(1e-12)


def _losses(logits, idx):
    C = logits.shape[-1]
    p = torch.softmax(logits, -1)
    f = torch.zeros(C, device=p.device, dtype=p.dtype)
    f.index_add_(0, idx.reshape(-1), torch.ones(idx.numel(), device=p.device, dtype=p.dtype))
    f = f / p.shape[0]
    return LB * C * (f * p.mean(0)).sum() + ZL * (torch.logsumexp(logits, -1) ** 2).mean()


def _row_norm(m, norm, eps=1e-6):
    if norm == "rms":
        return m / m.pow(2).mean(-1, keepdim=True).add(eps).sqrt()
    if norm == "layernorm":
        return F.layer_norm(m, (m.shape[-1],), eps=eps)
    return m


def _attend(q, keys, values, H):
    """softmax(q k^T / 8) v: q (L, H * 64), keys and values (N, HK * 64)."""
    L, N = q.shape[0], keys.shape[0]
    HK = keys.shape[1] // 64
    qh = q.view(L, HK, H // HK, 64).permute(1, 2, 0, 3).reshape(HK, -1, 64)
    kh = keys.view(N, HK, 64).permute(1, 2, 0).contiguous()
    vh = values.view(N, HK, 64).permute(1, 0, 2).contiguous()
    p = torch.softmax(torch.matmul(qh, kh) * 0.125, -1)
    return torch.matmul(p, vh).view(HK, H // HK, L, 64).permute(2, 0, 1, 3).reshape(L, H * 64)


def _leaf(t, train=True):
    return t.detach().double().requires_grad_(train)


def _exact_sequence(case, x):
    train = case["train"]
    h, bank = _leaf(x["h"], train), _leaf(x["bank"], train)
    w = {n: _leaf(t, train) for n, t in x["layers"][0].items()}
    br = torch.zeros(case["C"], device=h.device, dtype=torch.float64, requires_grad=train)
    B, L, d = h.shape
    if case["rolling"]:
        win = min(case["rolling"], L)
        cs = torch.cat([h.new_zeros(B, 1, d), h.cumsum(1)], 1)
        end = torch.arange(L, device=h.device) + 1
        start = (end - win).clamp_min(0)
        pooled = ((cs[:, end] - cs[:, start]) / (end - start).view(1, L, 1)).mean(1)
    else:
        pooled = h.mean(1)
    logits = pooled @ w["wr"].t() + br
    idx, wt = _route(logits, case["k"])
    ids, omega = _prepend(idx, wt)
    rows = (ids.unsqueeze(-1) * T + torch.arange(T, device=h.device)).reshape(-1)
    mem = _row_norm(bank.index_select(0, rows), case["norm"]).view(B, -1, d)
    mem = mem * omega.repeat_interleave(T, -1).unsqueeze(-1)
    outs = []
    for b in range(B):
        a = _attend(h[b] @ w["wq"].t(), mem[b] @ w["wk"].t(), mem[b] @ w["wv"].t(), case["H"])
        outs.append(a @ w["wo"].t())
    out = torch.stack(outs)
    return out, (_losses(logits, idx) if case["losses"] else None), [h, bank, w["wr"], br, w["wq"], w["wk"], w["wv"],
                                                                      w["wo"]]


def _blocks(q, keys, values, ids, wt, entry, HK, chunk_bytes=1 << 29):
    """Sparse attention in 64 bits over blocks keys / values [blocks][bs][HK * 64], ids (n, HK, S) block ids,
    wt (n, HK, S) or None; yields (first token, output (c, H * 64)) per chunk of tokens, for one backward each."""
    n, H = q.shape[0], q.shape[1] // 64
    bs, S = keys.shape[1], ids.shape[-1]
    kb = keys.view(-1, bs, HK, 64)
    vb = values.view(-1, bs, HK, 64)
    heads = torch.arange(HK, device=q.device).view(1, HK, 1)
    step = max(1, chunk_bytes // (HK * S * bs * 64 * 8))
    kp = kb.permute(0, 2, 1, 3)
    vp = vb.permute(0, 2, 1, 3)
    for at in range(0, n, step):
        i = ids[at:at + step]
        c = i.shape[0]
        kk = kp[i, heads].reshape(c, HK, S * bs, 64)
        vv = vp[i, heads].reshape(c, HK, S * bs, 64)
        qq = q[at:at + step].view(c, HK, H // HK, 64)
        s = torch.matmul(qq, kk.transpose(-1, -2).contiguous()) * 0.125
        g = H // HK
        if entry == "moe":
            p = torch.softmax(s.view(c, HK, g, S, bs), -1) * wt[at:at + step].view(c, HK, 1, S, 1)
            p = p.reshape(c, HK, g, S * bs)
        elif entry in ("bias", "block"):
            b = torch.log(wt[at:at + step].clamp_min(1e-20)).view(c, HK, 1, S, 1)
            p = torch.softmax((s.view(c, HK, g, S, bs) + b).reshape(c, HK, g, S * bs), -1)
        else:
            p = torch.softmax(s, -1)
        yield at, torch.matmul(p, vv).reshape(c, H * 64)


def _sparse_backward(q, keys, values, ids, wt, entry, HK, dout):
    """(out, grads of q, keys, values, wt) by chunks, each with its own backward."""
    cut = [t.detach().requires_grad_(True) for t in (q, keys, values)]
    wl = None if wt is None else wt.detach().requires_grad_(True)
    outs = []
    for at, o in _blocks(*cut, ids, wl, entry, HK):
        if dout is not None:
            o.backward(dout[at:at + o.shape[0]])
        outs.append(o.detach())
    return torch.cat(outs), [t.grad for t in cut] + [None if wl is None else wl.grad]


def _exact_token(case, x):
    train = case["train"]
    h, bank = _leaf(x["h"], train), _leaf(x["bank"], train)
    w = {n: _leaf(t, train) for n, t in x["layers"][0].items()}
    br = torch.zeros(case["C"], device=h.device, dtype=torch.float64, requires_grad=train)
    B, L, d = h.shape
    h2 = h.reshape(B * L, d)
    logits = h2 @ w["wr"].t() + br
    idx, wt = _route(logits, case["k"])
    q = h2 @ w["wq"].t()
    keys, values = bank[T:] @ w["wk"].t(), bank[T:] @ w["wv"].t()
    shared = _attend(q, bank[:T] @ w["wk"].t(), bank[:T] @ w["wv"].t(), case["H"])
    entry = "joint" if not case["weighted"] else "bias" if case["version"] == "v5" else "moe"
    HK = case["HK"]
    ids = (idx - 1).unsqueeze(1).expand(-1, HK, -1)
    wh = None if entry == "joint" else wt.unsqueeze(1).expand(-1, HK, -1)
    kb, vb = keys.view(-1, T, HK * 64), values.view(-1, T, HK * 64)
    d_pre = None
    if train:
        d_pre = (x["dout"].double().reshape(B * L, d) @ w["wo"]).detach()
    with torch.set_grad_enabled(train):
        routed, grads = _sparse_backward(q, kb, vb, ids, wh, entry, HK, None if d_pre is None else d_pre * SCALE)
    pre = shared + routed * SCALE
    out = (pre.detach() @ w["wo"].t()).view(B, L, d)
    if not train:
        return out
    # one backward through the outer graph: o_proj, the shared chapter, and the sparse part's gradients
    tensors, gs = [out, shared, q, kb, vb], [x["dout"].double(), d_pre, grads[0], grads[1], grads[2]]
    if wh is not None:
        tensors.append(wh)
        gs.append(grads[3])
    loss = None
    if case["losses"]:
        loss = _losses(logits, idx)
        tensors.append(loss)
        gs.append(None)
    torch.autograd.backward(tensors, gs)
    leaves = [h, bank, w["wr"], br, w["wq"], w["wk"], w["wv"], w["wo"]]
    for t in leaves:        # joint attention does not use the router's weights
        if t.grad is None:
            t.grad = torch.zeros_like(t)
    return out, loss, leaves


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "sparse":
        B, Tq, HQ, _ = x["q"].shape
        HK, bs, M = case["HK"], case["block"], case["Tk"] // case["block"]
        q = x["q"].double().reshape(B * Tq, HQ * 64)
        kb, vb = (x[n].double().reshape(B * M, bs, HK * 64) for n in ("k", "v"))
        ids = (x["idx"].long() + (torch.arange(B, device=q.device) * M).view(B, 1, 1, 1)).reshape(B * Tq, HK, -1)
        wt = None
        if "w" in x:
            wt = x["w"].double()
            wt = (wt if wt.dim() == 4 else wt.unsqueeze(2).expand(-1, -1, HK, -1)).reshape(B * Tq, HK, -1)
        out, g = _sparse_backward(q, kb, vb, ids, wt, case["entry"], HK, x["dout"].double().reshape(B * Tq, HQ * 64))
        grads = [g[0].view(x["q"].shape), g[1].view(x["k"].shape), g[2].view(x["v"].shape)]
        if wt is not None:
            gw = g[3].view(B, Tq, HK, -1)
            grads.append(gw if x["w"].dim() == 4 else gw.sum(2))
        return {"out": out.view(x["q"].shape), "grads": grads}
    if kind == "sublayer":
        h, mem, gam = _leaf(x["h"]), _leaf(x["mem"]), _leaf(x["g"])
        bet = None if x["b"] is None else _leaf(x["b"])
        w = {n: _leaf(t) for n, t in x["layers"][0].items()}
        d = case["d"]
        if case["rms"]:
            xn = h / h.pow(2).mean(-1, keepdim=True).add(1e-5).sqrt() * gam
        else:
            xn = F.layer_norm(h, (d,), gam, bet, 1e-5)
        outs = []
        for b in range(case["B"]):
            m = mem[b] if case["batched"] else mem
            a = _attend(xn[b] @ w["wq"].t(), m @ w["wk"].t(), m @ w["wv"].t(), case["H"])
            outs.append(h[b] + a @ w["wo"].t())
        out = torch.stack(outs)
        out.backward(x["dout"].double())
        leaves = [h, mem, gam] + ([] if bet is None else [bet]) + [w["wq"], w["wk"], w["wv"], w["wo"]]
        return {"out": out.detach(), "grads": [t.grad for t in leaves]}
    if kind in ("sequence", "token"):
        if not case["train"]:
            with torch.no_grad():
                return _exact_token(case, x) if kind == "token" else _exact_sequence(case, x)[0]
        out, loss, leaves = (_exact_token if kind == "token" else _exact_sequence)(case, x)
        if kind == "sequence":
            torch.autograd.backward([out] + ([] if loss is None else [loss]),
                                    [x["dout"].double()] + ([] if loss is None else [None]))
        # token routing's own weights' gradient is computed from bf16 logit gradients; compared as it is
        r = {"out": out.detach(), "grads": [t.grad for t in leaves]}
        if loss is not None:
            r["loss"] = loss.detach()
        return r
    outs = []
    bank = x["bank"].double()
    for w, h in zip(x["layers"], x["h"]):
        w = {n: t.double() for n, t in w.items()}
        pooled = x["prompt"].double()
        if kind == "reroute":
            pooled = torch.cat([pooled[:, -case["window"]:], h.double()], 1)[:, -case["window"]:]
        logits = pooled.mean(1) @ w["wr"].t()
        ids, omega = _prepend(*_route(logits, case["k"]))
        q = h.double()[:, 0] @ w["wq"].t()
        pre = []
        for b in range(case["B"]):
            rows = (ids[b].unsqueeze(-1) * T + torch.arange(T, device=bank.device)).reshape(-1)
            m = bank[rows] * omega[b].repeat_interleave(T).unsqueeze(-1)
            pre.append(_attend(q[b:b + 1], m @ w["wk"].t(), m @ w["wv"].t(), case["H"]))
        outs.append((torch.cat(pre) @ w["wo"].t()).unsqueeze(1))
    return {"out": outs[0], "logits": logits} if kind == "reroute" else outs
