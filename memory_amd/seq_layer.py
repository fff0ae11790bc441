"""The sequence-routed memory layer as one autograd function with a stream-scheduled backward.

Reference chain (one memory layer of MemoryTransformer.forward, memory_transformer/model.py:609-692,
and the sublayer call memory_block.py:549-558 without the caller-owned norm and residual):
mean-pool -> router linear -> softmax / top-k (router.py:96-149) -> shared-chapter prepend
(model.py:356-391) -> gather x omega -> k_proj / v_proj -> attention -> o_proj
(memory_attention.py:241-243, :269-478).

The same kernels as the per-op autograd functions of ``ops``, scheduled as one unit:

forward    main stream: pool -> router linear -> top-k + prepend (one launch) -> chapter plan ->
           K/V projection -> attention -> o_proj;
           aux stream, beside the router chain (which is latency-bound: a few workgroups per
           launch): the q projection and the [Wk; Wv] pack, which do not depend on the routing.
backward   main stream: o_proj dX -> attention backward (dQ, then dK/dV) -> K/V weight gradient ->
           dX of the projection into the bank rows;
           aux stream: o_proj dW beside the o_proj dX and the dQ kernel; after dQ the q projection's
           dX and dW beside the dK/dV kernel; after dK/dV the router's backward (d omega partials ->
           dlogits -> router linear backward) and the pooling's gradient added into dh, beside
           the K/V chapter GEMMs.  The main stream waits for the aux stream before returning.

Every tensor the aux stream writes and the caller sees is allocated on the main stream before
the fork, so the caching allocator never hands its memory to another stream early.

For a bf16 bank, row-normalised or not (no BankAdamW mirror, no row-sparse gradient), the same
schedule runs natively: moc_seq_layer_fwd_ex / moc_seq_layer_bwd_ex issue every launch, event and stream
wait from C++ (the q / o projections on the chapter GEMM, their transposed weights packed in the
forward), so a training step costs two host calls; PyTorch only allocates the outputs, one saved
buffer and one scratch buffer.  A forward that no backward follows (grad mode off, or no input that
requires a gradient) leaves out what only the backward reads, and its buffer is a temporary.
``NATIVE = False`` keeps the Python-scheduled sequence.

The float32 layer at the reference's small sizes runs as one host call each way on one stream
(moc_seq_layer_f32_fwd / _bwd): its launches take a few microseconds each and the step is what the
host needs to issue them.  Training steps that reduce over many tokens or bank rows, and backwards that
are themselves recorded, go through the per-op functions.
"""

from __future__ import annotations

import ctypes
import functools
from typing import Optional

import torch
import torch.nn.functional as F

from . import _lib as L
from . import ops
from ._lib import call, ptr, stream_ptr


def supported(h: torch.Tensor, bank: torch.Tensor, wq: torch.Tensor, wo: torch.Tensor, wr: torch.Tensor,
              num_shared: int, top_k: int, num_chapters: int, T: int) -> bool:
    """Whether the fused layer handles this configuration (otherwise the per-op path runs)."""
    d = h.shape[-1]
    return (h.is_cuda and h.dim() == 3 and h.dtype == torch.bfloat16 and wq.dtype == torch.bfloat16
            and wo.dtype == torch.bfloat16 and wr.dtype in (torch.float32, torch.bfloat16) and d % 8 == 0
            and 0 < num_shared <= 1024 and 0 < top_k <= 1024 and top_k <= num_chapters - num_shared
            and num_chapters <= 8192 and h.shape[0] <= 64 and T == 64 and h.shape[1] > 0)


NATIVE = True


@functools.lru_cache(maxsize=256)
def _layer_sizes(B, Lq, d, H, HK, C, S, k, norm):
    """(saved, scratch, inference) buffer bytes of the native layer, or None for shapes outside it."""
    n = (ctypes.c_size_t * 3)()
    at = [ctypes.addressof(n) + i * ctypes.sizeof(ctypes.c_size_t) for i in range(3)]
    return tuple(n) if L.query("moc_seq_layer_sizes", B, Lq, d, H, HK, C, S, k, norm, *at) == L.MOC_OK else None


def _native_sizes(h, bank, br, wq, wk, wv, wo, cfg):
    """_layer_sizes of a call that moc_seq_layer_fwd_ex / _bwd_ex take, or None (such calls run as the
    Python-scheduled sequence below)."""
    if not NATIVE:
        return None
    C, T, S, k, scale, H, HK, norm, eps, _train = cfg
    B, Lq, d = h.shape
    bf = torch.bfloat16
    if (bank.dtype != bf or bank.dim() != 2 or bank.shape[1] != d or T != 64 or d != 64 * H or d > 4096
            or wq.dtype != bf or wk.dtype != bf or wv.dtype != bf or wo.dtype != bf
            or (norm != L.MOC_NORM_NONE and bank.data_ptr() % 16)     # rows read in 16-byte pieces
            or getattr(bank, "_moc_bank_opt", None) is not None or getattr(bank, "_moc_row_grad", None) is not None
            or (br is not None and br.dtype not in (torch.float32, bf))):
        return None
    return _layer_sizes(B, Lq, d, H, HK, C, S, k, norm)


class _SeqRoutedLayer(torch.autograd.Function):
    @staticmethod
    def forward(ctx, h, bank, wr, br, wq, wk, wv, wo, coef, cfg):
        C, T, S, k, scale, H, HK, norm, eps, train = cfg
        dev = h.device
        B, Lq, d = h.shape
        Dh = d // H
        KV = HK * Dh
        NS = S + k
        h = h.contiguous()
        ctx.cfg = cfg
        ctx.wdt = (wr.dtype, None if br is None else br.dtype)
        ctx.set_materialize_grads(False)
        sizes = _native_sizes(h, bank, br, wq, wk, wv, wo, cfg)
        ctx.native = sizes is not None
        if ctx.native:
            # the whole forward in one host call (moc_seq_layer_fwd_ex); without a backward to come
            # `saved` is a temporary
            nbytes = sizes[0] if train else sizes[2]
            main = torch.cuda.current_stream(dev)
            aux = ops._side_stream(dev, "aux")
            wrc = wr.contiguous()
            brc = None if br is None else br.float().contiguous()
            cf = None if coef is None else coef.to(device=dev, dtype=torch.float32).contiguous()
            saved = torch.empty(nbytes, device=dev, dtype=torch.uint8)
            out = torch.empty(B, Lq, d, device=dev, dtype=h.dtype)
            logits = torch.empty(B, C, device=dev, dtype=torch.float32)
            idx = torch.empty(B, k, device=dev, dtype=torch.int32)
            idx_star = torch.empty(B, NS, device=dev, dtype=torch.int32)
            omega = torch.empty(B, NS, device=dev, dtype=torch.float32)
            wq, wk, wv, wo, bank = wq.contiguous(), wk.contiguous(), wv.contiguous(), wo.contiguous(), bank.contiguous()
            call("moc_seq_layer_fwd_ex", ptr(h), ptr(bank), ptr(wrc), L.dtype_code(wrc.dtype), ptr(brc), ptr(wq),
                 ptr(wk), ptr(wv), ptr(wo), ptr(cf), B, Lq, d, H, HK, C, S, k, scale, norm, eps, 1 if train else 0,
                 ptr(out), ptr(logits), ptr(idx), ptr(idx_star), ptr(omega), ptr(saved), nbytes, main.cuda_stream,
                 aux.cuda_stream)
            if train:
                ctx.save_for_backward(h, bank, wrc, cf, logits, idx, omega, saved)
                ctx.nscratch = sizes[1]
            ctx.mark_non_differentiable(idx, idx_star, omega)
            return out, logits, idx, idx_star, omega
        h2 = h.view(B * Lq, d)
        main = torch.cuda.current_stream(dev)
        aux = ops._side_stream(dev, "aux")

        # aux: q projection and the K/V weight pack (outputs allocated on the main stream)
        q = torch.empty(B * Lq, d, device=dev, dtype=h.dtype)
        wkv = torch.empty(2 * KV, d, device=dev, dtype=torch.bfloat16)
        wqc, wkc, wvc = wq.contiguous(), wk.contiguous(), wv.contiguous()
        aux.wait_stream(main)
        with torch.cuda.stream(aux):
            with L.region("lib_linear_fwd"):
                torch.matmul(h2, wqc.t(), out=q)
            call("moc_weight_pack", ptr(wkc), L.dtype_code(wkc.dtype), ptr(wvc), L.dtype_code(wvc.dtype), KV, d,
                 ptr(wkv), None, aux.cuda_stream)
        q_ready = torch.cuda.Event()
        q_ready.record(aux)

        # main: router (pool -> linear -> top-k + prepend)
        st = main.cuda_stream
        cf = None if coef is None else coef.to(device=dev, dtype=torch.float32).contiguous()
        pooled = torch.empty(B, d, device=dev, dtype=torch.float32)
        call("moc_router_pool1", ptr(h), L.dtype_code(h.dtype), B, Lq, d, ptr(cf), ptr(pooled), st)
        wrc = wr.contiguous()
        brc = None if br is None else br.float().contiguous()
        logits = torch.empty(B, C, device=dev, dtype=torch.float32)
        call("moc_router_linear", ptr(pooled), B, d, ptr(wrc), L.dtype_code(wrc.dtype), ptr(brc), C, ptr(logits), st)
        idx = torch.empty(B, k, device=dev, dtype=torch.int32)
        w = torch.empty(B, k, device=dev, dtype=torch.float32)
        idx_star = torch.empty(B, NS, device=dev, dtype=torch.int32)
        omega = torch.empty(B, NS, device=dev, dtype=torch.float32)
        call("moc_router_topk_prepend", ptr(logits), B, C, S, k, float(scale), ptr(idx), ptr(w), ptr(idx_star),
             ptr(omega), st)

        # main: plan, K/V projection, attention (waits for q and the packed weights)
        main.wait_event(q_ready)
        out_attn, saved, acfg = ops.routed_attn_forward(q.view(B, Lq, H, Dh), bank, wk, wv, omega, idx_star, C, T,
                                                        norm, eps, HK, wkv=wkv)
        a2 = out_attn.view(B * Lq, d)
        with L.region("lib_linear_fwd"):
            out = F.linear(a2, wo)
        ctx.row_grad = getattr(bank, "_moc_row_grad", None)
        ctx.save_for_backward(h, wrc, wqc, wo, pooled, logits, idx, w, cf, *saved)
        ctx.acfg = acfg
        ctx.mark_non_differentiable(idx, idx_star, omega)
        return out.view(B, Lq, d), logits, idx, idx_star, omega

    @staticmethod
    def backward(ctx, dout, dlogits, _didx, _didx_star, _domega):
        if ctx.native:
            return _native_backward(ctx, dout, dlogits)
        h, wrc, wqc, wo, pooled, logits, idx, w, cf = ctx.saved_tensors[:9]
        saved = ctx.saved_tensors[9:]
        C, T, S, k, scale, H, HK, norm, eps, _train = ctx.cfg
        need_h, need_bank, need_wr, need_br, need_wq, need_wk, need_wv, need_wo = ctx.needs_input_grad[:8]
        dev = h.device
        B, Lq, d = h.shape
        Dh = d // H
        a2 = saved[4].view(B * Lq, d)          # attention output (the o_proj input)
        main = torch.cuda.current_stream(dev)
        aux = ops._side_stream(dev, "aux")
        dh = dwr = dbr = dwq = dwo = None
        if dout is None:
            dout = torch.zeros(B, Lq, d, device=dev, dtype=h.dtype)
        dout2 = dout.reshape(B * Lq, d).to(h.dtype).contiguous()

        # aux: o_proj dW beside the o_proj dX and the attention backward's first kernels
        if need_wo:
            dwo = torch.empty(wo.shape, device=dev, dtype=wo.dtype)
            aux.wait_stream(main)
            with torch.cuda.stream(aux):
                ops.linear_wgrad(dout2, a2, wo.dtype, out=dwo)
        with L.region("lib_linear_dx"):
            d_attn = torch.matmul(dout2, wo)
        if need_h:
            dh = torch.empty(B, Lq, d, device=dev, dtype=h.dtype)
        if need_wq:
            dwq = torch.empty(wqc.shape, device=dev, dtype=wqc.dtype)

        def after_dq(dq):
            # aux: the q projection's dX (into dh) and dW beside the dK/dV kernel
            if not (need_h or need_wq):
                return
            aux.wait_stream(main)
            with torch.cuda.stream(aux):
                dq2 = dq.view(B * Lq, d)
                if need_h:
                    with L.region("lib_linear_dx"):
                        torch.matmul(dq2, wqc, out=dh.view(B * Lq, d))
                if need_wq:
                    ops.linear_wgrad(dq2, h.view(B * Lq, d), wqc.dtype, out=dwq)

        router_out = {}

        def after_dkv(dom_part):
            # aux: the router's backward and the pooling's gradient, beside the K/V chapter GEMMs
            if not (need_h or need_wr or need_br):
                return
            dz = torch.empty(B, C, device=dev, dtype=torch.float32)
            dpooled = torch.empty(B, d, device=dev, dtype=torch.float32) if need_h else None
            dW = torch.empty(C, d, device=dev, dtype=torch.float32) if need_wr else None
            db = torch.empty(C, device=dev, dtype=torch.float32) if need_br else None
            ws = None
            if dpooled is not None:
                ws = torch.empty(L.query("moc_router_linear_bwd_workspace", B, d, C) // 4, device=dev,
                                 dtype=torch.float32)
            dz_in = None if dlogits is None else dlogits.float().contiguous()
            aux.wait_stream(main)
            sa = aux.cuda_stream
            call("moc_router_seq_bwd", ptr(logits), ptr(idx), ptr(w), ptr(dom_part), HK, B, C, S, k, float(scale),
                 ptr(dz_in), ptr(dz), sa)
            call("moc_router_linear_bwd", ptr(dz), ptr(pooled), B, d, ptr(wrc), L.dtype_code(wrc.dtype), C,
                 ptr(dpooled), ptr(dW), ptr(db), ptr(ws), 0 if ws is None else ws.numel() * 4, sa)
            if dpooled is not None:
                call("moc_rows_add_bcast", ptr(dh), L.dtype_code(dh.dtype), B, Lq, d, ptr(dpooled), ptr(cf),
                     1.0 / Lq, sa)
            # kept alive (and unused by the main stream) until the main stream has waited for aux
            router_out.update(dz=dz, dpooled=dpooled, ws=ws, dz_in=dz_in, dom_part=dom_part, dW=dW, db=db)

        dq, dbank, dwk, dwv, _ = ops.routed_attn_backward(
            saved, ctx.acfg, d_attn.view(B, Lq, H, Dh), (True, need_bank, need_wk, need_wv, True),
            row_grad=ctx.row_grad, after_dq=after_dq, after_dkv=after_dkv)
        main.wait_stream(aux)
        if need_wr:
            dwr = router_out["dW"].to(ctx.wdt[0])
        if need_br:
            dbr = router_out["db"].to(ctx.wdt[1])
        return dh, dbank, dwr, dbr, dwq, dwk, dwv, dwo, None, None


def _trains(*tensors) -> bool:
    """Whether a backward may follow a call on these tensors (grad mode is off inside a function's forward)."""
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)


@functools.lru_cache(maxsize=256)
def _f32_trains(B, Lq, C, S, k) -> bool:
    return bool(L.query("moc_seq_layer_f32_trains", B, Lq, C, S, k))


@functools.lru_cache(maxsize=256)
def _f32_sizes(B, Lq, d, H, HK, C, S, k, norm):
    """(saved, scratch) buffer bytes of the native float32 layer, or None for shapes outside it."""
    n = (ctypes.c_size_t * 2)()
    at = [ctypes.addressof(n) + i * ctypes.sizeof(ctypes.c_size_t) for i in range(2)]
    return tuple(n) if L.query("moc_seq_layer_f32_sizes", B, Lq, d, H, HK, C, S, k, norm, *at) == L.MOC_OK else None


def supported_f32(h, bank, wr, br, wq, wk, wv, wo, *, num_chapters: int, tokens_per_chapter: int, num_shared: int,
                  top_k: int, num_heads: int, num_kv_heads: int, norm_type: Optional[str] = None) -> bool:
    """Whether moc_seq_layer_f32_fwd / _bwd take this call; every other float32 call keeps the per-op
    autograd functions.  Under autocast those cast, so such calls stay with them too."""
    f32 = torch.float32
    if not (h.dtype == f32 and h.is_cuda and h.dim() == 3 and h.shape[1] > 0 and tokens_per_chapter == 64
            and num_shared > 0 and top_k > 0 and not torch.is_autocast_enabled()):
        return False
    d = h.shape[2]
    KV = num_kv_heads * 64
    if (bank.dim() != 2 or bank.shape[0] < num_chapters * 64 or bank.shape[1] != d or wr.dtype not in (f32, torch.bfloat16)
            or wr.shape != (num_chapters, d) or wq.shape != (d, d) or wo.shape != (d, d) or wk.shape != (KV, d)
            or wv.shape != (KV, d) or getattr(bank, "_moc_bank_opt", None) is not None
            or getattr(bank, "_moc_row_grad", None) is not None):
        return False
    for t in (h, bank, wq, wk, wv, wo, wr, br):     # the kernels read 16-byte pieces of packed rows
        if t is not None and (t.device != h.device or not t.is_contiguous() or t.data_ptr() % 16
                              or (t is not wr and t.dtype != f32)):
            return False
    if (_trains(h, bank, wr, br, wq, wk, wv, wo)
            and not _f32_trains(h.shape[0], h.shape[1], num_chapters, num_shared, top_k)):
        return False
    return _f32_sizes(h.shape[0], h.shape[1], d, num_heads, num_kv_heads, num_chapters, num_shared, top_k,
                      ops.norm_code(norm_type)) is not None


def _f32_per_op(h, bank, wr, br, wq, wk, wv, wo, *, coef, cfg):
    """(out, logits) of the layer through the per-op autograd functions."""
    C, T, S, k, scale, H, HK, norm, eps, _train = cfg
    B, Lq, d = h.shape
    logits = ops.router_linear(ops.router_pool(h, coef), wr, br)
    idx_star, omega = ops.prepend_shared(*ops.router_topk(logits, k, S), S, scale)
    q = ops.linear(h, wq).view(B, Lq, H, d // H)
    a = ops.routed_attention(q, bank, wk, wv, omega, idx_star, num_chapters=C, tokens_per_chapter=T,
                             norm_type=ops.norm_name(norm), eps=eps, num_kv_heads=HK)
    return ops.linear(a.reshape(B, Lq, d), wo), logits


class _SeqF32Layer(torch.autograd.Function):
    """The float32 layer in one host call each way.  A recorded backward (create_graph) goes through the
    per-op functions instead, whose products of the projections are recorded."""

    @staticmethod
    def forward(ctx, h, bank, wr, br, wq, wk, wv, wo, coef, cfg):
        C, T, S, k, scale, H, HK, norm, eps, train = cfg
        dev = h.device
        B, Lq, d = h.shape
        nsaved, ctx.nscratch = _f32_sizes(B, Lq, d, H, HK, C, S, k, norm)
        cf = None if coef is None else coef.to(device=dev, dtype=torch.float32).contiguous()
        saved = torch.empty(nsaved, device=dev, dtype=torch.uint8)
        out = torch.empty(B, Lq, d, device=dev, dtype=torch.float32)
        logits = torch.empty(B, C, device=dev, dtype=torch.float32)
        idx = torch.empty(B, k, device=dev, dtype=torch.int32)
        idx_star = torch.empty(B, S + k, device=dev, dtype=torch.int32)
        omega = torch.empty(B, S + k, device=dev, dtype=torch.float32)
        call("moc_seq_layer_f32_fwd", ptr(h), ptr(bank), ptr(wr), L.dtype_code(wr.dtype), ptr(br), ptr(wq), ptr(wk),
             ptr(wv), ptr(wo), ptr(cf), B, Lq, d, H, HK, C, S, k, scale, norm, eps, ptr(out), ptr(logits), ptr(idx),
             ptr(idx_star), ptr(omega), ptr(saved), nsaved, stream_ptr(dev))
        ctx.cfg = cfg
        ctx.set_materialize_grads(False)
        if train:
            ctx.save_for_backward(h, bank, wr, br, wq, wk, wv, wo, cf, logits, idx, omega, saved)
        ctx.mark_non_differentiable(idx, idx_star, omega)
        return out, logits, idx, idx_star, omega

    @staticmethod
    def backward(ctx, dout, dlogits, _didx, _didx_star, _domega):
        h, bank, wr, br, wq, wk, wv, wo, cf, logits, idx, omega, saved = ctx.saved_tensors
        if torch.is_grad_enabled():     # create_graph: the backward is itself differentiated
            grads = ops.recorded_backward(functools.partial(_f32_per_op, coef=cf, cfg=ctx.cfg),
                                          (h, bank, wr, br, wq, wk, wv, wo), ctx.needs_input_grad[:8], (dout, dlogits))
            return (*grads, None, None)
        C, T, S, k, scale, H, HK, norm, eps, _train = ctx.cfg
        need_h, need_bank, need_wr, need_br, need_wq, need_wk, need_wv, need_wo = ctx.needs_input_grad[:8]
        dev = h.device
        B, Lq, d = h.shape
        KV = HK * 64

        def new(need, *shape):
            return torch.empty(shape, device=dev, dtype=torch.float32) if need else None

        dout = torch.zeros(B, Lq, d, device=dev) if dout is None else dout.contiguous()
        if dout.data_ptr() % 16:
            dout = dout.clone()
        dz = None if dlogits is None else dlogits.float().contiguous()
        dh, dbank, dwr, dbr = new(need_h, B, Lq, d), new(need_bank, *bank.shape), new(need_wr, C, d), new(need_br, C)
        dwq, dwkv, dwo = new(need_wq, d, d), new(need_wk or need_wv, 2 * KV, d), new(need_wo, d, d)
        scratch = torch.empty(ctx.nscratch, device=dev, dtype=torch.uint8)
        call("moc_seq_layer_f32_bwd", ptr(h), ptr(bank), ptr(wr), L.dtype_code(wr.dtype), ptr(wq), ptr(wk), ptr(wv),
             ptr(wo), ptr(cf), B, Lq, d, H, HK, C, S, k, scale, norm, ptr(logits), ptr(idx), ptr(omega), ptr(saved),
             saved.numel(), ptr(dout), ptr(dz), ptr(dh), ptr(dbank), bank.shape[0], ptr(dwr), ptr(dbr), ptr(dwq),
             ptr(dwkv), ptr(dwo), ptr(scratch), ctx.nscratch, stream_ptr(dev))
        dwk = dwkv[:KV] if need_wk else None
        dwv = dwkv[KV:] if need_wv else None
        return (dh, dbank, dwr if dwr is None else dwr.to(wr.dtype), dbr, dwq, dwk, dwv, dwo, None, None)


def _native_backward(ctx, dout, dlogits):
    """The whole backward in one host call (moc_seq_layer_bwd_ex)."""
    h, bank, wrc, cf, logits, idx, omega, saved = ctx.saved_tensors
    C, T, S, k, scale, H, HK, norm, eps, _train = ctx.cfg
    need_h, need_bank, need_wr, need_br, need_wq, need_wk, need_wv, need_wo = ctx.needs_input_grad[:8]
    dev = h.device
    B, Lq, d = h.shape
    KV = HK * 64
    if dout is None:
        dout = torch.zeros(B, Lq, d, device=dev, dtype=h.dtype)
    dout = dout.to(h.dtype).contiguous()
    dz_in = None if dlogits is None else dlogits.float().contiguous()
    dh = torch.empty(B, Lq, d, device=dev, dtype=h.dtype) if need_h else None
    dbank = torch.empty(bank.shape, device=dev, dtype=bank.dtype) if need_bank else None
    dwr = torch.empty(C, d, device=dev, dtype=torch.float32) if need_wr else None
    dbr = torch.empty(C, device=dev, dtype=torch.float32) if need_br else None
    dwq = torch.empty(d, d, device=dev, dtype=torch.bfloat16) if need_wq else None
    dwkv = torch.empty(2 * KV, d, device=dev, dtype=torch.bfloat16) if (need_wk or need_wv) else None
    dwo = torch.empty(d, d, device=dev, dtype=torch.bfloat16) if need_wo else None
    nscratch = ctx.nscratch
    scratch = torch.empty(nscratch, device=dev, dtype=torch.uint8)
    main = torch.cuda.current_stream(dev)
    aux = ops._side_stream(dev, "aux")
    fill = ops._side_stream(dev, "fill")
    call("moc_seq_layer_bwd_ex", ptr(h), ptr(bank), ptr(wrc), L.dtype_code(wrc.dtype), ptr(cf), B, Lq, d, H, HK, C, S,
         k, scale, norm, ptr(logits), ptr(idx), ptr(omega), ptr(saved), saved.numel(), ptr(dout), ptr(dz_in), ptr(dh),
         ptr(dbank), bank.shape[0], ptr(dwr), ptr(dbr), ptr(dwq), ptr(dwkv), L.MOC_BF16, ptr(dwo), ptr(scratch),
         nscratch, main.cuda_stream, aux.cuda_stream, fill.cuda_stream)
    dwk = dwkv[:KV] if need_wk else None
    dwv = dwkv[KV:] if need_wv else None
    if dwr is not None:
        dwr = dwr.to(ctx.wdt[0])
    if dbr is not None:
        dbr = dbr.to(ctx.wdt[1])
    return dh, dbank, dwr, dbr, dwq, dwk, dwv, dwo, None, None


def seq_routed_layer(h, bank, wr, br, wq, wk, wv, wo, *, num_chapters: int, tokens_per_chapter: int,
                     num_shared: int, top_k: int, routed_scale: float, num_heads: int, num_kv_heads: int,
                     norm_type: Optional[str] = None, eps: float = 1e-6, coef: Optional[torch.Tensor] = None):
    """(out (B, L, d), logits f32 (B, C), idx int32 (B, k), idx_star int32 (B, S+k), omega f32 (B, S+k))."""
    train = _trains(h, bank, wr, br, wq, wk, wv, wo)
    cfg = (int(num_chapters), int(tokens_per_chapter), int(num_shared), int(top_k), float(routed_scale),
           int(num_heads), int(num_kv_heads), ops.norm_code(norm_type), float(eps), train)
    layer = _SeqF32Layer if h.dtype == torch.float32 else _SeqRoutedLayer
    return layer.apply(h, bank, wr, br, wq, wk, wv, wo, coef, cfg)
