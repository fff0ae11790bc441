// Sequence-routed memory cross-attention, forward ("joint" combine).
//
// For sequence b, query i, query head h (kv head hk = h / (H / HK)) and the
// NS selected chapters c with router weights omega[b, c]:
//   s_ij  = omega_c * scale * q_i . k_j           (j ranges over chapter c's T keys)
//   o_i   = sum_j softmax_j(s_ij) * omega_c * v_j
// which is exactly MemoryCrossAttention over the omega-weighted gathered rows
// (memory_transformer/model.py:689-692 then memory_attention.py:458-478 /
// :269-318): (omega x) W^T = omega (x W^T), so the key and the value of every
// row of chapter c carry the factor omega_c.  k_j / v_j are read as (chapter, kv head)
// blocks of 64 rows through strides (projection rows [u*64 + t][K | V] on the training
// path, kv_project.hip's chapter-head tiles for the decode cache); slot_u[b, c] says which
// de-duplicated chapter holds slot c of sequence b (negative = skip the slot).
//
// Work decomposition (Dh = T = 64): one workgroup = 128 queries of one
// (sequence, head); 4 waves x 32 queries.  Every chapter is one 64-key tile,
// so omega is a scalar per tile and folds into the exp2 argument.  Each wave
// computes S^T = K Q^T (lane = one query, 16 keys), keeps the running max,
// accumulates O^T = V^T P^T, whose accumulator layout is again "lane = one
// query", so the online-softmax rescale needs no data movement, and takes the
// row sums from an MFMA of an all-ones operand with the same P^T fragments.
// K and V blocks (both [key][dim]) are double-buffered in
// LDS; the V^T operand is read from the V tile with the transposing LDS read, whose lane
// order is the key order of the P~^T fragments.
#include "moc_common.h"

namespace moc {

constexpr int kFwdThreads = 256;
constexpr int kDh = 64;
constexpr int kTch = 64;

// Running-max policy: a row's reference max m only moves up when the chapter
// max exceeds it by more than kRescaleSlack (log2 units), so most chapters skip
// the O / l rescale; probabilities stay <= 2^kRescaleSlack, far from overflow.
constexpr float kRescaleSlack = 8.f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float max3f(float a, float b, float c) { return fmax_fast(fmax_fast(a, b), c); }

// One 16-byte-per-lane LDS DMA (buffer_load_dwordx4 ... lds): lane l's 16 bytes at voff + soff
// of the buffer land at LDS address m0 + 16 l.  The wait on these loads is an explicit vmcnt(0).
typedef __attribute__((address_space(3))) void* fwd_lds_ptr_t;
__device__ __forceinline__ void fwd_dma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, const char* lds, uint32_t soff) {
  const uint32_t m0 = (uint32_t)(uintptr_t)(fwd_lds_ptr_t)lds;
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(r), "s"(soff), "{m0}"(m0) : "memory");
}

// SPLIT: the slots of a (sequence, head) are divided over nsplit workgroups per 128 queries, each
// writing normalised f32 partial rows part[split][b][l][h][64] and their log-sum-exp (log2 units,
// -inf when every slot was skipped) lse[split][b][h][Lp]; xattn_merge_kernel combines them.
template <typename T, bool SPLIT>
__global__ __launch_bounds__(kFwdThreads) void xattn_fwd_kernel(
    const T* __restrict__ q, const T* __restrict__ ktiles, const T* __restrict__ vtiles,
    const int32_t* __restrict__ slot_u, const float* __restrict__ omega, int B, int L, int H, int HK, int NS,
    int64_t kv_span, int64_t kv_su, int kv_sh, int kv_st, float scale_log2, T* __restrict__ out,
    float* __restrict__ lse, int nsplit, float* __restrict__ part) {
  typedef typename Frag<T>::type F8;
  using Tile = SwzTile<T, 64>;
  constexpr int TB = kTch * kDh * (int)sizeof(T);
  __shared__ __attribute__((aligned(16))) char sK[2][TB];
  __shared__ __attribute__((aligned(16))) char sV[2][TB];

  // tiles: (sequence, head) major, 128-query block minor, so the query blocks that read
  // the same chapter tiles share one XCD's L2
  const int nqb = (L + 127) / 128;
  const int nsp = SPLIT ? nsplit : 1;
  const int64_t t = xcd_tile((int64_t)B * H * nsp * nqb);
  if (t < 0) return;
  const int64_t bh = t / ((int64_t)nsp * nqb);
  const int b = (int)(bh / H), h = (int)(bh % H);
  const int sp = SPLIT ? (int)((t / nqb) % nsp) : 0;
  const int s_begin = SPLIT ? (int)((int64_t)NS * sp / nsp) : 0;
  const int s_end = SPLIT ? (int)((int64_t)NS * (sp + 1) / nsp) : NS;
  const int hk = h / (H / HK);
  const int q0 = (int)(t % nqb) * 128;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c16 = lane & 15;

  // Q^T fragments (B operand): query = q0 + 32*wave + 16*qb + c16, dims 32*ks + 8*g ..
  F8 qf[2][2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int qi = q0 + 32 * wave + 16 * qb + c16;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (qi < L)
        qf[qb][ks] = Load8<T, T>::run(q + ((size_t)(b * (size_t)L + qi) * H + h) * kDh + 32 * ks + 8 * g);
      else
        qf[qb][ks] = zero_frag<T>();
    }
  }

  float m[2] = {-INFINITY, -INFINITY};
  float lsum[2] = {0.f, 0.f};  // row sums of p (in units of exp2(m)), complete per lane
  float pend_ls[2] = {0.f, 0.f}, pend_rw = 0.f;   // last chapter's row sums, not yet folded in
  // all-ones A operand: the MFMA with it sums a P~^T fragment over its 32 keys, which
  // takes the row sums off the VALU (the sums use the same rounded P~ as O)
  F8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = from_f<T>(1.f);
  f32x4 o[4][2];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) o[db][qb] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int32_t* su = slot_u + (size_t)b * NS;
  const float* om = omega + (size_t)b * NS;
  TileIO<T, kFwdThreads> kio, vio;
  // block (u, hk) of K / V: element (t, dh) at u kv_su + hk kv_sh + t kv_st + dh of two buffers of
  // kv_span elements each
  const Buf kb(ktiles, (uint32_t)(kv_span * (int64_t)sizeof(T))), vb(vtiles, (uint32_t)(kv_span * (int64_t)sizeof(T)));
  auto tile_off = [&](int u) { return (uint32_t)(((size_t)u * kv_su + (size_t)hk * kv_sh) * sizeof(T)); };
  const uint32_t row_bytes = (uint32_t)(kv_st * (int)sizeof(T));
  // bf16: a slot's K and V tiles go global -> LDS by DMA (no registers held while in flight):
  // 8 instructions of 1 KB (8 rows of 128 B) per tile, wave w issuing 2w and 2w + 1; lane l fills
  // row 8 j + l / 8, physical chunk l % 8 = logical chunk (l % 8) ^ (row & 7) of Tile::off.
  // fp32: through registers.
  constexpr bool kDma = sizeof(T) == 2;
  static_assert(!kDma || (kFwdThreads == 256 && TB == 8192), "DMA staging geometry");
  const uint32_t dma_v0 = (uint32_t)((16 * wave + (lane >> 3)) * row_bytes + 16 * ((lane & 7) ^ (lane >> 3)));
  auto fetch = [&](int u, int buf) {
    if constexpr (kDma) {
      const uint32_t so = tile_off(u);
      fwd_dma16(kb.r, dma_v0, sK[buf] + 2048 * wave, so);
      fwd_dma16(kb.r, dma_v0 + 8 * row_bytes, sK[buf] + 2048 * wave + 1024, so);
      fwd_dma16(vb.r, dma_v0, sV[buf] + 2048 * wave, so);
      fwd_dma16(vb.r, dma_v0 + 8 * row_bytes, sV[buf] + 2048 * wave + 1024, so);
    } else {
      kio.load_rows(kb, tile_off(u), row_bytes, tid);
      vio.load_rows(vb, tile_off(u), row_bytes, tid);
    }
  };

  // S^T[kb][qb]: rows = keys 16*kb + 4*g + e, column = query c16 of block qb
  auto scores = [&](const char* Ks, f32x4 (&st)[4][2]) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) st[kb][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        F8 a = Tile::frag(Ks, 16 * kb + c16, 32 * ks + 8 * g);
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) mma(st[kb][qb], a, qf[qb][ks]);
      }
    }
  };
  // a row's maximum over the chapter (three-input max chains)
  auto row_max = [&](const f32x4 (&st)[4][2], int qb) {
    float mx = max3f(st[0][qb][0], st[0][qb][1], st[0][qb][2]);
    mx = max3f(mx, st[0][qb][3], st[1][qb][0]);
    mx = max3f(mx, st[1][qb][1], st[1][qb][2]);
    mx = max3f(mx, st[1][qb][3], st[2][qb][0]);
    mx = max3f(mx, st[2][qb][1], st[2][qb][2]);
    mx = max3f(mx, st[2][qb][3], st[3][qb][0]);
    mx = max3f(mx, st[3][qb][1], st[3][qb][2]);
    return quad_max_pl(fmax_fast(mx, st[3][qb][3]));
  };

  int u_cur = su[s_begin];
  if (u_cur >= 0) {
    fetch(u_cur, s_begin & 1);
    if constexpr (!kDma) {
      kio.store(sK[s_begin & 1], tid);
      vio.store(sV[s_begin & 1], tid);
    }
  }
  // A later split starts from the maximum over the row's first used chapter, as the unsplit loop does:
  // bf16 rounds P~ = 2^(logit - m) to 8 bits, and where a chapter's P~ falls in their binade, hence each
  // one's rounding, goes with m.  With one m the splits round every P~ as the unsplit kernel (until a
  // maximum grows by more than kRescaleSlack) and differ from it by f32 sums only; each with its own
  // first maximum, single prompts came out with up to 1.03 times its error.
  int s_first = s_begin;
  if constexpr (SPLIT && kDma) {
    s_first = 0;
    while (s_first < s_begin && su[s_first] < 0) ++s_first;
    s_first = __builtin_amdgcn_readfirstlane(s_first);   // the DMA's offset is a scalar operand
    if (s_first < s_begin) {
      const uint32_t so = tile_off(su[s_first]);
      fwd_dma16(kb.r, dma_v0, sK[(s_begin & 1) ^ 1] + 2048 * wave, so);
      fwd_dma16(kb.r, dma_v0 + 8 * row_bytes, sK[(s_begin & 1) ^ 1] + 2048 * wave + 1024, so);
    }
  }
  // Q fragments must have landed before the loop on every path (also when slot 0
  // is skipped); otherwise the wait for them inside the loop can't be told apart
  // from the prefetch and becomes a full vmcnt(0) ahead of the first MFMA.
  vm_wait_all();
  __syncthreads();
  if constexpr (SPLIT && kDma) {
    if (s_first < s_begin) {
      f32x4 st[4][2];
      scores(sK[(s_begin & 1) ^ 1], st);
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        const float cm = row_max(st, qb) * (om[s_first] * scale_log2);
        m[qb] = cm > m[qb] + kRescaleSlack ? cm : m[qb];
      }
      __syncthreads();   // the loop's first fetch overwrites this tile
    }
  }

  for (int s = s_begin; s < s_end; ++s) {
    const int buf = s & 1;
    const int u_next = (s + 1 < s_end) ? su[s + 1] : -1;
    // (buffer buf ^ 1 was last read in slot s - 1, which every wave has finished)
    if (u_next >= 0) fetch(u_next, buf ^ 1);
    if (u_cur >= 0) {
      const float w = om[s];
      const float c = w * scale_log2;
      const char* Ks = sK[buf];
      const char* Vs = sV[buf];
      f32x4 st[4][2];
      scores(Ks, st);
      // the previous chapter's row sums (their MFMA has long completed): folded in before any
      // rescale, in units of the reference max they were taken against
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) lsum[qb] += pend_ls[qb] * pend_rw;
      pend_rw = 0.f;
      // chapter max per row, lazy update of the reference max
      float cm[2];
      bool grow = false;
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        cm[qb] = row_max(st, qb) * c;  // c >= 0 (router weights are non-negative)
        grow |= cm[qb] > m[qb] + kRescaleSlack;
      }
      if (__any(grow)) {
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
          const float mn = cm[qb] > m[qb] + kRescaleSlack ? cm[qb] : m[qb];
          const float alpha = fast_exp2(m[qb] - mn);
          m[qb] = mn;
          lsum[qb] *= alpha;
#pragma unroll
          for (int db = 0; db < 4; ++db) o[db][qb] *= alpha;
        }
      }
      F8 pf[2][2];
      if (w > kTinyOmega) {
        // p~ = w * exp2(s*c - m): w folded into the exponent; the row sum needs sum(p~) / w
        const float lw = __builtin_amdgcn_logf(w);
        const float rw = __builtin_amdgcn_rcpf(w);
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
          const float off = m[qb] - lw;
#pragma unroll
          for (int ks2 = 0; ks2 < 2; ++ks2)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              pf[qb][ks2][e] = from_f<T>(fast_exp2(st[2 * ks2][qb][e] * c - off));
              pf[qb][ks2][4 + e] = from_f<T>(fast_exp2(st[2 * ks2 + 1][qb][e] * c - off));
            }
          f32x4 ls = f32x4{0.f, 0.f, 0.f, 0.f};
          mma(ls, ones, pf[qb][0]);
          mma(ls, ones, pf[qb][1]);
          pend_ls[qb] = ls[0];   // folded in at the next chapter (no wait on this MFMA here)
        }
        pend_rw = rw;
        // O^T[db][qb] += V^T(dims 16*db + c16, keys) * P~^T
#pragma unroll
        for (int ks2 = 0; ks2 < 2; ++ks2) {
#pragma unroll
          for (int db = 0; db < 4; ++db) {
            const F8 a = mk_frag<Tile, T>(Vs, 32 * ks2, 16 * db, lane);  // V^T, keys in MFMA key order
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) mma(o[db][qb], a, pf[qb][ks2]);
          }
        }
      } else {
        // zero (or below-floor) weight: keys and values vanish, every logit is 0 -> only the
        // denominator moves
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) lsum[qb] += 64.f * fast_exp2(-m[qb]);
      }
    }
    if (u_next >= 0) {
      if constexpr (kDma) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next slot's tiles landed
      } else {
        kio.store(sK[buf ^ 1], tid);
        vio.store(sV[buf ^ 1], tid);
      }
    }
    u_cur = u_next;
    __syncthreads();
  }

#pragma unroll
  for (int qb = 0; qb < 2; ++qb) lsum[qb] += pend_ls[qb] * pend_rw;
  // lse rows have stride Lp = round_up(L, 128); padded entries hold +inf so
  // that the backward's exp2(s - lse) is exactly 0 there (also for a row
  // whose every slot was skipped).
  const int Lp = nqb * 128;
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const float l = lsum[qb];
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const int qi = q0 + 32 * wave + 16 * qb + c16;
    if constexpr (SPLIT) {
      if (qi < L) {
        float* pp = part + ((((size_t)sp * B + b) * L + qi) * H + h) * kDh + 4 * g;
#pragma unroll
        for (int db = 0; db < 4; ++db) *reinterpret_cast<f32x4*>(pp + 16 * db) = o[db][qb] * inv;
      }
      if (g == 0) lse[(((size_t)sp * B + b) * H + h) * Lp + qi] = l > 0.f ? m[qb] + log2f(l) : -INFINITY;
      continue;
    }
    if (qi < L) {
      T* op = out + ((size_t)(b * (size_t)L + qi) * H + h) * kDh;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int e = 0; e < 4; ++e) op[16 * db + 4 * g + e] = from_f<T>(o[db][qb][e] * inv);
    }
    if (g == 0) lse[((size_t)b * H + h) * Lp + qi] = (qi < L && l > 0.f) ? m[qb] + log2f(l) : INFINITY;
  }
}

// out = sum_i 2^(lse_i - M) o_i / sum_i 2^(lse_i - M) over the splits of a (sequence, query, head) row
// and the row's log-sum-exp (+inf when every slot was skipped, and in the padding rows L .. Lp - 1):
// 16 lanes of 4 dims per row, rows in [b][l][h] order.
template <typename T>
__global__ __launch_bounds__(256) void xattn_merge_kernel(const float* __restrict__ part,
                                                          const float* __restrict__ lse_part, int nsplit, int B, int L,
                                                          int Lp, int H, T* __restrict__ out, float* __restrict__ lse) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = i >> 4;
  const int ch = (int)(i & 15);
  if (row >= (int64_t)B * Lp * H) return;
  const int h = (int)(row % H);
  const int64_t bl = row / H;
  const int b = (int)(bl / Lp), qi = (int)(bl % Lp);
  float* lo = lse + ((size_t)b * H + h) * Lp + qi;
  if (qi >= L) {
    if (ch == 0) *lo = INFINITY;
    return;
  }
  const size_t ls = (size_t)B * H * Lp, ps = (size_t)B * L * H * kDh;
  const float* lp = lse_part + ((size_t)b * H + h) * Lp + qi;
  const float* pp = part + (((size_t)b * L + qi) * H + h) * kDh + 4 * ch;
  float M = -INFINITY;
#pragma unroll 8
  for (int sp = 0; sp < nsplit; ++sp) M = fmaxf(M, lp[sp * ls]);
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  float den = 0.f;
#pragma unroll 8
  for (int sp = 0; sp < nsplit; ++sp) {
    const float a = M > -INFINITY ? fast_exp2(lp[sp * ls] - M) : 0.f;
    acc += *reinterpret_cast<const f32x4*>(pp + sp * ps) * a;
    den += a;
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
  T* op = out + (((size_t)b * L + qi) * H + h) * kDh + 4 * ch;
#pragma unroll
  for (int x = 0; x < 4; ++x) op[x] = from_f<T>(acc[x] * inv);
  if (ch == 0) *lo = den > 0.f ? M + log2f(den) : INFINITY;
}

// Attention weights of the forward above, materialised (MemoryCrossAttention.forward with
// return_attn_weights, memory_attention.py:437-447: softmax(q k^T * scale) over the sequence's
// selected keys, which carry omega): p_ij = exp2(omega_c scale log2(e) q_i . k_j - lse_i) with the
// forward's row log-sum-exp.  One workgroup = 64 queries x one slot of one (sequence, head), wave w
// owning queries 16 w .. 16 w + 15: S^T = K Q^T from global fragments (lane = query, 16 keys per
// lane), then 4 consecutive keys per store.  A skipped slot's keys get weight 0; a slot below the
// omega floor gets every logit 0 (its keys vanish), as in the forward.
template <typename T>
__global__ __launch_bounds__(256) void xattn_weights_kernel(
    const T* __restrict__ q, const T* __restrict__ ktiles, const int32_t* __restrict__ slot_u,
    const float* __restrict__ omega, int B, int L, int H, int HK, int NS, int64_t kv_span, int64_t kv_su, int kv_sh,
    int kv_st, float scale_log2, const float* __restrict__ lse, T* __restrict__ P) {
  typedef typename Frag<T>::type F8;
  const int nqb = (L + 63) / 64;
  const int64_t t = blockIdx.x;
  const int s = (int)(t % NS);
  const int64_t r = t / NS;
  const int qb = (int)(r % nqb);
  const int h = (int)((r / nqb) % H), b = (int)(r / ((int64_t)nqb * H));
  const int hk = h / (H / HK);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c16 = lane & 15;
  const int qi = qb * 64 + 16 * wave + c16;
  const int Lp = (L + 127) / 128 * 128;
  const int u = slot_u[(size_t)b * NS + s];
  const float w = omega[(size_t)b * NS + s];
  const float lq = qi < L ? lse[((size_t)b * H + h) * Lp + qi] : 0.f;
  f32x4 st[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) st[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (u >= 0 && w > kTinyOmega) {
    F8 qf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      qf[ks] = qi < L ? Load8<T, T>::run(q + ((size_t)(b * (size_t)L + qi) * H + h) * kDh + 32 * ks + 8 * g)
                      : zero_frag<T>();
    // K block (u, hk) through a bounded buffer resource (reads past kv_span return zero)
    const Buf kbuf(ktiles, (uint32_t)(kv_span * (int64_t)sizeof(T)));
    const uint32_t soff = (uint32_t)(((size_t)u * kv_su + (size_t)hk * kv_sh) * sizeof(T));
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const uint32_t voff = (uint32_t)(((16 * kb + c16) * kv_st + 32 * ks + 8 * g) * (int)sizeof(T));
        F8 a;
        if constexpr (sizeof(T) == 2) {
          a = __builtin_bit_cast(F8, kbuf.load16(voff, soff));
        } else {
          const V16 lo = kbuf.load16(voff, soff), hi = kbuf.load16(voff + 16, soff);
          a = F8{__uint_as_float(lo.w[0]), __uint_as_float(lo.w[1]), __uint_as_float(lo.w[2]), __uint_as_float(lo.w[3]),
                 __uint_as_float(hi.w[0]), __uint_as_float(hi.w[1]), __uint_as_float(hi.w[2]), __uint_as_float(hi.w[3])};
        }
        mma(st[kb], a, qf[ks]);
      }
  }
  if (qi >= L) return;
  const float c = w * scale_log2;
  T* row = P + (((size_t)b * H + h) * L + qi) * ((size_t)NS * kTch) + (size_t)s * kTch;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    T v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = from_f<T>(u < 0 ? 0.f : fast_exp2(st[kb][e] * c - lq));
    if constexpr (sizeof(T) == 2) {
      *reinterpret_cast<bf16x4*>(row + 16 * kb + 4 * g) = bf16x4{v[0], v[1], v[2], v[3]};
    } else {
      *reinterpret_cast<f32x4*>(row + 16 * kb + 4 * g) = f32x4{v[0], v[1], v[2], v[3]};
    }
  }
}

}  // namespace moc

using namespace moc;

// The loop over the slots is a serial chain, and a launch has one workgroup per (sequence, head, 128
// queries), a "tile".  A slot takes the longer the more workgroups a CU holds at once, at most three: bf16
// ~1.15 / 1.45 / 2.1 us; f32 ~6 us each, as if one after another (its registers fill a CU).  Splitting the
// slots n ways costs a merge launch (~5 us, ~0.2 a split) and f32 partial rows (~0.016 us per tile
// and split, written and read).  n is the one of least sum; 1, not split, has the chain alone.  Measured,
// unsplit -> split, forward / dQ, us:
//   bf16 65 slots:  48 tiles 72 -> 29 / 65 -> 25, 192 tiles 73 -> 52 / 66 -> 50, 384 tiles 95 -> 78 / 93 -> 84
//        64 slots: 128 tiles 71 -> 41 / 64 -> 40, 256 tiles 71 -> 62 / 65 -> 62
//        33 slots:  64 tiles 38 -> 23 / 35 -> 19, 256 tiles at three splits 39 -> 44 / 36 -> 42 (not split)
//        17 slots:  48 tiles 22 -> 17 / 20 -> 14;  9 slots: 24 tiles 13 -> 13 / 13 -> 11
//   f32  65 slots:  48 tiles 341 -> 84 / 441 -> 99, 192 tiles 342 -> 256 / 442 -> 357, 384 tiles 608 -> 488 /
//        881 -> 694; 64 slots: 256 tiles at three splits 337 -> 328 / 437 -> 462 (not split)
int moc::xattn_splits(int dtype, int64_t B, int64_t L, int H, int NS) {
  const int64_t tiles = B * H * ((L + 127) / 128);
  if (tiles <= 0 || NS <= 1) return 1;
  auto chain = [&](int64_t n) {
    const int64_t per_cu = (tiles * n + 255) / 256;
    const double slot = dtype == MOC_F32 ? 6.0 * per_cu : per_cu == 1 ? 1.15 : per_cu == 2 ? 1.45 : 2.1;
    return slot * (double)((NS + n - 1) / n);
  };
  int64_t best = 1;
  double least = chain(1);
  for (int64_t n = 2; n <= NS && n * tiles <= kXattnWgs; ++n) {
    const double cost = 5.0 + 0.2 * (double)n + chain(n) + 0.016 * (double)(n * tiles);
    if (cost < least) least = cost, best = n;
  }
  const int64_t per = (NS + best - 1) / best;
  return (int)((NS + per - 1) / per);
}

extern "C" {

size_t moc_xattn_split_workspace(int dtype, int64_t B, int64_t L, int H, int NS) {
  const int n = xattn_splits(dtype, B, L, H, NS);
  return n > 1 ? (size_t)n * ((size_t)B * L * H * kDh + (size_t)B * H * ((L + 127) / 128 * 128)) * sizeof(float) : 0;
}

int moc_xattn_fwd(int dtype, const void* q, const void* k_tiles, const void* v_tiles, int64_t kv_span, int64_t su,
                  int sh, int st, const int32_t* slot_u, const float* omega, int64_t B, int64_t L, int H, int HK, int Dh, int T,
                  int NS, float scale, void* out, float* lse, hipStream_t stream) {
  return moc_xattn_fwd_split(dtype, q, k_tiles, v_tiles, kv_span, su, sh, st, slot_u, omega, B, L, H, HK, Dh, T, NS,
                             scale, out, lse, nullptr, 0, stream);
}

int moc_xattn_fwd_split(int dtype, const void* q, const void* k_tiles, const void* v_tiles, int64_t kv_span,
                        int64_t su, int sh, int st, const int32_t* slot_u, const float* omega, int64_t B, int64_t L,
                        int H, int HK, int Dh, int T, int NS, float scale, void* out, float* lse, void* workspace,
                        size_t workspace_bytes, hipStream_t stream) {
  MOC_REQUIRE(q && k_tiles && v_tiles && slot_u && omega && out && lse, MOC_ERR_ARG, "moc_xattn_fwd: null pointer");
  MOC_REQUIRE(Dh == kDh && T == kTch, MOC_ERR_UNSUPPORTED, "moc_xattn_fwd: needs head_dim 64 and 64 tokens per chapter (got %d, %d)", Dh, T);
  MOC_REQUIRE(H > 0 && HK > 0 && H % HK == 0, MOC_ERR_ARG, "moc_xattn_fwd: H=%d HK=%d", H, HK);
  MOC_REQUIRE(NS > 0 && B >= 0 && L >= 0, MOC_ERR_ARG, "moc_xattn_fwd: bad shape");
  MOC_REQUIRE(B < 65536 && H < 65536, MOC_ERR_UNSUPPORTED, "moc_xattn_fwd: grid too large");
  if (int rc = check_kv_layout("moc_xattn_fwd", dtype, kv_span, su, sh, st)) return rc;
  MOC_REQUIRE(dtype == MOC_BF16 || dtype == MOC_F32, MOC_ERR_UNSUPPORTED, "moc_xattn_fwd: dtype %d", dtype);
  if (B == 0 || L == 0) return MOC_OK;
  MOC_REQUIRE(B * H * ((L + 127) / 128) < ((int64_t)1 << 31), MOC_ERR_UNSUPPORTED, "moc_xattn_fwd: grid too large");
  const float sl2 = scale * 1.4426950408889634f;
  const int ns = workspace ? xattn_splits(dtype, B, L, H, NS) : 1;
  MOC_REQUIRE(ns == 1 || (workspace_bytes >= moc_xattn_split_workspace(dtype, B, L, H, NS) &&
                          ((uintptr_t)workspace & 15) == 0),
              MOC_ERR_ARG, "moc_xattn_fwd: workspace of %zu bytes (16-byte aligned, at least %zu)", workspace_bytes,
              moc_xattn_split_workspace(dtype, B, L, H, NS));
  const int Lp = (int)((L + 127) / 128 * 128);
  float* part = (float*)workspace;
  float* lse_part = ns > 1 ? part + (size_t)ns * B * L * H * kDh : lse;
  dim3 grid(xcd_grid(B * H * ns * ((L + 127) / 128)));
#define XF(TT, SP)                                                                                                  \
  hipLaunchKernelGGL((xattn_fwd_kernel<TT, SP>), grid, dim3(kFwdThreads), 0, stream, (const TT*)q,                  \
                     (const TT*)k_tiles, (const TT*)v_tiles, slot_u, omega, (int)B, (int)L, H, HK, NS, kv_span, su, \
                     sh, st, sl2, (TT*)out, lse_part, ns, part)
  if (dtype == MOC_BF16) {
    if (ns > 1) XF(bf16, true); else XF(bf16, false);
  } else {
    if (ns > 1) XF(float, true); else XF(float, false);
  }
#undef XF
  if (int rc = check_launch("xattn_fwd_kernel")) return rc;
  if (ns == 1) return MOC_OK;
  const dim3 mgrid((unsigned)(((int64_t)B * Lp * H * 16 + 255) / 256));
  if (dtype == MOC_BF16)
    hipLaunchKernelGGL(xattn_merge_kernel<bf16>, mgrid, dim3(256), 0, stream, part, lse_part, ns, (int)B, (int)L, Lp, H,
                       (bf16*)out, lse);
  else
    hipLaunchKernelGGL(xattn_merge_kernel<float>, mgrid, dim3(256), 0, stream, part, lse_part, ns, (int)B, (int)L, Lp, H,
                       (float*)out, lse);
  return check_launch("xattn_merge_kernel");
}

int moc_xattn_weights(int dtype, const void* q, const void* k_tiles, int64_t kv_span, int64_t su, int sh, int st,
                      const int32_t* slot_u, const float* omega, int64_t B, int64_t L, int H, int HK, int Dh, int T,
                      int NS, float scale, const float* lse, void* weights, hipStream_t stream) {
  MOC_REQUIRE(q && k_tiles && slot_u && omega && lse && weights, MOC_ERR_ARG, "moc_xattn_weights: null pointer");
  MOC_REQUIRE(Dh == kDh && T == kTch, MOC_ERR_UNSUPPORTED,
              "moc_xattn_weights: needs head_dim 64 and 64 tokens per chapter (got %d, %d)", Dh, T);
  MOC_REQUIRE(H > 0 && HK > 0 && H % HK == 0 && NS > 0 && B >= 0 && L >= 0, MOC_ERR_ARG, "moc_xattn_weights: bad shape");
  if (int rc = check_kv_layout("moc_xattn_weights", dtype, kv_span, su, sh, st)) return rc;
  MOC_REQUIRE(((uintptr_t)q & 15) == 0 && ((uintptr_t)k_tiles & 15) == 0 && ((uintptr_t)weights & 15) == 0,
              MOC_ERR_ARG, "moc_xattn_weights: q, K and the weights must be 16-byte aligned");
  if (B == 0 || L == 0) return MOC_OK;
  const int64_t blocks = B * H * ((L + 63) / 64) * NS;
  MOC_REQUIRE(blocks < ((int64_t)1 << 31), MOC_ERR_UNSUPPORTED, "moc_xattn_weights: grid too large");
  const float sl2 = scale * 1.4426950408889634f;
  if (dtype == MOC_BF16)
    hipLaunchKernelGGL(xattn_weights_kernel<bf16>, dim3((unsigned)blocks), dim3(256), 0, stream, (const bf16*)q,
                       (const bf16*)k_tiles, slot_u, omega, (int)B, (int)L, H, HK, NS, kv_span, su, sh, st, sl2, lse,
                       (bf16*)weights);
  else if (dtype == MOC_F32)
    hipLaunchKernelGGL(xattn_weights_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, stream, (const float*)q,
                       (const float*)k_tiles, slot_u, omega, (int)B, (int)L, H, HK, NS, kv_span, su, sh, st, sl2, lse,
                       (float*)weights);
  else
    return set_error(MOC_ERR_UNSUPPORTED, "moc_xattn_weights: dtype %d", dtype);
  return check_launch("xattn_weights_kernel");
}

}  // extern "C"
