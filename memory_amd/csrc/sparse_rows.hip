// Sparse attention units with many query rows (bf16): grouped or multi-query heads over few blocks.
//
// A unit is one (block of KT = 64 or 128 keys, kv head) of the plan; its rows are the query heads
// of every (token, kv head) edge that selected it, G per edge.  The one-wave-per-unit kernels of
// sparse_xattn.hip are made for tens of rows: their row loop is a serial chain (edge id -> row ->
// products -> store), which 2,048 rows per unit (16 query heads on one kv head, 128 tokens per
// block) turn into 4 us per 32 rows with two waves per SIMD.  Here the chain is pipelined (edge ids
// two row blocks ahead, rows one block ahead), K and V operands stay in registers over the loop,
// and a unit's rows can be split over several workgroups when the units alone leave CUs idle.
// With KT = 128 a caller's 128-key block is one unit with one partial row per (edge, head): half
// the partial rows, their log-sum-exps and dQ parts through HBM (they bound the combines), and one
// softmax per block, which is what the per-block mixture needs.
// Layout of K / V (and dK / dV): [batch][Tk][HK][64].  Plan ids: (batch * nblk + block) * HK + hk,
// nblk = ceil(Tk / KT); the last block of a batch row may hold 64 keys only.
// Edge e = token' * S + slot with token' = token * HK + hk; its rows are q[(token' * G + r)][64],
// r < G, and partial rows e * G + r.
//
// Measured at 16,384 tokens, 16 query heads on one kv head, 8 blocks of 128 among 512 per sequence
// (1,024 units of ~2,048 rows; 206 GFLOP forward + backward), against the 64-key units before:
// forward 289 -> 153 us, backward 531 -> 310 us, the combines 324 -> 145 us.  What bounds them now:
// the forward the partial rows and gathered q rows (537 MB, 3.5 TB/s) beside its softmax VALU work;
// the backward MFMA + VALU issue (~180 us) and the transposing LDS reads (~170 us), partly
// overlapped at two waves per SIMD.  32-row blocks took 410 us against 339 (two barriers per 32
// rows), division by run-time S and G 50 us more; leaving the dQ row stores in flight over the wait for the
// next rows changed nothing.
#include "moc_common.h"

namespace moc {

constexpr int kSrDh = 64;

typedef __attribute__((address_space(3))) void* sr_lds_ptr_t;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sr_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
// 16-byte-per-lane LDS DMA: lane l's 16 bytes at voff of the buffer land at lds + 16 l; waited for
// by the explicit vmcnt(0).
__device__ __forceinline__ void sr_dma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, const char* lds) {
  const uint32_t m0 = (uint32_t)(uintptr_t)(sr_lds_ptr_t)lds;
  asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(r), "{m0}"(m0) : "memory");
}
__device__ __forceinline__ float sr_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float sr_logw(int mode, float w) {
  if (mode == 2) return w > 0.f ? log2f(w) : -INFINITY;
  if (mode == 3) return log2f(fmaxf(w, 1e-20f));
  return 0.f;
}

// n / d for 0 <= n < 2^31 by one 32-bit high product: m = floor(2^(31 + s) / d) + 1 < 2^32 with
// s = ceil(log2 d) is exact over that range (Granlund and Montgomery, "Division by invariant
// integers using multiplication"); d = 1 passes n through.  The row loops divide several times per
// row block, and a division by a run-time value costs ~25 VALU instructions.
struct SrDiv {
  uint32_t m;
  int sh, d;
  __device__ __forceinline__ int div(int n) const { return m ? (int)(__umulhi((uint32_t)n, m) >> sh) : n; }
  __device__ __forceinline__ int mod(int n) const { return n - div(n) * d; }
};
inline SrDiv sr_div(int d) {
  if (d <= 1) return SrDiv{0u, 0, 1};
  int s = 0;
  while ((1ll << s) < d) ++s;
  return SrDiv{(uint32_t)(((1ull << (31 + s)) / (uint64_t)d) + 1), s - 1, d};
}

struct SrUnit {
  int p0, nrows, nk;   // first edge (csr), rows, valid keys
  int64_t kv0;         // element offset of the block's first key row
};

__device__ __forceinline__ SrUnit sr_unit(int gid, int u, const int32_t* __restrict__ csr_off, int G, int HK,
                                          int nblk, int64_t Tk, int KT) {
  SrUnit r;
  const int hk = gid % HK, blk = gid / HK;
  const int b = blk / nblk, c = blk % nblk;
  r.p0 = csr_off[u];
  r.nrows = (csr_off[u + 1] - r.p0) * G;
  r.nk = (int)min((int64_t)KT, Tk - (int64_t)c * KT);
  r.kv0 = (((int64_t)b * Tk + (int64_t)c * KT) * HK + hk) * kSrDh;
  return r;
}

// ------------------------------------------------------------------ forward
// S^T = K Q^T (lane = query row), softmax over the unit's keys, O^T = V^T P^T, 16 rows per wave and
// step.  K fragments in registers, V in LDS read transposed.  The output dims of a row sit four per
// 16-lane group; row-swap permutes pair the groups up so that a row goes out in 16-byte pieces.
template <int KT>
__global__ __launch_bounds__(256) void sparse_rows_fwd_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v, int64_t Tk, int HK, int nblk,
    const int32_t* __restrict__ uniq, const int32_t* __restrict__ n_uniq, const int32_t* __restrict__ csr_off,
    const int32_t* __restrict__ csr_edge, int nsplit, SrDiv S, SrDiv G, float scale_log2, bf16* __restrict__ o_part,
    float* __restrict__ lse_part) {
  using Tile = SwzTile<bf16, 64>;
  constexpr int NKB = KT / 16;
  __shared__ __attribute__((aligned(1024))) char sV[KT * 128];
  const int u = blockIdx.x / nsplit, sp = blockIdx.x % nsplit;
  if (u >= n_uniq[0]) return;
  const SrUnit un = sr_unit(uniq[u], u, csr_off, G.d, HK, nblk, Tk, KT);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int step = 64 * nsplit;
  if (sp * 64 >= un.nrows) return;   // no rows for this workgroup's first wave, hence for none
  const int64_t rs = (int64_t)HK * kSrDh;
  {
    // instruction i fills LDS rows 8 i .. 8 i + 7: lane l -> row 8 i + l / 8, physical chunk l % 8 =
    // logical chunk (l % 8) ^ (row & 7); key rows past the block's end read as zeros
    const __amdgpu_buffer_rsrc_t vr = sr_rsrc(v + un.kv0, (uint32_t)(((un.nk - 1) * rs + 64) * 2));
#pragma unroll
    for (int i = 0; i < KT / 32; ++i) {
      const int blk = i * 4 + wave, row = 8 * blk + (lane >> 3), lch = (lane & 7) ^ (row & 7);
      sr_dma16(vr, row < un.nk ? (uint32_t)((row * rs + 8 * lch) * 2) : 0xFFFFFFF0u, sV + 1024 * blk);
    }
  }
  int r0 = sp * 64 + 16 * wave;
  auto edge_at = [&](int r) { return r < un.nrows ? csr_edge[un.p0 + G.div(r)] : -1; };
  bf16x8 qf[2];
  auto load_q = [&](int e, int r, bf16x8 (&f)[2]) {
    f[0] = f[1] = zero_frag<bf16>();
    if (e >= 0) {
      const bf16* qp = q + ((int64_t)S.div(e) * G.d + G.mod(r)) * kSrDh + 8 * g;
      f[0] = Load8<bf16, bf16>::run(qp);
      f[1] = Load8<bf16, bf16>::run(qp + 32);
    }
  };
  int e_cur = edge_at(r0 + c16), e_nxt = edge_at(r0 + step + c16);
  bf16x8 kf[NKB][2];
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      kf[kb][ks] = 16 * kb < un.nk
                       ? Load8<bf16, bf16>::run(k + un.kv0 + (16 * kb + c16) * rs + 32 * ks + 8 * g)
                       : zero_frag<bf16>();
  load_q(e_cur, r0 + c16, qf);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (; r0 < un.nrows; r0 += step) {
    // the next step's rows and the edge ids of the step after it
    bf16x8 qn[2];
    load_q(e_nxt, r0 + step + c16, qn);
    const int e_nn = edge_at(r0 + 2 * step + c16);
    f32x4 st[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      st[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
      mma(st[kb], kf[kb][0], qf[0]);
      mma(st[kb], kf[kb][1], qf[1]);
    }
    // 64 keys at a time, each with its own maximum: bf16 rounds P = 2^(s - max) to 8 bits, exactly for
    // the maximum's own key alone, so one maximum over 128 keys put 128-key units at 1.018 times the
    // error of 64-key ones (outputs, 8 blocks of 128; 1.001 so, the one rounding of a partial row in
    // place of two).  The halves are scaled to each other in f32.  Cross-lane maxima and sums go by row
    // swaps: the kernel 150 -> 161 us with the second maximum, 153 with them in place of LDS permutes.
    // (Row sums of the rounded P: for the partial rows alone 0.998 of that error, but 169 us, by dot products
    // or on the matrix cores; in lse as well dK / dV come out 1.0006 times as far off.)
    if (KT > 64 && un.nk < KT) {   // a half last block: its missing keys take no part
#pragma unroll
      for (int kb = 4; kb < NKB; ++kb) st[kb] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
    float m = -INFINITY, l = 0.f;
    f32x4 o[4];
#pragma unroll
    for (int h = 0; h < KT / 64; ++h) {
      float mx = st[4 * h][0];
#pragma unroll
      for (int kb = 4 * h; kb < 4 * h + 4; ++kb)
#pragma unroll
        for (int x = 0; x < 4; ++x) mx = fmax_fast(mx, st[kb][x]);
      const float mh = quad_max_pl(mx) * scale_log2;   // scale > 0 (host check)
      const float ref = mh > -INFINITY || KT == 64 ? mh : 0.f;   // a half of -inf scores adds nothing
      float ps = 0.f;
      bf16x8 pf[2];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float p = sr_exp2(st[4 * h + kb][x] * scale_log2 - ref);
          ps += p;
          pf[kb >> 1][4 * (kb & 1) + x] = (bf16)p;
        }
      const float lh = quad_sum_pl(ps);
      f32x4 oh[4];
#pragma unroll
      for (int db = 0; db < 4; ++db) oh[db] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int db = 0; db < 4; ++db) mma(oh[db], tr_frag_mk<Tile>(sV, 64 * h + 32 * ks, 16 * db, lane), pf[ks]);
      if (h == 0) {
        m = mh;
        l = lh;
#pragma unroll
        for (int db = 0; db < 4; ++db) o[db] = oh[db];
      } else {
        const float mn = fmaxf(m, mh), fa = sr_exp2(m - mn), fb = sr_exp2(mh - mn);
        m = mn;
        l = l * fa + lh * fb;
#pragma unroll
        for (int db = 0; db < 4; ++db) o[db] = o[db] * fa + oh[db] * fb;
      }
    }
    // dims 16 db + 4 g .. + 3 of two db in one lane -> dims 16 db + 8 (g / 2) .. + 7 of one: the
    // odd 16-lane groups' db = 2 j against the even groups' db = 2 j + 1
    const float inv = 1.f / l;
    const int r = r0 + c16;
    const int64_t prow = (int64_t)e_cur * G.d + G.mod(r);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      bf16x4 ha, hb;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        ha[x] = (bf16)(o[2 * j][x] * inv);
        hb[x] = (bf16)(o[2 * j + 1][x] * inv);
      }
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      u32x2 a = __builtin_bit_cast(u32x2, ha), b = __builtin_bit_cast(u32x2, hb);
      asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %2\n\tv_permlane16_swap_b32 %1, %3\n\ts_nop 1"
                   : "+v"(a[0]), "+v"(a[1]), "+v"(b[0]), "+v"(b[1]));
      if (e_cur >= 0) {
        V16 out{{a[0], a[1], b[0], b[1]}};
        st16(o_part + prow * kSrDh + 16 * (2 * j + (g & 1)) + 8 * (g >> 1), out);
      }
    }
    if (e_cur >= 0 && g == 0) lse_part[prow] = m + log2f(l);
    qf[0] = qn[0];
    qf[1] = qn[1];
    e_cur = e_nxt;
    e_nxt = e_nn;
  }
}

// ----------------------------------------------------------------- backward
// dS [key][32 rows] (64-byte rows, 16-byte chunks XOR-swizzled by key / 4)
struct SrDsTile {
  __device__ static __forceinline__ int off(int row, int col) {
    return row * 64 + ((((col >> 3) ^ (row >> 2)) & 3) << 4) + ((col & 7) << 1);
  }
};

// KT / 32 waves, wave w owning keys 32 w .. 32 w + 31 (K / V fragments and dK / dV accumulators in
// registers) and, for dQ, dims 16 NI w .. of all KT keys (K^T fragments in registers too).  Per
// block of RB rows, taken 32 at a time: S = Q K^T, dPu = dO V^T (lane = key, rows 4 g + x), P and dS, dV^T += dO^T P,
// dK^T += Q^T dS, dS through LDS, dQ^T = K^T dS^T.  Two barriers per block (three in mode 0, whose
// per-block softmax delta is a sum over the waves' keys): the rows of the next block arrive in the
// other LDS stage meanwhile, and a block's dQ rows, staged in LDS, are stored as whole 128-byte rows
// behind the next block's first barrier.
template <int KT, int RB, bool MOE>
__global__ __launch_bounds__(2 * KT) void sparse_rows_bwd_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ dout, const bf16* __restrict__ k, const bf16* __restrict__ v,
    int64_t Tk, int HK, int nblk, const int32_t* __restrict__ uniq, const int32_t* __restrict__ n_uniq,
    const int32_t* __restrict__ csr_off, const int32_t* __restrict__ csr_edge, int nsplit, SrDiv S, SrDiv G, int mode,
    const float* __restrict__ lse_row, float* __restrict__ delta_row, const float* __restrict__ w, float scale_log2,
    float scale, bf16* __restrict__ dk, bf16* __restrict__ dv, bf16* __restrict__ dq_part, float* __restrict__ dlog,
    float* __restrict__ part, uint32_t qbytes) {
  using Tile = SwzTile<bf16, 64>;
  constexpr int NW = KT / 32;      // waves
  constexpr int NI = 4 / NW;       // 16-dim tiles of dQ per wave
  constexpr int NKS = KT / 32;     // 32-key steps of the dQ product
  constexpr int NH = RB / 32;      // 32-row parts of a block
  constexpr int NR = RB / 8 / NW;  // row DMA instructions (8 rows each) per wave, for Q and for dO
  constexpr int kHalf = RB * 128, kStage = 2 * kHalf;   // Q rows, then dO rows
  // two row stages; at the start the K tile, at the end dK / dV staging
  __shared__ __attribute__((aligned(1024))) char sRows[2 * kStage];
  __shared__ __attribute__((aligned(1024))) char sDQ[RB * 128];
  __shared__ __attribute__((aligned(16))) char sDS[NH][KT * 64];
  __shared__ __attribute__((aligned(16))) float sC[2][RB], sDel[2][RB], sWr[2][RB];
  __shared__ float sPart[2][NW][RB];
  __shared__ int sEr[2][RB];
  static_assert(KT * 128 <= 2 * kStage && (RB == 32 || RB == 64), "K tile / staging fits the row stages");
  const int u = blockIdx.x / nsplit, sp = blockIdx.x % nsplit;
  if (u >= n_uniq[0]) return;
  const SrUnit un = sr_unit(uniq[u], u, csr_off, G.d, HK, nblk, Tk, KT);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int key0 = 32 * wave;
  const bool live = key0 < un.nk;   // this wave's keys exist (a half last block)
  const int64_t rs = (int64_t)HK * kSrDh;
  const int nb = (un.nrows + RB - 1) / RB;
  const int b0 = (int)((int64_t)nb * sp / nsplit), b1 = (int)((int64_t)nb * (sp + 1) / nsplit);
  const __amdgpu_buffer_rsrc_t qr = sr_rsrc(q, qbytes), dr = sr_rsrc(dout, qbytes);
  const int dlc = (lane & 7) ^ (lane >> 3);   // source chunk of this lane's DMA destination (row & 7 = lane / 8)

  // K tile -> LDS, then this wave's fragments
  bf16x8 kf[2][2], vf[2][2], kt[NI][NKS];
  {
    const __amdgpu_buffer_rsrc_t kr = sr_rsrc(k + un.kv0, (uint32_t)(((un.nk - 1) * rs + 64) * 2));
#pragma unroll
    for (int i = 0; i < KT / 8 / NW; ++i) {
      const int blk = i * NW + wave, row = 8 * blk + (lane >> 3);
      sr_dma16(kr, row < un.nk ? (uint32_t)((row * rs + 8 * dlc) * 2) : 0xFFFFFFF0u, sRows + 1024 * blk);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        vf[j][ks] = live ? Load8<bf16, bf16>::run(v + un.kv0 + (key0 + 16 * j + c16) * rs + 32 * ks + 8 * g)
                         : zero_frag<bf16>();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) kf[j][ks] = Tile::frag(sRows, key0 + 16 * j + c16, 32 * ks + 8 * g);
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) kt[i][ks] = tr_frag_mk<Tile>(sRows, 32 * ks, 16 * (NI * wave + i), lane);
    __syncthreads();
  }

  f32x4 dkt[4][2], dvt[4][2];   // [db][j]: lane = key key0 + 16 j + c16, dims 16 db + 4 g + x
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      dkt[db][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      dvt[db][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  // e_dma: the edge ids of the rows this lane's DMAs move, e_con of the constants' row (wave 0,
  // lane < RB)
  int e_dma[NR], e_con;
  auto edges = [&](int blk, int (&ed)[NR], int& ec) {
    const int r0 = RB * blk;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int r = r0 + 8 * (NR * wave + i) + (lane >> 3);
      ed[i] = blk < b1 && r < un.nrows ? csr_edge[un.p0 + G.div(r)] : -1;
    }
    const int r = r0 + (lane & (RB - 1));
    ec = wave == 0 && blk < b1 && r < un.nrows ? csr_edge[un.p0 + G.div(r)] : -1;
  };
  float c_c = -INFINITY, c_del = 0.f, c_w = 0.f;
  int c_er = -1;
  auto fetch = [&](int blk, int par) {   // rows and constants of block blk, its ids in e_dma / e_con
    char* st = sRows + par * kStage;
    const int r0 = RB * blk;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int r = r0 + 8 * (NR * wave + i) + (lane >> 3);
      const uint32_t off = e_dma[i] >= 0
                               ? (uint32_t)((((int64_t)S.div(e_dma[i]) * G.d + G.mod(r)) * kSrDh + 8 * dlc) * 2)
                               : 0xFFFFFFF0u;   // past the buffer: zeros
      sr_dma16(qr, off, st + 1024 * (NR * wave + i));
      sr_dma16(dr, off, st + kHalf + 1024 * (NR * wave + i));
    }
    c_c = -INFINITY;
    c_del = c_w = 0.f;
    c_er = -1;
    if (e_con >= 0) {   // wave 0 only
      const int r = G.mod(r0 + (lane & (RB - 1)));
      c_er = e_con * G.d + r;
      if (MOE) {
        c_c = -lse_row[c_er];
        c_w = w[e_con];
      } else {
        const int64_t trow = (int64_t)S.div(e_con) * G.d + r;
        c_c = sr_logw(mode, w ? w[e_con] : 1.f) - lse_row[trow];
        c_del = -delta_row[trow];
      }
    }
  };
  auto store_dq = [&](int par) {
#pragma unroll
    for (int t = 0; t < RB / (8 * NW); ++t) {
      const int cid = threadIdx.x + 64 * NW * t, row = cid >> 3, ch = cid & 7;
      const int er = sEr[par][row];
      if (er >= 0)
        *reinterpret_cast<bf16x8*>(dq_part + (int64_t)er * kSrDh + 8 * ch) =
            *reinterpret_cast<const bf16x8*>(sDQ + Tile::off(row, 8 * ch));
    }
  };
  if (b0 < b1) {
    edges(b0, e_dma, e_con);
    fetch(b0, 0);
    edges(b0 + 1, e_dma, e_con);
  }
  for (int blk = b0; blk < b1; ++blk) {
    const int par = (blk - b0) & 1;
    const char* sQ = sRows + par * kStage;
    const char* sD = sQ + kHalf;
    const int nh = NH == 1 || un.nrows - RB * blk > 32 ? NH : 1;   // parts that hold rows
    if (wave == 0 && lane < RB) {
      sC[par][lane] = c_c;
      sDel[par][lane] = c_del;
      sWr[par][lane] = c_w;
      sEr[par][lane] = c_er;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's rows of the block have landed
    __syncthreads();   // (A) rows and constants visible; the previous block's dQ rows staged
    if (blk > b0) store_dq(par ^ 1);
    if (blk + 1 < b1) {
      fetch(blk + 1, par ^ 1);
      edges(blk + 2, e_dma, e_con);
    }
    for (int h = 0; h < nh; ++h) {
    const int ro = 32 * h;
    f32x4 sc[2][2], dp[2][2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const f32x4 nd = MOE ? f32x4{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4*>(&sDel[par][ro + 16 * qb + 4 * g]);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        sc[qb][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        dp[qb][j] = nd;   // joint modes: dPu - delta
      }
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        const bf16x8 qa = Tile::frag(sQ, ro + 16 * qb + c16, 32 * ks + 8 * g);
        const bf16x8 da = Tile::frag(sD, ro + 16 * qb + c16, 32 * ks + 8 * g);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          mma(sc[qb][j], qa, kf[j][ks]);
          mma(dp[qb][j], da, vf[j][ks]);
        }
      }
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const f32x4 c = *reinterpret_cast<const f32x4*>(&sC[par][ro + 16 * qb + 4 * g]);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x)
          sc[qb][j][x] = live ? sr_exp2(__builtin_fmaf(sc[qb][j][x], scale_log2, c[x])) : 0.f;
    }
    if (MOE) {
      // the block's softmax delta per row: this wave's 32 keys, then the waves in order
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          float t = sc[qb][0][x] * dp[qb][0][x] + sc[qb][1][x] * dp[qb][1][x];
          t += __shfl_xor(t, 1, 16);
          t += __shfl_xor(t, 2, 16);
          t += __shfl_xor(t, 4, 16);
          t += __shfl_xor(t, 8, 16);
          if (c16 == 0) sPart[0][wave][ro + 16 * qb + 4 * g + x] = t;
        }
      __syncthreads();
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        f32x4 del = *reinterpret_cast<const f32x4*>(&sPart[0][0][ro + 16 * qb + 4 * g]);
#pragma unroll
        for (int i = 1; i < NW; ++i) del += *reinterpret_cast<const f32x4*>(&sPart[0][i][ro + 16 * qb + 4 * g]);
        const f32x4 wr = *reinterpret_cast<const f32x4*>(&sWr[par][ro + 16 * qb + 4 * g]);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            dp[qb][j][x] -= del[x];
            sc[qb][j][x] *= wr[x];
          }
      }
      if (wave == 0 && lane < 32) {
        const int er = sEr[par][ro + lane];
        float t = sPart[0][0][ro + lane];
#pragma unroll
        for (int i = 1; i < NW; ++i) t += sPart[0][i][ro + lane];
        if (er >= 0) delta_row[er] = t;
      }
    }
    bf16x8 pa[2], sa[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        float rsum = 0.f;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float ds = sc[qb][j][x] * dp[qb][j][x];
          rsum += ds;
          pa[j][4 * qb + x] = (bf16)sc[qb][j][x];
          sa[j][4 * qb + x] = (bf16)ds;
        }
        if (!MOE && dlog) {
          rsum += __shfl_xor(rsum, 1, 16);
          rsum += __shfl_xor(rsum, 2, 16);
          rsum += __shfl_xor(rsum, 4, 16);
          rsum += __shfl_xor(rsum, 8, 16);
          if (c16 == 0) sPart[1][wave][ro + 16 * qb + 4 * g + x] = rsum;
        }
      }
    // dS key-major for dQ
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int key = key0 + 16 * j + c16;
      const bf16x4 lo = {sa[j][0], sa[j][1], sa[j][2], sa[j][3]};
      const bf16x4 hi = {sa[j][4], sa[j][5], sa[j][6], sa[j][7]};
      *reinterpret_cast<bf16x4*>(sDS[h] + SrDsTile::off(key, 4 * g)) = lo;
      *reinterpret_cast<bf16x4*>(sDS[h] + SrDsTile::off(key, 16 + 4 * g)) = hi;
    }
    // dV^T += dO^T P, dK^T += Q^T dS
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      const bf16x8 ad = tr_frag_mk<Tile>(sD, ro, 16 * db, lane);
      const bf16x8 aq = tr_frag_mk<Tile>(sQ, ro, 16 * db, lane);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        mma(dvt[db][j], ad, pa[j]);
        mma(dkt[db][j], aq, sa[j]);
      }
    }
    }
    __syncthreads();   // (B) dS and the row sums visible; the block's rows are read
    if (!MOE && dlog && wave == 0 && lane < 32 * nh) {
      const int er = sEr[par][lane];
      float t = sPart[1][0][lane];
#pragma unroll
      for (int i = 1; i < NW; ++i) t += sPart[1][i][lane];
      if (er >= 0) dlog[er] = t;
    }
    // dQ^T = K^T dS^T: lane = row 32 h + 16 qb + c16, dims 16 (NI wave + i) + 4 g + x
    for (int h = 0; h < nh; ++h) {
    f32x4 dq[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) dq[i][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        const bf16x8 bs = tr_frag_mk<SrDsTile>(sDS[h], 32 * ks, 16 * qb, lane);
#pragma unroll
        for (int i = 0; i < NI; ++i) mma(dq[i][qb], kt[i][ks], bs);
      }
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const f32x4 t = dq[i][qb] * scale;
        const bf16x4 b = {(bf16)t[0], (bf16)t[1], (bf16)t[2], (bf16)t[3]};
        *reinterpret_cast<bf16x4*>(sDQ + Tile::off(32 * h + 16 * qb + c16, 16 * (NI * wave + i) + 4 * g)) = b;
      }
    }
  }
  __syncthreads();
  if (b0 < b1) store_dq((b1 - 1 - b0) & 1);
  if (nsplit > 1) {
    // f32 partial dK, dV in accumulator order, added in split order by sparse_rows_reduce_kernel
    f32x4* p = reinterpret_cast<f32x4*>(part) + ((int64_t)blockIdx.x * NW + wave) * 16 * 64 + lane;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        p[(db * 2 + j) * 64] = dkt[db][j];
        p[(8 + db * 2 + j) * 64] = dvt[db][j];
      }
    return;
  }
  // dK = scale (dK^T)^T, dV: staged as [key][dim] rows in this wave's 4 KB (the row stages are free:
  // every wave is past the last block), stored as whole 128-byte rows
  char* sW = sRows + 4096 * wave;
#pragma unroll
  for (int which = 0; which < 2; ++which) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        bf16x4 a;
#pragma unroll
        for (int x = 0; x < 4; ++x) a[x] = (bf16)(which == 0 ? dkt[db][j][x] * scale : dvt[db][j][x]);
        *reinterpret_cast<bf16x4*>(sW + Tile::off(16 * j + c16, 16 * db + 4 * g)) = a;
      }
    wave_lds_sync();
    bf16* dst = (which == 0 ? dk : dv) + un.kv0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = 8 * i + (lane >> 3), ch = lane & 7;
      if (live)
        *reinterpret_cast<bf16x8*>(dst + (key0 + key) * rs + 8 * ch) =
            *reinterpret_cast<const bf16x8*>(sW + Tile::off(key, 8 * ch));
    }
    wave_lds_sync();
  }
}

// dK / dV of a unit from its splits' partials, in split order: grid (unit, 16 accumulator tiles),
// wave w the keys of the backward's wave w; lane = key, four consecutive dims per 8-byte store.
template <int KT>
__global__ __launch_bounds__(2 * KT) void sparse_rows_reduce_kernel(const float* __restrict__ part, int nsplit,
                                                                    int64_t Tk, int HK, int nblk,
                                                                    const int32_t* __restrict__ uniq,
                                                                    const int32_t* __restrict__ n_uniq,
                                                                    const int32_t* __restrict__ csr_off, float scale,
                                                                    bf16* __restrict__ dk, bf16* __restrict__ dv) {
  constexpr int NW = KT / 32;
  const int u = blockIdx.x, i = blockIdx.y;
  if (u >= n_uniq[0]) return;
  const SrUnit un = sr_unit(uniq[u], u, csr_off, 1, HK, nblk, Tk, KT);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  if (32 * wave >= un.nk) return;
  const int64_t rs = (int64_t)HK * kSrDh;
  const f32x4* p = reinterpret_cast<const f32x4*>(part) + (((int64_t)u * nsplit * NW + wave) * 16 + i) * 64 + lane;
  f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int sp = 0; sp < nsplit; ++sp) s += p[(int64_t)sp * NW * 16 * 64];
  const int db = (i & 7) >> 1, j = i & 1;
  if (i < 8) s *= scale;
  bf16x4 o;
#pragma unroll
  for (int x = 0; x < 4; ++x) o[x] = (bf16)s[x];
  bf16* dst = (i < 8 ? dk : dv) + un.kv0 + (32 * wave + 16 * j + c16) * rs + 16 * db + 4 * g;
  *reinterpret_cast<bf16x4*>(dst) = o;
}

// Plan ids of per-head block choices: out[(tok * HK + hk) * S + s] = (b * nblk + c) * HK + hk for
// c = idx[tok][hk][s] in [0, nblk), -1 otherwise (skipped), b = tok / tok_per_batch (0 when K / V
// are shared by the batch).  The comparison is on the caller's id type.
template <typename I>
__global__ __launch_bounds__(256) void sparse_pack_ids_kernel(const I* __restrict__ idx, int64_t n, int heads, int HK,
                                                              int S, int64_t tok_per_batch, int64_t nblk,
                                                              int per_batch, int32_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int s = (int)(i % S);
  const int64_t t = i / S;
  const int hk = (int)(t % HK);
  const int64_t tok = t / HK;
  const int64_t c = (int64_t)idx[(tok * heads + hk) * S + s];
  const int64_t b = per_batch ? tok / tok_per_batch : 0;
  out[i] = c >= 0 && c < nblk ? (int32_t)((b * nblk + c) * HK + hk) : -1;
}

// dlog[e, r] -= P_e sum_e' dlog[e', r] over the valid slots of a (token, row), P_e = w_e 2^lse_e / 2^lse_joint:
// the joint softmax's log-weight gradients P_e (dP_e - D) add up to zero, and what they add up to is the
// error of D = dO . out, whose out is rounded to bf16.  That error was all of dw's (1.13e-3 in bf16 over 8
// blocks of 128 keys, a token with one valid block moved by 0.8 where the largest dw is 27; 3e-7 now), and
// 128-key units' roundings of out put it at 1.02 to 1.05 times that of 64-key ones.  Thread = (token, row).
__global__ __launch_bounds__(256) void sparse_dlog_center_kernel(float* __restrict__ dlog,
                                                                 const float* __restrict__ lse_part,
                                                                 const float* __restrict__ lse_joint,
                                                                 const float* __restrict__ w,
                                                                 const int32_t* __restrict__ edge_u, int mode, int S,
                                                                 int rpe, int64_t rows) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= rows) return;
  const int64_t tok = i / rpe, r = i - tok * rpe;
  float sum = 0.f;
  for (int s = 0; s < S; ++s)
    if (edge_u[tok * S + s] >= 0) sum += dlog[(tok * S + s) * rpe + r];
  const float lj = lse_joint[i];
  for (int s = 0; s < S; ++s) {
    const int64_t e = tok * S + s, at = e * rpe + r;
    if (edge_u[e] >= 0) dlog[at] -= sr_exp2(lse_part[at] + sr_logw(mode, w[e]) - lj) * sum;
  }
}

}  // namespace moc

using namespace moc;

namespace {

// Splits of a unit's rows: units alone fill the chip from about two workgroups per CU on; below
// that a unit is split as long as a split keeps kSrSplitRows rows (its K / V operands and, in the
// backward, 16 KB of f32 partials per wave and split are per split): 64 units of 1,024 rows, forward
// + backward of a call 100 us at 256 rows, 103 at 128, 127 at 512.
constexpr int kSrSplitRows = 256;
int sr_splits(int64_t rows, int64_t max_u, int64_t want) {
  if (max_u <= 0) return 1;
  const int64_t per_unit = rows / max_u;
  int64_t n = (want + max_u - 1) / max_u;
  if (n > per_unit / kSrSplitRows) n = per_unit / kSrSplitRows;
  return (int)(n < 1 ? 1 : n > 64 ? 64 : n);
}
constexpr int64_t kSrFwdWgs = 2048, kSrBwdWgs = 1024;
constexpr int64_t kSrMaxIds = 16384;   // what moc_chapter_plan takes
// Rows per unit (a lower bound: max_u counts every unit the plan could hold) from which the
// pipelined kernels win over the one-wave-per-unit ones of sparse_xattn.hip, forward + backward of
// a call (2,048 tokens, 8 slots, G = 4 on 4 kv heads): 32 rows 226 / 225 us, 48 rows 183 / 189,
// 128 rows 141 / 157, 1,024 rows 140 / 260; at 16 rows (G = 1) 141 / 131.
constexpr int64_t kSrMinRows = 48;
// A 128-key block as one unit instead of two 64-key ones wins from fewer rows on: 16 rows
// 189 / 205 us, 48 rows 122 / 136 (G = 1) and 252 / 322 (G = 4), 1,024 rows 170 / 316 (G = 16).
constexpr int64_t kSrMinRows128 = 16;
// Bytes of partial rows up to which all kv heads (and, per-block mixture, all slots) run at once: per-head
// segments hold one head's at a time, which a call of a million tokens with 64 slots on 16 kv heads needs
// (8 GiB a head, 128 GiB packed, in the forward and again in the backward).
constexpr int64_t kSrPartBytes = (int64_t)16 << 30;
bool sr_many_rows(int64_t rows, int64_t max_u, int64_t least) { return max_u > 0 && rows >= least * max_u; }
bool sr_use_rows(int dtype, int KT, int64_t rows, int64_t max_u, float scale) {
  return dtype == MOC_BF16 && (KT == 128 || (scale > 0.f && sr_many_rows(rows, max_u, kSrMinRows)));
}

int sr_check(const char* who, int dtype, const void* q, const void* k, const void* v, int64_t ntok, int64_t Bk,
             int64_t Tk, int HK, int G, int KT, int64_t max_u, int S) {
  MOC_REQUIRE(dtype == MOC_BF16 || dtype == MOC_F32, MOC_ERR_UNSUPPORTED, "%s: dtype %d", who, dtype);
  MOC_REQUIRE(KT == 64 || (KT == 128 && dtype == MOC_BF16), MOC_ERR_ARG, "%s: %d keys per block (64, bf16 also 128)",
              who, KT);
  MOC_REQUIRE(Bk > 0 && Tk > 0 && Tk % 64 == 0 && HK > 0 && G > 0 && S > 0 && max_u >= 0 && ntok >= 0, MOC_ERR_ARG,
              "%s: batches %lld, keys %lld (a multiple of 64), HK=%d, G=%d, S=%d", who, (long long)Bk, (long long)Tk, HK,
              G, S);
  const int64_t nblk = (Tk + KT - 1) / KT, es = dtype == MOC_F32 ? 4 : 2;
  MOC_REQUIRE(Bk * nblk * HK < ((int64_t)1 << 31) && ntok * S * G < ((int64_t)1 << 31) &&
                  ntok * G * kSrDh * es < ((int64_t)1 << 32) * (es / 2) - 16,
              MOC_ERR_UNSUPPORTED, "%s: too many blocks or rows", who);
  // (the float32 kernels take rows at any 4-byte boundary, such as a view into a flat buffer)
  MOC_REQUIRE(dtype == MOC_F32 || (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15) == 0, MOC_ERR_ARG,
              "%s: bf16 q, k and v must be 16-byte aligned", who);
  return MOC_OK;
}

}  // namespace

extern "C" {

int moc_sparse_pack_ids(const void* idx, int idx_bytes, int64_t ntok, int64_t tok_per_batch, int heads, int HK, int S,
                        int64_t nblk, int per_batch, int32_t* out, hipStream_t stream) {
  MOC_REQUIRE(idx && out, MOC_ERR_ARG, "moc_sparse_pack_ids: null pointer");
  MOC_REQUIRE((idx_bytes == 4 || idx_bytes == 8) && ntok >= 0 && tok_per_batch > 0 && HK > 0 && heads >= HK && S > 0 &&
                  nblk > 0,
              MOC_ERR_ARG, "moc_sparse_pack_ids: ids of %d bytes, %d heads for HK=%d, S=%d", idx_bytes, heads, HK, S);
  const int64_t n = ntok * HK * S;
  MOC_REQUIRE(n < ((int64_t)1 << 31), MOC_ERR_UNSUPPORTED, "moc_sparse_pack_ids: %lld edges", (long long)n);
  if (n == 0) return MOC_OK;
  const dim3 grid((unsigned)((n + 255) / 256));
  if (idx_bytes == 4)
    hipLaunchKernelGGL(sparse_pack_ids_kernel<int32_t>, grid, dim3(256), 0, stream, (const int32_t*)idx, n, heads, HK, S,
                       tok_per_batch, nblk, per_batch, out);
  else
    hipLaunchKernelGGL(sparse_pack_ids_kernel<int64_t>, grid, dim3(256), 0, stream, (const int64_t*)idx, n, heads, HK, S,
                       tok_per_batch, nblk, per_batch, out);
  return check_launch("sparse_pack_ids_kernel");
}

int moc_sparse_packed_block(int dtype, int64_t ntok, int G, int64_t S, int64_t Bk, int64_t Tk, int HK, int block_size,
                            int mode, float scale) {
  if (ntok < 0 || G <= 0 || S <= 0 || Bk <= 0 || Tk <= 0 || HK <= 0 || block_size < 64 || block_size % 64 != 0)
    return 0;
  const int m = block_size / 64;
  auto fits = [&](int kt) {
    const int64_t ids = Bk * ((Tk + kt - 1) / kt) * HK, edges = ntok * S * (block_size / kt);
    const int64_t bytes = edges * G * kSrDh * (dtype == MOC_F32 ? 4 : 2);
    return ids <= kSrMaxIds && edges * G < ((int64_t)1 << 31) && ntok * G * 256 < ((int64_t)1 << 32) - 16 &&
           (bytes <= kSrPartBytes || (HK == 1 && mode != 0));   // (one head, joint: its segment holds them too)
  };
  // A block's own softmax (mode 0) spans one unit at 128 keys and is otherwise the caller's one
  // call per slot; a joint softmax over 128-key units halves the partial rows, at a unit's cost in
  // registers and LDS that only many rows repay (kSrMinRows128).
  if (dtype == MOC_BF16 && scale > 0.f && m % 2 == 0 && (mode != 0 || m == 2) && fits(128)) {
    const int64_t ids = Bk * ((Tk + 127) / 128) * HK, edges = ntok * S * (m / 2);
    if (mode == 0 || sr_many_rows(edges * G, edges < ids ? edges : ids, kSrMinRows128)) return 128;
  }
  if (mode == 0 && m > 1) return 0;
  return fits(64) ? 64 : 0;
}

int moc_sparse_packed_fwd(int dtype, const void* q, int64_t ntok, int G, const void* k, const void* v, int64_t Bk,
                          int64_t Tk, int HK, int KT, const int32_t* uniq, const int32_t* n_uniq,
                          const int32_t* csr_off, const int32_t* csr_edge, int64_t max_u, int S, float scale,
                          void* o_part, float* lse_part, hipStream_t stream) {
  const char* who = "moc_sparse_packed_fwd";
  MOC_REQUIRE(q && k && v && uniq && n_uniq && csr_off && csr_edge && o_part && lse_part, MOC_ERR_ARG,
              "%s: null pointer", who);
  if (int rc = sr_check(who, dtype, q, k, v, ntok, Bk, Tk, HK, G, KT, max_u, S)) return rc;
  if (max_u == 0 || ntok == 0) return MOC_OK;
  const int64_t rows = ntok * S * G;
  if (!sr_use_rows(dtype, KT, rows, max_u, scale))
    return sparse_fwd_launch(dtype, q, G, k, v, (int64_t)64 * HK * kSrDh, kSrDh, (int64_t)HK * kSrDh, 1, uniq, n_uniq,
                             csr_off, csr_edge, max_u, S, 0, 1, 0, G, scale, nullptr, o_part, lse_part, stream, who,
                             nullptr, HK);
  MOC_REQUIRE(((uintptr_t)o_part & 15) == 0, MOC_ERR_ARG, "%s: o_part must be 16-byte aligned", who);
  MOC_REQUIRE(scale > 0.f, MOC_ERR_UNSUPPORTED, "%s: scale %g with 128-key blocks (needs > 0)", who, (double)scale);
  const int nblk = (int)((Tk + KT - 1) / KT);
  const int ns = sr_splits(rows, max_u, kSrFwdWgs);
  const dim3 grid((unsigned)(max_u * ns));
  const float sl2 = scale * 1.4426950408889634f;
#define SR_FWD(N)                                                                                                  \
  hipLaunchKernelGGL(sparse_rows_fwd_kernel<N>, grid, dim3(256), 0, stream, (const bf16*)q, (const bf16*)k,        \
                     (const bf16*)v, Tk, HK, nblk, uniq, n_uniq, csr_off, csr_edge, ns, sr_div(S), sr_div(G), sl2, (bf16*)o_part, \
                     lse_part)
  if (KT == 64) SR_FWD(64); else SR_FWD(128);
#undef SR_FWD
  return check_launch("sparse_rows_fwd_kernel");
}

size_t moc_sparse_packed_bwd_workspace(int dtype, int64_t ntok, int G, int S, int KT, int64_t max_u, float scale) {
  if (max_u <= 0 || dtype != MOC_BF16) return 0;
  const int64_t rows = ntok * S * G;
  if (!sr_use_rows(dtype, KT, rows, max_u, scale)) return (size_t)max_u * 32 * sizeof(int32_t);   // row table
  const int ns = sr_splits(rows, max_u, kSrBwdWgs);
  return ns > 1 ? (size_t)max_u * ns * KT * 64 * 2 * sizeof(float) : 0;
}

int moc_sparse_packed_bwd(int dtype, const void* q, const void* dout, int64_t ntok, int G, const void* k, const void* v,
                          int64_t Bk, int64_t Tk, int HK, int KT, const int32_t* uniq, const int32_t* n_uniq,
                          const int32_t* csr_off, const int32_t* csr_edge, int64_t max_u, int S, int mode,
                          const float* lse_row, float* delta_row, const float* w, float scale, void* dk, void* dv,
                          void* dq_part, float* dlog, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  const char* who = "moc_sparse_packed_bwd";
  MOC_REQUIRE(q && dout && k && v && uniq && n_uniq && csr_off && csr_edge && lse_row && delta_row && dk && dv &&
                  dq_part,
              MOC_ERR_ARG, "%s: null pointer", who);
  if (int rc = sr_check(who, dtype, q, k, v, ntok, Bk, Tk, HK, G, KT, max_u, S)) return rc;
  MOC_REQUIRE(mode >= 0 && mode <= 3 && (mode == 1 || w), MOC_ERR_ARG, "%s: mode %d / weights", who, mode);
  const size_t need = moc_sparse_packed_bwd_workspace(dtype, ntok, G, S, KT, max_u, scale);
  MOC_REQUIRE(workspace_bytes >= need && (need == 0 || workspace) && ((uintptr_t)workspace & 15) == 0, MOC_ERR_ARG,
              "%s: workspace of %zu bytes, needs %zu (16-byte aligned)", who, workspace_bytes, need);
  if (max_u == 0 || ntok == 0) return MOC_OK;
  const int64_t rows = ntok * S * G, rs = (int64_t)HK * kSrDh;
  if (!sr_use_rows(dtype, KT, rows, max_u, scale)) {
    int32_t* tab = dtype == MOC_BF16 ? (int32_t*)workspace : nullptr;
    if (tab)
      if (int rc = moc_plan_row_table(n_uniq, csr_off, csr_edge, max_u, 32, tab, stream)) return rc;
    return sparse_bwd_launch(dtype, q, dout, ntok, G, k, v, 64 * rs, kSrDh, rs, 1, kSrDh, uniq, n_uniq, csr_off, csr_edge,
                             max_u, S, 0, 1, 0, G, mode, lse_row, delta_row, w, scale, dk, dv, 64 * rs, kSrDh, rs,
                             dq_part, dlog, tab, stream, who, HK);
  }
  MOC_REQUIRE(((uintptr_t)dout & 15) == 0 && ((uintptr_t)dk & 15) == 0 && ((uintptr_t)dv & 15) == 0 &&
                  ((uintptr_t)dq_part & 15) == 0,
              MOC_ERR_ARG, "%s: dout, dk, dv and dq_part must be 16-byte aligned", who);
  MOC_REQUIRE(scale > 0.f, MOC_ERR_UNSUPPORTED, "%s: scale %g with 128-key blocks (needs > 0)", who, (double)scale);
  const int64_t qbytes = ntok * G * kSrDh * 2;
  const int nblk = (int)((Tk + KT - 1) / KT);
  const int ns = sr_splits(rows, max_u, kSrBwdWgs);
  const dim3 grid((unsigned)(max_u * ns));
  const float sl2 = scale * 1.4426950408889634f;
#define SR_BWD(N, R, M)                                                                                              \
  hipLaunchKernelGGL((sparse_rows_bwd_kernel<N, R, M>), grid, dim3(2 * N), 0, stream, (const bf16*)q, (const bf16*)dout, \
                     (const bf16*)k, (const bf16*)v, Tk, HK, nblk, uniq, n_uniq, csr_off, csr_edge, ns, sr_div(S), sr_div(G), mode, \
                     lse_row, delta_row, w, sl2, scale, (bf16*)dk, (bf16*)dv, (bf16*)dq_part, dlog,                 \
                     (float*)workspace, (uint32_t)qbytes)
  if (KT == 64) {
    if (mode == 0) SR_BWD(64, 32, true); else SR_BWD(64, 32, false);
  } else {
    if (mode == 0) SR_BWD(128, 64, true); else SR_BWD(128, 64, false);
  }
#undef SR_BWD
  if (int rc = check_launch("sparse_rows_bwd_kernel")) return rc;
  if (ns == 1) return MOC_OK;
#define SR_RED(N)                                                                                                    \
  hipLaunchKernelGGL(sparse_rows_reduce_kernel<N>, dim3((unsigned)max_u, 16), dim3(2 * N), 0, stream,                    \
                     (const float*)workspace, ns, Tk, HK, nblk, uniq, n_uniq, csr_off, scale, (bf16*)dk, (bf16*)dv)
  if (KT == 64) SR_RED(64); else SR_RED(128);
#undef SR_RED
  return check_launch("sparse_rows_reduce_kernel");
}

int moc_sparse_dlog_center(float* dlog, const float* lse_part, const float* lse_joint, const float* w,
                           const int32_t* edge_u, int mode, int S, int rpe, int64_t ntok, hipStream_t stream) {
  MOC_REQUIRE(dlog && lse_part && lse_joint && w && edge_u, MOC_ERR_ARG, "moc_sparse_dlog_center: null pointer");
  MOC_REQUIRE((mode == 2 || mode == 3) && S > 0 && rpe > 0 && ntok >= 0 && ntok * rpe < ((int64_t)1 << 38), MOC_ERR_ARG,
              "moc_sparse_dlog_center: mode %d, S=%d, %d rows of %lld tokens", mode, S, rpe, (long long)ntok);
  if (ntok == 0) return MOC_OK;
  const int64_t rows = ntok * rpe;
  hipLaunchKernelGGL(sparse_dlog_center_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, stream, dlog, lse_part,
                     lse_joint, w, edge_u, mode, S, rpe, rows);
  return check_launch("sparse_dlog_center_kernel");
}

}  // extern "C"
