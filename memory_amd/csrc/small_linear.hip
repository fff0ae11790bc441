// y = x W^T for few rows (decode: one token per sequence through q_proj / o_proj,
// memory_attention.py:140-143, :241, :456): x [M][K], W [N][K] bf16, M <= 256.
//
// A library GEMM tiles such a product into a handful of output tiles, each walking the whole
// K dimension on its own, so the launch is one long chain of dependent loads.  Here a
// workgroup owns one 16 x 16 output tile (64 rows x 768 columns make 192 workgroups), and its
// 4 waves split K: each wave issues all of its x and W fragment loads before its first MFMA
// (v_mfma_f32_16x16x32_bf16), and the four partial tiles are added through LDS in a fixed
// order.  Bound: the latency of one round of loads (each W slice is re-read by the M / 16 row
// tiles, mostly from L2).

#include "moc_common.h"

namespace moc {

constexpr int kSlWaves = 4;
constexpr int kSlTiles = 1;       // 16-row MFMA tiles per workgroup
constexpr int kSlRows = 16 * kSlTiles;
constexpr int kSlChunks = 6;      // 32-wide K chunks a wave holds in registers at once

template <typename TO>
__device__ __forceinline__ void small_linear_tile(const bf16* __restrict__ x, int M, int K, const bf16* __restrict__ W,
                                                  int N, TO* __restrict__ y) {
  __shared__ f32x4 red[kSlWaves][kSlTiles][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c16 = lane & 15;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * kSlRows;
  const int kw = K / kSlWaves;                 // this wave's K range: [wave * kw, wave * kw + kw)
  const int nch = kw / 32;
  f32x4 acc[kSlTiles];
#pragma unroll
  for (int mt = 0; mt < kSlTiles; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16* wrow = W + (size_t)(n0 + c16) * K + wave * kw + 8 * g;
  for (int c0 = 0; c0 < nch; c0 += kSlChunks) {
    bf16x8 a[kSlChunks][kSlTiles], b[kSlChunks];
#pragma unroll
    for (int j = 0; j < kSlChunks; ++j) {
      const bool live = c0 + j < nch;
      const int k = 32 * (c0 + j);
      b[j] = live ? *reinterpret_cast<const bf16x8*>(wrow + k) : bf16x8{};
#pragma unroll
      for (int mt = 0; mt < kSlTiles; ++mt) {
        const int m = m0 + 16 * mt + c16;
        a[j][mt] = (live && m < M) ? *reinterpret_cast<const bf16x8*>(x + (size_t)m * K + wave * kw + k + 8 * g)
                                   : bf16x8{};
      }
    }
#pragma unroll
    for (int j = 0; j < kSlChunks; ++j)
#pragma unroll
      for (int mt = 0; mt < kSlTiles; ++mt) mma(acc[mt], a[j][mt], b[j]);
  }
#pragma unroll
  for (int mt = 0; mt < kSlTiles; ++mt) red[wave][mt][lane] = acc[mt];
  __syncthreads();
  // wave t (< kSlTiles) sums tile t of its lane over the waves, in wave order
  const int mt = threadIdx.x >> 6;
  if (mt >= kSlTiles) return;
  f32x4 s = red[0][mt][lane];
#pragma unroll
  for (int w = 1; w < kSlWaves; ++w) {
    const f32x4 v = red[w][mt][lane];
    s = f32x4{s[0] + v[0], s[1] + v[1], s[2] + v[2], s[3] + v[3]};
  }
  // accumulator layout: column c16, rows 4 g + e of the 16-row tile
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int m = m0 + 16 * mt + 4 * g + e;
    if (m < M) y[(size_t)m * N + n0 + c16] = from_f<TO>(s[e]);
  }
}

template <typename TO>
__global__ __launch_bounds__(64 * kSlWaves) void small_linear_kernel(const bf16* __restrict__ x, int M, int K,
                                                                    const bf16* __restrict__ W, int N,
                                                                    TO* __restrict__ y) {
  small_linear_tile<TO>(x, M, K, W, N, y);
}

// The projections of several layers' decode steps in one launch (blockIdx.z = layer): q = x wq^T, or
// out = a wo^T with OUT.
template <bool OUT>
__global__ __launch_bounds__(64 * kSlWaves) void decode_linear_group_kernel(DecodeGroup grp, int M, int K, int N) {
  const DecodeLayer& l = grp.l[blockIdx.z];
  if constexpr (OUT)
    small_linear_tile<bf16>(l.a, M, K, l.wo, N, l.out);
  else
    small_linear_tile<bf16>(l.x, M, K, l.wq, N, l.q);
}

// The same idea for a few hundred rows (a prompt's q_proj / o_proj, few rows per training step): a
// workgroup owns 64 rows x 32 features and its 4 waves split K, each with every x / W fragment of up
// to CH 32-wide K chunks in flight before its first MFMA.  The persistent 128 x 256 tiles of
// chapter_gemm.hip put such a product on a handful of CUs, each walking K as a chain of staged loads:
// 509 x 768 x 768 takes 14 us there, 6.4 us here.  Features run along the MFMA's A operand, so a
// lane holds four consecutive features of a row; the waves' partial tiles are added in wave order.
constexpr int kMlRows = 64, kMlCols = 32;

template <int CH, bool RES>
__global__ __launch_bounds__(256) void mid_linear_kernel(const bf16* __restrict__ x, int64_t ldx, int M, int K,
                                                         const bf16* __restrict__ W, bf16* __restrict__ y, int64_t ldy,
                                                         const bf16* __restrict__ res, int64_t ldr) {
  __shared__ f32x4 red[4][8][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c16 = lane & 15;
  const int n0 = blockIdx.x * kMlCols, m0 = blockIdx.y * kMlRows;
  const int kw = K / 4, nch = kw / 32;
  f32x4 acc[2][4];   // [feature tile][row tile]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16* wp = W + (size_t)(n0 + c16) * K + wave * kw + 8 * g;
  const bf16* xp[4];
  bool live[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int m = m0 + 16 * j + c16;
    live[j] = m < M;
    xp[j] = x + (int64_t)(live[j] ? m : 0) * ldx + wave * kw + 8 * g;
  }
  for (int c0 = 0; c0 < nch; c0 += CH) {   // nch % CH == 0 (host rule)
    bf16x8 a[CH][2], b[CH][4];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        a[c][i] = *reinterpret_cast<const bf16x8*>(wp + (size_t)16 * i * K + 32 * (c0 + c));
#pragma unroll
      for (int j = 0; j < 4; ++j)
        b[c][j] = live[j] ? *reinterpret_cast<const bf16x8*>(xp[j] + 32 * (c0 + c)) : bf16x8{};
    }
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) mma(acc[i][j], a[c][i], b[c][j]);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) red[wave][4 * i + j][lane] = acc[i][j];
  __syncthreads();
  // wave w finishes tiles 2 w and 2 w + 1: lane = row 16 j + c16, features 16 i + 4 g .. + 3
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int tile = 2 * wave + t, i = tile >> 2, j = tile & 3;
    f32x4 s = red[0][tile][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) s += red[w][tile][lane];
    const int m = m0 + 16 * j + c16, n = n0 + 16 * i + 4 * g;
    if (m < M) {
      if constexpr (RES) {
        const bf16x4 r = *reinterpret_cast<const bf16x4*>(res + (int64_t)m * ldr + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += (float)r[e];
      }
      bf16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (bf16)s[e];
      *reinterpret_cast<bf16x4*>(y + (int64_t)m * ldy + n) = o;
    }
  }
}

// Up to two workgroups per CU; the chapter GEMM is as fast from there on.  Graph replays, us here
// against there: 768 x 768: 64 rows 6.1 / 13.1, 509 rows (192 workgroups) 6.4 / 14.1, 1,024 rows (384)
// 10.2 / 14.0, 1,536 rows (576) 14.3 / 14.3; 256 x 256: 4,096 rows (512) 5.2 / 7.4; 1,024 x 1,024:
// 1,024 rows (512) 13.0 / 17.6.
constexpr int64_t kMlTiles = 512;
bool mid_linear_takes(int64_t M, int N, int K) {
  return M > 0 && N % kMlCols == 0 && K % 128 == 0 &&
         (M + kMlRows - 1) / kMlRows * (N / kMlCols) <= kMlTiles;
}

int mid_linear(const void* x, int64_t ldx, int64_t M, const void* w, int N, int K, void* y, int64_t ldy,
               const void* res, int64_t ldr, hipStream_t stream) {
  const dim3 grid((unsigned)(N / kMlCols), (unsigned)((M + kMlRows - 1) / kMlRows));
  const int nch = K / 128;
#define ML(CH, RES)                                                                                                  \
  hipLaunchKernelGGL((mid_linear_kernel<CH, RES>), grid, dim3(256), 0, stream, (const bf16*)x, ldx, (int)M, K,       \
                     (const bf16*)w, (bf16*)y, ldy, (const bf16*)res, ldr)
  if (nch % 6 == 0) {
    if (res) ML(6, true); else ML(6, false);
  } else if (nch % 4 == 0) {
    if (res) ML(4, true); else ML(4, false);
  } else if (nch % 2 == 0) {
    if (res) ML(2, true); else ML(2, false);
  } else {
    if (res) ML(1, true); else ML(1, false);
  }
#undef ML
  return check_launch("mid_linear_kernel");
}

}  // namespace moc

using namespace moc;

int moc::decode_linear_group(const DecodeGroup& grp, int layers, bool out, int64_t M, int64_t K, int64_t N,
                             hipStream_t stream) {
  MOC_REQUIRE(M > 0 && M <= 256 && K > 0 && N > 0 && K % (32 * kSlWaves) == 0 && N % 16 == 0 && K <= 65536 && N <= 65536,
              MOC_ERR_UNSUPPORTED, "decode_linear_group: M=%lld (at most 256 rows), K=%lld, N=%lld", (long long)M,
              (long long)K, (long long)N);
  const dim3 grid((unsigned)(N / 16), (unsigned)((M + kSlRows - 1) / kSlRows), (unsigned)layers);
  if (out)
    hipLaunchKernelGGL(decode_linear_group_kernel<true>, grid, dim3(64 * kSlWaves), 0, stream, grp, (int)M, (int)K, (int)N);
  else
    hipLaunchKernelGGL(decode_linear_group_kernel<false>, grid, dim3(64 * kSlWaves), 0, stream, grp, (int)M, (int)K,
                       (int)N);
  return check_launch("decode_linear_group_kernel");
}

extern "C" {

int moc_linear_rows(const void* x, int64_t M, int64_t K, const void* W, int64_t N, int out_dtype, void* y,
                    hipStream_t stream) {
  MOC_REQUIRE(x && W && y, MOC_ERR_ARG, "moc_linear_rows: null pointer");
  MOC_REQUIRE(M >= 0 && M <= 256 && K > 0 && N > 0, MOC_ERR_UNSUPPORTED,
              "moc_linear_rows: M=%lld (at most 256 rows), K=%lld, N=%lld", (long long)M, (long long)K, (long long)N);
  MOC_REQUIRE(K % (32 * kSlWaves) == 0 && N % 16 == 0 && K <= 65536 && N <= 65536, MOC_ERR_UNSUPPORTED,
              "moc_linear_rows: K=%lld must be a multiple of %d and N=%lld of 16", (long long)K, 32 * kSlWaves,
              (long long)N);
  MOC_REQUIRE(((uintptr_t)x & 15) == 0 && ((uintptr_t)W & 15) == 0, MOC_ERR_ARG,
              "moc_linear_rows: x and W must be 16-byte aligned");
  if (M == 0) return MOC_OK;
  dim3 grid((unsigned)(N / 16), (unsigned)((M + kSlRows - 1) / kSlRows));
  if (out_dtype == MOC_BF16)
    hipLaunchKernelGGL(small_linear_kernel<bf16>, grid, dim3(64 * kSlWaves), 0, stream, (const bf16*)x, (int)M, (int)K,
                       (const bf16*)W, (int)N, (bf16*)y);
  else if (out_dtype == MOC_F32)
    hipLaunchKernelGGL(small_linear_kernel<float>, grid, dim3(64 * kSlWaves), 0, stream, (const bf16*)x, (int)M,
                       (int)K, (const bf16*)W, (int)N, (float*)y);
  else
    return set_error(MOC_ERR_UNSUPPORTED, "moc_linear_rows: out dtype %d", out_dtype);
  return check_launch("small_linear_kernel");
}

}  // extern "C"
