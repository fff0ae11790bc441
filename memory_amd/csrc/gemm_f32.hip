// Small float32 products C = op(A) op(B) on the fp32 matrix cores (the float32 layers' projections,
// input and weight gradients, memory_attention.py:140-143, :241-243, :456 at the reference's small
// configurations).  A library GEMM takes one 256 x 256 tile of the reduction-long chain per CU for such
// a product (256 x 256 x 256: 64 us); here a workgroup owns 32 x 64 outputs and its 4 waves take the
// reduction's 32-long chunks in turn, with every operand load of two chunks in flight before the first
// product.  Exact fp32 operands (v_mfma_f32_16x16x4_f32), fp32 accumulation; the waves' partial tiles
// are added through LDS in wave order (256^3: 6.5 us, relative error against 64 bits 1.5e-7, the
// library's 2.9e-7).  Bound: latency of a few rounds of loads; the line to the library is in
// moc_gemm_f32_takes.
#include "moc_common.h"

namespace moc {

constexpr int kGfRows = 32, kGfCols = 64;

// 8 reduction elements k .. k + 7 of row r of an operand; KC: the reduction index is contiguous
// (element (r, k) at p[r * ld + k], 16-byte pieces), else element (r, k) at p[k * ld + r].
template <bool KC>
__device__ __forceinline__ f32x8 gf_load(const float* __restrict__ p, int64_t ld, int r, int rows, int k, int K) {
  f32x8 v;
  if constexpr (KC) {   // K % 8 == 0: a piece is whole or past the end
    f32x4 lo = f32x4{0.f, 0.f, 0.f, 0.f}, hi = lo;
    if (r < rows && k < K) {
      const float* q = p + (int64_t)r * ld + k;
      lo = *reinterpret_cast<const f32x4*>(q);
      hi = *reinterpret_cast<const f32x4*>(q + 4);
    }
    v = f32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = r < rows && k + e < K ? p[(int64_t)(k + e) * ld + r] : 0.f;
  }
  return v;
}

// AK / BK: A's rows m / B's rows n have the reduction contiguous
template <bool AK, bool BK>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ a, int64_t lda,
                                                       const float* __restrict__ b, int64_t ldb, int M, int N, int K,
                                                       float* __restrict__ c, int64_t ldc, int add) {
  __shared__ f32x4 red[4][8][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c16 = lane & 15;
  const int n0 = blockIdx.x * kGfCols, m0 = blockIdx.y * kGfRows;
  const int nch = (K + 31) / 32;
  f32x4 acc[4][2];   // [n tile][m tile]: lane = m, four consecutive n
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int ch = wave; ch < nch; ch += 8) {
    f32x8 fb[2][4], fa[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int k = 32 * (ch + 4 * u) + 8 * g;
#pragma unroll
      for (int i = 0; i < 4; ++i) fb[u][i] = gf_load<BK>(b, ldb, n0 + 16 * i + c16, N, k, K);
#pragma unroll
      for (int j = 0; j < 2; ++j) fa[u][j] = gf_load<AK>(a, lda, m0 + 16 * j + c16, M, k, K);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (ch + 4 * u < nch) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) mma(acc[i][j], fb[u][i], fa[u][j]);
      }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) red[wave][2 * i + j][lane] = acc[i][j];
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int tile = 2 * wave + t, i = tile >> 1, j = tile & 1;
    f32x4 s = red[0][tile][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) s += red[w][tile][lane];
    const int m = m0 + 16 * j + c16, n = n0 + 16 * i + 4 * g;
    if (m < M && n < N) {   // N % 4 == 0
      f32x4* o = reinterpret_cast<f32x4*>(c + (int64_t)m * ldc + n);
      *o = add ? *o + s : s;
    }
  }
}

int gemm_f32(int ta, int tb, int64_t M, int64_t N, int64_t K, const float* a, int64_t lda, const float* b, int64_t ldb,
             float* c, int64_t ldc, int add, hipStream_t stream) {
  MOC_REQUIRE(M > 0 && N > 0 && K > 0 && N % 4 == 0 && M < (1 << 21) && N < (1 << 21) && K < (1 << 21) &&
                  ((ta && !tb) || K % 8 == 0),
              MOC_ERR_UNSUPPORTED, "moc_gemm_f32: M=%lld, N=%lld, K=%lld", (long long)M, (long long)N, (long long)K);
  MOC_REQUIRE(lda >= (ta ? M : K) && ldb >= (tb ? K : N) && ldc >= N && ldc % 4 == 0 && (ta || lda % 4 == 0) &&
                  (!tb || ldb % 4 == 0) && (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15) == 0,
              MOC_ERR_ARG, "moc_gemm_f32: row strides %lld, %lld, %lld (multiples of 4, 16-byte aligned operands)",
              (long long)lda, (long long)ldb, (long long)ldc);
  const dim3 grid((unsigned)((N + kGfCols - 1) / kGfCols), (unsigned)((M + kGfRows - 1) / kGfRows));
  MOC_REQUIRE(grid.y < 65536, MOC_ERR_UNSUPPORTED, "moc_gemm_f32: M=%lld", (long long)M);
#define GF(AK, BK)                                                                                                   \
  hipLaunchKernelGGL((gemm_f32_kernel<AK, BK>), grid, dim3(256), 0, stream, a, lda, b, ldb, (int)M, (int)N, (int)K, \
                     c, ldc, add)
  if (!ta) {
    if (tb) GF(true, true); else GF(true, false);
  } else {
    if (tb) GF(false, true); else GF(false, false);
  }
#undef GF
  return check_launch("gemm_f32_kernel");
}

}  // namespace moc

using namespace moc;

extern "C" {

int moc_gemm_f32_takes(int ta, int tb, int64_t M, int64_t N, int64_t K) {
  // us here / hipBLASLt (graph replays, forward / input-gradient / weight-gradient form alike): 256^3
  // 6.5 / 63, 640 x 512 x 256 7 / 6.3, 512 x 512 x 256 6.6 / 5.6, 8,192 x 64 x 64 5 / 4.5, 320 x 256 x 512
  // 10 / 6.5, 64 x 64 x 512 10 / 10.7, 512 x 1024 x 1024 18 / 12, 256 x 256 x 2048 29 / 9.  From the host a
  // call of either is longer than that, 8 us here against 19 to 20 of the library, which is what a step of
  // such sizes waits for: calls back to back take 8 to 11 us here and 19 to 20 there at every one of them.
  constexpr int64_t kMaxWork = 100000000, kMaxK = 512;
  if (M <= 0 || N <= 0 || K <= 0 || N % 4 != 0 || M > (1 << 20) || N > (1 << 20) || K > (1 << 20)) return 0;
  if ((!ta || tb) && K % 8 != 0) return 0;   // an operand with a contiguous reduction is read 8 at a time
  return K <= kMaxK && M * N * K <= kMaxWork;
}

int moc_gemm_f32(int ta, int tb, int64_t M, int64_t N, int64_t K, const float* a, int64_t lda, const float* b,
                 int64_t ldb, float* c, int64_t ldc, hipStream_t stream) {
  MOC_REQUIRE(a && b && c, MOC_ERR_ARG, "moc_gemm_f32: null pointer");
  MOC_REQUIRE(moc_gemm_f32_takes(ta, tb, M, N, K), MOC_ERR_UNSUPPORTED, "moc_gemm_f32: M=%lld, N=%lld, K=%lld",
              (long long)M, (long long)N, (long long)K);
  return gemm_f32(ta, tb, M, N, K, a, lda, b, ldb, c, ldc, 0, stream);
}

}  // extern "C"
