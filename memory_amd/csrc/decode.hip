// Single-token decode over precomputed per-layer K / V chapter tiles.
//
// Step of the sequence-routed memory layer with L = 1 (the decode use of
// memory_transformer/model.py:612-692 -> memory_attention.py:458-478) when the
// chapters and their weights omega are fixed for the generation: K / V of every
// chapter are precomputed once per layer (kv_project over all chapters), so a step
// only reads the selected tiles.  HBM-bound: each distinct (chapter, kv head) tile
// is read once per step however many sequences selected it (chapter plan over the
// (sequence, slot) edges).
//
// The omega-weighted memory rows of the reference (memory = memory * omega before the
// K/V projection) give K = omega K_c and V = omega V_c, so per edge (b, slot) and query
// head: s_j = omega * scale * q . k_j, o = omega * sum_j p_j v_j / sum_j p_j and
// lse = log2 sum_j 2^(s_j log2 e): exactly the chapter-centric partial attention of the
// token-routed path with a per-edge logit and output factor (sparse_fwd_launch: one
// wave per (chapter, kv head) unit, K fragments from HBM, V^T through transposing LDS
// reads).  moc_sparse_combine (joint mode, rpe = H) merges the slots of a sequence.  The plan is
// fixed for a whole generation, so the first 16 edges of every chapter are tabulated once
// (moc_decode_row_table): a unit then requests its rows' edge ids together with its plan entries
// instead of after them, and its q rows go out together with its K / V tiles.
#include "moc_common.h"

#include <algorithm>

using namespace moc;

namespace {

// row_tab[u * W + j] = the j-th edge (csr order) of distinct chapter u, -1 past its edges or past
// n_uniq; one thread per entry.
__global__ __launch_bounds__(256) void decode_row_table_kernel(const int32_t* __restrict__ n_uniq,
                                                               const int32_t* __restrict__ csr_off,
                                                               const int32_t* __restrict__ csr_edge, int64_t max_u,
                                                               int W, int32_t* __restrict__ row_tab) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t u = i / W;
  const int j = (int)(i % W);
  if (u >= max_u) return;
  int32_t e = -1;
  if (u < n_uniq[0]) {
    const int32_t p0 = csr_off[u], cnt = csr_off[u + 1] - p0;
    if (j < cnt) e = csr_edge[p0 + j];
  }
  row_tab[i] = e;
}

}  // namespace

extern "C" {

int moc_plan_row_table(const int32_t* n_uniq, const int32_t* csr_off, const int32_t* csr_edge, int64_t max_u,
                       int width, int32_t* row_tab, hipStream_t stream) {
  MOC_REQUIRE(n_uniq && csr_off && csr_edge && row_tab, MOC_ERR_ARG, "moc_plan_row_table: null pointer");
  MOC_REQUIRE(width == 16 || width == 32, MOC_ERR_ARG, "moc_plan_row_table: width %d (16 or 32)", width);
  MOC_REQUIRE(max_u >= 0 && max_u < ((int64_t)1 << 25), MOC_ERR_ARG, "moc_plan_row_table: max_u %lld",
              (long long)max_u);
  if (max_u == 0) return MOC_OK;
  hipLaunchKernelGGL(decode_row_table_kernel, dim3((unsigned)((max_u * width + 255) / 256)), dim3(256), 0, stream,
                     n_uniq, csr_off, csr_edge, max_u, width, row_tab);
  return check_launch("decode_row_table_kernel");
}

int moc_decode_row_table(const int32_t* n_uniq, const int32_t* csr_off, const int32_t* csr_edge, int64_t max_u,
                         int32_t* row_tab, hipStream_t stream) {
  return moc_plan_row_table(n_uniq, csr_off, csr_edge, max_u, 16, row_tab, stream);
}

int moc_decode_partial(int dtype, const void* q, int64_t B, int H, const void* k_tiles, const void* v_tiles, int HK,
                       int Dh, int T, const int32_t* uniq, const int32_t* n_uniq, const int32_t* csr_off,
                       const int32_t* csr_edge, int64_t max_u, const float* omega, int NS, float scale, void* o_part,
                       float* lse_part, const int32_t* row_tab, hipStream_t stream) {
  MOC_REQUIRE(q && k_tiles && v_tiles && uniq && n_uniq && csr_off && csr_edge && omega && o_part && lse_part,
              MOC_ERR_ARG, "moc_decode_partial: null pointer");
  MOC_REQUIRE(Dh == 64 && T == 64, MOC_ERR_UNSUPPORTED, "moc_decode_partial: needs head_dim 64 and T 64");
  MOC_REQUIRE(H > 0 && HK > 0 && H % HK == 0 && NS > 0, MOC_ERR_ARG, "moc_decode_partial: bad heads");
  if (B == 0 || max_u == 0) return MOC_OK;
  // tiles [chapter][HK][64 keys][64 dims]; edge e = b * NS + slot serves query heads 0 .. H-1
  return sparse_fwd_launch(dtype, q, H, k_tiles, v_tiles, (int64_t)HK * 4096, 4096, 64, HK, uniq, n_uniq, csr_off,
                           csr_edge, max_u, NS, 0, HK, 0, H, scale, omega, o_part, lse_part, stream,
                           "moc_decode_partial", row_tab);
}

int moc_decode_route(const float* pooled, int64_t B, int64_t d, const void* W, int w_dtype, const float* bias, int64_t C,
                     int S, int k, float scale, float* logits, int32_t* idx, float* w, int32_t* idx_star, float* omega,
                     void* plan_ws, size_t plan_ws_bytes, int32_t* uniq, int32_t* n_uniq, int32_t* edge_u,
                     int32_t* csr_off, int32_t* csr_edge, int64_t max_u, int32_t* row_tab, hipStream_t stream) {
  const int64_t E = B * (S + k);
  MOC_REQUIRE(max_u >= 0 && max_u <= E && max_u <= C, MOC_ERR_ARG, "moc_decode_route: max_u %lld", (long long)max_u);
  if (int rc = moc_router_linear(pooled, B, d, W, w_dtype, bias, C, logits, stream)) return rc;
  if (int rc = moc_router_topk_prepend(logits, B, C, S, k, scale, idx, w, idx_star, omega, stream)) return rc;
  if (int rc = moc_chapter_plan(idx_star, E, C, plan_ws, plan_ws_bytes, uniq, n_uniq, edge_u, csr_off, csr_edge, stream))
    return rc;
  return moc_decode_row_table(n_uniq, csr_off, csr_edge, max_u, row_tab, stream);
}

namespace {
struct StepLayout {
  size_t q, o_part, a, lse_part, lse, bytes;
  StepLayout(int64_t B, int H, int NS) {
    const size_t row = (size_t)B * H * 64 * 2;
    size_t o = 0;
    auto take = [&](size_t n) { const size_t at = o; o += (n + 255) / 256 * 256; return at; };
    q = take(row);
    o_part = take(row * NS);
    a = take(row);
    lse_part = take((size_t)B * NS * H * 4);
    lse = take((size_t)B * H * 4);
    bytes = o;
  }
};
}  // namespace

size_t moc_decode_step_workspace(int64_t B, int H, int NS) {
  return B < 0 || H <= 0 || NS <= 0 ? 0 : StepLayout(B, H, NS).bytes;
}

int moc_decode_step(const void* x, int64_t B, int64_t d, const void* wq, int H, const void* k_tiles, const void* v_tiles,
                    int HK, int T, const int32_t* uniq, const int32_t* n_uniq, const int32_t* csr_off,
                    const int32_t* csr_edge, const int32_t* edge_u, int64_t max_u, const float* omega, int NS,
                    float scale, const void* wo, int64_t N, void* workspace, size_t workspace_bytes, void* out,
                    const int32_t* row_tab, hipStream_t stream) {
  MOC_REQUIRE(x && wq && wo && workspace && out && edge_u, MOC_ERR_ARG, "moc_decode_step: null pointer");
  MOC_REQUIRE(B > 0 && H > 0 && NS > 0, MOC_ERR_ARG, "moc_decode_step: B=%lld H=%d NS=%d", (long long)B, H, NS);
  const StepLayout y(B, H, NS);
  MOC_REQUIRE(workspace_bytes >= y.bytes, MOC_ERR_ARG, "moc_decode_step: workspace %zu < %zu bytes", workspace_bytes,
              y.bytes);
  char* ws = (char*)workspace;
  if (int rc = moc_linear_rows(x, B, d, wq, (int64_t)H * 64, MOC_BF16, ws + y.q, stream)) return rc;
  if (int rc = moc_decode_partial(MOC_BF16, ws + y.q, B, H, k_tiles, v_tiles, HK, 64, T, uniq, n_uniq, csr_off, csr_edge,
                                  max_u, omega, NS, scale, ws + y.o_part, (float*)(ws + y.lse_part), row_tab, stream))
    return rc;
  if (int rc = moc_sparse_combine(MOC_BF16, ws + y.o_part, (const float*)(ws + y.lse_part), edge_u, nullptr, 1, NS, H, B,
                                  H, 0, ws + y.a, (float*)(ws + y.lse), stream))
    return rc;
  return moc_linear_rows(ws + y.a, B, (int64_t)H * 64, wo, N, MOC_BF16, out, stream);
}

// 9 to 68 slots and 16,384 rows are what the one combine kernel with a grouped form takes
// (sparse_combine_small_kernel): fewer slots and more rows have combines of their own, which would need one
// too, and run a chain of kernels per layer.
int moc_decode_step_group(const moc_decode_layer* layers, int n, int64_t B, int64_t d, int H, int HK, int T, int NS,
                          float scale, int64_t N, size_t workspace_bytes, hipStream_t stream) {
  MOC_REQUIRE(layers && n > 0, MOC_ERR_ARG, "moc_decode_step_group: no layers");
  MOC_REQUIRE(T == 64 && B > 0 && H > 0 && HK > 0 && H % HK == 0 && NS > 8 && NS <= 68 && B * H <= 16384,
              MOC_ERR_UNSUPPORTED, "moc_decode_step_group: B=%lld H=%d HK=%d T=%d NS=%d", (long long)B, H, HK, T, NS);
  const StepLayout y(B, H, NS);
  MOC_REQUIRE(workspace_bytes >= y.bytes, MOC_ERR_ARG, "moc_decode_step_group: workspace %zu < %zu bytes",
              workspace_bytes, y.bytes);
  for (int i = 0; i < n; ++i) {
    const moc_decode_layer& l = layers[i];
    MOC_REQUIRE(l.x && l.wq && l.k_tiles && l.v_tiles && l.wo && l.uniq && l.n_uniq && l.csr_off && l.csr_edge && l.edge_u &&
                    l.omega && l.workspace && l.out && l.max_u >= 0 && l.max_u < (1 << 24) &&
                    (((uintptr_t)l.x | (uintptr_t)l.wq | (uintptr_t)l.wo | (uintptr_t)l.workspace) & 15) == 0,
                MOC_ERR_ARG, "moc_decode_step_group: layer %d: null or unaligned pointer", i);
  }
  for (int i0 = 0; i0 < n; i0 += kDecodeGroup) {
    const int m = std::min(kDecodeGroup, n - i0);
    DecodeGroup grp{};
    for (int i = 0; i < m; ++i) {
      const moc_decode_layer& l = layers[i0 + i];
      char* ws = (char*)l.workspace;
      grp.l[i] = DecodeLayer{(const bf16*)l.x, (const bf16*)l.wq, (const bf16*)l.k_tiles, (const bf16*)l.v_tiles,
                             (const bf16*)l.wo, l.uniq, l.n_uniq, l.csr_off, l.csr_edge, l.edge_u, l.row_tab, l.omega,
                             (bf16*)(ws + y.q), (bf16*)(ws + y.o_part), (bf16*)(ws + y.a), (bf16*)l.out,
                             (float*)(ws + y.lse_part), (float*)(ws + y.lse), l.max_u};
    }
    if (int rc = decode_linear_group(grp, m, false, B, d, (int64_t)H * 64, stream)) return rc;
    if (int rc = decode_attend_group(grp, m, B, H, HK, NS, scale, stream)) return rc;
    if (int rc = decode_linear_group(grp, m, true, B, (int64_t)H * 64, N, stream)) return rc;
  }
  return MOC_OK;
}

}  // extern "C"
