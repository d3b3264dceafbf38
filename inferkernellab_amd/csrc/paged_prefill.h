// Parameters and block-table helpers shared by the paged prefill kernels
// (paged_prefill.hip: 16-bit matrix cores and the wide-row fallback;
// paged_prefill_split.hip: 16-bit matrix cores, keys split between waves;
// paged_prefill_f32.hip: fp32 matrix cores).
#pragma once

#include "ikl_common.h"
#include "paged_attn.h"

namespace ikl {

struct PrefillParams {
  const char *q;
  int64_t q_sb, q_sh, q_st;  // elements
  const char *kc;
  const char *vc;
  int64_t k_sb, k_st, k_sh;
  int64_t v_sb, v_st, v_sh;
  const void *tables;
  int64_t t_sb;
  int64_t table_width;
  const void *starts;
  const void *lens;
  char *out;
  int64_t o_sb, o_sh, o_st;
  int64_t batch;
  int64_t width;       // query rows per request (T)
  int64_t num_blocks;
  int64_t cap_tokens;  // table_width * block_size
  int64_t row_blocks;  // workgroups per (request, kv head) of the MFMA kernel
  int64_t bh_pad;      // batch * num_kv_heads rounded up to a multiple of 8
  int32_t stream_major;  // each XCD takes its (request, kv head) prefixes one after another
  int32_t paired;        // one resident round: the shortest row blocks share CUs with the longest
  int32_t num_heads;
  int32_t num_kv_heads;
  int32_t heads_per_kv;
  int32_t head_dim;
  int32_t block_size;
  int32_t bs_shift;  // log2(block_size) or -1
  int32_t table_i64;
  int32_t idx_i64;   // starts / lens element type
  float scale_log2;  // scale * log2(e)
  // FP8 KV cache: E4M3 codes, one fp32 scale per (token, head) row in
  // k_scale / v_scale [blocks, kv heads, block_size]
  int32_t kv_fp8;
  const float *k_scale;
  const float *v_scale;
  int64_t s_sb, s_sh;  // elements
};

// Launches paged_prefill_f32_kernel (head_dim <= PREFILL_F32_MAX_DIM, caches
// in the query's dtype) for queries of `dtype`; p.row_blocks and p.bh_pad are
// set here.
constexpr int PREFILL_F32_MAX_DIM = 256;
hipError_t launch_prefill_f32(PrefillParams p, int dtype, hipStream_t s);

// Launches paged_prefill_split_kernel (what the 16-bit kernel takes) with
// `groups` (1, 2 or 4) waves on every row; p.row_blocks and p.bh_pad are set
// here.
hipError_t launch_prefill_split(PrefillParams p, int dtype, int groups, hipStream_t s);

namespace {

__device__ inline int64_t pf_index(const void *base, int64_t i, int i64) {
  return i64 ? load_index<int64_t>(base, i) : load_index<int32_t>(base, i);
}

// Block-table entry (b, lb), or -1 when it is outside the table or names a
// block outside the cache.
__device__ inline int pf_block(const PrefillParams &p, int64_t b, int64_t lb) {
  if (lb < 0 || lb >= p.table_width) return -1;
  const int64_t e = pf_index(p.tables, b * p.t_sb + lb, p.table_i64);
  return e >= 0 && e < p.num_blocks ? (int)e : -1;
}

// Prefill range of request b: start (clamped to [0, end]), end (clamped to
// [0, cap_tokens]) and the number of attending rows (<= width).
__device__ inline void pf_range(const PrefillParams &p, int64_t b, int64_t *start, int64_t *end, int64_t *rows) {
  int64_t e = pf_index(p.lens, b, p.idx_i64);
  e = e < 0 ? 0 : (e < p.cap_tokens ? e : p.cap_tokens);
  int64_t s = pf_index(p.starts, b, p.idx_i64);
  s = s < 0 ? 0 : (s < e ? s : e);
  *start = s;
  *end = e;
  *rows = e - s < p.width ? e - s : p.width;
}

__device__ inline int64_t pf_logical(const PrefillParams &p, int64_t pos) {
  return p.bs_shift >= 0 ? (pos >> p.bs_shift) : pos / p.block_size;
}

// Two E4M3 codes times one fp32 scale -> two 16-bit values (one rounding).
template <typename Tag>
__device__ inline uint32_t fp8x2_scaled(uint32_t w, float scale, bool hi);
template <>
__device__ inline uint32_t fp8x2_scaled<bf16_tag>(uint32_t w, float scale, bool hi) {
  return __builtin_bit_cast(uint32_t, hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, scale, true)
                                        : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, scale, false));
}
template <>
__device__ inline uint32_t fp8x2_scaled<f16_tag>(uint32_t w, float scale, bool hi) {
  return __builtin_bit_cast(uint32_t, hi ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, scale, true)
                                        : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, scale, false));
}

}  // namespace
}  // namespace ikl
