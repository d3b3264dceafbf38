// Paged prefill on the fp32 matrix cores: the shapes the 16-bit kernel of
// paged_prefill.hip does not take (fp32 caches, head dims other than 32 / 64
// / 96 / 128, block sizes that are not a multiple of 16), with every product
// and probability in fp32. Same semantics: row t of request b attends the
// keys at positions <= start_b + t; rows past the chunk receive the value at
// position 0; keys of blocks outside the cache are dropped.
//
// Bound: the fp32 matrix rate (256 flop per clock and CU; a large fp32
// matrix product reaches 137 TFLOP/s). One K/V element read from LDS feeds
// 16 rows, so LDS runs at a quarter of the matrix time and global memory far
// below that; what is lost is the softmax between the two products and the
// start and end of each workgroup.
//
// A workgroup of 4 waves takes 64 query rows of one (request, kv head) - a
// row is one (token, query head) pair, token-major - and streams the keys in
// 32-key tiles staged in LDS as fp32. Each wave owns 16 rows:
//
//   S^T[32 keys x 16 rows] = K . Q^T     2 * D/4 v_mfma_f32_16x16x4_f32
//   online softmax (lane = one row x 8 keys)
//   O^T[D x 16 rows]     += V^T . P      8 * D/16 v_mfma_f32_16x16x4_f32
//
// v_mfma_f32_16x16x4_f32: lane l supplies A[l%16][l/16], B[l/16][l%16] and
// receives D[4(l/16)+i][l%16], i < 4. The order of a contraction and of the
// output rows is free, so that every LDS read is 16 bytes wide:
//   * QK^T contracts dims 16s + 4g + j (g = l/16) in MFMA j of step s: one
//     16-byte read of a K row feeds four MFMAs;
//   * the scores' layout (row l%16, keys 4g + i) is the B operand of the PV
//     MFMA i over keys {4g + i}; output row m of MFMA t in a 64-dim window
//     is dim 4m + t, so one 16-byte read of a V row feeds four MFMAs and
//     each lane ends with 16 consecutive dims of its row.
//
// Measured on 4 ragged prompts of 257-512 tokens, 32/8 heads of 64, fp32:
// 51 us (49 TFLOP/s of attended pairs), against 1050 us with one wave per row
// walking the keys in sequence.
#include "ikl_common.h"
#include "mfma_ops.h"
#include "paged_attn.h"
#include "paged_prefill.h"

namespace ikl {
namespace {

constexpr int FT = 32;          // keys per tile
constexpr int FWAVES = 4;       // waves per workgroup
constexpr int FROWS = 16 * FWAVES;

// Waves per SIMD the register allocation aims at. Up to 64 dims three fit
// without scratch: 51.4 us on the prompts above against 54.5 at two and 71.4
// at four (156 bytes of scratch per lane).
constexpr int f32_waves(int dp) { return dp <= 64 ? 3 : dp <= 128 ? 2 : 1; }

__device__ inline f32x4_t mma4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Four consecutive elements of a row, as loaded.
template <typename Tag>
struct quad;
template <>
struct quad<f32_tag> {
  static constexpr int EB = 4;
  typedef f32x4_t raw;
  __device__ static inline raw load(const char *p) { return *reinterpret_cast<const raw *>(p); }
  // n < 4 elements, or a row that is not aligned to four
  __device__ static inline raw load_some(const char *p, int n) {
    const float *f = reinterpret_cast<const float *>(p);
    raw r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n) r[i] = f[i];
    return r;
  }
  __device__ static inline raw zero() { return raw{0.f, 0.f, 0.f, 0.f}; }
  __device__ static inline f32x4_t wide(raw r) { return r; }
  __device__ static inline void store(char *p, f32x4_t x) { *reinterpret_cast<f32x4_t *>(p) = x; }
  __device__ static inline void store_some(char *p, f32x4_t x, int n) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n) reinterpret_cast<float *>(p)[i] = x[i];
  }
};
template <typename Tag>
struct quad16 {
  static constexpr int EB = 2;
  typedef u32x2_t raw;
  __device__ static inline raw load(const char *p) { return *reinterpret_cast<const raw *>(p); }
  // rows of 16-bit elements are whole 4-byte words (n is even)
  __device__ static inline raw load_some(const char *p, int n) {
    const uint32_t *w = reinterpret_cast<const uint32_t *>(p);
    raw r = {0u, 0u};
    if (n > 0) r[0] = w[0];
    if (n > 2) r[1] = w[1];
    return r;
  }
  __device__ static inline raw zero() { return raw{0u, 0u}; }
  __device__ static inline f32x4_t wide(raw r) {
    return f32x4_t{mfma_ops<Tag>::lo(r[0]), mfma_ops<Tag>::hi(r[0]), mfma_ops<Tag>::lo(r[1]), mfma_ops<Tag>::hi(r[1])};
  }
  __device__ static inline raw narrow(f32x4_t x) {
    return raw{elem<Tag>::pack2(x[0], x[1]), elem<Tag>::pack2(x[2], x[3])};
  }
  __device__ static inline void store(char *p, f32x4_t x) { *reinterpret_cast<raw *>(p) = narrow(x); }
  __device__ static inline void store_some(char *p, f32x4_t x, int n) {
    const raw r = narrow(x);
    if (n > 0) reinterpret_cast<uint32_t *>(p)[0] = r[0];
    if (n > 2) reinterpret_cast<uint32_t *>(p)[1] = r[1];
  }
};
template <>
struct quad<f16_tag> : quad16<f16_tag> {};
template <>
struct quad<bf16_tag> : quad16<bf16_tag> {};

__device__ inline bool not_finite(f32x4_t x) {
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) bad |= (__float_as_uint(x[i]) & 0x7f800000u) == 0x7f800000u;
  return bad;
}

// DP: head_dim rounded up to a compiled width; dims past head_dim are zero
// in LDS and in Q. `vec` (kernel argument): every Q, K, V and out row starts
// on a whole quad and head_dim is a multiple of 4.
template <typename Tag, int DP>
__global__ __launch_bounds__(64 * FWAVES, f32_waves(DP)) void paged_prefill_f32_kernel(const PrefillParams p, int vec) {
  static_assert(DP % 32 == 0, "head dims are padded to a multiple of 32");
  using Q4 = quad<Tag>;
  constexpr int EB = Q4::EB;
  constexpr int KS = DP / 16;          // QK^T steps of 16 dims
  constexpr int NW = DP / 64;          // 64-dim windows of V
  constexpr bool TAIL = DP % 64 != 0;  // and a 32-dim one
  constexpr int MT = DP / 16;          // PV accumulators
  constexpr int CH = DP / 4;           // quads per row
  constexpr int PPT = FT * CH / (64 * FWAVES);  // staged quads per thread, of K and of V
  // Row pitch of a staged tile: 4 words past a multiple of 32 put the 16
  // rows of a K read on distinct banks.
  constexpr int PITCH = DP + 4;
  __shared__ __attribute__((aligned(16))) float ks[FT * PITCH];
  __shared__ __attribute__((aligned(16))) float vs[FT * PITCH];
  __shared__ int64_t koff[2][FT], voff[2][FT];  // byte offset of a tile's key rows, -1: no such key

  const int tid = threadIdx.x;
  const int lane = tid & 63, hl = lane & 15, grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // All row blocks of one (request, kv head) share blockIdx.x mod 8, hence
  // one XCD and its L2; those nearest the end of the prompts start first.
  const int64_t idx = blockIdx.x;
  const int64_t bh = idx % p.bh_pad, rb = p.row_blocks - 1 - idx / p.bh_pad;
  if (bh >= p.batch * p.num_kv_heads) return;
  const int64_t b = bh / p.num_kv_heads;
  const int kvh = (int)(bh % p.num_kv_heads);
  const int G = p.heads_per_kv, D = p.head_dim;

  int64_t start, end, nrows;
  pf_range(p, b, &start, &end, &nrows);
  const int64_t rows_valid = nrows * G, rows_all = p.width * G;
  const int64_t row0 = rb * FROWS, wr0 = row0 + 16 * wave;
  const int64_t wg_last = (row0 + FROWS < rows_valid ? row0 + FROWS : rows_valid) - 1;
  const int64_t kv_hi = wg_last >= row0 ? start + wg_last / G + 1 : 0;  // keys the workgroup needs
  const int64_t n_tiles = (kv_hi + FT - 1) / FT;
  const int64_t w_last = (wr0 + 16 < rows_valid ? wr0 + 16 : rows_valid) - 1;
  const int64_t w_hi = w_last >= wr0 ? start + w_last / G + 1 : 0;  // keys [0, w_hi) reach some row of the wave
  const int64_t w_lo = start + wr0 / G;                             // every row of the wave sees keys <= w_lo
  const int64_t wg_lo = start + row0 / G;                           // ... of the workgroup

  const int64_t r = wr0 + hl;  // this lane's row
  const bool row_ok = r < rows_valid;
  const int64_t t = r < rows_all ? r / G : 0;
  const int h = r < rows_all ? (int)(r % G) : 0;
  const int64_t qpos = row_ok ? start + t : -1;
  const int64_t head = (int64_t)kvh * G + h;

  f32x4_t q[KS];
  {
    const char *qrow = p.q + (b * p.q_sb + head * p.q_sh + t * p.q_st) * EB;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int d = 16 * s + 4 * grp;
      typename Q4::raw w = Q4::zero();
      if (row_ok && d < D) w = vec ? Q4::load(qrow + d * EB) : Q4::load_some(qrow + d * EB, D - d);
      q[s] = Q4::wide(w);
    }
  }

  f32x4_t acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = NEG_SENTINEL;    // running max of the lane's row, log2 domain
  float thr = NEG_SENTINEL;  // (m + RESCALE_LOG2) in raw score units
  float l = 0.f;             // this lane's share of the row's sum
  const float inv_scale_log2 = 1.f / p.scale_log2;

  const char *kbase = p.kc + (int64_t)kvh * p.k_sh * EB;
  const char *vbase = p.vc + (int64_t)kvh * p.v_sh * EB;

  // Key rows of tile j, one per thread of the first half wave: the block id,
  // loaded a tile ahead of its use and put into LDS by put_rows.
  int blk = -1;
  auto load_rows = [&](int64_t j) {
    const int64_t pos = j * FT + tid;
    blk = tid < FT && pos < kv_hi ? pf_block(p, b, pf_logical(p, pos)) : -1;
  };
  auto put_rows = [&](int64_t j) {
    if (tid < FT) {
      const int64_t pos = j * FT + tid, in = pos - pf_logical(p, pos) * p.block_size;
      koff[j & 1][tid] = blk >= 0 ? (blk * p.k_sb + in * p.k_st) * EB : -1;
      voff[j & 1][tid] = blk >= 0 ? (blk * p.v_sb + in * p.v_st) * EB : -1;
    }
  };
  // Global -> registers for tile j; rows that do not exist read as zero.
  typename Q4::raw kr[PPT], vr[PPT];
  auto fetch = [&](int64_t j) {
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
      const int i = tid + 64 * FWAVES * u, row = i / CH, d = 4 * (i % CH);
      const int64_t ko = koff[j & 1][row], vo = voff[j & 1][row];
      kr[u] = Q4::zero();
      vr[u] = Q4::zero();
      if (ko >= 0 && d < D) {
        if (vec) {
          kr[u] = Q4::load(kbase + ko + d * EB);
          vr[u] = Q4::load(vbase + vo + d * EB);
        } else {
          kr[u] = Q4::load_some(kbase + ko + d * EB, D - d);
          vr[u] = Q4::load_some(vbase + vo + d * EB, D - d);
        }
      }
    }
  };

  // One tile. `hole`: bit k set when the tile's key k lies in a block
  // outside the cache. `odd_v`: some staged V element is not finite and some
  // row of the workgroup does not see all keys: a masked key's probability
  // of 0 must not meet it in a matrix product.
  auto compute = [&](int64_t base, uint32_t hole, bool odd_v) {
    if (base >= w_hi) return;  // no row of this wave reaches the tile
    // Four chains per half, one for each dim of a quad, added in pairs: a
    // single chain of D/4 products is four times as long, in time and in
    // rounding (error against 64 bits at 64 dims: 2.7e-7 with one, 2.1e-7
    // with four, 2.4e-7 for the lane-parallel tree of one wave per row).
    f32x4_t sc[2], sj[2][4];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int j = 0; j < 4; ++j) sj[hf][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const f32x4_t k0 = *reinterpret_cast<const f32x4_t *>(&ks[hl * PITCH + 16 * s + 4 * grp]);
      const f32x4_t k1 = *reinterpret_cast<const f32x4_t *>(&ks[(16 + hl) * PITCH + 16 * s + 4 * grp]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sj[0][j] = mma4(k0[j], q[s][j], sj[0][j]);
        sj[1][j] = mma4(k1[j], q[s][j], sj[1][j]);
      }
    }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) sc[hf] = (sj[hf][0] + sj[hf][1]) + (sj[hf][2] + sj[hf][3]);
    // lane: row hl, keys 16 hf + 4 grp + i
    uint32_t dead = hole;
    if (base + FT - 1 > w_lo) {
      const int64_t seen = qpos - base + 1;  // keys below this are visible
      dead |= seen <= 0 ? 0xffffffffu : seen < FT ? 0xffffffffu << (int)seen : 0u;
    }
    if (dead != 0u) {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if ((dead >> (16 * hf + 4 * grp + i)) & 1u) sc[hf][i] = -INFINITY;
    }
    const float lmax = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])),
                             fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
    // The maximum moves, and sums are rescaled, only where a score passes it
    // by 2^RESCALE_LOG2: fp32 sums lose nothing by that.
    if (__builtin_amdgcn_ballot_w64(lmax > thr) != 0ull) {
      const float tmax = max_xor32(max_xor16(lmax)) * p.scale_log2;
      const bool need = tmax > m + RESCALE_LOG2;
      const float alpha = need ? fast_exp2(m - tmax) : 1.f;
      m = need ? tmax : m;
      thr = (m + RESCALE_LOG2) * inv_scale_log2;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i] *= alpha;
    }
    f32x4_t pr[2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pr[hf][i] = fast_exp2(fmaf(sc[hf][i], p.scale_log2, -m));
        l += pr[hf][i];
      }
    if (!odd_v) {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float *vrow = &vs[(16 * hf + 4 * grp + i) * PITCH];
#pragma unroll
          for (int w = 0; w < NW; ++w) {
            const f32x4_t v4 = *reinterpret_cast<const f32x4_t *>(vrow + 64 * w + 4 * hl);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[4 * w + j] = mma4(v4[j], pr[hf][i], acc[4 * w + j]);
          }
          if constexpr (TAIL) {
            const f32x2_t v2 = *reinterpret_cast<const f32x2_t *>(vrow + 64 * NW + 2 * hl);
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[4 * NW + j] = mma4(v2[j], pr[hf][i], acc[4 * NW + j]);
          }
        }
      return;
    }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll 1
        for (int g = 0; g < 4; ++g) {
          const int key = 16 * hf + 4 * g + i;
          const float pk = __shfl(pr[hf][i], hl + 16 * g, 64);
          const bool see = ((dead >> key) & 1u) == 0u;
          const float *vrow = &vs[key * PITCH];
#pragma unroll
          for (int a = 0; a < MT; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int mrow = 4 * grp + e;  // output row of MFMA a's window
              const int d = a < 4 * NW ? 64 * (a / 4) + 4 * mrow + a % 4 : 64 * NW + 2 * mrow + (a - 4 * NW);
              if (see) acc[a][e] = fmaf(pk, vrow[d], acc[a][e]);
            }
        }
  };

  if (n_tiles > 0) {
    load_rows(0);
    put_rows(0);
    load_rows(1);
    put_rows(1);
    __syncthreads();
    fetch(0);
    load_rows(2);
  }
  for (int64_t j = 0; j < n_tiles; ++j) {
    const int64_t base = j * FT;
    const bool masked = base + FT - 1 > wg_lo;
    __syncthreads();  // every wave is done with tile j - 1 and with the row offsets of tile j
    bool odd = false;
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
      const int i = tid + 64 * FWAVES * u, row = i / CH, d = 4 * (i % CH);
      const f32x4_t k4 = Q4::wide(kr[u]), v4 = Q4::wide(vr[u]);
      if (masked) odd |= not_finite(v4);
      *reinterpret_cast<f32x4_t *>(&ks[row * PITCH + d]) = k4;
      *reinterpret_cast<f32x4_t *>(&vs[row * PITCH + d]) = v4;
    }
    // keys below kv_hi without a row: their block lies outside the cache
    const uint32_t hole =
        (uint32_t)__builtin_amdgcn_ballot_w64(lane < FT && base + lane < kv_hi && koff[j & 1][lane & 31] < 0);
    if (masked) odd = __syncthreads_or(odd);
    else __syncthreads();
    put_rows(j + 2);  // into the offsets of tile j, read by every wave before the barrier
    if (j + 1 < n_tiles) fetch(j + 1);
    load_rows(j + 3);
    compute(base, hole, odd);
  }

  // Normalise and store: lane (hl, grp) holds 16 (tail: 8) consecutive dims
  // of row r per 64-dim window.
  if (r >= rows_all) return;
  char *dst = p.out + (b * p.o_sb + head * p.o_sh + t * p.o_st) * EB;
  if (row_ok) {
    l = sum_xor32(sum_xor16(l));
    const float inv = 1.f / l;  // no attended key: 0/0 -> NaN
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = 64 * w + 16 * grp + 4 * e;
        const f32x4_t o = f32x4_t{acc[4 * w][e], acc[4 * w + 1][e], acc[4 * w + 2][e], acc[4 * w + 3][e]} * inv;
        if (vec && d < D) Q4::store(dst + d * EB, o);
        else Q4::store_some(dst + d * EB, o, D - d);
      }
    if constexpr (TAIL) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int d = 64 * NW + 8 * grp + 4 * e;
        const f32x4_t o =
            f32x4_t{acc[4 * NW][2 * e], acc[4 * NW + 1][2 * e], acc[4 * NW][2 * e + 1], acc[4 * NW + 1][2 * e + 1]} * inv;
        if (vec && d < D) Q4::store(dst + d * EB, o);
        else Q4::store_some(dst + d * EB, o, D - d);
      }
    }
  } else {
    // padding row: the value at position 0 (zero when its block is masked),
    // the row's four lanes taking every fourth quad, or word
    const int ph = end > 0 ? pf_block(p, b, 0) : -1;
    const char *src = ph >= 0 ? vbase + ph * p.v_sb * EB : nullptr;
    if (vec) {
      typename Q4::raw w[DP / 16];
#pragma unroll
      for (int i = 0; i < DP / 16; ++i) {
        const int d = 16 * i + 4 * grp;
        w[i] = src && d < D ? Q4::load(src + d * EB) : Q4::zero();
      }
#pragma unroll
      for (int i = 0; i < DP / 16; ++i) {
        const int d = 16 * i + 4 * grp;
        if (d < D) *reinterpret_cast<typename Q4::raw *>(dst + d * EB) = w[i];
      }
    } else {
      for (int i = grp; i < D * EB / 4; i += 4)
        reinterpret_cast<uint32_t *>(dst)[i] = src ? reinterpret_cast<const uint32_t *>(src)[i] : 0u;
    }
  }
}

template <typename Tag>
hipError_t launch_dim(const PrefillParams &p, int vec, hipStream_t s) {
  const dim3 grid((unsigned)(p.row_blocks * p.bh_pad)), wg(64 * FWAVES);
  if (p.head_dim <= 32) paged_prefill_f32_kernel<Tag, 32><<<grid, wg, 0, s>>>(p, vec);
  else if (p.head_dim <= 64) paged_prefill_f32_kernel<Tag, 64><<<grid, wg, 0, s>>>(p, vec);
  else if (p.head_dim <= 96) paged_prefill_f32_kernel<Tag, 96><<<grid, wg, 0, s>>>(p, vec);
  else if (p.head_dim <= 128) paged_prefill_f32_kernel<Tag, 128><<<grid, wg, 0, s>>>(p, vec);
  else paged_prefill_f32_kernel<Tag, 256><<<grid, wg, 0, s>>>(p, vec);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_prefill_f32(PrefillParams p, int dtype, hipStream_t s) {
  const int64_t rows = p.width * p.heads_per_kv;
  p.row_blocks = (rows + FROWS - 1) / FROWS;
  p.bh_pad = (p.batch * p.num_kv_heads + 7) / 8 * 8;
  if (p.row_blocks * p.bh_pad > 0x7fffffffLL) return hipErrorInvalidValue;
  // whole-quad loads: every row of every tensor aligned to four elements
  const int64_t strides[] = {p.q_sb, p.q_sh, p.q_st, p.k_sb, p.k_st, p.k_sh, p.v_sb,
                             p.v_st, p.v_sh, p.o_sb, p.o_sh, p.o_st, p.head_dim};
  const uintptr_t bytes = dtype == IKL_F32 ? 16 : 8;
  int vec = (((uintptr_t)p.q | (uintptr_t)p.kc | (uintptr_t)p.vc | (uintptr_t)p.out) & (bytes - 1)) == 0;
  for (int64_t st : strides) vec &= st % 4 == 0;
  if (dtype == IKL_BF16) return launch_dim<bf16_tag>(p, vec, s);
  if (dtype == IKL_F16) return launch_dim<f16_tag>(p, vec, s);
  return launch_dim<f32_tag>(p, vec, s);
}

}  // namespace ikl
