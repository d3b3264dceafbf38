// Paged prefill for launches of long contexts that leave the chip idle (the
// rule is prefill_key_groups in paged_prefill.hip): the shapes and results
// of paged_prefill_mfma_kernel (paged_prefill.hip), where a workgroup's 4
// waves own 128 rows and walk the keys together. There few rows over long
// prefixes are few workgroups, each a serial chain of all its key tiles, and
// a launch of one or two rounds ends with half-empty CUs.
//
// Here KG waves (1, 2 or 4) share every 32 rows: wave group kg takes the
// 32-key tiles kg, kg + KG, ..., and the groups' (maximum, denominator,
// product) meet in LDS at the end. The chain is KG times shorter and there
// are KG times as many workgroups, for KG times the copies per product.
//
// Bound: the latency of one step (copy to LDS, QK^T, softmax, PV), about
// 0.7 us at KG = 1, times the steps of the longest workgroup. So the loop
// favours few instructions (32x32x16 MFMAs: half as many, one softmax row per
// lane, 8 dot products for the denominators) and runs the next tile's QK^T
// under this one's exponentials. 9 % fewer cycles than the 16x16x32 loop on
// the ragged chunks below. At 8 x 4096 it is 6 % fewer (2.68 -> 2.52 M), but
// that launch meets the power limit: the clock falls from 2219-2226 to
// 2000-2040 MHz and it takes 1234-1260 us against 1201-1207 (medians of two
// counter runs), which is why the other kernel stays.
//
// 32/8 heads of 128, bf16, against paged_prefill_mfma_kernel: 4 requests x
// (2000 + 64 tokens) 57.6 -> 28.9 us, 1 x 1024 tokens 32.1 -> 23.8, 2 x 1024
// 36.6 -> 32.8; 4 ragged chunks (1024-3072 + 517-1024) over the FP8 cache
// 222 -> 205.
#include "ikl_common.h"
#include "mfma_ops.h"
#include "paged_attn.h"
#include "paged_prefill.h"

namespace ikl {
namespace {

constexpr int PT = 32;     // keys per tile
constexpr int PWAVES = 4;  // waves per workgroup

// KV8: the cache holds E4M3 codes with per-row scales; the copy stages
// round(code * scale) as 16-bit values.
template <typename Tag, int D, int KG, bool KV8>
__global__ __launch_bounds__(64 * PWAVES, KG == 4 && D == 128 ? 1 : 2) void paged_prefill_split_kernel(
    const PrefillParams p) {
  static_assert(D % 32 == 0 && D <= 128, "head_dim = 32k <= 128");
  static_assert(KG == 1 || KG == 2 || KG == 4, "waves per row");
  using ops = mfma_ops<Tag>;
  constexpr int EB = 2;
  constexpr int ROWB = D * EB;           // bytes per staged row
  constexpr int PIECES = ROWB / 16;      // 16-byte pieces per staged row
  constexpr int KSTEPS = D / 16;         // QK^T k-steps
  constexpr int MTILES = D / 32;         // PV output tiles of 32 dims
  constexpr int RG = PWAVES / KG;        // row groups of 32
  constexpr int RWG = 32 * RG;           // query rows per workgroup
  constexpr int TILE_BYTES = PT * ROWB;  // one staged K or V tile
  constexpr int CEB = KV8 ? 1 : EB;      // bytes per cache element
  constexpr int CPIECES = D * CEB / 16;  // 16-byte pieces per cache row
  constexpr int PPL = (16 * CPIECES + 63) / 64;  // pieces per lane of a 16-key half
  // Who copies what: KG = 1: each wave a 16-key half of the step's K or V
  // tile; KG = 2: each wave the K or V tile of its key group; both stage it
  // twice, one barrier a step. KG = 4: a tile is one wave's own, both
  // matrices, staged once.
  constexpr int STAGES = KG == 4 ? 1 : 2;
  constexpr int MATS = KG == 4 ? 2 : 1;   // matrices a wave copies
  constexpr int HALVES = KG == 1 ? 1 : 2;  // halves of each
  // merge: per wave past the first group, 64 lanes x (16 MTILES sums, maximum, denominator)
  constexpr int MERGE_BYTES = 64 * 4 * (16 * MTILES + 2);
  constexpr int LDS_BYTES = STAGES * KG * 2 * TILE_BYTES;
  __shared__ __attribute__((aligned(16))) char
      lds[LDS_BYTES > (PWAVES - RG) * MERGE_BYTES ? LDS_BYTES : (PWAVES - RG) * MERGE_BYTES];

  // Place of 16-byte piece c of a staged K / V row (bijective per row).
  // gfx950 serves a 16-byte LDS read conflict-free when each 16 consecutive
  // lanes hit 16 distinct pieces of a 256-byte window and lanes l and l + 16
  // stay in the same 64-byte quarter of it. A K read's lanes take one piece
  // of 32 rows: the rows of a 16-row half (and, alike, of the other) spread
  // it over the window. A transposing V read takes 64 bytes of four
  // consecutive rows, which go to distinct quarters. Rows of 12 pieces do
  // most of that by their pitch.
  auto kpos = [](int row, int c) {
    if constexpr (PIECES == 12) return row * ROWB + (c + ((row >> 2) & 3)) % 12 * 16;
    else return row * ROWB + ((c ^ (row * PIECES >> 4)) & (PIECES - 1)) * 16;
  };
  auto vpos = [](int row, int c) {
    if constexpr (PIECES < 8 || PIECES == 12) return row * ROWB + c * 16;
    else return row * ROWB + (c ^ (4 * ((PIECES == 16 ? row : row >> 1) & (PIECES / 4 - 1)))) * 16;
  };

  const int tid = threadIdx.x;
  const int lane = tid & 63, hl = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave % RG, kg = wave / RG;

  // All row blocks of one (request, kv head) share blockIdx.x mod 8, hence
  // one XCD and its L2; those nearest the end of the prompts start first.
  // paired (one resident round, two workgroups per CU): the second half of
  // the launch takes the short row blocks in rising order, so that the
  // longest share their CU with the shortest (2 x 1024 tokens 34.0 -> 32.8 us,
  // over the FP8 cache 36.3 -> 34.5; nothing at two groups).
  const int64_t idx = blockIdx.x;
  const int64_t bh = idx % p.bh_pad, turn = idx / p.bh_pad;
  const int64_t rb = p.paired && 2 * turn >= p.row_blocks ? turn - (p.row_blocks + 1) / 2 : p.row_blocks - 1 - turn;
  if (bh >= p.batch * p.num_kv_heads) return;
  const int64_t b = bh / p.num_kv_heads;
  const int kvh = (int)(bh % p.num_kv_heads);
  const int G = p.heads_per_kv;

  int64_t start64, end64, nrows;
  pf_range(p, b, &start64, &end64, &nrows);
  // positions fit in 31 bits (the host bounds table_width * block_size)
  const int start = (int)start64, end = (int)end64;
  const int64_t rows_valid = nrows * G, rows_all = p.width * G;
  const int64_t row0 = rb * RWG;
  const int64_t wr0 = row0 + 32 * rg;

  // keys the workgroup needs, and the wave's own causal window
  const int64_t wg_last = (row0 + RWG < rows_valid ? row0 + RWG : rows_valid) - 1;
  const int kv_hi = wg_last >= row0 ? start + (int)(wg_last / G) + 1 : 0;
  const int n_tiles = (kv_hi + PT - 1) / PT;
  const int n_steps = (n_tiles + KG - 1) / KG;
  const int64_t w_last = (wr0 + 32 < rows_valid ? wr0 + 32 : rows_valid) - 1;
  const int w_hi = w_last >= wr0 ? start + (int)(w_last / G) + 1 : 0;  // keys [0, w_hi) reach some row
  const int w_lo = start + (int)(wr0 / G);                             // every row sees keys <= w_lo

  // Q^T operands and the position of the lane's row (-1: not attending)
  v4u32 qb[KSTEPS];
  int qpos;
  {
    const int64_t r = wr0 + hl;
    const bool ok = r < rows_valid;
    const int64_t t = ok ? r / G : 0;
    const int h = ok ? (int)(r % G) : 0;
    qpos = ok ? start + (int)t : -1;
    const char *qrow = p.q + (b * p.q_sb + ((int64_t)kvh * G + h) * p.q_sh + t * p.q_st + 8 * half) * EB;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) qb[s] = ok ? load16v_global(qrow + 32 * s) : zero4();
  }
  // Wait for Q here: otherwise the loop's first MFMA would wait for every
  // load in flight, the next tiles' prefetch included.
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s) asm volatile("" ::"v"(qb[s]));

  f32x16_t acc[MTILES];
#pragma unroll
  for (int mt = 0; mt < MTILES; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[mt][i] = 0.f;
  float m = NEG_SENTINEL;    // running max of the lane's row, log2 domain (scaled)
  float thr = NEG_SENTINEL;  // (m + RESCALE_LOG2) in raw score units (scale > 0)
  float lsum = 0.f;          // this lane's share of the row's denominator
  const float inv_scale_log2 = 1.f / p.scale_log2;

  // LDS offsets. MFMA row rho of S^T holds key kappa(rho), chosen so that
  // the 16 scores of a lane are keys 16 (i / 8) + 8 half + i % 8: the P
  // operands of the two 16-deep PV steps.
  const int kappa = 16 * (hl >> 4) + 8 * ((hl >> 2) & 1) + 4 * ((hl >> 3) & 1) + (hl & 3);
  int k_off[KSTEPS];
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s) k_off[s] = kpos(kappa, 2 * s + half);
  // ds_read_b64_tr_b16: lane 4k + d of a 16-lane group supplies key k, dims
  // 4d..4d+3 of the group's four keys x 16 dims. Keys 4, 8 and 16 further on
  // keep a row's swizzle: constants.
  const int vrow = 8 * half + ((lane >> 2) & 3);
  int v_off[MTILES];
#pragma unroll
  for (int mt = 0; mt < MTILES; ++mt)
    v_off[mt] = vpos(vrow, 4 * mt + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + 8 * (lane & 1);

  // The copy. Matrix x of this wave: K (0) or V (1).
  auto mat = [&](int x) { return KG == 4 ? x : KG == 2 ? rg : wave >> 1; };
  const int hf0 = KG == 1 ? wave & 1 : 0;  // first half copied
  int row_bytes[MATS];
  const char *cp_base[MATS], *cp_scale[MATS];
#pragma unroll
  for (int x = 0; x < MATS; ++x) {
    const bool v = mat(x) != 0;
    row_bytes[x] = (int)((v ? p.v_st : p.k_st) * CEB);
    cp_base[x] = v ? p.vc + (int64_t)kvh * p.v_sh * CEB : p.kc + (int64_t)kvh * p.k_sh * CEB;
    cp_scale[x] = KV8 ? (const char *)(v ? p.v_scale : p.k_scale) + (int64_t)kvh * p.s_sh * 4 : nullptr;
  }
  // Piece u of this lane: cache piece c of row r of a 16-key half.
  int cp_row[PPL], cp_c[PPL];
  bool cp_ok[PPL];
#pragma unroll
  for (int u = 0; u < PPL; ++u) {
    const int pi = u * 64 + lane, r = pi / CPIECES;
    cp_ok[u] = pi < 16 * CPIECES;
    cp_row[u] = r < 16 ? r : 15;
    cp_c[u] = pi % CPIECES;
  }

  // The block table as a window of 64 consecutive 16-key halves, one per
  // lane: the byte offset of the half's first row from the matrix' base (and,
  // for FP8, of its first row scale), plus a bit of `holes_w` for each half
  // whose block lies outside the cache (block_size % 16 == 0: a half never
  // straddles two blocks).
  int hbase = 0;
  uint32_t woff_lo[MATS], woff_hi[MATS], wsc_lo = 0, wsc_hi = 0;
  uint64_t holes_w;
  auto load_window = [&](int h0) {
    const uint32_t pos = 16u * (uint32_t)(h0 + lane);
    const uint32_t lb = pos / (uint32_t)p.block_size;
    const int ph = pf_block(p, b, lb);
    const int64_t in_blk = pos - (int64_t)lb * p.block_size;
#pragma unroll
    for (int x = 0; x < MATS; ++x) {
      const int64_t sb = (mat(x) ? p.v_sb : p.k_sb) * CEB, st = row_bytes[x];
      const int64_t off = ph >= 0 ? ph * sb + in_blk * st : 0;
      woff_lo[x] = (uint32_t)off;
      woff_hi[x] = (uint32_t)((uint64_t)off >> 32);
    }
    if constexpr (KV8) {
      const int64_t so = ph >= 0 ? (ph * p.s_sb + in_blk) * 4 : 0;
      wsc_lo = (uint32_t)so;
      wsc_hi = (uint32_t)((uint64_t)so >> 32);
    }
    holes_w = __builtin_amdgcn_ballot_w64(ph < 0);
#pragma unroll
    for (int x = 0; x < MATS; ++x) asm volatile("" ::"v"(woff_lo[x]), "v"(woff_hi[x]));
  };
  load_window(0);

  // Global -> registers for this wave's part of its group's tile of step j,
  // matrix x. A half is one block window addressed by a buffer resource whose
  // record count ends at the half's last valid row: rows past it (and a whole
  // half whose block is masked) read as zero without a branch.
  v4u32 cd[MATS][HALVES][PPL];
  float cs[MATS][HALVES][PPL];
  uint32_t hb = 0u;  // hole bits of 16 steps, two per step
  auto fetch = [&](int x, int j) {
    const int want = j * KG + kg, tile = want < n_tiles ? want : n_tiles - 1;
    if (2 * tile + 1 - hbase >= 64) {
      hbase = tile > KG ? 2 * (tile - KG) : 0;  // V's tiles follow K's a step behind
      load_window(hbase);
    }
    const int i0 = 2 * tile - hbase;
    const uint32_t holes = (uint32_t)(holes_w >> i0) & 3u;
    const int sh = 2 * (j & 15);
    hb = (hb & ~(3u << sh)) | (holes << sh);
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      const int hf = hf0 + h, left = end - 16 * (2 * tile + hf);
      const int nv = (holes >> hf) & 1u ? 0 : (left <= 0 ? 0 : (left < 16 ? left : 16));
      const uint64_t off = ((uint64_t)__builtin_amdgcn_readlane(woff_hi[x], i0 + hf) << 32) |
                           __builtin_amdgcn_readlane(woff_lo[x], i0 + hf);
      const __amdgpu_buffer_rsrc_t rs =
          __builtin_amdgcn_make_buffer_rsrc((void *)(cp_base[x] + off), (short)0, nv * row_bytes[x], 0x00020000);
#pragma unroll
      for (int u = 0; u < PPL; ++u)
        if (cp_ok[u])
          cd[x][h][u] = __builtin_amdgcn_raw_buffer_load_b128(rs, cp_row[u] * row_bytes[x] + cp_c[u] * 16, 0, 0);
      if constexpr (KV8) {
        const uint64_t so = ((uint64_t)__builtin_amdgcn_readlane(wsc_hi, i0 + hf) << 32) |
                            __builtin_amdgcn_readlane(wsc_lo, i0 + hf);
        const __amdgpu_buffer_rsrc_t ss =
            __builtin_amdgcn_make_buffer_rsrc((void *)(cp_scale[x] + so), (short)0, nv * 4, 0x00020000);
#pragma unroll
        for (int u = 0; u < PPL; ++u)
          if (cp_ok[u]) cs[x][h][u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ss, cp_row[u] * 4, 0, 0));
      }
    }
  };
  // registers -> the group's tile of step j (FP8 codes widened with their row scale)
  auto stage = [&](int j) { return lds + ((j % STAGES) * KG + kg) * 2 * TILE_BYTES; };
  auto store = [&](int x, int j) {
    char *base = stage(j) + mat(x) * TILE_BYTES;
#pragma unroll
    for (int h = 0; h < HALVES; ++h)
#pragma unroll
      for (int u = 0; u < PPL; ++u) {
        if (!cp_ok[u]) continue;
        const int row = 16 * (hf0 + h) + cp_row[u];
        auto at = [&](int c) { return base + (mat(x) ? vpos(row, c) : kpos(row, c)); };
        const v4u32 w = cd[x][h][u];
        if constexpr (KV8) {
          const float sc = cs[x][h][u];
          *reinterpret_cast<v4u32 *>(at(2 * cp_c[u])) =
              v4u32{fp8x2_scaled<Tag>(w.x, sc, false), fp8x2_scaled<Tag>(w.x, sc, true),
                    fp8x2_scaled<Tag>(w.y, sc, false), fp8x2_scaled<Tag>(w.y, sc, true)};
          *reinterpret_cast<v4u32 *>(at(2 * cp_c[u] + 1)) =
              v4u32{fp8x2_scaled<Tag>(w.z, sc, false), fp8x2_scaled<Tag>(w.z, sc, true),
                    fp8x2_scaled<Tag>(w.w, sc, false), fp8x2_scaled<Tag>(w.w, sc, true)};
        } else {
          *reinterpret_cast<v4u32 *>(at(cp_c[u])) = w;
        }
      }
  };

  // S^T of a tile
  auto scores = [&](const char *kt, f32x16_t &S) {
    v4u32 ka[KSTEPS];
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) ka[s] = *reinterpret_cast<const v4u32 *>(kt + k_off[s]);
#pragma unroll
    for (int i = 0; i < 16; ++i) S[i] = 0.f;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) S = ops::mma_32(ka[s], qb[s], S);
  };

  // Everything of a tile's softmax that branches: masks and the rescale.
  // Raw (unscaled) scores: the scale is folded into the exponent.
  auto bound = [&](f32x16_t &S, int base, uint32_t holes_t) {
    if (base + PT - 1 > w_lo) {  // diagonal tile: per-key causal test
      const int lim = qpos - base - 8 * half;
#pragma unroll
      for (int i = 0; i < 16; ++i) S[i] = 16 * (i >> 3) + (i & 7) <= lim ? S[i] : -INFINITY;
    }
    if (holes_t != 0u) {  // halves in blocks outside the cache
#pragma unroll
      for (int i = 0; i < 16; ++i) S[i] = (holes_t >> (i >> 3)) & 1u ? -INFINITY : S[i];
    }
    // Lazy rescale: the row maximum is only needed when a score passes
    // m + RESCALE_LOG2 (scaled), and each lane can test its own 16 scores
    // against that bound in raw units, so the cross-lane reduction runs
    // on those tiles only (the first one and rare growth).
    float lmax = S[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) lmax = fmaxf(lmax, S[i]);
    if (__builtin_amdgcn_ballot_w64(lmax > thr) != 0ull) {
      const float tmax = max_xor32(lmax) * p.scale_log2;
      const bool need = tmax > m + RESCALE_LOG2;
      const float alpha = need ? fast_exp2(m - tmax) : 1.f;
      m = need ? tmax : m;
      thr = (m + RESCALE_LOG2) * inv_scale_log2;
      lsum *= alpha;
#pragma unroll
      for (int mt = 0; mt < MTILES; ++mt) acc[mt] *= alpha;
    }
  };

  // The probabilities of a bounded tile and their product with its V. The
  // denominator sums the rounded probabilities that the product uses.
  auto attend = [&](const f32x16_t &S, const char *vt) {
    v4u32 pb[2];
    const float neg_m = -m;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float a = fast_exp2(fmaf(S[2 * i], p.scale_log2, neg_m));
      const float c = fast_exp2(fmaf(S[2 * i + 1], p.scale_log2, neg_m));
      pb[i >> 2][i & 3] = ops::pack(a, c);
      lsum = elem<Tag>::dot2(pb[i >> 2][i & 3], ops::ONE2, lsum);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int mt = 0; mt < MTILES; ++mt) {
        const char *at = vt + v_off[mt] + 16 * s * ROWB;
        const u32x2_t v0 = lds_read_tr(at), v1 = lds_read_tr(at + 4 * ROWB);
        acc[mt] = ops::mma_32(v4u32{v0.x, v0.y, v1.x, v1.y}, pb[s], acc[mt]);
      }
  };

  // Software pipeline: step j computes the scores of step j + 1's tile and
  // the probabilities and PV product of step j's, so that one tile's
  // exponentials run under the next one's MFMAs. K is therefore staged one
  // step further ahead than V: step j stores K of step j + 2 over K of step j
  // (read in step j - 1) and V of step j + 1 over V of step j - 1, and refills
  // the registers a step further on.
  f32x16_t sa, sb;
  auto lead = [&](int x) { return mat(x) ? 1 : 2; };
  auto refill = [&](int j) {
#pragma unroll
    for (int x = 0; x < MATS; ++x) {
      store(x, j + lead(x));
      fetch(x, j + lead(x) + 1);
    }
  };
  auto compute = [&](int j, f32x16_t &cur, f32x16_t &next) {
    const int base = (j * KG + kg) * PT;
    if (base >= w_hi) return;  // no row of this wave reaches the tile
    bound(cur, base, (hb >> (2 * (j & 15))) & 3u);
    scores(stage(j + 1), next);  // past the last step: of stale rows, never used
    attend(cur, stage(j) + TILE_BYTES);
  };
  auto step = [&](int j, f32x16_t &cur, f32x16_t &next) {
    if constexpr (STAGES == 2) {
      refill(j);
      compute(j, cur, next);
      __syncthreads();
    } else {
      compute(j, cur, next);
      wave_lds_sync();
      refill(j);
      wave_lds_sync();
    }
  };
  if (n_steps > 0) {
    // tiles of steps 0 and (K) 1, then the first scores
#pragma unroll
    for (int x = 0; x < MATS; ++x) {
      fetch(x, 0);
      store(x, 0);
      fetch(x, 1);
    }
    if constexpr (STAGES == 2) {
      if (mat(0) == 0) {
        store(0, 1);
        fetch(0, 2);
      }
      __syncthreads();
      scores(stage(0), sa);
      __syncthreads();
    } else {
      wave_lds_sync();
      scores(stage(0), sa);
      wave_lds_sync();
      store(0, 1);
      fetch(0, 2);
      wave_lds_sync();
    }
  }
  int j = 0;
  for (; j + 1 < n_steps; j += 2) {
    step(j, sa, sb);
    step(j + 1, sb, sa);
  }
  if (j < n_steps) step(j, sa, sb);
  if constexpr (KG == 4) __syncthreads();

  // The groups meet: groups 1.. leave their sums in LDS, group 0 takes them.
  lsum = sum_xor32(lsum);
  if (KG > 1 && kg > 0) {
    float *mine = reinterpret_cast<float *>(lds + (wave - RG) * MERGE_BYTES);
    mine[lane] = m;
    mine[64 + lane] = lsum;
#pragma unroll
    for (int mt = 0; mt < MTILES; ++mt)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *reinterpret_cast<f32x4_t *>(mine + 128 + (4 * mt + c) * 256 + 4 * lane) =
            f32x4_t{acc[mt][4 * c], acc[mt][4 * c + 1], acc[mt][4 * c + 2], acc[mt][4 * c + 3]};
  }
  if constexpr (KG > 1) __syncthreads();
  if (kg > 0) return;
#pragma unroll
  for (int g = 1; g < KG; ++g) {
    const float *theirs = reinterpret_cast<const float *>(lds + (g * RG + rg - RG) * MERGE_BYTES);
    const float mo = theirs[lane], mn = fmaxf(m, mo);
    const float a = fast_exp2(m - mn), c = fast_exp2(mo - mn);
    m = mn;
    lsum = lsum * a + theirs[64 + lane] * c;
#pragma unroll
    for (int mt = 0; mt < MTILES; ++mt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t o = *reinterpret_cast<const f32x4_t *>(theirs + 128 + (4 * mt + q) * 256 + 4 * lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[mt][4 * q + i] = acc[mt][4 * q + i] * a + o[i] * c;
      }
  }

  // Normalise and store. The lane holds dims 32 mt + 8 c + 4 half + i of
  // row hl.
  const int64_t r = wr0 + hl;
  if (r >= rows_all) return;
  const int64_t t = r / G;
  char *dst = p.out + (b * p.o_sb + ((int64_t)kvh * G + r % G) * p.o_sh + t * p.o_st + 4 * half) * EB;
  if (r < rows_valid) {
    const float inv = 1.f / lsum;  // no attended key: 0/0 -> NaN
#pragma unroll
    for (int mt = 0; mt < MTILES; ++mt)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const f32x16_t &o = acc[mt];
        const u32x2_t w = u32x2_t{ops::pack(o[4 * c] * inv, o[4 * c + 1] * inv),
                                  ops::pack(o[4 * c + 2] * inv, o[4 * c + 3] * inv)};
        *reinterpret_cast<u32x2_t *>(dst + 64 * mt + 16 * c) = w;
      }
    return;
  }
  // padding row: the value at position 0 (zero when its block is masked)
  const int ph_first = pf_block(p, b, 0);
  const char *v0row = ph_first >= 0 && end > 0 ? p.vc + (int64_t)kvh * p.v_sh * CEB + (int64_t)ph_first * p.v_sb * CEB : nullptr;
  const float v0scale = KV8 && v0row ? p.v_scale[(int64_t)ph_first * p.s_sb + (int64_t)kvh * p.s_sh] : 0.f;
#pragma unroll
  for (int c = 0; c < 4 * MTILES; ++c) {
    u32x2_t w = u32x2_t{0u, 0u};
    if (v0row) {
      if constexpr (KV8) {
        const uint32_t codes = *reinterpret_cast<const uint32_t *>(v0row + 8 * c + 4 * half);
        w = u32x2_t{fp8x2_scaled<Tag>(codes, v0scale, false), fp8x2_scaled<Tag>(codes, v0scale, true)};
      } else {
        w = *reinterpret_cast<const u32x2_t *>(v0row + (8 * c + 4 * half) * EB);
      }
    }
    *reinterpret_cast<u32x2_t *>(dst + 16 * c) = w;
  }
}

template <typename Tag, int KG, bool KV8>
hipError_t launch_dim(const PrefillParams &p, hipStream_t s) {
  const dim3 grid((unsigned)(p.row_blocks * p.bh_pad)), wg(64 * PWAVES);
  switch (p.head_dim) {
    case 32: paged_prefill_split_kernel<Tag, 32, KG, KV8><<<grid, wg, 0, s>>>(p); break;
    case 64: paged_prefill_split_kernel<Tag, 64, KG, KV8><<<grid, wg, 0, s>>>(p); break;
    case 96: paged_prefill_split_kernel<Tag, 96, KG, KV8><<<grid, wg, 0, s>>>(p); break;
    case 128: paged_prefill_split_kernel<Tag, 128, KG, KV8><<<grid, wg, 0, s>>>(p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename Tag>
hipError_t launch_tag(const PrefillParams &p, int groups, hipStream_t s) {
  if (groups == 1) return p.kv_fp8 ? launch_dim<Tag, 1, true>(p, s) : launch_dim<Tag, 1, false>(p, s);
  if (groups == 2) return p.kv_fp8 ? launch_dim<Tag, 2, true>(p, s) : launch_dim<Tag, 2, false>(p, s);
  if (groups == 4) return p.kv_fp8 ? launch_dim<Tag, 4, true>(p, s) : launch_dim<Tag, 4, false>(p, s);
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_prefill_split(PrefillParams p, int dtype, int groups, hipStream_t s) {
  const int64_t rows = p.width * p.heads_per_kv, per_wg = 32 * PWAVES / groups;
  p.row_blocks = (rows + per_wg - 1) / per_wg;
  p.bh_pad = (p.batch * p.num_kv_heads + 7) / 8 * 8;
  if (p.row_blocks * p.bh_pad > 0x7fffffffLL) return hipErrorInvalidValue;
  p.paired = groups == 1 && p.row_blocks * p.bh_pad <= 512;
  return dtype == IKL_BF16 ? launch_tag<bf16_tag>(p, groups, s) : launch_tag<f16_tag>(p, groups, s);
}

}  // namespace ikl
