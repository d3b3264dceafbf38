// The layer work around the paged attention of a Llama step: RMSNorm with
// the residual add before it, SiLU times the up projection, and the linear
// layers of a decode step with both folded in. Every value is rounded to the
// tensors' dtype where the module sequence rounds (hf_benchmark.py:408-454):
// linear outputs, residual sums, normalised rows, their product with the
// norm's weight, SiLU and its product; sums and products inside an op are
// fp32.
#include "ikl_common.h"
#include "mfma_ops.h"

namespace ikl {
namespace {

// Two elements of a 16-bit dtype, or one fp32, per 32-bit word.
template <typename Tag>
struct words {
  static constexpr int PER = 2;
  __device__ static inline void get(uint32_t w, float *x) {
    x[0] = mfma_ops<Tag>::lo(w);
    x[1] = mfma_ops<Tag>::hi(w);
  }
  __device__ static inline uint32_t put(const float *x) { return mfma_ops<Tag>::pack(x[0], x[1]); }
};
template <>
struct words<f32_tag> {
  static constexpr int PER = 1;
  __device__ static inline void get(uint32_t w, float *x) { x[0] = __uint_as_float(w); }
  __device__ static inline uint32_t put(const float *x) { return __float_as_uint(x[0]); }
};

__device__ inline float wave_sum64(float v) { return sum_xor32(sum_xor16(group_sum<16>(v))); }

// ------------------------------------------------------- RMSNorm (+ residual)
// One workgroup per row, the row in registers between the sum of squares and
// the scaling: each tensor crosses memory once. As separate torch launches
// (seven for the norm, one for the add) 4096 rows of 2048 bf16 took 64 us and
// 16 rows 18 us, all launch gaps and fp32 intermediates; here 6.1 us (5.5 TB/s;
// 9.4 with the add) and 2.1 us.
constexpr int NORM_THREADS = 256;
constexpr int NORM_VECS = 4;  // 16-byte pieces a thread holds: rows of up to 16 KB

struct NormParams {
  const char *x;
  const char *delta;  // nullptr: no residual add
  const char *weight;
  char *sum;          // x + delta (may be x); nullptr without delta
  char *out;
  int64_t x_st, d_st, s_st, o_st;  // row strides, bytes
  int32_t pieces;                  // 16-byte pieces per row
  int32_t packed;                  // out in the order of packed_piece()
  float inv_cols, eps;
};

// Operand order of up to 16 rows of 16-bit elements: the 16-byte pieces that
// the lanes of a wave take for 32 columns of the contraction side by side,
// lane l = row l % 16, piece l / 16, so that a B operand is one contiguous
// 1 KB load. Piece c (8 columns) of a row sits at:
__device__ inline int64_t packed_piece(int64_t row, int64_t c) { return (c >> 2) * 64 + (c & 3) * 16 + row; }

template <typename Tag>
__global__ __launch_bounds__(NORM_THREADS) void add_rms_norm_kernel(const NormParams p) {
  using W = words<Tag>;
  constexpr int PER = W::PER;
  __shared__ float part[NORM_THREADS / 64];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x;
  v4u32 v[NORM_VECS];
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < NORM_VECS; ++u) {
    const int c = tid + NORM_THREADS * u;
    if (c >= p.pieces) continue;
    v[u] = load16v_global(p.x + row * p.x_st + 16 * c);
    if (p.delta) {
      const v4u32 d = load16v_global(p.delta + row * p.d_st + 16 * c);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float a[PER], b[PER];
        W::get(v[u][i], a);
        W::get(d[i], b);
#pragma unroll
        for (int e = 0; e < PER; ++e) a[e] += b[e];
        v[u][i] = W::put(a);
      }
      *reinterpret_cast<v4u32 *>(p.sum + row * p.s_st + 16 * c) = v[u];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float a[PER];
      W::get(v[u][i], a);
#pragma unroll
      for (int e = 0; e < PER; ++e) ss = fmaf(a[e], a[e], ss);
    }
  }
  ss = wave_sum64(ss);
  if ((tid & 63) == 0) part[tid >> 6] = ss;
  __syncthreads();
  ss = (part[0] + part[1]) + (part[2] + part[3]);
  const float r = rsqrtf(ss * p.inv_cols + p.eps);
#pragma unroll
  for (int u = 0; u < NORM_VECS; ++u) {
    const int c = tid + NORM_THREADS * u;
    if (c >= p.pieces) continue;
    const v4u32 w = load16v_global(p.weight + 16 * c);
    v4u32 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float a[PER], g[PER];
      W::get(v[u][i], a);
      W::get(w[i], g);
#pragma unroll
      for (int e = 0; e < PER; ++e) a[e] *= r;
      W::get(W::put(a), a);
#pragma unroll
      for (int e = 0; e < PER; ++e) a[e] *= g[e];
      o[i] = W::put(a);
    }
    *reinterpret_cast<v4u32 *>(p.out + (p.packed ? 16 * packed_piece(row, c) : row * p.o_st + 16 * c)) = o;
  }
}

// ------------------------------------------------------------- SiLU(gate) * up
__device__ inline float silu(float x) { return x / (1.f + expf(-x)); }

// One pass instead of two launches with a tensor between them: 4096 x 5632
// bf16 20 us (6.9 TB/s), 16 rows 2.1 us.
template <typename Tag>
__global__ __launch_bounds__(256) void silu_mul_kernel(const v4u32 *gate, const v4u32 *up, v4u32 *out, int64_t pieces) {
  using W = words<Tag>;
  constexpr int PER = W::PER;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= pieces) return;
  const v4u32 g = load16v_global(gate + i), u = load16v_global(up + i);
  v4u32 o;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float a[PER], b[PER];
    W::get(g[k], a);
    W::get(u[k], b);
#pragma unroll
    for (int e = 0; e < PER; ++e) a[e] = silu(a[e]);
    W::get(W::put(a), a);
#pragma unroll
    for (int e = 0; e < PER; ++e) a[e] *= b[e];
    o[k] = W::put(a);
  }
  out[i] = o;
}

// ------------------------------------------------------- decode linear layers
// y = x W^T for the at most 16 rows of a decode step (one per request).
// Bound: the read of W, once; at these sizes (2-46 MB) as much the latency of
// one load and the launch. So one workgroup owns 16 output columns (16 rows
// of W) and its 8 waves split the contraction in steps of 64, every load of
// up to four steps in flight at once; their partial sums meet in LDS. W goes
// from memory straight into the MFMA's A operand (lane l: 16 bytes of row
// l % 16; the two loads of a step use whole 128-byte lines, the second out of
// the cache: streaming loads were 0.3-1.7 us slower), x into its B operand.
// What follows the product runs here instead of in launches of its own: the
// residual add or SiLU(gate) * up; up to three weights that share x (q, k and
// v) are one launch. Where x comes from a norm or from SiLU(gate) * up, that
// kernel leaves it in operand order: every workgroup reads all of x, and 16
// rows of 64 bytes per load cost 1-2 us more than 1 KB in one piece.
//
// us per launch in a captured graph, weights from memory (columns x
// contraction, 16 rows of bf16 in operand order; in brackets plain rows, then
// the library's product alone):
//   2048 x 2048 + residual  4.5 (5.7; 8.0)   2048 x 5632 + residual 11.2 (14.1; 10.6)
//   5632 x 2048 gate * up  14.1 (15.8; 2 x 12.1)   4096 x 4096  10.1 (12.0; 15.3)
// The read floor of 5632 x 2048 gate * up is 8.9 us at 5.2 TB/s.
//
// RMSNorm of x stays a launch: folded in here, every workgroup repeated it,
// which cost 2.4-3 us (11 us at 5632 columns) against 2.1 us.
constexpr int LIN_WAVES = 8;
constexpr int LIN_STEPS = 4;  // steps of 64 in flight per wave; 8 and 12 measured within noise or slower
enum { LIN_PLAIN = 0, LIN_RESIDUAL = 1, LIN_SILU = 2 };

struct LinearParams {
  const char *x;
  int64_t x_st;  // row stride, bytes; 0: x in operand order (packed_piece)
  const char *w[3];
  char *y[3];
  int64_t y_st[3];   // row strides, bytes
  int32_t tiles[3];  // cumulative 16-column tiles
  const char *res;   // LIN_RESIDUAL: added to y[0] (may be y[0])
  int64_t res_st;
  int32_t rows, steps;  // rows of x; contraction steps of 64
  int32_t y_packed;     // y[0] in operand order
};

template <typename Tag, int EPI>
__global__ __launch_bounds__(64 * LIN_WAVES) void decode_linear_kernel(const LinearParams p) {
  using ops = mfma_ops<Tag>;
  using W2 = words<Tag>;
  constexpr int NB = EPI == LIN_SILU ? 2 : 1;  // weights a workgroup multiplies
  __shared__ __attribute__((aligned(16))) float red[LIN_WAVES][NB][64][4];
  const int tid = threadIdx.x, lane = tid & 63, hl = lane & 15, grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = blockIdx.x;
  const int seg = EPI == LIN_PLAIN ? (tile >= p.tiles[0]) + (tile >= p.tiles[1]) : 0;
  const int t0 = seg == 0 ? tile : tile - p.tiles[seg - 1];
  const int64_t w_st = (int64_t)p.steps * 128;
  const char *wrow[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) wrow[n] = p.w[EPI == LIN_SILU ? n : seg] + (16 * (int64_t)t0 + hl) * w_st + 16 * grp;
  // rows past the last read it again; their columns are not stored
  const bool packed = p.x_st == 0;
  const char *xrow = packed ? p.x + 16 * lane : p.x + (hl < p.rows ? hl : p.rows - 1) * p.x_st + 16 * grp;
  const int64_t x_step = packed ? 2048 : 128, x_half = packed ? 1024 : 64;

  f32x4_t acc[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) acc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // Steps wave, wave + LIN_WAVES, ...: the waves walk neighbouring lines of
  // the same rows.
  for (int s0 = wave; s0 < p.steps; s0 += LIN_WAVES * LIN_STEPS) {
    v4u32 wr[NB][2 * LIN_STEPS], xr[2 * LIN_STEPS];
#pragma unroll
    for (int i = 0; i < 2 * LIN_STEPS; ++i) {
      const int s = s0 + LIN_WAVES * (i >> 1);
      if (s >= p.steps) continue;
      const int64_t off = (int64_t)s * 128 + 64 * (i & 1);
#pragma unroll
      for (int n = 0; n < NB; ++n) wr[n][i] = load16v_global(wrow[n] + off);
      xr[i] = load16v_global(xrow + s * x_step + (i & 1) * x_half);
    }
#pragma unroll
    for (int i = 0; i < 2 * LIN_STEPS; ++i) {
      if (s0 + LIN_WAVES * (i >> 1) >= p.steps) continue;
#pragma unroll
      for (int n = 0; n < NB; ++n) acc[n] = ops::mma_k32(wr[n][i], xr[i], acc[n]);
    }
  }
#pragma unroll
  for (int n = 0; n < NB; ++n) *reinterpret_cast<f32x4_t *>(red[wave][n][lane]) = acc[n];
  __syncthreads();
  // lane l of an accumulator: columns (rows of W) 4 (l / 16) + i, row l % 16.
  // A thread finishes two neighbouring columns of a row.
  if (tid >= 128) return;
  const int row = tid >> 3, c = 2 * (tid & 7), l = row + 16 * (c >> 2), i = c & 3;
  if (row >= p.rows) return;
  float v[NB][2];
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    v[n][0] = v[n][1] = 0.f;
#pragma unroll
    for (int w = 0; w < LIN_WAVES; ++w) {
      v[n][0] += red[w][n][l][i];
      v[n][1] += red[w][n][l][i + 1];
    }
    W2::get(W2::put(v[n]), v[n]);
  }
  const int64_t col = 2 * (16 * (int64_t)t0 + c);  // bytes
  if constexpr (EPI == LIN_RESIDUAL) {
    float h[2];
    W2::get(*reinterpret_cast<const uint32_t *>(p.res + row * p.res_st + col), h);
    v[0][0] += h[0];
    v[0][1] += h[1];
  } else if constexpr (EPI == LIN_SILU) {
    float g[2] = {silu(v[0][0]), silu(v[0][1])};
    W2::get(W2::put(g), g);
    v[0][0] = g[0] * v[1][0];
    v[0][1] = g[1] * v[1][1];
  }
  const int64_t at = EPI == LIN_SILU && p.y_packed ? 16 * packed_piece(row, col >> 4) + (col & 15) : row * p.y_st[seg] + col;
  *reinterpret_cast<uint32_t *>(p.y[seg] + at) = W2::put(v[0]);
}

template <typename Tag>
hipError_t launch_linear(const LinearParams &p, int epi, int grid, hipStream_t s) {
  const dim3 g((unsigned)grid), wg(64 * LIN_WAVES);
  if (epi == LIN_SILU) decode_linear_kernel<Tag, LIN_SILU><<<g, wg, 0, s>>>(p);
  else if (epi == LIN_RESIDUAL) decode_linear_kernel<Tag, LIN_RESIDUAL><<<g, wg, 0, s>>>(p);
  else decode_linear_kernel<Tag, LIN_PLAIN><<<g, wg, 0, s>>>(p);
  return hipGetLastError();
}

bool off16(const void *ptr) { return ((uintptr_t)ptr & 15u) != 0; }

int launched(const char *what, hipError_t e) {
  return e == hipSuccess ? IKL_OK : fail(IKL_ELAUNCH, std::string(what) + ": " + hipGetErrorString(e));
}

}  // namespace
}  // namespace ikl

using namespace ikl;

extern "C" int ikl_add_rms_norm(const ikl_norm_args *a, void *stream) {
  if (!a) return fail(IKL_EINVAL, "rms norm: args is NULL");
  if (a->rows == 0) return IKL_OK;
  if (a->rows < 0 || a->rows > 0x7fffffffLL || a->cols <= 0)
    return fail(IKL_EINVAL, "rms norm: sizes must be positive");
  if (a->dtype != IKL_F16 && a->dtype != IKL_BF16 && a->dtype != IKL_F32)
    return fail(IKL_EINVAL, "rms norm: unknown dtype");
  if (!a->x || !a->weight || !a->out || (a->delta && !a->sum)) return fail(IKL_EINVAL, "rms norm: NULL tensor pointer");
  const int64_t eb = a->dtype == IKL_F32 ? 4 : 2;
  if (a->cols * eb % 16 != 0 || a->cols * eb > 16LL * NORM_THREADS * NORM_VECS)
    return fail(IKL_EUNSUPPORTED, "rms norm: rows must be whole 16-byte pieces of at most 16 KB");
  if (off16(a->x) || off16(a->weight) || off16(a->out) || off16(a->delta) || off16(a->sum) ||
      (a->x_stride * eb | a->delta_stride * eb | a->sum_stride * eb | a->out_stride * eb) % 16 != 0)
    return fail(IKL_EINVAL, "rms norm: rows must be 16-byte aligned");
  NormParams p;
  p.x = (const char *)a->x;
  p.delta = (const char *)a->delta;
  p.weight = (const char *)a->weight;
  p.sum = (char *)a->sum;
  p.out = (char *)a->out;
  p.x_st = a->x_stride * eb;
  p.d_st = a->delta_stride * eb;
  p.s_st = a->sum_stride * eb;
  p.o_st = a->out_stride * eb;
  p.pieces = (int32_t)(a->cols * eb / 16);
  p.packed = a->packed;
  if (a->packed && (eb != 2 || a->cols % 64 != 0 || a->rows > IKL_DECODE_LINEAR_MAX_ROWS))
    return fail(IKL_EINVAL, "rms norm: operand order is for up to 16 rows of whole 64-column steps, 16-bit");
  p.inv_cols = 1.f / (float)a->cols;
  p.eps = a->eps;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)a->rows);
  if (a->dtype == IKL_BF16) add_rms_norm_kernel<bf16_tag><<<grid, NORM_THREADS, 0, s>>>(p);
  else if (a->dtype == IKL_F16) add_rms_norm_kernel<f16_tag><<<grid, NORM_THREADS, 0, s>>>(p);
  else add_rms_norm_kernel<f32_tag><<<grid, NORM_THREADS, 0, s>>>(p);
  return launched("rms norm", hipGetLastError());
}

extern "C" int ikl_silu_mul(const void *gate, const void *up, void *out, int64_t count, int32_t dtype, void *stream) {
  if (count == 0) return IKL_OK;
  if (!gate || !up || !out || count < 0) return fail(IKL_EINVAL, "silu mul: NULL tensor pointer or negative size");
  if (dtype != IKL_F16 && dtype != IKL_BF16 && dtype != IKL_F32) return fail(IKL_EINVAL, "silu mul: unknown dtype");
  const int64_t eb = dtype == IKL_F32 ? 4 : 2, pieces = count * eb / 16, grid = (pieces + 255) / 256;
  if (count * eb % 16 != 0 || off16(gate) || off16(up) || off16(out))
    return fail(IKL_EINVAL, "silu mul: tensors must be whole 16-byte pieces, 16-byte aligned");
  if (grid > 0x7fffffffLL) return fail(IKL_EINVAL, "silu mul: launch too large");
  hipStream_t s = (hipStream_t)stream;
  const v4u32 *g = (const v4u32 *)gate, *u = (const v4u32 *)up;
  if (dtype == IKL_BF16) silu_mul_kernel<bf16_tag><<<dim3((unsigned)grid), 256, 0, s>>>(g, u, (v4u32 *)out, pieces);
  else if (dtype == IKL_F16) silu_mul_kernel<f16_tag><<<dim3((unsigned)grid), 256, 0, s>>>(g, u, (v4u32 *)out, pieces);
  else silu_mul_kernel<f32_tag><<<dim3((unsigned)grid), 256, 0, s>>>(g, u, (v4u32 *)out, pieces);
  return launched("silu mul", hipGetLastError());
}

extern "C" int ikl_decode_linear(const ikl_decode_linear_args *a, void *stream) {
  if (!a) return fail(IKL_EINVAL, "decode linear: args is NULL");
  if (a->rows <= 0 || a->rows > IKL_DECODE_LINEAR_MAX_ROWS || a->cols <= 0)
    return fail(IKL_EINVAL, "decode linear: rows must lie in [1, IKL_DECODE_LINEAR_MAX_ROWS]");
  if (a->dtype != IKL_F16 && a->dtype != IKL_BF16)
    return fail(IKL_EUNSUPPORTED, "decode linear: fp16 and bf16 only");
  if (a->cols % 64 != 0 || a->cols > (1 << 24))
    return fail(IKL_EUNSUPPORTED, "decode linear: cols must be a multiple of 64, at most 2^24");
  if (a->epilogue < LIN_PLAIN || a->epilogue > LIN_SILU) return fail(IKL_EINVAL, "decode linear: unknown epilogue");
  const int want = a->epilogue == LIN_SILU ? 2 : a->epilogue == LIN_RESIDUAL ? 1 : 0;
  if (a->num_weights < 1 || a->num_weights > 3 || (want && a->num_weights != want))
    return fail(IKL_EINVAL, "decode linear: wrong number of weights");
  if (!a->x || off16(a->x) || a->x_stride % 8 != 0)
    return fail(IKL_EINVAL, "decode linear: x rows must be 16-byte aligned");
  if (a->x_packed == 0 && a->x_stride == 0 && a->rows > 1)
    return fail(IKL_EINVAL, "decode linear: x rows must not share a stride of 0");
  if (a->y_packed && (a->epilogue != LIN_SILU || off16(a->y[0]) || a->out_cols[0] % 64 != 0))
    return fail(IKL_EINVAL, "decode linear: only gate * up leaves its output in operand order, in 64-column steps");
  LinearParams p{};
  p.x = (const char *)a->x;
  p.x_st = a->x_packed ? 0 : a->rows > 1 ? a->x_stride * 2 : 16;
  p.y_packed = a->y_packed;
  p.rows = a->rows;
  p.steps = (int32_t)(a->cols / 64);
  int64_t tiles = 0;
  for (int i = 0; i < 3; ++i) {
    if (i < a->num_weights) {
      if (!a->weight[i] || off16(a->weight[i]) || a->out_cols[i] <= 0 || a->out_cols[i] % 16 != 0)
        return fail(IKL_EINVAL, "decode linear: weights must be 16-byte aligned with a multiple of 16 rows");
      p.w[i] = (const char *)a->weight[i];
      if (a->epilogue != LIN_SILU || i == 0) {
        if (!a->y[i] || ((uintptr_t)a->y[i] & 3u) || a->y_stride[i] % 2 != 0)
          return fail(IKL_EINVAL, "decode linear: output rows must be 4-byte aligned");
        p.y[i] = (char *)a->y[i];
        p.y_st[i] = a->y_stride[i] * 2;
        tiles += a->out_cols[i] / 16;
      } else if (a->out_cols[1] != a->out_cols[0]) {
        return fail(IKL_EINVAL, "decode linear: gate and up must have the same size");
      }
    }
    if (tiles > 0x7fffffffLL) return fail(IKL_EINVAL, "decode linear: launch too large");
    p.tiles[i] = (int32_t)tiles;
  }
  if (a->epilogue == LIN_RESIDUAL) {
    if (!a->residual || ((uintptr_t)a->residual & 3u) || a->residual_stride % 2 != 0)
      return fail(IKL_EINVAL, "decode linear: residual rows must be 4-byte aligned");
    p.res = (const char *)a->residual;
    p.res_st = a->residual_stride * 2;
  }
  hipStream_t s = (hipStream_t)stream;
  const hipError_t e = a->dtype == IKL_BF16 ? launch_linear<bf16_tag>(p, a->epilogue, (int)tiles, s)
                                            : launch_linear<f16_tag>(p, a->epilogue, (int)tiles, s);
  return launched("decode linear", e);
}
