// Value checks of a decode launch's block tables and context lengths
// (triton_ops.py:439-457 makes them with three torch reductions, each read
// back to the host): one kernel over both tensors, whose findings go
// straight to pinned host memory that the host polls.
//
// Bound: latency. As eight elementwise and reduction launches with four
// read-backs the checks were two thirds of an eager call; with one launch,
// polled while the host prepares the attention's arguments, a pass of append
// + checked attention went from 133-144 us to 56 us (32/8 heads of 64; fp32
// 4 x 512 and fp16 16 x 2048).
#include <atomic>

#include "ikl_common.h"

namespace ikl {
namespace {

constexpr int CHECK_THREADS = 512;
constexpr int CHECK_WAVES = CHECK_THREADS / 64;
constexpr int CHECK_SEG = 256;  // table entries a wave takes at a time: four loads in flight per lane

struct CheckParams {
  const void *tables;
  const void *lens;
  int64_t t_sb, t_sw, l_sb;  // elements
  int64_t batch, width, segs;
  int64_t capacity, num_blocks, max_context;
  int32_t table_i64, lens_i64;
  uint32_t *flags;  // one word per workgroup, host memory
};

__device__ inline int64_t entry(const void *base, int64_t i, int i64) {
  return i64 ? load_index<int64_t>(base, i) : load_index<int32_t>(base, i);
}

__global__ __launch_bounds__(CHECK_THREADS) void check_metadata_kernel(const CheckParams p) {
  __shared__ uint32_t found;
  if (threadIdx.x == 0) found = 0u;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  uint32_t bits = 0u;
  const int64_t waves = (int64_t)gridDim.x * CHECK_WAVES;
  for (int64_t i = (int64_t)blockIdx.x * CHECK_WAVES + (threadIdx.x >> 6); i < p.batch * p.segs; i += waves) {
    const int64_t b = i / p.segs, w0 = (i - b * p.segs) * CHECK_SEG;
#pragma unroll
    for (int u = 0; u < CHECK_SEG / 64; ++u) {
      const int64_t w = w0 + 64 * u + lane;
      if (w < p.width) {
        const int64_t e = entry(p.tables, b * p.t_sb + w * p.t_sw, p.table_i64);
        if (e < 0 || e >= p.num_blocks) bits |= IKL_CHECK_BLOCK_ID;
      }
    }
  }
  for (int64_t b = (int64_t)blockIdx.x * CHECK_THREADS + threadIdx.x; b < p.batch;
       b += (int64_t)gridDim.x * CHECK_THREADS) {
    const int64_t n = entry(p.lens, b * p.l_sb, p.lens_i64);
    if (n <= 0) bits |= IKL_CHECK_LENGTH_POSITIVE;
    if (n > p.capacity) bits |= IKL_CHECK_LENGTH_CAPACITY;
    if (n > p.max_context) bits |= IKL_CHECK_LENGTH_MAX;
  }
  if (bits) atomicOr(&found, bits);
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(&p.flags[blockIdx.x], found, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace
}  // namespace ikl

using namespace ikl;

extern "C" int32_t ikl_check_metadata(const void *tables, int32_t table_type, int64_t table_stride_b,
                                      int64_t table_stride_w, const void *lens, int32_t lens_type,
                                      int64_t lens_stride, int64_t batch, int64_t width, int64_t block_size,
                                      int64_t num_blocks, int64_t max_context, uint32_t *flags, int32_t num_flags,
                                      void *stream) {
  if (!tables || !lens || !flags) return fail(IKL_EINVAL, "check metadata: null pointer");
  if (batch <= 0 || width <= 0 || block_size <= 0 || num_blocks <= 0 || num_flags <= 0)
    return fail(IKL_EINVAL, "check metadata: sizes must be positive");
  if ((table_type != IKL_I32 && table_type != IKL_I64) || (lens_type != IKL_I32 && lens_type != IKL_I64))
    return fail(IKL_EINVAL, "check metadata: unknown index type");
  if (width > INT64_MAX / block_size) return fail(IKL_EINVAL, "check metadata: table_width * block_size is too large");
  hipStream_t s = (hipStream_t)stream;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return fail(IKL_ELAUNCH, "check metadata: the result is read back, which a stream under capture cannot do");
  }
  CheckParams p;
  p.tables = tables;
  p.lens = lens;
  p.t_sb = table_stride_b;
  p.t_sw = table_stride_w;
  p.l_sb = lens_stride;
  p.batch = batch;
  p.width = width;
  p.segs = (width + CHECK_SEG - 1) / CHECK_SEG;
  p.capacity = width * block_size;
  p.num_blocks = num_blocks;
  p.max_context = max_context != 0 ? max_context : INT64_MAX;
  p.table_i64 = table_type == IKL_I64;
  p.lens_i64 = lens_type == IKL_I64;
  p.flags = flags;
  // a workgroup per 16 segments: two for each of its eight waves
  const int64_t want = (batch * p.segs + 2 * CHECK_WAVES - 1) / (2 * CHECK_WAVES);
  const int32_t grid = (int32_t)(want < num_flags ? want : num_flags);
  for (int32_t i = 0; i < grid; ++i) reinterpret_cast<volatile uint32_t *>(flags)[i] = IKL_CHECK_PENDING;
  std::atomic_thread_fence(std::memory_order_seq_cst);
  check_metadata_kernel<<<dim3((unsigned)grid), dim3(CHECK_THREADS), 0, s>>>(p);
  const int rc = check_launch("check metadata");
  return rc < 0 ? rc : grid;
}

extern "C" int32_t ikl_check_metadata_wait(const uint32_t *flags, int32_t count, void *stream) {
  if (!flags || count <= 0) return fail(IKL_EINVAL, "check metadata: no flags to wait for");
  const volatile uint32_t *f = flags;
  uint32_t bits = 0u;
  for (int32_t i = 0; i < count; ++i) {
    // The words arrive within microseconds of the kernel; the stream is
    // asked now and then, so that a launch that failed ends the wait.
    for (int64_t spin = 1; f[i] == IKL_CHECK_PENDING; ++spin) {
      __builtin_ia32_pause();
      if (spin % 4096 != 0) continue;
      const hipError_t e = hipStreamQuery((hipStream_t)stream);
      if (e == hipErrorNotReady) {
        (void)hipGetLastError();
        continue;
      }
      if (e != hipSuccess) return fail(IKL_ELAUNCH, std::string("check metadata: ") + hipGetErrorString(e));
      std::atomic_thread_fence(std::memory_order_seq_cst);
      if (f[i] == IKL_CHECK_PENDING) return fail(IKL_ELAUNCH, "check metadata: the kernel left no result");
    }
    bits |= f[i];
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  return (int32_t)bits;
}
