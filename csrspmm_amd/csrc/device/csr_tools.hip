// Device-side CSR tooling: dense -> CSR, the longest row, and int64 -> int32
// index narrowing, all on the caller's stream with no host synchronisation.
//
// dense -> CSR follows the reference's host dense2csr (src/host/csr_utils.cpp
// :70-111): an element is kept when fabsf(v) > tol (so +-0 and NaN are
// dropped), in row-major order.  It runs in two steps because the output
// size is data-dependent: csrspmm_dense2csr_count_f32 writes rowptr and the
// nonzero count (both in device memory); the caller allocates colidx/vals
// from the count and calls csrspmm_dense2csr_fill_f32.  With a scratch (the
// _ex forms) the first step keeps each element's verdict and the kept values,
// and the second does not read the dense matrix again.

#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../../include/csrspmm_c.h"
#include "common.hpp"
#include "spmm_internal.h"

namespace csrspmm_hip {
namespace {

constexpr int kToolBlock = 256;
constexpr int kToolMaxBlocks = 8192;
constexpr int kScanThreads = 1024;
constexpr int kWavesPerBlock = kToolBlock / 64;

__device__ __forceinline__ bool keep(float v, float tol) { return fabsf(v) > tol; }

// Dense -> CSR reads the matrix once where the scratch allows, and is bound by
// that read.  A wave takes a part of a row, kStepCols columns a step, eight
// consecutive ones a lane (two 16-byte loads, which need 4-byte alignment
// only): 32 bytes a lane in flight and the next step's before this one is
// used, where one 4-byte load a lane and step had left the read waiting.  The
// verdicts of a lane make one byte of the part's mask (1/32 of the matrix),
// and the kept values go to the part's stage, in order, as far as it holds
// them; the fill then writes columns from the mask and copies the values, and
// only a part with more reads its columns of the matrix again (figures at
// dense2csr_layout).
constexpr int kStepCols = 512;
constexpr int kPartCols = 4 * kStepCols;  // columns of a part, at most

typedef float f4_unaligned __attribute__((ext_vector_type(4), aligned(4)));

// Lane's eight values of columns c .. c + 7 below c_end (0 past it).
__device__ __forceinline__ void load8(const float* a, int c, int c_end, float (&v)[8]) {
  if (c + 8 <= c_end) {
    const f4 x = *reinterpret_cast<const f4_unaligned*>(a + c);
    const f4 y = *reinterpret_cast<const f4_unaligned*>(a + c + 4);
    v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
    v[4] = y.x, v[5] = y.y, v[6] = y.z, v[7] = y.w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = c + i < c_end ? a[c + i] : 0.0f;
  }
}

// The columns [c_begin, c_end) of a row by one wave: emit(column, lane's
// first kept index, verdict bits, values) each step; returns the kept count.
template <class Emit>
__device__ __forceinline__ int scan_columns(const float* a, int c_begin, int c_end, float tol, Emit&& emit) {
  const int lane = lane_id();
  int n = 0;
  float v[8];
  load8(a, c_begin + lane * 8, c_end, v);
  for (int c0 = c_begin; c0 < c_end; c0 += kStepCols) {
    float next[8];
    if (c0 + kStepCols < c_end) load8(a, c0 + kStepCols + lane * 8, c_end, next);
    const int c = c0 + lane * 8;
    unsigned bits = 0;
    int at = n;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bool k = c + i < c_end && keep(v[i], tol);
      bits |= (unsigned)k << i;
      const unsigned long long m = __ballot(k);
      at = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)at));
      n += __popcll(m);
    }
    emit(c, at, bits, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = next[i];
  }
  return n;
}

// Writes the kept elements of columns [c_begin, c_end) at colidx / vals.
__device__ __forceinline__ void write_columns(const float* a, int c_begin, int c_end, float tol, int* colidx,
                                              float* vals) {
  scan_columns(a, c_begin, c_end, tol, [&](int c, int at, unsigned bits, const float(&v)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (bits & (1u << i)) {
        colidx[at] = c + i;
        vals[at] = v[i];
        ++at;
      }
    }
  });
}

// One wave per row: rowptr[row + 1] = kept elements of the row.
__global__ __launch_bounds__(kToolBlock) void d2c_count_kernel(int M, int K, const float* A,
                                                               long long lda, float tol,
                                                               int* rowptr) {
  for (int row = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6); row < M; row += gridDim.x * kWavesPerBlock) {
    const int cnt = scan_columns(A + (long long)row * lda, 0, K, tol,
                                 [](int, int, unsigned, const float(&)[8]) {});
    if (lane_id() == 0) rowptr[row + 1] = cnt;
  }
}

// One wave per row: its kept elements, in column order.
__global__ __launch_bounds__(kToolBlock) void d2c_fill_kernel(int M, int K, const float* A,
                                                              long long lda, float tol,
                                                              const int* rowptr, int* colidx,
                                                              float* vals) {
  for (int row = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6); row < M; row += gridDim.x * kWavesPerBlock) {
    const int at = rowptr[row];
    write_columns(A + (long long)row * lda, 0, K, tol, colidx + at, vals + at);
  }
}

// Scratch of the one-read form.  Unit u = row * parts + part: its count at
// cnt[u], the index of its first kept element, from the scan, at at[u] (one
// more holds the total), its verdicts at mask + u * width / 8, bit by column, and up to
// `cap` of its kept values at stage + u * cap.  Three values in eight stay in
// the stage: beyond, writing and reading them back costs as much as reading
// the part again.  Below kScratchMinCols columns the mask and stage of a part
// exceed the row itself, and beyond kScratchMaxBytes the scratch is refused:
// both read the matrix twice.
// Measured on MI355X through dense_to_csr, two reads of one 4-byte load a
// lane -> one read: 8192^2 at 5%: count 61.8 -> 53.8 us (5.4 TB/s), scan 7.7 ->
// 7.1, fill 79.3 -> 18.1; the whole call 186 -> 95 us, with the count written
// to host memory by the scan instead of copied.
constexpr int kScratchMinCols = 256;
constexpr long long kScratchMaxUnits = 1 << 26;
constexpr size_t kScratchMaxBytes = (size_t)8 << 30;
struct D2cLayout {
  int parts, width, cap;
  long long units;
  size_t at_off, mask_off, stage_off, total;  // cnt at 0; total 0: no scratch
};
D2cLayout dense2csr_layout(int M, int K) {
  D2cLayout L{};
  if (M <= 0 || K < kScratchMinCols) return L;
  const int n = (int)(((long long)K + kPartCols - 1) / kPartCols);
  L.width = (int)((((long long)K + n - 1) / n + kStepCols - 1) / kStepCols * kStepCols);
  L.parts = (int)(((long long)K + L.width - 1) / L.width);
  L.cap = L.width / 8 * 3;
  L.units = (long long)M * L.parts;
  if (L.units > kScratchMaxUnits) return L;
  auto align = [](size_t x) { return (x + 255) & ~size_t(255); };
  L.at_off = align((size_t)L.units * sizeof(int));
  L.mask_off = align(L.at_off + ((size_t)L.units + 1) * sizeof(int));
  L.stage_off = align(L.mask_off + (size_t)L.units * (L.width / 8));
  const size_t total = align(L.stage_off + (size_t)L.units * L.cap * sizeof(float));
  if (total <= kScratchMaxBytes) L.total = total;
  return L;
}

// One wave per unit: its verdicts, the values its stage holds, its count.
__global__ __launch_bounds__(kToolBlock) void d2c_stage_kernel(int K, const float* A, long long lda, float tol,
                                                               D2cLayout L, char* scratch) {
  const long long u = (long long)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
  if (u >= L.units) return;
  const int row = (int)(u / L.parts);
  const int c_begin = (int)(u - (long long)row * L.parts) * L.width;
  const int c_end = min(K, c_begin + L.width);
  unsigned char* mask = reinterpret_cast<unsigned char*>(scratch) + L.mask_off + u * (L.width / 8);
  float* stage = reinterpret_cast<float*>(scratch + L.stage_off) + u * L.cap;
  const int n = scan_columns(A + (long long)row * lda, c_begin, c_end, tol,
                             [&](int c, int at, unsigned bits, const float(&v)[8]) {
                               mask[(c - c_begin) >> 3] = (unsigned char)bits;
#pragma unroll
                               for (int i = 0; i < 8; ++i) {
                                 if (bits & (1u << i)) {
                                   if (at < L.cap) stage[at] = v[i];
                                   ++at;
                                 }
                               }
                             });
  if (lane_id() == 0) reinterpret_cast<int*>(scratch)[u] = n;
}

// One wave per unit, after the scan.
__global__ __launch_bounds__(kToolBlock) void d2c_unstage_kernel(int K, const float* A, long long lda, float tol,
                                                                 D2cLayout L, const char* scratch, int* colidx,
                                                                 float* vals) {
  const long long u = (long long)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
  if (u >= L.units) return;
  const int* first = reinterpret_cast<const int*>(scratch + L.at_off);
  const int row = (int)(u / L.parts);
  const int c_begin = (int)(u - (long long)row * L.parts) * L.width;
  const int at = first[u];
  const int n = first[u + 1] - at;
  if (n > L.cap) {
    write_columns(A + (long long)row * lda, c_begin, min(K, c_begin + L.width), tol, colidx + at, vals + at);
    return;
  }
  const int lane = lane_id();
  const float* stage = reinterpret_cast<const float*>(scratch + L.stage_off) + u * L.cap;
  for (int i = lane; i < n; i += 64) vals[at + i] = stage[i];
  // a lane per 32 columns (width / 32 is at most 64); the steps past c_end
  // wrote no verdicts
  const int steps = div_up(min(K - c_begin, L.width), kStepCols);
  unsigned w = 0;
  if (lane < steps * (kStepCols / 32))
    w = reinterpret_cast<const unsigned*>(scratch + L.mask_off + u * (L.width / 8))[lane];
  const int mine = __popc(w);
  int incl = mine;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off);
    if (lane >= off) incl += o;
  }
  int pos = at + incl - mine;
  for (; w; w &= w - 1) colidx[pos++] = c_begin + lane * 32 + __ffs((int)w) - 1;
}

// Sum of x over the block, in every thread; wave_tot: one entry per wave.
__device__ __forceinline__ long long block_sum(long long x, long long* wave_tot) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
  if (lane_id() == 0) wave_tot[threadIdx.x >> 6] = x;
  __syncthreads();
  long long sum = 0;
#pragma unroll
  for (int w = 0; w < kScanThreads / 64; ++w) sum += wave_tot[w];
  __syncthreads();
  return sum;
}

// Exclusive scan of cnt[0 .. units) into at[0 .. units] (at[units] the total);
// rowptr[r] = the scan at unit r * parts, and the 64-bit total goes to
// *total.  Block b scans `chunk` units (a multiple of the block's 4 per
// thread), kScanThreads * 4 a step, after summing all units before them by
// itself: at most kScanBlocks readings of the counts, in parallel, in place of
// one block's chain of steps (32768 units: 19.7 us by one block).
constexpr int kScanBlocks = 32;
__global__ __launch_bounds__(kScanThreads) void scan_units_kernel(const int* cnt, int* at, int units, int parts,
                                                                  int chunk, int* rowptr, long long* total) {
  __shared__ long long wave_tot[kScanThreads / 64];
  const int lane = lane_id();
  const int wave = threadIdx.x >> 6;
  const int begin = (int)blockIdx.x * chunk;
  const int end = min(units, begin + chunk);
  long long mine = 0;
  for (int i = (int)threadIdx.x * 4; i < begin; i += kScanThreads * 4) {
    const int4 x = *reinterpret_cast<const int4*>(cnt + i);
    mine += (long long)x.x + x.y + x.z + x.w;
  }
  long long carry = block_sum(mine, wave_tot);
  for (int base = begin; base < end; base += kScanThreads * 4) {
    const int i0 = base + (int)threadIdx.x * 4;
    int v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = i0 + i < end ? cnt[i0 + i] : 0;
    const int t = v[0] + v[1] + v[2] + v[3];
    int x = t;  // inclusive scan of the thread totals across the wave
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(x, off);
      if (lane >= off) x += y;
    }
    if (lane == 63) wave_tot[wave] = x;
    __syncthreads();
    long long before = carry + x - t;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w) {
      if (w < wave) before += wave_tot[w];
      carry += wave_tot[w];
    }
    int o = (int)before;
    int r = i0 / parts;
    int past = i0 - r * parts;  // units since the row's first
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i0 + i < end) {
        at[i0 + i] = o;
        if (past == 0) rowptr[r] = o;
      }
      o += v[i];
      if (++past == parts) {
        past = 0;
        ++r;
      }
    }
    __syncthreads();  // wave_tot is rewritten by the next step
  }
  if (end == units && threadIdx.x == 0) {
    at[units] = (int)carry;
    rowptr[units / parts] = (int)carry;
    *total = carry;
  }
}

// In-place inclusive scan of rowptr[1..M] by one workgroup, 4096 entries per
// step with the running total carried between steps; rowptr[0] = 0 and the
// 64-bit total goes to *total.
__global__ __launch_bounds__(kScanThreads) void scan_rowptr_kernel(int* rowptr, int M,
                                                                   long long* total) {
  __shared__ long long wave_tot[kScanThreads / 64];
  constexpr int kItems = 4;
  const int lane = lane_id();
  const int wave = threadIdx.x >> 6;
  long long carry = 0;
  for (int base = 1; base <= M; base += kScanThreads * kItems) {
    const int i0 = base + threadIdx.x * kItems;
    long long v[kItems];
    long long t = 0;
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      v[i] = (i0 + i <= M) ? rowptr[i0 + i] : 0;
      t += v[i];
      v[i] = t;  // inclusive within the thread
    }
    // inclusive scan of the thread totals across the wave
    long long x = t;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const long long y = __shfl_up(x, off);
      if (lane >= off) x += y;
    }
    if (lane == 63) wave_tot[wave] = x;
    __syncthreads();
    long long before = carry;
    long long step = 0;
    for (int w = 0; w < kScanThreads / 64; ++w) {
      if (w < wave) before += wave_tot[w];
      step += wave_tot[w];
    }
    before += x - t;  // exclusive prefix of this thread
#pragma unroll
    for (int i = 0; i < kItems; ++i)
      if (i0 + i <= M) rowptr[i0 + i] = static_cast<int>(before + v[i]);
    carry += step;
    __syncthreads();  // wave_tot is rewritten by the next step
  }
  if (threadIdx.x == 0) {
    rowptr[0] = 0;
    *total = carry;
  }
}

__global__ void zero_int_kernel(int* p) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0;
}

// *out = max over rows of rowptr[r + 1] - rowptr[r] (0 when M == 0).
__global__ __launch_bounds__(kToolBlock) void max_row_kernel(int M, const int* rowptr, int* out) {
  __shared__ int s_max;
  if (threadIdx.x == 0) s_max = 0;
  __syncthreads();
  int mx = 0;
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < M; r += gridDim.x * blockDim.x)
    mx = max(mx, rowptr[r + 1] - rowptr[r]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = max(mx, __shfl_xor(mx, off));
  if (lane_id() == 0 && mx > 0) atomicMax(&s_max, mx);
  __syncthreads();
  if (threadIdx.x == 0 && s_max > 0) atomicMax(out, s_max);
}

// dst[i] = src[i] for values that fit int32; *overflow = 1 if any does not
// (dst then holds the low 32 bits there).
__global__ __launch_bounds__(kToolBlock) void narrow_kernel(const long long* src, int* dst,
                                                            long long n, int* overflow) {
  bool bad = false;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const long long v = src[i];
    bad |= v < INT32_MIN || v > INT32_MAX;
    dst[i] = static_cast<int>(v);
  }
  if (overflow && __ballot(bad) && lane_id() == 0) *overflow = 1;
}

// dst0[i] = src0[i] for i < n0 and dst1[i] = src1[i] for i < n1, the low 32 bits:
// both index arrays of a CSR in one launch (2^21 entries: 2 x 5.2 us before).
__global__ __launch_bounds__(kToolBlock) void narrow_csr_kernel(const long long* src0, int* dst0, long long n0,
                                                                const long long* src1, int* dst1,
                                                                long long n1) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n0 + n1;
       i += (long long)gridDim.x * blockDim.x) {
    if (i < n0) {
      dst0[i] = static_cast<int>(src0[i]);
    } else {
      dst1[i - n0] = static_cast<int>(src1[i - n0]);
    }
  }
}

int tool_blocks(long long work, int per_block) {
  return static_cast<int>(std::max<long long>(1, std::min<long long>(kToolMaxBlocks, (work + per_block - 1) / per_block)));
}

int status_of(hipError_t e) { return e == hipSuccess ? CSRSPMM_STATUS_SUCCESS : static_cast<int>(e); }

}  // namespace
}  // namespace csrspmm_hip

using namespace csrspmm_hip;

extern "C" {

int csrspmm_dense2csr_count_f32(int M, int K, const float* dense, long long ld, float tol,
                                int* rowptr, long long* nnz_out, void* stream) {
  if (M < 0 || K < 0 || !rowptr || !nnz_out || (M > 0 && K > 0 && (!dense || ld < K)))
    return CSRSPMM_STATUS_INVALID_VALUE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  if (M > 0) {  // K == 0 leaves every count 0 without touching dense
    hipLaunchKernelGGL(d2c_count_kernel, dim3(tool_blocks(M, kToolBlock / 64)), dim3(kToolBlock), 0,
                       s, M, K, dense, ld, tol, rowptr);
  }
  hipLaunchKernelGGL(scan_rowptr_kernel, dim3(1), dim3(kScanThreads), 0, s, rowptr, M, nnz_out);
  return status_of(hipGetLastError());
}

int csrspmm_dense2csr_fill_f32(int M, int K, const float* dense, long long ld, float tol,
                               const int* rowptr, int* colidx, float* vals, void* stream) {
  if (M < 0 || K < 0 || !rowptr || (M > 0 && K > 0 && (!dense || ld < K)))
    return CSRSPMM_STATUS_INVALID_VALUE;
  if (M == 0 || K == 0) return CSRSPMM_STATUS_SUCCESS;
  hipStream_t s = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  hipLaunchKernelGGL(d2c_fill_kernel, dim3(tool_blocks(M, kToolBlock / 64)), dim3(kToolBlock), 0,
                     s, M, K, dense, ld, tol, rowptr, colidx, vals);
  return status_of(hipGetLastError());
}

size_t csrspmm_dense2csr_scratch_bytes(int M, int K) { return dense2csr_layout(M, K).total; }

int csrspmm_dense2csr_count_f32_ex(int M, int K, const float* dense, long long ld, float tol, int* rowptr,
                                   long long* nnz_out, void* scratch, size_t scratch_bytes, void* stream) {
  const D2cLayout L = dense2csr_layout(M, K);
  if (L.total == 0 || !scratch)
    return csrspmm_dense2csr_count_f32(M, K, dense, ld, tol, rowptr, nnz_out, stream);
  if (!rowptr || !nnz_out || !dense || ld < K || (reinterpret_cast<uintptr_t>(scratch) & 255))
    return CSRSPMM_STATUS_INVALID_VALUE;
  if (scratch_bytes < L.total) return CSRSPMM_STATUS_WORKSPACE_TOO_SMALL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  const int blocks = (int)((L.units + kWavesPerBlock - 1) / kWavesPerBlock);
  hipLaunchKernelGGL(d2c_stage_kernel, dim3(blocks), dim3(kToolBlock), 0, s, K, dense, ld, tol, L,
                     static_cast<char*>(scratch));
  const int step = kScanThreads * 4;
  const int chunk = (int)((L.units + (long long)kScanBlocks * step - 1) / ((long long)kScanBlocks * step)) * step;
  hipLaunchKernelGGL(scan_units_kernel, dim3((unsigned)((L.units + chunk - 1) / chunk)), dim3(kScanThreads), 0, s,
                     static_cast<const int*>(scratch),
                     reinterpret_cast<int*>(static_cast<char*>(scratch) + L.at_off), (int)L.units, L.parts,
                     chunk, rowptr, nnz_out);
  return status_of(hipGetLastError());
}

int csrspmm_dense2csr_fill_f32_ex(int M, int K, const float* dense, long long ld, float tol, const int* rowptr,
                                  int* colidx, float* vals, const void* scratch, size_t scratch_bytes,
                                  void* stream) {
  const D2cLayout L = dense2csr_layout(M, K);
  if (L.total == 0 || !scratch)
    return csrspmm_dense2csr_fill_f32(M, K, dense, ld, tol, rowptr, colidx, vals, stream);
  if (!rowptr || !dense || ld < K || (reinterpret_cast<uintptr_t>(scratch) & 255))
    return CSRSPMM_STATUS_INVALID_VALUE;
  if (scratch_bytes < L.total) return CSRSPMM_STATUS_WORKSPACE_TOO_SMALL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  const int blocks = (int)((L.units + kWavesPerBlock - 1) / kWavesPerBlock);
  hipLaunchKernelGGL(d2c_unstage_kernel, dim3(blocks), dim3(kToolBlock), 0, s, K, dense, ld, tol, L,
                     static_cast<const char*>(scratch), colidx, vals);
  return status_of(hipGetLastError());
}

int csrspmm_csr_max_row_nnz(int M, const int* rowptr, int* max_out, void* stream) {
  if (M < 0 || !max_out || (M > 0 && !rowptr)) return CSRSPMM_STATUS_INVALID_VALUE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  hipLaunchKernelGGL(zero_int_kernel, dim3(1), dim3(64), 0, s, max_out);
  if (M > 0)
    hipLaunchKernelGGL(max_row_kernel, dim3(tool_blocks(M, kToolBlock)), dim3(kToolBlock), 0, s, M,
                       rowptr, max_out);
  return status_of(hipGetLastError());
}

int csrspmm_indices_i64_to_i32(const long long* src, int* dst, long long n, int* overflow_out,
                               void* stream) {
  if (n < 0 || (n > 0 && (!src || !dst))) return CSRSPMM_STATUS_INVALID_VALUE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  if (overflow_out) hipLaunchKernelGGL(zero_int_kernel, dim3(1), dim3(64), 0, s, overflow_out);
  if (n > 0)
    hipLaunchKernelGGL(narrow_kernel, dim3(tool_blocks(n, kToolBlock)), dim3(kToolBlock), 0, s, src,
                       dst, n, overflow_out);
  return status_of(hipGetLastError());
}

int csrspmm_csr_i64_to_i32(const long long* rowptr, int* rowptr_out, long long n_rowptr, const long long* colidx,
                           int* colidx_out, long long n_colidx, void* stream) {
  if (n_rowptr < 0 || n_colidx < 0 || (n_rowptr > 0 && (!rowptr || !rowptr_out)) ||
      (n_colidx > 0 && (!colidx || !colidx_out)))
    return CSRSPMM_STATUS_INVALID_VALUE;
  if (n_rowptr + n_colidx == 0) return CSRSPMM_STATUS_SUCCESS;
  hipStream_t s = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  hipLaunchKernelGGL(narrow_csr_kernel, dim3(tool_blocks(n_rowptr + n_colidx, kToolBlock)), dim3(kToolBlock), 0, s,
                     rowptr, rowptr_out, n_rowptr, colidx, colidx_out, n_colidx);
  return status_of(hipGetLastError());
}

}  // extern "C"
