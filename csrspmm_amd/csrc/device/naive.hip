// Naive and NaiveSmem for gfx950 (reference src/device/csrspmm_naive.cu:11-39,
// src/device/csrspmm_naive_smem.cu:5-44).
//
// Both keep the reference's "one thread per output element C[row, col]"
// decomposition and its sequential CSR-order accumulation, laid out for
// wave64: a wave covers 64 consecutive columns of one row, so the row index,
// its rowptr bounds and every (col, val) pair are wave-uniform and come in
// through the scalar cache (s_load), while each lane gathers one float of the
// B row (256 B per wave per nonzero, coalesced).
//
// NaiveSmem: a block covers up to 256 columns of one row and stages the row's
// (col, val) pairs through LDS in 256-entry chunks, so each pair is read from
// global memory once per block instead of once per wave.  Barriers sit at
// block-uniform trip counts (the reference places __syncthreads inside a
// per-row loop after an early return, csrspmm_naive_smem.cu:19,37,40).

#include "common.hpp"

namespace csrspmm_hip {

namespace {

// Waves of a naive_kernel block; build-time tunable.  Measured on MI355X,
// power-law rows of up to 4096 (65536^2 x 96): 2 waves 114 us, 4 75, 8 85;
// R-MAT N = 64 4 waves 1732 us, 8 1845.
#ifndef CSRSPMM_NAIVE_WAVES
#define CSRSPMM_NAIVE_WAVES 4
#endif
constexpr int kNaiveWaves = CSRSPMM_NAIVE_WAVES;
constexpr int kNaiveUnroll = 8;
// A row is one wave's (or block's) chain of dependent batches: batches of
// kNaiveLongUnroll gathers in flight come before the 8-wide ones and the
// tail.  Measured on MI355X per call against 8 throughout: medium 63.7 ->
// 57.8 us; NaiveSmem XL 1792 -> 1451 us, R-MAT 3858 -> 2913 us (16 or 64 in
// flight: slower).
#ifndef CSRSPMM_NAIVE_LONG_UNROLL
#define CSRSPMM_NAIVE_LONG_UNROLL 32
#endif
constexpr int kNaiveLongUnroll = CSRSPMM_NAIVE_LONG_UNROLL;

// A long row (more than relay_row_min nonzeros) is relayed by a whole block:
// its waves take batches of kNaiveLongUnroll nonzeros in turn, each with its
// batch's gathers in flight while the others add, and hand the 64 sums on
// through LDS, so the products are still added one by one in CSR order.
// Which rows are long: those whose chain by one wave, about 16 nonzeros a
// microsecond, would outlast the whole product at the 8 TB/s that gathers past
// the L2s reach, so at most a few thousand rows are; shorter ones are better
// off side by side, a wave each (4096^2 x 128 with 1229 per row, all relayed:
// 202 -> 2600 us).  A turn is bound by its 32 dependent fmas and the handing
// on, about 17 ns a nonzero against 65 of one wave, which waited for its
// batch's gathers.  Measured on MI355X per call with both (and the scalar row
// offsets below): 65536^2 x 96, rows up to 4096, 266 -> 75 us; XL 1320 -> 676;
// R-MAT N = 64 3110 -> 1732.
constexpr int kNaiveRelayMin = 512;
constexpr long long kNaiveRelayWork = 125000;  // elements gathered per nonzero of chain
inline int relay_row_min(int N, int nnz) {
  return (int)std::min<long long>(0x7fffffff, std::max<long long>(kNaiveRelayMin, (long long)nnz * N / kNaiveRelayWork));
}

// One column of B, gathered row by row (wave-uniform rows).  BUF: B's extent
// is below 4 GiB, so a row is a 32-bit scalar offset of a buffer load (one
// scalar multiply) instead of a 64-bit address a lane.  The address arithmetic
// had bound the short rows: measured on MI355X per call, 16384^2 x 128 with 82
// per row 58 -> 42 us, 30000 x 20000 x 40 with 0-500 171 -> 115, 4096^2 x 128
// with 1229 202 -> 142.
template <bool BUF>
struct BColumn {
  __amdgpu_buffer_rsrc_t rsrc;
  const float* base;
  unsigned rowbytes, colbytes;
  long long ldb;
  __device__ __forceinline__ BColumn(const Problem& p, int col) {
    const int c = min(col, p.N - 1);  // lanes past the last column read it again
    if constexpr (BUF) {
      const long long bytes = (long long)(p.K - 1) * p.ldb * 4 + (long long)p.N * 4;
      rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.B), (short)0, (int)(unsigned)bytes, 0x00020000);
      rowbytes = (unsigned)(p.ldb * 4);
      colbytes = (unsigned)c * 4u;
    } else {
      base = p.B + c;
      ldb = p.ldb;
    }
  }
  __device__ __forceinline__ float operator[](int row) const {
    if constexpr (BUF) {
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                           rsrc, (int)colbytes, (int)((unsigned)row * rowbytes), 0));
    } else {
      return base[(long long)row * ldb];
    }
  }
};

// One tile of 64 columns of one long row [start, end), by the whole block.
// The block's batches are numbered on from `done` over all its rows; *turn is
// the number of the batch to be added next, and the wave that has added batch
// k sets it to k + 1 after the sums, so every wait ends.
template <bool BUF>
__device__ __forceinline__ void relay_row(const Problem& p, int row, int start, int end, int col, int wave, int lane,
                                          float* sums, int* turn, int& done) {
  constexpr int U = kNaiveLongUnroll;
  constexpr int W = kNaiveWaves;
  const int batches = div_up(end - start, U);
  const BColumn<BUF> bc(p, col);
  float b[U];
  // lane u: column and value of nonzero u of batch k; past the row's end the
  // last one's, which are not added
  auto entry = [&](int k, int& c, float& v) {
    const int j = min(start + k * U + (lane & (U - 1)), end - 1);
    c = p.colidx[j];
    v = p.vals[j];
  };
  auto gather = [&](int c) {
#pragma unroll
    for (int u = 0; u < U; ++u) b[u] = bc[__builtin_amdgcn_readlane(c, u)];
  };
  auto value = [&](float v, int u) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), u));
  };
  int k = wave;
  if (k < batches) {
    __builtin_amdgcn_s_setprio(3);
    int c, cn;  // of this batch and of the wave's next one
    float v, vn;
    entry(k, c, v);
    gather(c);
    entry(min(k + W, batches - 1), cn, vn);
    for (;;) {
      float sv[U];  // the values in scalar registers before the turn comes
#pragma unroll
      for (int u = 0; u < U; ++u) sv[u] = value(v, u);
      while (__hip_atomic_load(turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != done + k)
        __builtin_amdgcn_s_sleep(1);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
      float sum = k == 0 ? 0.0f : sums[lane];
      const int n = end - start - k * U;
      if (n >= U) {
#pragma unroll
        for (int u = 0; u < U; ++u) sum = __builtin_fmaf(sv[u], b[u], sum);
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float next = __builtin_fmaf(sv[u], b[u], sum);
          sum = u < n ? next : sum;
        }
      }
      sums[lane] = sum;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __hip_atomic_store(turn, done + k + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (k == batches - 1 && col < p.N) {
        float* cp = p.C + (long long)row * p.ldc + col;
        st_c(cp, epi1(p.epi, p.alpha, p.beta, sum, cp));
      }
      k += W;
      if (k >= batches) break;
      v = vn;
      gather(cn);
      entry(min(k + W, batches - 1), cn, vn);
    }
    __builtin_amdgcn_s_setprio(0);
  }
  done += batches;
}

// The first long_blocks * ntile blocks relay the rows of more than long_row
// nonzeros: block i checks rows i, i + long_blocks, ... (64 of them, so that
// neighbouring long rows go to different blocks); the others take a row a
// wave.
template <bool BUF>
__global__ __launch_bounds__(kNaiveWaves * 64) __attribute__((amdgpu_waves_per_eu(8))) void naive_kernel(
    Problem p, int ntile, int long_blocks, int long_row) {
  __shared__ float sums[64];
  __shared__ int turn;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = lane_id();
  const int tile = blockIdx.x % ntile;
  const int block = blockIdx.x / ntile;
  const int col = tile * 64 + lane;
  if (block < long_blocks) {
    const long long r = block + (long long)lane * long_blocks;
    int start = 0, end = 0;
    if (r < p.M) {
      start = p.rowptr[r];
      end = p.rowptr[r + 1];
    }
    unsigned long long rows = __ballot(end - start > long_row);  // the same in every wave
    if (threadIdx.x == 0) turn = 0;
    __syncthreads();
    int done = 0;
    while (rows) {
      const int l = __ffsll((long long)rows) - 1;
      rows &= rows - 1;
      relay_row<BUF>(p, block + l * long_blocks, __builtin_amdgcn_readlane(start, l),
                     __builtin_amdgcn_readlane(end, l), col, wave, lane, sums, &turn, done);
    }
    return;
  }
  const int row = (block - long_blocks) * kNaiveWaves + wave;
  if (row >= p.M) return;
  const int start = p.rowptr[row];
  const int end = p.rowptr[row + 1];
  if (end - start > long_row) return;
  const BColumn<BUF> bc(p, col);
  float sum = 0.0f;
  int j = start;
  // U gathers of the row in flight, then the next U, in CSR order
  auto batch = [&](auto u_const) {
    constexpr int U = decltype(u_const)::value;
    int c[U];
    float v[U];
    float b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      c[u] = p.colidx[j + u];
      v[u] = p.vals[j + u];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) b[u] = bc[c[u]];
#pragma unroll
    for (int u = 0; u < U; ++u) sum = __builtin_fmaf(v[u], b[u], sum);
    j += U;
  };
  while (j + kNaiveLongUnroll <= end) batch(std::integral_constant<int, kNaiveLongUnroll>{});
  while (j + kNaiveUnroll <= end) batch(std::integral_constant<int, kNaiveUnroll>{});
  for (; j < end; ++j) sum = __builtin_fmaf(p.vals[j], bc[p.colidx[j]], sum);
  if (col < p.N) {
    float* cp = p.C + (long long)row * p.ldc + col;
    st_c(cp, epi1(p.epi, p.alpha, p.beta, sum, cp));
  }
}

constexpr int kSmemChunk = 256;

__global__ __launch_bounds__(256) void naive_smem_kernel(Problem p, int ntile, int cols_per_block) {
  __shared__ int s_col[kSmemChunk];
  __shared__ float s_val[kSmemChunk];
  const int tile = blockIdx.x % ntile;
  const int row = blockIdx.x / ntile;  // block-uniform: every barrier below is reached by all threads
  const int t = threadIdx.x;
  const int col = tile * cols_per_block + t;
  const bool valid = col < p.N;
  const int start = p.rowptr[row];
  const int end = p.rowptr[row + 1];
  const float* bc = p.B + col;
  float sum = 0.0f;
  const int nthreads = blockDim.x;
  for (int base = start; base < end; base += kSmemChunk) {
    const int cnt = min(kSmemChunk, end - base);
    for (int i = t; i < cnt; i += nthreads) {
      s_col[i] = ld_stream(p.colidx + base + i);
      s_val[i] = ld_stream(p.vals + base + i);
    }
    __syncthreads();
    int k = 0;
    auto batch = [&](auto u_const) {
      constexpr int U = decltype(u_const)::value;
      float b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) b[u] = valid ? bc[(long long)s_col[k + u] * p.ldb] : 0.0f;
#pragma unroll
      for (int u = 0; u < U; ++u) sum = __builtin_fmaf(s_val[k + u], b[u], sum);
      k += U;
    };
    while (k + kNaiveLongUnroll <= cnt) batch(std::integral_constant<int, kNaiveLongUnroll>{});
    while (k + kNaiveUnroll <= cnt) batch(std::integral_constant<int, kNaiveUnroll>{});
    for (; k < cnt; ++k) {
      const float b = valid ? bc[(long long)s_col[k] * p.ldb] : 0.0f;
      sum = __builtin_fmaf(s_val[k], b, sum);
    }
    __syncthreads();  // chunk fully consumed before the next overwrite
  }
  if (valid) {
    float* cp = p.C + (long long)row * p.ldc + col;
    st_c(cp, epi1(p.epi, p.alpha, p.beta, sum, cp));
  }
}

// Unused LDS that leaves room for 5 blocks (20 waves) a CU instead of 8, for
// rows that average kNaiveCapMean nonzeros or more on a B beyond kNaiveCapBytes:
// their batches of 32 gathers, cheap as they are to issue, push each other's
// B rows out of the L2s.  Measured on MI355X per call, 8 blocks -> 6 -> 5:
// 65536^2 x 256 with 66 per row 504 -> 498 -> 486 us, with 0-200 (60000^2) 681
// -> 667 -> 650, 131072^2 x 128 with 40 352 -> 349 -> 339; but with 30 per row
// 237 -> 258 -> 309, and the relays of skewed rows (mean 16) 75 -> 88 -> 115.
constexpr int kNaiveCapMean = 36;
constexpr long long kNaiveCapBytes = 32LL << 20;
constexpr int kNaiveCapBlocks = 5;
inline unsigned naive_pad_lds(const Problem& p) {
  if (p.nnz < (long long)kNaiveCapMean * p.M || (long long)p.K * p.N * 4 <= kNaiveCapBytes) return 0;
  return (unsigned)(kLdsPerCu / kNaiveCapBlocks / 512 * 512 - 1024);  // the static sums take 512
}

}  // namespace

hipError_t launch_naive(const Problem& p, hipStream_t s) {
  if (p.M == 0 || p.N == 0) return hipSuccess;
  const int ntile = div_up_host(p.N, 64);
  const int long_row = relay_row_min(p.N, p.nnz);
  const int long_blocks = p.nnz > long_row ? div_up_host(p.M, 64) | 1 : 0;
  const long long blocks = ((long long)div_up_host(p.M, kNaiveWaves) + long_blocks) * ntile;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  timing_before_main(s);
  const unsigned pad_lds = naive_pad_lds(p);
  const bool buf = p.K > 0 && (long long)(p.K - 1) * p.ldb * 4 + (long long)p.N * 4 < (1LL << 32);
  if (buf) {
    hipLaunchKernelGGL((naive_kernel<true>), dim3((unsigned)blocks), dim3(kNaiveWaves * 64), pad_lds, s, p,
                       ntile, long_blocks, long_row);
  } else {
    hipLaunchKernelGGL((naive_kernel<false>), dim3((unsigned)blocks), dim3(kNaiveWaves * 64), pad_lds, s, p,
                       ntile, long_blocks, long_row);
  }
  const hipError_t e = hipGetLastError();
  timing_after_main(s);
  return e;
}

hipError_t launch_naive_smem(const Problem& p, hipStream_t s) {
  if (p.M == 0 || p.N == 0) return hipSuccess;
  const int cols_per_block = p.N >= 256 ? 256 : ((p.N + 63) / 64) * 64;
  const int ntile = div_up_host(p.N, cols_per_block);
  const long long blocks = (long long)p.M * ntile;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  timing_before_main(s);
  hipLaunchKernelGGL(naive_smem_kernel, dim3((unsigned)blocks), dim3(cols_per_block), 0, s, p, ntile,
                     cols_per_block);
  const hipError_t e = hipGetLastError();
  timing_after_main(s);
  return e;
}

}  // namespace csrspmm_hip
