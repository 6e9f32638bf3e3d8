// NF4 quantizer with double-quantized absmax, on the GPU.
//
// Upstream of the hot path: it produces the packed weights the dequant and GEMM kernels
// consume, with the algorithm bitsandbytes' quantize_4bit(quant_type="nf4",
// compress_statistics=True) follows as the reference calls it (solution/test_nf4.py:33,
// tools/bench_nf4.py:30-35): per-64 absmax, nearest NF4 value by midpoints, high nibble first;
// offset = mean(absmax); (absmax - offset) quantized per 256 blocks with a signed 8-bit code book
// to the nearest entry.  Every step is deterministic (fixed reduction order), so the result is
// reproducible run to run.
#include "common.h"
#include "mxs_nf4.h"

namespace mxs {

// The code of x in [-1, 1] is the number of midpoints below it.  No two midpoints are closer than
// 1/16 (the smallest gap is 0.08), so the sixteenth of the interval x falls in holds at most one:
// a table of (codes below the bin, its midpoint or +inf) gives the code with one compare, where
// the chain over 15 midpoints took 30 instructions a value and bounded the kernel (8960 x 1536:
// 19.6 us against 10.8; its 34 MB take 6.7 at the copy rate).  x * 16 is exact and the sum
// with 16 rounds only near a bin's edge, from which every midpoint is at least 0.0016 away, so a
// value rounded into the next bin still gets its own code.  NaN (an infinite weight times the
// zero reciprocal of its block's maximum) clamps to bin 0 and compares false: code 0, as counting
// gives.
constexpr int kBins = 33;

struct CodeBin {
  float mid;
  uint32_t below;
};

// Lane group of 8 lanes = one 64-value block; lane handles 8 consecutive values.
__global__ __launch_bounds__(256) void k_quant_blocks(const uint16_t* __restrict__ w,
                                                     int64_t n_blocks, uint8_t* __restrict__ packed,
                                                     float* __restrict__ absmax) {
  __shared__ CodeBin s_bin[kBins];
  const int64_t chunk = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t blk = chunk >> 3;
  const bool live = blk < n_blocks;
  u32x4 raw = {0u, 0u, 0u, 0u};
  if (live) raw = reinterpret_cast<const u32x4*>(w)[chunk];
  if (threadIdx.x < kBins) {
    const float lo = (float)threadIdx.x * 0.0625f - 1.0f, hi = lo + 0.0625f;
    CodeBin b = {__builtin_inff(), 0u};
    for (int i = 0; i < 15; i++) {
      const float mid = (float)(((double)kNF4[i] + (double)kNF4[i + 1]) * 0.5);
      if (mid < lo) b.below = i + 1;
      else if (mid < hi) b.mid = mid;
    }
    s_bin[threadIdx.x] = b;
  }
  __syncthreads();
  float v[8];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    v[2 * j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(raw[j] & 0xffffu));
    v[2 * j + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(raw[j] >> 16));
  }
  float m = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; j++) m = fmaxf(m, fabsf(v[j]));
  // max over the 8 lanes of the block (lane groups are aligned to 8 within the wave)
#pragma unroll
  for (int d = 1; d < 8; d <<= 1) m = fmaxf(m, __shfl_xor(m, d, 8));
  const float inv = m > 0.0f ? 1.0f / m : 0.0f;
  uint32_t word = 0;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float x = v[j] * inv;
    const int bin = (int)fminf(fmaxf(x * 16.0f + 16.0f, 0.0f), (float)(kBins - 1));
    const CodeBin b = s_bin[bin];
    const uint32_t q = b.below + (x > b.mid ? 1u : 0u);
    // value j -> byte j/2, high nibble for even j
    word |= q << (8 * (j >> 1) + ((j & 1) ? 0 : 4));
  }
  if (live) {
    reinterpret_cast<uint32_t*>(packed)[chunk] = word;
    if ((chunk & 7) == 0) absmax[blk] = m;
  }
}

// Partial sums of absmax in double: workgroup g sums blocks [g*4096, g*4096+4096) with a fixed
// tree (lane-strided, then pairwise in LDS).
constexpr int kSumSpan = 4096;
__global__ __launch_bounds__(256) void k_absmax_partial(const float* __restrict__ absmax,
                                                       int64_t n_blocks,
                                                       double* __restrict__ partial) {
  __shared__ double s[256];
  const int64_t base = (int64_t)blockIdx.x * kSumSpan;
  float v[kSumSpan / 256];  // every load before the first add
#pragma unroll
  for (int i = 0; i < kSumSpan / 256; i++) {
    const int64_t b = base + i * 256 + threadIdx.x;
    v[i] = b < n_blocks ? absmax[b] : 0.0f;  // absmax >= 0: adding +0 changes nothing
  }
  double acc = 0.0;
#pragma unroll
  for (int i = 0; i < kSumSpan / 256; i++) acc += (double)v[i];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int d = 128; d > 32; d >>= 1) {
    if ((int)threadIdx.x < d) s[threadIdx.x] += s[threadIdx.x + d];
    __syncthreads();
  }
  if (threadIdx.x >= 64) return;
  acc = s[threadIdx.x];  // the tree's last six levels within one wave
  for (int d = 32; d > 0; d >>= 1) acc += __shfl_down(acc, d, 64);
  if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

// The mean from the partials, added in order: for more of them than the workgroups below take.
__global__ void k_absmax_mean(const double* __restrict__ partial, int n_partial, int64_t n_blocks,
                              float* __restrict__ offset) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double acc = 0.0;
  for (int i = 0; i < n_partial; i++) acc += partial[i];
  offset[0] = (float)(acc / (double)n_blocks);
}

// Partials a workgroup of the next kernel adds itself (in order, from LDS), so that a weight of up
// to 2^26 values needs no launch for its mean (3.6 us of a 30 us quantization of 1536 x 8960).
constexpr int kMeanHere = 256;

// One workgroup per 256-block group: absmax2 = max |absmax - offset|; q8 = nearest code entry
// (code ascending; ties to the lower index).  n_partial > 0: the offset is their mean, which
// workgroup 0 stores; else it is read.
__global__ __launch_bounds__(256) void k_quant_absmax(const float* __restrict__ absmax,
                                                     int64_t n_blocks,
                                                     const double* __restrict__ partial,
                                                     int n_partial,
                                                     float* __restrict__ offset,
                                                     const float* __restrict__ code,
                                                     uint8_t* __restrict__ q8,
                                                     float* __restrict__ absmax2) {
  __shared__ float s_code[256];
  __shared__ float s_max[4];
  __shared__ double s_part[kMeanHere];
  __shared__ float s_off;
  const int t = threadIdx.x;
  s_code[t] = code[t];
  const int64_t b = (int64_t)blockIdx.x * 256 + t;
  const float am = b < n_blocks ? absmax[b] : 0.0f;
  if (t < n_partial) s_part[t] = partial[t];
  __syncthreads();
  if (t == 0) {
    if (n_partial > 0) {
      double acc = 0.0;
      for (int i = 0; i < n_partial; i++) acc += s_part[i];
      s_off = (float)(acc / (double)n_blocks);
      if (blockIdx.x == 0) offset[0] = s_off;
    } else {
      s_off = offset[0];
    }
  }
  __syncthreads();
  const float off = s_off;
  const float v = b < n_blocks ? am - off : 0.0f;
  float m = fabsf(v);
  for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  if ((t & 63) == 0) s_max[t >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
  if (t == 0) absmax2[blockIdx.x] = m;
  if (b >= n_blocks) return;
  const float inv = m > 0.0f ? 1.0f / m : 0.0f;
  const float x = v * inv;
  int idx;
  if (x <= s_code[0]) {
    idx = 0;
  } else if (x >= s_code[255]) {
    idx = 255;
  } else {
    int lo = 0, hi = 255;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (s_code[mid] <= x) lo = mid; else hi = mid;
    }
    const float dlo = x - s_code[lo], dhi = s_code[hi] - x;
    idx = dhi < dlo ? hi : lo;
  }
  q8[b] = (uint8_t)idx;
}

}  // namespace mxs

using namespace mxs;

extern "C" {

int mxs_nf4_quantize_workspace_bytes(int64_t n_values) {
  const int64_t n_blocks = n_values / 64;
  const int64_t n_partial = (n_blocks + kSumSpan - 1) / kSumSpan;
  return (int)(n_partial * (int64_t)sizeof(double) + 256);
}

int mxs_nf4_quantize(const void* w_f16, int64_t n_values, const float* code, void* packed,
                     float* absmax_f32, void* absmax8, float* absmax2, float* offset,
                     void* workspace, hipStream_t stream) {
  if (n_values < 0 || (n_values % 64) != 0) return MXS_ERR_SIZE;
  if (!w_f16 || !code || !packed || !absmax_f32 || !absmax8 || !absmax2 || !offset ||
      !workspace)
    return MXS_ERR_ARG;
  if (((uintptr_t)w_f16 % 16) != 0 || ((uintptr_t)packed % 4) != 0 ||
      ((uintptr_t)workspace % 8) != 0)
    return MXS_ERR_ALIGN;
  if (n_values == 0) return MXS_OK;
  const int64_t n_blocks = n_values / 64;
  const int64_t n_chunks = n_blocks * 8;
  const int64_t n_partial = (n_blocks + kSumSpan - 1) / kSumSpan;
  const int64_t n_groups = (n_blocks + 255) / 256;
  if ((n_chunks + 255) / 256 > 0x7fffffff) return MXS_ERR_SIZE;
  double* partial = static_cast<double*>(workspace);
  hipLaunchKernelGGL(k_quant_blocks, dim3((unsigned)((n_chunks + 255) / 256)), dim3(256), 0,
                     stream, static_cast<const uint16_t*>(w_f16), n_blocks,
                     static_cast<uint8_t*>(packed), absmax_f32);
  hipLaunchKernelGGL(k_absmax_partial, dim3((unsigned)n_partial), dim3(256), 0, stream,
                     absmax_f32, n_blocks, partial);
  const bool here = n_partial <= kMeanHere;
  if (!here)
    hipLaunchKernelGGL(k_absmax_mean, dim3(1), dim3(64), 0, stream, partial, (int)n_partial,
                       n_blocks, offset);
  hipLaunchKernelGGL(k_quant_absmax, dim3((unsigned)n_groups), dim3(256), 0, stream, absmax_f32,
                     n_blocks, partial, here ? (int)n_partial : 0, offset, code,
                     static_cast<uint8_t*>(absmax8), absmax2);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? MXS_OK : (int)e;
}

}  // extern "C"
