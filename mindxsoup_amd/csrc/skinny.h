// Forward NF4 GEMMs of a few tokens (generation): at most 16 rows of x against the
// whole weight.  Included by nf4_gemm.hip (GemmArgs, AccStart::lora_row).
//
// Bound by the weight's bytes (gate_proj: 7 MB) and by latency: the tile kernels run a few tokens
// as one 128- or 256-row tile per column strip, so their 24 K-steps are a serial chain of barriers
// (27 us for gate and up, 12 us for a 1536 x 1536 projection, whatever the token count).  Here a
// workgroup owns 16 output columns and its waves split the reduction: each wave's whole share of
// the weight is one or two batches of 16-byte loads, decoded in registers straight into the
// operand of v_mfma_f32_16x16x32_f16, and the waves' sums meet once in LDS, in wave order.  One
// more wave forms bias + LoRA.
#pragma once

namespace mxs {

constexpr int kSkinnyRows = 16;    // most tokens (one row block of the multiply)
constexpr int kSkinnyWaves = 12;   // most waves splitting the reduction (and one for the LoRA term)
constexpr int kSkinnyChunk = 128;  // reduction indices per wave and load: 4 lane groups x 32 values
constexpr int kSkinnyBatch = 2;    // chunks a wave loads together

struct SkinnyGroup {
  GemmArgs p[4];
  int start[5];  // workgroups of problem i: [start[i], start[i + 1])
  int nw[4];     // waves splitting problem i's reduction (its own, so that a group keeps the bits)
  int n;
};

// The rotated output of row m, column col (column c of the workgroup): the lane 8 away in c holds
// the value 64 columns away in the head.  Every lane of the wave calls it.
__device__ __forceinline__ float skinny_rotate(const GemmArgs& a, float sum, int m, int c,
                                               int col) {
#pragma clang fp contract(off)
  const float x = (float)(_Float16)sum, other = __shfl_xor(x, 8, 64);
  if (m >= a.M) return x;
  const int b = m / a.rope_T, t = m - b * a.rope_T;
  const int64_t at = (int64_t)b * a.rope_cs_b + (int64_t)t * a.rope_cs_t + (col & 127);
  const float s = a.rope_sin[at];
  return x * a.rope_cos[at] + other * (c & 8 ? s : -s);
}

// Lane l holds column l % 16 of the workgroup's 16 and row l % 16 of x, lane group g = l / 16 the
// 32 reduction indices 32 g of its chunk; multiply j takes 8 j .. 8 j + 7 of them on both sides.
// The workgroup's columns are 16 neighbours, or, where the output is rotated, 8 of a head's first
// half and the 8 they pair with 64 further on, so that a rotation's two values meet in one wave:
// rope_rotate's arithmetic on the fp16 values, a group then having the bits of the same group
// followed by the rotation launch (q, k and v of 1 token: 5.3 us rotated, 4.7 not; rotated on the
// tile kernels 12.7).  ROPE: some problem of the launch is rotated.
template <bool ROPE>
__global__ __launch_bounds__(64 * (kSkinnyWaves + 1)) void k_nf4_skinny(SkinnyGroup grp) {
  __shared__ float s_nf4[16];
  __shared__ float s_code[256];
  __shared__ float red[kSkinnyWaves + 1][16][17];
  int pi = 0;
  while (pi + 1 < grp.n && (int)blockIdx.x >= grp.start[pi + 1]) pi++;
  const GemmArgs& a = grp.p[pi];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nw = grp.nw[pi];
  const int lw = ((int)blockDim.x >> 6) - 1;  // the wave of bias and LoRA
  const int c16 = lane & 15, g = lane >> 4;
  const int n0 = ((int)blockIdx.x - grp.start[pi]) * 16;
  const bool rot = ROPE && a.rope_cos;
  // output column of the workgroup's column c
  auto column = [&](int c) {
    return rot ? (n0 & ~127) + ((n0 & 127) >> 1) + (c & 7) + ((c & 8) << 3) : n0 + c;
  };
  const int n = min(column(c16), a.Nc - 1);
  const int chunks = (a.Kr + kSkinnyChunk - 1) / kSkinnyChunk;
  const float off = a.offset[0];
  const int64_t row = (int64_t)n * a.Kr;
  const _Float16* xrow = a.A + (int64_t)min(c16, a.M - 1) * a.lda;

  u32x4 w[kSkinnyBatch];
  uint32_t q8[kSkinnyBatch];
  float a2[kSkinnyBatch];
  half8_t x[kSkinnyBatch][4];
  // one batch's loads: chunks c, c + nw, .. ; lanes past the reduction's end read its start
  auto issue = [&](int c) {
#pragma unroll
    for (int u = 0; u < kSkinnyBatch; u++) {
      const int cu = c + u * nw;
      if (cu >= chunks) break;
      const int k0 = cu * kSkinnyChunk + 32 * g, k = k0 < a.Kr ? k0 : 0;
      w[u] = *reinterpret_cast<const u32x4*>(a.packed + (row + k) / 2);
      const int64_t blk = (row + k) >> 6;
      q8[u] = a.absmax8[blk];
      a2[u] = a.absmax2[blk >> 8];
#pragma unroll
      for (int j = 0; j < 4; j++)
        x[u][j] = *reinterpret_cast<const half8_t*>(xrow + k + 8 * j);
    }
  };
  float4_t acc = {0.f, 0.f, 0.f, 0.f};
  if (wave < nw) issue(wave);  // in flight over the tables' loads and the barrier
  for (int i = t; i < 256; i += (int)blockDim.x) s_code[i] = a.code[i];
  if (t < 16) s_nf4[t] = kNF4[t];
  __syncthreads();
  if (wave < nw) {
    for (int c = wave; c < chunks; c += kSkinnyBatch * nw) {
      if (c != wave) issue(c);
#pragma unroll
      for (int u = 0; u < kSkinnyBatch; u++) {
        const int cu = c + u * nw;
        if (cu >= chunks) break;
        const bool live = cu * kSkinnyChunk + 32 * g < a.Kr;
        const float s = nested_scale(s_code[q8[u]], a2[u], off);
#pragma unroll
        for (int j = 0; j < 4; j++) {
          half8_t wf = __builtin_bit_cast(half8_t, decode8(w[u][j], s, s_nf4));
          if (!live) wf = (half8_t){};
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(live ? x[u][j] : (half8_t){}, wf, acc, 0, 0,
                                                       0);
        }
      }
    }
  } else if (wave == lw) {
    // bias + LoRA, and the transposed LoRA operand from the first columns' workgroup
    if (a.bias) {
      const float bv = (float)a.bias[n];
      acc = (float4_t){bv, bv, bv, bv};
    }
    if (a.lora_h || a.lora_hp) {
      for (int r0 = 0; r0 < a.r; r0 += 32) {
        const int rank = r0 + 8 * g;
        const bool live = rank < a.r;
        const half8_t wf = live
            ? *reinterpret_cast<const half8_t*>(a.lora_w + (int64_t)n * a.r + rank) : (half8_t){};
        const half8_t hf =
            live ? AccStart<1, 1, false>::lora_row(a, c16, rank & ~15, g & 1) : (half8_t){};
        if (live && n0 == 0 && a.lora_hp && a.lora_ht && c16 < a.ldt) {
#pragma unroll
          for (int e = 0; e < 8; e++) a.lora_ht[(int64_t)(rank + e) * a.ldt + c16] = hf[e];
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(hf, wf, acc, 0, 0, 0);
      }
      if (n0 == 0 && a.lora_hp && a.lora_ht) {  // a row length past the 16 rows: zeros
        const int pad = a.ldt - kSkinnyRows;
        for (int i = lane; i < a.r * pad; i += 64)
          a.lora_ht[(int64_t)(i / pad) * a.ldt + kSkinnyRows + i % pad] = (_Float16)0.0f;
      }
    }
  }
  // acc[v] = C[4 g + v][n0 + c16]; waves past nw have none
  if (wave < nw || wave == lw)
#pragma unroll
    for (int v = 0; v < 4; v++) red[wave][4 * g + v][c16] = acc[v];
  __syncthreads();
  for (int i = t; i < 256; i += (int)blockDim.x) {
    const int m = i >> 4, c = i & 15, col = column(c);
    float sum = red[lw][m][c];  // bias and LoRA first, as the tile kernels' accumulators start
    for (int v = 0; v < nw; v++) sum += red[v][m][c];
    if constexpr (ROPE) {
      if (rot) sum = skinny_rotate(a, sum, m, c, col);
    }
    if (m >= a.M || col >= a.Nc) continue;
    a.C[(int64_t)m * a.ldc + col] = (_Float16)sum;
  }
}

// Waves splitting the reduction, at 1 token (16 are within 2 us of it): with at most one workgroup
// per CU the reduction's latency decides (1536 x 1536: 12 waves 4.2 us, 6 waves 4.8, 3 waves 5.6;
// 1536 x 8960 10.2, 12.8, 19.7; 4096 x 4096 7.0, 8.3, 11.3), with more of them how many share a CU
// (8960 x 1536: 3 waves 7.5 us, 6 waves 8.1, 12 waves 9.4; 14336 x 4096 18.2, 20.0, 22.3).
static int skinny_waves(int Nc, int Kr) {
  const int chunks = (Kr + kSkinnyChunk - 1) / kSkinnyChunk, wgs = (Nc + 15) / 16;
  const int most = wgs <= 256 ? kSkinnyWaves : 3;
  return chunks < most ? chunks : most;
}

// n problems over one x, each with its own output, in one launch.
static int launch_skinny(const GemmArgs* probs, int n, hipStream_t stream) {
  if (n < 1 || n > 4) return MXS_ERR_ARG;
  SkinnyGroup g{};
  g.n = n;
  int64_t total = 0;
  int nw = 1;
  bool rope = false;
  for (int i = 0; i < n; i++) {
    g.p[i] = probs[i];
    rope = rope || probs[i].rope_cos;
    g.start[i] = (int)total;
    total += (probs[i].Nc + 15) / 16;
    g.nw[i] = skinny_waves(probs[i].Nc, probs[i].Kr);
    nw = g.nw[i] > nw ? g.nw[i] : nw;
  }
  if (total > 0x7fffffff) return MXS_ERR_SIZE;
  g.start[n] = (int)total;
  const dim3 grid((unsigned)total), block(64 * (nw + 1));
  if (rope) hipLaunchKernelGGL(k_nf4_skinny<true>, grid, block, 0, stream, g);
  else hipLaunchKernelGGL(k_nf4_skinny<false>, grid, block, 0, stream, g);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? MXS_OK : (int)e;
}

}  // namespace mxs
