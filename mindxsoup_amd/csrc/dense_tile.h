// The dense route of the NF4 GEMMs, for token counts where decoding once pays: the weight is
// decoded to fp16 once per call into the caller's workspace (k_w16_decode; the input gradient's
// weight transposed on the way, so that both directions read B [Nc, Kr] with the reduction
// contiguous), then a plain fp16 GEMM whose eight waves all multiply.  Included by nf4_gemm.hip
// (GemmArgs, AccStart, LoraStage, MaskStage, StagedStore, epilogue_staged).
//
// The fused kernels decode every weight tile once per 256-row band of C: at 8192 tokens 32
// times.  Their K-step is bound by the producers' chain and its barrier with four consumer
// waves (one per SIMD); here the producers and their tables are gone, B arrives by direct
// global -> LDS copies like A, and two multiplying waves per SIMD cover each other's LDS reads.
// The products, their order and the accumulator start are the fused kernels' (the same decoded
// fp16 values, v_mfma_f32_32x32x16_f16 over the same K sequence), so at one split count the
// results have the same bits.
#pragma once

namespace mxs {

// ---- weight decode --------------------------------------------------------------------------

struct W16Problem {
  const uint32_t* packed;
  const uint8_t* absmax8;
  const float* code;
  const float* absmax2;
  const float* offset;
  _Float16* out;  // W [N, K] or, transposed, W^T [K, N]
  int N, K;
};

struct W16Group {
  W16Problem p[4];
  int start[5];  // workgroups of problem i: [start[i], start[i + 1])
  int n;
};

constexpr int kW16Chunks = 1024;         // forward: 8-value chunks per workgroup
constexpr int kW16TR = 64, kW16TC = 128;  // transposed: W rows x columns per workgroup

// Forward: 256 lanes x 4 chunks of one dword (8 values, 16 output bytes), as k_dequant_wide, but
// with cached stores: the GEMM behind it reads the result back at once.
__device__ __forceinline__ void w16_decode_rows(const W16Problem& p, int wg, float* s_nf4,
                                                float* s_scale) {
  const int t = threadIdx.x;
  const int64_t c0 = (int64_t)wg * kW16Chunks;
  const int64_t n_chunks = (int64_t)p.N * p.K / 8;
  uint32_t w[4];
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int64_t c = c0 + u * 256 + t;
    w[u] = c < n_chunks ? __builtin_nontemporal_load(p.packed + c) : 0u;
  }
  if (t < 16) s_nf4[t] = kNF4[t];
  if (t < kW16Chunks / 8) {
    const int64_t blk = (c0 >> 3) + t;
    s_scale[t] = blk * 8 < n_chunks
        ? nested_scale(p.code[p.absmax8[blk]], p.absmax2[blk >> 8], p.offset[0]) : 0.0f;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int local = u * 256 + t;
    if (c0 + local >= n_chunks) break;
    reinterpret_cast<u32x4*>(p.out)[c0 + local] = decode8(w[u], s_scale[local >> 3], s_nf4);
  }
}

// Transposed: a 64 x 128 tile of W through LDS.  A lane decodes 16 consecutive values of two
// neighbouring rows and writes them as (row n, row n + 1) pairs, one dword per column; the
// 16-byte groups of a column's 64 rows are XOR-ed with bits 4..6 of the column, so that the
// eight lanes sharing a row pair write different banks.  Each column's 64 values then leave as
// one 128-byte line.
__device__ __forceinline__ void w16_decode_cols(const W16Problem& p, int wg, float* s_nf4,
                                                uint32_t* s_tile) {
  const int t = threadIdx.x;
  const int gx = (p.K + kW16TC - 1) / kW16TC;
  const int k0 = (wg % gx) * kW16TC, n0 = (wg / gx) * kW16TR;
  const int pair = t >> 3, part = t & 7;  // rows n0 + 2 pair, +1; columns k0 + 16 part .. +15
  const int k = k0 + 16 * part;
  const bool live = k < p.K;
  u32x2 w[2] = {};
  float s[2] = {};
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int64_t v0 = (int64_t)(n0 + 2 * pair + j) * p.K + (live ? k : 0);
    w[j] = *reinterpret_cast<const u32x2*>(p.packed + v0 / 8);
    const int64_t blk = v0 >> 6;
    s[j] = nested_scale(p.code[p.absmax8[blk]], p.absmax2[blk >> 8], p.offset[0]);
  }
  if (t < 16) s_nf4[t] = kNF4[t];
  __syncthreads();
  if (live) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const u32x4 a = decode8(w[0][h], s[0], s_nf4), b = decode8(w[1][h], s[1], s_nf4);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int c = 16 * part + 8 * h + 2 * e;
        const int col = pair ^ (part << 2);
        s_tile[c * 32 + col] = (a[e] & 0xffffu) | (b[e] << 16);
        s_tile[(c + 1) * 32 + col] = (a[e] >> 16) | (b[e] & 0xffff0000u);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kW16TC / 32; u++) {
    const int c = u * 32 + (t >> 3), g = t & 7;
    if (k0 + c >= p.K) break;
    const u32x4 v = *reinterpret_cast<const u32x4*>(s_tile + c * 32 + 4 * (g ^ (c >> 4)));
    *reinterpret_cast<u32x4*>(p.out + (int64_t)(k0 + c) * p.N + n0 + 8 * g) = v;
  }
}

template <bool T>
__global__ __launch_bounds__(256) void k_w16_decode(W16Group g) {
  __shared__ float s_nf4[16];
  __shared__ uint32_t s_buf[T ? kW16TC * kW16TR / 2 : kW16Chunks / 8];
  const int bid = (int)blockIdx.x;
  int i = 0;
  while (i + 1 < g.n && bid >= g.start[i + 1]) i++;
  if constexpr (T) w16_decode_cols(g.p[i], bid - g.start[i], s_nf4, s_buf);
  else w16_decode_rows(g.p[i], bid - g.start[i], s_nf4, reinterpret_cast<float*>(s_buf));
}

// ---- GEMM -------------------------------------------------------------------------------------

// Direct global -> LDS copies of a [ROWS][64] fp16 tile by the eight waves: wave w copies the
// 8-row groups w, w + 8, ... (64 lanes x 16 B each, consecutive in LDS), each lane fetching the
// segment that lds_off's swizzle keeps at its slot.  Rows past the operand's end repeat its last
// one (their products are not stored).  Inline asm as in ACopy; completion is awaited by hand.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <int ROWS>
struct TileCopy {
  static constexpr int N = ROWS / 64;  // copies per wave per K-step
  uint32_t off[N];
  const char* base;  // row row0 of the operand (uniform)
  uint32_t lds;      // LDS byte address of this wave's first row group in stage 0 (uniform)

  __device__ __forceinline__ void init(const _Float16* src, int64_t ld, int row0, int rows,
                                       const _Float16* tile, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int row = wave * 8 + 64 * i + (lane >> 3);
      const int seg = ((lane & 7) ^ (row >> 1)) & 7;
      off[i] = ((uint32_t)(min(row0 + row, rows - 1) - row0) * (uint32_t)ld + seg * 8) * 2;
    }
    base = reinterpret_cast<const char*>(src + (int64_t)row0 * ld);
    lds = __builtin_amdgcn_readfirstlane(
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>(tile + wave * 8 * kBK)));
  }

  // copy i of K-step k into the stage at byte offset `stage`
  __device__ __forceinline__ void copy(uint32_t stage, int k, int i) const {
    const char* src = base + (size_t)k * kBK * sizeof(_Float16);
    const uint32_t dst = lds + stage + i * 64 * kBK * sizeof(_Float16);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(dst), "v"(off[i]), "s"(src)
                 : "memory", "m0");
  }
};
#pragma clang diagnostic pop

constexpr int kDenseBM = 256;

constexpr int kDenseNT = 512;  // threads: eight waves, 4 x 2 over the tile

// Dwords of one wave's staging area in the epilogue: 320-column tiles never split (fp16 rows).
template <int BN>
constexpr int dense_area() {
  using SS = StagedStore<2, BN / 64>;
  return 32 * (BN > 256 ? SS::S16 : SS::S32);
}

// Dynamic LDS of the dense kernel: two stages of A and B, or the epilogue's staging areas.
template <int BN>
constexpr int dense_lds_bytes() {
  constexpr int stages = 2 * (kDenseBM + BN) * kBK * 2, areas = 8 * 4 * dense_area<BN>();
  return stages > areas ? stages : areas;
}

// SwiGLU adjoint of down_proj's input gradient (GemmArgs.glu == 2): the tile is d(hidden);
// gate <- d(gate), up <- d(up).  Staged through the wave's LDS area like epilogue_staged; the
// gate / up chunks of half a slice are loaded together.
template <int TM, int TN>
__device__ __forceinline__ void epilogue_glu_bwd(const GemmArgs& a, float16_t (&acc)[TM][TN],
                                                 int mb, int nb, int lane, uint32_t* area) {
  using SS = StagedStore<TM, TN>;
  constexpr int CPR = SS::WN / 8, NC = CPR / 2, G = (NC + 1) / 2;
  const int lrow = lane & 31, lseg = lane >> 5;
#pragma unroll
  for (int i = 0; i < TM; i++) {
    const int row0 = mb + i * 32;
    if (row0 >= a.M) break;
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        u32x2 v;
        v[0] = pack_f16x2(acc[i][j][4 * g], acc[i][j][4 * g + 1]);
        v[1] = pack_f16x2(acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
        *reinterpret_cast<u32x2*>(area + lrow * SS::S16 + 16 * j + 4 * g + 2 * lseg) = v;
      }
#pragma unroll
    for (int q0 = 0; q0 < NC; q0 += G) {
      u32x4 gv[G], uv[G];
#pragma unroll
      for (int u = 0; u < G; u++) {
        const int c = (q0 + u) * 64 + lane, m = row0 + c / CPR, n = nb + 8 * (c % CPR);
        const bool ok = q0 + u < NC && m < a.M && n < a.Nc;  // Nc % 8 == 0: whole chunks
        const int64_t o = (int64_t)m * a.ldc + n;
        gv[u] = ok ? *reinterpret_cast<const u32x4*>(a.glu_g + o) : (u32x4){};
        uv[u] = ok ? *reinterpret_cast<const u32x4*>(a.glu_u + o) : (u32x4){};
      }
#pragma unroll
      for (int u = 0; u < G; u++) {
        const int c = (q0 + u) * 64 + lane, r = c / CPR, m = row0 + r, n = nb + 8 * (c % CPR);
        if (q0 + u >= NC || m >= a.M || n >= a.Nc) continue;
        const half8_t h = __builtin_bit_cast(
            half8_t, *reinterpret_cast<const u32x4*>(area + r * SS::S16 + 4 * (c % CPR)));
        const half8_t g8 = __builtin_bit_cast(half8_t, gv[u]);
        const half8_t u8 = __builtin_bit_cast(half8_t, uv[u]);
        half8_t dg, du;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          _Float16 x, y;
          swiglu_bwd((float)h[e], (float)g8[e], (float)u8[e], x, y);
          dg[e] = x;
          du[e] = y;
        }
        const int64_t o = (int64_t)m * a.ldc + n;
        *reinterpret_cast<half8_t*>(a.glu_g + o) = dg;
        *reinterpret_cast<half8_t*>(a.glu_u + o) = du;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // reads done before the next slice
  }
}

// RoPE on a wave's 128 columns (one head, in order: blocks j and j + 2 hold head columns d and
// d + 64 in the same lane and element), before the fp16 store: rope_rotate's arithmetic.
__device__ __forceinline__ void rope_rotate_head(const GemmArgs& a, float16_t (&acc)[4], int m,
                                                 int lseg) {
#pragma clang fp contract(off)
  if (m >= a.M) return;
  const int b = m / a.rope_T, t = m - b * a.rope_T;
  const int64_t cr = (int64_t)b * a.rope_cs_b + (int64_t)t * a.rope_cs_t;
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int d = 32 * j + 8 * g + 4 * lseg;
      const float4_t c1 = *reinterpret_cast<const float4_t*>(a.rope_cos + cr + d);
      const float4_t c2 = *reinterpret_cast<const float4_t*>(a.rope_cos + cr + d + 64);
      const float4_t s1 = *reinterpret_cast<const float4_t*>(a.rope_sin + cr + d);
      const float4_t s2 = *reinterpret_cast<const float4_t*>(a.rope_sin + cr + d + 64);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float x1 = (float)(_Float16)acc[j][4 * g + e];
        const float x2 = (float)(_Float16)acc[j + 2][4 * g + e];
        acc[j][4 * g + e] = x1 * c1[e] + x2 * -s1[e];
        acc[j + 2][4 * g + e] = x2 * c2[e] + x1 * s2[e];
      }
    }
}

// One 256 x BN output tile, eight waves of 64 x BN/2 (4 x 2, two per SIMD).  Two LDS stages of one
// 64-deep K-step (A and B) each.  A K-step's last sub-step is multiplied behind the barrier that
// ends it, over the next step's first fragment reads; the stage that barrier frees takes the
// copies of the K-step after next, spread over the MFMAs of that sub-step and the next two, so
// that the last of them has a whole sub-step to land (with the last third of the copies issued in
// the sub-step before the wait, down_proj forward at 8192 tokens took 233 us instead of 220).  The
// order of MFMAs, fragment reads and copies is pinned.
// What bounds it: with every CU multiplying, the clock the part sustains (a K-step of 256 columns
// takes 1.45 us against 1.2 with a fifth of the CUs busy), and per tile 13 us at its ends that
// nothing overlaps: the operands and LoRA term before the first multiply and the stores, which
// every CU issues at the same time (7.5 us of the 58 of a 1536-long, 320-wide tile).  Measured
// and not kept: four waves of 128 x BN/2 (two thirds of the LDS reads: the same K-steps, longer
// ends: 55 against 49 us at 8192 x 1536 x 1536); two workgroups per CU on 128-row tiles with
// 32-deep K-steps, so that one's ends hide behind the other's multiplies (1.5 times the copies:
// 280 against 220 us).
// NSUM > 1: up to NSUM problems with one output, their reductions one after the other into the
// same accumulators (GemmArgs as[0..nsum)).  Every problem has keep bits or none does: with the
// test per problem the compiler spilled inside the K loop (gate and up's dX at 8192 tokens: 1099 us
// instead of 506), so the host keeps mixed masks on the fused kernel.
template <int BN, bool BWD, bool GLU, int NSUM, bool ROPE>
__device__ __forceinline__ void dense_tile(const GemmArgs* as, int nsum, int bx, int by) {
  constexpr int BM = kDenseBM, TM = 2, TN = BN / 64, NT = kDenseNT;
  constexpr int LDS_A = BM * kBK, LDS_B = BN * kBK;
  constexpr uint32_t STAGE = (LDS_A + LDS_B) * sizeof(_Float16);
  static_assert(!ROPE || TN == 4, "a wave holds one head");
  extern __shared__ __attribute__((aligned(16))) _Float16 smem[];
  const GemmArgs& a = as[0];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int m0 = by * BM, n0 = bx * BN;
  const int wm0 = (wave >> 1) * 64, wn0 = (wave & 1) * (BN / 2);
  const int lrow = lane & 31, lseg = lane >> 5;
  int n_steps = 0;
  if constexpr (NSUM == 1) {
    n_steps = a.Kr / kBK;
  } else {
    for (int q = 0; q < nsum; q++) n_steps += as[q].Kr / kBK;
  }
  const int kt0 = ((int)blockIdx.z - a.zf) * a.steps_per_split;
  const int kt1 = min(n_steps, kt0 + a.steps_per_split);

  // the copies' operands: problem q's from K-step `first` on
  TileCopy<BM> ca;
  TileCopy<BN> cb;
  int q = 0, first = 0, end = 0;
  auto enter = [&](int k) {  // the problem of K-step k (k never decreases)
    while (q + 1 < nsum && k >= end) {
      q++;
      first = end;
      end += as[q].Kr / kBK;
    }
    ca.init(as[q].A, as[q].lda, m0, a.M, smem, wave, lane);
    cb.init(as[q].w16, as[q].Kr, n0, a.Nc, smem + LDS_A, wave, lane);
  };
  end = a.Kr / kBK;
  enter(kt0);
  // copy c (A's, then B's) of K-step k into stage k - kt0
  constexpr int NCP = TileCopy<BM>::N + TileCopy<BN>::N;
  auto copy = [&](int k, int c) {
    const uint32_t st = ((k - kt0) & 1) * STAGE;
    if (c < TileCopy<BM>::N) ca.copy(st, k - first, c);
    else cb.copy(st, k - first, c - TileCopy<BM>::N);
  };
  if (kt0 < kt1) {
#pragma unroll
    for (int c = 0; c < NCP; c++) copy(kt0, c);
  }

  // accumulator start: bias and the LoRA term (first split), its operands staged in stage 1
  const bool lora = (int)blockIdx.z == a.zf && (a.lora_hp || a.lora_h);
  const bool lora16 = lora && a.r == 16;
  const bool kmask = BWD && lora && a.mask;
  using MS = MaskStage<BM, BN, NT>;
  constexpr int LSH = (BM + BN) * 16;
  static_assert(LSH * 2 + BM * MS::KST <= (int)STAGE, "staged operands fit a stage");
  _Float16* Ls = smem + LDS_A + LDS_B;
  uint8_t* Ks = reinterpret_cast<uint8_t*>(Ls + LSH);
  float16_t acc[TM][TN];
  AccStart<TM, TN, BWD> start;
  auto begin = [&](const GemmArgs& p, float16_t (&c)[TM][TN]) {
    if (lora16 || kmask) {
      LoraStage<BM, BN, NT> lst;
      MS mst;
      if (lora16) lst.issue(p, t, m0, n0);
      if (kmask) mst.issue(p, t, m0, n0);
      if (lora16) lst.commit(p, Ls, t);
      if (kmask) mst.commit(Ks, t);
      lds_barrier();
    }
    if (lora16)
      start.finish_staged(p, c, m0 + wm0, n0 + wn0, lrow, lseg, wm0, wn0, Ls, BM,
                          kmask ? Ks : nullptr, MS::KST);
    else
      start.finish(p, c, m0 + wm0, n0 + wn0, lrow, lseg, wm0, wn0, nullptr, 0,
                   kmask ? Ks : nullptr, MS::KST);
    if (lora16 || kmask) lds_barrier();  // read before stage 1 is written again
  };
  start.load(a, n0 + wn0, lseg);
  begin(a, acc);
  if constexpr (NSUM > 1) {
    if (lora) {
      for (int p = 1; p < nsum; p++) {
        float16_t part[TM][TN];
        begin(as[p], part);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++) acc[i][j] += part[i][j];
      }
    }
  }

  if (kt0 < kt1) {
    wait_vmem_all();
    lds_barrier();  // K-step kt0 ready
    half8_t fa[2][TM], fb[2][TN];
    const int xs = (lrow >> 1) & 7;
    int aoff[4], boff[4];  // halfs: the lane's A / B fragment of sub-step kk, block 0
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
      const int seg = (((2 * kk + lseg) ^ xs) & 7) << 3;
      aoff[kk] = (wm0 + lrow) * kBK + seg;
      boff[kk] = LDS_A + (wn0 + lrow) * kBK + seg;
    }
    // fragment e of sub-step kk, in the order its MFMAs need them: A block 0, B's, A 1..
    constexpr int NRD = TM + TN, NMF = TM * TN;
    auto read = [&](int set, const _Float16* s, int kk, int e) {
      if (e == 0 || e > TN) {
        const int i = e == 0 ? 0 : e - TN;
        fa[set][i] = *reinterpret_cast<const half8_t*>(s + aoff[kk] + i * 32 * kBK);
      } else {
        fb[set][e - 1] = *reinterpret_cast<const half8_t*>(s + boff[kk] + (e - 1) * 32 * kBK);
      }
    };
    // One sub-step: multiply set `set`; read sub-step kk of stage `s` into the other set (s
    // null: none); copies part * NCP / 3 .. of K-step ck (part < 0: none).
    auto sub = [&](int set, const _Float16* s, int kk, int ck, int part) {
      const int c0 = part < 0 ? 0 : part * NCP / 3, c1 = part < 0 ? 0 : (part + 1) * NCP / 3;
      int c = c0;
#pragma unroll
      for (int e = 0; e < NMF; e++) {
        const int i = e / TN, j = e % TN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[set][j], fa[set][i], acc[i][j], 0,
                                                           0, 0);
        if (s && e < NRD) read(set ^ 1, s, kk, e);
        if (c < c1 && (e + 1) * (c1 - c0) >= (c - c0 + 1) * NMF) {
          copy(ck, c);
          c++;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto stage = [&](int k) { return smem + ((k - kt0) & 1) * (LDS_A + LDS_B); };
#pragma unroll
    for (int e = 0; e < NRD; e++) read(0, smem, 0, e);
    if (kt0 + 1 < kt1) {
      if constexpr (NSUM > 1) {
        if (kt0 + 1 >= end) enter(kt0 + 1);
      }
#pragma unroll
      for (int c = 0; c < NCP / 3; c++) copy(kt0 + 1, c);
    }
    int kt = kt0;
    for (; kt + 2 < kt1; kt++) {
      sub(0, stage(kt), 1, kt + 1, 1);
      sub(1, stage(kt), 2, kt + 1, 2);
      sub(0, stage(kt), 3, 0, -1);
      wait_vmem_all();  // K-step kt + 1
      lds_barrier();    // (its lgkmcnt(0) covers sub-step 3's fragments)
      if constexpr (NSUM > 1) {
        if (kt + 2 >= end) enter(kt + 2);
      }
      sub(1, stage(kt + 1), 0, kt + 2, 0);
    }
    if (kt + 1 < kt1) {
      sub(0, stage(kt), 1, kt + 1, 1);
      sub(1, stage(kt), 2, kt + 1, 2);
      sub(0, stage(kt), 3, 0, -1);
      wait_vmem_all();
      lds_barrier();
      sub(1, stage(kt + 1), 0, 0, -1);
      kt++;
    }
    sub(0, stage(kt), 1, 0, -1);
    sub(1, stage(kt), 2, 0, -1);
    sub(0, stage(kt), 3, 0, -1);
    sub(1, nullptr, 0, 0, -1);
  }
  lds_barrier();  // every wave has read its last fragments: the stages hold the staged stores
  const bool split = gridDim.z > 1;
  float* area = reinterpret_cast<float*>(smem) + wave * dense_area<BN>();
  const int mb = m0 + wm0, nb = n0 + wn0;
  if constexpr (GLU) {
    if (!split) {
      epilogue_glu_bwd<TM, TN>(a, acc, mb, nb, lane, reinterpret_cast<uint32_t*>(area));
      return;
    }
  }
  if constexpr (ROPE) {
    if (a.rope_cos) {
#pragma unroll
      for (int i = 0; i < TM; i++) rope_rotate_head(a, acc[i], mb + i * 32 + lrow, lseg);
    }
  }
  epilogue_staged<TM, TN>(a, acc, mb, nb, lane, area);
}

// Up to four problems over the same rows, each with its own output (SUM = false), or up to three
// whose outputs are summed into problem 0's.
struct DenseGroup {
  GemmArgs p[4];
  int start[5];  // tiles of problem i: [start[i], start[i + 1])
  int gy;        // row bands
  int n;
};

// Tile of workgroup `bid` of `total`: the hardware hands workgroups to the eight XCDs in turn,
// so XCD x takes a contiguous run of tiles.  Tiles run down a column of row bands first: an XCD's
// L2 then keeps the few B panels of its run, and A once, instead of every B panel (8192 x 8960
// output: 27 MB of B).  A permutation of [0, total) for every total.
__device__ __forceinline__ int xcd_tile(int bid, int total) {
  const int x = bid & 7, j = bid >> 3, per = total >> 3, rem = total & 7;
  return x * per + min(x, rem) + j;
}

template <int BN, bool BWD, bool GLU, int NSUM, bool ROPE>
__global__ __launch_bounds__(kDenseNT) void k_dense_gemm(DenseGroup g) {
  const int tile = xcd_tile((int)blockIdx.x, (int)gridDim.x);
  if constexpr (NSUM > 1) {
    dense_tile<BN, BWD, GLU, NSUM, ROPE>(g.p, g.n, tile / g.gy, tile % g.gy);
  } else {
    int i = 0;
    while (i + 1 < g.n && tile >= g.start[i + 1]) i++;
    const int local = tile - g.start[i];
    dense_tile<BN, BWD, GLU, 1, ROPE>(&g.p[i], 1, local / g.gy, local % g.gy);
  }
}

}  // namespace mxs
