// gemm_planes.hip — the weight-only int8 and fp32 GEMMs on bf16 MFMA
// (v_mfma_f32_32x32x16_bf16, fp32 accumulation) with every operand already
// in bf16 "planes", so the main loop only moves bytes and multiplies.
//
//  * Weight-only int8 (replaces MatMulPacked8, internal/tensor/pack8.go:80-126
//    and gemm4x16i8, gemm8_amd64.s:14-79): the int8 weights are stored once,
//    at pack time, as a bf16 plane of the same integers (exact: |q| <= 127
//    needs 7 significant bits). The fp32 activations are split by one light
//    pass into hi = bf16(a) and lo = bf16(a - hi), so a·q keeps ~16
//    significant bits of a; the per-channel scale multiplies the fp32
//    accumulator in the epilogue, as the reference does.
//  * fp32 (replaces MatMulPacked, pack.go:123-210 and gemm4x16,
//    gemm_amd64.s:14-64): weights split into hi/lo planes at pack time,
//    activations by the same pass; three products hi·hi + hi·lo + lo·hi (the
//    lo·lo term is ~2^-16 of the others, below the fp32 rounding of the sum
//    at these magnitudes).
//
// Main loop: BM x BN tile per workgroup, a WGM x WGN grid of waves of 32x32
// MFMA tiles, K in stages of BK bf16 per row and plane. Stages reach LDS by
// global_load_lds_dwordx4 (no register staging): lane l of a wave instruction
// writes LDS bytes [16l, 16l+16) of a 1 KiB block, so each lane loads the
// global 16-byte chunk that belongs at that slot, rows permuted for
// conflict-free fragment reads. NS stages in flight, one barrier per stage; a
// step's fragments are read from LDS under the products of the step before.
//
// What bounds it: what one CU pulls. Probes of global_load_lds on MI355X, one
// workgroup per CU and L2 hits, B/ns per CU: 16 rows of 64 bytes per
// instruction 53 with four waves and 69-72 with eight, 8 rows of 128 bytes
// 59 and 84-89. Hence 128-byte rows (BK 64) and eight waves on a CU: one
// 512-thread workgroup, two 64-KiB ones, or four multiplying waves and LW more
// that only load.
//
// The epilogue parks each 32-row band of accumulators in LDS and reads rows
// back 4 columns per lane: scale, bias, activation (or the gated pair) and a
// 4-wide vector store.
#include "gemm_common.h"

namespace rh {

// Wait until this wave's loads of at most min(MAX, later) stages are pending.
template <int LOADS, int MAX>
__device__ __forceinline__ void wait_stages(int later) {
  if constexpr (MAX == 0) {
    wait_vmcnt<0>();
  } else {
    if (later >= MAX) wait_vmcnt<MAX * LOADS>();
    else wait_stages<LOADS, MAX - 1>(later);
  }
}

// WGM x WGN waves multiply, LW more only load. BK: k elements per stage and
// row, 32 (64-byte rows, i8_slot permutation) or 64 (128-byte rows, lds_off
// permutation; half the barriers).
// QKN: the QK-norm + RoPE epilogue of the decoders' q|k|v projection (bf16
// rows to p.qk_out; see GemmPlArgs).
template <int BM, int BN, int NS, int AT, int BT, bool GLU, int BK, int WGM, int WGN, int LW = 0,
          bool QKN = false>
__global__ __launch_bounds__(64 * (WGM * WGN + LW)) void gemm_planes_kernel(GemmPlArgs p) {
  constexpr int NW = WGM * WGN;        // waves that multiply
  constexpr int NT = 64 * (NW + LW);   // threads
  constexpr int CPR = BK / 8;    // 16-byte chunks per row
  static_assert(BK == 32 || BK == 64, "stage depth");
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int kA = BM * BK * 2, kB = BN * BK * 2;  // bytes per plane
  constexpr int kStage = AT * kA + BT * kB;
  constexpr int LA = kA / (NT * 16), LB = kB / (NT * 16);  // loads per thread and plane
  constexpr int kLoads = AT * LA + BT * LB;
  constexpr int kEpiStride = WN + 4;  // floats per row of the epilogue transpose
  static_assert(LA >= 1 && LB >= 1 && TN >= 1, "tile too small for the wave grid");
  // A stage's slot is refilled right after the barrier that follows the
  // last reads of it, so two slots suffice.
  static_assert(NS >= 2, "ring");
  constexpr int kEpi = NW * 32 * kEpiStride * 4;  // epilogue bands
  constexpr int kLds = NS * kStage > kEpi ? NS * kStage : kEpi;
  static_assert(kLds <= 160 * 1024, "LDS");
  static_assert((NS - 1) * kLoads < 64, "vmcnt range");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLds];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const int tiles_n = (p.N + BN - 1) / BN;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  int rb, cb;
  tile_origin(tile, (p.M + BM - 1) / BM, tiles_n, p.tile_group, rb, cb);
  const int row0 = rb * BM;
  const int col0 = cb * BN;
  const int nk = (p.K + BK - 1) / BK;

  // Element offsets of this thread's loads (fixed across stages). Rows past
  // M read row M-1 (their outputs are never stored); weight rows are
  // zero-padded to a multiple of 256; both operands are zero past K up to a
  // multiple of 64, so a stage never masks.
  int aoff[LA], boff[LB];
#pragma unroll
  for (int j = 0; j < LA; j++) {
    const int slot = (wave * LA + j) * 64 + lane;
    const int r = slot / CPR;
    const int chunk = stage_slot_chunk<BK * 2>(r, slot % CPR);
    const int gr = row0 + r;
    aoff[j] = (gr < p.M ? gr : p.M - 1) * p.lda + chunk * 8;
  }
#pragma unroll
  for (int j = 0; j < LB; j++) {
    const int slot = (wave * LB + j) * 64 + lane;
    const int r = slot / CPR;
    const int chunk = stage_slot_chunk<BK * 2>(r, slot % CPR);
    boff[j] = (col0 + r) * p.ldb + chunk * 8;
  }

  auto issue = [&](int kt) {
    uint8_t* s = lds + (kt % NS) * kStage;
    const int k0 = kt * BK;
#pragma unroll
    for (int j = 0; j < LA; j++) {
      lds_dma16(p.Ah + aoff[j] + k0, s + (wave * LA + j) * 1024);
      if constexpr (AT == 2) lds_dma16(p.Al + aoff[j] + k0, s + kA + (wave * LA + j) * 1024);
    }
#pragma unroll
    for (int j = 0; j < LB; j++) {
      lds_dma16(p.Bh + boff[j] + k0, s + AT * kA + (wave * LB + j) * 1024);
      if constexpr (BT == 2)
        lds_dma16(p.Bl + boff[j] + k0, s + AT * kA + kB + (wave * LB + j) * 1024);
    }
  };

  v16f acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

  const int fr = lane & 31, fg = lane >> 5;
  // The fragments of one 16-k step, held twice: step s + 1 (the next stage's
  // first, past the barrier, after a stage's last) is read from LDS under the
  // products of step s.
  struct Frags {
    v8bf a[AT][TM], b[BT][TN];
  };
  auto read = [&](Frags& f, int kt, int s) {
    const uint8_t* sA = lds + (kt % NS) * kStage;
    const uint8_t* sB = sA + AT * kA;
    const int c = 2 * s + fg;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const int off = stage_frag_off<BK * 2>(wm * WM + i * 32 + fr, c);
#pragma unroll
      for (int x = 0; x < AT; x++) f.a[x][i] = *reinterpret_cast<const v8bf*>(sA + x * kA + off);
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int off = stage_frag_off<BK * 2>(wn * WN + j * 32 + fr, c);
#pragma unroll
      for (int x = 0; x < BT; x++) f.b[x][j] = *reinterpret_cast<const v8bf*>(sB + x * kB + off);
    }
  };
  // hi·hi, then hi·lo, then lo·hi of every tile: an output's sums keep their
  // order and no product waits for the one before it
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int x = 0; x < AT + BT - 1; x++)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              f.a[x == BT ? 1 : 0][i], f.b[x == 1 && BT == 2 ? 1 : 0][j], acc[i][j], 0, 0, 0);
  };

  // The one-term 256x256 tile keeps no fragments past a step: its 128 accumulators
  // leave the compiler to place a stage's reads by itself, and holding the next
  // step's across the barrier took 1-4 % longer (M = 16384: K = 768, N = 3072 104 µs
  // against 100, K = 3072, N = 768 99 against 96). Its next stage is requested as a
  // stage begins.
  constexpr bool kPlain = AT + BT == 2 && BM == 256 && BN == 256;
  if constexpr (kPlain) {
    static_assert(NS == 2, "two stages");
    issue(0);
    for (int kt = 0; kt < nk; kt++) {
      wait_vmcnt<0>();   // stage kt has landed for this wave,
      wait_lgkmcnt0();   // which has read all of stage kt - 1,
      stage_barrier();   // and so has and did every other
      if (kt + 1 < nk) issue(kt + 1);
      const uint8_t* sA = lds + (kt % NS) * kStage;
      const uint8_t* sB = sA + kA;
#pragma unroll
      for (int s = 0; s < BK / 16; s++) {
        const int c = 2 * s + fg;
        v8bf fa[TM], fb[TN];
#pragma unroll
        for (int i = 0; i < TM; i++)
          fa[i] = *reinterpret_cast<const v8bf*>(
              sA + stage_frag_off<BK * 2>(wm * WM + i * 32 + fr, c));
#pragma unroll
        for (int j = 0; j < TN; j++)
          fb[j] = *reinterpret_cast<const v8bf*>(
              sB + stage_frag_off<BK * 2>(wn * WN + j * 32 + fr, c));
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++)
            acc[i][j] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
      }
    }
  } else {
#pragma unroll
    for (int st = 0; st < NS; st++)
      if (st < nk) issue(st);
    wait_stages<kLoads, NS - 1>(nk - 1);  // stage 0 has landed for this wave
    stage_barrier();                      // and for the others
    // To stage kt + 1: this wave's loads of it have landed once only those of the
    // later stages issued are pending. Past the barrier that holds for every wave
    // (a __syncthreads() fence would drain the ring) and all reads of stage kt are
    // done, so its slot can be refilled.
    auto advance = [&](int kt) {
      wait_stages<kLoads, NS - 2>(nk - 2 - kt);
      stage_barrier();
      if (kt + NS < nk) issue(kt + NS);
    };
    if (LW > 0 && wave >= NW) {
      for (int kt = 0; kt + 1 < nk; kt++) advance(kt);
    } else {
      constexpr int S = BK / 16;
      Frags f[2];
      read(f[0], 0, 0);
      for (int kt = 0; kt + 1 < nk; kt++) {
#pragma unroll
        for (int s = 0; s < S; s++) {
          if (s + 1 < S) {
            read(f[(s + 1) & 1], kt, s + 1);
          } else {
            wait_lgkmcnt0();
            advance(kt);
            read(f[0], kt + 1, 0);
          }
          multiply(f[s & 1]);
        }
      }
#pragma unroll
      for (int s = 0; s < S; s++) {
        if (s + 1 < S) read(f[(s + 1) & 1], nk - 1, s + 1);
        multiply(f[s & 1]);
      }
    }
  }

  // ---- epilogue ----------------------------------------------------------
  // applyDense order (bert.go:282-301, pack8.go:118-122): fp32 sum, ·scale
  // (weight-only int8), + bias, then the activation.
  __syncthreads();
  if (LW > 0 && wave >= NW) return;
  float* ep = reinterpret_cast<float*>(lds) + wave * 32 * kEpiStride;
  // QKN: this lane's column scales, bias and norm weights (fixed columns
  // 4*lane..+3 of the tile for every row)
  v4f qk_cs = {1.0f, 1.0f, 1.0f, 1.0f}, qk_bs = {0.0f, 0.0f, 0.0f, 0.0f};
  v4f qk_g = {1.0f, 1.0f, 1.0f, 1.0f};
  // and the positions of this wave row's WM rows (lane r: row r), read per row
  // with readlane: no dependent global load before a row's cos/sin loads
  int qk_pos0 = 0;
  if constexpr (QKN) {
    static_assert(WM <= 64, "one position register covers the wave row");
    const int r = row0 + wm * WM + lane;
    qk_pos0 = r < p.M ? p.qk_pos[r] : 0;
    const int gcol = col0 + lane * 4, h = gcol / p.qk_dh, d = gcol % p.qk_dh;
    if (p.col_scales) qk_cs = *reinterpret_cast<const v4f*>(p.col_scales + gcol);
    if (p.bias) qk_bs = *reinterpret_cast<const v4f*>(p.bias + gcol);
    if (h < p.qk_nq + p.qk_nkv)
      qk_g = *reinterpret_cast<const v4f*>((h < p.qk_nq ? p.qk_qg : p.qk_kg) + d);
  }
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++)
        ep[((r >> 2) * 8 + fg * 4 + (r & 3)) * kEpiStride + j * 32 + fr] = acc[i][j][r];
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    const int grow_base = row0 + wm * WM + i * 32;
    if constexpr (QKN) {
      // The band's 32 rows x BN columns are parked across the WGN waves of
      // this wave row (wave wn holds columns [wn*WN, wn*WN + WN)). A pass
      // takes one tile row: lane l holds columns 4l..4l+3, a head is dh/4
      // consecutive lanes (the separate QK-norm pass's layout), and wave wn
      // takes rows wn, wn + WGN, ... of the band. The arithmetic is the
      // separate pass's, element for element (the sum of squares adds lane
      // pairs, then a butterfly over the head's lanes).
      static_assert(BN == 256, "a pass is one 256-column tile row of 64 lanes");
      __syncthreads();  // every wave of the band row has parked its columns
      const int dh = p.qk_dh, lph = dh >> 2, half = dh >> 1;
      const int c = lane * 4, l = lane % lph, d = l * 4;
      const int gcol = col0 + c, h = gcol / dh;
      const bool vh = h >= p.qk_nq + p.qk_nkv;  // v head: conversion only
      const bool first = l < (lph >> 1);        // columns d < dh/2
      const int dp = first ? d : d - half;
      const float* src0 = reinterpret_cast<const float*>(lds) +
                          (wm * WGN + c / WN) * 32 * kEpiStride + c % WN;
      typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
      // This wave's rows of the band, RPW at a time: their cos/sin pieces are loaded
      // before the first row's store, so no table load queues behind a store
      // (vmcnt counts both in order). All eight at once would take 64 registers
      // beside the accumulators not yet parked: 138 in all and one workgroup per
      // CU, or spills at the 128 that two allow. With four it is 112.
      constexpr int RPW = 4;
      static_assert(32 / WGN % RPW == 0, "rows per wave and band");
#pragma unroll
      for (int k0 = 0; k0 < 32 / WGN; k0 += RPW) {
        v4f ccs[RPW], sns[RPW];
#pragma unroll
        for (int k = 0; k < RPW; k++) {
          const int wr = i * 32 + wn + (k0 + k) * WGN;  // row within the wave row (uniform)
          const int pos = __builtin_amdgcn_readlane(qk_pos0, wr);
          ccs[k] = *reinterpret_cast<const v4f*>(p.qk_cos + (size_t)pos * half + dp);
          sns[k] = *reinterpret_cast<const v4f*>(p.qk_sin + (size_t)pos * half + dp);
        }
#pragma unroll
        for (int k = 0; k < RPW; k++) {
          const int rr = wn + (k0 + k) * WGN;
          v4f x = *reinterpret_cast<const v4f*>(src0 + rr * kEpiStride);
          const int grow = grow_base + rr;
          const bool ok = grow < p.M;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            if (p.col_scales) x[e] = x[e] * qk_cs[e];
            if (p.bias) x[e] = x[e] + qk_bs[e];
          }
          float ss = (x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]);
          for (int o = lph >> 1; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
          v4bf* out = reinterpret_cast<v4bf*>(p.qk_out + (size_t)grow * p.ldc + gcol);
          const v4f cc = ccs[k], sn = sns[k];
          const float inv = rms_inv(ss, dh, p.qk_eps);
          v4f xn, pn;
#pragma unroll
          for (int e = 0; e < 4; e++) xn[e] = x[e] * inv * qk_g[e];
#pragma unroll
          for (int e = 0; e < 4; e++) pn[e] = __shfl_xor(xn[e], lph >> 1, 64);
          v4f o;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float a = first ? xn[e] : pn[e], b = first ? pn[e] : xn[e];
            o[e] = first ? a * cc[e] - b * sn[e] : b * cc[e] + a * sn[e];
          }
          if (vh) o = x;
          if (ok) *out = v4bf{(__bf16)o[0], (__bf16)o[1], (__bf16)o[2], (__bf16)o[3]};
        }
      }
      __syncthreads();  // the next band overwrites the parked columns
    } else if constexpr (GLU) {
      // Gated weight: tile columns 8t..8t+3 are gate rows, 8t+4..8t+7 the
      // matching up rows. A lane reads both halves of one group of 8 and
      // writes act(gate) * up at output column (packed column) / 2.
      constexpr int kL8 = WN / 8, kR8 = 64 / kL8;
      const int c8 = (lane % kL8) * 8;
      const int gpk = col0 + wn * WN + c8;
      const bool pk_ok = gpk < p.N;
      v4f csg = {1.0f, 1.0f, 1.0f, 1.0f}, csu = csg;
      v4f bg = {0.0f, 0.0f, 0.0f, 0.0f}, bu = bg;
      if (pk_ok) {
        if (p.col_scales) {
          csg = *reinterpret_cast<const v4f*>(p.col_scales + gpk);
          csu = *reinterpret_cast<const v4f*>(p.col_scales + gpk + 4);
        }
        if (p.bias) {
          bg = *reinterpret_cast<const v4f*>(p.bias + gpk);
          bu = *reinterpret_cast<const v4f*>(p.bias + gpk + 4);
        }
      }
      for (int rr = lane / kL8; rr < 32; rr += kR8) {
        const int grow = grow_base + rr;
        const v4f ag = *reinterpret_cast<const v4f*>(ep + rr * kEpiStride + c8);
        const v4f au = *reinterpret_cast<const v4f*>(ep + rr * kEpiStride + c8 + 4);
        if (grow < p.M && pk_ok) {
          v4f o;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            float g = ag[e], u = au[e];
            if (p.col_scales) {
              g = g * csg[e];
              u = u * csu[e];
            }
            if (p.bias) {
              g = g + bg[e];
              u = u + bu[e];
            }
            o[e] = glu_act(g, u, p.act);
          }
          if (p.Ch) store_planes4(p.Ch, p.Cl, (size_t)grow * p.ldc + gpk / 2, o);
          else *reinterpret_cast<v4f*>(p.C + (size_t)grow * p.ldc + gpk / 2) = o;
        }
      }
    } else {
      constexpr int kLanesPerRow = WN / 4;
      constexpr int kRowsPerPass = 64 / kLanesPerRow;
      const int c4 = (lane % kLanesPerRow) * 4;
      const int gcol = col0 + wn * WN + c4;
      const bool col_ok = gcol < p.N;
      v4f cs = {1.0f, 1.0f, 1.0f, 1.0f}, bs = {0.0f, 0.0f, 0.0f, 0.0f};
      if (col_ok) {
        if (p.col_scales) cs = *reinterpret_cast<const v4f*>(p.col_scales + gcol);
        if (p.bias) bs = *reinterpret_cast<const v4f*>(p.bias + gcol);
      }
#pragma unroll 2
      for (int rr = lane / kLanesPerRow; rr < 32; rr += kRowsPerPass) {
        const int grow = grow_base + rr;
        const v4f a = *reinterpret_cast<const v4f*>(ep + rr * kEpiStride + c4);
        if (grow < p.M && col_ok) {
          v4f v;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            float x = a[e];
            if (p.col_scales) x = x * cs[e];
            if (p.bias) x = x + bs[e];
            v[e] = apply_act(x, p.act);
          }
          if (p.Ch) store_planes4(p.Ch, p.Cl, (size_t)grow * p.ldc + gcol, v);
          else *reinterpret_cast<v4f*>(p.C + (size_t)grow * p.ldc + gcol) = v;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// a [M][lda_f] fp32 -> hi/lo [M][ldk] bf16 planes, zero in [K, ldk). One
// thread per 4 columns; rows with 16-byte aligned 4-groups load as float4.
__global__ __launch_bounds__(256) void split_bf16_kernel(const float* __restrict__ a,
                                                         int lda_f, int M, int K,
                                                         __bf16* __restrict__ hi,
                                                         __bf16* __restrict__ lo, int ldk,
                                                         int vec) {
  typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
  const int groups = ldk >> 2;
  const size_t total = (size_t)M * groups;
  for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < total;
       g += (size_t)gridDim.x * blockDim.x) {
    const int row = (int)(g / groups);
    const int c = (int)(g % groups) * 4;
    const float* src = a + (size_t)row * lda_f + c;
    v4f x;
    if (vec && c + 4 <= K) {
      x = *reinterpret_cast<const v4f*>(src);
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = c + e < K ? src[e] : 0.0f;
    }
    v4bf h, l;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      __bf16 a, b;
      split_hi_lo(x[e], a, b);
      h[e] = a;
      l[e] = b;
    }
    *reinterpret_cast<v4bf*>(hi + (size_t)row * ldk + c) = h;
    if (lo) *reinterpret_cast<v4bf*>(lo + (size_t)row * ldk + c) = l;
  }
}

hipError_t launch_split_bf16(const float* a, int lda_f, int M, int K, __bf16* hi, __bf16* lo,
                             int ldk, hipStream_t s) {
  if (M <= 0) return hipSuccess;
  if (ldk % 64 != 0 || ldk < K) return hipErrorInvalidValue;
  const int vec = (lda_f % 4 == 0) && ((reinterpret_cast<uintptr_t>(a) & 15) == 0);
  const size_t total = (size_t)M * (ldk / 4);
  const size_t blocks = std::min<size_t>((total + 255) / 256, 256 * 16);
  timed_launch(split_bf16_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a, lda_f, M, K,
                     hi, lo, ldk, vec);
  return hipGetLastError();
}

template <int BM, int BN, int NS, int AT, int BT, int BK, int WGM, int WGN, int LW = 0>
static hipError_t launch_pl(const GemmPlArgs& a, hipStream_t s) {
  const int tiles = ceil_div(a.M, BM) * ceil_div(a.N, BN);
  if (is_glu(a.act))
    timed_launch((gemm_planes_kernel<BM, BN, NS, AT, BT, true, BK, WGM, WGN, LW>), dim3(tiles),
                 dim3(64 * (WGM * WGN + LW)), 0, s, a);
  else
    timed_launch((gemm_planes_kernel<BM, BN, NS, AT, BT, false, BK, WGM, WGN, LW>), dim3(tiles),
                 dim3(64 * (WGM * WGN + LW)), 0, s, a);
  return hipGetLastError();
}

// Tiles: 1, 4 and 6 = 256x256, 2, 5 and 7 = 256x128, 3 = 128x128, 8 = 64x64,
// 9 = 128x64, 10 = 128x256 (one term; else 128x128). All 32-bit sums run over K
// in the same order, so a row has the same bits on every tile.
//
// One term, fp32: the tile whose rounds of the chip take the least. One-term
// tiles cost, in µs, c0 + full rounds * (r + rk*K) + (h + hk*K) if a last round
// of two-per-CU tiles puts at most one workgroup on a CU (fitted to 300 sizes of
// M 256..32768, K 200..3200, N 320..6400 on MI355X; the choice is within 0.5 % of
// the fastest tile on average). 128x128 is ahead on up to a few rounds of short
// K, 256x256 on many or deep ones, where its operands are read half as often
// (weight-only int8, µs on 128x128 against 256x256: M = 32768, K = 3072, N = 1024
// 250 - 195; M = 16384, K = 2048, N = 1024 76.9 - 66.5; M = 16384, K = 768, N = 3072
// 101 - 91.8, N = 2304 72.7 - 89); 64x64 where they leave CUs idle (M = 2048,
// K = 2048, N = 1024 22.8 - 17.4 on 64x64). Gated rows leave a 256x256 workgroup
// alone on its CU for a long epilogue; 128x256, two to a CU, hides it (M = 16384,
// K = 768, N = 6144 213 - 201).
// fp32: as units of 1e-8 s per k (256x256 86, 256x128 47.8 and 128x128 27.5 with
// one workgroup per CU, 64x64 8 with two; measured at M = 16384, K = 1024, N =
// 6144). µs before -> now: M = 16384 620 -> 586, M = 3896, K = 3072, N = 1024
// 113 -> 71, M = 4012, K = 1152, N = 768 46.5 -> 26.9, M = 2408, K = 1536, N = 384
// 17.4 -> 15.1, M = 349, K = 3072, N = 768 28.5 -> 23.4.
// Weight-only int8 on two activation terms: 256x256 while its grid fills the
// chip, 256x128 down to 96 tiles, 128x128 down to 192, then 64x64.
int pick_planes_tile(int M, int N, int K, int a_terms, int b_terms, bool glu) {
  auto tiles = [&](int bm, int bn) { return (long long)ceil_div(M, bm) * ceil_div(N, bn); };
  if (a_terms == 1 && b_terms == 1) {
    auto cost = [&](long long t, int per_cu, double c0, double r, double rk, double h, double hk) {
      const long long round = 256LL * per_cu, rest = t % round;
      const bool half = per_cu == 2 && rest > 0 && rest <= 256;
      const long long full = t / round + (rest > 0 && !half);
      return c0 + full * (r + rk * K) + (half ? h + hk * K : 0.0);
    };
    const double t1 = cost(tiles(256, 256), 1, -2.5, glu ? 19.0 : 13.0, 0.0216, 0.0, 0.0);
    const double t3 = cost(tiles(128, 128), 2, 1.8, glu ? 4.7 : 3.6, 0.0160, glu ? 3.7 : 2.6, 0.0076);
    const double t8 = cost(tiles(64, 64), 2, 2.8, glu ? 2.0 : 1.6, 0.0058, glu ? 2.0 : 1.3, 0.0038);
    int best = t1 < t3 ? 1 : 3;
    double us = std::min(t1, t3);
    if (t8 < us) {
      best = 8;
      us = t8;
    }
    if (glu && cost(tiles(128, 256), 2, 0.3, 7.4, 0.0310, 9.5, 0.0146) < us) best = 10;
    return best;
  }
  if (b_terms == 1) {
    if (tiles(256, 256) >= 256) return 1;
    if (tiles(256, 128) >= 96) return 2;
    return tiles(128, 128) >= 192 ? 3 : 8;
  }
  const double t1 = 86.0 * ((tiles(256, 256) + 255) / 256);
  const double t2 = 47.8 * ((tiles(256, 128) + 255) / 256);
  const double t3 = 27.5 * ((tiles(128, 128) + 255) / 256);
  const double t8 = 16.0 * ((tiles(64, 64) + 511) / 512);
  if (t8 <= t1 && t8 <= t2 && t8 <= t3) return 8;
  if (t3 <= t1 && t3 <= t2) return 3;
  return t2 <= t1 ? 2 : 1;
}

hipError_t launch_gemm_planes_qk(const GemmPlArgs& a, hipStream_t s) {
  if (a.M <= 0) return hipSuccess;
  if (a.N % 256 != 0 || a.lda % 64 != 0 || a.ldb % 64 != 0 || a.ldc % 4 != 0 || !a.qk_out ||
      !(a.qk_dh == 64 || a.qk_dh == 128 || a.qk_dh == 256) || is_glu(a.act))
    return hipErrorInvalidValue;
  // µs on 256x256 tiles, here with eight rows of cos/sin at once, here (one stream):
  // K = 768, N = 1280: M = 32768 155, 132, 125, M = 16384 100, 82, 74; K = 1024,
  // N = 4096: M = 16384 222, 208, 198, M = 8192 110, 108, 104
  const int tiles = ceil_div(a.M, 128) * (a.N / 256);
  timed_launch((gemm_planes_kernel<128, 256, 3, 1, 1, false, 32, 2, 4, 0, true>), dim3(tiles),
               dim3(512), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_gemm_planes(const GemmPlArgs& a, int a_terms, int b_terms, int tile,
                              hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if (a.lda % 64 != 0 || a.ldb % 64 != 0) return hipErrorInvalidValue;
  if (tile <= 0 || tile > kPlanesTileConfigs) {
    if (const int small = pick_small_tile(a.M, a.N, a_terms + b_terms)) {
      GemmSmallArgs g{};
      g.A = a.Ah;
      g.Al = a.Al;
      g.lda = 2 * a.lda;
      g.B = a.Bh;
      g.Bl = a.Bl;
      g.ldb = 2 * a.ldb;
      g.M = a.M;
      g.N = a.N;
      g.kbytes = 2 * a.K;
      g.col_scales = a.col_scales;
      g.bias = a.bias;
      g.out = a.Ch ? static_cast<void*>(a.Ch) : static_cast<void*>(a.C);
      g.out_lo = a.Cl;
      g.ldo = a.ldc;
      g.act = a.act;
      g.epi = a.Ch ? EPI_PLANES : EPI_F32;
      return launch_gemm_small_planes(g, a_terms, b_terms, small, s);
    }
    tile = pick_planes_tile(a.M, a.N, a.K, a_terms, b_terms, is_glu(a.act));
  }
  if (a_terms == 1 && b_terms == 1) {
    switch (tile) {
      case 1:
      case 4:
      case 6: return launch_pl<256, 256, 2, 1, 1, 64, 2, 4>(a, s);
      case 2:
      case 5:
      case 7: return launch_pl<256, 128, 3, 1, 1, 32, 4, 2>(a, s);
      case 8: return launch_pl<64, 64, 4, 1, 1, 64, 2, 2, 4>(a, s);
      case 9: return launch_pl<128, 64, 2, 1, 1, 64, 2, 2>(a, s);
      case 10: return launch_pl<128, 256, 3, 1, 1, 32, 2, 4>(a, s);
      default: return launch_pl<128, 128, 2, 1, 1, 64, 4, 2>(a, s);
    }
  }
  if (a_terms == 2 && b_terms == 1) {
    switch (tile) {
      case 1:
      case 4:
      case 6: return launch_pl<256, 256, 3, 2, 1, 32, 2, 4>(a, s);
      case 2:
      case 5:
      case 7: return launch_pl<256, 128, 4, 2, 1, 32, 4, 2>(a, s);
      case 8: return launch_pl<64, 64, 3, 2, 1, 64, 2, 2, 4>(a, s);
      case 9: return launch_pl<128, 64, 4, 2, 1, 32, 2, 2>(a, s);
      default: return launch_pl<128, 128, 3, 2, 1, 32, 4, 2>(a, s);
    }
  }
  if (a_terms == 2 && b_terms == 2) {
    switch (tile) {
      case 1:
      case 4:
      case 6: return launch_pl<256, 256, 2, 2, 2, 32, 2, 4>(a, s);
      case 2:
      case 5:
      case 7: return launch_pl<256, 128, 3, 2, 2, 32, 4, 2>(a, s);
      case 8:  // four stages in flight with one workgroup per CU, else two with two
        // (M = 349, K = 3072, N = 768, 72 tiles: 23.4 against 31.8; M = 349, K = 768,
        // N = 3072, 288 tiles: 16.1 against 12.8)
        if ((long long)ceil_div(a.M, 64) * ceil_div(a.N, 64) <= 256)
          return launch_pl<64, 64, 4, 2, 2, 64, 2, 2, 4>(a, s);
        return launch_pl<64, 64, 2, 2, 2, 64, 2, 2, 4>(a, s);
      case 9: return launch_pl<128, 64, 3, 2, 2, 64, 2, 2, 4>(a, s);
      default: return launch_pl<128, 128, 2, 2, 2, 64, 4, 2>(a, s);
    }
  }
  return hipErrorInvalidValue;
}

}  // namespace rh
