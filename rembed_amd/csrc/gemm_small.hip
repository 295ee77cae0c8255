// gemm_small.hip — the GEMMs of few rows (a query, a page of short texts):
// full int8 on v_mfma_i32_16x16x64_i8 and the bf16-planes products (weight-only
// int8, fp32) on v_mfma_f32_16x16x32_bf16.
//
// With few rows the tiled kernels (gemm_i8.hip, gemm_planes.hip) launch a
// handful of workgroups that each walk the whole of K stage by stage, one
// memory latency and one barrier per stage: at 28 rows a full-int8 768x768
// linear ran 6 workgroups of 12 stages. What bounds such a call is that chain
// and the bytes one CU can pull, so here a workgroup owns a small output tile,
// 16·RT rows x 16·CT columns, its NW waves hold different shares of K, and
// fragments go straight from global memory to registers (a wave's share is
// read by nobody else in the workgroup, so LDS staging would share nothing):
// the loads of all shares are in flight at once. The epilogue's scales and
// bias are loaded with them, so no memory latency follows the last product.
//
//   * int8: each wave sums its share; the int32 partials meet in LDS (exact in
//     any order).
//   * planes: the fp32 sum of one output runs over K in the tiled kernels'
//     order, so a row's result does not depend on how many rows are computed
//     with it (an instruction adds groups of 4 consecutive k in ascending
//     order: one 16x16x32 product equals two chained 32x32x16 ones bit for
//     bit). The shares therefore take turns: the accumulators pass from wave to
//     wave through LDS in K order, while the later shares are still loading.
//     The two-term products interleave hi·hi, hi·lo and lo·hi per 16 k, so
//     those run each half of a 32-k fragment with the other half zeroed.
//
// Measured per launch on MI355X (HIP events, six weights used in turn), tiled
// kernels -> here, µs, at 28 rows (K x N):
//   768 x 768   int8 10.4 -> 5.1, weight-only int8 6.4 -> 4.0, fp32 9.1 -> 6.9
//   768 x 3072  int8 10.8 -> 5.5, weight-only int8 7.0 -> 4.7
//   3072 x 768  int8 24.9 -> 6.6, weight-only int8 17.7 -> 7.7, fp32 25.7 -> 17.8
// About 4.0 µs of each is the launch itself (no kernel of this size measured
// less). What bounds the deep ones is the 0.2-0.4 MB one CU pulls at ~50 B/ns
// and, for fp32, six dependent products per 32 k.
#include "gemm_common.h"

namespace rh {

typedef __bf16 v4bf __attribute__((ext_vector_type(4)));

namespace {

__device__ __forceinline__ uint32_t small_qbyte(float v, float inv) {
  int q = (int)rintf(v * inv) + 128;
  return (uint32_t)(q < 0 ? 0 : (q > 255 ? 255 : q));
}

// The workgroup's output tile: an XCD owns consecutive tiles, row blocks
// first, so the tiles that share a column block's weights read them through
// one L2.
template <int R, int C>
__device__ __forceinline__ void small_tile(const GemmSmallArgs& p, int& row0, int& col0) {
  const int tiles_m = (p.M + R - 1) / R;
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  row0 = (t % tiles_m) * R;
  col0 = (t / tiles_m) * C;
}

// Epilogue over an R x C tile: a thread finishes 4 columns (8 packed ones of a
// gated weight) of GPT rows, GR rows apart. Its operands are loaded by the
// constructor, before the main loop.
template <bool I8, int R, int C, int NW>
struct SmallEpilogue {
  static constexpr int GPT = R * C / 4 > 64 * NW ? R * C / 4 / (64 * NW) : 1, GR = R / GPT;
  static_assert(GPT == 1 || GR * C / 4 == 64 * NW, "groups");
  static_assert(R * C / 8 <= 64 * NW, "gated groups");
  const GemmSmallArgs& p;
  int row0, col0, er, ec;
  bool glu;
  float rs[GPT];
  v4f cs0 = {1.0f, 1.0f, 1.0f, 1.0f}, cs1 = cs0, bs0 = {0.0f, 0.0f, 0.0f, 0.0f}, bs1 = bs0;

  __device__ __forceinline__ SmallEpilogue(const GemmSmallArgs& a, int r0, int c0)
      : p(a), row0(r0), col0(c0), glu(is_glu(a.act)) {
    const int tid = threadIdx.x;
    er = glu ? tid / (C / 8) : tid / (C / 4);
    ec = glu ? tid % (C / 8) * 8 : tid % (C / 4) * 4;
#pragma unroll
    for (int k = 0; k < GPT; k++) {
      const int row = row0 + er + k * GR;
      rs[k] = I8 && p.epi != EPI_ACC && er < R && row < p.M ? p.row_scales[row] : 1.0f;
    }
    if (er < R && col0 + ec < p.N) {
      if (p.col_scales) {
        cs0 = *reinterpret_cast<const v4f*>(p.col_scales + col0 + ec);
        if (glu) cs1 = *reinterpret_cast<const v4f*>(p.col_scales + col0 + ec + 4);
      }
      if (p.bias) {
        bs0 = *reinterpret_cast<const v4f*>(p.bias + col0 + ec);
        if (glu) bs1 = *reinterpret_cast<const v4f*>(p.bias + col0 + ec + 4);
      }
    }
  }

  // applyDense's order: the int32 sum to float32 ·row scale (int8), ·column
  // scale (not fp32), + bias.
  template <class A>
  __device__ __forceinline__ v4f dense(const A& a, float rsv, const v4f& cs, const v4f& bs) {
    v4f v;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      v[e] = (float)a[e];
      if constexpr (I8) v[e] = v[e] * rsv;
      if (p.col_scales) v[e] = v[e] * cs[e];
      if (p.bias) v[e] = v[e] + bs[e];
    }
    return v;
  }

  // sum4(r, c): the raw sums of tile row r, columns c..c+3.
  template <class F>
  __device__ __forceinline__ void finish(F&& sum4) {
    if (er >= R) return;
    const int col = col0 + ec;
#pragma unroll
    for (int k = 0; k < GPT; k++) {
      const int r = er + k * GR, row = row0 + r;
      const bool ok = row < p.M && col < p.N;
      if (glu) {  // packed columns 8t..8t+3 gate, 8t+4..8t+7 up
        if (!ok || k > 0) continue;  // all of them in one go
        const v4f ga = dense(sum4(r, ec), rs[k], cs0, bs0);
        const v4f up = dense(sum4(r, ec + 4), rs[k], cs1, bs1);
        v4f o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = glu_act(ga[e], up[e], p.act);
        const size_t at = (size_t)row * p.ldo + col / 2;
        if (p.epi == EPI_PLANES)
          store_planes4(static_cast<__bf16*>(p.out), static_cast<__bf16*>(p.out_lo), at, o);
        else
          *reinterpret_cast<v4f*>(static_cast<float*>(p.out) + at) = o;
        continue;
      }
      const size_t at = (size_t)row * p.ldo + col;
      if constexpr (I8) {
        if (p.epi == EPI_ACC) {
          if (!ok) continue;
          const v4i a = sum4(r, ec);
          v4i w;
#pragma unroll
          for (int e = 0; e < 4; e++)
            w[e] = (int)((uint32_t)a[e] + 128u * (uint32_t)p.colsum[col + e]);
          *reinterpret_cast<v4i*>(static_cast<int32_t*>(p.out) + at) = w;
          continue;
        }
      }
      v4f v = {0.0f, 0.0f, 0.0f, 0.0f};
      if (ok) {
        v = dense(sum4(r, ec), rs[k], cs0, bs0);
        if (p.act == ACT_GELU) {
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = gelu_avx2(v[e]);
        }
      }
      if constexpr (I8) {
        if (p.epi == EPI_ABSMAX) {  // row |max| over the tile's columns; whole waves are here
          float m = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
#pragma unroll
          for (int o = C / 8; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
          if (row < p.M && ec == 0)
            atomicMax(reinterpret_cast<unsigned int*>(p.row_absmax) + row, __float_as_uint(m));
          continue;
        }
      }
      if (!ok) continue;
      switch (p.epi) {
        case EPI_F32:
          *reinterpret_cast<v4f*>(static_cast<float*>(p.out) + at) = v;
          break;
        case EPI_BF16:
          *reinterpret_cast<v4bf*>(static_cast<__bf16*>(p.out) + at) =
              v4bf{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
          break;
        case EPI_PLANES:
          store_planes4(static_cast<__bf16*>(p.out), static_cast<__bf16*>(p.out_lo), at, v);
          break;
        case EPI_QUANT: {
          float scale = p.row_absmax[row] / 127.0f;
          if (scale == 0.0f) scale = 1.0f;
          const float inv = 1.0f / scale;
          *reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(p.out) + at) =
              small_qbyte(v[0], inv) | (small_qbyte(v[1], inv) << 8) |
              (small_qbyte(v[2], inv) << 16) | (small_qbyte(v[3], inv) << 24);
          if (col == 0) p.rs_out[row] = scale;
          break;
        }
      }
    }
  }
};

}  // namespace

// u8 rows x s8 weights. A 16x16 step is 64 bytes of K: lane l holds row (column)
// l % 16 and the 16 bytes at 16·(l / 16); output column l % 16, rows
// 4·(l / 16) + r. Two register buffers of U steps per wave.
template <int RT, int CT, int NW, int U>
__global__ __launch_bounds__(64 * NW) void gemm_small_i8_kernel(GemmSmallArgs p) {
  constexpr int R = 16 * RT, C = 16 * CT;
  constexpr int S = C + 4;  // words per row of a partial tile (spreads the banks)
  static_assert(NW * R * S * 4 <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(16))) int part[NW * R * S];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int row0, col0;
  small_tile<R, C>(p, row0, col0);
  // this wave's share of the k steps
  const int steps = (p.kbytes + 63) / 64;
  const int per = (steps + NW - 1) / NW;
  const int s0 = min(wave * per, steps), s1 = min(s0 + per, steps);

  const int fr = lane & 15, fo = (lane >> 4) * 16;
  const uint8_t* arow[RT];
  const uint8_t* brow[CT];
#pragma unroll
  for (int i = 0; i < RT; i++)  // rows past M read row M-1; their outputs are never stored
    arow[i] = static_cast<const uint8_t*>(p.A) + (size_t)min(row0 + 16 * i + fr, p.M - 1) * p.lda;
#pragma unroll
  for (int j = 0; j < CT; j++)  // weight rows are zero-padded to a multiple of 256
    brow[j] = static_cast<const uint8_t*>(p.B) + (size_t)(col0 + 16 * j + fr) * p.ldb;

  struct Frags {
    v4i a[RT], b[CT];
  };
  auto load = [&](Frags& f, int s) {
    // steps past the wave's share re-read its last one (never multiplied)
    const int kb = min(s, s1 - 1) * 64 + fo;
    // A's rows end at lda >= round_up(K, 16); the weight is zero past K
    const int ka = kb + 16 > p.lda ? 0 : kb;
#pragma unroll
    for (int i = 0; i < RT; i++) f.a[i] = *reinterpret_cast<const v4i*>(arow[i] + ka);
#pragma unroll
    for (int j = 0; j < CT; j++) f.b[j] = *reinterpret_cast<const v4i*>(brow[j] + kb);
  };
  v4i acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int j = 0; j < CT; j++) acc[i][j] = v4i{0, 0, 0, 0};
  auto multiply = [&](Frags& f) {
#pragma unroll
    for (int i = 0; i < RT; i++) {
      f.a[i] = f.a[i] ^ (int)0x80808080;  // u8 ^ 0x80 = q, QuantizeRowU8's byte less 128
#pragma unroll
      for (int j = 0; j < CT; j++)
        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
    }
  };

  Frags f0[U], f1[U];
  if (s0 < s1) {
#pragma unroll
    for (int u = 0; u < U; u++) load(f0[u], s0 + u);
  }
  SmallEpilogue<true, R, C, NW> epi(p, row0, col0);
  if (s0 < s1) {
    for (int s = s0; s < s1; s += 2 * U) {
      if (s + U < s1) {
#pragma unroll
        for (int u = 0; u < U; u++) load(f1[u], s + U + u);
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (s + u < s1) multiply(f0[u]);
      if (s + 2 * U < s1) {
#pragma unroll
        for (int u = 0; u < U; u++) load(f0[u], s + 2 * U + u);
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (s + U + u < s1) multiply(f1[u]);
    }
  }
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int j = 0; j < CT; j++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        part[(wave * R + 16 * i + 4 * (lane >> 4) + r) * S + 16 * j + fr] = acc[i][j][r];
  __syncthreads();
  epi.finish([&](int r, int c) {
    v4i v = *reinterpret_cast<const v4i*>(&part[r * S + c]);
#pragma unroll
    for (int w = 1; w < NW; w++) v = v + *reinterpret_cast<const v4i*>(&part[(w * R + r) * S + c]);
    return v;
  });
}

// The planes products. A 16x16 step is 32 bf16 of K (64 bytes, the same lane
// layout); turn t is U consecutive steps and belongs to wave t % NW, which
// loads its next turn's fragments as soon as it has multiplied this one's.
template <int RT, int CT, int AT, int BT, int NW, int U>
__global__ __launch_bounds__(64 * NW) void gemm_small_planes_kernel(GemmSmallArgs p) {
  constexpr int R = 16 * RT, C = 16 * CT, S = C + 4;
  __shared__ __attribute__((aligned(16))) float part[R * S];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int row0, col0;
  small_tile<R, C>(p, row0, col0);
  const int steps = (p.kbytes + 63) / 64;
  const int turns = (steps + U - 1) / U;

  const int fr = lane & 15, fo = (lane >> 4) * 16;
  const uint8_t* arow[AT][RT];
  const uint8_t* brow[BT][CT];
#pragma unroll
  for (int i = 0; i < RT; i++) {
    const size_t off = (size_t)min(row0 + 16 * i + fr, p.M - 1) * p.lda + fo;
    arow[0][i] = static_cast<const uint8_t*>(p.A) + off;
    if constexpr (AT == 2) arow[1][i] = static_cast<const uint8_t*>(p.Al) + off;
  }
#pragma unroll
  for (int j = 0; j < CT; j++) {
    const size_t off = (size_t)(col0 + 16 * j + fr) * p.ldb + fo;
    brow[0][j] = static_cast<const uint8_t*>(p.B) + off;
    if constexpr (BT == 2) brow[1][j] = static_cast<const uint8_t*>(p.Bl) + off;
  }

  v4i fa[U][AT][RT], fb[U][BT][CT];
  auto load = [&](int t) {  // both operands are zero past K up to a multiple of 64
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kb = min(t * U + u, steps - 1) * 64;  // past the end: never multiplied
#pragma unroll
      for (int x = 0; x < AT; x++)
#pragma unroll
        for (int i = 0; i < RT; i++)
          fa[u][x][i] = *reinterpret_cast<const v4i*>(arow[x][i] + kb);
#pragma unroll
      for (int x = 0; x < BT; x++)
#pragma unroll
        for (int j = 0; j < CT; j++)
          fb[u][x][j] = *reinterpret_cast<const v4i*>(brow[x][j] + kb);
    }
  };
  v4f acc[RT][CT];
  auto mma = [&](int i, int j, const v4i& a, const v4i& b) {
    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        __builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), acc[i][j], 0, 0, 0);
  };
  auto multiply = [&](int u) {
    if constexpr (AT == 1 && BT == 1) {
#pragma unroll
      for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < CT; j++) mma(i, j, fa[u][0][i], fb[u][0][j]);
    } else {
#pragma unroll
      for (int h = 0; h < 2; h++) {  // k 0..15 sit in lanes 0..31, 16..31 in the others
        const bool mine = (lane >> 5) == h;
        v4i a[AT][RT], b[BT][CT];
#pragma unroll
        for (int e = 0; e < 4; e++) {
#pragma unroll
          for (int x = 0; x < AT; x++)
#pragma unroll
            for (int i = 0; i < RT; i++) a[x][i][e] = mine ? fa[u][x][i][e] : 0;
#pragma unroll
          for (int x = 0; x < BT; x++)
#pragma unroll
            for (int j = 0; j < CT; j++) b[x][j][e] = mine ? fb[u][x][j][e] : 0;
        }
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
          for (int j = 0; j < CT; j++) {
            mma(i, j, a[0][i], b[0][j]);
            if constexpr (BT == 2) mma(i, j, a[0][i], b[1][j]);
            if constexpr (AT == 2) mma(i, j, a[1][i], b[0][j]);
          }
      }
    }
  };

  if (wave < turns) load(wave);
  SmallEpilogue<false, R, C, NW> epi(p, row0, col0);
  // where this lane's accumulators pass: row 4·(lane / 16) + r, column lane % 16
  float* mine = part + 4 * (lane >> 4) * S + fr;
  for (int t = 0; t < turns; t++) {
    if (t % NW == wave) {
#pragma unroll
      for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < CT; j++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            acc[i][j][r] = t == 0 ? 0.0f : mine[(16 * i + r) * S + 16 * j];
#pragma unroll
      for (int u = 0; u < U; u++)
        if (t * U + u < steps) multiply(u);
#pragma unroll
      for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < CT; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) mine[(16 * i + r) * S + 16 * j] = acc[i][j][r];
      if (t + NW < turns) load(t + NW);
      wait_lgkmcnt0();  // the accumulators are in LDS (the loads stay in flight)
    }
    stage_barrier();
  }
  epi.finish([&](int r, int c) { return *reinterpret_cast<const v4f*>(&part[r * S + c]); });
}

namespace {

template <int RT, int CT, int NW, int U>
hipError_t launch_i8(const GemmSmallArgs& a, hipStream_t s) {
  const int tiles = ceil_div(a.M, 16 * RT) * ceil_div(a.N, 16 * CT);
  timed_launch((gemm_small_i8_kernel<RT, CT, NW, U>), dim3(tiles), dim3(64 * NW), 0, s, a);
  return hipGetLastError();
}

template <int RT, int CT, int AT, int BT, int NW, int U>
hipError_t launch_pl(const GemmSmallArgs& a, hipStream_t s) {
  const int tiles = ceil_div(a.M, 16 * RT) * ceil_div(a.N, 16 * CT);
  timed_launch((gemm_small_planes_kernel<RT, CT, AT, BT, NW, U>), dim3(tiles), dim3(64 * NW), 0,
               s, a);
  return hipGetLastError();
}

}  // namespace

// Which calls run here, and on which tile (1..5 = 16x16, 32x16, 32x32, 64x32,
// 64x64; 0 = the tiled kernels): the finest tile whose grid still fits one
// workgroup per CU. Finer tiles put more CUs on the weights; past one round
// the re-read operands cost more than the idle CUs did (weight-only int8, µs:
// K = 768, N = 768, 64 rows, 192 tiles of 16x16: 4.0 against 4.7 with 32x16;
// 128 rows, 384 of them: 5.3 against 4.7; N = 3072, 96 rows, 288 tiles of
// 32x32: 8.2 against 7.2 tiled).
// terms: 0 = int8, else the planes' terms in all. Products of two and three
// terms take 16x16 only: their chain of instructions, not the loads, is what
// a workgroup waits for, and it grows with the tile (fp32, K = 768, N = 768, 64
// rows: 6.9 with 16x16, 9.6 with 32x16; 96 rows, 288 tiles: 9.7 against 9.0
// tiled). int8 is worth the grids of 64x32 and 64x64 too: the tiled kernel that
// runs otherwise, 64x256, has a twelfth to a quarter of the workgroups (µs, here
// against 64x256: K = 3072, N = 768: 349 rows 12.9 - 19.1, 1344 rows 17.5 - 19.8;
// K = 768, N = 768: 700 rows 8.3 - 10.0, 1344 rows 9.3 - 10.6; N = 3072: 320 rows
// 8.9 - 10.7; past 256 tiles, 1408 rows of K = 768, N = 768, it takes 10.6).
int pick_small_tile(int M, int N, int terms) {
  static const int rt[] = {1, 2, 2, 4, 4}, ct[] = {1, 1, 2, 2, 4};
  const int most = terms == 0 ? 5 : terms == 2 ? 3 : 1;
  for (int t = 0; t < most; t++)
    if ((long long)ceil_div(M, 16 * rt[t]) * ceil_div(N, 16 * ct[t]) <= 256) return t + 1;
  return 0;
}

hipError_t launch_gemm_small_i8(const GemmSmallArgs& a, int tile, hipStream_t s) {
  switch (tile) {
    case 1: return launch_i8<1, 1, 4, 3>(a, s);
    case 2: return launch_i8<2, 1, 4, 3>(a, s);
    case 3: return launch_i8<2, 2, 4, 3>(a, s);
    case 4: return launch_i8<4, 2, 8, 3>(a, s);
    case 5: return launch_i8<4, 4, 8, 2>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_gemm_small_planes(const GemmSmallArgs& a, int a_terms, int b_terms, int tile,
                                    hipStream_t s) {
  if (a_terms == 1 && b_terms == 1) {
    switch (tile) {
      case 1: return launch_pl<1, 1, 1, 1, 8, 6>(a, s);
      case 2: return launch_pl<2, 1, 1, 1, 8, 6>(a, s);
      case 3: return launch_pl<2, 2, 1, 1, 8, 4>(a, s);
      default: return hipErrorInvalidValue;
    }
  }
  if (tile != 1 || a_terms != 2) return hipErrorInvalidValue;
  if (b_terms == 1) return launch_pl<1, 1, 2, 1, 8, 3>(a, s);
  if (b_terms == 2) return launch_pl<1, 1, 2, 2, 8, 3>(a, s);
  return hipErrorInvalidValue;
}

}  // namespace rh
