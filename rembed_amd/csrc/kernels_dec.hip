// kernels_dec.hip — row kernels of the decoder-family embedders (Qwen3,
// EmbeddingGemma) that keep activations in HBM between the GEMMs: token
// embedding gather, the residual + RMSNorm sandwich, per-head QK-norm with
// rotate-half RoPE, and EmbeddingGemma's Dense head.
//
// One 64-lane wave owns one row (or one head of one row); rows are 16-byte
// aligned and every width here is a multiple of 4, so rows move as float4.
#include "gemm_common.h"
#include "rows_common.h"

namespace rh {

namespace {

constexpr int kRows = 4;  // 256 threads = 4 waves = 4 rows

__device__ __forceinline__ uint8_t qbyte(float v, float inv) {
  int q = (int)rintf(v * inv) + 128;
  return (uint8_t)(q < 0 ? 0 : (q > 255 ? 255 : q));
}

// RMSNorm's scale (tensor.go:459-471): 1 / float32(sqrt(float64(ss/n + eps))).

}  // namespace

// ---- embeddings ---------------------------------------------------------------
// embed_tokens rows (qwen3.go:460-467), scaled by float32(sqrt(H)) for Gemma
// (gemma3.go:262-275), plus an optional row added to each (nomic's segment-0
// row: w[j] + t[j], nomic.go:177-188), and each row's position in its text
// for RoPE.
__global__ __launch_bounds__(256) void embed_gather_kernel(
    const int32_t* __restrict__ ids, int stride, const int32_t* __restrict__ cu,
    int batch, const float* __restrict__ word, const float* __restrict__ add_row, int H,
    int vocab, float scale, float* __restrict__ x, int32_t* __restrict__ pos, int* err_flag,
    int total) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRows + (threadIdx.x >> 6);
  if (row >= total) return;
  int lo = 0, hi = batch;  // text b with cu[b] <= row < cu[b+1]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu[mid] <= row) lo = mid;
    else hi = mid;
  }
  const int t = row - cu[lo];
  int id = ids[(size_t)lo * stride + t];
  if (id < 0 || id >= vocab) {
    if (lane == 0) *err_flag = 1;
    id = id < 0 ? 0 : vocab - 1;  // stay in bounds; the call reports failure
  }
  if (lane == 0) pos[row] = t;
  const float* src = word + (size_t)id * H;
  float* dst = x + (size_t)row * H;
  for (int j = lane * 4; j < H; j += 256) {
    v4f v = *reinterpret_cast<const v4f*>(src + j);
    if (scale != 1.0f) v = v * scale;
    if (add_row) v = v + *reinterpret_cast<const v4f*>(add_row + j);
    *reinterpret_cast<v4f*>(dst + j) = v;
  }
}

hipError_t launch_embed_gather(const int32_t* ids, int stride, const int32_t* cu,
                               int batch, const float* word, const float* add_row, int H,
                               int vocab, float scale, float* x, int32_t* pos, int* err_flag,
                               int total_rows, hipStream_t s) {
  if (total_rows <= 0) return hipSuccess;
  if (H % 4) return hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_gather_kernel, dim3(ceil_div(total_rows, kRows)), dim3(256), 0,
                     s, ids, stride, cu, batch, word, add_row, H, vocab, scale, x, pos,
                     err_flag, total_rows);
  return hipGetLastError();
}

// ---- residual + norm sandwich ----------------------------------------------------
//   y' = post_g ? RMSNorm(y, post_g) : y   (Gemma post-norms, gemma3.go:357,376)
//   x += y'                                 (Add, tensor.go:383-387)
//   out = RMSNorm(x, pre_g)                 (the next sublayer's pre-norm)
// or, with layer_norm set, out = LayerNorm(x, pre_g, ln_b) (tensor.go:430-452:
// biased variance, 1 / float32(sqrt(var + eps)), (v - mean) * inv * g + b;
// a null ln_b adds zero, as ModernBERT's shared zero beta does). out goes to
// fp32 rows and/or to the bf16 hi/lo planes of the next GEMM's input, plus
// an optional QuantizeRowU8 of it for a full-int8 GEMM. When out is x itself
// (a post-norm block, or the final norm) the sum is not stored first. V
// float4 per lane.
template <int V>
__global__ __launch_bounds__(256) void rms_residual_kernel(RmsArgs p) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRows + (threadIdx.x >> 6);
  if (row >= p.m) return;
  const int H = p.H;
  float* xr = p.x + (size_t)row * H;
  v4f v[V];
#pragma unroll
  for (int e = 0; e < V; e++) {
    const int j = (lane + 64 * e) * 4;
    v[e] = j < H ? *reinterpret_cast<const v4f*>(xr + j) : v4f{0.0f, 0.0f, 0.0f, 0.0f};
  }
  if (p.y) {
    const float* yr = p.y + (size_t)row * H;
    v4f w[V];
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < V; e++) {
      const int j = (lane + 64 * e) * 4;
      w[e] = j < H ? *reinterpret_cast<const v4f*>(yr + j) : v4f{0.0f, 0.0f, 0.0f, 0.0f};
      ss += (w[e][0] * w[e][0] + w[e][1] * w[e][1]) + (w[e][2] * w[e][2] + w[e][3] * w[e][3]);
    }
    if (p.post_g) {
      const float inv = rms_inv(wave_sum(ss), H, p.eps);
#pragma unroll
      for (int e = 0; e < V; e++) {
        const int j = (lane + 64 * e) * 4;
        if (j < H) {
          const v4f g = *reinterpret_cast<const v4f*>(p.post_g + j);
#pragma unroll
          for (int c = 0; c < 4; c++) w[e][c] = w[e][c] * inv * g[c];
        }
      }
    }
    const bool store_sum = p.out != p.x;
#pragma unroll
    for (int e = 0; e < V; e++) {
      const int j = (lane + 64 * e) * 4;
      if (j < H) {
        v[e] = v[e] + w[e];
        if (store_sum) *reinterpret_cast<v4f*>(xr + j) = v[e];
      }
    }
  }
  float inv, mean = 0.0f;
  if (p.layer_norm) {
    float s = 0.0f;  // lanes past H hold zeros
#pragma unroll
    for (int e = 0; e < V; e++) s += (v[e][0] + v[e][1]) + (v[e][2] + v[e][3]);
    mean = wave_sum(s) / (float)H;
    float s2 = 0.0f;
#pragma unroll
    for (int e = 0; e < V; e++) {
      const int j = (lane + 64 * e) * 4;
      if (j < H) {
        const v4f d = v[e] - mean;
        s2 += (d[0] * d[0] + d[1] * d[1]) + (d[2] * d[2] + d[3] * d[3]);
      }
    }
    inv = 1.0f / sqrtf(wave_sum(s2) / (float)H + p.eps);
  } else {
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < V; e++)
      ss += (v[e][0] * v[e][0] + v[e][1] * v[e][1]) + (v[e][2] * v[e][2] + v[e][3] * v[e][3]);
    inv = rms_inv(wave_sum(ss), H, p.eps);
  }
  float mx = 0.0f;
#pragma unroll
  for (int e = 0; e < V; e++) {
    const int j = (lane + 64 * e) * 4;
    if (j < H) {
      const v4f g = *reinterpret_cast<const v4f*>(p.pre_g + j);
      v4f o;
      if (p.layer_norm) {
        const v4f b = p.ln_b ? *reinterpret_cast<const v4f*>(p.ln_b + j)
                             : v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < 4; c++) o[c] = (v[e][c] - mean) * inv * g[c] + b[c];
      } else {
#pragma unroll
        for (int c = 0; c < 4; c++) o[c] = v[e][c] * inv * g[c];
      }
      v[e] = o;
      if (p.out) *reinterpret_cast<v4f*>(p.out + (size_t)row * H + j) = o;
      if (p.ph) store_planes4(p.ph, p.pl, (size_t)row * p.ldp + j, o);
      mx = fmaxf(mx, fmaxf(fmaxf(fabsf(o[0]), fabsf(o[1])), fmaxf(fabsf(o[2]), fabsf(o[3]))));
    }
  }
  if (p.qa) {  // QuantizeRowU8 (pack_vnni.go:85-117) of the normalized row
    mx = wave_max(mx);
    float scale = mx / 127.0f;
    if (scale == 0.0f) scale = 1.0f;
    const float qinv = 1.0f / scale;
    uint8_t* q = p.qa + (size_t)row * p.ldq;
#pragma unroll
    for (int e = 0; e < V; e++) {
      const int j = (lane + 64 * e) * 4;
      if (j < H)
        *reinterpret_cast<uint32_t*>(q + j) =
            (uint32_t)qbyte(v[e][0], qinv) | ((uint32_t)qbyte(v[e][1], qinv) << 8) |
            ((uint32_t)qbyte(v[e][2], qinv) << 16) | ((uint32_t)qbyte(v[e][3], qinv) << 24);
    }
    for (int j = H + lane * 4; j < p.ldq; j += 256) *reinterpret_cast<uint32_t*>(q + j) = 0u;
    if (lane == 0) p.row_scales[row] = scale;
  }
}

hipError_t launch_rms_residual(const RmsArgs& a, hipStream_t s) {
  if (a.m <= 0) return hipSuccess;
  if (a.H % 4 || a.H > 4096 || (a.qa && a.ldq % 4) || (a.ph && (a.ldp % 64 || a.ldp < a.H)) ||
      (a.layer_norm && a.post_g))
    return hipErrorInvalidValue;
  const dim3 grid(ceil_div(a.m, kRows)), block(256);
  const int v = ceil_div(a.H, 256);
  if (v <= 1) hipLaunchKernelGGL((rms_residual_kernel<1>), grid, block, 0, s, a);
  else if (v <= 2) hipLaunchKernelGGL((rms_residual_kernel<2>), grid, block, 0, s, a);
  else if (v <= 3) hipLaunchKernelGGL((rms_residual_kernel<3>), grid, block, 0, s, a);
  else if (v <= 4) hipLaunchKernelGGL((rms_residual_kernel<4>), grid, block, 0, s, a);
  else if (v <= 8) hipLaunchKernelGGL((rms_residual_kernel<8>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((rms_residual_kernel<16>), grid, block, 0, s, a);
  return hipGetLastError();
}

// ---- QK-norm + RoPE -----------------------------------------------------------------
// Items are (row, head) over the q heads then the k heads of a fused q|k|v
// row: RMSNorm of the head's dh values with its norm weight (none when the
// norm weights are null: nomic and ModernBERT rotate the raw projections,
// nomic.go:210-211, modernbert.go:256-257), then rotate-half RoPE at the
// row's position (applyRoPE, modernbert.go:130-143: each product rounded to
// float32 before the add). The results go to bf16 rows `outh` of the same layout
// (round to nearest even), and the v heads are converted too: the operands of a
// bf16 attention. With `outl`, outh and outl receive the bf16 hi/lo split of the
// results, the operands of an fp32-grade attention.
// A wave takes kQkItems consecutive items, loading all of them before it
// reduces, so their memory latencies overlap.
constexpr int kQkItems = 4;

__global__ __launch_bounds__(256) void qk_norm_rope_kernel(
    const float* __restrict__ qkv, int ldqkv, int m, int nq, int nkv, int dh,
    const float* __restrict__ q_g, const float* __restrict__ k_g, float eps,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t,
    const int32_t* __restrict__ pos, __bf16* __restrict__ outh, __bf16* __restrict__ outl) {
  const int lane = threadIdx.x & 63;
  const int item0 = (blockIdx.x * kRows + (threadIdx.x >> 6)) * kQkItems;
  const int nh = nq + 2 * nkv;
  const int total = m * nh;
  const int half = dh >> 1;
  // lane holds pairs (d, d + half) for d = lane, lane + 64 (dh <= 256)
  float x1[kQkItems][2], x2[kQkItems][2];
#pragma unroll
  for (int it = 0; it < kQkItems; it++) {
    const int item = min(item0 + it, total - 1);
    const float* v = qkv + (size_t)(item / nh) * ldqkv + (item % nh) * dh;
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int d = lane + 64 * e;
      x1[it][e] = d < half ? v[d] : 0.0f;
      x2[it][e] = d < half ? v[d + half] : 0.0f;
    }
  }
#pragma unroll
  for (int it = 0; it < kQkItems; it++) {
    const int item = item0 + it;
    if (item >= total) return;
    const int row = item / nh, h = item % nh;
    __bf16* o = outh + (size_t)row * ldqkv + h * dh;
    __bf16* ol = outl ? outl + (size_t)row * ldqkv + h * dh : nullptr;
    auto store = [&](int d, float x) {
      __bf16 hi, lo;
      split_hi_lo(x, hi, lo);
      o[d] = hi;
      if (ol) ol[d] = lo;
    };
    if (h >= nq + nkv) {  // v head: conversion only
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int d = lane + 64 * e;
        if (d < half) {
          store(d, x1[it][e]);
          store(d + half, x2[it][e]);
        }
      }
      continue;
    }
    const float* g = h < nq ? q_g : k_g;  // null: no QK-norm, RoPE only
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 2; e++) ss += x1[it][e] * x1[it][e] + x2[it][e] * x2[it][e];
    const float inv = rms_inv(wave_sum(ss), dh, eps);
    const int p = pos[row];
    const float* c = cos_t + (size_t)p * half;
    const float* sn = sin_t + (size_t)p * half;
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int d = lane + 64 * e;
      if (d < half) {
        const float a = g ? x1[it][e] * inv * g[d] : x1[it][e];
        const float b = g ? x2[it][e] * inv * g[d + half] : x2[it][e];
        const float cc = c[d], ssn = sn[d];
        const float t0 = a * cc, t1 = b * ssn, t2 = b * cc, t3 = a * ssn;
        store(d, t0 - t1);
        store(d + half, t2 + t3);
      }
    }
  }
}

// Vector form for dh in {64, 128, 256}: one workgroup per row; a head is
// dh/4 consecutive lanes holding 4 columns each (16-byte loads, 8- or
// 16-byte stores), so a wave covers 64/(dh/4) heads at once. The head's
// sum of squares reduces over its lanes; lane l and l ^ (dh/8) hold the
// RoPE pair (d, d + dh/2). Same per-element operations as the scalar form
// (only the sum of squares is added in another order).
template <int DH>
__global__ __launch_bounds__(256) void qk_norm_rope_vec_kernel(
    const float* __restrict__ qkv, int ldqkv, int nq, int nkv, const float* __restrict__ q_g,
    const float* __restrict__ k_g, float eps, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, const int32_t* __restrict__ pos,
    __bf16* __restrict__ outh, __bf16* __restrict__ outl) {
  constexpr int LPH = DH / 4;    // lanes per head
  constexpr int HPW = 64 / LPH;  // heads per wave
  constexpr int HALF = DH / 2;
  constexpr int IT = 4;          // passes whose loads are issued together
  const int row = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l = lane % LPH, d = l * 4;
  const int nh = nq + 2 * nkv;
  const float* rowp = qkv + (size_t)row * ldqkv;
  const int p = pos[row];
  for (int base = 0; base < nh; base += IT * 4 * HPW) {
    v4f x[IT];
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int h = base + (it * 4 + wave) * HPW + lane / LPH;
      x[it] = h < nh ? *reinterpret_cast<const v4f*>(rowp + h * DH + d)
                     : v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int h0 = base + (it * 4 + wave) * HPW;  // first head of this wave's pass
      if (h0 >= nh) break;
      const int h = h0 + lane / LPH;
      const size_t off = (size_t)row * ldqkv + h * DH + d;
      float ss = (x[it][0] * x[it][0] + x[it][1] * x[it][1]) +
                 (x[it][2] * x[it][2] + x[it][3] * x[it][3]);
#pragma unroll
      for (int o = LPH / 2; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
      if (h >= nh) continue;
      if (h >= nq + nkv) {  // v head: conversion only
        store_planes4(outh, outl, off, x[it]);
        continue;
      }
      const float inv = rms_inv(ss, DH, eps);
      const float* gp = h < nq ? q_g : k_g;  // null: no QK-norm, RoPE only
      v4f xn, pn;
      if (gp) {
        const v4f g = *reinterpret_cast<const v4f*>(gp + d);
#pragma unroll
        for (int c = 0; c < 4; c++) xn[c] = x[it][c] * inv * g[c];
      } else {
        xn = x[it];
      }
#pragma unroll
      for (int c = 0; c < 4; c++) pn[c] = __shfl_xor(xn[c], LPH / 2, 64);
      const bool first = l < LPH / 2;  // columns d < dh/2
      const int dp = first ? d : d - HALF;
      const v4f cc = *reinterpret_cast<const v4f*>(cos_t + (size_t)p * HALF + dp);
      const v4f sn = *reinterpret_cast<const v4f*>(sin_t + (size_t)p * HALF + dp);
      v4f o;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const float a = first ? xn[c] : pn[c], b = first ? pn[c] : xn[c];
        o[c] = first ? a * cc[c] - b * sn[c] : b * cc[c] + a * sn[c];
      }
      store_planes4(outh, outl, off, o);
    }
  }
}

hipError_t launch_qk_norm_rope(const float* qkv, int ldqkv, int m, int nq, int nkv, int dh,
                               const float* q_g, const float* k_g, float eps,
                               const float* cos_t, const float* sin_t,
                               const int32_t* pos, __bf16* outh, __bf16* outl, hipStream_t s) {
  if (m <= 0) return hipSuccess;
  if (dh % 2 || dh > 256 || !outh) return hipErrorInvalidValue;
  const bool vec = ldqkv % 4 == 0 && ((reinterpret_cast<uintptr_t>(qkv) & 15) == 0) &&
                   ((reinterpret_cast<uintptr_t>(outh) & 7) == 0) &&
                   ((reinterpret_cast<uintptr_t>(outl) & 7) == 0);
  if (vec && (dh == 64 || dh == 128 || dh == 256)) {
    if (dh == 64)
      hipLaunchKernelGGL((qk_norm_rope_vec_kernel<64>), dim3(m), dim3(256), 0, s, qkv, ldqkv, nq,
                         nkv, q_g, k_g, eps, cos_t, sin_t, pos, outh, outl);
    else if (dh == 128)
      hipLaunchKernelGGL((qk_norm_rope_vec_kernel<128>), dim3(m), dim3(256), 0, s, qkv, ldqkv,
                         nq, nkv, q_g, k_g, eps, cos_t, sin_t, pos, outh, outl);
    else
      hipLaunchKernelGGL((qk_norm_rope_vec_kernel<256>), dim3(m), dim3(256), 0, s, qkv, ldqkv,
                         nq, nkv, q_g, k_g, eps, cos_t, sin_t, pos, outh, outl);
    return hipGetLastError();
  }
  const int items = m * (nq + 2 * nkv);
  hipLaunchKernelGGL(qk_norm_rope_kernel, dim3(ceil_div(items, kRows * kQkItems)), dim3(256), 0,
                     s, qkv, ldqkv, m, nq, nkv, dh, q_g, k_g, eps, cos_t, sin_t, pos, outh, outl);
  return hipGetLastError();
}

// ---- EmbeddingGemma Dense head --------------------------------------------------------
// applyGemmaDenseHead (gemma3.go:174-198): hid[o] = sum_i w1[o][i] * pooled[i],
// out[o] = sum_i w2[o][i] * hid[i], each a sequential float32 sum in ascending
// i (no FMA) over transposed weights (wT[i][o]). A workgroup takes 32 outputs of
// 8 texts: 128 rows of its weight columns at a time go through LDS (ColChunk)
// with the texts' inputs, and half-wave h adds text h's products, 4*G at a time.
// Bound by the chain of additions and what a CU pulls of the weights while every
// workgroup has a CU to itself (G = 4), by LDS reads and additions beyond, where
// G = 2 leaves registers for two workgroups per CU (95 against 151). µs for both
// products (768 -> 3072, 3072 -> 768) with a text's 256 outputs per workgroup,
// with 256-row chunks and G = 4 throughout, and now:
//   16 texts 73, 44, 45; 96 texts 110, 111, 76; 1024 texts 734, 837, 512
constexpr int kDenseTexts = 8, kDenseRows = 128;
template <int G>
__global__ __launch_bounds__(512) void dense_matvec_kernel(const float* __restrict__ wT,
                                                           int in, int outn, int batch,
                                                           const float* __restrict__ x,
                                                           float* __restrict__ y) {
  constexpr int kStride = ColChunk<kDenseRows>::kStride;
  __shared__ __attribute__((aligned(16))) float w[2][kColCols * kStride];
  __shared__ __attribute__((aligned(16))) float xs[2][kDenseTexts][kDenseRows];
  const int b0 = blockIdx.y * kDenseTexts, nb = min(kDenseTexts, batch - b0);
  const bool loads = threadIdx.x >= 256;  // waves 4..7
  const int tid = threadIdx.x & 255;
  const int h = tid >> 5;  // text b0 + h
  const int o = blockIdx.x * kColCols + (tid & 31);
  const float* src = wT + min(o, outn - 1);
  const int chunks = (in + kDenseRows - 1) / kDenseRows;
  ColChunk<kDenseRows> ch;
  // the inputs: row tid % 128 of the texts tid / 128, 2 + tid / 128, ...
  constexpr int kTextsEach = kDenseTexts * kDenseRows / 256;
  const int xi = tid % kDenseRows, xt = tid / kDenseRows;
  float xv[kTextsEach];
  auto fetch = [&](int c) {
    const int i = min(c * kDenseRows + xi, in - 1);
#pragma unroll
    for (int t = 0; t < kTextsEach; t++)
      xv[t] = x[(size_t)(b0 + min(2 * t + xt, nb - 1)) * in + i];
    ch.fetch(src, outn, c * kDenseRows, in);
  };
  auto stash = [&](int c) {
    const int n = in - c * kDenseRows;
    ch.stash(w[c & 1], n);
#pragma unroll
    for (int t = 0; t < kTextsEach; t++) xs[c & 1][2 * t + xt][xi] = xi < n ? xv[t] : 0.0f;
  };
  if (loads) {
    fetch(0);
    stash(0);
    if (chunks > 1) fetch(1);
  }
  float acc = 0.0f;
  for (int c = 0; c < chunks; c++) {
    __syncthreads();  // chunk c is in LDS, and chunk c - 1 has been read
    if (loads) {
      if (c + 1 < chunks) stash(c + 1);
      if (c + 2 < chunks) fetch(c + 2);
    } else if (h < nb) {
      const float* pw = w[c & 1] + (tid & 31) * kStride;
      const float* px = xs[c & 1][h];
      // whole groups of 4*G, a group read under the additions of the one before;
      // products past `in` are zeros, which change no sum
      const int n = min(kDenseRows, in - c * kDenseRows);
      v4f a[2][G], v[2][G];
      auto read = [&](int g, int i) {
#pragma unroll
        for (int q = 0; q < G; q++) {
          a[g][q] = *reinterpret_cast<const v4f*>(pw + i + 4 * q);
          v[g][q] = *reinterpret_cast<const v4f*>(px + i + 4 * q);
        }
      };
      auto add = [&](int g) {
#pragma unroll
        for (int q = 0; q < G; q++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc = acc + a[g][q][e] * v[g][q][e];
      };
      read(0, 0);
      for (int i = 0; i < n; i += 8 * G) {
        read(1, i + 4 * G);  // at most the chunk's last group
        add(0);
        if (i + 8 * G < n) read(0, i + 8 * G);
        if (i + 4 * G < n) add(1);
      }
    }
  }
  if (!loads && h < nb && o < outn) y[(size_t)(b0 + h) * outn + o] = acc;
}

static void launch_dense(const float* wT, int in, int outn, int batch, const float* x, float* y,
                         hipStream_t s) {
  const dim3 grid(ceil_div(outn, kColCols), ceil_div(batch, kDenseTexts));
  if ((long long)grid.x * grid.y <= 256)
    hipLaunchKernelGGL((dense_matvec_kernel<4>), grid, dim3(512), 0, s, wT, in, outn, batch, x, y);
  else
    hipLaunchKernelGGL((dense_matvec_kernel<2>), grid, dim3(512), 0, s, wT, in, outn, batch, x, y);
}

hipError_t launch_dense_head(const float* pooled, int batch, int H, int D, const float* w1T,
                             const float* w2T, int normalize, float* hid, float* out,
                             hipStream_t s) {
  if (batch <= 0) return hipSuccess;
  launch_dense(w1T, H, D, batch, pooled, hid, s);
  launch_dense(w2T, D, H, batch, hid, out, s);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && normalize) e = launch_l2_rows(out, batch, H, s);
  return e;
}

// Gated-MLP glue over separate gate and up rows (qwen3.go:530-539,
// gemma3.go:365-374): out = act(gate) * up element by element, with the same
// float32 glu_act the fused gated epilogues apply, so the result equals the
// fused form bit for bit. Used when newDense packed gate and up in different
// modes. out may alias gate.
__global__ void glu_rows_kernel(const float* gate, const float* up, float* out, size_t n,
                                int act) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = glu_act(gate[i], up[i], act);
}

hipError_t launch_glu_rows(const float* gate, const float* up, float* out, size_t n, int act,
                           hipStream_t s) {
  if (n == 0) return hipSuccess;
  if (!is_glu(act)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(glu_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, gate,
                     up, out, n, act);
  return hipGetLastError();
}

}  // namespace rh
