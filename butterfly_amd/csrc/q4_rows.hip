// Products of 1..32 activation rows with 4-bit affine weights on gfx950 (a batched decode step, a
// short prompt): Y = X W^T from the codes, on the matrix cores.
//
// Reference: the quantized linear layers of the swapped decoder (mlx.nn.QuantizedLinear,
// bna/integrations/qwen_mlx.py:1115-1157); w = code * scale + bias per group of 64 inputs, as
// bfly_q4_gemv reads it.  The product is taken group by group in factorised form,
//   y_mn = sum_g ( scale_ng sum_{i in g} x_mi (16 + code_ni) + (bias_ng - 16 scale_ng) sum_{i in g} x_mi ):
// 16 + code is exact in bf16 (bits 0x4180 | code << 3, one and-or per two codes), so
// v_mfma_f32_16x16x32_bf16 multiplies the codes themselves, the group sums are fp32 and W is never
// expanded or rounded; y is rounded once to bf16.
//
// Weights: lane (lg, lq) of a wave reads the 16 bytes (32 codes) at 16 lg of a 64-byte span (two
// groups) of weight row lq: the MFMA's B operand holds one output row per lane, so a group's scale
// and bias are one word per lane.  v_permlane32_swap then trades the upper lanes' first 8 bytes
// (group g + 1) for the lower lanes' last 8 (group g), so that each register holds codes of one
// group: k-step s of a group is codes q4_first(lg) + 8 s .. + 7.
//
// q4_rows_kernel (a layer's products): R tiles of 16 output rows, by S waves that each take every
// S-th run of 256 inputs (four groups) and add their fp32 parts through LDS; x straight from L2,
// sum x of a group from the same MFMA with ones for codes, in the layout of the products.
// q4_rows_wide_kernel (the lm_head): x is laid out in LDS once per workgroup in fragment order, with
// its group sums, and each wave streams whole tiles, one run of weights ahead.
//
// What bounds it: HBM for large outputs (the weights are read once whatever the row count), launch
// and first-request latency for a layer's small ones.
#include "bfly_common.h"
#include "../../include/butterfly_amd_decoder.h"

namespace bfly {

constexpr int kQ4RowsMax = 32;      // activation rows
constexpr int kQ4RowsQuad = 256;    // inputs of a run: four groups of 64

typedef unsigned int q4_u32x4 __attribute__((ext_vector_type(4)));

// First code (within its group) of lane group lg's k-step 0.
__device__ __forceinline__ int q4_first(int lg) { return ((lg & 1) << 5) | ((lg >> 1) << 4); }

// Words 0, 1 of w become the two k-steps of the span's first group, words 2, 3 the second group's.
__device__ __forceinline__ void q4_split_groups(q4_u32x4& w) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto t = __builtin_amdgcn_permlane32_swap(w[i], w[i + 2], false, false);
    w[i] = t[0];
    w[i + 2] = t[1];
  }
}

// Eight codes of a word as bf16 16 + code, in the order 0 4 1 5 2 6 3 7.
__device__ __forceinline__ bf16x8 q4_codes(uint32_t w) {
  const q4_u32x4 r = {((w << 3) & 0x00780078u) | 0x41804180u, ((w >> 1) & 0x00780078u) | 0x41804180u,
                      ((w >> 5) & 0x00780078u) | 0x41804180u, ((w >> 9) & 0x00780078u) | 0x41804180u};
  return __builtin_bit_cast(bf16x8, r);
}
// Eight consecutive bf16 in that order.
__device__ __forceinline__ bf16x8 q4_order(q4_u32x4 x) {
  const q4_u32x4 r = {__builtin_amdgcn_perm(x[2], x[0], 0x05040100u), __builtin_amdgcn_perm(x[2], x[0], 0x07060302u),
                      __builtin_amdgcn_perm(x[3], x[1], 0x05040100u), __builtin_amdgcn_perm(x[3], x[1], 0x07060302u)};
  return __builtin_bit_cast(bf16x8, r);
}

// SiLU(gate) * up with the rounding points of bfly_silu_mul over the two bf16 outputs.
__device__ __forceinline__ __bf16 q4_rows_silu(float g, float u) {
#pragma clang fp contract(off)
  const float x = (float)(__bf16)g;
  const float sg = (float)(__bf16)(x / (1.f + expf(-x)));
  return (__bf16)(sg * (float)(__bf16)u);
}

// NaN once `z` is one or `v` holds an infinity or NaN, else zero.
__device__ __forceinline__ float q4_watch(float z, f32x4 v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) z = fmaf(v[i], 0.f, z);
  return z;
}

// A tile's products over runs q0, q0 + step, .. with the weights expanded to bf16 (code * scale + bias), as the
// GEMM over `weight` takes them, for those that the factorised form left infinite or NaN: an infinite x gives
// inf - inf there (scale * inf + (bias - 16 scale) * inf), and a finite one above about 1e37 overflows the sum with
// 16 + code.  Looking for them costs a product at most 1%.  x: this lane's activation row, w: its weight row, both from the row's start; every lane calls it.
__device__ __forceinline__ f32x4 q4_expanded(const __bf16* x, const uint8_t* w, const uint32_t* sb, int lg, int q0,
                                             int step, int quads) {
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int q = q0; q < quads; q += step)
#pragma unroll 1
    for (int g = 4 * q; g < 4 * q + 4; ++g) {
      const float scale = __uint_as_float(sb[g] << 16), bias = __uint_as_float(sb[g] & 0xffff0000u);
      const int at = 64 * g + q4_first(lg);      // 16 inputs: this lane's two k-steps
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const uint32_t codes = *reinterpret_cast<const uint32_t*>(w + (at + 8 * c) / 2);
        bf16x8 wf;
#pragma unroll
        for (int e = 0; e < 8; ++e) wf[e] = (__bf16)fmaf((float)((codes >> (4 * e)) & 15u), scale, bias);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(x + at + 8 * c), wf, acc, 0, 0, 0);
      }
    }
  return acc;
}
// `plain` where `v` is an infinity or NaN.
__device__ __forceinline__ f32x4 q4_mend(f32x4 v, f32x4 plain) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = fabsf(v[i]) < INFINITY ? v[i] : plain[i];
  return v;
}

struct Q4RowsArgs {
  const __bf16* x;         // [rows, in_f]
  const uint8_t* w;        // [.., in_f / 2]
  const uint32_t* sb;      // [.., in_f / 64] words: bf16 scale low, bias high
  __bf16* y;               // [rows, n_out]
  int rows, in_f;
  int64_t n_out, up_off;
};

// kSilu: tiles 0 .. R/2 - 1 are gate rows, the others the up rows up_off further.  (MT = 1: at most 128
// registers, for two 512-thread workgroups a CU; with one more, gate|up at 8 rows takes 10.1 us instead of 8.5.)
template <int MT, int R, int S, bool kSilu>
__global__ void __launch_bounds__(64 * S, MT == 1 ? 4 : 2) q4_rows_kernel(Q4RowsArgs a) {
  constexpr int OT = kSilu ? R / 2 : R;
  __shared__ __attribute__((aligned(16))) float part[S][R][MT][64][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lg = lane >> 4, lq = lane & 15;
  const int64_t n0 = (int64_t)blockIdx.x * (16 * OT);
  const int groups = a.in_f / 64, quads = a.in_f / kQ4RowsQuad;

  const uint8_t* wp[R];
  const uint32_t* sp[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t n = n0 + 16 * (r % OT) + lq;      // rows past the end read the last one, never stored
    const int64_t row = (n < a.n_out ? n : a.n_out - 1) + (kSilu && r >= OT ? a.up_off : 0);
    wp[r] = a.w + row * (a.in_f / 2) + 16 * lg;
    sp[r] = a.sb + row * groups;
  }
  const __bf16* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xp[m] = a.x + (int64_t)min(16 * m + lq, a.rows - 1) * a.in_f + q4_first(lg);

  f32x4 acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[r][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const q4_u32x4 one4 = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  const bf16x8 ones = __builtin_bit_cast(bf16x8, one4);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

  q4_u32x4 wv[R][2], sv[R];
  auto load = [&](int q) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // a row's two 64-byte spans are one 128-byte line: requested together, fetched once
#pragma unroll
      for (int j = 0; j < 2; ++j) wv[r][j] = *reinterpret_cast<const q4_u32x4*>(wp[r] + (int64_t)q * 128 + 64 * j);
      sv[r] = *reinterpret_cast<const q4_u32x4*>(sp[r] + 4 * q);
    }
  };
  if (wave < quads) load(wave);
  for (int q = wave; q < quads; q += S) {
    q4_u32x4 wc[R][2], sc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      wc[r][0] = wv[r][0];
      wc[r][1] = wv[r][1];
      sc[r] = sv[r];
    }
    q4_u32x4 xr[MT][4][2];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          xr[m][j][c] = *reinterpret_cast<const q4_u32x4*>(xp[m] + (int64_t)q * kQ4RowsQuad + 64 * j + 8 * c);
    if (q + S < quads) load(q + S);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      q4_split_groups(wc[r][0]);
      q4_split_groups(wc[r][1]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bf16x8 xa[MT][2];
      f32x4 xs[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        xa[m][0] = q4_order(xr[m][j][0]);
        xa[m][1] = q4_order(xr[m][j][1]);
        xs[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[m][0], ones, zero, 0, 0, 0);
        xs[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[m][1], ones, xs[m], 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const bf16x8 c0 = q4_codes(wc[r][j / 2][2 * (j % 2)]), c1 = q4_codes(wc[r][j / 2][2 * (j % 2) + 1]);
        const float scale = __uint_as_float(sc[r][j] << 16), bias = __uint_as_float(sc[r][j] & 0xffff0000u);
        const float b16 = fmaf(-16.f, scale, bias);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          f32x4 t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[m][0], c0, zero, 0, 0, 0);
          t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[m][1], c1, t, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[r][m][i] = fmaf(scale, t[i], fmaf(b16, xs[m][i], acc[r][m][i]));
        }
      }
    }
  }
  float watch = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < MT; ++m) watch = q4_watch(watch, acc[r][m]);
  if (__any(watch != watch)) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[r][m] = q4_mend(acc[r][m], q4_expanded(xp[m] - q4_first(lg), wp[r] - 16 * lg, sp[r], lg, wave, S, quads));
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(part[wave][r][m][lane]) = acc[r][m];
  __syncthreads();
  // lane (lg, lq) of a part holds output row lq of the tile for activation rows 4 lg + i
  auto total = [&](int r, int m, int l, int i) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < S; ++w) s += part[w][r][m][l][i];
    return s;
  };
  for (int o = tid; o < MT * 16 * OT * 16; o += 64 * S) {
    const int nn = o % 16, r = (o / 16) % OT, mi = o / (16 * OT);    // a row's outputs are consecutive
    const int64_t n = n0 + 16 * r + nn;
    if (mi >= a.rows || n >= a.n_out) continue;
    const int l = ((mi % 16) >> 2) * 16 + nn, i = mi & 3, m = mi / 16;
    const float g = total(r, m, l, i);
    if constexpr (kSilu) a.y[(int64_t)mi * a.n_out + n] = q4_rows_silu(g, total(r + OT, m, l, i));
    else a.y[(int64_t)mi * a.n_out + n] = (__bf16)g;
  }
}

// The lm_head's form: at most 16 activation rows, each wave whole tiles of 16 output rows.
// LDS: x fragments [in_f / 64 groups][2 k-steps][64 lanes], then the group sums [groups][16 rows].
// One 1024-thread workgroup per CU: at 8 x 2048 inputs and 151936 outputs (175 MB of weights) 40.5 us
// (4.3 TB/s) on 256 of them, 42.9 on 256 of 512 threads, 44.3 on 512; q4_rows_kernel takes 52.2 at
// its best split (every workgroup reads x from L2 again), a bf16 GEMM over the expanded weights 205.
constexpr int kQ4WideThreads = 1024, kQ4WideGrid = 256;
template <int kInMax>
__global__ void __launch_bounds__(kQ4WideThreads) q4_rows_wide_kernel(Q4RowsArgs a, int tiles) {
  constexpr int kThreads = kQ4WideThreads;
  __shared__ __attribute__((aligned(16))) q4_u32x4 xf[kInMax / 64 * 2 * 64];
  __shared__ __attribute__((aligned(16))) float xsum[kInMax / 64 * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lg = lane >> 4, lq = lane & 15;
  const int groups = a.in_f / 64, quads = a.in_f / kQ4RowsQuad;
  const int nwaves = (int)gridDim.x * (kThreads / 64);
  int tile = (int)blockIdx.x + wave * (int)gridDim.x;   // a workgroup's waves take tiles far apart

  const uint8_t* wp = nullptr;
  const uint32_t* sp = nullptr;
  auto point = [&](int t) {      // rows past the end read the last one, never stored
    const int64_t n = (int64_t)t * 16 + lq, row = n < a.n_out ? n : a.n_out - 1;
    wp = a.w + row * (a.in_f / 2) + 16 * lg;
    sp = a.sb + row * groups;
  };
  q4_u32x4 wv[2], sv;
  auto load = [&](int q) {
    wv[0] = *reinterpret_cast<const q4_u32x4*>(wp + (int64_t)q * 128);
    wv[1] = *reinterpret_cast<const q4_u32x4*>(wp + (int64_t)q * 128 + 64);
    sv = *reinterpret_cast<const q4_u32x4*>(sp + 4 * q);
  };
  point(min(tile, tiles - 1));
  load(0);                       // in flight while x is laid out
  // x: thread t of 64 a group: lane t's two fragments and its part of the row's sum
  for (int g = wave; g < groups; g += kThreads / 64) {
    const q4_u32x4* src = reinterpret_cast<const q4_u32x4*>(a.x + (int64_t)min(lq, a.rows - 1) * a.in_f + 64 * g + q4_first(lg));
    const q4_u32x4 x0 = src[0], x1 = src[1];
    const bf16x8 f0 = q4_order(x0), f1 = q4_order(x1);
    *reinterpret_cast<bf16x8*>(xf + (2 * g) * 64 + lane) = f0;
    *reinterpret_cast<bf16x8*>(xf + (2 * g + 1) * 64 + lane) = f1;
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += (float)f0[e] + (float)f1[e];
    s = col_sum4(s);
    if (lg == 0) xsum[g * 16 + lq] = s;
  }
  __syncthreads();
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // (tile + nwaves stays below 2 * 2^30: the host bounds tiles)
  for (; tile < tiles; tile += nwaves) {
    f32x4 acc = zero;
    const int64_t n = (int64_t)tile * 16 + lq;
    for (int q = 0; q < quads; ++q) {
      q4_u32x4 wc[2] = {wv[0], wv[1]};
      const q4_u32x4 sc = sv;
      if (q + 1 < quads) {
        load(q + 1);
      } else {                   // the next tile's first run
        point(min(tile + nwaves, tiles - 1));
        load(0);
      }
      q4_split_groups(wc[0]);
      q4_split_groups(wc[1]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bf16x8 x0 = __builtin_bit_cast(bf16x8, xf[(2 * (4 * q + j)) * 64 + lane]);
        const bf16x8 x1 = __builtin_bit_cast(bf16x8, xf[(2 * (4 * q + j) + 1) * 64 + lane]);
        const f32x4 xs = *reinterpret_cast<const f32x4*>(xsum + (4 * q + j) * 16 + 4 * lg);
        const float scale = __uint_as_float(sc[j] << 16), bias = __uint_as_float(sc[j] & 0xffff0000u);
        const float b16 = fmaf(-16.f, scale, bias);
        f32x4 t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x0, q4_codes(wc[j / 2][2 * (j % 2)]), zero, 0, 0, 0);
        t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x1, q4_codes(wc[j / 2][2 * (j % 2) + 1]), t, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = fmaf(scale, t[i], fmaf(b16, xs[i], acc[i]));
      }
    }
    const float watch = q4_watch(0.f, acc);
    if (__any(watch != watch)) {
      const int64_t row = n < a.n_out ? n : a.n_out - 1;
      acc = q4_mend(acc, q4_expanded(a.x + (int64_t)min(lq, a.rows - 1) * a.in_f, a.w + row * (a.in_f / 2),
                                     a.sb + row * groups, lg, 0, 1, quads));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * lg + i < a.rows && n < a.n_out) a.y[(int64_t)(4 * lg + i) * a.n_out + n] = (__bf16)acc[i];
  }
}

template <bool kSilu>
static int q4_rows_launch(const void* x, int64_t rows, const void* packed, const void* scale_bias, int64_t n_out,
                          int64_t in_f, int group, int64_t up_off, void* out, hipStream_t stream, const char* what) {
  BFLY_CHECK_ARG(x && packed && scale_bias && out, "null pointer");
  BFLY_CHECK_ARG(rows > 0 && rows <= kQ4RowsMax, "rows=%lld must be in 1..%d", (long long)rows, kQ4RowsMax);
  BFLY_CHECK_ARG(n_out > 0 && in_f > 0 && in_f <= 1 << 20 && in_f % kQ4RowsQuad == 0,
                 "in_features=%lld must be a positive multiple of %d", (long long)in_f, kQ4RowsQuad);
  BFLY_CHECK_ARG(group == 64, "group=%d: groups of 64 only", group);
  BFLY_CHECK_ARG(aligned16(x) && aligned16(packed) && aligned16(scale_bias),
                 "x, packed and scale_bias must be 16-byte aligned");
  BFLY_CHECK_ARG(!kSilu || up_off >= n_out, "up_row_offset=%lld overlaps the gate rows", (long long)up_off);
  Q4RowsArgs a{static_cast<const __bf16*>(x), static_cast<const uint8_t*>(packed),
               static_cast<const uint32_t*>(scale_bias), static_cast<__bf16*>(out), (int)rows, (int)in_f, n_out, up_off};
  auto go = [&](auto kernel, int r, int s) -> int {
    const int tiles = kSilu ? r / 2 : r;
    const int64_t grid = (n_out + 16 * tiles - 1) / (16 * tiles);
    BFLY_CHECK_ARG(grid <= INT32_MAX, "%s: grid too large", what);
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * s), 0, stream, a);
    BFLY_CHECK_LAUNCH(what);
    return BFLY_OK;
  };
  // Splits measured on layers of in x out, 8 / 16 / 32 rows (us; the bf16 GEMM over expanded weights in
  // brackets).  2048 x 3072: one tile on 8 waves 4.66 / 5.20 / 7.13, on 2 waves 5.43 / 5.71 / 7.95, two
  // tiles on 8 waves 5.50 / 6.18 / 8.40 [8.5].  6144 x 2048: 8 waves 7.84 / 9.69 / 15.2, 2 waves
  // 10.6 / 11.6 / 17.2 [12.2, at 32 rows 16.7].  gate|up with SiLU, 2048 x 2 * 6144: a tile pair on 8
  // waves 8.38 / 9.43 / 15.3, on 4 waves 8.65 / 9.70 / 14.3 [18.9, two launches].  2048 x 151936, 32
  // rows: two tiles on 4 waves 100, on 8 waves 137 [150].
  if (rows <= 16) {
    if constexpr (kSilu) {
      return go(q4_rows_kernel<1, 2, 8, true>, 2, 8);
    } else {
      // from 16384 outputs on (2 / 8 / 16 rows, us, weights beyond the caches; this form, then q4_rows_kernel):
      // 2048 x 16384 10.7 / 11.2 / 11.8, 10.0 / 11.5 / 13.6; 2048 x 32768 12.6 / 13.1 / 13.8, 17.9 / 20.5 / 23.6;
      // 512 x 16384 4.5 / 4.7 / 4.9, 5.1 / 5.3 / 5.7; 4096 x 16384 17.3 / 17.8 / 19.2, 14.8 / 17.8 / 22.8
      if (n_out >= 16384 && in_f <= 4096) {
        const int64_t tiles = (n_out + 15) / 16;
        BFLY_CHECK_ARG(tiles <= INT32_MAX / 2, "%s: out_features too large", what);
        hipLaunchKernelGGL(in_f <= 2048 ? q4_rows_wide_kernel<2048> : q4_rows_wide_kernel<4096>, dim3(kQ4WideGrid),
                           dim3(kQ4WideThreads), 0, stream, a, (int)tiles);
        BFLY_CHECK_LAUNCH(what);
        return BFLY_OK;
      }
      return go(q4_rows_kernel<1, 1, 8, false>, 1, 8);
    }
  }
  if constexpr (kSilu) return go(q4_rows_kernel<2, 2, 4, true>, 2, 4);
  else return n_out >= 16384 ? go(q4_rows_kernel<2, 2, 4, false>, 2, 4) : go(q4_rows_kernel<2, 1, 8, false>, 1, 8);
}

}  // namespace bfly

using namespace bfly;

extern "C" int bfly_q4_rows(const void* x, int64_t rows, const void* packed, const void* scale_bias,
                            int64_t out_features, int64_t in_features, int group, void* out, hipStream_t stream) {
  return q4_rows_launch<false>(x, rows, packed, scale_bias, out_features, in_features, group, 0, out, stream,
                               "bfly_q4_rows");
}

extern "C" int bfly_q4_rows_silu(const void* x, int64_t rows, const void* packed, const void* scale_bias,
                                 int64_t out_features, int64_t in_features, int group, int64_t up_row_offset, void* out,
                                 hipStream_t stream) {
  return q4_rows_launch<true>(x, rows, packed, scale_bias, out_features, in_features, group, up_row_offset, out, stream,
                              "bfly_q4_rows_silu");
}
