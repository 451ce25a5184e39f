// bf16 window + summary attention for windows of up to 128 tokens with every key of a unit in one
// softmax (head_dim 64, 128 or 256): what the windows of 65..128 tokens run on.
//
// Semantics and work unit as page_attn.h: (batch, kv head, HW * NH of its query heads, 64 consecutive
// query positions).  The unit's keys are 192 window rows (positions 64 c - 128 .. 64 c + 63) and a
// 16-slot tile of routed summaries.  Two phases share one LDS buffer of 208 rows:
//   * K staged; each wave (16 query rows, HW heads) scores its nine window tiles and the summary tile
//     (S^T = K Q^T, one K fragment read for the wave's heads), one maximum and one sum per row in fp32
//     registers, P = hi + mid + lo exactly in three bf16 parts;
//   * V, requested with K and held in registers until every wave is done with K, staged in the same
//     rows; O^T = V^T P^T tile by tile (one V fragment read for HW heads times three parts), stored as
//     each 64 columns are done.
// No running softmax: one maximum per row and chunk, no rescaling, and no output accumulators held
// across the keys (page_attn_kernel holds D / 4 registers a head and runs 7 barriers a unit; 3 here).
// The buffer is 110 KB at d = 256 (one workgroup of 512 threads per CU), 57 KB at d = 128 and 29 KB at
// d = 64 (workgroups of 256 threads and two heads, two per CU by registers).
//
// An infinity or NaN in V: its rows are flagged when V is staged; a unit with any takes fragments with
// such elements zeroed and adds them afterwards to the rows that attend to them.
//
// What bounds it: the chain request, scores, softmax, V, store within a workgroup (two of them per CU at
// d = 128), with the VALU about 36% and the matrix cores about 25% busy.  2 x 10007 tokens, 16/4 heads of d 128,
// W 128, with the compressor's 8 us: 82 us a call (40 by bytes); 20011 tokens of d 256 streamed in chunks of 512:
// 306.  With P in two parts, 17 of its 24 bits: 78 and 288 here, 109 and 407 on page_attn_kernel.
#pragma once

#include "page_attn.h"

namespace bfly {

constexpr int kWinMax = 128;                  // window
constexpr int kWinRows = 192;                 // staged window rows
constexpr int kWinSlots = 16;                 // summary slots
constexpr int kWinAll = kWinRows + kWinSlots;

// max(a, b, c) in one instruction (fmaxf first quiets each operand that may be a signalling NaN)
__device__ __forceinline__ float win_max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// The larger of `m`'s halves and those of a piece's bf16 without their signs, half by half.
__device__ __forceinline__ unsigned win_magnitude(unsigned m, page_u32x4 x) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  u16x2 r = __builtin_bit_cast(u16x2, m);
#pragma unroll
  for (int i = 0; i < 4; ++i) r = __builtin_elementwise_max(r, __builtin_bit_cast(u16x2, x[i] & 0x7fff7fffu));
  return __builtin_bit_cast(unsigned, r);
}

template <int D, int HW, int NH, int MODE, bool kBatch = false>
__global__ void __launch_bounds__(256 * NH, 2)
win_attn_kernel(PageArgs a_in, std::conditional_t<kBatch, PageBatch, PageNoBatch> cb) {
  PageArgs a = a_in;
  constexpr int NTHR = 256 * NH, KP = D + 8, KSTEPS = D / 32, PIECES = D / 8, MT = D / 32;
  constexpr int RSTEP = NTHR / PIECES;                       // rows between a thread's pieces
  constexpr int LD = (kWinAll + RSTEP - 1) / RSTEP;          // K (and V) pieces per thread
  constexpr int NT = MODE == kPageSwa ? 9 : 10;              // key tiles of a wave: 9 window, the summaries
  static_assert(MODE == kPageFused || MODE == kPageSwa, "window modes");
  static_assert(!kBatch || MODE == kPageFused, "batches are the streaming loop's");
  static_assert(64 % RSTEP == 0 && RSTEP >= kWinSlots && LD * RSTEP >= kWinAll && (LD - 1) * RSTEP == kWinRows,
                "a round of pieces lies in one page, the summary slots in the last");
  __shared__ __attribute__((aligned(16))) unsigned char smem[kWinAll * KP * 2];
  __shared__ int s_n[kWinSlots], s_b[kWinSlots];
  __shared__ int s_bad[kWinAll + 1];                         // rows of V with an infinity or NaN, and whether any
  __bf16* Ks = reinterpret_cast<__bf16*>(smem);              // [kWinAll][KP], then V [kWinAll][D] swizzled
  if constexpr (kBatch) {
    static_assert(sizeof(smem) >= NH * 256 * 8 * 4, "pooling scratch aliases the staging rows");
    if ((int)blockIdx.x >= cb.attn_blocks) {
      page_update<NH>(cb, reinterpret_cast<float*>(smem));
      return;
    }
  }
  int row, chunk, zc;
  if (!page_unit<kBatch>(a, cb, row, chunk, zc)) return;
  const int bh = row / a.nparts, hpart = row - bh * a.nparts;
  const int bi = bh / a.hkv, kvh = bh - bi * a.hkv;
  const int gsz = a.hq / a.hkv;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lg = lane >> 4, lq = lane & 15;
  const int qwave = wave & 3;
  const int h0 = (hpart * NH + (wave >> 2)) * HW;      // the wave's first head in the group

  const int pw = chunk * kPageRows + qwave * 16;
  const int qp = pw + lq;                               // this lane's query position (column lq)
  const bool row_ok = qp >= a.qlo && qp < a.qhi;
  const bool wave_on = pw + 15 >= a.qlo && pw < a.qhi && h0 < gsz;
  auto blk_of = [&](int p) { return min(max(p / a.bs, 0), a.nblocks - 1); };
  const int qblk = MODE == kPageSwa ? 0 : blk_of(qp);
  const float sl2 = a.scale * 1.4426950408889634f;      // > 0 (the host's rule)

  // ---- requests: Q, then every K row, then every V row
  bf16x8 qf[HW][KSTEPS];
  const int64_t qhead0 = ((int64_t)bi * a.hq + (int64_t)kvh * gsz) * a.tq;
  const int qrow = row_ok ? qp - a.qlo : 0;
#pragma unroll
  for (int u = 0; u < HW; ++u) {
    const __bf16* qs = reinterpret_cast<const __bf16*>(a.q) +
                       (qhead0 + (int64_t)min(h0 + u, gsz - 1) * a.tq + qrow) * D + lg * (D / 4);
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) qf[u][ks] = *reinterpret_cast<const bf16x8*>(qs + 8 * ks);
  }
  const int p_lo = chunk * kPageRows - 128;             // position of LDS row 0
  const int last = a.kv_len - 1, key0 = max(a.key_lo, 0);
  const __bf16* kb = reinterpret_cast<const __bf16*>(a.k) + (int64_t)bh * a.kv_rows * D;
  const __bf16* vb = reinterpret_cast<const __bf16*>(a.v) + (int64_t)bh * a.kv_rows * D;
  page_u32x4 kst[LD], vst[LD];
  // thread: piece pc of rows r0, r0 + RSTEP, ...; the window rows are three pages of 64
  constexpr int RPP = 64 / RSTEP;                       // rounds per page
  const int pc = tid % PIECES, r0 = tid / PIECES;
  const unsigned voff = (unsigned)(r0 * D + pc * 8);
  // Page g's rows, K or V (kv): a page whose 64 positions all exist and lie in one run of rows is read at
  // uniform addresses plus voff.  In any other, a position that does not exist reads the nearest one
  // that does (masked; its V is finite or flagged like any other), each row found by itself.
  struct Run {
    const __bf16 *k, *v;
    bool whole;
  } run[3];
#pragma unroll
  for (int g = 0; g < 3; ++g) {
    const int p0 = p_lo + 64 * g;
    const __bf16 *kx = kb, *vx = vb;
    int x = p0 - a.key_lo;
    bool whole = p0 >= key0 && p0 + 63 <= last;
    bool ring = a.ring != 0;
    if constexpr (kBatch) {
      if (cb.from_inputs && p0 >= cb.c[0].qlo) {
        // the chunk of the batch that holds the page: this one or one before it
        int zp = zc;
        while (zp > 0 && p0 < cb.c[zp].qlo) --zp;
        const int len = cb.c[zp].tq;
        kx = reinterpret_cast<const __bf16*>(cb.c[zp].k) + (int64_t)bh * len * D;
        vx = reinterpret_cast<const __bf16*>(cb.c[zp].v) + (int64_t)bh * len * D;
        x = p0 - cb.c[zp].qlo;
        ring = false;
      }
    }
    if (ring && whole) {
      x = (int)((unsigned)p0 % (unsigned)a.ring);
      whole = x + 64 <= a.ring;
    }
    run[g].k = whole ? kx + (int64_t)x * D : kx;
    run[g].v = whole ? vx + (int64_t)x * D : vx;
    run[g].whole = whole;
  }
  auto load_pages = [&](int kv, page_u32x4 (&dst)[LD]) {
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      const __bf16* src = kv ? run[g].v : run[g].k;
      if (run[g].whole) {
#pragma unroll
        for (int i = 0; i < RPP; ++i)
          dst[g * RPP + i] = *reinterpret_cast<const page_u32x4*>(src + (unsigned)(i * RSTEP * D) + voff);
      } else {
        const int p0 = p_lo + 64 * g;
        int lo = key0, hi = last, first = a.key_lo, ring = a.ring;
        if constexpr (kBatch) {
          if (cb.from_inputs) {
            if (p0 >= cb.c[0].qlo) {                    // (its chunk ends in the page or past it)
              int zp = zc;
              while (zp > 0 && p0 < cb.c[zp].qlo) --zp;
              first = lo = cb.c[zp].qlo;
              hi = min(last, lo + cb.c[zp].tq - 1);
              ring = 0;
            } else {
              hi = cb.c[0].qlo - 1;                     // the batch's own tokens need not be in the ring
            }
          }
        }
#pragma unroll
        for (int i = 0; i < RPP; ++i) {
          const int p = min(max(p0 + i * RSTEP + r0, lo), hi);
          const int64_t x = ring ? (int64_t)((unsigned)p % (unsigned)ring) : (int64_t)(p - first);
          dst[g * RPP + i] = *reinterpret_cast<const page_u32x4*>(src + x * D + pc * 8);
        }
      }
    }
  };
  const int q_first = max(chunk * kPageRows, a.qlo), q_last = min((chunk + 1) * kPageRows, a.qhi) - 1;
  const int bA = MODE == kPageSwa ? 0 : blk_of(q_first), bB = MODE == kPageSwa ? 0 : blk_of(q_last);
  for (int i = tid; i < kWinAll + 1; i += NTHR) s_bad[i] = 0;
  load_pages(0, kst);
  if constexpr (MODE == kPageFused) page_slots<kBatch>(a, cb, zc, bA, bB, kWinSlots, s_n, s_b);
  load_pages(1, vst);
  __syncthreads();   // the summary slots
  if constexpr (MODE == kPageFused) {
    // (without summaries their tile is masked and its rows are the window buffer's first)
    const __bf16* ks = a.nsum > 0 ? reinterpret_cast<const __bf16*>(a.ks) + (int64_t)bh * a.pool_rows * D : kb;
    const __bf16* vs = a.nsum > 0 ? reinterpret_cast<const __bf16*>(a.vs) + (int64_t)bh * a.pool_rows * D : vb;
    const int64_t off = (int64_t)max(s_n[r0 & (kWinSlots - 1)], 0) * D + pc * 8;
    kst[LD - 1] = *reinterpret_cast<const page_u32x4*>(ks + off);
    vst[LD - 1] = *reinterpret_cast<const page_u32x4*>(vs + off);
  }
  // rows staged (the last round of d = 64 runs past the summary slots)
  auto staged = [&](int j) { return (j + 1) * RSTEP <= kWinRows || (MODE == kPageFused && r0 + j * RSTEP < kWinAll); };
#pragma unroll
  for (int j = 0; j < LD; ++j)
    if (staged(j)) *reinterpret_cast<page_u32x4*>(Ks + (r0 + j * RSTEP) * KP + pc * 8) = kst[j];
  __syncthreads();   // K staged

  // ---- scores and softmax: key 4 lg + i of tile t (window tiles: positions pw - 128 + 16 t .., rows
  // 16 (qwave + t) ..; tile 9: the summary slots)
  bf16x8 hi[HW][5], mid[HW][5], lo[HW][5];
  float inv[HW];
  const int wlo = max(max(qp - a.W + 1, a.key_lo), 0);
  const int qcut = max(0, (a.token_cutoff ? qp : qblk * a.bs) - a.W + 1);
  auto sum_ok = [&](int s) {
    const int n = s_n[s];
    return n >= 0 && s_b[s] == qblk && (n + 1) * a.bs <= qcut;
  };
  if (wave_on) {
    f32x4 s[HW][10];
    const __bf16* kl = Ks + (16 * qwave + lq) * KP + lg * (D / 4);
    const __bf16* kq = Ks + (kWinRows + lq) * KP + lg * (D / 4);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      bf16x8 kf[KSTEPS];
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks)
        kf[ks] = *reinterpret_cast<const bf16x8*>((t < 9 ? kl + 16 * t * KP : kq) + 8 * ks);
#pragma unroll
      for (int u = 0; u < HW; ++u) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], qf[u][ks], acc, 0, 0, 0);
        s[u][t] = acc;
      }
    }
    // window keys [wlo, qp] as offsets from this lane group's first key of tile 0; tiles before pw hold no
    // key above the queries, and those from the 16 rows' highest lower end on need no mask
    const int off = pw - 128 + 4 * lg, klo = wlo - off, khi = min(qp, last) - off;
    const int full = max(max(pw + 15 - a.W + 1, a.key_lo), 0) - (pw - 128);
#pragma unroll
    for (int t = 0; t < 8; ++t)
      if (16 * t < full) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int u = 0; u < HW; ++u) s[u][t][i] = 16 * t + i >= klo ? s[u][t][i] : -INFINITY;
      }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool own = 128 + i >= klo && 128 + i <= khi;
      const bool sum = MODE == kPageFused && sum_ok(4 * lg + i);
#pragma unroll
      for (int u = 0; u < HW; ++u) {
        s[u][8][i] = own ? s[u][8][i] : -INFINITY;
        if (MODE == kPageFused) s[u][9][i] = sum ? s[u][9][i] : -INFINITY;
      }
    }
#pragma unroll
    for (int u = 0; u < HW; ++u) {
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < NT; ++t) mx = win_max3(win_max3(mx, s[u][t][0], s[u][t][1]), s[u][t][2], s[u][t][3]);
      mx = col_max4(mx);
      const float nm = mx == -INFINITY ? 0.f : -mx * sl2;
      float l = 0.f;
#pragma unroll
      for (int pr = 0; pr < 5; ++pr) {
        Parts4 x[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
          const int t = 2 * pr + tt;
          f32x4 e = {0.f, 0.f, 0.f, 0.f};
          if (t < NT) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              e[i] = __builtin_amdgcn_exp2f(fmaf(s[u][t][i], sl2, nm));
              l += e[i];
            }
          }
          x[tt] = split_parts(e);
        }
        hi[u][pr] = join8(x[0].h, x[1].h);
        mid[u][pr] = join8(x[0].m, x[1].m);
        lo[u][pr] = join8(x[0].l, x[1].l);
        __builtin_amdgcn_sched_barrier(0);      // two tiles at a time: the parts take the scores' registers
      }
      l = col_sum4(l);
      if constexpr (MODE == kPageFused) {
        inv[u] = 1.f / fmaxf(l, 1e-30f);
        // every window score -inf (or NaN): 0 / 0, as one softmax over the row's keys gives
        if (mx == -INFINITY && wlo <= min(qp, last)) inv[u] = NAN;
      } else {
        const bool any = mx != -INFINITY;
        inv[u] = any ? 1.f / l : 0.f;
        if (lg == 0 && row_ok && h0 + u < gsz) {
          const int64_t r = qhead0 + (int64_t)(h0 + u) * a.tq + (qp - a.qlo);
          a.l[r] = any ? l : 0.f;
          a.m[r] = any ? mx * a.scale : kPageNeg;
        }
      }
    }
  }
  __syncthreads();   // every wave is done with K
  __bf16* Vs = Ks;
  unsigned worst = 0;      // per half: the largest magnitude
#pragma unroll
  for (int j = 0; j < LD; ++j)
    if (staged(j)) {
      const int r = r0 + j * RSTEP;
      *reinterpret_cast<page_u32x4*>(Vs + r * D + (pc ^ vrow_swizzle<D>(r)) * 8) = vst[j];
      worst = win_magnitude(worst, vst[j]);
    }
  if (max(worst << 16, worst & 0xffff0000u) >= 0x7f800000u) {
#pragma unroll
    for (int j = 0; j < LD; ++j)
      if (staged(j) && page_nonfinite(vst[j])) s_bad[r0 + j * RSTEP] = s_bad[kWinAll] = 1;
  }
  __syncthreads();   // V staged
  if (!wave_on) return;
  const bool bad = s_bad[kWinAll] != 0;

  // ---- O^T = V^T P^T.  V fragments (transposing reads): row 4 lg + (lq >> 2) of a tile, 8-byte unit
  // mt * 8 + (lq & 3) * 2 + half XOR the row's swizzle, which is this lane's alone
  const int xs = D == 64 ? (lq >> 3) & 1 : (lq >> 2) & 3;
  const __bf16* vrow = Vs + (4 * lg + (lq >> 2)) * D;
  const int vcol = (lq & 3) * 8;
  const bool lo8 = lq < 8;
  const int pA = pw + (lq & 7), pB = pA + 8;
  const bool okA = pA >= a.qlo && pA < a.qhi, okB = pB >= a.qlo && pB < a.qhi;
  __bf16* ob = reinterpret_cast<__bf16*>(a.out) + (qhead0 + (int64_t)h0 * a.tq) * D;
  const int64_t hstride = (int64_t)a.tq * D;
  const int64_t oA = (int64_t)(okA ? pA - a.qlo : 0) * D, oB = (int64_t)(okB ? pB - a.qlo : 0) * D;
  auto finite = [](bf16x4 x) {      // infinities and NaN as zeros
    typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
    u16x4 b = __builtin_bit_cast(u16x4, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = (b[e] & 0x7f80) == 0x7f80 ? 0 : b[e];
    return __builtin_bit_cast(bf16x4, b);
  };
  // output tiles mt = 2 mp, 2 mp + 1: one 128-byte line per position
  auto columns = [&](int mp, auto has_bad) {
    constexpr bool kBad = decltype(has_bad)::value;
    bf16x8 w[HW][2];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int mt = 2 * mp + sub;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        f32x4 o[HW];
#pragma unroll
        for (int u = 0; u < HW; ++u) o[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        const __bf16* vp = vrow + (mt ^ xs) * 32 + vcol + half * 4;
#pragma unroll
        for (int pr = 0; pr < 5; ++pr) {
          bf16x4 va = read_tr(vp + 16 * (qwave + 2 * pr) * D);
          bf16x4 vc = {};
          if (pr < 4) vc = read_tr(vp + 16 * (qwave + 2 * pr + 1) * D);
          else if (MODE == kPageFused) vc = read_tr(vp + kWinRows * D);
          if constexpr (kBad) {
            va = finite(va);
            vc = finite(vc);
          }
          const bf16x8 vf = __builtin_shufflevector(va, vc, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
          for (int u = 0; u < HW; ++u) {
            o[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, hi[u][pr], o[u], 0, 0, 0);
            o[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, mid[u][pr], o[u], 0, 0, 0);
            o[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, lo[u][pr], o[u], 0, 0, 0);
          }
        }
        if constexpr (kBad) {
          // flagged rows one by one: this lane's 4 d of the rows that its query attends to
#pragma unroll 1
          for (int r = 0; r < kWinAll; ++r) {
            if (!s_bad[r]) continue;
            const int rel = r < kWinRows ? r - 16 * qwave : 144 + r - kWinRows;   // row of the wave's ten tiles
            if (rel < 0 || (r < kWinRows && rel >= 144)) continue;
            const bool take = r < kWinRows ? p_lo + r >= wlo && p_lo + r <= min(qp, last) : sum_ok(r - kWinRows);
            const int src = lq + 16 * ((rel >> 2) & 3), pick = (rel >> 4) * 4 + (rel & 3);
            const int unit = mt * 8 + lg * 2 + half;
            const bf16x4 x = *reinterpret_cast<const bf16x4*>(Vs + r * D + (unit ^ (2 * vrow_swizzle<D>(r))) * 4);
#pragma unroll
            for (int u = 0; u < HW; ++u) {
              // (times an infinity or NaN: the high part of the weight says all that its value does)
              unsigned word = 0;
#pragma unroll
              for (int w32 = 0; w32 < 20; ++w32)
                word = pick >> 1 == w32 ? __builtin_bit_cast(page_u32x4, hi[u][w32 / 4])[w32 % 4] : word;
              float p = __uint_as_float(pick & 1 ? word & 0xffff0000u : word << 16);
              p = __shfl(p, src);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float xv = (float)x[e];
                if (take && !(fabsf(xv) < INFINITY)) o[u][e] = fmaf(p, xv, o[u][e]);
              }
            }
          }
        }
#pragma unroll
        for (int u = 0; u < HW; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) w[u][sub][4 * half + i] = (__bf16)(o[u][i] * inv[u]);
      }
    }
    // lanes lq and lq ^ 8 swap a 16-byte piece so that each store writes 8 whole lines
    const int dA = (2 * mp + (lo8 ? 0 : 1)) * 32 + lg * 8;
#pragma unroll
    for (int u = 0; u < HW; ++u) {
      if (h0 + u >= gsz) continue;
      const bf16x8 x = page_xchg8(lo8 ? w[u][1] : w[u][0]);
      const bf16x8 sa = lo8 ? w[u][0] : x, sb = lo8 ? x : w[u][1];
      if (okA) __builtin_nontemporal_store(sa, reinterpret_cast<bf16x8*>(ob + u * hstride + oA + dA));
      if (okB) __builtin_nontemporal_store(sb, reinterpret_cast<bf16x8*>(ob + u * hstride + oB + dA));
    }
  };
  if (!bad) {
#pragma unroll
    for (int mp = 0; mp < MT / 2; ++mp) columns(mp, std::false_type{});
  } else {
#pragma unroll 1
    for (int mp = 0; mp < MT / 2; ++mp) columns(mp, std::true_type{});
  }
}

// Whether win_attn_kernel takes a launch that page_attn_kernel takes: 64 < W <= 128 (a shorter window
// wastes most of its nine tiles), summaries in one tile, rows to stand in for those that do not
// exist.
static inline bool win_path(int64_t W, int64_t slots, float scale, int64_t key_lo, int64_t kv_len) {
  return W > 64 && W <= kWinMax && slots <= kWinSlots && scale > 0.f && key_lo < kv_len;
}

// Whether the grid fills the chip with the split that launch_win_attn takes (two heads per workgroup, or
// the group's one).  Smaller launches leave most CUs idle either way and page_attn_kernel, which starts
// on its first 64 keys, ends sooner: 512 rows over a 32k plain cache, 16/4 heads of d 128, 28.6 us with
// the compressor against 32.4.
static inline bool win_fills(int64_t qlo, int64_t tq, int64_t batch, int hq, int hkv) {
  const int64_t chunks = (qlo + tq - 1) / kPageRows - qlo / kPageRows + 1;
  const int gsz = hq / hkv;
  return chunks * batch * hkv * (gsz > 1 ? (gsz + 1) / 2 : 1) >= 256;
}

template <int MODE>
static inline void launch_win_attn(PageArgs a, int d, hipStream_t stream) {
  a.c_first = a.qlo / kPageRows;
  a.nchunks = (a.qhi - 1) / kPageRows - a.c_first + 1;
  const int gsz = a.hq / a.hkv;
  const int64_t units = (int64_t)a.nchunks * a.batch * a.hkv;
  auto go = [&](auto kernel, int heads, int nh) {
    a.nparts = (gsz + heads - 1) / heads;
    a.items = (int)(units * a.nparts);
    a.per_xcd = (a.items + 7) / 8;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * a.per_xcd)), dim3(256 * nh), 0, stream, a, PageNoBatch{});
  };
  const bool two = gsz >= 2;
  if (d == 256) {
    // four heads a workgroup on whatever grid win_fills lets through: 16/4 heads, window 128, 2100 / 3840 tokens
    // (132 / 240 such workgroups) 28.1 / 30.5 us a call, 35.0 / 38.8 with two heads in twice as many
    if (gsz >= 3) go(win_attn_kernel<256, 2, 2, MODE>, 4, 2);
    else go(win_attn_kernel<256, 1, 2, MODE>, 2, 2);
  } else if (d == 128) {
    if (two) go(win_attn_kernel<128, 2, 1, MODE>, 2, 1);
    else go(win_attn_kernel<128, 1, 1, MODE>, 1, 1);
  } else {
    if (two) go(win_attn_kernel<64, 2, 1, MODE>, 2, 1);
    else go(win_attn_kernel<64, 1, 1, MODE>, 1, 1);
  }
}

}  // namespace bfly
