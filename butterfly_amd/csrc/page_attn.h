// Paged bf16 attention on MFMA with a running softmax: what windows above 64 tokens, blocks
// below 64 tokens and the stream-level entries run on (head_dim 64, 128 or 256).
//
// Reference semantics: butterfly_compressed_attention(_active)
// (bna/torch/attention_wayfinder_permute.py:1046-1197) and the two streams on their own,
// _swa_stream_attention (bna/mlx/attention.py:304-369) and _compressed_stream_attention (:372-516).
//
// Work unit: (batch, kv head, up to HW * NH of its query heads, 64 consecutive query positions).
// Its keys come in pages of 64 rows, each staged once in LDS (K row-major, V row-major with its
// 16-byte pieces swizzled) while the next page's rows are on their way into registers:
//   kFused:  the window's pages from the queries' own one downwards, then one page of routed
//            block summaries (slot s = entry s % kcap of the routed row of the unit's block s / kcap);
//   kSwa:    the window's pages alone;
//   kDense:  the summaries of every earlier block, 64 a page;
//   kRouted: each query block's routed list, 64 entries a page (one query head per unit: the
//            lists are per head).
// 4 NH waves: wave w takes query rows 16 (w % 4) .. + 15 and HW heads.  Keys are taken 32 at a
// time (two 16-row tiles): S^T = K Q^T, running maximum and sum, O^T += V^T P^T, all on
// v_mfma_f32_16x16x32_bf16 with fp32 accumulators.  32-key groups without a key for the wave's 16
// rows are passed over.
//   * P enters the product whole, all 24 bits of its fp32 value, as three bf16 parts P = hi + mid + lo:
//     three MFMAs on one V fragment.
//   * The accumulators are rescaled only when a row's maximum outgrows the reference value by
//     2^8 (P then stays below 2^8, far inside fp32), or at all for a page with a V of 2^100 or more (whose
//     sums would overflow): a rescale is D / 4 multiplications per head.
//   * A page whose V holds an infinity or NaN goes through plain fp32 sums over the keys each row
//     attends to (0 * inf in the matrix product would reach rows that do not attend to it).
//
// What bounds it: VALU (masks, exponentials, splitting P) and LDS fragment reads beside the MFMAs;
// HBM traffic is Q and O once and the K/V pages about once per XCD (consecutive units of one kv
// head share their pages in an L2).  Measured, whole calls: 2 x 10007 tokens, 16/4 heads of d 128,
// W 256 3185 us on the generic kernel, 152 here (141 with P in two parts, 17 of its 24 bits); 512 rows over
// 32k tokens 135 and 28 to 29 (compressor included); window stream, dense summaries and merge over 8192 tokens,
// 8/2 heads 680 and 45.
#pragma once

#include "bfly_topology.h"
#include "cache_update.h"

namespace bfly {

enum PageMode { kPageFused = 0, kPageSwa = 1, kPageDense = 2, kPageRouted = 3 };

constexpr int kPageRows = 64;
constexpr float kPageNeg = -1e30f;     // row maximum of an empty stream row

struct PageArgs {
  const void* q;          // [batch, hq, tq, D]
  const void* k;          // window keys: linear [batch, hkv, kv_rows, D] (row = p - key_lo) or ring
  const void* v;
  const void* ks;         // summaries [batch, hkv, pool_rows, D]
  const void* vs;
  void* out;
  float* l;               // stream modes: row sums and maxima [batch, hq, tq]
  float* m;
  const int32_t* nbr;     // kFused: [nblocks, kcap]; kRouted: [hq, routed_blocks, kcap]
  int64_t kv_rows, pool_rows, routed_blocks;
  int batch, hq, hkv, tq;
  int qlo, qhi;           // query positions [qlo, qhi)
  int key_lo, kv_len;     // window keys are positions [key_lo, kv_len)
  int ring;               // 0, or position p lives at row p mod ring (ring >= 64)
  int nblocks, nsum, kcap, bs, W;
  int token_cutoff;
  float scale;
  // grid: items = chunks x (batch x hkv x head parts), item = (row, chunk), 8 contiguous runs
  int c_first, nchunks, nparts, per_xcd, items;
};

// A batched streaming launch: the attention of up to kMaxUpdateParts consecutive chunks whose
// cache updates are all done, each with the arguments of its own cache state (the counters right
// after its update), so its results are those of a launch of its own.
struct ChunkArgs {
  const void* q;
  void* out;
  const void* k;          // the chunk's own keys and values, [batch x kv heads, tq, d]
  const void* v;
  int tq, qlo, qhi, key_lo, kv_len, nsum, nblocks, c_first, nchunks;
  bfly_topology_t topo;
};
// page_attn_kernel's batch.  Workgroups from attn_blocks on run a cache update instead
// (cache_update_body over upd_x x upd_rows x K|V items, upd_wgs in all, one per 256 threads).
struct PageBatch {
  int nch;
  int from_inputs;        // 1: every chunk starts on a page boundary; pages of the batch's own
                          // tokens come from the chunk inputs (else every page from the ring)
  int attn_blocks, upd_x, upd_rows;
  int64_t upd_wgs;
  UpdateJob upd;
  ChunkArgs c[kMaxUpdateParts];
};
struct PageNoBatch {};

template <int D, int NH>
struct PageCfg {
  static constexpr int NTHR = 256 * NH;
  static constexpr int KP = D + 8;             // bf16 per K row (16-byte pad)
  static constexpr int KSTEPS = D / 32;
  static constexpr int PIECES = D / 8;         // 16-byte pieces per row
  static constexpr int LD = kPageRows * PIECES / NTHR;   // K (and V) pieces per thread per page
  static constexpr int K_BYTES = kPageRows * KP * 2;
  static constexpr int LDS = K_BYTES + kPageRows * D * 2;
};

typedef unsigned int page_u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes from lane ^ 8 of each row of 16 (DPP row_ror:8)
__device__ __forceinline__ bf16x8 page_xchg8(bf16x8 v) {
  page_u32x4 u = __builtin_bit_cast(page_u32x4, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) u[i] = (unsigned)__builtin_amdgcn_mov_dpp((int)u[i], 0x128, 0xf, 0xf, false);
  return __builtin_bit_cast(bf16x8, u);
}

// The largest magnitude of a piece's 8 bf16, its exponent in the upper 8 bits.
__device__ __forceinline__ unsigned page_magnitude(page_u32x4 x) {
  unsigned t = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned a = x[i] << 1, b = x[i] << 17;
    t = max(t, max(a, b));
  }
  return t;
}
// From kPageLarge (2^100) on a V is too large for weights of 2^8; kPageNonfinite: an infinity or NaN.
constexpr unsigned kPageLarge = (127u + 100u) << 24, kPageNonfinite = 0xff000000u;
__device__ __forceinline__ bool page_nonfinite(page_u32x4 x) { return page_magnitude(x) >= kPageNonfinite; }

// The three bf16 parts (bit patterns, two per dword, element 0 in the low half) of four floats: together
// exactly the float, 8 bits of its 24 each.
struct Parts4 {
  uint2 h, m, l;
};
__device__ __forceinline__ Parts4 split_parts(f32x4 x) {
  uint32_t hb[4], mb[4], lb[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hb[i] = __float_as_uint(x[i]) & 0xffff0000u;
    const float rest = x[i] - __uint_as_float(hb[i]);          // exact
    mb[i] = __float_as_uint(rest) & 0xffff0000u;
    lb[i] = __float_as_uint(rest - __uint_as_float(mb[i]));     // exact, low 16 bits zero
  }
  auto pk = [](uint32_t e0, uint32_t e1) { return (e0 >> 16) | (e1 & 0xffff0000u); };
  return {{pk(hb[0], hb[1]), pk(hb[2], hb[3])}, {pk(mb[0], mb[1]), pk(mb[2], mb[3])},
          {pk(lb[0], lb[1]), pk(lb[2], lb[3])}};
}
__device__ __forceinline__ bf16x8 join8(uint2 a, uint2 b) {
  return __builtin_bit_cast(bf16x8, uint4{a.x, a.y, b.x, b.y});
}

// This workgroup's (row, 64-position chunk) item, and in a batch its chunk's arguments put into `a` and its
// index into zc; false for a workgroup past the items.  Workgroups go round-robin over the 8 XCDs: XCD x
// takes items x per_xcd .. , whose consecutive chunks share pages in its L2.
template <bool kBatch>
__device__ __forceinline__ bool page_unit(PageArgs& a, const std::conditional_t<kBatch, PageBatch, PageNoBatch>& cb,
                                          int& row, int& chunk, int& zc) {
  const int item = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
  if (item >= a.items) return false;   // the whole workgroup
  row = item / a.nchunks;
  chunk = a.c_first + item - row * a.nchunks;
  zc = 0;
  if constexpr (kBatch) {
    // item = (row, chunk of the batch, 64 positions): a.nchunks is the longest chunk's
    const int c64 = item - row * a.nchunks;
    zc = row % cb.nch;
    row /= cb.nch;
    const ChunkArgs& ck = cb.c[zc];
    if (c64 >= ck.nchunks) return false;
    chunk = ck.c_first + c64;
    a.q = ck.q;
    a.out = ck.out;
    a.tq = ck.tq;
    a.qlo = ck.qlo;
    a.qhi = ck.qhi;
    a.key_lo = ck.key_lo;
    a.kv_len = ck.kv_len;
    a.nsum = ck.nsum;
    a.nblocks = ck.nblocks;
  }
  return true;
}

// A batch's update work of this workgroup (blockIdx.x >= attn_blocks); `part`: 256 * 8 floats of LDS per
// 256 threads.  A group of 256 threads whose item is past the end exits (it no longer counts at a barrier).
template <int NH>
__device__ __forceinline__ void page_update(const PageBatch& cb, float* part) {
  const int grp = (int)threadIdx.x >> 8;
  const int64_t lin = (int64_t)((int)blockIdx.x - cb.attn_blocks) * NH + grp;
  if (lin >= cb.upd_wgs) return;
  const int64_t per_kv = (int64_t)cb.upd_x * cb.upd_rows;
  const int kv = (int)(lin / per_kv);
  const int64_t r = lin - kv * per_kv, urow = r / cb.upd_x;
  cache_update_body<__bf16, 8>(cb.upd, r - urow * cb.upd_x, urow, kv, part + grp * 256 * 8, (int)threadIdx.x & 255);
}

// The batch chunk that holds the page of positions p0 .. (it lies in one), by selects over the slots
// (uniform): its keys and values [batch x kv heads, len, d], the first of them position lo.
__device__ __forceinline__ void page_input(const PageBatch& cb, int p0, const void*& k, const void*& v, int& lo,
                                           int& len) {
  k = cb.c[0].k;
  v = cb.c[0].v;
  lo = cb.c[0].qlo;
  len = cb.c[0].tq;
#pragma unroll
  for (int j = 1; j < kMaxUpdateParts; ++j) {
    const bool in = j < cb.nch && p0 >= cb.c[j].qlo;
    k = in ? cb.c[j].k : k;
    v = in ? cb.c[j].v : v;
    lo = in ? cb.c[j].qlo : lo;
    len = in ? cb.c[j].tq : len;
  }
}

// The routed summary slots of query blocks bA .. bB into LDS: slot s holds entry s % kcap of block
// bA + s / kcap's row (s_n: the block, -1 where there is none before the row's or not yet summarised;
// s_b: the row's block), `cap` slots in all.
template <bool kBatch>
__device__ __forceinline__ void page_slots(const PageArgs& a, const std::conditional_t<kBatch, PageBatch, PageNoBatch>& cb,
                                           int zc, int bA, int bB, int cap, int* s_n, int* s_b) {
  const int tid = threadIdx.x, nslots = (bB - bA + 1) * a.kcap;
  if constexpr (kBatch) {
    // no table: thread t < blocks writes the row of block bA + t (neighbor_row, the table
    // builder's), the first wave clears the slots past them
    if (tid >= nslots && tid < cap) s_n[tid] = -1;
    const int bb = bA + tid;
    if (bb <= bB) {
      int32_t* list = s_n + tid * a.kcap;
      const int len = neighbor_row(bb, a.nblocks, cb.c[zc].topo, list, a.kcap);
      for (int j = 0; j < a.kcap; ++j) {
        const int n = j < len ? list[j] : -1;
        list[j] = n < bb && n < a.nsum ? n : -1;
        s_b[tid * a.kcap + j] = bb;
      }
    }
  } else if (tid < cap) {
    const int bb = bA + tid / a.kcap;
    int n = -1;
    if (tid < nslots) {
      n = a.nbr[(int64_t)bb * a.kcap + tid % a.kcap];
      if (n >= bb || n >= a.nsum) n = -1;
    }
    s_n[tid] = n;
    s_b[tid] = bb;
  }
}

template <int D, int HW, int NH, int MODE, bool kBatch = false>
__global__ void __launch_bounds__(256 * NH, (HW == 1 && D <= 128) ? 3 : 2)
page_attn_kernel(PageArgs a_in, std::conditional_t<kBatch, PageBatch, PageNoBatch> cb) {
  PageArgs a = a_in;
  using C = PageCfg<D, NH>;
  constexpr int NTHR = C::NTHR, KP = C::KP, KSTEPS = C::KSTEPS, LD = C::LD, MT = D / 32;
  constexpr bool kWin = MODE == kPageFused || MODE == kPageSwa;
  static_assert(MODE != kPageRouted || HW * NH == 1, "routed lists are per head");
  __shared__ __attribute__((aligned(16))) unsigned char smem[C::LDS];
  __shared__ __attribute__((aligned(16))) int s_n[kPageRows];   // summary page: block of each slot, -1 none
  __shared__ __attribute__((aligned(16))) int s_b[kPageRows];   // and the query block that lists it
  __shared__ int s_bad[2];
  __bf16* Ks = reinterpret_cast<__bf16*>(smem);
  __bf16* Vs = reinterpret_cast<__bf16*>(smem + C::K_BYTES);

  static_assert(!kBatch || MODE == kPageFused, "batches are the streaming loop's");
  if constexpr (kBatch) {
    static_assert(C::LDS >= NH * 256 * 8 * 4, "pooling scratch aliases the staging tiles");
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
  const float sl2 = a.scale * 1.4426950408889634f;

  // ---- Q fragments: lane (lg, lq) holds row lq at d = lg D/4 + 8 ks + 0..7 of k-step ks (the K
  // fragments use the same map, so the order of d cancels); rows outside the range read row 0
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

  // ---- the unit's pages
  const int q_first = max(chunk * kPageRows, a.qlo), q_last = min((chunk + 1) * kPageRows, a.qhi) - 1;
  int nwin = 0;
  if constexpr (kWin) {
    const int first = max(max(q_first - a.W + 1, a.key_lo), 0);
    nwin = q_last >= first ? chunk - first / kPageRows + 1 : 0;   // 0: every key is past the queries
  }
  const int bA = MODE == kPageSwa ? 0 : blk_of(q_first), bB = MODE == kPageSwa ? 0 : blk_of(q_last);
  // (without summaries there is no summary page: its row 0 would not exist)
  int npages = nwin, per_list = 1, nslots = 0;
  if constexpr (MODE == kPageFused) {
    nslots = (bB - bA + 1) * a.kcap;                    // at most 64 (the host's rule)
    npages = nwin + (a.nsum > 0 ? 1 : 0);
  } else if constexpr (MODE == kPageDense) {
    nslots = min(bB, a.nsum);
    npages = (nslots + kPageRows - 1) / kPageRows;
  } else if constexpr (MODE == kPageRouted) {
    per_list = (a.kcap + kPageRows - 1) / kPageRows;
    npages = a.nsum > 0 ? (bB - bA + 1) * per_list : 0;
  }
  const int64_t kv_off = (int64_t)bh * a.kv_rows * D, pool_off = (int64_t)bh * a.pool_rows * D;
  const __bf16* kb = reinterpret_cast<const __bf16*>(a.k) + kv_off;
  const __bf16* vb = reinterpret_cast<const __bf16*>(a.v) + kv_off;
  const __bf16* ksb = reinterpret_cast<const __bf16*>(a.ks) + pool_off;
  const __bf16* vsb = reinterpret_cast<const __bf16*>(a.vs) + pool_off;

  page_u32x4 kst[LD], vst[LD];
  int cand[LD];      // kRouted: the staged rows' list entries
  // Loads are unconditional: the page's nearest position that exists (a window page has one) or summary row 0
  // stands in for a row that does not.  Such a row is masked in the scores, and no value of it is needed (its
  // V takes weight 0; were it infinite, the page would be summed key by key), so nothing waits for the loads
  // before the page is stored.
  auto fetch = [&](int it) {
    int rr[LD];
    const __bf16 *kr = ksb, *vr = vsb;
    if (kWin && it < nwin) {
      const int p0 = (chunk - it) * kPageRows;
      int r0 = p0 - a.key_lo, wrap = a.ring;
      if (a.ring) r0 = (int)((unsigned)p0 % (unsigned)a.ring);   // p0 >= 0
      kr = kb;
      vr = vb;
      if constexpr (kBatch) {
        if (cb.from_inputs && p0 >= cb.c[0].qlo) {
          const void *kc, *vc;
          int lo, len;
          page_input(cb, p0, kc, vc, lo, len);
          kr = reinterpret_cast<const __bf16*>(kc) + (int64_t)bh * len * D;
          vr = reinterpret_cast<const __bf16*>(vc) + (int64_t)bh * len * D;
          r0 = p0 - lo;      // rows past the chunk's end are past kv_len, the attended chunk's end
          wrap = 0;
        }
      }
#pragma unroll
      for (int j = 0; j < LD; ++j) {
        const int r = min(max((tid + j * NTHR) / C::PIECES, a.key_lo - p0), a.kv_len - 1 - p0);
        int x = r0 + r;
        if (wrap && x >= wrap) x -= wrap;
        rr[j] = x;
      }
    } else if constexpr (MODE == kPageFused) {
#pragma unroll
      for (int j = 0; j < LD; ++j) rr[j] = max(s_n[(tid + j * NTHR) / C::PIECES], 0);
    } else if constexpr (MODE == kPageDense) {
#pragma unroll
      for (int j = 0; j < LD; ++j) {
        const int n = it * kPageRows + (tid + j * NTHR) / C::PIECES;
        rr[j] = n < nslots ? n : 0;
      }
    } else if constexpr (MODE == kPageRouted) {
      const int li = it / per_list, bb = bA + li, s0 = (it - li * per_list) * kPageRows;
      const int32_t* list = a.nbr + ((int64_t)(kvh * gsz + h0) * a.routed_blocks + bb) * a.kcap;
#pragma unroll
      for (int j = 0; j < LD; ++j) {
        const int s = s0 + (tid + j * NTHR) / C::PIECES;
        const int n = list[min(s, a.kcap - 1)];
        cand[j] = s < a.kcap && n >= 0 && n < bb && n < a.nsum ? n : -1;
        rr[j] = max(cand[j], 0);
      }
    }
#pragma unroll
    for (int j = 0; j < LD; ++j)
      kst[j] = *reinterpret_cast<const page_u32x4*>(kr + (int64_t)rr[j] * D + (tid + j * NTHR) % C::PIECES * 8);
#pragma unroll
    for (int j = 0; j < LD; ++j)
      vst[j] = *reinterpret_cast<const page_u32x4*>(vr + (int64_t)rr[j] * D + (tid + j * NTHR) % C::PIECES * 8);
  };

  if (npages > 0 && (MODE != kPageFused || nwin > 0)) fetch(0);
  if (tid < 2) s_bad[tid] = 0;
  if constexpr (MODE == kPageFused) {
    page_slots<kBatch>(a, cb, zc, bA, bB, kPageRows, s_n, s_b);
  }
  __syncthreads();   // s_bad and the summary slots
  if (MODE == kPageFused && nwin == 0 && npages > 0) fetch(0);

  const int wlo = max(max(qp - a.W + 1, a.key_lo), 0);
  const int qcut = max(0, (a.token_cutoff ? qp : qblk * a.bs) - a.W + 1);
  // V fragments (transposing reads): row 4 lg + (lq >> 2) of a tile, 8-byte unit
  // mt * 8 + (lq & 3) * 2 + half XOR the row's swizzle, which is this lane's alone
  const int xs = D == 64 ? (lq >> 3) & 1 : (lq >> 2) & 3;
  int vlane[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) vlane[r] = (4 * lg + (lq >> 2)) * D + ((r ^ xs) * 8 + (lq & 3) * 2) * 4;
  const int klane = lq * KP + lg * (D / 4);

  f32x4 o[HW][MT][2];
  float mref[HW], mtop[HW], lsum[HW];
#pragma unroll
  for (int u = 0; u < HW; ++u) {
    mref[u] = mtop[u] = -INFINITY;
    lsum[u] = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) o[u][mt][0] = o[u][mt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  for (int it = 0; it < npages; ++it) {
    unsigned worst = 0;
#pragma unroll
    for (int j = 0; j < LD; ++j) {
      const int i = tid + j * NTHR, r = i / C::PIECES, pc = i % C::PIECES;
      *reinterpret_cast<page_u32x4*>(Ks + r * KP + pc * 8) = kst[j];
      *reinterpret_cast<page_u32x4*>(Vs + r * D + (pc ^ vrow_swizzle<D>(r)) * 8) = vst[j];
      worst = max(worst, page_magnitude(vst[j]));
      if constexpr (MODE == kPageRouted) {
        if (pc == 0) s_n[r] = cand[j];
      }
    }
    if (worst >= kPageLarge) atomicMax(&s_bad[it & 1], worst >= kPageNonfinite ? 2 : 1);
    __syncthreads();   // the page is staged
    if (tid == 0) s_bad[(it + 1) & 1] = 0;
    const int flag = s_bad[it & 1];
    const bool page_bad = flag == 2;
    const float slack = flag != 0 ? 0.f : 8.f;
    if (it + 1 < npages) fetch(it + 1);

    const bool win = kWin && it < nwin;
    const int p0 = win ? (chunk - it) * kPageRows : 0;
    if (wave_on) {
#pragma unroll 1
      for (int pr = 0; pr < 2; ++pr) {
        // is any of the 32 keys one of this wave's rows', and does every row take all of them
        bool any, all;
        if (win) {
          const int k0 = p0 + 32 * pr;
          any = k0 <= pw + 15 && k0 + 31 >= pw - a.W + 1 && k0 + 31 >= a.key_lo;
          all = k0 + 31 <= pw && k0 >= pw + 15 - a.W + 1 && k0 >= a.key_lo;
        } else if constexpr (MODE == kPageRouted) {
          any = (it % per_list) * kPageRows + 32 * pr < a.kcap;
          all = false;
        } else {
          any = (MODE == kPageDense ? it * kPageRows : 0) + 32 * pr < nslots;
          all = false;
        }
        if (!any) continue;
        f32x4 s[HW][2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
          bf16x8 kf[KSTEPS];
#pragma unroll
          for (int ks = 0; ks < KSTEPS; ++ks)
            kf[ks] = *reinterpret_cast<const bf16x8*>(Ks + klane + (32 * pr + 16 * tt) * KP + 8 * ks);
#pragma unroll
          for (int u = 0; u < HW; ++u) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], qf[u][ks], acc, 0, 0, 0);
            s[u][tt] = acc * sl2;
          }
        }
        // is key `slot` of the page one that this lane's row attends to
        auto win_ok = [&](int slot) { return p0 + slot >= wlo && p0 + slot <= qp; };
        auto sum_ok = [&](int slot) {
          if constexpr (MODE == kPageFused) {
            const int n = s_n[slot];
            return n >= 0 && s_b[slot] == qblk && (n + 1) * a.bs <= qcut;
          } else if constexpr (MODE == kPageDense) {
            const int n = it * kPageRows + slot;
            return n < nslots && n < qblk;
          } else {
            return s_n[slot] >= 0 && bA + it / per_list == qblk;
          }
        };
        auto mask = [&](auto ok_of) {
#pragma unroll
          for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const bool ok = ok_of(32 * pr + 16 * tt + 4 * lg + i);
#pragma unroll
              for (int u = 0; u < HW; ++u) s[u][tt][i] = ok ? s[u][tt][i] : -INFINITY;
            }
        };
        if (win) {
          if (!all) mask(win_ok);
        } else {
          mask(sum_ok);
        }
        bf16x8 hi[HW], mid[HW], lo[HW];
#pragma unroll
        for (int u = 0; u < HW; ++u) {
          float mx = fmaxf(fmaxf(fmaxf(s[u][0][0], s[u][0][1]), fmaxf(s[u][0][2], s[u][0][3])),
                           fmaxf(fmaxf(s[u][1][0], s[u][1][1]), fmaxf(s[u][1][2], s[u][1][3])));
          mx = col_max4(mx);
          if constexpr (MODE != kPageFused) mtop[u] = fmaxf(mtop[u], mx);
          if (__any(mx > mref[u] + slack)) {
            const float mn = fmaxf(mref[u], mx);
            const float al = __builtin_amdgcn_exp2f(mref[u] - (mn == -INFINITY ? 0.f : mn));   // 0 at first
            mref[u] = mn;
            lsum[u] *= al;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
              o[u][mt][0] *= al;
              o[u][mt][1] *= al;
            }
          }
          const float mr = mref[u] == -INFINITY ? 0.f : mref[u];
#pragma unroll
          for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float e = __builtin_amdgcn_exp2f(s[u][tt][i] - mr);   // exp2(-inf) = 0
              s[u][tt][i] = e;
              lsum[u] += e;
            }
          const Parts4 x0 = split_parts(s[u][0]), x1 = split_parts(s[u][1]);
          hi[u] = join8(x0.h, x1.h);
          mid[u] = join8(x0.m, x1.m);
          lo[u] = join8(x0.l, x1.l);
        }
        if (!page_bad) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
              const __bf16* vp = Vs + vlane[mt & 3] + (mt >> 2) * 128 + half * 4 + 32 * pr * D;
              const bf16x4 va = read_tr(vp), vc = read_tr(vp + 16 * D);
              const bf16x8 vf = __builtin_shufflevector(va, vc, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
              for (int u = 0; u < HW; ++u) {
                o[u][mt][half] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, hi[u], o[u][mt][half], 0, 0, 0);
                o[u][mt][half] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, mid[u], o[u][mt][half], 0, 0, 0);
                o[u][mt][half] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, lo[u], o[u][mt][half], 0, 0, 0);
              }
            }
        } else {
          // key by key, only those the row attends to (a key's weight from the lane group
          // that scored it): O[d] of tile (mt, half) in lane (lg, lq) is d = 32 mt + 8 lg + 4 half + i
#pragma unroll
          for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll 1
              for (int src = 0; src < 4; ++src) {
                const int key = 32 * pr + 16 * tt + 4 * src + i;
                const bool take = win ? win_ok(key) : sum_ok(key);
#pragma unroll
                for (int u = 0; u < HW; ++u) {
                  const float p = __shfl(s[u][tt][i], lq + 16 * src);
#pragma unroll
                  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                      const int unit = mt * 8 + lg * 2 + half;
                      const bf16x4 x = *reinterpret_cast<const bf16x4*>(Vs + key * D + (unit ^ (2 * vrow_swizzle<D>(key))) * 4);
#pragma unroll
                      for (int e = 0; e < 4; ++e)
                        o[u][mt][half][e] = take ? fmaf(p, (float)x[e], o[u][mt][half][e]) : o[u][mt][half][e];
                    }
                }
              }
        }
      }
    }
    __syncthreads();   // every wave is done with the page
  }
  if (!wave_on) return;

  // ---- outputs: tiles mt, mt + 1 hold one 128-byte line per position; lanes lq and lq ^ 8 swap a
  // 16-byte piece so that each store writes 8 whole lines
  const bool lo8 = lq < 8;
  const int pA = pw + (lq & 7), pB = pA + 8;
  const bool okA = pA >= a.qlo && pA < a.qhi, okB = pB >= a.qlo && pB < a.qhi;
#pragma unroll
  for (int u = 0; u < HW; ++u) {
    const float l = col_sum4(lsum[u]);
    const bool live = h0 + u < gsz;
    float inv;
    if constexpr (MODE == kPageFused) {
      inv = 1.f / fmaxf(l, 1e-30f);
      // every window score -inf (or NaN): 0 / 0, as one softmax over the row's keys gives
      if (mref[u] == -INFINITY && wlo <= min(qp, a.kv_len - 1)) inv = NAN;
    } else {
      const bool any = mref[u] != -INFINITY;
      inv = any ? 1.f / l : 0.f;
      if (lg == 0 && row_ok && live) {
        const int64_t r = qhead0 + (int64_t)(h0 + u) * a.tq + (qp - a.qlo);
        // the sum is relative to mref: bring it to the row's true maximum
        a.l[r] = any ? l * __builtin_amdgcn_exp2f(mref[u] - mtop[u]) : 0.f;
        a.m[r] = any ? mtop[u] * 0.6931471805599453f : kPageNeg;
      }
    }
    __bf16* ob = reinterpret_cast<__bf16*>(a.out) + (qhead0 + (int64_t)min(h0 + u, gsz - 1) * a.tq) * D;
    __bf16* oA = ob + (int64_t)(okA ? pA - a.qlo : 0) * D;
    __bf16* oB = ob + (int64_t)(okB ? pB - a.qlo : 0) * D;
#pragma unroll
    for (int mp = 0; mp < MT / 2; ++mp) {
      bf16x8 w[2];
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          w[sub][i] = (__bf16)(o[u][2 * mp + sub][0][i] * inv);
          w[sub][4 + i] = (__bf16)(o[u][2 * mp + sub][1][i] * inv);
        }
      const bf16x8 x = page_xchg8(lo8 ? w[1] : w[0]);
      const bf16x8 sa = lo8 ? w[0] : x, sb = lo8 ? x : w[1];
      const int dA = (2 * mp + (lo8 ? 0 : 1)) * 32 + lg * 8;
      if (okA && live) __builtin_nontemporal_store(sa, reinterpret_cast<bf16x8*>(oA + dA));
      if (okB && live) __builtin_nontemporal_store(sb, reinterpret_cast<bf16x8*>(oB + dA));
    }
  }
}

// Query heads per workgroup: four where the GQA group has them and the grid still covers the chip
// twice over (a K or V fragment read then feeds two heads' MFMAs), else fewer heads in more
// workgroups, which stage the same pages again from L2.
template <int MODE>
static inline void launch_page_attn(PageArgs a, int d, hipStream_t stream) {
  a.c_first = a.qlo / kPageRows;
  a.nchunks = (a.qhi - 1) / kPageRows - a.c_first + 1;
  const int gsz = a.hq / a.hkv;
  const int64_t units = (int64_t)a.nchunks * a.batch * a.hkv;
  auto go = [&](auto kernel, int heads, int threads) {
    a.nparts = (gsz + heads - 1) / heads;
    a.items = (int)(units * a.nparts);
    a.per_xcd = (a.items + 7) / 8;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * a.per_xcd)), dim3(threads), 0, stream, a, PageNoBatch{});
  };
  if constexpr (MODE == kPageRouted) {
    if (d == 64) go(page_attn_kernel<64, 1, 1, MODE>, 1, 256);
    else if (d == 128) go(page_attn_kernel<128, 1, 1, MODE>, 1, 256);
    else go(page_attn_kernel<256, 1, 1, MODE>, 1, 256);
  } else {
    const bool four = gsz >= 3 && units * ((gsz + 3) / 4) >= 256;
    const bool two = gsz >= 2 && units * ((gsz + 1) / 2) >= 256;
    if (d == 64) {
      if (four) go(page_attn_kernel<64, 2, 2, MODE>, 4, 512);
      else if (two) go(page_attn_kernel<64, 2, 1, MODE>, 2, 256);
      else go(page_attn_kernel<64, 1, 1, MODE>, 1, 256);
    } else if (d == 128) {
      if (four) go(page_attn_kernel<128, 2, 2, MODE>, 4, 512);
      else if (two) go(page_attn_kernel<128, 2, 1, MODE>, 2, 256);
      else go(page_attn_kernel<128, 1, 1, MODE>, 1, 256);
    } else {
      go(page_attn_kernel<256, 1, 2, MODE>, 2, 512);   // (with one head the other waves only stage)
    }
  }
}

// Items of the widest split (one head per workgroup) that the kernel's 32-bit grid arithmetic takes.
static inline bool page_grid_fits(int64_t tq, int64_t batch, int64_t hq) {
  return (tq / kPageRows + 2) * batch * hq < (int64_t)1 << 30;
}

}  // namespace bfly
