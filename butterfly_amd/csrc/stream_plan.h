// Host rules of the streaming chunk loop (bfly_stream_chunks): which ring rows a launch may read, and when an
// update may write beside it.  No device code: a host compiler builds it for the tests.
#pragma once

#include <stdint.h>

namespace bfly {

constexpr int64_t kStreamPage = 64;

// The attention kernel of a stream's batches: attn_mfma_kernel, page_attn_kernel or win_attn_kernel.
enum class StreamKernel { kMfma, kPaged, kWindow };

// The lowest position whose ring row the kernel may read for queries from position q0 on.  Pages are staged
// whole: also rows that every query masks are read, and must not be written meanwhile.
inline int64_t stream_ring_lo(StreamKernel kernel, int64_t q0, int64_t window) {
  const int64_t page = q0 / kStreamPage * kStreamPage;
  int64_t lo = page - kStreamPage;                                        // the page before the queries' own
  if (kernel == StreamKernel::kWindow) lo = page - 2 * kStreamPage;       // three pages whatever the window
  if (kernel == StreamKernel::kPaged) {
    lo = q0 - (window - 1);
    lo = lo > 0 ? lo / kStreamPage * kStreamPage : 0;                     // the window's pages
  }
  return lo > 0 ? lo : 0;
}

// An upper bound of q0 - stream_ring_lo(kernel, q0, window), in whole pages.
inline int64_t stream_halo(StreamKernel kernel, int64_t window) {
  if (kernel == StreamKernel::kMfma) return 2 * kStreamPage;
  if (kernel == StreamKernel::kWindow) return 3 * kStreamPage;
  return (window - 1 + kStreamPage - 1) / kStreamPage * kStreamPage + kStreamPage;
}

// Whether an update that appends `next` tokens may run beside the attention of the `cur` tokens before them,
// whichever of their rows the attention reads from the ring: [P - cur - halo, P) against [P, P + next).
inline bool stream_apart(int64_t cur, int64_t next, int64_t halo, int64_t ring) { return cur + next + halo <= ring; }

// Whether positions [w_lo, w_hi) and the earlier positions [r_lo, r_hi) (r_hi <= w_lo) share no ring
// slot: no difference w - r is a multiple of the ring.
inline bool ring_disjoint(int64_t w_lo, int64_t w_hi, int64_t r_lo, int64_t r_hi, int64_t ring) {
  if (w_lo >= w_hi || r_lo >= r_hi) return true;
  const int64_t least = w_lo - (r_hi - 1), most = w_hi - 1 - r_lo;
  return (least - 1) / ring == most / ring;
}

}  // namespace bfly
