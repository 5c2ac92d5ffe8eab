// Shared parts of the contrastive forward kernels (contrastive_tiled_kernel,
// contrastive_kloop_kernel): their arguments, the document chunks and the
// host's choice of how many.
#pragma once

#include "maxsim_common.h"
#include "maxsim_host.h"

#include <algorithm>

namespace maxsim {

constexpr int kDocWork = 32;            // work of a document beyond its rows, in rows
constexpr int kLptKeys = 128;           // sort keys of the dealt lists: tile counts, clamped
// Dealt lists when chunks average fewer documents than this: with 8 per
// chunk (64 queries x 512 C5 documents) contiguous chunks of whole documents
// hold up to 17 % more tiles than the mean (forward 139.6 -> 128.4 us
// dealt); with 64 (C5) within 2 %, and the ranking costs more (952.7 against
// 955 us)
constexpr int kDealtBelowDocsPerChunk = 32;

struct TiledArgs {
  const void* q;
  const void* d;
  const int32_t* doff;
  int64_t nq;
  int64_t nb;
  int64_t total_d;
  int lq;
  int dim;
  int nblk;   // blocks per query
  int qpg;    // queries per workgroup (query group)
  int n_qg;   // query groups
  int n_dc;   // document chunks
  int by_rank;  // one document per chunk: 1 longest first, 2 long and short paired
  bool qfrag; // contrastive_kloop_kernel: q holds fragments in order
  float* scores;
  int32_t* argmax;
};

// Position in the (document, tile) walk of a workgroup.  All fields are
// wave-uniform 32-bit values (document offsets are int32), so the walk stays
// in scalar registers.
struct TileCursor {
  int b;          // entry of the workgroup's document list
  int row0;       // its first row
  int ld;         // its length (0 when past the end)
  int t;          // tile within the document
  int id;         // its document index
};

// The documents of chunk dc, as a list in LDS (rows [s, e) and index of
// entry bl).  Two ways to form the chunks:
//  * dealt (more than one chunk, fewer than kDealtBelowDocsPerChunk
//    documents per chunk on average, at most one document per thread):
//    the documents sorted by tile count, longest
//    first (ties by index), and dealt in snake order, place p of round r
//    to chunk p (r even) or n_dc - 1 - p (r odd), so every chunk gets a
//    near-equal share of the tiles whatever the lengths.  Every workgroup
//    ranks all documents itself (the same ranks everywhere): one thread
//    per document, RankScratch (a mask per wave and key set by LDS atomic
//    ORs, then a scan over the keys);
//  * contiguous: the documents whose work prefix W(b) = off[b] + kDocWork
//    * b falls in [dc, dc + 1) * W / n_dc, W = total_d + kDocWork * nb
//    (rows, plus one tile's worth per document for its last partial tile
//    and its document-end work), so chunks hold equal work, not equal
//    counts.  The bounds are counts of documents below each threshold, one
//    parallel pass over the offsets; counts partition [0, nb) for any
//    offsets.
// kThreads = 64 kWaves threads build the list of at most kMaxDocs entries; the
// ranking's scratch of kScratchBytes may be the tile ring, which no load has
// touched yet.  Returns the number of entries, or -1 and the run [b_begin,
// b_end) when it is longer than the list; ends with LDS writes that the
// caller's barrier makes visible.
template <int kWaves, int kMaxDocs, int kScratchBytes>
__device__ __forceinline__ int chunk_documents(const TiledArgs& a, int dc, void* scratch,
                                               int* tab_s, int* tab_e, int* tab_id,
                                               int64_t& b_begin, int64_t& b_end) {
  constexpr int kThreads = 64 * kWaves;
  const int tid = threadIdx.x;
  int n_docs = 0;
  if (a.n_dc > 1 && a.n_dc < a.nb && a.nb <= kThreads &&
      a.nb < (int64_t)kDealtBelowDocsPerChunk * a.n_dc) {
    // scratch in the tile ring, which no load has touched yet (half the
    // keys where the ring is small: 32-element rows)
    constexpr int kKeys =
        RankScratch<kWaves, kLptKeys>::kBytes <= kScratchBytes ? kLptKeys : kLptKeys / 2;
    using Rank = RankScratch<kWaves, kKeys>;
    static_assert(Rank::kBytes <= kScratchBytes, "ranking scratch fits the tile ring");
    const Rank rs(scratch);
    rs.clear();
    const bool own = tid < a.nb;
    int s0 = 0, e0 = 0, key = 0;
    if (own) {
      s0 = a.doff[tid];
      e0 = a.doff[tid + 1];
      const bool ok = (s0 >= 0) && (e0 > s0) && ((int64_t)e0 <= a.total_d);
      const int t = ok ? (e0 - s0 + kTileRows - 1) / kTileRows : 0;
      key = t < kKeys - 1 ? t : kKeys - 1;
    }
    const int r = rs.rank(own, key);
    const int nc = a.n_dc, nbd = (int)a.nb;
    if (own) {
      const int rd = r / nc, p = r - rd * nc;
      if (((rd & 1) ? nc - 1 - p : p) == dc) {
        tab_s[rd] = s0;
        tab_e[rd] = e0;
        tab_id[rd] = tid;
      }
    }
    const int full = nbd / nc, tail = nbd - full * nc;
    n_docs = full + (tail > 0 && ((full & 1) ? nc - 1 - dc : dc) < tail ? 1 : 0);
  } else {
    __shared__ int chunk_cnt[2];
    if (threadIdx.x < 2) chunk_cnt[threadIdx.x] = 0;
    __syncthreads();
    if (a.n_dc >= a.nb) {
      // one document per chunk: nothing to balance
      if (threadIdx.x == 0) {
        chunk_cnt[0] = dc;
        chunk_cnt[1] = (int)min((int64_t)dc + 1, a.nb);
      }
    } else {
      const int64_t w_all = a.total_d + (int64_t)kDocWork * a.nb;
      const int64_t w_lo = w_all * dc / a.n_dc;
      const int64_t w_hi = w_all * (dc + 1) / a.n_dc;
      int c_lo = 0, c_hi = 0;
      for (int64_t bb = threadIdx.x; bb < a.nb; bb += kThreads) {
        const int64_t w = (int64_t)a.doff[bb] + (int64_t)kDocWork * bb;
        c_lo += w < w_lo ? 1 : 0;
        c_hi += w < w_hi ? 1 : 0;
      }
      if (c_lo) atomicAdd(&chunk_cnt[0], c_lo);
      if (c_hi) atomicAdd(&chunk_cnt[1], c_hi);
    }
    __syncthreads();
    b_begin = dc == 0 ? 0 : chunk_cnt[0];
    b_end = dc == a.n_dc - 1 ? a.nb : chunk_cnt[1];
    // With non-decreasing offsets consecutive documents are kDocWork apart
    // in W, so the host's chunk count keeps every chunk within the list.
    // Only offsets that decrease or overrun total_d can break that; such a
    // chunk is reported like documents with invalid offsets.
    if (b_end - b_begin > kMaxDocs) return -1;
    n_docs = (int)(b_end - b_begin);
    for (int i = tid; i < n_docs; i += kThreads) {
      tab_s[i] = a.doff[b_begin + i];
      tab_e[i] = a.doff[b_begin + i + 1];
      tab_id[i] = (int)(b_begin + i);
    }
  }
  return n_docs;
}

// Chunks of one document each, by length (at most one document per thread):
// the document of chunk dc in entry 0 of the list (as chunk_documents).  More
// workgroups than the chip holds start longest first and the short ones fill
// in; where all are resident at once (a.by_rank == 2), the second half of an
// XCD's workgroups, which share the CUs of the first, comes in the opposite
// order.
template <int kWaves, int kScratchBytes>
__device__ __forceinline__ void ranked_document(const TiledArgs& a, int dc, void* scratch,
                                                int* tab_s, int* tab_e, int* tab_id) {
  const int tid = threadIdx.x;
  using Rank = RankScratch<kWaves, kLptKeys>;
  static_assert(Rank::kBytes <= kScratchBytes, "ranking scratch fits the tile ring");
  const Rank rs(scratch);
  rs.clear();
  const bool own = tid < a.nb;
  int s0 = 0, e0 = 0, key = 0;
  if (own) {
    s0 = a.doff[tid];
    e0 = a.doff[tid + 1];
    const bool ok = (s0 >= 0) && (e0 > s0) && ((int64_t)e0 <= a.total_d);
    const int t = ok ? (e0 - s0 + kTileRows - 1) / kTileRows : 0;
    key = t < kLptKeys - 1 ? t : kLptKeys - 1;
  }
  const int r = rs.rank(own, key);
  // chunk dc is the k-th of XCD x; its rank counts the chunks (k', x') before
  // (k, x), so every XCD gets documents of all lengths, longest first
  const int nbd = (int)a.nb;
  const int per = (nbd + kXcds - 1) / kXcds;
  const int full = nbd / per, rem = nbd - full * per;
  const int x = dc / per;
  int k = dc - x * per;
  if (a.by_rank == 2 && rem == 0 && k >= (per + 1) / 2) k = per - 1 - (k - (per + 1) / 2);
  if (own && r == k * full + min(k, rem) + x) {
    tab_s[0] = s0;
    tab_e[0] = e0;
    tab_id[0] = tid;
  }
}

// Document chunks for n_qg query groups, one workgroup per (group, chunk) and
// `resident` workgroups on the chip at a time (one per CU for the tiled
// kernel): the launch takes rounds of that many, each as long as a chunk, and
// every round costs a pipeline fill of kRoundTiles tiles more.
// One round where the groups divide the CUs (C5: 32 groups, 8 chunks); with 3
// groups, 86 chunks are 258 workgroups, a second round for two of them, where
// 85 are one (21 queries of 64 tokens x 700 documents, bf16: 82.9 against
// 51.5 us).
constexpr int64_t kRoundTiles = 8;
inline int64_t chunks_for_rounds(int64_t n_qg, int64_t tiles, int64_t resident) {
  int64_t best = 0;
  double best_cost = 0.0;
  const int64_t r0 = (n_qg + resident - 1) / resident;
  for (int64_t r = r0; r < r0 + 4; ++r) {
    const int64_t n = r * resident / n_qg;
    const double cost = (double)r * ((double)tiles / (double)n + (double)kRoundTiles);
    if (best == 0 || cost < best_cost) {
      best = n;
      best_cost = cost;
    }
  }
  return best;
}

// contrastive_kloop_kernel (maxsim_kloop.hip): embedding rows that the tiled
// kernel does not hold in registers.  Rows of whole 16-element chunks on
// 16-byte boundaries are taken as they are; with a workspace, kloop_prepare()
// first brings the queries, and the documents if copy_d, into the kernel's
// layout (and points `a` at them).  `a` comes without the launch's own fields
// (qpg, n_qg, n_dc).
constexpr int kKloopBlocks = 8;  // query blocks of a workgroup
bool kloop_supported(maxsim_dtype dtype, int64_t dim, int64_t nblk);
size_t kloop_workspace_bytes(maxsim_dtype dtype, int64_t nq, int64_t nblk, int64_t total_d,
                             int64_t dim, bool copy_d);
int kloop_prepare(maxsim_dtype dtype, TiledArgs& a, bool copy_d, void* workspace, hipStream_t st);
int launch_contrastive_kloop(maxsim_dtype dtype, TiledArgs a, hipStream_t st);

}  // namespace maxsim
