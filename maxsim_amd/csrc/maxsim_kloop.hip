// Contrastive forward for rows that contrastive_tiled_kernel does not keep in
// registers: of other widths than its own (16-bit 32, 64 and 128, fp32 32 and
// 64) or off 16-byte boundaries, from 33 fp32 or 65 16-bit elements (two
// slices) up.
#include "maxsim_tiled.h"

#include <type_traits>

namespace maxsim {

// ---------------------------------------------------------------------------
// contrastive_kloop_kernel: a workgroup of four waves scores 256 query tokens
// (two 32-token blocks per wave) against four 32-row document tiles at a time,
// looping over the embedding dimension in slices of 128 bytes.  Per slice
// (a "unit") the document part, 128 rows, comes into LDS by direct
// global->LDS loads, wave w loading tile w; each wave's query part goes
// straight from L2 to its B fragments, since no other wave needs it.  The
// eight accumulators (128 VGPRs) stay in registers over the slices; after
// the last one the four tiles' maxima are taken in row order, and the running
// max and argmax carry over to the next four tiles until a document ends.
//
// Why this split: a 32 x 32 x 16 MFMA needs one A and one B fragment; with
// four tiles by two blocks six fragments feed eight MFMAs, four of them from
// LDS (64 bytes per clock of the CU's 128), and a unit moves (128 + 256) rows
// x 128 bytes through L2 for 2 x 128 x 256 x 64 operations, 48 bytes per clock
// and CU at the full MFMA rate.  Two workgroups per CU (at most 256 VGPRs,
// 44 KB of LDS each): one's MFMAs run under the other's epilogue and waits.
//
// Unit u computes from ring slot u % 2 while unit u + 1's loads are in
// flight: at its start every wave waits for its own loads, then the barrier
// makes the slot visible to all and frees the other one.  K chunks are taken
// in order into accumulators that start at zero, so every similarity has the
// bits that pair_kernel and wide_pair_kernel give it.
//
// Measured against those kernels (same process): bf16 dim 768, 64 queries of
// 32 tokens x 64 documents of 64-512 rows 496 -> 75 us, 256 x 256 documents of
// 100-400 rows 8480 -> 950 us (852 TFLOP/s; a large library product reaches
// about 1210 here); fp16 dim 384, 128 x 300: 2337 -> 312 us; fp32 dim 128,
// 200 x 200: 1082 -> 752 us (118 TFLOP/s of the 150 that a large fp32 product
// reaches).  Bound by L2 -> CU traffic and the per-unit waits in 16 bits, by
// the fp32 MFMA rate and, in small batches, by whole documents per workgroup
// (72 x 72: 185 -> 137 us, 83 TFLOP/s).
// ---------------------------------------------------------------------------
constexpr int kKlWaves = 4;
constexpr int kKlThreads = 64 * kKlWaves;
constexpr int kKlTiles = 4;                   // document tiles per step (one per wave to load)
constexpr int kKlBlocks = 2;                  // query blocks per wave
constexpr int kKlSlots = 2;                   // LDS ring, in units
constexpr int kKlSliceBytes = 128;            // of a row, per unit
constexpr int kKlPieces = kKlSliceBytes / 16;
constexpr int kKlTilePieces = kTileRows * kKlPieces;
constexpr int kKlUnitPieces = kKlTiles * kKlTilePieces;
constexpr int kKlMaxDocs = 1024;              // document list per workgroup
static_assert(kKlTiles == kKlWaves, "wave w loads tile w");
static_assert(kKlWaves * kKlBlocks == kKloopBlocks, "as the route counts them");

template <typename T, bool ARGMAX>
__global__ __launch_bounds__(kKlThreads, 2) void contrastive_kloop_kernel(TiledArgs a) {
  using S = typename T::storage;
  constexpr int kSliceElems = kKlSliceBytes / T::bytes;
  constexpr int kChunks = kSliceElems / kChunk;          // MFMA chunks per unit
  constexpr int kGroupBlocks = kKlWaves * kKlBlocks;
  __shared__ uint4 ring[kKlSlots * kKlUnitPieces];
  __shared__ int tab_s[kKlMaxDocs], tab_e[kKlMaxDocs], tab_id[kKlMaxDocs];
  __shared__ float part_sums[kKlTiles * kGroupBlocks];

  // XCD-aware mapping as in contrastive_tiled_kernel: an XCD takes a run of
  // chunks, the query groups of a chunk side by side
  const int64_t total = (int64_t)a.n_qg * a.n_dc;
  const int64_t per_xcd = gridDim.x / kXcds;
  const int64_t L = (int64_t)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
  if (L >= total) return;
  const int qg = (int)(L % a.n_qg);
  const int dc = (int)(L / a.n_qg);
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 31;
  const int h = lane >> 5;
  const S* __restrict__ D = static_cast<const S*>(a.d);
  const uint32_t row_bytes = (uint32_t)a.dim * (uint32_t)sizeof(S);
  float* __restrict__ scores = a.scores;
  int32_t* __restrict__ argmax_out = a.argmax;

  // this wave's blocks: part blk_part[j] of query blk_q[j]
  int64_t blk_q[kKlBlocks];
  int blk_part[kKlBlocks];
  bool blk_on[kKlBlocks];
  // this lane's fragment of chunk k at q_base + q_off + k * q_step (fp32: its
  // second half q_half further): rows as the caller has them, or fragments in
  // order (kloop_prepare_kernel)
  const MAXSIM_GLOBAL char* q_base[kKlBlocks];
  uint32_t q_off[kKlBlocks];
  const uint32_t frag_bytes = 64 * 16;
  const uint32_t q_step = a.qfrag ? frag_bytes * (T::bytes / 2) : kChunk * T::bytes;
  const uint32_t q_half = a.qfrag ? frag_bytes : 16;
#pragma unroll
  for (int j = 0; j < kKlBlocks; ++j) {
    const int g = wave * kKlBlocks + j;
    blk_q[j] = (int64_t)qg * a.qpg + g / a.nblk;
    blk_part[j] = g % a.nblk;
    blk_on[j] = g < a.qpg * a.nblk && blk_q[j] < a.nq;
    const int64_t q = min(blk_q[j], a.nq - 1);
    const int tok0 = blk_part[j] * kTileCols;
    if (a.qfrag) {
      q_base[j] = uniform_gptr(static_cast<const char*>(a.q) +
                               (q * a.nblk + blk_part[j]) * (int64_t)kTileCols * row_bytes);
      q_off[j] = lane * 16;
    } else {
      q_base[j] = uniform_gptr(static_cast<const char*>(a.q) + (q * a.lq + tok0) * row_bytes);
      q_off[j] = (uint32_t)min(c, a.lq - 1 - tok0) * row_bytes + (uint32_t)(8 * h * sizeof(S));
    }
  }

  int64_t b_begin = 0, b_end = 0;
  constexpr int kRingBytes = kKlSlots * kKlUnitPieces * (int)sizeof(uint4);
  int n_docs = 1;
  if (a.by_rank)
    ranked_document<kKlWaves, kRingBytes>(a, dc, ring, tab_s, tab_e, tab_id);
  else
    n_docs = chunk_documents<kKlWaves, kKlMaxDocs, kRingBytes>(a, dc, ring, tab_s, tab_e, tab_id,
                                                               b_begin, b_end);
  // NaN score and zero argmax for this wave's queries against document b
  auto write_invalid = [&](int64_t b) {
#pragma unroll
    for (int j = 0; j < kKlBlocks; ++j) {
      if (!blk_on[j]) continue;
      const int tok = blk_part[j] * kTileCols + c;
      if (ARGMAX && h == 0 && tok < a.lq) argmax_out[(blk_q[j] * a.nb + b) * a.lq + tok] = 0;
      if (blk_part[j] == 0 && lane == 0) scores[blk_q[j] * a.nb + b] = __builtin_nanf("");
    }
  };
  if (n_docs < 0) {
    for (int64_t b = b_begin; b < b_end; ++b) write_invalid(b);
    return;
  }
  __syncthreads();
  auto doc_ok = [&](int s, int e) { return (s >= 0) && (e > s) && ((int64_t)e <= a.total_d); };
  int ntiles = 0;
  for (int bl0 = 0; bl0 < n_docs; bl0 += 64) {
    const int bl = bl0 + lane;
    bool bad = false;
    if (bl < n_docs) {
      const int s = tab_s[bl], e = tab_e[bl];
      if (doc_ok(s, e))
        ntiles += (e - s + kTileRows - 1) / kTileRows;
      else
        bad = true;
    }
    for (uint64_t mb = __ballot(bad); mb; mb &= mb - 1)
      write_invalid(__builtin_amdgcn_readfirstlane(
          tab_id[bl0 + __ffsll((unsigned long long)mb) - 1]));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ntiles += __shfl_xor(ntiles, o);
  ntiles = __builtin_amdgcn_readfirstlane(ntiles);
  if (ntiles == 0) return;
  auto seek = [&](int bl) -> TileCursor {
    TileCursor cur{n_docs, 0, 0, 0, 0};
    for (; bl < n_docs; ++bl) {
      const int s = __builtin_amdgcn_readfirstlane(tab_s[bl]);
      const int e = __builtin_amdgcn_readfirstlane(tab_e[bl]);
      if (doc_ok(s, e)) {
        cur.b = bl;
        cur.row0 = s;
        cur.ld = e - s;
        cur.id = __builtin_amdgcn_readfirstlane(tab_id[bl]);
        break;
      }
    }
    return cur;
  };
  auto advance = [&](TileCursor cur) -> TileCursor {
    if (cur.b >= n_docs) return cur;
    if ((cur.t + 1) * kTileRows < cur.ld) {
      ++cur.t;
      return cur;
    }
    return seek(cur.b + 1);
  };

  const int nslices = (int)((row_bytes + kKlSliceBytes - 1) / kKlSliceBytes);  // >= 2
  const int nchunks = (a.dim + kChunk - 1) / kChunk;  // of a row (a.dim % kChunk == 0)
  const int nsteps = (ntiles + kKlTiles - 1) / kKlTiles;

  // ---- document loads: unit (step, slice) of tile `wave`
  TileCursor lc = seek(0);
  for (int i = 0; i < wave; ++i) lc = advance(lc);
  int ls = 0;  // slice of the next load
  const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(lds_addr(ring));
  auto load_docs = [&](int slot) __attribute__((always_inline)) {
    if (lc.b < n_docs) {
      const char* base = reinterpret_cast<const char*>(D) +
                         (int64_t)(lc.row0 + lc.t * kTileRows) * row_bytes +
                         (int64_t)ls * kKlSliceBytes;
      const int last = lc.ld - 1 - lc.t * kTileRows;
      // pieces past the row's end (the last slice) repeat its last one: their
      // chunks are not multiplied
      const int pmax = min(kKlPieces, (int)(row_bytes - ls * kKlSliceBytes) / 16) - 1;
#pragma unroll
      for (int i = 0; i < kKlTilePieces / 64; ++i) {
        const int r = i * (64 / kKlPieces) + lane / kKlPieces;
        const int p = min((lane % kKlPieces) ^ (r % kKlPieces), pmax);
        lds_dma16(base, (uint32_t)min(r, last) * row_bytes + (uint32_t)(p * 16),
                  ring_lds + (uint32_t)((slot * kKlUnitPieces + wave * kKlTilePieces + i * 64) *
                                        sizeof(uint4)));
      }
    }
    if (++ls == nslices) {
      ls = 0;
#pragma unroll
      for (int i = 0; i < kKlTiles; ++i) lc = advance(lc);
    }
  };
  // ---- query fragments of slice s
  auto load_query = [&](int s, Frag<T> (&f)[kKlBlocks][kChunks]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < kChunks; ++k) {
      if (s * kChunks + k < nchunks) {
#pragma unroll
        for (int j = 0; j < kKlBlocks; ++j) {
          const uint32_t off = q_off[j] + (uint32_t)(s * kChunks + k) * q_step;
          if constexpr (T::bytes == 2) {
            f[j][k].v = load16(q_base[j], off);
          } else {
            f[j][k].lo = load16(q_base[j], off);
            f[j][k].hi = load16(q_base[j], off + q_half);
          }
        }
      }
    }
  };
  // this lane's A fragment of chunk k of tile t in a slot
  auto read_doc = [&](int slot, int t, int k) __attribute__((always_inline)) {
    const uint4* tile = ring + slot * kKlUnitPieces + t * kKlTilePieces + c * kKlPieces;
    Frag<T> f;
    if constexpr (T::bytes == 2) {
      f.v = tile[(2 * k + h) ^ (c % kKlPieces)];
    } else {
      f.lo = tile[(4 * k + 2 * h) ^ (c % kKlPieces)];
      f.hi = tile[(4 * k + 2 * h + 1) ^ (c % kKlPieces)];
    }
    return f;
  };
  auto barrier = [&]() __attribute__((always_inline)) {
    __asm__ __volatile__("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ __volatile__("" ::: "memory");
  };

  float m[kKlBlocks];
  int am[kKlBlocks];
#pragma unroll
  for (int j = 0; j < kKlBlocks; ++j) {
    m[j] = -__builtin_inff();
    am[j] = 0;
  }
  f32x16 acc[kKlTiles][kKlBlocks];
  TileCursor ec = seek(0);
  // the documents whose last tile was tile t of the step before (-1: none)
  int done_id[kKlTiles];
#pragma unroll
  for (int t = 0; t < kKlTiles; ++t) done_id[t] = -1;
  // a document's block sums meet in part_sums; between the two barriers that
  // follow (a step has at least two units) one wave adds and writes them
  auto flush_scores = [&](int step) __attribute__((always_inline)) {
    if (wave == (step & (kKlWaves - 1))) {
#pragma unroll
      for (int t = 0; t < kKlTiles; ++t) {
        const int64_t q = (int64_t)qg * a.qpg + lane;
        if (done_id[t] >= 0 && lane < a.qpg && q < a.nq) {
          const float* ps = part_sums + t * kGroupBlocks + lane * a.nblk;
          float sum = 0.0f;
          for (int part = 0; part < a.nblk; ++part) sum += ps[part];
          scores[q * a.nb + done_id[t]] = sum;
        }
      }
    }
#pragma unroll
    for (int t = 0; t < kKlTiles; ++t) done_id[t] = -1;
  };
  auto epilogue = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < kKlTiles; ++t) {
      if (ec.b < n_docs) {
#pragma unroll
        for (int j = 0; j < kKlBlocks; ++j)
          tile_update<ARGMAX>(acc[t][j], m[j], am[j], ec.t * kTileRows + 4 * h);
        if (ec.ld - ec.t * kTileRows <= kTileRows) {  // the document's last tile
          done_id[t] = ec.id;
#pragma unroll
          for (int j = 0; j < kKlBlocks; ++j) {
            merge_halves(m[j], am[j]);
            const int tok = blk_part[j] * kTileCols + c;
            const bool vtok = tok < a.lq;
            const float sm = half_sum(vtok ? m[j] : 0.0f);
            if (lane == kHalfSumLane) part_sums[t * kGroupBlocks + wave * kKlBlocks + j] = sm;
            if (ARGMAX && blk_on[j] && h == 0 && vtok)
              argmax_out[(blk_q[j] * a.nb + ec.id) * a.lq + tok] = am[j];
            m[j] = -__builtin_inff();
            am[j] = 0;
          }
        }
        ec = advance(ec);
      }
    }
  };

  // ---- the units
  Frag<T> qa[kKlBlocks][kChunks], qb[kKlBlocks][kChunks];
  load_docs(0);
  load_query(0, qa);
  int step = 0, slice = 0;
  // One unit; `cur` holds its query fragments, `nxt` gets the next unit's.
  // Returns true after the last.
  auto unit = [&](auto slot_c, Frag<T> (&cur)[kKlBlocks][kChunks],
                  Frag<T> (&nxt)[kKlBlocks][kChunks]) __attribute__((always_inline)) -> bool {
    constexpr int SLOT = decltype(slot_c)::value;
    // this wave's loads have landed and its LDS accesses are done
    __builtin_amdgcn_s_waitcnt(0x0070);
    barrier();
    const bool last_slice = slice + 1 == nslices;
    const bool more = !(last_slice && step + 1 == nsteps);
    if (more) {
      load_docs(SLOT ^ 1);
      load_query(last_slice ? 0 : slice + 1, nxt);
    }
    if (slice == 0) {
      if (step > 0) flush_scores(step);
#pragma unroll
      for (int t = 0; t < kKlTiles; ++t)
#pragma unroll
        for (int j = 0; j < kKlBlocks; ++j) acc[t][j] = f32x16{};
    }
    const int left = nchunks - slice * kChunks;
#pragma unroll
    for (int k = 0; k < kChunks; ++k) {
      if (k < left) {
        Frag<T> df[kKlTiles];
#pragma unroll
        for (int t = 0; t < kKlTiles; ++t) df[t] = read_doc(SLOT, t, k);
#pragma unroll
        for (int t = 0; t < kKlTiles; ++t)
#pragma unroll
          for (int j = 0; j < kKlBlocks; ++j) mma_chunk(df[t], cur[j][k], acc[t][j]);
      }
    }
    if (last_slice) {
      epilogue();
      ++step;
      slice = 0;
    } else {
      ++slice;
    }
    return !more;
  };
  while (true) {
    if (unit(std::integral_constant<int, 0>{}, qa, qb)) break;
    if (unit(std::integral_constant<int, 1>{}, qb, qa)) break;
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);
  barrier();
  flush_scores(step);
}

// ---------------------------------------------------------------------------
// kloop_prepare_kernel: the queries as B fragments in the order in which the
// K-loop kernel loads them ([query, block][chunk][fp32: half][lane] x 16
// bytes, so that a wave's load is one run of 1 KB instead of 32 rows' 32
// bytes: 64 x 64 documents at dim 768 121 -> 88 us, 256 x 256 1259 -> 954 us),
// zero past the embedding dimension; and, where the document rows are
// not whole aligned chunks, a copy of them padded with zeros.
// ---------------------------------------------------------------------------
struct KlPrepArgs {
  const void* q;
  const void* d;      // null: the documents are used in place
  void* qf;
  void* dp;
  int64_t nq;
  int64_t total_d;
  int lq;
  int nblk;
  int dim;
  int dim_p;          // multiple of kChunk
  bool vec_q;         // rows of q in 16-byte pieces
};

template <typename T>
__global__ __launch_bounds__(256) void kloop_prepare_kernel(KlPrepArgs a) {
  using S = typename T::storage;
  const int chunks = a.dim_p / kChunk;
  const int64_t n_frag = a.nq * a.nblk * chunks * 64;  // one lane's 8 elements each
  const int pieces = a.dim_p / 8;
  const int64_t n = n_frag + (a.d ? a.total_d * pieces : 0);
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    if (i < n_frag) {
      const int lane = (int)(i & 63);
      const int64_t f = i >> 6;
      const int k = (int)(f % chunks);
      const int64_t blk = f / chunks;
      const int64_t q = blk / a.nblk;
      const int tok = min((int)(blk % a.nblk) * kTileCols + (lane & 31), a.lq - 1);
      const S* row = static_cast<const S*>(a.q) + (q * a.lq + tok) * (int64_t)a.dim;
      const Frag<T> v = load_frag<T>(row, kChunk * k + 8 * (lane >> 5), a.dim, a.vec_q);
      uint4* out = static_cast<uint4*>(a.qf) + f * (64 * (T::bytes / 2)) + lane;
      if constexpr (T::bytes == 2) {
        out[0] = v.v;
      } else {
        out[0] = v.lo;
        out[64] = v.hi;
      }
    } else {
      const int64_t x = i - n_frag;
      const int64_t r = x / pieces;
      const int p = (int)(x - r * pieces);
      const Frag<T> v =
          load_frag<T>(static_cast<const S*>(a.d) + r * (int64_t)a.dim, 8 * p, a.dim, false);
      uint4* out = reinterpret_cast<uint4*>(static_cast<S*>(a.dp) + r * (int64_t)a.dim_p + 8 * p);
      if constexpr (T::bytes == 2) {
        out[0] = v.v;
      } else {
        out[0] = v.lo;
        out[1] = v.hi;
      }
    }
  }
}

static int64_t padded_dim(int64_t dim) { return (dim + kChunk - 1) / kChunk * kChunk; }

// Workspace: the query fragments, then (documents not in whole aligned
// chunks) the padded documents.
static size_t kloop_frag_bytes(maxsim_dtype dtype, int64_t nq, int64_t nblk, int64_t dim) {
  return (size_t)(nq * nblk * kTileCols * padded_dim(dim)) * (dtype == MAXSIM_FLOAT32 ? 4 : 2);
}
size_t kloop_workspace_bytes(maxsim_dtype dtype, int64_t nq, int64_t nblk, int64_t total_d,
                             int64_t dim, bool copy_d) {
  return kloop_frag_bytes(dtype, nq, nblk, dim) +
         (copy_d ? (size_t)(total_d * padded_dim(dim)) * (dtype == MAXSIM_FLOAT32 ? 4 : 2) : 0);
}

template <typename T>
static void launch_prepare(const KlPrepArgs& a, hipStream_t st) {
  const int64_t n = a.nq * a.nblk * (a.dim_p / kChunk) * 64 +
                    (a.d ? a.total_d * (a.dim_p / 8) : 0);
  const int64_t grid = std::min<int64_t>((n + 255) / 256, 16 * (int64_t)device_cus());
  hipLaunchKernelGGL(kloop_prepare_kernel<T>, dim3((unsigned)grid), dim3(256), 0, st, a);
}

int kloop_prepare(maxsim_dtype dtype, TiledArgs& a, bool copy_d, void* workspace,
                  hipStream_t st) {
  KlPrepArgs p{};
  p.q = a.q;
  p.d = copy_d ? a.d : nullptr;
  p.qf = workspace;
  p.dp = static_cast<char*>(workspace) + kloop_frag_bytes(dtype, a.nq, a.nblk, a.dim);
  p.nq = a.nq;
  p.total_d = a.total_d;
  p.lq = a.lq;
  p.nblk = a.nblk;
  p.dim = a.dim;
  p.dim_p = (int)padded_dim(a.dim);
  p.vec_q = a.dim == p.dim_p && (reinterpret_cast<uintptr_t>(a.q) & 15u) == 0;
  switch (dtype) {
    case MAXSIM_BFLOAT16: launch_prepare<BF16>(p, st); break;
    case MAXSIM_FLOAT16: launch_prepare<F16>(p, st); break;
    default: launch_prepare<F32>(p, st); break;
  }
  a.q = p.qf;
  a.qfrag = true;
  if (copy_d) a.d = p.dp;
  a.dim = p.dim_p;
  return check_launch("kloop_prepare_kernel");
}

bool kloop_supported(maxsim_dtype dtype, int64_t dim, int64_t nblk) {
  const int bytes = dtype == MAXSIM_FLOAT32 ? 4 : 2;
  return padded_dim(dim) * bytes > kKlSliceBytes &&  // at least two slices
         nblk <= kKlWaves * kKlBlocks;
}

template <typename T>
static void launch_kloop(const TiledArgs& a, dim3 grid, hipStream_t st) {
  hipLaunchKernelGGL((a.argmax ? contrastive_kloop_kernel<T, true>
                               : contrastive_kloop_kernel<T, false>),
                     grid, dim3(kKlThreads), 0, st, a);
}

int launch_contrastive_kloop(maxsim_dtype dtype, TiledArgs a, hipStream_t st) {
  a.qpg = kKlWaves * kKlBlocks / a.nblk;
  a.n_qg = (int)((a.nq + a.qpg - 1) / a.qpg);
  const int64_t w_all = a.total_d + (int64_t)kDocWork * a.nb;
  const int64_t per_table = (int64_t)kDocWork * (kKlMaxDocs - 1);
  const int64_t resident = 2 * (int64_t)device_cus();
  int64_t n_dc = chunks_for_rounds(a.n_qg, w_all / kTileRows, resident);
  // Fewer than two documents per chunk cannot be balanced by dealing whole
  // documents: one workgroup each, by length (64 x 64 documents of 64-512
  // rows at dim 768: 88 us in document order, 75 us long and short paired).
  a.by_rank = 0;
  if (2 * n_dc > a.nb && a.nb <= kKlThreads) {
    n_dc = a.nb;
    a.by_rank = a.n_qg * a.nb <= resident ? 2 : 1;
  }
  n_dc = std::max<int64_t>(n_dc, (w_all + per_table - 1) / per_table);
  n_dc = std::max<int64_t>(1, std::min<int64_t>(n_dc, a.nb));
  a.n_dc = (int)n_dc;
  const int64_t total = (int64_t)a.n_qg * a.n_dc;
  const dim3 grid((unsigned)((total + kXcds - 1) / kXcds * kXcds));
  switch (dtype) {
    case MAXSIM_BFLOAT16: launch_kloop<BF16>(a, grid, st); break;
    case MAXSIM_FLOAT16: launch_kloop<F16>(a, grid, st); break;
    default: launch_kloop<F32>(a, grid, st); break;
  }
  return check_launch("contrastive_kloop_kernel");
}

}  // namespace maxsim
