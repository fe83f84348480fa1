// Rank-deduplicated expert-parallel payloads on gfx950: the per-rank halves
// of PlaceMoE's dispatch and combine around the all-to-all.
//
// Dispatch (sender): every assignment (t, k) goes to rank r = slot / slots_per_rank.
// A token sends its hidden row once per distinct target rank; the assignments
// travel as (unique ordinal within the rank, local slot, token) plus weight,
// ordered by (rank, token, k).  Both orders, assignments by rank and the first
// assignment of each (rank, token) pair by rank, come out of one stable
// counting sort with 2R columns (chunks of whole tokens, one wave each): three
// launches, each bound by latency, instead of two sorts of one column per rank
// with the keys, metadata and counts beside them, ten launches (131072
// assignments, 8 ranks: 17 us of kernels against 50).
//
// Combine (receiver): weighted expert outputs of the received assignments,
// summed in fp32 per run of equal (source rank, source token) - the runs are
// contiguous because each sender's assignments arrive ordered by token.

#include "common.h"


namespace {

constexpr int kPayloadMaxTopK = 32;

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

constexpr int kPayloadLdsRanks = 4096;       // 2R counters in LDS up to this many ranks
constexpr int kPayloadMaxRanks = (1 << 24) - 1;

// Chunks of whole tokens: segments of 64 / K tokens, one lane per assignment,
// four a chunk (their loads are in flight together), more of them past 1024
// chunks or 2^24 table entries.
struct PayloadGeom {
  int32_t seg;      // assignments per segment
  int64_t chunk;    // ... per chunk
  int64_t nchunks;  // >= 1
};

constexpr int kPayloadSegs = 4;

int64_t payload_max_chunks(int64_t A, int32_t R) {
  const int64_t most = (int64_t(1) << 23) / R;
  const int64_t cap = most > 1024 ? 1024 : most < 1 ? 1 : most;
  const int64_t n = A / (kPayloadSegs * 33) + 1;  // a segment has at least 33 lanes in use
  return n < cap ? n : cap;
}

PayloadGeom payload_geom(int64_t A, int32_t K, int32_t R) {
  PayloadGeom g;
  const int64_t max_chunks = payload_max_chunks(A, R);
  g.seg = 64 / K * K;
  g.chunk = (int64_t)kPayloadSegs * g.seg;
  if ((A + g.chunk - 1) / g.chunk > max_chunks)
    g.chunk = ((A + max_chunks - 1) / max_chunks + g.seg - 1) / g.seg * g.seg;
  g.nchunks = (A + g.chunk - 1) / g.chunk;
  if (g.nchunks < 1) g.nchunks = 1;
  return g;
}

// Target rank of a slot (clamped into [0, R*L); bad: it was not inside).
__device__ __forceinline__ int32_t rank_of(int32_t p, int32_t hi, int32_t L, int& bad) {
  if (p < 0 || p > hi) {
    bad = 1;
    p = p < 0 ? 0 : hi;
  }
  return p / L;
}

// The lanes of a segment with this lane's rank (same), the first of them in
// every token (first), and the lanes of this lane's token (tok).
struct Peers {
  uint64_t same, first, tok;
};
__device__ __forceinline__ Peers peers(int32_t r, bool valid, int nbits, int lane, int32_t K) {
  Peers q;
  q.same = match_any(r, valid, nbits);
  q.tok = ((1ull << K) - 1) << (lane / K * K);
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  q.first = __ballot(valid && (q.same & q.tok & lt) == 0) & q.same;
  return q;
}

// Per chunk: target ranks, and the counts of the chunk's assignments (columns
// 0 .. R-1 of its table row) and of its (rank, token) pairs (R .. 2R-1) per rank.
// (I: the index type of the caller's slots, ranks and tokens, of which the low
// 32 bits count.)
template <bool USE_LDS, class I>
__global__ __launch_bounds__(64) void payload_hist_kernel(const I* __restrict__ phys, int64_t A, int32_t K,
                                                          int32_t R, int32_t L, int32_t seg, int64_t chunk, int nbits,
                                                          I* __restrict__ target_rank,
                                                          int32_t* __restrict__ table, int32_t* __restrict__ flags,
                                                          int32_t* __restrict__ status) {
  extern __shared__ int32_t lds_hist[];
  const int lane = threadIdx.x;
  int32_t* row = table + (int64_t)blockIdx.x * 2 * R;
  int32_t* hist = USE_LDS ? lds_hist : row;
  for (int c = lane; c < 2 * R; c += 64) hist[c] = 0;
  __syncthreads();
  const int64_t begin = (int64_t)blockIdx.x * chunk;
  const int64_t end = begin + chunk < A ? begin + chunk : A;
  const int32_t hi = R * L - 1;
  int bad = 0;
  for (int64_t s = begin; s < end; s += kPayloadSegs * seg) {
    int32_t p[kPayloadSegs];
#pragma unroll
    for (int u = 0; u < kPayloadSegs; ++u) {
      const int64_t a = s + u * seg + lane;
      p[u] = lane < seg && a < end ? (int32_t)phys[a] : 0;
    }
#pragma unroll
    for (int u = 0; u < kPayloadSegs; ++u) {
      const int64_t a = s + u * seg + lane;
      const bool valid = lane < seg && a < end;
      const int32_t r = rank_of(p[u], hi, L, bad);
      if (valid) target_rank[a] = r;
      const Peers q = peers(r, valid, nbits, lane, K);
      if (valid && lane == 63 - __clzll(q.same)) {
        atomicAdd(&hist[r], __popcll(q.same));
        atomicAdd(&hist[R + r], __popcll(q.first));
      }
    }
  }
  __syncthreads();
  if (USE_LDS)
    for (int c = lane; c < 2 * R; c += 64) row[c] = hist[c];
  const bool any_bad = __ballot(bad) != 0;
  if (lane == 0) {
    flags[blockIdx.x] = 0;
    if (any_bad) atomicOr(status, 1);
  }
}

// Per assignment: its metadata row and weight at its place in (rank, token,
// k) order; per (rank, token) pair its token and, at its first assignment,
// its row (upos; -1 at the others).  `table` holds the chunks' start
// positions, those of the pairs behind the A assignments.  Block 0 writes the
// counts and offsets out.
template <bool USE_LDS, class I>
__global__ __launch_bounds__(64) void payload_place_kernel(
    const I* __restrict__ phys, const bf16_t* __restrict__ weights, int64_t A, int32_t K, int32_t R, int32_t L,
    int32_t seg, int64_t chunk, int nbits, int32_t* __restrict__ table, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ offsets, int32_t* __restrict__ assign_counts, int32_t* __restrict__ assign_offsets,
    int32_t* __restrict__ unique_counts, int32_t* __restrict__ unique_offsets, int32_t* __restrict__ send_meta,
    bf16_t* __restrict__ send_weights, I* __restrict__ unique_tokens, int32_t* __restrict__ upos) {
  extern __shared__ int32_t lds_pos[];
  const int lane = threadIdx.x;
  if (blockIdx.x == 0) {
    for (int r = lane; r <= R; r += 64) {
      if (r < R) assign_counts[r] = counts[r], unique_counts[r] = counts[R + r];
      assign_offsets[r] = offsets[r];
      unique_offsets[r] = (int32_t)((uint32_t)offsets[R + r] - (uint32_t)A);
    }
  }
  int32_t* row = table + (int64_t)blockIdx.x * 2 * R;
  int32_t* next = USE_LDS ? lds_pos : row;
  if (USE_LDS) {
    for (int c = lane; c < 2 * R; c += 64) next[c] = row[c];
    __syncthreads();
  }
  const int64_t begin = (int64_t)blockIdx.x * chunk;
  const int64_t end = begin + chunk < A ? begin + chunk : A;
  const int32_t hi = R * L - 1;
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  // The counters are read and written by this wave only; atomics keep the
  // global-table form coherent between its lanes.
  constexpr int kScope = USE_LDS ? __HIP_MEMORY_SCOPE_WORKGROUP : __HIP_MEMORY_SCOPE_AGENT;
  for (int64_t s = begin; s < end; s += kPayloadSegs * seg) {
    int32_t p[kPayloadSegs];
    bf16_t w[kPayloadSegs];
#pragma unroll
    for (int u = 0; u < kPayloadSegs; ++u) {
      const int64_t a = s + u * seg + lane;
      const bool valid = lane < seg && a < end;
      p[u] = valid ? (int32_t)phys[a] : 0;
      w[u] = valid ? weights[a] : (bf16_t)0;
    }
#pragma unroll
    for (int u = 0; u < kPayloadSegs; ++u) {
      const int64_t a = s + u * seg + lane;
      const bool valid = lane < seg && a < end;
      int bad = 0;
      const int32_t r = rank_of(p[u], hi, L, bad);
      const Peers q = peers(r, valid, nbits, lane, K);
      int32_t abase = 0, ubase = 0;
      if (valid) {
        abase = __hip_atomic_load(&next[r], __ATOMIC_RELAXED, kScope);
        ubase = (int32_t)((uint32_t)__hip_atomic_load(&next[R + r], __ATOMIC_RELAXED, kScope) - (uint32_t)A);
      }
      __builtin_amdgcn_wave_barrier();
      if (valid) {
        const int f = __ffsll((unsigned long long)(q.same & q.tok)) - 1;  // the token's first lane with this rank
        const uint64_t before_f = f == 0 ? 0ull : (~0ull >> (64 - f));
        const int32_t urow = ubase + __popcll(q.first & before_f);
        const int64_t o = abase + __popcll(q.same & lt);
        const int32_t slot = p[u] < 0 ? 0 : (p[u] > hi ? hi : p[u]);
        const int32_t t = (int32_t)(a / K);
        send_meta[o * 3 + 0] = (int32_t)((uint32_t)urow + (uint32_t)A - (uint32_t)offsets[R + r]);
        send_meta[o * 3 + 1] = slot - r * L;
        send_meta[o * 3 + 2] = t;
        send_weights[o] = w[u];
        if (f == lane) unique_tokens[urow] = t;
        upos[a] = f == lane ? urow : -1;
        if (lane == 63 - __clzll(q.same)) {
          __hip_atomic_store(&next[r], abase + __popcll(q.same), __ATOMIC_RELAXED, kScope);
          __hip_atomic_store(&next[R + r], (int32_t)((uint32_t)ubase + (uint32_t)A) + __popcll(q.first),
                             __ATOMIC_RELAXED, kScope);
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// send_hidden[upos[a]] = hidden[t] for the first assignment a of each
// (rank, token) pair.  One wave per token: the row is read once, four 16-byte
// chunks a lane, and stored to every rank that takes it.
__global__ __launch_bounds__(256) void payload_rows_kernel(const bf16_t* __restrict__ hidden,
                                                           const int32_t* __restrict__ upos, int64_t T, int32_t K,
                                                           int64_t H, bf16_t* __restrict__ send_hidden) {
  constexpr int U = 4;
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t >= T) return;
  const int64_t n8 = H / 8;
  const uint4* src = reinterpret_cast<const uint4*>(hidden + t * H);
  const int32_t my_row = lane < K ? upos[t * K + lane] : -1;
  const uint64_t rows = __ballot(my_row >= 0);
  for (int64_t i0 = lane; i0 - lane < n8; i0 += 64 * U) {
    uint4 v[U] = {};
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i0 + 64 * u < n8) v[u] = ld_stream(src + i0 + 64 * u);
    for (uint64_t m = rows; m != 0; m &= m - 1) {
      const int k = __ffsll((unsigned long long)m) - 1;
      uint4* dst = reinterpret_cast<uint4*>(send_hidden + (int64_t)__builtin_amdgcn_readlane(my_row, k) * H);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i0 + 64 * u < n8) dst[i0 + 64 * u] = v[u];
    }
  }
}

__global__ void fill_kernel(int32_t* __restrict__ p, int32_t n) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------------------
// Combine aggregation
// ---------------------------------------------------------------------------

constexpr int kScanBlock = 1024;

// flag[a] = 1 where a run of equal (src_rank, src_token) starts; per-block
// sums of the flags; rank_runs cleared for the counts that follow.
template <class I>
__global__ __launch_bounds__(kScanBlock) void run_flags_kernel(const I* __restrict__ src_rank,
                                                               const I* __restrict__ src_token, int64_t N,
                                                               int32_t* __restrict__ flag,
                                                               int32_t R, int32_t* __restrict__ rank_runs,
                                                               int32_t* __restrict__ block_sum) {
  __shared__ int32_t red[kScanBlock / 64];
  const int64_t a = (int64_t)blockIdx.x * kScanBlock + threadIdx.x;
  for (int64_t r = a; r < R; r += (int64_t)gridDim.x * kScanBlock) rank_runs[r] = 0;
  int32_t f = 0;
  if (a < N) {
    f = (a == 0 || (int32_t)src_rank[a] != (int32_t)src_rank[a - 1] ||
         (int32_t)src_token[a] != (int32_t)src_token[a - 1])
            ? 1
            : 0;
    flag[a] = f;
  }
  const uint64_t m = __ballot(f != 0);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = __popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t s = 0;
    for (int w = 0; w < kScanBlock / 64; ++w) s += red[w];
    block_sum[blockIdx.x] = s;
  }
}

// Exclusive scan of the block sums in one block; total -> *num_runs.
__global__ __launch_bounds__(kScanBlock) void scan_blocks_kernel(int32_t* __restrict__ block_sum, int64_t nblocks,
                                                                 int32_t* __restrict__ num_runs) {
  __shared__ int32_t sums[kScanBlock];
  __shared__ int32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int64_t base = 0; base < nblocks; base += kScanBlock) {
    const int64_t i = base + threadIdx.x;
    const int32_t v = i < nblocks ? block_sum[i] : 0;
    sums[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < kScanBlock; off <<= 1) {
      const int32_t add = threadIdx.x >= off ? sums[threadIdx.x - off] : 0;
      __syncthreads();
      sums[threadIdx.x] += add;
      __syncthreads();
    }
    const int32_t c = carry;
    if (i < nblocks) block_sum[i] = c + sums[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == kScanBlock - 1) carry = c + sums[kScanBlock - 1];
    __syncthreads();
  }
  if (threadIdx.x == 0) *num_runs = carry;
}

// Run starts -> run_offsets[run] = a (and run_offsets[U] = N); runs per
// source rank, counted in LDS per block (up to kLdsRanks ranks) and added to
// the global counts once per block and rank: the ranks are sorted, so one
// block touches few of them, and a global atomic per run would serialise on
// R counters.
constexpr int kLdsRanks = 4096;

template <class I>
__global__ __launch_bounds__(kScanBlock) void run_offsets_kernel(const int32_t* __restrict__ flag,
                                                                 const int32_t* __restrict__ block_base,
                                                                 const I* __restrict__ src_rank, int64_t N,
                                                                 int32_t R, const int32_t* __restrict__ num_runs,
                                                                 int32_t* __restrict__ run_offsets,
                                                                 int32_t* __restrict__ rank_runs,
                                                                 int32_t* __restrict__ status) {
  __shared__ int32_t wsum[kScanBlock / 64];
  __shared__ int32_t cnt[kLdsRanks];
  const bool lds = R <= kLdsRanks;
  if (lds)
    for (int i = threadIdx.x; i < R; i += kScanBlock) cnt[i] = 0;
  const int64_t a = (int64_t)blockIdx.x * kScanBlock + threadIdx.x;
  const int32_t f = a < N ? flag[a] : 0;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t m = __ballot(f != 0);
  if (lane == 0) wsum[w] = __popcll(m);
  __syncthreads();
  int32_t before = block_base[blockIdx.x];
  for (int i = 0; i < w; ++i) before += wsum[i];
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  if (f) {
    const int32_t run = before + __popcll(m & lt);
    run_offsets[run] = (int32_t)a;
    const int32_t r = (int32_t)src_rank[a];
    if (r >= 0 && r < R) {
      if (lds) atomicAdd(&cnt[r], 1);
      else atomicAdd(&rank_runs[r], 1);
    } else {
      atomicOr(status, 1);
    }
  }
  if (a == 0) run_offsets[*num_runs] = (int32_t)N;
  if (lds) {
    __syncthreads();
    for (int i = threadIdx.x; i < R; i += kScanBlock)
      if (cnt[i]) atomicAdd(&rank_runs[i], cnt[i]);
  }
}

// out[run] = bf16( sum_{a in run} fp32( bf16(Y[pos[a]] * w[a]) ) ).  Bound by
// HBM: every row of Y is read once, every sum written once, and a run has 1-2
// rows.  One wave per run (four to a block): a lane takes four 16-byte chunks
// of a row at a time and two rows together, so that a wave has up to 8 KB on
// its way behind one read of the run's positions; rows are added in order.
template <class E, class I>
__global__ __launch_bounds__(256) void run_combine_kernel(const bf16_t* __restrict__ Y,
                                                          const I* __restrict__ pos,
                                                          const bf16_t* __restrict__ w,
                                                          const int32_t* __restrict__ run_offsets,
                                                          const int32_t* __restrict__ num_runs, int64_t H,
                                                          bf16_t* __restrict__ out) {
  constexpr int U = 4;
  const int lane = threadIdx.x & 63;
  const int64_t run = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (run >= *num_runs) return;
  const int32_t b = run_offsets[run], e = run_offsets[run + 1];
  const int64_t n8 = H / 8;
  for (int64_t i0 = lane; i0 - lane < n8; i0 += 64 * U) {
    float acc[U][8] = {};
    for (int32_t a0 = b; a0 < e; a0 += 64) {
      const int n = e - a0 < 64 ? e - a0 : 64;
      const int32_t my_pos = lane < n ? (int32_t)pos[a0 + lane] : 0;
      const int32_t my_w = lane < n ? (int32_t)w[a0 + lane] : 0;
      auto load = [&](int j, uint4 (&v)[U]) __attribute__((always_inline)) {
        const uint4* row = reinterpret_cast<const uint4*>(Y + (int64_t)__builtin_amdgcn_readlane(my_pos, j) * H);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (i0 + 64 * u < n8) v[u] = ld_stream(row + i0 + 64 * u);
      };
      auto add = [&](int j, const uint4 (&v)[U]) __attribute__((always_inline)) {
        const float wk = E::to_f32((uint32_t)__builtin_amdgcn_readlane(my_w, j));
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float f[8];
          unpack8e<E>(v[u], f);
#pragma unroll
          for (int x = 0; x < 8; ++x) acc[u][x] += E::round(f[x] * wk);
        }
      };
      for (int j = 0; j < n; j += 2) {
        uint4 v0[U] = {}, v1[U] = {};
        load(j, v0);
        if (j + 1 < n) {
          load(j + 1, v1);
          add(j, v0);
          add(j + 1, v1);
        } else {
          add(j, v0);
        }
      }
    }
    uint4* o = reinterpret_cast<uint4*>(out + run * H);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i0 + 64 * u < n8) st_stream(o + i0 + 64 * u, pack8e<E>(acc[u]));
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

extern "C" {

size_t pmx_ep_payload_workspace_bytes(int64_t num_assign, int32_t num_ranks) {
  if (num_assign < 0 || num_ranks <= 0) return 0;
  // the chunk table (K decides the chunks: at most 1024, or one, rows), one
  // flag a chunk, upos, counts, offsets, the scan's status word
  const size_t chunks = payload_max_chunks(num_assign, num_ranks);
  return align256(chunks * 2 * (size_t)num_ranks * sizeof(int32_t)) + align256(chunks * sizeof(int32_t)) +
         align256((size_t)num_assign * sizeof(int32_t)) + 2 * align256((size_t)(2 * (int64_t)num_ranks + 1) * sizeof(int32_t)) +
         256;
}

}  // extern "C"

namespace {

template <class I>
int ep_dispatch_payload_t(const I* phys, const void* hidden, const void* weights, int64_t T, int32_t K,
                            int64_t H, int32_t R, int32_t slots_per_rank, int32_t* assign_counts,
                            int32_t* assign_offsets, int32_t* unique_counts, int32_t* unique_offsets,
                            void* send_hidden, I* unique_tokens, int32_t* send_meta, void* send_weights,
                            I* target_rank, int32_t* status, void* workspace, size_t workspace_bytes,
                            pmx_stream_t stream) {
  if (T < 0 || K <= 0 || K > kPayloadMaxTopK || H < 0 || R <= 0 || slots_per_rank <= 0) return PMX_ERR_ARG;
  if (R > kPayloadMaxRanks) return PMX_ERR_ARG;
  if ((int64_t)R * slots_per_rank > (int64_t)INT32_MAX) return PMX_ERR_SHAPE;
  if (H % 8) return PMX_ERR_SHAPE;
  if (!assign_counts || !assign_offsets || !unique_counts || !unique_offsets || !status || !workspace)
    return PMX_ERR_ARG;
  const int64_t A = T * K;
  if (A > (int64_t)INT32_MAX) return PMX_ERR_SHAPE;
  if (A > 0 && (!phys || !weights || !unique_tokens || !send_meta || !send_weights || !target_rank))
    return PMX_ERR_ARG;
  if (A > 0 && H > 0 && (!hidden || !send_hidden || !aligned16(hidden) || !aligned16(send_hidden)))
    return PMX_ERR_ARG;
  if (workspace_bytes < pmx_ep_payload_workspace_bytes(A, R)) return PMX_ERR_ARG;

  char* ws = reinterpret_cast<char*>(workspace);
  size_t off = 0;
  auto carve = [&](size_t n) {
    int32_t* p = reinterpret_cast<int32_t*>(ws + off);
    off += align256(n * sizeof(int32_t));
    return p;
  };
  const PayloadGeom g = payload_geom(A, K, R);
  int32_t* table = carve((size_t)g.nchunks * 2 * R);
  int32_t* flags = carve((size_t)g.nchunks);
  int32_t* upos = carve((size_t)A);
  int32_t* counts = carve((size_t)2 * R);
  int32_t* offsets = carve((size_t)2 * R + 1);
  int32_t* scan_status = carve(1);

  const bool lds = R <= kPayloadLdsRanks;
  const size_t lds_bytes = lds ? (size_t)2 * R * sizeof(int32_t) : 0;
  const unsigned chunks = (unsigned)g.nchunks;
  int nbits = 0;
  while ((1 << nbits) < R) ++nbits;
  auto hist = lds ? payload_hist_kernel<true, I> : payload_hist_kernel<false, I>;
  auto place = lds ? payload_place_kernel<true, I> : payload_place_kernel<false, I>;
  hist<<<chunks, 64, lds_bytes, stream>>>(phys, A, K, R, slots_per_rank, g.seg, g.chunk, nbits, target_rank, table, flags,
                                          status);
  PMX_LAUNCH_CHECK();
  const int rc = pmx_route_scan_launch(table, g.nchunks, 2 * R, flags, counts, offsets, scan_status, stream);
  if (rc != PMX_OK) return rc;
  place<<<chunks, 64, lds_bytes, stream>>>(phys, static_cast<const bf16_t*>(weights), A, K, R, slots_per_rank, g.seg,
                                           g.chunk, nbits, table, counts, offsets, assign_counts, assign_offsets,
                                           unique_counts, unique_offsets, send_meta,
                                           static_cast<bf16_t*>(send_weights), unique_tokens, upos);
  PMX_LAUNCH_CHECK();
  if (A == 0) return PMX_OK;
  if (H > 0) {
    payload_rows_kernel<<<(unsigned)((T + 3) / 4), 256, 0, stream>>>(static_cast<const bf16_t*>(hidden), upos, T, K, H,
                                                         static_cast<bf16_t*>(send_hidden));
    PMX_LAUNCH_CHECK();
  }
  return PMX_OK;
}

}  // namespace

extern "C" {

int pmx_ep_dispatch_payload(const int32_t* phys, const void* hidden, const void* weights, int64_t T, int32_t K,
                            int64_t H, int32_t R, int32_t slots_per_rank, int32_t* assign_counts,
                            int32_t* assign_offsets, int32_t* unique_counts, int32_t* unique_offsets,
                            void* send_hidden, int32_t* unique_tokens, int32_t* send_meta, void* send_weights,
                            int32_t* target_rank, int32_t* status, void* workspace, size_t workspace_bytes,
                            pmx_stream_t stream) {
  return ep_dispatch_payload_t(phys, hidden, weights, T, K, H, R, slots_per_rank, assign_counts, assign_offsets,
                               unique_counts, unique_offsets, send_hidden, unique_tokens, send_meta, send_weights,
                               target_rank, status, workspace, workspace_bytes, stream);
}

int pmx_ep_dispatch_payload_i64(const int64_t* phys, const void* hidden, const void* weights, int64_t T, int32_t K,
                            int64_t H, int32_t R, int32_t slots_per_rank, int32_t* assign_counts,
                            int32_t* assign_offsets, int32_t* unique_counts, int32_t* unique_offsets,
                            void* send_hidden, int64_t* unique_tokens, int32_t* send_meta, void* send_weights,
                            int64_t* target_rank, int32_t* status, void* workspace, size_t workspace_bytes,
                            pmx_stream_t stream) {
  return ep_dispatch_payload_t(phys, hidden, weights, T, K, H, R, slots_per_rank, assign_counts, assign_offsets,
                               unique_counts, unique_offsets, send_hidden, unique_tokens, send_meta, send_weights,
                               target_rank, status, workspace, workspace_bytes, stream);
}

size_t pmx_ep_combine_workspace_bytes(int64_t num_recv) {
  if (num_recv < 0) return 0;
  const int64_t nblocks = (num_recv + kScanBlock - 1) / kScanBlock + 1;
  return align256((size_t)num_recv * sizeof(int32_t)) + align256((size_t)nblocks * sizeof(int32_t)) + 256;
}

}  // extern "C"

namespace {

template <class E, class I>
int ep_combine_aggregate_t(const void* Y, const I* pos, const void* w, const I* src_rank, const I* src_token, int64_t N, int64_t H, int32_t R, void* out,
                             int32_t* run_offsets, int32_t* rank_runs, int32_t* num_runs, int32_t* status,
                             void* workspace, size_t workspace_bytes, pmx_stream_t stream) {
  if (N < 0 || H < 0 || R <= 0) return PMX_ERR_ARG;
  if (H % 8) return PMX_ERR_SHAPE;
  if (N > (int64_t)INT32_MAX) return PMX_ERR_SHAPE;
  if (!run_offsets || !rank_runs || !num_runs || !status || !workspace) return PMX_ERR_ARG;
  if (N > 0 && (!pos || !w || !src_rank || !src_token)) return PMX_ERR_ARG;
  if (N > 0 && H > 0 && (!Y || !out || !aligned16(Y) || !aligned16(out))) return PMX_ERR_ARG;
  if (workspace_bytes < pmx_ep_combine_workspace_bytes(N)) return PMX_ERR_ARG;
  int32_t* flag = reinterpret_cast<int32_t*>(workspace);
  int32_t* block_sum = reinterpret_cast<int32_t*>(reinterpret_cast<char*>(workspace) +
                                                  align256((size_t)N * sizeof(int32_t)));
  const int64_t nblocks = (N + kScanBlock - 1) / kScanBlock;
  if (N == 0) {
    // Device-side zeroing (no memset nodes, so the path can sit in a graph).
    fill_kernel<<<(unsigned)((R + 255) / 256), 256, 0, stream>>>(rank_runs, R);
    PMX_LAUNCH_CHECK();
    fill_kernel<<<1, 64, 0, stream>>>(num_runs, 1);
    PMX_LAUNCH_CHECK();
    fill_kernel<<<1, 64, 0, stream>>>(run_offsets, 1);
    PMX_LAUNCH_CHECK();
    return PMX_OK;
  }
  run_flags_kernel<<<(unsigned)nblocks, kScanBlock, 0, stream>>>(src_rank, src_token, N, flag, R, rank_runs, block_sum);
  PMX_LAUNCH_CHECK();
  scan_blocks_kernel<<<1, kScanBlock, 0, stream>>>(block_sum, nblocks, num_runs);
  PMX_LAUNCH_CHECK();
  run_offsets_kernel<<<(unsigned)nblocks, kScanBlock, 0, stream>>>(flag, block_sum, src_rank, N, R, num_runs,
                                                                   run_offsets, rank_runs, status);
  PMX_LAUNCH_CHECK();
  if (H > 0) {
    run_combine_kernel<E, I><<<(unsigned)((N + 3) / 4), 256, 0, stream>>>(static_cast<const bf16_t*>(Y), pos,
                                                        static_cast<const bf16_t*>(w), run_offsets, num_runs, H,
                                                        static_cast<bf16_t*>(out));
    PMX_LAUNCH_CHECK();
  }
  return PMX_OK;
}

}  // namespace

extern "C" {

int pmx_ep_combine_aggregate(const void* Y, const int32_t* pos, const void* w, const int32_t* src_rank,
                             const int32_t* src_token, int64_t N, int64_t H, int32_t R, void* out,
                             int32_t* run_offsets, int32_t* rank_runs, int32_t* num_runs, int32_t* status,
                             void* workspace, size_t workspace_bytes, pmx_stream_t stream) {
  return ep_combine_aggregate_t<EltBF16>(Y, pos, w, src_rank, src_token, N, H, R, out, run_offsets, rank_runs,
                                     num_runs, status, workspace, workspace_bytes, stream);
}

int pmx_ep_combine_aggregate_f16(const void* Y, const int32_t* pos, const void* w, const int32_t* src_rank,
                             const int32_t* src_token, int64_t N, int64_t H, int32_t R, void* out,
                             int32_t* run_offsets, int32_t* rank_runs, int32_t* num_runs, int32_t* status,
                             void* workspace, size_t workspace_bytes, pmx_stream_t stream) {
  return ep_combine_aggregate_t<EltF16>(Y, pos, w, src_rank, src_token, N, H, R, out, run_offsets, rank_runs,
                                     num_runs, status, workspace, workspace_bytes, stream);
}

int pmx_ep_combine_aggregate_i64(const void* Y, const int64_t* pos, const void* w, const int64_t* src_rank,
                             const int64_t* src_token, int64_t N, int64_t H, int32_t R, void* out,
                             int32_t* run_offsets, int32_t* rank_runs, int32_t* num_runs, int32_t* status,
                             void* workspace, size_t workspace_bytes, pmx_stream_t stream) {
  return ep_combine_aggregate_t<EltBF16>(Y, pos, w, src_rank, src_token, N, H, R, out, run_offsets, rank_runs,
                                     num_runs, status, workspace, workspace_bytes, stream);
}

int pmx_ep_combine_aggregate_i64_f16(const void* Y, const int64_t* pos, const void* w, const int64_t* src_rank,
                             const int64_t* src_token, int64_t N, int64_t H, int32_t R, void* out,
                             int32_t* run_offsets, int32_t* rank_runs, int32_t* num_runs, int32_t* status,
                             void* workspace, size_t workspace_bytes, pmx_stream_t stream) {
  return ep_combine_aggregate_t<EltF16>(Y, pos, w, src_rank, src_token, N, H, R, out, run_offsets, rank_runs,
                                     num_runs, status, workspace, workspace_bytes, stream);
}

}  // extern "C"
