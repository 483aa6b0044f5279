// 1-bit Hamming full-scan top-k for k above the list-based scans' 1024 (up to 8192): LiNR V3's
// candidate pools (retrieve/src/retrieve/modules/linr.py:112-162, candidate_pool = 5000 by
// default; the shortlist is oporp_1bit_match_topk_full, ops/triton/oporp_1bit_match_topk.py:
// 261-273, then torch.topk). Same result as the scan: top-k by (score desc, id asc) of
// score = 64 W - 2 popcount(q ^ item) over the items that pass the mask.
//
// A Hamming score takes only 64 W + 1 values, so the selection is a counting sort by (popcount h,
// range of ids):
//   1. count pass: each workgroup scores one contiguous range of items for its queries and
//      writes how many passing items it met at each popcount (its own row of counts: no
//      clearing, no global atomics);
//   2. prefix: per query and popcount the running sums of those counts over the ranges, in
//      place, and the totals;
//   3. cut: per query the popcount h* of the k-th best, where each popcount's entries start in
//      the result, and how many there are (kk = min(k, passing items));
//   4. emit pass: the same ranges scored again; an item with h <= h* goes to its popcount's
//      start plus its range's running sum plus an LDS counter. Ties at h* are emitted by the
//      ranges up to the one where they reach kk, whose ties may run past it;
//   5. rank: entries of one popcount and range (a cell) lie together in no order; each finds its
//      place among them by id and is written there if that is below kk.
// Two passes over the codes, whose bound is the popcounts (2 W XOR and 2 W bit counts an item
// and query) and the mask bits. Counting into one histogram a query and appending through one
// counter a query (same-address atomics, a third pass for the ties and two block sorts) took
// 516 us for 3M 128-bit codes, 16 queries at k = 5000 under a 10 % mask; these five launches take
// 108 (count 40, prefix 12, cut 4, emit 46, rank 6).
#include "scan_common.h"

namespace rt {
namespace {

constexpr int kLkThreads = 256;
constexpr int kLkWaves = kLkThreads / kWave;
constexpr int kLkQpw = 8;           // queries a workgroup scores
constexpr int kLkTiles = 2;         // 64-item tiles a wave scores together
constexpr int64_t kLkMaxRows = 8192;  // items of a range at most (its ties may overrun k)
constexpr int64_t kLkMinRows = 1024;  // and at least, where the table allows
constexpr int64_t kLkTargetWgs = 2048;
constexpr int kLkRankWalk = 64;     // entries of a cell that each of them walks
constexpr int kLkPrefixThreads = 1024;
constexpr int kLkPrefixSegs = kLkPrefixThreads / kWave;
// Counts and entries of the queries taken at a time (the others follow on the same workspace), or
// those of eight queries where they are more: at most 3.2 % of the codes' bytes and 1 MiB.
constexpr size_t kLkMaxBytes = size_t{256} << 20;

typedef __attribute__((address_space(4))) const uint32_t ku32;
typedef __attribute__((address_space(4))) const uint64_t ku64;

struct LkArgs {
  const uint64_t* q;
  int64_t B;         // queries of this batch
  const uint64_t* items;
  int64_t N;
  int64_t rows;      // items of a range, a multiple of 64
  int gx;            // ranges
  int k;
  const uint64_t* mask;
  int64_t mask_words;
  int nb;            // 64 W + 1 popcounts
  int nbp;           // a row of counts: nb rounded up to 64
  uint16_t* counts;  // [B][gx][nbp]: items of the range at a popcount, then the sums before it
  uint32_t* totals;  // [B][nbp]: items at a popcount, then its entries' start
  int32_t* cut;      // [B][4]: h* (-1: nothing passes), kk, entries emitted
  int64_t cap;       // entries of a query's buffer: k + rows
  uint64_t* buf;     // [B][cap]
};

template <int W>
__device__ inline void lk_load(const uint32_t* __restrict__ I, int64_t item, uint32_t* iw) {
  if constexpr (W % 2 == 1) {
    const uint2* p = reinterpret_cast<const uint2*>(I + item * (2 * W));
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const uint2 v = p[j];
      iw[2 * j] = v.x;
      iw[2 * j + 1] = v.y;
    }
  } else {
    const uint4* p = reinterpret_cast<const uint4*>(I + item * (2 * W));
#pragma unroll
    for (int j = 0; j < W / 2; ++j) {
      const uint4 v = p[j];
      iw[4 * j] = v.x;
      iw[4 * j + 1] = v.y;
      iw[4 * j + 2] = v.z;
      iw[4 * j + 3] = v.w;
    }
  }
}

// One range of items for kLkQpw queries. EMIT: the entries up to the cut, else the counts.
template <int W, bool EMIT>
__global__ void __launch_bounds__(kLkThreads) lk_pass_kernel(LkArgs a) {
  extern __shared__ uint32_t lh[];  // [kLkQpw][nb]: counts, or the next entry of each popcount
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t q0 = static_cast<int64_t>(blockIdx.y) * kLkQpw;
  const int nq = static_cast<int>(a.B - q0 < kLkQpw ? a.B - q0 : kLkQpw);
  const int64_t wg = blockIdx.x;
  // EMIT: the highest popcount the range emits (-1: none), and where its ties start
  __shared__ int hs[kLkQpw];
  __shared__ int first_tie[kLkQpw];
  if constexpr (EMIT) {
    for (int qi = 0; qi < nq; ++qi) {
      const int64_t q = q0 + qi;
      const int h = a.cut[q * 4];
      const int kk = a.cut[q * 4 + 1];
      const uint16_t* before = a.counts + (q * a.gx + wg) * a.nbp;
      // ties start in this range at the sums before it (saturated far above any k)
      const int tie = h < 0 ? 0 : static_cast<int>(a.totals[q * a.nbp + h] + before[h]);
      const int top = h >= 0 && tie >= kk ? h - 1 : h;
      for (int i = threadIdx.x; i <= top; i += kLkThreads) {
        lh[qi * a.nb + i] = a.totals[q * a.nbp + i] + before[i];
      }
      if (threadIdx.x == 0) {
        hs[qi] = top;
        first_tie[qi] = tie;
      }
    }
  } else {
    for (int i = threadIdx.x; i < kLkQpw * a.nb; i += kLkThreads) lh[i] = 0;
  }
  __syncthreads();
  ku32* qc = (ku32*)(a.q) + q0 * 2 * W;
  const uint32_t* I = reinterpret_cast<const uint32_t*>(a.items);
  const int64_t r0 = wg * a.rows;
  const int64_t r1 = r0 + a.rows < a.N ? r0 + a.rows : a.N;
  // waves take kLkTiles consecutive tiles in turn
  constexpr int64_t kStep = static_cast<int64_t>(kLkWaves) * kLkTiles * kWave;
  for (int64_t t0 = r0 + wave * (kLkTiles * kWave); t0 < r1; t0 += kStep) {
    uint32_t iw[kLkTiles][2 * W];
#pragma unroll
    for (int t = 0; t < kLkTiles; ++t) {
      const int64_t row = t0 + t * kWave + lane;
      lk_load<W>(I, row < r1 ? row : r1 - 1, iw[t]);
    }
    for (int qi = 0; qi < nq; ++qi) {
      uint64_t m[kLkTiles];
#pragma unroll
      for (int t = 0; t < kLkTiles; ++t) {
        // bit 63 - lane of the tile's word: the row passes (ranges are whole words)
        const int64_t left = r1 - (t0 + t * kWave);
        m[t] = left >= kWave ? ~0ull : (left > 0 ? ~(~0ull >> left) : 0ull);
      }
      if (a.mask != nullptr) {
        ku64* mrow = (ku64*)(a.mask) + (q0 + qi) * a.mask_words;
#pragma unroll
        for (int t = 0; t < kLkTiles; ++t) {
          if (m[t] != 0ull) m[t] &= mrow[(t0 >> 6) + t];
        }
      }
#pragma unroll
      for (int t = 0; t < kLkTiles; ++t) {
        if (m[t] == 0ull) continue;  // (wave-uniform)
        int h = 0;
#pragma unroll
        for (int d = 0; d < 2 * W; ++d) h = __builtin_popcount(iw[t][d] ^ qc[qi * 2 * W + d]) + h;
        const bool ok = (m[t] >> (63 - lane)) & 1ull;
        if constexpr (!EMIT) {
          if (ok) atomicAdd(&lh[qi * a.nb + h], 1u);
        } else {
          if (ok && h <= hs[qi]) {
            const uint32_t row = static_cast<uint32_t>(t0 + t * kWave + lane);
            const uint32_t pos = atomicAdd(&lh[qi * a.nb + h], 1u);
            if (pos < a.cap) {
              a.buf[(q0 + qi) * a.cap + pos] = composite(key_of_i32(64 * W - 2 * h), row);
            }
          }
        }
      }
    }
  }
  __syncthreads();
  if constexpr (EMIT) {
    // the range in which the ties reach kk knows how many entries there are
    if (threadIdx.x < nq) {
      const int qi = threadIdx.x;
      int32_t* cut = a.cut + (q0 + qi) * 4;
      const int h = cut[0];
      const int kk = cut[1];
      if (h >= 0 && hs[qi] == h) {
        const int end = static_cast<int>(lh[qi * a.nb + h]);
        if (first_tie[qi] < kk && end >= kk) cut[2] = end;
      }
    }
  } else {
    for (int qi = 0; qi < nq; ++qi) {
      uint16_t* out = a.counts + ((q0 + qi) * a.gx + wg) * a.nbp;
      for (int i = threadIdx.x; i < a.nbp; i += kLkThreads) {
        out[i] = i < a.nb ? static_cast<uint16_t>(lh[qi * a.nb + i]) : uint16_t{0};
      }
    }
  }
}

// Per query (grid y) and 64 popcounts (grid x): each range's counts become the sums before it,
// saturated at 65535 (sums that matter stay below k <= 8192), and the totals are written. A wave
// takes a segment of the ranges, a lane a popcount.
__global__ void __launch_bounds__(kLkPrefixThreads) lk_prefix_kernel(LkArgs a) {
  __shared__ uint32_t seg_sum[kLkPrefixSegs][kWave];
  const int lane = lane_id();
  const int seg = threadIdx.x >> 6;
  const int64_t q = blockIdx.y;
  const int h = blockIdx.x * kWave + lane;  // < nbp
  uint16_t* c = a.counts + q * a.gx * a.nbp + h;
  const int per = (a.gx + kLkPrefixSegs - 1) / kLkPrefixSegs;
  const int g0 = seg * per;
  const int g1 = g0 + per < a.gx ? g0 + per : a.gx;
  uint32_t sum = 0;
#pragma unroll 8
  for (int g = g0; g < g1; ++g) sum += c[static_cast<int64_t>(g) * a.nbp];
  seg_sum[seg][lane] = sum;
  __syncthreads();
  uint32_t run = 0;
  for (int s = 0; s < seg; ++s) run += seg_sum[s][lane];
  constexpr int kAhead = 8;
  for (int g = g0; g < g1; g += kAhead) {
    uint32_t v[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      v[i] = g + i < g1 ? c[static_cast<int64_t>(g + i) * a.nbp] : 0u;
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (g + i < g1) {
        c[static_cast<int64_t>(g + i) * a.nbp] =
            static_cast<uint16_t>(run < 0xffffu ? run : 0xffffu);
      }
      run += v[i];
    }
  }
  if (seg == kLkPrefixSegs - 1) a.totals[q * a.nbp + h] = run;
}

// Per query (one wave): the totals become each popcount's start (saturated: only starts up to
// h* matter), h* and kk.
__global__ void __launch_bounds__(kWave) lk_cut_kernel(LkArgs a) {
  const int64_t q = blockIdx.x;
  const int lane = lane_id();
  uint32_t* t = a.totals + q * a.nbp;
  uint64_t run = 0;
  int hs = -1;
  for (int c0 = 0; c0 < a.nbp; c0 += kWave) {
    const uint64_t v = t[c0 + lane];
    uint64_t incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint64_t y = __shfl_up(incl, off);
      incl += lane >= off ? y : 0ull;
    }
    const uint64_t before = run + incl - v;
    t[c0 + lane] = static_cast<uint32_t>(before < 0x7fffffffull ? before : 0x7fffffffull);
    // the popcount of the k-th best, or the last one that holds an item
    const uint64_t here = __ballot(v != 0ull && before < static_cast<uint64_t>(a.k));
    if (here != 0ull) hs = c0 + 63 - __builtin_clzll(here);
    run += __shfl(incl, kWave - 1);
  }
  if (lane == 0) {
    const int kk = run < static_cast<uint64_t>(a.k) ? static_cast<int>(run) : a.k;
    a.cut[q * 4] = hs;
    a.cut[q * 4 + 1] = kk;
    a.cut[q * 4 + 2] = 0;  // (the emit pass writes it where kk > 0)
  }
}

// An entry's place: its cell (entries of one popcount and range, which lie together in no order)
// starts at the sums that the emit pass started from, and it follows those of the cell that have
// lower ids. A cell of few entries is walked by each of them (random codes: one or two entries).
// Tables of many equal codes have cells of up to kLkMaxRows, where the walks are quadratic: those
// are ranked by a bitmap of the range's ids in LDS, one cell of the block's entries after another
// (at most five a block). 3M 128-bit codes, 16 queries at k = 5000, the whole call: all codes equal
// 875 us walked, 235 now (163 of it the count pass' same-address adds, 14 this kernel); random
// codes 97, 94.
__global__ void __launch_bounds__(kLkThreads) lk_rank_kernel(LkArgs a, int64_t* out_ids,
                                                             void* out_scores, int score_kind) {
  __shared__ uint32_t bits[kLkThreads];    // the cell's ids, a bit an item of the range
  __shared__ int before[kLkThreads];       // ids of the cell in the words before
  __shared__ int first[kLkWaves];
  __shared__ int part[kLkWaves];
  __shared__ int cell_at[3];               // the cell's first entry, its end, its range
  static_assert(kLkMaxRows == 32 * kLkThreads, "a thread a word of the bitmap");
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = tid >> 6;
  const int64_t q = blockIdx.y;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kLkThreads + tid;
  const int kk = a.cut[q * 4 + 1];
  const int n = a.cut[q * 4 + 2];
  auto put = [&](int64_t at, int64_t id, int32_t score, bool pad) {
    out_ids[q * a.k + at] = id;
    if (score_kind == kScoreI32) {
      static_cast<int32_t*>(out_scores)[q * a.k + at] = pad ? INT32_MIN : score;
    } else {
      static_cast<float*>(out_scores)[q * a.k + at] =
          pad ? -INFINITY : static_cast<float>(score);
    }
  };
  if (i >= kk && i < a.k) put(i, -1, 0, true);
  if (i - tid >= n) return;  // (the whole block)
  const bool have = i < n;
  const uint64_t* e = a.buf + q * a.cap;
  const uint64_t c = have ? e[i] : 0ull;
  const uint32_t rows = static_cast<uint32_t>(a.rows);
  const uint32_t id = have ? composite_item(c) : 0u;
  const int cell = static_cast<int>(id / rows);
  const int32_t score = have ? i32_of_key(composite_key(c)) : 0;
  int s0 = 0;
  int s1 = 0;
  if (have) {
    const int h = (a.nb - 1 - score) / 2;
    const uint32_t* starts = a.totals + q * a.nbp + h;
    const uint16_t* sums = a.counts + (q * a.gx + cell) * a.nbp + h;
    s0 = static_cast<int>(starts[0] + sums[0]);
    // (saturated sums and starts lie past n)
    const uint32_t end = cell + 1 < a.gx ? starts[0] + sums[a.nbp]
                                         : (h + 1 < a.nb ? starts[1] : 0x7fffffffu);
    s1 = end < static_cast<uint32_t>(n) ? static_cast<int>(end) : n;
  }
  int at = s0;
  bool pending = s1 - s0 > kLkRankWalk;
  if (!pending) {
    for (int j = s0; j < s1; ++j) at += e[j] > c ? 1 : 0;  // (greater composite: lower id)
  }
  while (true) {
    // the first entry that is not placed yet names the cell
    const uint64_t bal = __ballot(pending);
    if (lane == 0) first[wave] = bal != 0ull ? tid + __builtin_ctzll(bal) : kLkThreads;
    __syncthreads();
    int f = kLkThreads;
#pragma unroll
    for (int w = 0; w < kLkWaves; ++w) f = first[w] < f ? first[w] : f;
    if (f == kLkThreads) break;  // (the whole block)
    if (tid == f) {
      cell_at[0] = s0;
      cell_at[1] = s1;
      cell_at[2] = cell;
    }
    bits[tid] = 0u;
    __syncthreads();
    const uint32_t id0 = static_cast<uint32_t>(cell_at[2]) * rows;
    for (int j = cell_at[0] + tid; j < cell_at[1]; j += kLkThreads) {
      const uint32_t off = composite_item(e[j]) - id0;
      atomicOr(&bits[off >> 5], 1u << (off & 31u));
    }
    __syncthreads();
    const int own = __builtin_popcount(bits[tid]);
    int incl = own;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int y = __shfl_up(incl, off);
      incl += lane >= off ? y : 0;
    }
    if (lane == kWave - 1) part[wave] = incl;
    __syncthreads();
    int base = incl - own;
    for (int w = 0; w < wave; ++w) base += part[w];
    before[tid] = base;
    __syncthreads();
    if (pending && s0 == cell_at[0]) {
      const uint32_t off = id - id0;
      at = s0 + before[off >> 5] +
           __builtin_popcount(bits[off >> 5] & ((1u << (off & 31u)) - 1u));
      pending = false;
    }
    __syncthreads();  // (read before the next cell's replace them)
  }
  if (have && at < kk) put(at, id, score, false);
}

struct LkPlan {
  int64_t rows, gx, nbp, cap, batch;
  size_t totals, cut, counts, buf, total;
};

LkPlan lk_plan(int64_t B, int64_t N, int64_t W, int64_t k) {
  LkPlan p{};
  const int64_t gy = cdiv(B, kLkQpw);
  // ranges of at most kLkMaxRows items, and enough of them to fill the GPU where they stay
  // above kLkMinRows
  int64_t gx = cdiv(kLkTargetWgs, gy);
  const int64_t most = cdiv(N, kLkMinRows);
  gx = gx < most ? gx : most;
  const int64_t least = cdiv(N, kLkMaxRows);
  gx = gx > least ? gx : least;
  p.rows = cdiv(cdiv(N, gx), kWave) * kWave;
  p.gx = cdiv(N, p.rows);
  p.nbp = cdiv(64 * W + 1, kWave) * kWave;
  p.cap = k + p.rows;
  const size_t per = static_cast<size_t>(p.gx * p.nbp) * sizeof(uint16_t) +
                     static_cast<size_t>(p.cap) * sizeof(uint64_t);
  p.batch = static_cast<int64_t>(kLkMaxBytes / per) / kLkQpw * kLkQpw;
  p.batch = p.batch < kLkQpw ? kLkQpw : p.batch;
  p.batch = p.batch < B ? p.batch : B;
  p.totals = 0;
  p.cut = align_up(static_cast<size_t>(p.batch * p.nbp) * sizeof(uint32_t), 256);
  p.counts = p.cut + align_up(static_cast<size_t>(p.batch) * 16, 256);
  p.buf = p.counts + align_up(static_cast<size_t>(p.batch * p.gx * p.nbp) * sizeof(uint16_t), 256);
  p.total = p.buf + static_cast<size_t>(p.batch * p.cap) * sizeof(uint64_t);
  return p;
}

template <int W>
int lk_dispatch(int64_t w, const LkArgs& a, dim3 grid, hipStream_t stream, bool emit) {
  if (w == W) {
    const size_t lds = static_cast<size_t>(kLkQpw) * a.nb * sizeof(uint32_t);
    if (emit) {
      lk_pass_kernel<W, true><<<grid, kLkThreads, lds, stream>>>(a);
    } else {
      lk_pass_kernel<W, false><<<grid, kLkThreads, lds, stream>>>(a);
    }
    RT_CHECK_HIP(hipGetLastError());
    return kOk;
  }
  if constexpr (W < 16) {
    return lk_dispatch<W + 1>(w, a, grid, stream, emit);
  } else {
    set_error("Hamming scan supports W in [1, 16], got %lld", static_cast<long long>(w));
    return kInvalidArgument;
  }
}

}  // namespace

size_t hamming_large_k_workspace(int64_t B, int64_t N, int64_t W, int64_t k) {
  if (B <= 0 || N <= 0 || W <= 0) return 256;
  return lk_plan(B, N, W, k).total;
}

int hamming_large_k(const uint64_t* query_bits, int64_t B, const uint64_t* item_bits, int64_t N,
                    int64_t W, int64_t k, const uint64_t* mask, int64_t mask_words,
                    int64_t* out_ids, void* out_scores, int score_kind, void* workspace,
                    size_t workspace_bytes, hipStream_t stream) {
  RT_CHECK_ARG(k > kMaxK && k <= kMaxKHamming, "k must be in (%lld, %lld] here",
               static_cast<long long>(kMaxK), static_cast<long long>(kMaxKHamming));
  const LkPlan p = lk_plan(B, N, W, k);
  if (workspace_bytes < p.total) {
    set_error("workspace too small: %zu < %zu", workspace_bytes, p.total);
    return kWorkspaceTooSmall;
  }
  RT_CHECK_ARG(p.gx < (int64_t{1} << 31), "N too large");
  char* ws = static_cast<char*>(workspace);
  const int64_t elem = score_kind == kScoreI32 ? sizeof(int32_t) : sizeof(float);
  for (int64_t b0 = 0; b0 < B; b0 += p.batch) {
    LkArgs a{};
    a.q = query_bits + b0 * W;
    a.B = B - b0 < p.batch ? B - b0 : p.batch;
    a.items = item_bits;
    a.N = N;
    a.rows = p.rows;
    a.gx = static_cast<int>(p.gx);
    a.k = static_cast<int>(k);
    a.mask = mask != nullptr ? mask + b0 * mask_words : nullptr;
    a.mask_words = mask_words;
    a.nb = static_cast<int>(64 * W + 1);
    a.nbp = static_cast<int>(p.nbp);
    a.counts = reinterpret_cast<uint16_t*>(ws + p.counts);
    a.totals = reinterpret_cast<uint32_t*>(ws + p.totals);
    a.cut = reinterpret_cast<int32_t*>(ws + p.cut);
    a.cap = p.cap;
    a.buf = reinterpret_cast<uint64_t*>(ws + p.buf);
    const int64_t gy = cdiv(a.B, kLkQpw);
    RT_CHECK_ARG(gy <= 65535 && a.B <= 65535, "too many queries");
    const dim3 grid(static_cast<unsigned>(p.gx), static_cast<unsigned>(gy));
    int st = lk_dispatch<1>(W, a, grid, stream, false);
    if (st != kOk) return st;
    lk_prefix_kernel<<<dim3(static_cast<unsigned>(p.nbp / kWave), static_cast<unsigned>(a.B)),
                       kLkPrefixThreads, 0, stream>>>(a);
    RT_CHECK_HIP(hipGetLastError());
    lk_cut_kernel<<<static_cast<unsigned>(a.B), kWave, 0, stream>>>(a);
    RT_CHECK_HIP(hipGetLastError());
    st = lk_dispatch<1>(W, a, grid, stream, true);
    if (st != kOk) return st;
    lk_rank_kernel<<<dim3(static_cast<unsigned>(cdiv(p.cap, kLkThreads)),
                          static_cast<unsigned>(a.B)),
                     kLkThreads, 0, stream>>>(a, out_ids + b0 * k,
                                              static_cast<char*>(out_scores) + b0 * k * elem,
                                              score_kind);
    RT_CHECK_HIP(hipGetLastError());
  }
  return kOk;
}

}  // namespace rt
