// SilverTorch's search after phase 1 (silvertorch/.../ops/csrc/fork_search_cuda.cu:1256-1524):
// query quantization, the int8 scorer over each query's probed clusters, the selection by
// (key desc, slot asc) and the epilogue id = sort_perm[position], score = dequantized dot.
//
// Slots: query row b's probed clusters c_j = probe_ids[b, j] hold the items at sorted positions
// cluster_offsets[c_j] .. + cluster_sizes[c_j]. The row's slots are the reference scorer's write
// order: the full 32-item warps of every probed cluster in probe order, then every cluster's
// remaining (< 32) items in probe order (fork_search_cuda.cu:989-991 and :1051-1053;
// fused_kmean_ann_cuda.cu:592-598 and :443-453). Ties go to the lower slot. The row holds at most
// `width` slots (max_tensor_size_per_row rounded up to 32, as the reference's score buffer); the
// reference requires a row's clusters to fit its width, and slots at or past it are dropped here.
// A filtered-out item keeps its slot (the scorer skips it), so the filter never renumbers slots.
//
// Keys: the int32 dot (divisor -1), or the fp16 score fp16(float(dot) / divisor) of the serving
// path (index_mm_helpers.cuh:48-65), ordered as fp16 values (ties merge distinct dots).
//
// The range scan filters 64 slots of a wave at a time and queues the ones that pass; queued rows
// are scored by groups of lanes, several rows in flight a group; every wave keeps a candidate
// list under a rising threshold; the shared merge picks the k best composites.
#include "scan_common.h"
#include "wave_lists.h"

namespace rt {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kQuantThreads = 256;
constexpr int64_t kQuantMaxGrid = 4096;  // sixteen workgroups a CU: two rounds of eight
constexpr int kIvfThreads = 256;
constexpr int kIvfWaves = kIvfThreads / kWave;
constexpr int kIvfMaxProbe = 1024;
constexpr int kIvfMaxWgsPerRow = 256;

// ---- query quantization (A1 / A2) ------------------------------------------------------------

// Per row: abs_max = max(max |x|, 1e-8); scale = abs_max * fp32(1/127); code =
// clamp(rint(fp32(fp64(x) / fp64(abs_max)) * 127), -128, 127) (fork_search_cuda.cu:680-699;
// retrieve/src/retrieve/indexing/quantize.py:9-18).
// scale_div: scales = abs_max / 127 (quantize_int8, indexing/quantize.py:9-18); else
// abs_max * fp32(1/127) (probe_prep_kernel, fork_search_cuda.cu:689). The codes are the same.
//
// The quotient is one fp32 division: the fp64 quotient of two fp32 values rounded to fp32 is the
// correctly rounded fp32 quotient (53 >= 2 * 24 + 2 bits, so the double rounding is harmless)
// but for results below the normal range, whose codes are 0 either way.
__device__ inline int8_t code_of(float x, float abs_max) {
  const float v = (x / abs_max) * 127.0f;
  return static_cast<int8_t>(fminf(fmaxf(rintf(v), -128.0f), 127.0f));
}

__device__ inline float row_scale(float abs_max, int scale_div) {
  return scale_div ? abs_max / 127.0f : abs_max * (1.0f / 127.0f);
}

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int8_t v4c __attribute__((ext_vector_type(4)));

// Four codes of one lane.
__device__ inline v4c codes_of(v4f x, float abs_max) {
  return v4c{code_of(x[0], abs_max), code_of(x[1], abs_max), code_of(x[2], abs_max),
             code_of(x[3], abs_max)};
}

// Any row length and alignment, one workgroup per row, the row read twice.
__global__ void __launch_bounds__(kQuantThreads) quantize_rows_kernel(const float* x,
                                                                      int64_t dim, int8_t* codes,
                                                                      float* scales,
                                                                      int scale_div) {
  __shared__ float red[kQuantThreads / kWave];
  const int64_t row = blockIdx.x;
  const float* xr = x + row * dim;
  float m = 0.f;
  for (int64_t d = threadIdx.x; d < dim; d += kQuantThreads) m = fmaxf(m, fabsf(xr[d]));
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if (lane_id() == 0) red[threadIdx.x / kWave] = m;
  __syncthreads();
  m = red[0];
  for (int w = 1; w < kQuantThreads / kWave; ++w) m = fmaxf(m, red[w]);
  m = fmaxf(m, 1e-8f);
  if (threadIdx.x == 0) scales[row] = row_scale(m, scale_div);
  int8_t* out = codes + row * dim;
  for (int64_t d = threadIdx.x; d < dim; d += kQuantThreads) out[d] = code_of(xr[d], m);
}

// Rows of whole 16-byte chunks at 16-byte alignment, at most kQuantMaxChunks chunks a lane: L
// lanes hold a row in registers (chunk c of lane l is floats 4 (c L + l) .. + 3), so it is read
// once, and the groups of a wave take 64 / L neighbouring rows, whose loads and stores are
// contiguous. HBM-bound (5 bytes a value): 3M x 128 in 0.38 ms, 5.0 TB/s. The general kernel
// above spends a workgroup and two barriers on each row and took 2.00 ms.
constexpr int kQuantMaxChunks = 8;

template <int L, int NC>
__global__ void __launch_bounds__(kQuantThreads) quantize_rows_vec_kernel(
    const float* __restrict__ x, int64_t rows, int dim, int8_t* __restrict__ codes,
    float* __restrict__ scales, int scale_div) {
  constexpr int R = kQuantThreads / L;  // rows a workgroup takes at a time
  const int gl = threadIdx.x % L;
  const int chunks = dim / 4;
  const int64_t step = static_cast<int64_t>(gridDim.x) * R;
  int64_t row = static_cast<int64_t>(blockIdx.x) * R + threadIdx.x / L;
  v4f v[NC];
  auto load = [&](int64_t r) {
    const v4f* src = reinterpret_cast<const v4f*>(x + r * dim);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int i = c * L + gl;
      v[c] = r < rows && i < chunks ? __builtin_nontemporal_load(src + i) : v4f{0.f, 0.f, 0.f, 0.f};
    }
  };
  load(row);
  while (row < rows) {
    v4f cur[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) cur[c] = v[c];
    load(row + step);  // in flight while this row is coded
    float m = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
#pragma unroll
      for (int e = 0; e < 4; ++e) m = fmaxf(m, fabsf(cur[c][e]));
    }
#pragma unroll
    for (int off = L / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    m = fmaxf(m, 1e-8f);
    if (gl == 0) scales[row] = row_scale(m, scale_div);
    v4c* out = reinterpret_cast<v4c*>(codes + row * dim);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int i = c * L + gl;
      if (i < chunks) out[i] = codes_of(cur[c], m);
    }
    row += step;
  }
}

template <int L, int NC>
static void launch_quantize_vec(const float* x, int64_t rows, int64_t dim, int8_t* codes,
                                float* scales, int scale_div, hipStream_t stream) {
  const int64_t want = cdiv(rows, kQuantThreads / L);
  const unsigned grid = static_cast<unsigned>(want < kQuantMaxGrid ? want : kQuantMaxGrid);
  quantize_rows_vec_kernel<L, NC><<<grid, kQuantThreads, 0, stream>>>(
      x, rows, static_cast<int>(dim), codes, scales, scale_div);
}

// One scale for the whole table (quantize_int8_global, retrieve/src/retrieve/indexing/quantize.py:
// 25-52): abs_max = max(max x, -min x) floored at 1e-8 (fabsf's maximum, the same value), code
// = clamp(rint(fp32(x / abs_max) * 127), -128, 127) in fp32, row i of the codes from row
// perm[i] of x when a permutation is given. NaN inputs are outside the contract (max ignores
// them here; the reference's int8 cast of a NaN code is unspecified).
constexpr int kGlobalThreads = 256;

__global__ void abs_max_init_kernel(uint32_t* bits) { bits[0] = 0u; }

// Grid-stride max |x| over n floats, 16-byte loads when x is 16-byte aligned; one atomic per
// workgroup on the bits of the (non-negative) float, whose unsigned order is the float order.
__global__ void __launch_bounds__(kGlobalThreads) abs_max_kernel(const float* x, int64_t n,
                                                                 uint32_t* bits) {
  __shared__ float red[kGlobalThreads / kWave];
  float m = 0.f;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kGlobalThreads;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kGlobalThreads + threadIdx.x;
  if (reinterpret_cast<uintptr_t>(x) % 16 == 0) {
    const v4f* x4 = reinterpret_cast<const v4f*>(x);
    const int64_t n4 = n / 4;
    for (int64_t i = t0; i < n4; i += stride) {
      const v4f v = __builtin_nontemporal_load(x4 + i);
      m = fmaxf(fmaxf(m, fmaxf(fabsf(v[0]), fabsf(v[1]))), fmaxf(fabsf(v[2]), fabsf(v[3])));
    }
    for (int64_t i = 4 * n4 + t0; i < n; i += stride) m = fmaxf(m, fabsf(x[i]));
  } else {
    for (int64_t i = t0; i < n; i += stride) m = fmaxf(m, fabsf(x[i]));
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if (lane_id() == 0) red[threadIdx.x / kWave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kGlobalThreads / kWave; ++w) m = fmaxf(m, red[w]);
    atomicMax(bits, __float_as_uint(m));
  }
}

// Any row length and alignment, one value a thread at a time.
__global__ void __launch_bounds__(kGlobalThreads) quantize_global_kernel(
    const float* x, int64_t rows, int64_t dim, const int64_t* perm, const uint32_t* bits,
    int8_t* codes, float* abs_max_out) {
  const float m = fmaxf(__uint_as_float(bits[0]), 1e-8f);
  const int64_t total = rows * dim;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kGlobalThreads;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kGlobalThreads + threadIdx.x;
  if (t0 == 0) abs_max_out[0] = m;
  for (int64_t i = t0; i < total; i += stride) {
    const int64_t r = i / dim;
    const int64_t c = i - r * dim;
    const int64_t src = perm != nullptr ? perm[r] : r;
    codes[i] = code_of(x[src * dim + c], m);
  }
}

// Rows of whole 16-byte chunks at 16-byte alignment: L lanes take a row, NC chunks each, as
// quantize_rows_vec_kernel's do, with the next row's chunks and the source index of the one
// after it in flight, so a permuted read waits for neither. HBM-bound (5 bytes a value and the
// permutation): 3M x 128 in a random order in 0.41 ms, 4.8 TB/s. One value a thread, each with
// a 64-bit division for its row, took 0.93 ms.
template <int L, int NC>
__global__ void __launch_bounds__(kGlobalThreads) quantize_global_vec_kernel(
    const float* __restrict__ x, int64_t rows, int dim, const int64_t* __restrict__ perm,
    const uint32_t* __restrict__ bits, int8_t* __restrict__ codes, float* abs_max_out) {
  constexpr int R = kGlobalThreads / L;
  const float m = fmaxf(__uint_as_float(bits[0]), 1e-8f);
  if (blockIdx.x == 0 && threadIdx.x == 0) abs_max_out[0] = m;
  const int gl = threadIdx.x % L;
  const int chunks = dim / 4;
  const int64_t step = static_cast<int64_t>(gridDim.x) * R;
  int64_t row = static_cast<int64_t>(blockIdx.x) * R + threadIdx.x / L;
  auto source = [&](int64_t r) { return r >= rows ? -1 : (perm != nullptr ? perm[r] : r); };
  v4f v[NC];
  auto load = [&](int64_t src_row) {
    const v4f* src = reinterpret_cast<const v4f*>(x + src_row * dim);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int i = c * L + gl;
      v[c] = src_row >= 0 && i < chunks ? __builtin_nontemporal_load(src + i)
                                        : v4f{0.f, 0.f, 0.f, 0.f};
    }
  };
  load(source(row));
  int64_t next = source(row + step);
  while (row < rows) {
    v4f cur[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) cur[c] = v[c];
    load(next);
    next = source(row + 2 * step);
    v4c* out = reinterpret_cast<v4c*>(codes + row * dim);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int i = c * L + gl;
      if (i < chunks) out[i] = codes_of(cur[c], m);
    }
    row += step;
  }
}

template <int L, int NC>
static void launch_quantize_global_vec(const float* x, int64_t rows, int64_t dim,
                                       const int64_t* perm, const uint32_t* bits, int8_t* codes,
                                       float* abs_max, hipStream_t stream) {
  const int64_t want = cdiv(rows, kGlobalThreads / L);
  const unsigned grid = static_cast<unsigned>(want < kQuantMaxGrid ? want : kQuantMaxGrid);
  quantize_global_vec_kernel<L, NC><<<grid, kGlobalThreads, 0, stream>>>(
      x, rows, static_cast<int>(dim), perm, bits, codes, abs_max);
}

// Sign bits of float rows, LSB-first: bit b of word w of row r is x[r, 64 w + b] > 0
// (_pack_signs_to_int64, retrieve/src/retrieve/indexing/quantize.py:63-72). One wave per word:
// lane b reads element 64 w + b and the ballot is the word (NaN and -0 give 0 bits, as the
// reference's comparison does).
__global__ void __launch_bounds__(256) pack_signs_kernel(const float* x, int64_t words_total,
                                                         uint64_t* words) {
  const int64_t w = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) / kWave;
  if (w >= words_total) return;  // whole waves
  const bool pos = x[w * kWave + lane_id()] > 0.0f;
  const uint64_t word = __ballot(pos);
  if (lane_id() == 0) words[w] = word;
}

// Sign-OPORP codes with one dimension a bin: bit b of word w of row r is set where, for
// p = perm[64 w + b], (x[r, p] * signs[p]) / max(norm, 1e-8) > 0 with norm the fp32 2-norm of the
// row's products (indexing/quantize.py:97-140; a NaN anywhere in the row makes every bit 0, an
// infinite norm those of the finite values). A quotient of positive floats rounds to 0 only at
// or below 2^-150, so it is above 0 iff x * sign > floor(norm / 2) * 2^-149: a compare, no
// division.
//
// L lanes hold a row in registers, NC 16-byte chunks each; each of the 4 NC components of a lane
// gives one ballot over the wave's 64 / L rows, kept in LDS, and an output bit is bit `lane` of
// the ballot that holds its permuted dimension (`src`, from perm once a workgroup), so the
// gather moves single bits and x is read once in order. HBM-bound (4 bytes a value): 3M x 128 in
// 0.37 ms, 4.3 TB/s. Composed of a product, an index_select, a sum, a norm, a division and the
// packing it took 4.0 ms in 46 chunks of launches.
constexpr int kOporpThreads = 256;
constexpr int kOporpMaxChunks = 8;
constexpr int kOporpMaxDim = 4 * kWave * kOporpMaxChunks;

template <int L, int NC, bool VEC>
__global__ void __launch_bounds__(kOporpThreads) pack_oporp_kernel(
    const float* __restrict__ x, int64_t rows, int dim, const int8_t* __restrict__ signs,
    const int64_t* __restrict__ perm, uint64_t* __restrict__ words) {
  constexpr int R = kWave / L;        // rows a wave takes at a time
  constexpr int kWaves = kOporpThreads / kWave;
  __shared__ uint16_t src[4 * L * NC];  // output bit -> ballot << 6 | lane of the row
  __shared__ uint64_t bal[kWaves][4 * NC];
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  const int gl = lane % L;
  const int chunks = dim / 4;
  const int W = dim / 64;
  for (int i = threadIdx.x; i < dim; i += kOporpThreads) {
    int64_t p = perm[i];
    p = p < 0 ? 0 : (p < dim ? p : dim - 1);  // (a permutation: kept inside the row regardless)
    const int chunk = static_cast<int>(p) / 4;
    src[i] = static_cast<uint16_t>(((chunk / L * 4 + static_cast<int>(p) % 4) << 6) | chunk % L);
  }
  v4f sg[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = c * L + gl;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sg[c][e] = i < chunks ? static_cast<float>(signs[4 * i + e]) : 0.f;
    }
  }
  __syncthreads();
  const int64_t step = static_cast<int64_t>(gridDim.x) * kWaves * R;
  int64_t row0 = (static_cast<int64_t>(blockIdx.x) * kWaves + wave) * R;
  v4f v[NC];
  auto load = [&](int64_t r) {
    const float* src_row = x + r * dim;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int i = c * L + gl;
      v[c] = v4f{0.f, 0.f, 0.f, 0.f};
      if (r < rows && i < chunks) {
        if constexpr (VEC) {
          v[c] = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(src_row) + i);
        } else {
          const v4f u = {src_row[4 * i], src_row[4 * i + 1], src_row[4 * i + 2],
                         src_row[4 * i + 3]};
          v[c] = u;
        }
      }
    }
  };
  load(row0 + lane / L);
  for (; row0 < rows; row0 += step) {
    v4f y[NC];
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[c][e] = v[c][e] * sg[c][e];
        ss = __builtin_fmaf(y[c][e], y[c][e], ss);
      }
    }
    load(row0 + step + lane / L);  // in flight while these rows are packed
#pragma unroll
    for (int off = L / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    const float norm = sqrtf(ss);
    // (norm below 2: 0, every positive product counts; NaN stays NaN and passes nothing)
    const float t = floorf((norm < 1e-8f ? 1e-8f : norm) * 0.5f) * 0x1p-149f;
    uint64_t mine = 0ull;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint64_t b = __ballot(y[c][e] > t);
        mine = lane == 4 * c + e ? b : mine;
      }
    }
    if (lane < 4 * NC) bal[wave][lane] = mine;
    wave_sync_memory();
    uint64_t out = 0ull;
    for (int r = 0; r < R; ++r) {
      for (int w = 0; w < W; ++w) {
        const int s = src[64 * w + lane];
        const uint64_t word = __ballot((bal[wave][s >> 6] >> (r * L + (s & 63))) & 1ull);
        out = lane == r * W + w ? word : out;
      }
    }
    if (lane < R * W && row0 + lane / W < rows) words[row0 * W + lane] = out;
    wave_sync_memory();  // (the ballots are read before the next rows' replace them)
  }
}

template <int L, int NC>
static void launch_pack_oporp(const float* x, int64_t rows, int dim, const int8_t* signs,
                              const int64_t* perm, uint64_t* words, hipStream_t stream) {
  const int64_t want = cdiv(rows, (kOporpThreads / kWave) * (kWave / L));
  const unsigned grid = static_cast<unsigned>(want < kQuantMaxGrid ? want : kQuantMaxGrid);
  if (reinterpret_cast<uintptr_t>(x) % 16 == 0) {
    pack_oporp_kernel<L, NC, true><<<grid, kOporpThreads, 0, stream>>>(x, rows, dim, signs, perm,
                                                                       words);
  } else {
    pack_oporp_kernel<L, NC, false><<<grid, kOporpThreads, 0, stream>>>(x, rows, dim, signs, perm,
                                                                        words);
  }
}

// ---- range scan ------------------------------------------------------------------------------

struct IvfArgs {
  const int8_t* q;  // [B, RB] codes
  int64_t B;
  const int8_t* items;  // [N, RB]
  int64_t N;
  int RB;
  const int64_t* probe_ids;  // [B, n_probe]
  int64_t n_probe;
  const int64_t* cluster_offsets;  // [n_lists]
  const int64_t* cluster_sizes;    // [n_lists]
  int64_t n_lists;
  int64_t width;
  const uint64_t* mask;  // [B, mask_words], item position d at bit 63 - d % 64, or null
  int64_t mask_words;
  // or the probed payloads' Bloom words (rt_bloom_search_columns' layout): entry e = b * n_probe
  // + j covers probe j's docs from bit pfirst[e] of words pcum[e - 1] ... (null: none)
  const int32_t* pcum;
  const int8_t* pfirst;
  const uint64_t* pwords;
  int64_t p_entries;
  int64_t p_words;
  // and / or the exact clauses in the slot layout (slots [R, N] int32, clause c in rows
  // cslots[c] .. cslots[c + 1], query values qv [B, C], -1 inactive; null: none)
  const int32_t* slots;
  int64_t R;
  const int64_t* cslots;
  int C;
  const int8_t* reverse;  // [C], non-zero: a reverse clause
  const int32_t* qv;
  int divisor;  // -1: int32 keys
  int k;
  int capw;
  uint64_t* lists;
  int* list_counts;
};

constexpr int kIvfMaxClauses = 32;
constexpr int kIvfUnroll = 4;  // 64-slot steps a wave filters together
constexpr int kIvfQueue = kIvfUnroll * kWave + kWave;  // a step's slots and an unscored rest

// The row's 2 n_probe slot ranges in slot order: range j < n_probe is probe j's full warps
// (its first len_j / 32 * 32 items), range n_probe + j probe j's remaining len_j % 32 items.
// start[r] is range r's first sorted position and prefix[r] the slots before it (prefix[2n] =
// total, clamped at width). Invalid clusters, or clusters reaching outside the table, are empty.
// The lengths are summed by a block scan (a serial sum over 2 n_probe LDS entries took longer
// than a workgroup's scoring). `part` holds kIvfThreads / kWave int64.
__device__ inline uint32_t load_ranges(const IvfArgs& a, int64_t b, int64_t* start,
                                       uint32_t* prefix, int64_t* part) {
  const int tid = threadIdx.x;
  const int np = static_cast<int>(a.n_probe);
  const int nr = 2 * np;
  for (int j = tid; j < np; j += kIvfThreads) {
    const int64_t c = a.probe_ids[b * np + j];
    int64_t s = 0;
    int64_t len = 0;
    if (c >= 0 && c < a.n_lists) {
      s = a.cluster_offsets[c];
      len = a.cluster_sizes[c];
      if (s < 0 || len < 0 || s > a.N || len > a.N - s) len = 0;
    }
    // (a range longer than the width ends the row either way)
    const int64_t full = len / 32 * 32;
    start[j] = s;
    prefix[j + 1] = static_cast<uint32_t>(full < a.width ? full : a.width);
    start[np + j] = s + full;
    prefix[np + j + 1] = static_cast<uint32_t>(len - full);
  }
  __syncthreads();
  // each thread takes a run of lengths, then the runs' sums are scanned across the block
  const int per = (nr + kIvfThreads - 1) / kIvfThreads;
  int64_t run = 0;
  for (int i = 0; i < per; ++i) {
    const int r = tid * per + i;
    if (r < nr) run += prefix[r + 1];
  }
  int64_t incl = run;
  const int lane = lane_id();
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int64_t t = __shfl_up(incl, off);
    incl += lane >= off ? t : 0;
  }
  if (lane == kWave - 1) part[tid / kWave] = incl;
  __syncthreads();
  int64_t sum = incl - run;
  for (int w = 0; w < tid / kWave; ++w) sum += part[w];
  for (int i = 0; i < per; ++i) {
    const int r = tid * per + i;
    if (r < nr) {
      sum += prefix[r + 1];
      prefix[r + 1] = static_cast<uint32_t>(sum < a.width ? sum : a.width);
    }
  }
  if (tid == 0) prefix[0] = 0;
  __syncthreads();
  return prefix[nr];
}

// LDS bytes of a row's ranges (start[2 n], the scan's partial sums, prefix[2 n + 1]), rounded to
// whole 16-byte chunks.
__host__ __device__ inline size_t ranges_lds(int64_t n_probe) {
  return (static_cast<size_t>(2 * n_probe + kIvfWaves) * sizeof(int64_t) +
          static_cast<size_t>(2 * n_probe + 1) * sizeof(uint32_t) + 15) / 16 * 16;
}

// the range holding slot s: the last j with prefix[j] <= s
__device__ inline int range_of(const uint32_t* prefix, int n, uint32_t s) {
  int lo = 0;
  int hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (prefix[mid] <= s) {
      lo = mid;
    } else {
      hi = mid - 1;
    }
  }
  return lo;
}

__device__ inline uint32_t search_key(int32_t dot, int divisor) {
  if (divisor == -1) return key_of_i32(dot);
  const _Float16 h = static_cast<_Float16>(static_cast<float>(dot) / static_cast<float>(divisor));
  return key_of_f32(static_cast<float>(h));
}

// The row's active exact clauses (LDS): value, slot rows [r0, r1) inside the table, reverse. A
// doc passes a clause when one of its values equals the query's, negated for a reverse clause
// (fork_filters.cuh:15-41).
struct IvfClauses {
  int n;
  int32_t value[kIvfMaxClauses];
  int32_t reverse[kIvfMaxClauses];
  int64_t r0[kIvfMaxClauses];
  int64_t r1[kIvfMaxClauses];
};

// Fills the row's clauses in clause order; called by the block, followed by a barrier.
__device__ inline void load_clauses(const IvfArgs& a, int64_t b, IvfClauses* cl) {
  const int tid = threadIdx.x;
  if (tid >= kWave) return;
  const bool have = a.qv != nullptr && tid < a.C;
  const int32_t v = have ? a.qv[b * a.C + tid] : -1;
  const uint64_t active = __ballot(v != -1);
  if (v != -1) {
    const int i = __popcll(active & ((1ull << tid) - 1ull));
    cl->value[i] = v;
    cl->reverse[i] = a.reverse[tid] != 0;
    const int64_t r0 = a.cslots[tid];
    const int64_t r1 = a.cslots[tid + 1];
    cl->r0[i] = r0 > 0 ? r0 : 0;
    cl->r1[i] = r1 < a.R ? r1 : a.R;
  }
  if (tid == 0) cl->n = __popcll(active);
}

// The LDS of a scan workgroup beside the ranges.
struct IvfLds {
  int64_t qpos[kIvfWaves][kIvfQueue];  // per wave: sorted positions of the slots that passed
  uint32_t qslot[kIvfWaves][kIvfQueue];
  IvfClauses clauses;
  int cnt[kIvfWaves];
};

__host__ __device__ constexpr size_t ivf_lds_bytes() { return (sizeof(IvfLds) + 15) / 16 * 16; }

// One workgroup's share of a row's slots. Each wave takes one contiguous run of them: the range
// of a slot is found once by bisection and then only walked forward. kIvfUnroll x 64 slots a
// step are filtered lane by lane (neighbouring slots are neighbouring docs, so their mask words
// and attribute rows coalesce, kIvfUnroll loads in flight a lane), and those that pass are
// queued in LDS; then the queue is scored R * V rows at a time: a group of L lanes holds the
// query's chunks and loads V rows of NC 16-byte chunks a lane before it uses the first, and V
// partial dots are folded across the lanes by halves (each exchange hands half of the values to
// the other lane), so a lane ends with one row's dot. Bound: the latency of the dependent loads
// (filter, then row), hidden by the rows in flight and three to five workgroups a CU (81
// to 144 registers; the LDS of a full list's sort allows one at k = 1000). Docs that the
// filter drops cost no row load and no reduction, and plain (not streaming) loads keep rows that
// other queries of the batch probe in the caches. Filtering and scoring one slot a group step by
// step, the same scans took (before, now): 3M x 128, 64 queries of 64 probes in 1024 lists under
// the exact filter 992, 80 us; 10M x 256, 16 queries of 128 probes in 4096 lists under Bloom
// words and the recheck 917, 56 us; unfiltered 2M x 512, 16 queries, the whole search 587, 301.
template <int L, int NC, int V>
__global__ void __launch_bounds__(kIvfThreads) ivf_scan_kernel(IvfArgs a) {
  constexpr int R = kWave / L;
  constexpr int E = R * V;  // rows scored at a time
  static_assert(V <= L && E <= kWave, "a lane owns at most one of the rows scored together");
  extern __shared__ __attribute__((aligned(16))) uint64_t smem[];
  const int nr = static_cast<int>(2 * a.n_probe);  // slot ranges
  int64_t* start = reinterpret_cast<int64_t*>(smem);
  int64_t* part = start + nr;
  uint32_t* prefix = reinterpret_cast<uint32_t*>(part + kIvfWaves);
  char* after = reinterpret_cast<char*>(smem) + ranges_lds(a.n_probe);
  IvfLds* lds = reinterpret_cast<IvfLds*>(after);
  uint64_t* scratch = reinterpret_cast<uint64_t*>(after + ivf_lds_bytes());
  // per probe: the payload's first Bloom word and its first doc's bit there (-1: no entry)
  uint32_t* pw = reinterpret_cast<uint32_t*>(scratch + kIvfWaves * a.capw);
  int32_t* pb = reinterpret_cast<int32_t*>(pw + a.n_probe);
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = lane / L;
  const int gl = lane % L;
  const int64_t b = blockIdx.y;
  const int64_t S = static_cast<int64_t>(gridDim.x) * kIvfWaves;
  const int64_t list_at = static_cast<int64_t>(blockIdx.x) * kIvfWaves + wave;
  uint64_t* list = a.lists + (b * S + list_at) * a.capw;
  scratch += wave * a.capw;
  int64_t* qpos = lds->qpos[wave];
  uint32_t* qslot = lds->qslot[wave];

  load_clauses(a, b, &lds->clauses);
  if (a.pwords != nullptr) {
    for (int j = tid; j < a.n_probe; j += kIvfThreads) {
      const int64_t e = b * a.n_probe + j;
      const bool have = e < a.p_entries;
      pw[j] = have && e > 0 ? static_cast<uint32_t>(a.pcum[e - 1]) : 0u;
      pb[j] = have ? static_cast<int32_t>(a.pfirst[e]) : INT32_MIN;
    }
  }
  const uint32_t total = load_ranges(a, b, start, prefix, part);  // (its barriers cover both)
  const int ncl = lds->clauses.n;

  const int nchunks = a.RB / 16;
  v4i qv[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int c = gl + j * L;
    qv[j] = c < nchunks ? *reinterpret_cast<const v4i*>(a.q + b * a.RB + c * 16)
                        : v4i{0, 0, 0, 0};
  }
  const uint64_t* mrow = a.mask != nullptr ? a.mask + b * a.mask_words : nullptr;

  uint64_t tau = 0;
  int cnt = 0;     // entries of this wave's list
  int queued = 0;  // slots waiting to be scored
  const bool cut = total > kCutRows;
  // the row of the scored batch that this lane owns: the folds below leave lane gl (its low bits
  // reversed) with row v of its group
  int own = 0;
#pragma unroll
  for (int i = 1, v = V / 2; v > 0; i <<= 1, v >>= 1) own |= (gl & i) ? v : 0;

  // scores queue entries [at, at + n), n <= E; `more`: the wave may append again, or its list is
  // to be cut to k for the merge's sake
  auto score = [&](int at, int n, bool more) {
    v4i x[V][NC];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int e = v * R + grp;
      const int8_t* row = a.items + qpos[at + (e < n ? e : 0)] * a.RB;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const int c = gl + j * L;
        x[v][j] = c < nchunks && e < n ? *reinterpret_cast<const v4i*>(row + c * 16)
                                       : v4i{0, 0, 0, 0};
      }
    }
    int32_t d[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      d[v] = 0;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          d[v] = __builtin_amdgcn_sdot4(x[v][j][i], qv[j][i], d[v], false);
        }
      }
    }
#pragma unroll
    for (int off = 1, half = V / 2; half > 0; off <<= 1, half >>= 1) {
      const bool up = (gl & off) != 0;
#pragma unroll
      for (int v = 0; v < half; ++v) {
        const int32_t send = up ? d[v] : d[v + half];
        const int32_t keep = up ? d[v + half] : d[v];
        d[v] = keep + __shfl_xor(send, off);
      }
    }
#pragma unroll
    for (int off = V; off < L; off <<= 1) d[0] += __shfl_xor(d[0], off);
    const int e = own * R + grp;
    const bool mine = gl < V && e < n;
    const uint32_t s = qslot[at + (mine ? e : 0)];
    const uint64_t c = composite(search_key(d[0], a.divisor), s);
    const bool keep = mine && c >= tau;
    const uint64_t bal = __ballot(keep);
    if (bal == 0ull) return;
    if (keep) list[cnt + __popcll(bal & ((1ull << lane) - 1ull))] = c;
    cnt += __popcll(bal);
    if (more && cnt > a.capw - E) {
      if (lane == 0) lds->cnt[wave] = cnt;
      const uint64_t nt = wave_compact(list, &lds->cnt[wave], scratch, a.capw, a.k);
      cnt = lds->cnt[wave];
      tau = nt > tau ? nt : tau;
    }
  };

  // this wave's slots: equal runs, in 16s (in 64s, 3100 slots over 16 waves left four of them idle:
  // 128 rows at k = 500 the search 139 us, 129 so; 16 of 1 KB rows 271, 256)
  const uint64_t per = static_cast<uint64_t>(S) * 16;
  const uint32_t span = static_cast<uint32_t>((total + per - 1) / per * 16);
  const uint64_t first = static_cast<uint64_t>(list_at) * span;
  const uint32_t s0 = first < total ? static_cast<uint32_t>(first) : total;
  const uint32_t s1 = total - s0 < span ? total : s0 + span;
  int jr = s0 < s1 ? range_of(prefix, nr, s0) : 0;  // the range of the step's first slot
  for (uint32_t base = s0; base < s1; base += kIvfUnroll * kWave) {
    bool ok[kIvfUnroll];
    int64_t pos[kIvfUnroll];
    const uint64_t* word[kIvfUnroll];
    int bit[kIvfUnroll];
    int j = jr;
#pragma unroll
    for (int u = 0; u < kIvfUnroll; ++u) {
      const uint32_t s = base + u * kWave + lane;  // (below total + 256 < 2^32)
      ok[u] = s < s1 && s >= base;
      while (true) {
        const bool next = ok[u] && s >= prefix[j + 1];
        if (!__any(next)) break;
        j += next ? 1 : 0;
      }
      pos[u] = ok[u] ? start[j] + (s - prefix[j]) : 0;
      word[u] = nullptr;
      bit[u] = 0;
      if (mrow != nullptr) {
        word[u] = mrow + (pos[u] >> 6);
        bit[u] = 63 - static_cast<int>(pos[u] & 63);
      } else if (a.pwords != nullptr) {
        // as fused_kmean_ann_with_partial_masks reads it (fused_kmean_ann_cuda.cu:2264-2501);
        // outside the words: no match
        const int p = j < a.n_probe ? j : j - static_cast<int>(a.n_probe);
        const int64_t at = static_cast<int64_t>(pb[p]) + (pos[u] - start[p]);
        const int64_t w = static_cast<int64_t>(pw[p]) + (at >> 6);
        ok[u] = ok[u] && at >= 0 && pb[p] != INT32_MIN && w < a.p_words;
        word[u] = a.pwords + w;
        bit[u] = 63 - static_cast<int>(at & 63);
      }
      // (lanes are in slot order, so the last one holds the furthest range; lanes past the run
      // keep theirs)
      j = __builtin_amdgcn_readlane(j, kWave - 1);
    }
    jr = j;
    if (mrow != nullptr || a.pwords != nullptr) {
      uint64_t m[kIvfUnroll];
#pragma unroll
      for (int u = 0; u < kIvfUnroll; ++u) m[u] = ok[u] ? *word[u] : 0ull;
#pragma unroll
      for (int u = 0; u < kIvfUnroll; ++u) ok[u] = ok[u] && ((m[u] >> bit[u]) & 1ull);
    }
    for (int c = 0; c < ncl; ++c) {
      const int32_t v = lds->clauses.value[c];
      bool eq[kIvfUnroll] = {};
      for (int64_t r = lds->clauses.r0[c]; r < lds->clauses.r1[c]; ++r) {
        const int32_t* slot_row = a.slots + r * a.N;
        int32_t x[kIvfUnroll];
#pragma unroll
        for (int u = 0; u < kIvfUnroll; ++u) x[u] = ok[u] ? slot_row[pos[u]] : -1;
#pragma unroll
        for (int u = 0; u < kIvfUnroll; ++u) eq[u] |= x[u] == v;
      }
      const bool rev = lds->clauses.reverse[c] != 0;
      bool any = false;
#pragma unroll
      for (int u = 0; u < kIvfUnroll; ++u) {
        ok[u] = ok[u] && eq[u] != rev;
        any |= ok[u];
      }
      if (!__any(any)) break;
    }
#pragma unroll
    for (int u = 0; u < kIvfUnroll; ++u) {
      const uint64_t bal = __ballot(ok[u]);
      if (ok[u]) {
        const int at = queued + __popcll(bal & ((1ull << lane) - 1ull));
        qpos[at] = pos[u];
        qslot[at] = base + u * kWave + lane;
      }
      queued += __popcll(bal);
    }
    wave_sync_memory();
    const bool last = s1 - base <= kIvfUnroll * kWave;
    int at = 0;
    for (; queued - at >= E; at += E) score(at, E, cut || !last || queued - at > E);
    if (last) {
      if (at < queued) score(at, queued - at, cut);
      break;
    }
    // the remainder (fewer than E <= 64) moves to the front
    queued -= at;
    if (at > 0 && queued > 0) {
      const int64_t mp = lane < queued ? qpos[at + lane] : 0;
      const uint32_t ms = lane < queued ? qslot[at + lane] : 0;
      wave_sync_memory();
      if (lane < queued) {
        qpos[lane] = mp;
        qslot[lane] = ms;
      }
    }
    wave_sync_memory();
  }
  if (lane == 0) a.list_counts[b * S + list_at] = cnt;
}

// ---- epilogue -------------------------------------------------------------------------------

struct EpiArgs {
  int64_t* ids;     // in: slots (ranges) or positions, -1 empty; out: sort_perm ids
  const void* raw;  // [B, k] int32 dots, or float fp16 scores
  float* scores;    // out [B, k]
  int64_t B;
  int64_t k;
  bool ranges;  // ids are slots of the probed ranges (else item positions)
  IvfArgs a;    // the ranges (when `ranges`)
  const int64_t* sort_perm;
  int64_t n_perm;
  const float* q_scales;
  const float* global_scale;
  int divisor;
};

// One workgroup per row. Scores (fork_search_cuda.cu:585-591): int32 path
// (fp32(dot) * q_scale) * global_scale; fp16 path score16 * ((q_scale * divisor) *
// global_scale), each product rounded to nearest.
__global__ void __launch_bounds__(kIvfThreads) search_epilogue_kernel(EpiArgs e) {
  extern __shared__ uint64_t smem[];
  const int64_t b = blockIdx.x;
  const int nr = e.ranges ? static_cast<int>(2 * e.a.n_probe) : 0;  // slot ranges
  int64_t* start = reinterpret_cast<int64_t*>(smem);
  uint32_t* prefix = reinterpret_cast<uint32_t*>(start + nr + kIvfWaves);
  if (e.ranges) load_ranges(e.a, b, start, prefix, start + nr);
  const float qs = e.q_scales[b];
  const float gs = e.global_scale[0];
  for (int64_t i = threadIdx.x; i < e.k; i += blockDim.x) {
    const int64_t x = e.ids[b * e.k + i];
    int64_t id = -1;
    float score = -INFINITY;
    if (x >= 0) {
      int64_t pos = x;
      if (e.ranges) {
        const int j = range_of(prefix, nr, static_cast<uint32_t>(x));
        pos = start[j] + (x - prefix[j]);
      }
      if (pos >= 0 && pos < e.n_perm) {
        id = e.sort_perm[pos];
        if (e.divisor == -1) {
          const float dot = static_cast<float>(static_cast<const int32_t*>(e.raw)[b * e.k + i]);
          score = __fmul_rn(__fmul_rn(dot, qs), gs);
        } else {
          const float s16 = static_cast<const float*>(e.raw)[b * e.k + i];
          score = __fmul_rn(s16, __fmul_rn(__fmul_rn(qs, static_cast<float>(e.divisor)), gs));
        }
      }
    }
    e.ids[b * e.k + i] = id;
    e.scores[b * e.k + i] = score;
  }
}

template <int L, int NC, int V>
static int launch_ivf(const IvfArgs& a, dim3 grid, size_t lds, hipStream_t stream) {
  if (lds > 64 * 1024) {
    RT_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&ivf_scan_kernel<L, NC, V>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                     static_cast<int>(lds)));
  }
  ivf_scan_kernel<L, NC, V><<<grid, kIvfThreads, lds, stream>>>(a);
  RT_CHECK_HIP(hipGetLastError());
  return kOk;
}

// L lanes of NC chunks a row: narrow groups fold few partial dots (8 lanes take a 128-byte line
// together); V rows in flight a group, 64 or fewer registers of them. (Rows of 16 and 32 bytes in
// groups of four lanes leave most of the lanes idle: 2M rows, 64 queries of 64 of 1024 lists, the
// scan 126 and 128 us so, 109 and 120 in one and two.)
static int dispatch_ivf(int64_t D, const IvfArgs& a, dim3 grid, size_t lds, hipStream_t stream) {
  if (D <= 16) return launch_ivf<1, 1, 1>(a, grid, lds, stream);
  if (D <= 32) return launch_ivf<2, 1, 2>(a, grid, lds, stream);
  if (D <= 64) return launch_ivf<4, 1, 4>(a, grid, lds, stream);
  if (D <= 128) return launch_ivf<8, 1, 8>(a, grid, lds, stream);
  if (D <= 192) return launch_ivf<4, 3, 4>(a, grid, lds, stream);
  if (D <= 256) return launch_ivf<8, 2, 8>(a, grid, lds, stream);
  if (D <= 512) return launch_ivf<16, 2, 8>(a, grid, lds, stream);
  if (D <= 1024) return launch_ivf<32, 2, 8>(a, grid, lds, stream);
  if (D <= 2048) return launch_ivf<64, 2, 8>(a, grid, lds, stream);
  if (D <= 4096) return launch_ivf<64, 4, 4>(a, grid, lds, stream);
  return launch_ivf<64, 8, 2>(a, grid, lds, stream);
}

// List capacity: k and a batch's appends, a power of two (sorted whole), or the slots of a wave's run
// and those appends where they are fewer (such a list never fills and is never sorted).
static int ivf_capw(int64_t k, int64_t width, int64_t S) {
  const int64_t full = next_pow2(k + kWave);
  const int64_t run = cdiv(width, S * kWave) * kWave + kWave;
  return static_cast<int>(run < full ? run : full);
}

// A row's lists hold up to k entries each (a wave starts without a bound), so its merge is split
// from far fewer lists than a seeded scan's, up to a batch whose merges fill the CUs: 64 rows of
// 128 lists and 19K entries 63 us in one launch, 32 + 14 us split.
constexpr int kIvfPartSlots = 16;
constexpr int64_t kIvfSplitMaxB = 128;

static int64_t ivf_gx(int64_t B, int64_t width) {
  int64_t gx = cdiv(2048, B > 0 ? B : 1);
  const int64_t by_rows = cdiv(width, 1024);
  gx = gx < by_rows ? gx : by_rows;
  gx = gx < 1 ? 1 : gx;
  return gx < kIvfMaxWgsPerRow ? gx : kIvfMaxWgsPerRow;
}

}  // namespace rt

using namespace rt;

// The lane-group quantizers' form: whole 16-byte chunks of every row, codes in 4-byte stores.
static bool quant_vec(const float* x, int64_t dim, const int8_t* codes) {
  return dim % 4 == 0 && dim <= 4 * kWave * kQuantMaxChunks &&
         reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(codes) % 4 == 0;
}

extern "C" int rt_quantize_int8_rows(const float* x, int64_t rows, int64_t dim, int8_t* codes,
                                     float* scales, int scale_div, hipStream_t stream) {
  RT_CHECK_ARG(rows >= 0 && dim >= 1, "rows must be >= 0 and dim >= 1");
  RT_CHECK_ARG(rows <= (int64_t{1} << 31) - 1, "too many rows");
  if (rows == 0) return kOk;
  if (!quant_vec(x, dim, codes)) {
    quantize_rows_kernel<<<static_cast<unsigned>(rows), kQuantThreads, 0, stream>>>(
        x, dim, codes, scales, scale_div);
  } else if (dim <= 64) {
    launch_quantize_vec<16, 1>(x, rows, dim, codes, scales, scale_div, stream);
  } else if (dim <= 128) {
    launch_quantize_vec<32, 1>(x, rows, dim, codes, scales, scale_div, stream);
  } else if (dim <= 256) {
    launch_quantize_vec<64, 1>(x, rows, dim, codes, scales, scale_div, stream);
  } else if (dim <= 512) {
    launch_quantize_vec<64, 2>(x, rows, dim, codes, scales, scale_div, stream);
  } else if (dim <= 1024) {
    launch_quantize_vec<64, 4>(x, rows, dim, codes, scales, scale_div, stream);
  } else {
    launch_quantize_vec<64, kQuantMaxChunks>(x, rows, dim, codes, scales, scale_div, stream);
  }
  RT_CHECK_HIP(hipGetLastError());
  return kOk;
}

extern "C" int rt_quantize_int8_global(const float* x, int64_t rows, int64_t dim,
                                       const int64_t* perm, int8_t* codes, float* abs_max,
                                       uint32_t* scratch4, hipStream_t stream) {
  RT_CHECK_ARG(rows >= 0 && dim >= 1, "rows must be >= 0 and dim >= 1");
  RT_CHECK_ARG(abs_max != nullptr && scratch4 != nullptr, "abs_max and scratch4 must be given");
  RT_CHECK_ARG(rows == 0 || (x != nullptr && codes != nullptr), "x and codes must not be null");
  const int64_t total = rows * dim;
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) {
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  }
  const int64_t want = cdiv(total, kGlobalThreads * 4);
  const unsigned grid = static_cast<unsigned>(want < 8 * cus ? (want > 0 ? want : 1) : 8 * cus);
  abs_max_init_kernel<<<1, 1, 0, stream>>>(scratch4);
  if (total > 0) abs_max_kernel<<<grid, kGlobalThreads, 0, stream>>>(x, total, scratch4);
  if (rows == 0 || !quant_vec(x, dim, codes)) {
    quantize_global_kernel<<<grid, kGlobalThreads, 0, stream>>>(x, rows, dim, perm, scratch4,
                                                                codes, abs_max);
  } else if (dim <= 64) {
    launch_quantize_global_vec<16, 1>(x, rows, dim, perm, scratch4, codes, abs_max, stream);
  } else if (dim <= 128) {
    launch_quantize_global_vec<32, 1>(x, rows, dim, perm, scratch4, codes, abs_max, stream);
  } else if (dim <= 256) {
    launch_quantize_global_vec<64, 1>(x, rows, dim, perm, scratch4, codes, abs_max, stream);
  } else if (dim <= 512) {
    launch_quantize_global_vec<64, 2>(x, rows, dim, perm, scratch4, codes, abs_max, stream);
  } else if (dim <= 1024) {
    launch_quantize_global_vec<64, 4>(x, rows, dim, perm, scratch4, codes, abs_max, stream);
  } else {
    launch_quantize_global_vec<64, kQuantMaxChunks>(x, rows, dim, perm, scratch4, codes, abs_max,
                                                    stream);
  }
  RT_CHECK_HIP(hipGetLastError());
  return kOk;
}

extern "C" int rt_pack_signs(const float* x, int64_t rows, int64_t dim, uint64_t* words,
                             hipStream_t stream) {
  RT_CHECK_ARG(rows >= 0 && dim >= 1, "rows must be >= 0 and dim >= 1");
  RT_CHECK_ARG(dim % 64 == 0, "dim must be a multiple of 64, got %lld",
               static_cast<long long>(dim));
  const int64_t total = rows * (dim / 64);
  if (total == 0) return kOk;
  const int64_t blocks = cdiv(total * kWave, 256);
  RT_CHECK_ARG(blocks < (int64_t{1} << 31), "too many rows");
  pack_signs_kernel<<<static_cast<unsigned>(blocks), 256, 0, stream>>>(x, total, words);
  RT_CHECK_HIP(hipGetLastError());
  return kOk;
}

extern "C" int rt_pack_oporp(const float* x, int64_t rows, int64_t dim, const int8_t* signs,
                             const int64_t* perm, uint64_t* words, hipStream_t stream) {
  RT_CHECK_ARG(rows >= 0 && dim >= 64 && dim % 64 == 0 && dim <= kOporpMaxDim,
               "dim must be a multiple of 64 in [64, %d], got %lld", kOporpMaxDim,
               static_cast<long long>(dim));
  if (rows == 0) return kOk;
  RT_CHECK_ARG(x != nullptr && signs != nullptr && perm != nullptr && words != nullptr,
               "x, signs, perm and words must not be null");
  const int d = static_cast<int>(dim);
  if (d <= 64) {
    launch_pack_oporp<16, 1>(x, rows, d, signs, perm, words, stream);
  } else if (d <= 128) {
    launch_pack_oporp<32, 1>(x, rows, d, signs, perm, words, stream);
  } else if (d <= 256) {
    launch_pack_oporp<64, 1>(x, rows, d, signs, perm, words, stream);
  } else if (d <= 512) {
    launch_pack_oporp<64, 2>(x, rows, d, signs, perm, words, stream);
  } else if (d <= 1024) {
    launch_pack_oporp<64, 4>(x, rows, d, signs, perm, words, stream);
  } else {
    launch_pack_oporp<64, kOporpMaxChunks>(x, rows, d, signs, perm, words, stream);
  }
  RT_CHECK_HIP(hipGetLastError());
  return kOk;
}

extern "C" size_t rt_ivf_search_workspace(int64_t B, int64_t width, int64_t k) {
  if (B <= 0 || k <= 0) return 256;
  const int64_t S = ivf_gx(B, width) * kIvfWaves;
  return align_up(static_cast<size_t>(B * S) * ivf_capw(k, width, S) * sizeof(uint64_t), 256) +
         align_up(static_cast<size_t>(B * S) * sizeof(int), 256) +
         align_up(static_cast<size_t>(B * k) * sizeof(float), 256) +
         (B <= kIvfSplitMaxB ? static_cast<size_t>(B) * kMergeParts * k * sizeof(uint64_t) : 0);
}

// Top-k over each row's probed ranges of int8 codes (slots, ties to the lower slot), then the
// epilogue: out_ids = sort_perm[position] (-1 pads), out_scores dequantized (-inf pads).
static int ivf_search(const int8_t* q_codes, const float* q_scales, int64_t B,
                      const int8_t* item_codes, int64_t N, int64_t D, const int64_t* probe_ids,
                      int64_t n_probe, const int64_t* cluster_offsets,
                      const int64_t* cluster_sizes, int64_t n_lists, int64_t width,
                      const uint64_t* mask, int64_t mask_words, const IvfArgs& filters,
                      int64_t divisor, const int64_t* sort_perm, int64_t n_perm,
                      const float* global_scale, int64_t k, int64_t* out_ids, float* out_scores,
                      void* workspace, size_t workspace_bytes, hipStream_t stream) {
  RT_CHECK_ARG(B >= 0 && N >= 0 && n_probe >= 0 && n_lists >= 0 && width >= 0,
               "sizes must be >= 0");
  RT_CHECK_ARG(k >= 1 && k <= kMaxK, "k must be in [1, %lld], got %lld",
               static_cast<long long>(kMaxK), static_cast<long long>(k));
  RT_CHECK_ARG(D % 16 == 0 && D >= 16 && D <= 8192, "D must be a multiple of 16 in [16, 8192]");
  RT_CHECK_ARG(n_probe <= kIvfMaxProbe, "n_probe must be <= %d", kIvfMaxProbe);
  RT_CHECK_ARG(divisor == -1 || divisor >= 1, "divisor_for_int8 must be -1 or >= 1");
  RT_CHECK_ARG(width < 0xffffffffll, "width must be < 2**32 - 1");
  RT_CHECK_ARG(mask == nullptr || mask_words >= cdiv(N, 64), "mask must cover every item");
  RT_CHECK_ARG(reinterpret_cast<uintptr_t>(item_codes) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(q_codes) % 16 == 0,
               "codes must be 16-byte aligned");
  RT_CHECK_ARG(B <= 65535, "B must be <= 65535");
  if (B == 0) return kOk;
  const size_t need = rt_ivf_search_workspace(B, width, k);
  if (workspace_bytes < need) {
    set_error("workspace too small: %zu < %zu", workspace_bytes, need);
    return kWorkspaceTooSmall;
  }
  const int64_t gx = ivf_gx(B, width);
  const int64_t S = gx * kIvfWaves;
  const int capw = ivf_capw(k, width, S);
  IvfArgs a{};
  a.q = q_codes;
  a.B = B;
  a.items = item_codes;
  a.N = N;
  a.RB = static_cast<int>(D);
  a.probe_ids = probe_ids;
  a.n_probe = n_probe;
  a.cluster_offsets = cluster_offsets;
  a.cluster_sizes = cluster_sizes;
  a.n_lists = n_lists;
  a.width = width;
  a.mask = mask;
  a.mask_words = mask_words;
  a.pcum = filters.pcum;
  a.pfirst = filters.pfirst;
  a.pwords = filters.pwords;
  a.p_entries = filters.p_entries;
  a.p_words = filters.p_words;
  a.slots = filters.slots;
  a.R = filters.R;
  a.cslots = filters.cslots;
  a.C = filters.C;
  a.reverse = filters.reverse;
  a.qv = filters.qv;
  a.divisor = static_cast<int>(divisor);
  a.k = static_cast<int>(k);
  a.capw = capw;
  char* ws = static_cast<char*>(workspace);
  a.lists = reinterpret_cast<uint64_t*>(ws);
  ws += align_up(static_cast<size_t>(B * S) * capw * sizeof(uint64_t), 256);
  a.list_counts = reinterpret_cast<int*>(ws);
  ws += align_up(static_cast<size_t>(B * S) * sizeof(int), 256);
  void* raw = ws;
  ws += align_up(static_cast<size_t>(B * k) * sizeof(float), 256);
  uint64_t* parts = B <= kIvfSplitMaxB ? reinterpret_cast<uint64_t*>(ws) : nullptr;
  const int score_kind = divisor == -1 ? kScoreI32 : kScoreF32;
  if (n_probe > 0) {
    const size_t lds = ranges_lds(n_probe) + ivf_lds_bytes() +
                       static_cast<size_t>(kIvfWaves) * capw * sizeof(uint64_t) +
                       static_cast<size_t>(n_probe) * 2 * sizeof(uint32_t);
    const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(B));
    int st = dispatch_ivf(D, a, grid, lds, stream);
    if (st != kOk) return st;
    MergeArgs m{};
    m.lists = a.lists;
    m.counts = a.list_counts;
    m.capw = capw;
    m.qpw = 1;
    m.S = S;
    m.B = B;
    m.k = static_cast<int>(k);
    m.out_ids = out_ids;
    m.out_scores = raw;
    m.score_kind = score_kind;
    m.part_buf = parts;
    m.part_slots = kIvfPartSlots;
    m.max_entries = width;
    st = launch_merge(m, stream);
    if (st != kOk) return st;
  } else {
    const int st = launch_pad(out_ids, raw, B, k, score_kind, stream);
    if (st != kOk) return st;
  }
  EpiArgs e{};
  e.ids = out_ids;
  e.raw = raw;
  e.scores = out_scores;
  e.B = B;
  e.k = k;
  e.ranges = true;
  e.a = a;
  e.sort_perm = sort_perm;
  e.n_perm = n_perm;
  e.q_scales = q_scales;
  e.global_scale = global_scale;
  e.divisor = static_cast<int>(divisor);
  const size_t lds = ranges_lds(n_probe);
  search_epilogue_kernel<<<static_cast<unsigned>(B), kIvfThreads, lds, stream>>>(e);
  RT_CHECK_HIP(hipGetLastError());
  return kOk;
}

extern "C" int rt_ivf_search(const int8_t* q_codes, const float* q_scales, int64_t B,
                             const int8_t* item_codes, int64_t N, int64_t D,
                             const int64_t* probe_ids, int64_t n_probe,
                             const int64_t* cluster_offsets, const int64_t* cluster_sizes,
                             int64_t n_lists, int64_t width, const uint64_t* mask,
                             int64_t mask_words, int64_t divisor, const int64_t* sort_perm,
                             int64_t n_perm, const float* global_scale, int64_t k,
                             int64_t* out_ids, float* out_scores, void* workspace,
                             size_t workspace_bytes, hipStream_t stream) {
  const IvfArgs none{};
  return ivf_search(q_codes, q_scales, B, item_codes, N, D, probe_ids, n_probe, cluster_offsets,
                    cluster_sizes, n_lists, width, mask, mask_words, none, divisor, sort_perm,
                    n_perm, global_scale, k, out_ids, out_scores, workspace, workspace_bytes,
                    stream);
}

// rt_ivf_search with the reference's per-payload filters in place of a full-N mask: the probed
// payloads' Bloom words (partial response, may be null) and / or the exact clause recheck over
// the probed docs (slot layout, may be null); a doc is scored when both pass.
extern "C" int rt_ivf_search_payload_filters(
    const int8_t* q_codes, const float* q_scales, int64_t B, const int8_t* item_codes, int64_t N,
    int64_t D, const int64_t* probe_ids, int64_t n_probe, const int64_t* cluster_offsets,
    const int64_t* cluster_sizes, int64_t n_lists, int64_t width,
    const int32_t* partial_counts_cumsum, const int8_t* partial_first_offsets,
    const uint64_t* partial_words, int64_t partial_entries, int64_t partial_n_words,
    const int32_t* clause_slot_values, int64_t R, const int64_t* clause_slots, int64_t C,
    const int8_t* clause_is_reverse, const int32_t* query_clause_values, int64_t divisor,
    const int64_t* sort_perm, int64_t n_perm, const float* global_scale, int64_t k,
    int64_t* out_ids, float* out_scores, void* workspace, size_t workspace_bytes,
    hipStream_t stream) {
  RT_CHECK_ARG(partial_words == nullptr ||
                   (partial_counts_cumsum != nullptr && partial_first_offsets != nullptr &&
                    partial_entries >= 0 && partial_n_words >= 0),
               "the partial masks need their counts and first offsets");
  RT_CHECK_ARG(query_clause_values == nullptr ||
                   (clause_slots != nullptr && clause_is_reverse != nullptr && C >= 0 &&
                    C <= 32 && R >= 0 && (R == 0 || clause_slot_values != nullptr)),
               "the exact clauses need slots, clause_slots and clause_is_reverse, C <= 32");
  IvfArgs f{};
  f.pcum = partial_counts_cumsum;
  f.pfirst = partial_first_offsets;
  f.pwords = partial_words;
  f.p_entries = partial_entries;
  f.p_words = partial_n_words;
  f.slots = clause_slot_values;
  f.R = R;
  f.cslots = clause_slots;
  f.C = static_cast<int>(C);
  f.reverse = clause_is_reverse;
  f.qv = query_clause_values;
  return ivf_search(q_codes, q_scales, B, item_codes, N, D, probe_ids, n_probe, cluster_offsets,
                    cluster_sizes, n_lists, width, nullptr, 0, f, divisor, sort_perm, n_perm,
                    global_scale, k, out_ids, out_scores, workspace, workspace_bytes, stream);
}

// The epilogue alone, for a full scan's results: in_ids are item positions (-1 empty), raw the
// int32 dots [B, k].
extern "C" int rt_search_epilogue(int64_t* ids, const int32_t* raw_dots, float* out_scores,
                                  int64_t B, int64_t k, const int64_t* sort_perm, int64_t n_perm,
                                  const float* q_scales, const float* global_scale,
                                  hipStream_t stream) {
  RT_CHECK_ARG(B >= 0 && k >= 1, "B must be >= 0 and k >= 1");
  if (B == 0) return kOk;
  EpiArgs e{};
  e.ids = ids;
  e.raw = raw_dots;
  e.scores = out_scores;
  e.B = B;
  e.k = k;
  e.ranges = false;
  e.sort_perm = sort_perm;
  e.n_perm = n_perm;
  e.q_scales = q_scales;
  e.global_scale = global_scale;
  e.divisor = -1;
  search_epilogue_kernel<<<static_cast<unsigned>(B), kIvfThreads, 0, stream>>>(e);
  RT_CHECK_HIP(hipGetLastError());
  return kOk;
}
