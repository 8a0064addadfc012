// Split-K flash-decoding over per-head segments of the packed circular cache.
//
// Replaces the external decode op the reference calls at
// MoA/kernels/mixture_of_attention.py:465-473.  Every (batch row b, head h)
// attends one query row to rows [start[b,h], start[b,h]+len[b,h]) of
// kc/vc [B, sumC, D].  The work is pure HBM streaming (each K and V byte is
// used once), so the kernel is built around wide coalesced loads:
//
//   * a K/V row of D 16-bit elements is read by D/8 adjacent lanes, 16 bytes
//     each, so one wave-wide load instruction covers 1 KiB of consecutive
//     cache memory (4 rows at D=128);
//   * every wave issues kBatch K loads and kBatch V loads before it consumes
//     any of them (16 KiB in flight per wave);
//   * q.k is a lane-local dot2 chain plus a 4-step DPP sum inside the D/8
//     lanes of a row; the softmax is the usual running (max, sum) in fp32,
//     base 2, rescaled once per batch of rows;
//   * segments differ in length by ~80x between heads, so the unit of work is
//     a fixed-size chunk of rows, not a head: a work-group walks every n-th
//     chunk of a batch row, locating (head, chunk) through a
//     prefix sum over the row's heads that every wave forms from
//     head_valid_len (no host knowledge of the lengths, no host sync);
//   * a head with one chunk writes its output directly; otherwise chunks
//     write fp32 partial (acc, max, sum) triples and a small second kernel
//     merges them (in launches of few chunks the head's last chunk to arrive
//     does, when the caller brings counters);
//   * grouped-query attention (G = Hq / Hkv query heads per ring, which the
//     reference does not have): the G query rows of a ring share every K/V
//     row that a wave loads, so the cache is still read once.  This kernel is
//     written for any G but instantiated for G = 1 only; G = 2 to 8 run on the
//     matrix cores (decode_gqa_kernel below).
#include "moa_mfma.h"

#include <hip/hip_fp16.h>

#include <mutex>
#include <type_traits>

namespace moa {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kDecThreads = 256;
constexpr int kDecWaves = kDecThreads / 64;
constexpr int kBatch = 8;           // wave-wide loads in flight per tensor
constexpr int kMaxHeads = 256;     // heads per batch row: four to a lane of the wave that finds the chunks
constexpr float kLog2e = 1.4426950408889634f;

struct F16 {};
struct BF16 {};

template <typename T>
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c);
template <>
__device__ __forceinline__ float dot2<F16>(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
}
template <>
__device__ __forceinline__ float dot2<BF16>(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c,
                                         false);
}

template <typename T>
__device__ __forceinline__ void unpack2(uint32_t x, float& lo, float& hi);
template <>
__device__ __forceinline__ void unpack2<F16>(uint32_t x, float& lo, float& hi) {
  f16x2 h = __builtin_bit_cast(f16x2, x);
  lo = (float)h.x;
  hi = (float)h.y;
}
template <>
__device__ __forceinline__ void unpack2<BF16>(uint32_t x, float& lo, float& hi) {
  lo = __builtin_bit_cast(float, x << 16);
  hi = __builtin_bit_cast(float, x & 0xffff0000u);
}

template <typename T>
__device__ __forceinline__ uint16_t pack1(float x);
template <>
__device__ __forceinline__ uint16_t pack1<F16>(float x) {
  return __builtin_bit_cast(uint16_t, (_Float16)x);
}
template <>
__device__ __forceinline__ uint16_t pack1<BF16>(float x) {
  // round to nearest even
  uint32_t u = __builtin_bit_cast(uint32_t, x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

template <int N>
struct DecInt {
  static constexpr int value = N;
};

typedef const uint16_t __attribute__((address_space(1))) * GlobalPtr;
// Sixteen bytes of a cache row, which a step reads once.  NT marks the load non-temporal: it leaves no line
// behind in the caches, which a launch that reads more than they hold only pays for (see kNtBytes).
template <bool NT>
__device__ __forceinline__ u32x4 load_once16(GlobalPtr p) {
  typedef const u32x4 __attribute__((address_space(1))) * Global16;
  const Global16 s = (Global16)p;
  if constexpr (NT) return __builtin_nontemporal_load(s);
  else return *s;
}

// Rows of a segment are numbered in 32 bits, without a sign: a segment has up to 2^31 - 1 rows, and where its last
// chunk, or the load batch at its end, would stop lies up to a chunk past that.
constexpr __host__ __device__ __forceinline__ int chunks_of(int len, int size) {
  return (int)(((unsigned)len + (unsigned)size - 1u) / (unsigned)size);
}
// first row of a wave's share of a chunk, and the first row behind it
constexpr __host__ __device__ __forceinline__ unsigned share_begin(int chunk, int chunk_rows, int wave, int share_rows) {
  return (unsigned)chunk * (unsigned)chunk_rows + (unsigned)wave * (unsigned)share_rows;
}
constexpr __host__ __device__ __forceinline__ unsigned share_end(unsigned begin, int share_rows, int len) {
  return begin + (unsigned)share_rows < (unsigned)len ? begin + (unsigned)share_rows : (unsigned)len;
}
// the largest segment: whole chunks, the last one a row short (an overflow with a sign does not compile here)
constexpr int kMaxRows = 0x7fffffff;
static_assert(chunks_of(kMaxRows, 512) == 1 << 22 && chunks_of(kMaxRows, 2048) == 1 << 20);
static_assert(chunks_of(0, 512) == 0 && chunks_of(1, 512) == 1 && chunks_of(512, 512) == 1 && chunks_of(513, 512) == 2);
static_assert(share_end(share_begin((1 << 22) - 1, 512, 3, 128), 128, kMaxRows) == 0x7fffffffu);
static_assert(share_end(share_begin((1 << 22) - 1, 512, 2, 128), 128, kMaxRows) == 0x7fffff80u);

__device__ __forceinline__ int wave_sum(int x) { return __builtin_amdgcn_readlane(wave_scan(x), 63); }
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}

// The chunks of one batch row, worked out by every wave for itself: lane i holds heads i, i + 64, ... and no LDS, no
// barrier and one memory latency stand between the launch and the first cache row (a table in LDS built by the whole
// work-group cost 1 us of a launch).  Chunks are numbered head by head; chunk numbers are clamped to `cap`, the
// partial slots a batch row owns: with disjoint segments the clamp never acts; with overlapping ones (lengths that sum
// to more than the row holds) the chunks past the cap do not exist for any kernel, so none of them is written, read
// or merged.  Segments are clamped into the row, so that a bad index cannot fault.
//
// Three policies.  Fixed: chunks of CHUNK rows.  Short (kShortChunks, only with EVEN): chunks of kEvenMinChunk rows, for
// launches whose batch rows cannot have more of them than their share of the CUs: what Even comes to there, without its
// search and divisions (0.5 to 1 us in front of the first load).  Even (even_target > 0, only with EVEN): with a fixed length the last
// chunk of every head is a remainder and the number of chunks is whatever it comes to; here the caller names the
// number of chunks a batch row should not exceed, and the row takes the shortest chunk length c (whole steps of
// kEvenStep rows, at least kEvenMinChunk) for which sum_h ceil(len_h / c) <= target; head h is then split evenly into
// ceil(len_h / c) chunks.  The search starts at total / target and goes up step by step (the sum exceeds the target by
// at most the number of heads at the start, so a few steps do), and gives up after kEvenTries: the result is valid for
// any c, the target is a wish.  Integer arithmetic only: the split and the merge kernel must agree on every entry.
constexpr int kEvenMinChunk = 256;   // also the chunk length the partial slots of a batch row are sized for
constexpr int kEvenStep = 128;
constexpr int kEvenTries = 24;
constexpr int kShortChunks = -1;     // instead of an even_target
struct Chunk {
  int head, index, count;   // its head, its place among the head's chunks, how many those are
  int seg0, len, rows;      // first row and valid rows of the head's segment, rows per chunk of the head
};
template <int CHUNK, bool EVEN>
struct RowChunks {
  static constexpr int kGroups = kMaxHeads / 64;
  int seg0[kGroups], len[kGroups], rows[kGroups], last[kGroups];   // last: chunks up to and including this head, clamped
  int total;                                                       // chunks of the batch row, clamped

  __device__ __forceinline__ RowChunks(const int64_t* __restrict__ valid_row, const int64_t* __restrict__ start_row,
                                       int H, int64_t sumC, int cap, int even_target) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) {
      seg0[k] = len[k] = 0;
      const int i = k * 64 + lane;
      if (i < H) {
        int64_t l = valid_row[i];
        const int64_t first = start_row[i];
        if (l < 0 || first < 0 || first >= sumC) l = 0;
        if (l > sumC - first) l = sumC - first;
        seg0[k] = (int)(l > 0 ? first : 0);
        len[k] = (int)l;
      }
    }
    static_assert((CHUNK & (CHUNK - 1)) == 0 && (kEvenMinChunk & (kEvenMinChunk - 1)) == 0, "fixed chunks divide by a shift");
    int c = EVEN && even_target == kShortChunks ? kEvenMinChunk : CHUNK;
    const bool even = EVEN && even_target > 0;
    const int shift = __builtin_ctz(c);
    if (even) {
      auto chunks = [&](int size) __attribute__((always_inline)) {
        int n = 0;
#pragma unroll
        for (int k = 0; k < kGroups; ++k)
          if (k * 64 < H) n += chunks_of(len[k], size);
        return wave_sum(n);
      };
      // rows in steps (a sum of at most 256 heads of < 2^31 rows each fits 32 bits in steps)
      c = max(kEvenMinChunk, ((chunks(kEvenStep) + even_target - 1) / even_target) * kEvenStep);
#pragma unroll 1   // unrolled, its divisions cost every launch 0.3 us
      for (int t = 0; t < kEvenTries && chunks(c) > even_target; ++t) c += kEvenStep;
    }
    int base = 0;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) {
      rows[k] = c;
      last[k] = base;
      if (k * 64 < H) {
        int n = (int)(((unsigned)len[k] + (unsigned)c - 1u) >> shift);
        if (even) n = chunks_of(len[k], c);
        if (even && n > 0) {
          rows[k] = chunks_of(chunks_of(len[k], n), kEvenStep) * kEvenStep;   // even split, <= c
          n = chunks_of(len[k], rows[k]);
        }
        const int incl = wave_scan(n);
        last[k] = min(base + incl, cap);
        base += __builtin_amdgcn_readlane(incl, 63);
      }
    }
    total = min(base, cap);
  }
  // an entry of head h (h is uniform)
  __device__ __forceinline__ int of(const int (&x)[kGroups], int h) const {
    int r = 0;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) {
      const int in_group = __builtin_amdgcn_readlane(x[k], h & 63);
      r = (h >> 6) == k ? in_group : r;
    }
    return r;
  }
  __device__ __forceinline__ int first_of(int h) const {
    const int before = of(last, max(h - 1, 0));
    return h > 0 ? before : 0;
  }
  // chunk w, 0 <= w < total (uniform)
  __device__ __forceinline__ Chunk at(int w, int H) const {
    int h = 0;   // heads that end before w
#pragma unroll
    for (int k = 0; k < kGroups; ++k)
      if (k * 64 < H) h += __popcll(__ballot(last[k] <= w && k * 64 + (int)(threadIdx.x & 63) < H));
    const int first = first_of(h);
    return {h, w - first, of(last, h) - first, of(seg0, h), of(len, h), of(rows, h)};
  }
};

// What a wave knows of a head once it has gone through its share of the chunks: its VEC columns of the weighted sum
// (of its share) and the sum of weights (of all chunks).
template <int D>
struct Merged {
  static constexpr int VEC = D / 64;   // columns per lane
  typedef float fvec __attribute__((ext_vector_type(VEC)));
  fvec a;
  float L;
};
// One wave's part of the merge of a head's n partials: chunks first, first + stride, ...  `acc` and `ml` are the head's
// first partial (uniform), `G` partials lie between a chunk's and the next one's.  The constructor sends the wave's loads
// out, sum() looks at them: a wave that merges several heads asks for all of theirs first.  COHERENT: the partials come from work-groups of this launch, on other XCDs perhaps:
// device-scope loads.
// A wave that takes every chunk (stride 1) sums them in kDecWaves strands, as kDecWaves waves with a stride of
// kDecWaves and their final sum do: every way of merging gives the same bits.
template <int D, bool COHERENT, int kFirst /* chunks asked for at once */, int kMore /* and in every round behind */,
          bool STRANDS = false>
struct WaveMerge {
  typedef typename Merged<D>::fvec fvec;
  static constexpr int VEC = Merged<D>::VEC;
  static_assert(64 % kMore == 0 && kFirst % kMore == 0, "rounds do not straddle a block of 64 factors");
  const float* acc;
  const f32x2* ml;
  int G, n, first, stride;
  int step;          // from a chunk's accumulator to the next one's
  fvec x[kFirst];    // a chunk past the head's last repeats that one: no branch stands between the loads
  f32x2 mine;        // chunk `lane`

  template <typename V>
  static __device__ __forceinline__ V load(const V* p) {
    if constexpr (!COHERENT) {
      return *p;
    } else if constexpr (sizeof(V) == 8) {
      return __builtin_bit_cast(V, __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT));
    } else {
      return __builtin_bit_cast(V, __hip_atomic_load(reinterpret_cast<const uint32_t*>(p), __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT));
    }
  }
  __device__ __forceinline__ WaveMerge(const float* acc_, const f32x2* ml_, int G_, int n_, int first_, int stride_)
      : acc(acc_), ml(ml_), G(G_), n(n_), first(first_), stride(stride_), step(G_ * D) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < kFirst; ++j)
      x[j] = load(reinterpret_cast<const fvec*>(acc + min(first + stride * j, n - 1) * step + lane * VEC));
    mine = f32x2{-INFINITY, 0.f};
    if (lane < n) mine = load(ml + (int64_t)lane * G);
  }
  __device__ __forceinline__ Merged<D> sum() const;
};
template <int D, bool COHERENT, int kFirst, int kMore, bool STRANDS>
__device__ __forceinline__ Merged<D> WaveMerge<D, COHERENT, kFirst, kMore, STRANDS>::sum() const {
  const int lane = threadIdx.x & 63;
  float M = mine.x;
  for (int i = 64 + lane; i < n; i += 64) M = fmaxf(M, load(ml + (int64_t)i * G).x);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
  const float m_use = (M == -INFINITY) ? 0.f : M;
  float f = fast_exp2(mine.x - m_use);   // the factor of chunk `lane`
  float L = mine.y * f;
  auto factor = [&](int i) __attribute__((always_inline)) {   // of the chunk at lane i (uniform)
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), i));
  };
  constexpr int kStrands = STRANDS ? kDecWaves : 1;
  static_assert(kMore % kStrands == 0, "a round starts at strand 0");
  fvec a[kStrands] = {};
#pragma unroll
  for (int j = 0; j < kFirst; ++j)
    if (first + stride * j < n) a[j % kStrands] += x[j] * factor(first + stride * j);
  int i = first + stride * kFirst;   // the rest; factors in blocks of 64 chunks
  for (int i0 = 0; i0 < n; i0 += 64) {
    if (i0 > 0) {
      f = 0.f;
      if (i0 + lane < n) {
        const f32x2 v = load(ml + (int64_t)(i0 + lane) * G);
        f = fast_exp2(v.x - m_use);
        L += v.y * f;
      }
    }
    const int end = min(i0 + 64, n);
    for (; i < end; i += kMore * stride) {
      fvec y[kMore];
#pragma unroll
      for (int j = 0; j < kMore; ++j)
        y[j] = load(reinterpret_cast<const fvec*>(acc + (int64_t)min(i + stride * j, end - 1) * step + lane * VEC));
#pragma unroll
      for (int j = 0; j < kMore; ++j)
        if (i + stride * j < end) a[j % kStrands] += y[j] * factor(i + stride * j - i0);
    }
  }
  Merged<D> r;
  r.a = a[0];
#pragma unroll
  for (int k = 1; k < kStrands; ++k) r.a += a[k];
  r.L = wave_sum(L);
  return r;
}

// Launches of few chunks merge inside the split kernel: the work-group whose chunk is the head's last to arrive sums
// the head's partials up, and the merge launch (4.5 us of a step's GPU time, as much again of the host's) falls away.
// Partials are stored and read with device-scope accesses and the arrival is counted with a device-scope atomic, each
// wave waiting for its stores before the count; no fence, which would write back and drop the XCD's whole L2.
// `counters` holds one zero per (batch row, ring) and is left at zero.
__device__ __forceinline__ void store_partial(float* p, float x, bool coherent) {
  if (coherent) __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = x;
}
// Called by the whole work-group behind its partials' stores; true for the last of the ring's n chunks to arrive.
__device__ __forceinline__ bool arrived_last(unsigned* counter, int n) {
  __shared__ unsigned s_before;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    s_before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (s_before == (unsigned)n - 1) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return s_before == (unsigned)n - 1;
}
// The zero output of a batch row's rings without a chunk (the merge kernel's in launches of two kernels).
template <typename ROW>
__device__ __forceinline__ void zero_empty_rings(const ROW& row, uint16_t* o_row, int H, int row_elems) {
  const int lane = threadIdx.x & 63;
  int before = 0;   // chunks of the groups of heads so far
#pragma unroll
  for (int k = 0; k < ROW::kGroups; ++k) {
    if (k * 64 >= H) break;
    const int up = __shfl_up(row.last[k], 1, 64);
    unsigned long long empty = __ballot(k * 64 + lane < H && row.last[k] == (lane > 0 ? up : before));
    before = __builtin_amdgcn_readlane(row.last[k], 63);
    for (; empty != 0; empty &= empty - 1) {
      const int h = k * 64 + __builtin_ctzll(empty);
      for (int i = threadIdx.x; i < row_elems; i += blockDim.x) o_row[(int64_t)h * row_elems + i] = 0;
    }
  }
}

// H: kv heads (rings) per batch row; query head hk*G + g reads ring hk.
// PIPE: the wave keeps two half-batches of loads going (the next one is issued before the current
// one is consumed) instead of loading a full batch, waiting for it and consuming it (kDecPipeFrom).
template <typename T, int D, int CHUNK, int G, bool PIPE, bool NT>
__global__ __launch_bounds__(kDecThreads) void decode_split_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    uint16_t* __restrict__ o, float* __restrict__ part_acc, float* __restrict__ part_ml,
    const int64_t* __restrict__ head_start, const int64_t* __restrict__ head_valid, int H,
    int64_t sumC, float scale_log2, int cap /* partial slots per batch row */,
    unsigned* __restrict__ counters /* one per (b, ring): merge here; null: decode_merge_kernel does */) {
  constexpr bool MERGE = !PIPE;       // the launches that may merge inside (the code costs the others 1 %)
  constexpr int LPR = D / 8;          // lanes per row
  constexpr int RPL = 64 / LPR;       // rows per wave-wide load
  constexpr int KB = (G >= 8) ? kBatch / 2 : kBatch;   // loads in flight per tensor (registers bound it at G = 8)
  constexpr int ROWS = RPL * KB;      // rows per wave per batch of loads
  constexpr int WCHUNK = CHUNK / kDecWaves;
  static_assert(WCHUNK % ROWS == 0, "chunk must split evenly over waves and load batches");

  __shared__ float s_acc[kDecWaves][G][D];
  __shared__ float s_m[kDecWaves][G];
  __shared__ float s_l[kDecWaves][G];

  const int b = blockIdx.x;   // batch rows side by side (see kDecBlocksPerCu)
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane % LPR;   // which 8-element slice of the row
  const int sub = lane / LPR;   // which row of a wave-wide load

  const RowChunks<CHUNK, false> row(head_valid + (int64_t)b * H, head_start + (int64_t)b * H, H, sumC, cap, 0);

  if (MERGE && counters && blockIdx.y == 0) zero_empty_rings(row, o + (int64_t)b * H * G * D, H, G * D);

  for (int w = blockIdx.y; w < row.total; w += gridDim.y) {
    const Chunk ck = row.at(w, H);
    const int c = ck.index, n_chunks = ck.count;
    const int64_t bh = (int64_t)b * H + ck.head;
    const unsigned r_begin = share_begin(c, CHUNK, wave, WCHUNK);
    const unsigned r_end = share_end(r_begin, WCHUNK, ck.len);

    // this lane's 8 query elements of each of the G query heads, kept packed for dot2
    u32x4 qv[G];
#pragma unroll
    for (int g = 0; g < G; ++g) qv[g] = *reinterpret_cast<const u32x4*>(q + (bh * G + g) * D + col * 8);

    GlobalPtr kbase = (GlobalPtr)kc + ((int64_t)b * sumC + ck.seg0) * D + col * 8;
    GlobalPtr vbase = (GlobalPtr)vc + ((int64_t)b * sumC + ck.seg0) * D + col * 8;
    // Opaque from here on: loads the compiler can prove to read constant memory are moved next to their uses, across
    // any barrier, to save registers, and go out one at a time.
    asm volatile("" : "+v"(kbase), "+v"(vbase));

    float m[G], l[G];
    float acc[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      m[g] = -INFINITY;
      l[g] = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[g][j] = 0.f;
    }

    // n wave-wide loads of K and of V starting at row r0 of the wave's share
    auto load_rows = [&](auto N, u32x4* kr, u32x4* vr, unsigned r0) __attribute__((always_inline)) {
      constexpr int n = decltype(N)::value;
#pragma unroll
      for (int i = 0; i < n; ++i) {
        const unsigned row = r0 + i * RPL + sub;
        const int64_t rr = row < r_end ? row : r_begin;  // any valid row: keeps the load in bounds
        kr[i] = load_once16<NT>(kbase + rr * D);
        vr[i] = load_once16<NT>(vbase + rr * D);
      }
      __builtin_amdgcn_sched_barrier(0);   // all of them before what uses them
    };
    // online-softmax update with those rows
    auto consume_rows = [&](auto N, const u32x4* kr, const u32x4* vr, unsigned r0) __attribute__((always_inline)) {
      constexpr int n = decltype(N)::value;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float s[n];
        float bm = -INFINITY;
#pragma unroll
        for (int i = 0; i < n; ++i) {
          float d = 0.f;
          d = dot2<T>(qv[g].x, kr[i].x, d);
          d = dot2<T>(qv[g].y, kr[i].y, d);
          d = dot2<T>(qv[g].z, kr[i].z, d);
          d = dot2<T>(qv[g].w, kr[i].w, d);
          d = group_sum<LPR>(d) * scale_log2;
          const bool ok = (r0 + i * RPL + sub) < r_end;
          s[i] = ok ? d : -INFINITY;
          bm = fmaxf(bm, s[i]);
        }
        const float m_new = fmaxf(m[g], bm);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = fast_exp2(m[g] - m_use);
        l[g] *= alpha;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[g][j] *= alpha;
#pragma unroll
        for (int i = 0; i < n; ++i) {
          const float p = fast_exp2(s[i] - m_use);
          l[g] += p;
          float lo, hi;
          unpack2<T>(vr[i].x, lo, hi); acc[g][0] = fmaf(p, lo, acc[g][0]); acc[g][1] = fmaf(p, hi, acc[g][1]);
          unpack2<T>(vr[i].y, lo, hi); acc[g][2] = fmaf(p, lo, acc[g][2]); acc[g][3] = fmaf(p, hi, acc[g][3]);
          unpack2<T>(vr[i].z, lo, hi); acc[g][4] = fmaf(p, lo, acc[g][4]); acc[g][5] = fmaf(p, hi, acc[g][5]);
          unpack2<T>(vr[i].w, lo, hi); acc[g][6] = fmaf(p, lo, acc[g][6]); acc[g][7] = fmaf(p, hi, acc[g][7]);
        }
        m[g] = m_new;
      }
    };
    if (!PIPE) {
      for (unsigned r0 = r_begin; r0 < r_end; r0 += ROWS) {
        u32x4 kr[KB], vr[KB];
        load_rows(DecInt<KB>{}, kr, vr, r0);
        consume_rows(DecInt<KB>{}, kr, vr, r0);
      }
    } else {
      // Every half-batch is asked for without a condition (past the end: the first row again, cached): behind a
      // branch the compiler cannot count the loads in flight and waits for all of them in front of each use.
      constexpr int KH = KB / 2, HROWS = ROWS / 2;
      u32x4 ka[KH], va[KH], kb2[KH], vb2[KH];
      if (r_begin < r_end) {
        load_rows(DecInt<KH>{}, ka, va, r_begin);
        for (unsigned r0 = r_begin; r0 < r_end; r0 += ROWS) {
          load_rows(DecInt<KH>{}, kb2, vb2, r0 + HROWS);
          consume_rows(DecInt<KH>{}, ka, va, r0);
          load_rows(DecInt<KH>{}, ka, va, r0 + ROWS);
          if (r0 + HROWS < r_end) consume_rows(DecInt<KH>{}, kb2, vb2, r0 + HROWS);
        }
      }
    }

    // ---- combine the RPL row-groups of the wave ----
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float mw = m[g];
#pragma unroll
      for (int off = LPR; off < 64; off <<= 1) mw = fmaxf(mw, __shfl_xor(mw, off, 64));
      {
        const float m_use = (mw == -INFINITY) ? 0.f : mw;
        const float f = fast_exp2(m[g] - m_use);
        l[g] *= f;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[g][j] *= f;
      }
#pragma unroll
      for (int off = LPR; off < 64; off <<= 1) {
        l[g] += __shfl_xor(l[g], off, 64);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[g][j] += __shfl_xor(acc[g][j], off, 64);
      }
      if (lane < LPR) {
#pragma unroll
        for (int j = 0; j < 8; ++j) s_acc[wave][g][lane * 8 + j] = acc[g][j];
        if (lane == 0) {
          s_m[wave][g] = mw;
          s_l[wave][g] = l[g];
        }
      }
    }
    __syncthreads();

    // ---- combine the waves; thread d owns output column d of every query head of the ring ----
    if (tid < D) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float M = s_m[0][g];
#pragma unroll
        for (int i = 1; i < kDecWaves; ++i) M = fmaxf(M, s_m[i][g]);
        const float m_use = (M == -INFINITY) ? 0.f : M;
        float L = 0.f, a = 0.f;
#pragma unroll
        for (int i = 0; i < kDecWaves; ++i) {
          const float f = fast_exp2(s_m[i][g] - m_use);
          L += s_l[i][g] * f;
          a += s_acc[i][g][tid] * f;
        }
        if (n_chunks == 1) {
          const float out = (L > 0.f) ? a / L : 0.f;
          o[(bh * G + g) * D + tid] = pack1<T>(out);
        } else {
          const int64_t slot = ((int64_t)b * cap + w) * G + g;
          store_partial(part_acc + slot * D + tid, a, MERGE && counters != nullptr);
          if (tid == 0) {
            store_partial(part_ml + slot * 2 + 0, M, MERGE && counters != nullptr);
            store_partial(part_ml + slot * 2 + 1, L, MERGE && counters != nullptr);
          }
        }
      }
    }
    if (MERGE && counters && n_chunks > 1 && arrived_last(counters + bh, n_chunks)) {
      float* const s_sum = &s_acc[0][0][0];   // [kDecWaves][D]
      for (int g = 0; g < G; ++g) {
        const int64_t slot0 = ((int64_t)b * cap + w - c) * G + g;
        const Merged<D> m = WaveMerge<D, true, 8, 4>(part_acc + slot0 * D, reinterpret_cast<const f32x2*>(part_ml) + slot0, G,
                                                     n_chunks, wave, kDecWaves).sum();
        *reinterpret_cast<typename Merged<D>::fvec*>(s_sum + wave * D + lane * Merged<D>::VEC) = m.a;
        __syncthreads();
        if (tid < D) {
          const float t = s_sum[tid] + s_sum[D + tid] + s_sum[2 * D + tid] + s_sum[3 * D + tid];
          o[(bh * G + g) * D + tid] = pack1<T>((m.L > 0.f) ? t / m.L : 0.f);
        }
        __syncthreads();
      }
    }
    __syncthreads();  // s_acc / s_m / s_l are reused by the next chunk
  }
}

// Merge of the per-chunk partials of heads with more than one chunk, and the zero output of empty heads.
// Latency is all there is to it (a few MB at most): one work-group per query head, each of its waves finds the
// head's chunks by itself (one memory latency), then asks for the (max, sum) pairs of all chunks, a lane each,
// and for its share of the accumulators, every fourth chunk, before it looks at any of them (a second one);
// the waves meet once, in LDS, for the final sum.  Against two heads to a work-group, a table of the row in LDS and the
// loads behind it: four layers at batch 1 of 16k tokens 112.0 -> 108.9 us a pass, batch 4 grouped 185.0 -> 180.5 us.
template <typename T, int D, int CHUNK>
__global__ __launch_bounds__(kDecThreads) void decode_merge_kernel(
    uint16_t* __restrict__ o, const float* __restrict__ part_acc, const float* __restrict__ part_ml,
    const int64_t* __restrict__ head_start, const int64_t* __restrict__ head_valid, int H,
    int G /* query heads per ring */, int64_t sumC, int cap,
    int even_target /* of the split kernel's chunks */) {
  __shared__ float s_a[kDecWaves][D];
  const int hq = blockIdx.x, b = blockIdx.y;
  const int h = hq / G, g = hq % G;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const RowChunks<CHUNK, true> row(head_valid + (int64_t)b * H, head_start + (int64_t)b * H, H, sumC, cap, even_target);
  const int w0 = row.first_of(h), n = row.of(row.last, h) - w0;
  if (n == 1) return;   // written by the split kernel
  uint16_t* const out = o + ((int64_t)b * H * G + hq) * D;
  if (n == 0) {
    if (tid < D) out[tid] = 0;
    return;
  }
  const int64_t slot0 = ((int64_t)b * cap + w0) * G + g;
  const Merged<D> m = WaveMerge<D, false, 8, 4>(part_acc + slot0 * D, reinterpret_cast<const f32x2*>(part_ml) + slot0, G, n,
                                                wave, kDecWaves).sum();
  const float L = m.L;
  *reinterpret_cast<typename Merged<D>::fvec*>(&s_a[wave][lane * Merged<D>::VEC]) = m.a;
  __syncthreads();
  if (tid < D) {
    float t = s_a[0][tid];
#pragma unroll
    for (int w = 1; w < kDecWaves; ++w) t += s_a[w][tid];
    out[tid] = pack1<T>((L > 0.f) ? t / L : 0.f);
  }
}

// ---- grouped-query decode on the matrix cores (G >= 2) ---------------------------------------
// With G query heads per ring the vector ALU version above does G times the arithmetic per cache
// byte and stops being HBM bound (measured: 65 % of peak at G = 2, 46 % at G = 8).  Here the G query rows of a ring are the
// columns of a 16-wide MFMA tile (columns >= G are zero padding; the matrix pipe has the room):
//   S^T[key][q] = sum_d K[key][d] Q[q][d]      A = K (LDS), B = Q^T (registers)
//   O^T[d][q]   = sum_key V[key][d] P[q][key]   A = V^T (LDS, transposing read), B = P^T
// the same transposed pair of products as the prefill kernel, 32 keys at a time, so the softmax
// state of a query head stays in its column's four lanes (a quarter of the keys each).  v_mfma_f32_16x16x32 leaves in lane
// 16 g + n rows 4 g + i of column n, which is the B operand of the second product as it is, when its contraction slots are
// numbered that way.  Each wave streams its own share of the chunk through a
// private two-stage LDS ring with asynchronous copies (16-byte chunks XOR-permuted as in the
// prefill kernel), so no work-group barrier is needed inside the loop.  Chunks, partials and the
// merge kernel are those of the vector version, with a longer chunk.
// A CU has one wave per SIMD (the LDS rings fill it), so nothing hides what a wave does to a tile between two copies.  With
// 32-wide tiles half of the matrix cycles, of the exponentials and of the packing went into padding, for up to 8 heads three
// quarters; with 16-wide ones, and K and V waited for and copied each by itself, a call takes, before and now (GPU time):
// batch 4 of 8 rings, 164 MB, 8 heads 34.9 -> 33.5 us; batch 2, 82 MB 23.1 -> 21.8; batch 1, 8 rings of up to 500 rows,
// 4 heads 9.7 -> 8.7; batch 4 of 64-element rows, 66 MB, 2 heads 18.2 -> 16.5; batch 16, 655 MB 109.5 -> 107.7.
// Work-groups per CU the grid may hold.  A CU runs one at a time (the LDS rings fill it), so the hardware
// dispatcher hands out chunks as CUs become free when every chunk is a work-group of its own: 602 us at
// batch 64 of the 70B shape against 612-628 us with 2-16 per CU, each walking several chunks in a fixed order.
// The grid has batch rows side by side, chunk numbers outside: a row's chunks are fewer than the host can count on, and the
// work-groups that find none come last then.  Between the rows they delay what stands behind them, since work-groups go to
// the XCDs strictly in turn: a chunk waits for its XCD while another has CUs free.  Batch 32 of 8 rings of up to 6800 rows,
// 4 heads 107.1 -> 89.0 us, batch 12 of up to 17000, 8 heads 96.7 -> 87.4, batch 24 of 2 rings 25.8 -> 19.6.
constexpr int kGqaBlocksPerCu = 64;
// Largest number of cache rows per work-group step (a quarter per wave) the launch aims for; the actual
// chunk lengths come out of an even split of every batch row (RowChunks).  A chunk start costs a
// wave full memory latencies with nothing in flight, so long chunks win: with one fixed length, 2048 was
// the best of 512..4096 at batch 64 and at batch 4.
constexpr int kGqaChunk = 2048;
constexpr int kGqaTile = 32;      // keys per stage (two MFMA tiles of scores, one contraction of P.V)
constexpr int kGqaMaxG = 8;       // query heads per ring the per-wave result buffers are sized for
constexpr int kGqaWaves = 4;      // waves per work-group (8 waves with one stage each measure the same)
constexpr int kGqaThreads = 64 * kGqaWaves;
constexpr int kGqaStages = 2;     // LDS stages per wave (8 stages of 16 KiB at D = 128 in all)

template <typename T> struct MfmaElem;
template <> struct MfmaElem<F16> { typedef PF16 type; };
template <> struct MfmaElem<BF16> { typedef PBF16 type; };

template <int D>
constexpr size_t gqa_lds_bytes() { return (size_t)kGqaWaves * kGqaStages * 2 * kGqaTile * D * 2; }

template <typename T, int D, bool NT>
__global__ __launch_bounds__(kGqaThreads) void decode_gqa_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    uint16_t* __restrict__ o, float* __restrict__ part_acc, float* __restrict__ part_ml,
    const int64_t* __restrict__ head_start, const int64_t* __restrict__ head_valid, int H,
    int G /* query heads per ring, <= kGqaMaxG */, int64_t sumC, float scale_log2_signed, int cap,
    int target /* > 0: chunks a batch row is split into; 0 or kShortChunks: chunks of a fixed length (RowChunks) */,
    unsigned* __restrict__ counters /* as in decode_split_kernel */) {
  typedef typename MfmaElem<T>::type M;
  // the row maximum is taken over unscaled scores: a negative softmax scale goes into Q (sign flip, exact)
  const float scale_log2 = __builtin_fabsf(scale_log2_signed);
  const uint32_t q_sign = scale_log2_signed < 0.f ? 0x80008000u : 0u;
  constexpr bool MERGE = !NT;                   // as in decode_split_kernel
  constexpr int KS = D / 32;                    // MFMA k-steps of Q.K^T
  constexpr int DT = D / 16;                    // 16-wide d tiles of the output
  constexpr int KT = kGqaTile / 16;             // 16-key tiles of the scores
  constexpr int CPR = D / 8;                    // 16-byte chunks per cache row
  constexpr int ROW_B = D * 2;
  constexpr int RSH = 16 / CPR;                 // rows per 256 bytes of LDS
  constexpr int TILE_B = kGqaTile * ROW_B;      // bytes of one K or V tile
  constexpr int NCP = TILE_B / 1024;            // async copies per tile and tensor
  constexpr int STAGE_B = 2 * TILE_B;           // K tile, then V tile
  constexpr float kRescaleStep = 8.f;
  static_assert((kEvenStep / kGqaWaves) % kGqaTile == 0, "a wave's share of a chunk is whole tiles");

  extern __shared__ __attribute__((aligned(1024))) char s_mem[];
  // the per-wave results (m, l, O[d] per query head) go into the first 4.5 KiB of the wave's own ring
  // once its loop is over
  __shared__ float s_m[kGqaWaves][kGqaMaxG];
  __shared__ float s_l[kGqaWaves][kGqaMaxG];
  static_assert(kGqaMaxG * D * 4 <= kGqaStages * STAGE_B, "the result buffer fits the wave's ring");

  const int b = blockIdx.x;   // batch rows side by side (see kGqaBlocksPerCu)
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mcol = lane & 15;   // query head inside the ring (the MFMA column); >= G: padding
  const int g = lane >> 4;      // quarter of the wave
  const uint32_t ring0 = lds_address(s_mem) + wave * (kGqaStages * STAGE_B);   // this wave's stages

  // copy i of a tile moves chunks [64 i, 64 i + 64): chunk c = row * CPR + position
  uint32_t koff[NCP], voff[NCP];
  int crow[NCP];
#pragma unroll
  for (int i = 0; i < NCP; ++i) {
    const int L = i * 64 + lane;
    const int row = L / CPR, pos = L % CPR;
    crow[i] = row;
    koff[i] = (uint32_t)(row * ROW_B + (pos ^ ((row / RSH) % CPR)) * 16);
    voff[i] = (uint32_t)(row * ROW_B + (pos ^ (2 * ((row / RSH) % (CPR / 2)))) * 16);
  }
  // Operand read addresses inside stage 0.  K: sixteen lanes read one chunk of sixteen rows.  V: the transposing read of
  // half a wave covers 32 bytes of each of eight rows, which the permutation spreads over all banks.
  uint32_t k_ad[KS], v_ad[DT];
  {
    const uint32_t k_rd = (uint32_t)(mcol * ROW_B) | (uint32_t)(((g ^ ((mcol / RSH) % CPR)) & (CPR - 1)) * 16);
#pragma unroll
    for (int s = 0; s < KS; ++s) k_ad[s] = ring0 + (k_rd ^ (uint32_t)(64 * s));
    const int v_row = 4 * g + (mcol >> 2);
    const uint32_t v_rd = (uint32_t)(v_row * ROW_B) +
                          (uint32_t)((((mcol & 3) >> 1) ^ (2 * ((v_row / RSH) % (CPR / 2)))) * 16 + 8 * (mcol & 1));
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_ad[dt] = ring0 + TILE_B + (v_rd ^ (uint32_t)(32 * dt));
  }

  const RowChunks<kGqaChunk, true> row(head_valid + (int64_t)b * H, head_start + (int64_t)b * H, H, sumC, cap, target);

  if (MERGE && counters && blockIdx.y == 0) zero_empty_rings(row, o + (int64_t)b * H * G * D, H, G * D);

  for (int w = blockIdx.y; w < row.total; w += gridDim.y) {
    const Chunk ck = row.at(w, H);
    const int c = ck.index, n_chunks = ck.count;
    const int64_t bh = (int64_t)b * H + ck.head;
    const int64_t seg0 = ck.seg0;
    const int64_t len = ck.len;
    const int clen = ck.rows;                  // rows of one chunk of this head
    const int wchunk = clen / kGqaWaves;       // a wave's share: whole tiles
    const int64_t r_begin = (int64_t)c * clen + (int64_t)wave * wchunk;
    int64_t r_end = r_begin + wchunk;
    if (r_end > len) r_end = len;
    const int n_rows = __builtin_amdgcn_readfirstlane(r_end > r_begin ? (int)(r_end - r_begin) : 0);
    const int n_t = (n_rows + kGqaTile - 1) / kGqaTile;
    const char* kbase = reinterpret_cast<const char*>(kc + ((int64_t)b * sumC + seg0 + r_begin) * D);
    const char* vbase = reinterpret_cast<const char*>(vc + ((int64_t)b * sumC + seg0 + r_begin) * D);

    // Q^T fragments: column mcol = query head, k-step s holds Q[mcol][32 s + 8 g .. +7]
    u32x4 qf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4 z = {0, 0, 0, 0};
      qf[s] = (mcol < G) ? *reinterpret_cast<const u32x4*>(q + (bh * G + mcol) * D + 32 * s + 8 * g) : z;
      qf[s] ^= u32x4{q_sign, q_sign, q_sign, q_sign};
    }
    f32x4 oacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;

    // tile t: rows [32 t, 32 t + 32) of the wave's share, into stage t % kGqaStages; rows past the
    // end repeat the last row (their scores are masked)
    auto issue = [&](const char* base, const uint32_t (&off)[NCP], uint32_t dst, int t) __attribute__((always_inline)) {
      const char* src = base + (int64_t)t * TILE_B;
      dst += (t % kGqaStages) * STAGE_B;
      const int last = n_rows - 1 - t * kGqaTile;   // last valid row of the tile, >= 0
      if (last >= kGqaTile - 1) {
#pragma unroll
        for (int i = 0; i < NCP; ++i) async_copy16<NT>(src, off[i], dst + i * 1024);
      } else {
#pragma unroll
        for (int i = 0; i < NCP; ++i)
          async_copy16<NT>(src, off[i] - (uint32_t)(max(crow[i] - last, 0) * ROW_B), dst + i * 1024);
      }
    };
    auto issue_k = [&](int t) __attribute__((always_inline)) { issue(kbase, koff, ring0, t); };
    auto issue_v = [&](int t) __attribute__((always_inline)) { issue(vbase, voff, ring0 + TILE_B, t); };
    static_assert(kGqaStages == 2, "the waits below count two stages");
    if (n_t > 0) { issue_k(0); issue_v(0); }
    if (n_t > 1) { issue_k(1); issue_v(1); }
    // The Q rows are waited for here, by the compiler, which does not know of the copies behind them and waits for those too:
    // the first two tiles have landed when the loop starts.  (Without the pin it would do so inside the loop.)
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s]));

    // K and V of a tile are waited for, and their stages filled again, each by itself: from the first refills on three or
    // four of the wave's four half stages are in flight (with whole tiles one of two stages while a tile is worked on).
    for (int t = 0; t < n_t; ++t) {
      if (t + 1 < n_t) wait_vm(3 * NCP); else wait_vm(NCP);   // K(t) has landed; V(t), K(t+1), V(t+1) may be in flight
      const uint32_t so = (uint32_t)((t % kGqaStages) * STAGE_B);
      // ---- S^T = K . Q^T ----
      f32x4 st[KT];
      {
        u32x4 kf[KT][KS];
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int k = 0; k < KT; ++k) kf[k][s] = lds_load16(k_ad[s] + so, 16 * k * ROW_B);
#pragma unroll
        for (int k = 0; k < KT; ++k) st[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int k = 0; k < KT; ++k) st[k] = M::mfma16(kf[k][s], qf[s], st[k]);
      }
      if (t + kGqaStages < n_t) {
        wait_lds();   // this K stage has been read
        issue_k(t + kGqaStages);
      }
      // ---- softmax over the 32 keys (element i of tile k: key 16 k + 4 g + i) ----
      const int n_valid = n_rows - t * kGqaTile;
      if (n_valid < kGqaTile) {
        const int thr = n_valid - 4 * g;
#pragma unroll
        for (int k = 0; k < KT; ++k)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (16 * k + i >= thr) st[k][i] = -INFINITY;
      }
      // a lane has a quarter of its column's keys: that one of them is too large is seen by the lane that has it, and
      // the column's maximum is needed only then
      float mx = st[0][0];
#pragma unroll
      for (int k = 0; k < KT; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, st[k][i]);
      if (__any(mx * scale_log2 > m_run + kRescaleStep)) {
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = max_with_other_half(mx);
        // an integer reference exponent: the rounding of the weights below is then independent of it
        const float m_new = __builtin_ceilf(fmaxf(m_run, mx * scale_log2));   // finite: key 0 of the tile is valid
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[dt][i] *= alpha;
        m_run = m_new;
      }
      uint32_t pf[4];   // P^T in B-operand order: contraction slot 8 g + 4 k + i is key 16 k + 4 g + i
      float psum = 0.f;
#pragma unroll
      for (int k = 0; k < KT; ++k)
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[k][i], scale_log2, -m_run));
          const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[k][i + 1], scale_log2, -m_run));
          pf[2 * k + (i >> 1)] = M::pack_rne(p0, p1);
          psum += p0 + p1;
        }
      l_run += psum;
      // V(t) has landed; K(t+1), V(t+1), K(t+2) may be in flight
      if (t + 2 < n_t) wait_vm(3 * NCP); else if (t + 1 < n_t) wait_vm(2 * NCP); else wait_vm(0);
      // ---- O^T += V^T . P^T ----
      const u32x4 bfrag = {pf[0], pf[1], pf[2], pf[3]};
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const u32x2 lo = lds_load_tr16(v_ad[dt] + so, 0);
        const u32x2 hi = lds_load_tr16(v_ad[dt] + so, 16 * ROW_B);
        oacc[dt] = M::mfma16(u32x4{lo.x, lo.y, hi.x, hi.y}, bfrag, oacc[dt]);
      }
      if (t + kGqaStages < n_t) {
        wait_lds();   // this V stage has been read
        issue_v(t + kGqaStages);
      }
    }

    // ---- the wave's result per query head: (m, l, O[d]) ----
    {
      float l_tot = l_run + __shfl_xor(l_run, 16, 64);
      l_tot += __shfl_xor(l_tot, 32, 64);
      float* s_acc_w = reinterpret_cast<float*>(s_mem + wave * (kGqaStages * STAGE_B));
      if (mcol < G) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(s_acc_w + mcol * D + 16 * dt + 4 * g) = oacc[dt];
        if (g == 0) {
          s_m[wave][mcol] = m_run;
          s_l[wave][mcol] = l_tot;
        }
      }
    }
    __syncthreads();

    // ---- combine the waves; a thread owns an output column of every second (fourth at D = 64) query head of the ring ----
    {
      const int d = tid % D;
#pragma unroll 2
      for (int gq = tid / D; gq < G; gq += kGqaThreads / D) {
        float Mx = s_m[0][gq];
#pragma unroll
        for (int i = 1; i < kGqaWaves; ++i) Mx = fmaxf(Mx, s_m[i][gq]);
        const float m_use = (Mx == -INFINITY) ? 0.f : Mx;
        float L = 0.f, a = 0.f;
#pragma unroll
        for (int i = 0; i < kGqaWaves; ++i) {
          const float f = fast_exp2(s_m[i][gq] - m_use);
          L += s_l[i][gq] * f;
          a += reinterpret_cast<const float*>(s_mem + i * (kGqaStages * STAGE_B))[gq * D + d] * f;
        }
        if (n_chunks == 1) {
          o[(bh * G + gq) * D + d] = pack1<T>((L > 0.f) ? a / L : 0.f);
        } else {
          const int64_t slot = ((int64_t)b * cap + w) * G + gq;
          store_partial(part_acc + slot * D + d, a, MERGE && counters != nullptr);
          if (d == 0) {
            store_partial(part_ml + slot * 2 + 0, Mx, MERGE && counters != nullptr);
            store_partial(part_ml + slot * 2 + 1, L, MERGE && counters != nullptr);
          }
        }
      }
    }
    if (MERGE && counters && n_chunks > 1 && arrived_last(counters + bh, n_chunks)) {
      // a wave has query heads wave and wave + 4: the loads of both go out together
      typedef WaveMerge<D, true, 16, 16, true> HeadMerge;
      auto part = [&](int gq) __attribute__((always_inline)) {
        const int64_t slot0 = ((int64_t)b * cap + w - c) * G + gq;
        return HeadMerge(part_acc + slot0 * D, reinterpret_cast<const f32x2*>(part_ml) + slot0, G, n_chunks, 0, 1);
      };
      auto finish = [&](int gq, const HeadMerge& h) __attribute__((always_inline)) {
        const Merged<D> m = h.sum();
#pragma unroll
        for (int j = 0; j < D / 64; ++j) o[(bh * G + gq) * D + lane * (D / 64) + j] = pack1<T>((m.L > 0.f) ? m.a[j] / m.L : 0.f);
      };
      static_assert(kGqaMaxG <= 2 * kGqaWaves, "two heads to a wave");
      if (wave + kGqaWaves < G) {
        const HeadMerge h0 = part(wave), h1 = part(wave + kGqaWaves);
        __builtin_amdgcn_sched_barrier(0);
        finish(wave, h0);
        finish(wave + kGqaWaves, h1);
      } else if (wave < G) {
        finish(wave, part(wave));
      }
    }
    __syncthreads();  // s_acc / s_m / s_l are reused by the next chunk
  }
}

constexpr int kChunk = 512;           // cache rows per work-group step of the one-query-head kernel
// Work-groups per CU over the whole grid, never more per batch row than it can have chunks (8 leaves a visible tail, 32 is no
// better).  The batch rows lie side by side, chunk numbers outside (see kGqaBlocksPerCu).  Row by row, with the work-groups
// that find no chunk between the rows, it is a matter of luck which CUs those meet: where a row is a multiple of two, four
// or eight of them, the same ones every time.  GPU time over 9400 random launches (batch 1 to 64, 4 to 40 rings of 64 and
// 128, full and ragged) against row by row with work-groups for the shortest chunks: 0.99 of it below 256 chunks, 0.95 from
// there to four work-groups per CU (0.63 to 1.25, at most 1.07 in 95 of 100), 0.98 above (0.65 to 1.10).  Row by row with
// no more of them than chunks of 512 rows is 0.99 in the middle range, but up to 1.7 where those are an even few: batch 64
// of rings of 700, 500, 200 and 162 rows of 128, 8 places to a row, 11.5 us, 18.9 and, side by side, 12.1.  32 full rings
// of 128, 157888 rows to a batch row, batch 64: 815 -> 807 us, batch 16 210 -> 204.5, batch 8 102.5 -> 101.0.
constexpr int kDecBlocksPerCu = 16;
// Work-groups per CU (full-length chunks by the rings' capacity) below which the chunks are half as long, and from
// which the waves pipeline their own loads.  Half-length chunks pay only where full ones leave CUs idle: 32 rings of 128,
// 288 chunks 17.3 us with half-length, 15.9 with full ones, 469 chunks 26.4 and 23.6, 8 rings 445 chunks 30.6 and 24.5;
// 160 chunks 11.3 with half-length ones.  Pipelining pays where several work-groups follow each other on a CU: 814 chunks of
// 64-element rows 23.5 us with, 22.6 without, 864 of 128 40.2 and 39.6, 1152 49.5 and 49.4, 1440 59.2 both.
constexpr int kDecSmallBelow = 1;
constexpr int kDecPipeFrom = 4;

// From this many bytes of K and V per launch on they are read non-temporally.  What a step reads of one layer
// is read again a token later, after the rings of all other layers: with several layers of this size that is
// past the 256 MB of the last-level cache, and lines kept for it only cost.  Measured with graphs of 16
// layers, ordinary against non-temporal loads: one query head per ring, D = 128, 67 MB a layer 21.2 -> 19.7 us,
// 268 MB 55.4 -> 51.0 us, 2.1 GB 382 -> 337 us (6.4 TB/s); eight query heads 134 MB 36.1 -> 34.7 us, 268 MB
// 57.5 -> 53.9 us.  Below, the rings of some layers do stay cached and ordinary loads win: 16.8 MB a layer
// 14.1 against 15.1 us.
// The launch knows its own layer only.  Where the rings of all layers together stay cached over a step (up to about
// 270 MB, and nothing else read in between: no decoder, whose weights pass through the cache too, but a loop over one
// or a few layers) non-temporal loads lose: one layer of 134 MB, eight query heads, 34.5 -> 37.2 us, of 268 MB 56.4 ->
// 58.6; of 67 MB, seven heads of 64, 25.8 -> 26.8; four of 67 MB, one head, 19.4 -> 20.2.  Four layers of 134 MB already
// win, 37.1 -> 34.9 us, and single ones from 537 MB on, 106.5 -> 93.7 us.
constexpr int64_t kNtBytes = (int64_t)64 << 20;
static inline bool read_nontemporal(int B, int64_t sumC, int D) { return (int64_t)B * sumC * D * 4 >= kNtBytes; }

// Which launches with counters merge inside the split kernel.  What is saved is a launch; what is added stands behind
// every chunk, and where several chunks follow each other on a CU it is no longer hidden.  One query head per ring: the
// launches that do not pipeline their loads (kDecPipeFrom).  GPU time with the merge launch and without, 32 rings of
// 128: 256 rows 7.5 -> 5.9 us, 2048 rows 12.6 -> 11.6 us, batch 4 of 4096 rows (1152 chunks) 49.8 -> 49.6 us, batch 8
// 90.0 -> 92.4 us; a step called from Python, bound by its launches, 24 -> 21 us.
// Skewed rings do not change that: one of 100000 rows beside seven short ones 30.5 -> 25.4 us.
// Grouped kernel: only below kNtBytes (above, a chunk is alone on its CU and nothing hides the merge: batch 4 of 8 rings
// at 32k tokens, 8 query heads, 43.9 us a layer with the merge launch, 46.2 us without, with 32-wide tiles), and by what
// the last work-group of a ring has to do alone.  A wave merges up to two query heads, whose partials it asks for
// together, 16 chunks of each at once.  GPU time of a call among others in a graph, with the merge launch -> without:
//   G = 4, 8 rings of 128:  8 chunks a ring 9.7 -> 9.3 us, 16 10.4 -> 10.2, 32 12.5 -> 13.2
//   G = 2, 8 rings of 128:  8 chunks 9.4 -> 8.7, 16 10.2 -> 9.7, 32 12.0 -> 12.7
//   G = 7, 4 rings of 64:   4 chunks 8.5 -> 8.1, 8 8.5 -> 8.2, 16 8.5 -> 8.6, 32 8.7 -> 10.5
//   G = 8, 8 rings of 128:  2 chunks 10.4 -> 10.3, 4 10.4 -> 10.4, 8 10.5 -> 11.0, 16 10.5 -> 12.1
// Up to 16 chunks of up to four heads, 8 of seven and 4 of eight the launch saved is GPU time won, or it is even; from there
// to the lines it costs at most 0.7 us (1.5 above four heads), less than the host's time for a launch (3.5), which is
// what is won there: a small step called from Python waits for its launches.
// The rings of a plan are not equally long, and the host knows only how many rows they hold together.  So there are two
// bounds: on the chunks of an average ring, where the gain ends, and on the chunks of a whole batch row, which is the
// most its largest ring can have.  One ring with nearly all rows is then the worst case: G = 4, 60 chunks 10.8 -> 12.3 us;
// G = 8, 20 chunks 10.3 -> 12.1 us; without the second bound 235 chunks 22.5 -> 29.2 us and 24.6 -> 45.5 us.
struct MergeInside {
  int64_t ring_chunks, row_chunks;   // at most: of a ring of average size, of a batch row
};
static inline MergeInside merge_inside_up_to(int G) { return G <= kGqaWaves ? MergeInside{32, 64} : MergeInside{16, 24}; }

constexpr int kSmallChunk = kChunk / 2;   // chunk length of the one-query-head kernel when the grid is small

// partial slots per batch row: at most this many chunks exist when the rings do not overlap (sized
// for the shortest chunk any of the kernels uses)
static inline int64_t decode_cap(int64_t sumC, int H) { return (sumC + kSmallChunk - 1) / kSmallChunk + H; }
// every chunk keeps one partial per query head of its ring
static inline size_t decode_slots(int B, int Hq, int Hkv, int64_t sumC) {
  return (size_t)B * (size_t)decode_cap(sumC, Hkv) * (size_t)((Hq + Hkv - 1) / Hkv);
}

template <typename T, int D, int G>
static int launch_decode(const void* q, const void* kc, const void* vc, void* o, float* part_acc,
                         float* part_ml, const int64_t* head_start, const int64_t* head_valid, int B,
                         int H, int64_t sumC, float sm_scale, unsigned* counters, hipStream_t st) {
  const int cap = (int)decode_cap(sumC, H);
  const int64_t chunks = (sumC + kChunk - 1) / kChunk + H;   // per batch row, at the normal chunk length
  const bool pipe = (int64_t)B * chunks >= (int64_t)256 * kDecPipeFrom;
  const bool small = (int64_t)B * chunks < (int64_t)256 * kDecSmallBelow;
  int64_t bx = (256 * kDecBlocksPerCu + B - 1) / B;
  if (bx > (small ? cap : chunks)) bx = small ? cap : chunks;
  if (bx < 1) bx = 1;
  auto launch = [&](auto split, auto merge) {
    hipLaunchKernelGGL(split, dim3(B, (unsigned)bx), dim3(kDecThreads), 0, st, (const uint16_t*)q, (const uint16_t*)kc,
                       (const uint16_t*)vc, (uint16_t*)o, part_acc, part_ml, head_start, head_valid, H, sumC,
                       sm_scale * kLog2e, cap, counters);
    if (int rc = check_launch("moa_decode_fwd(split)")) return rc;
    if (counters) return MOA_OK;
    hipLaunchKernelGGL(merge, dim3(H * G, B), dim3(kDecThreads), 0, st, (uint16_t*)o, part_acc, part_ml, head_start,
                       head_valid, H, G, sumC, cap, 0);
    return check_launch("moa_decode_fwd(merge)");
  };
  if (pipe && !small) counters = nullptr;
  const bool nt = read_nontemporal(B, sumC, D);
  if (small) {
    if (nt) return launch(&decode_split_kernel<T, D, kSmallChunk, G, false, true>, &decode_merge_kernel<T, D, kSmallChunk>);
    return launch(&decode_split_kernel<T, D, kSmallChunk, G, false, false>, &decode_merge_kernel<T, D, kSmallChunk>);
  }
  // the pipelined kernel's launches are past kNtBytes but for short rings of 64-element rows
  if (pipe && nt) return launch(&decode_split_kernel<T, D, kChunk, G, true, true>, &decode_merge_kernel<T, D, kChunk>);
  if (pipe) return launch(&decode_split_kernel<T, D, kChunk, G, true, false>, &decode_merge_kernel<T, D, kChunk>);
  if (nt) return launch(&decode_split_kernel<T, D, kChunk, G, false, true>, &decode_merge_kernel<T, D, kChunk>);
  return launch(&decode_split_kernel<T, D, kChunk, G, false, false>, &decode_merge_kernel<T, D, kChunk>);
}


template <typename T, int D>
static int launch_decode_gqa(const void* q, const void* kc, const void* vc, void* o, float* part_acc,
                             float* part_ml, const int64_t* head_start, const int64_t* head_valid, int B,
                             int H, int G, int64_t sumC, float sm_scale, unsigned* counters, hipStream_t st) {
  const int cap = (int)decode_cap(sumC, H);   // partial slots per batch row the workspace was sized for
  // Chunk policy.  A chunk start costs three dependent memory latencies (ring index, query rows, first tiles), so chunks of
  // kGqaChunk rows are the rule.  Where those leave many CUs idle, all the time or in the last of few rounds, every batch row is split
  // evenly into its share of one or two rounds of 256 chunks instead.  By the number of chunks of kGqaChunk rows, GPU time
  // with those and with (256 chunks, 512 chunks):
  //   D = 128: 54 32.4 (25.8)   129 30.8 us (27.3, 31.1)   140 31.8 (28.7, 32.8)   172 33.2 (33.1)   176 32.6 (33.7, 35.9)
  //     215 37.9 (39.6, 42.0)   258 57.4 (46.2, 48.4)   344 67.6 (59.5, 59.7)   516 88.5 (85.2, 83.5)   688 108.8 (115.7, 109.5)
  //   D = 64: 136 19.2 (17.9, 19.6)   220 21.7 (23.2, 22.3)   264 30.9 (28.9, 29.5)   280 30.2 (29.9, 28.8)
  // The host does not know how full the rings are; it plans with their capacity.
  const int64_t fixed_chunks = (int64_t)B * (sumC / kGqaChunk + (H + 1) / 2);
  int64_t target = 0;   // 0: chunks of kGqaChunk rows; kShortChunks: of kEvenMinChunk
  if (fixed_chunks <= 160 || (fixed_chunks > 240 && fixed_chunks <= 560)) {
    const int64_t all = fixed_chunks <= 400 ? 256 : 512;
    target = fixed_chunks <= 128 ? (all + B - 1) / B : all / B;   // past one round by a few, those cost a round of their own
    if (fixed_chunks > 128 && 2 * target < 3 * H) target = 0;   // short rings: a chunk or two each either way
    if (target > cap) target = cap;
    if (target > 0 && (sumC + kEvenMinChunk - 1) / kEvenMinChunk + H <= target) target = kShortChunks;
  }
  // at most this many chunks per batch row (a work-group without a chunk still holds a CU while it finds that out)
  const int64_t fixed_rows = target == kShortChunks ? kEvenMinChunk : kGqaChunk;
  const int64_t chunks = target > 0 ? target + H : (sumC + fixed_rows - 1) / fixed_rows + H;
  const int64_t chunk_rows = target == kShortChunks ? kEvenMinChunk : target > 0 ? (sumC / target > kEvenMinChunk ? sumC / target : kEvenMinChunk) : kGqaChunk;
  const int64_t ring_chunks = (sumC / H + chunk_rows - 1) / chunk_rows;   // of a ring of average size
  const int64_t row_chunks = (sumC + chunk_rows - 1) / chunk_rows;        // of a ring that is all of the batch row
  const bool nt = read_nontemporal(B, sumC, D);
  const MergeInside limit = merge_inside_up_to(G);
  if (nt || ring_chunks > limit.ring_chunks || row_chunks > limit.row_chunks) counters = nullptr;
  int64_t bx = (256 * kGqaBlocksPerCu + B - 1) / B;   // in practice one work-group per chunk (see kGqaBlocksPerCu)
  if (bx > chunks) bx = chunks;
  if (bx > cap) bx = cap;
  if (bx < 1) bx = 1;
  constexpr size_t lds = gqa_lds_bytes<D>();
  static bool lds_reserved[2][kMaxDevices] = {};   // per template instance
  const auto kernel = nt ? &decode_gqa_kernel<T, D, true> : &decode_gqa_kernel<T, D, false>;
  if (int rc = reserve_lds(reinterpret_cast<const void*>(kernel), lds, lds_reserved[nt], "moa_decode_fwd"))
    return rc;
  hipLaunchKernelGGL(kernel, dim3(B, (unsigned)bx), dim3(kGqaThreads), lds, st,
                     (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, (uint16_t*)o,
                     part_acc, part_ml, head_start, head_valid, H, G, sumC, mfma_softmax_scale(sm_scale), cap,
                     (int)target, counters);
  int rc = check_launch("moa_decode_fwd(grouped split)");
  if (rc || counters) return rc;
  hipLaunchKernelGGL((decode_merge_kernel<T, D, kGqaChunk>), dim3(H * G, B), dim3(kDecThreads), 0, st,
                     (uint16_t*)o, part_acc, part_ml, head_start, head_valid, H, G, sumC, cap, (int)target);
  return check_launch("moa_decode_fwd(merge)");
}

// Launches the decode kernels with their partials in `workspace` (at least
// moa_decode_workspace_bytes(...) bytes; arguments and size are checked by the entry points).
static int decode_dispatch(const void* q, const void* kc, const void* vc, void* o,
                           void* workspace, const int64_t* head_start, const int64_t* head_valid_len,
                           int B, int Hq, int Hkv, int D, int64_t sumC, float sm_scale, int dtype,
                           unsigned* counters, void* stream) {
  const int G = Hq / Hkv;
  const size_t slots = decode_slots(B, Hq, Hkv, sumC);
  float* part_acc = reinterpret_cast<float*>(workspace);
  float* part_ml = part_acc + slots * (size_t)D;
  hipStream_t st = (hipStream_t)stream;
#define MOA_DEC_ARGS q, kc, vc, o, part_acc, part_ml, head_start, head_valid_len, B, Hkv
#define MOA_DEC_TAIL sumC, sm_scale, counters, st
  // one query head per ring: vector ALU kernel; more: matrix-core kernel
  if (dtype == MOA_DTYPE_F16) {
    if (D == 128) return G == 1 ? launch_decode<F16, 128, 1>(MOA_DEC_ARGS, MOA_DEC_TAIL) : launch_decode_gqa<F16, 128>(MOA_DEC_ARGS, G, MOA_DEC_TAIL);
    return G == 1 ? launch_decode<F16, 64, 1>(MOA_DEC_ARGS, MOA_DEC_TAIL) : launch_decode_gqa<F16, 64>(MOA_DEC_ARGS, G, MOA_DEC_TAIL);
  }
  if (D == 128) return G == 1 ? launch_decode<BF16, 128, 1>(MOA_DEC_ARGS, MOA_DEC_TAIL) : launch_decode_gqa<BF16, 128>(MOA_DEC_ARGS, G, MOA_DEC_TAIL);
  return G == 1 ? launch_decode<BF16, 64, 1>(MOA_DEC_ARGS, MOA_DEC_TAIL) : launch_decode_gqa<BF16, 64>(MOA_DEC_ARGS, G, MOA_DEC_TAIL);
#undef MOA_DEC_TAIL
#undef MOA_DEC_ARGS
}

static int decode_check_args(const char* who, const void* q, const void* kc, const void* vc, const void* o,
                             const int64_t* head_start, const int64_t* head_valid_len, int B, int Hq,
                             int Hkv, int D, int64_t sumC, int dtype) {
  if (!q || !kc || !vc || !o || !head_start || !head_valid_len) return fail(MOA_ERR_ARG, "%s: null pointer", who);
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || sumC <= 0) return fail(MOA_ERR_ARG, "%s: B, H, sumC must be positive", who);
  if (B > 65535) return fail(MOA_ERR_UNSUPPORTED, "%s: B <= 65535", who);
  if (sumC >= ((int64_t)1 << 31)) return fail(MOA_ERR_UNSUPPORTED, "%s: at most 2^31 - 1 cache rows per batch row", who);
  if (Hq % Hkv != 0) return fail(MOA_ERR_ARG, "%s: Hq=%d is not a multiple of Hkv=%d", who, Hq, Hkv);
  const int G = Hq / Hkv;
  if (G > kGqaMaxG) return fail(MOA_ERR_UNSUPPORTED, "%s: %d query heads per kv head (at most %d)", who, G, kGqaMaxG);
  if (Hkv > kMaxHeads) return fail(MOA_ERR_UNSUPPORTED, "%s: at most %d kv heads", who, kMaxHeads);
  if (D != 64 && D != 128) return fail(MOA_ERR_UNSUPPORTED, "%s: head_dim %d (64 or 128)", who, D);
  if (dtype != MOA_DTYPE_F16 && dtype != MOA_DTYPE_BF16) return fail(MOA_ERR_UNSUPPORTED, "%s: dtype %d (f16 or bf16)", who, dtype);
  if (!aligned16(q) || !aligned16(kc) || !aligned16(vc) || !aligned16(o))
    return fail(MOA_ERR_ARG, "%s: pointers must be 16-byte aligned", who);
  return MOA_OK;
}

// ---- scratch of the entry point that allocates nothing -------------------------------------------
// The split-K partials of moa_decode_fwd_noalloc live in this file-scope array instead of a caller's
// workspace.  Every GPU the library runs on holds its own copy at its own address until the process
// ends.  In host code the array's name is only a handle for hipGetSymbolAddress: the kernels get the
// device address looked up below, once per device.
static __device__ __align__(256) unsigned char scratch[MOA_DECODE_NOALLOC_MAX_BYTES];

static int noalloc_scratch(void** out) {
  static void* ptr_of_device[kMaxDevices] = {};
  static std::mutex mu;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(MOA_ERR_LAUNCH, "moa_decode_fwd_noalloc: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(MOA_ERR_UNSUPPORTED, "moa_decode_fwd_noalloc: device %d (at most %d devices)", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr_of_device[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));   // the copy of the array on the current device
    if (e != hipSuccess || !p)
      return fail(MOA_ERR_LAUNCH, "moa_decode_fwd_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
    ptr_of_device[dev] = p;
  }
  *out = ptr_of_device[dev];
  return MOA_OK;
}

}  // namespace moa

using namespace moa;

extern "C" size_t moa_decode_workspace_bytes(int B, int Hq, int Hkv, int D, int64_t sumC) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || D <= 0 || sumC <= 0) return 0;
  const size_t slots = decode_slots(B, Hq, Hkv, sumC);
  return ((slots * ((size_t)D + 2) * sizeof(float)) + 255) & ~(size_t)255;
}

extern "C" int moa_decode_fwd(const void* q, const void* kc, const void* vc, void* o, void* workspace,
                              size_t workspace_bytes, const int64_t* head_start,
                              const int64_t* head_valid_len, int B, int Hq, int Hkv, int D, int64_t sumC,
                              float sm_scale, int dtype, void* stream) {
  if (int rc = decode_check_args("moa_decode_fwd", q, kc, vc, o, head_start, head_valid_len, B, Hq, Hkv, D, sumC, dtype))
    return rc;
  const size_t need = moa_decode_workspace_bytes(B, Hq, Hkv, D, sumC);
  if (!workspace || workspace_bytes < need)
    return fail(MOA_ERR_WORKSPACE, "moa_decode_fwd: workspace %zu < %zu bytes", workspace_bytes, need);
  return decode_dispatch(q, kc, vc, o, workspace, head_start, head_valid_len, B, Hq, Hkv, D,
                         sumC, sm_scale, dtype, nullptr, stream);
}

extern "C" int moa_decode_fwd_counted(const void* q, const void* kc, const void* vc, void* o, void* workspace,
                                      size_t workspace_bytes, uint32_t* counters, size_t n_counters,
                                      const int64_t* head_start, const int64_t* head_valid_len, int B, int Hq, int Hkv,
                                      int D, int64_t sumC, float sm_scale, int dtype, void* stream) {
  if (int rc = decode_check_args("moa_decode_fwd_counted", q, kc, vc, o, head_start, head_valid_len, B, Hq, Hkv, D, sumC, dtype))
    return rc;
  const size_t need = moa_decode_workspace_bytes(B, Hq, Hkv, D, sumC);
  if (!workspace || workspace_bytes < need)
    return fail(MOA_ERR_WORKSPACE, "moa_decode_fwd_counted: workspace %zu < %zu bytes", workspace_bytes, need);
  if (n_counters < (size_t)B * (size_t)Hkv) counters = nullptr;
  return decode_dispatch(q, kc, vc, o, workspace, head_start, head_valid_len, B, Hq, Hkv, D, sumC, sm_scale, dtype, counters,
                         stream);
}

extern "C" int moa_decode_fwd_noalloc(const void* q, const void* kc, const void* vc, void* o,
                                      const int64_t* head_start, const int64_t* head_valid_len, int B,
                                      int Hq, int Hkv, int D, int64_t sumC, float sm_scale, int dtype,
                                      void* stream) {
  if (int rc = decode_check_args("moa_decode_fwd_noalloc", q, kc, vc, o, head_start, head_valid_len, B, Hq, Hkv, D, sumC, dtype))
    return rc;
  const size_t need = moa_decode_workspace_bytes(B, Hq, Hkv, D, sumC);
  if (need > (size_t)MOA_DECODE_NOALLOC_MAX_BYTES)
    return fail(MOA_ERR_WORKSPACE,
                "moa_decode_fwd_noalloc: these sizes need %zu bytes of partials, the built-in scratch holds %zu; "
                "use moa_decode_fwd with a workspace",
                need, (size_t)MOA_DECODE_NOALLOC_MAX_BYTES);
  void* ws = nullptr;
  if (int rc = noalloc_scratch(&ws)) return rc;
  return decode_dispatch(q, kc, vc, o, ws, head_start, head_valid_len, B, Hq, Hkv, D,
                         sumC, sm_scale, dtype, nullptr, stream);
}
