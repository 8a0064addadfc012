// Block-sparse causal prefill attention for per-head sink + sliding-window
// spans, on the gfx950 matrix cores.
//
// Replaces the reference's prefill kernels (Triton
// _sparse_attention_prefill_moa_fwd_kernel, MoA/kernels/block_sparse_attention_prefill.py:473-629,
// and the external moa_prefill op, MoA/kernels/mixture_of_attention.py:435-444).
// For query block m (64 rows) of a head with ns sink blocks and nl local
// blocks the live key blocks are {0..min(ns-1,m)} U {max(0,m+1-nl)..m}, with
// the causal test inside the diagonal block (:558-580).
//
// Work decomposition
//   * a work item is 256 consecutive query rows (four 64-row query blocks) of
//     one (batch, head); a work-group of 8 waves takes one item at a time, each
//     wave 32 rows of it;
//   * one work-group per CU stays resident for the whole launch and takes items
//     from a queue (a few counters in device memory): the hardware dispatcher
//     hands work-groups to the XCDs strictly round-robin, so with one
//     work-group per item a CU that falls free waits until it is its XCD's turn
//     (measured: 7 % of CU time at the benchmark shape);
//   * wave 0 turns a queue ticket into an item descriptor (base pointers, tile
//     schedule) once and leaves it in LDS; it does so for item i+1 a few
//     iterations before item i ends, and item i's last iteration asks for the
//     Q rows and starts the first copies of item i+1;
//   * a work-group walks the union of the live 64-key tiles of its four query
//     blocks; a wave skips the math of a tile that is dead for ITS query block;
//   * K and V tiles are copied global -> LDS asynchronously (no registers),
//     four stages deep, rows unpadded with XOR-permuted 16-byte chunks so
//     that every operand read is bank-conflict free;
//   * the band of a work-group is walked circularly from the tile whose index is
//     a multiple of the band length, so that neighbouring query tiles of a head
//     (resident on one XCD at the same time) ask for the same tile at the same
//     step and share it in L2.
//
// Matrix layout.  Both GEMMs are computed transposed so that every per-row
// softmax quantity lives in ONE lane:
//   S^T[n][m] = sum_d K[n][d] Q[m][d]      A = K (LDS), B = Q^T (registers)
//   O^T[d][m] = sum_n V[n][d] P[m][n]      A = V^T (LDS, transposing read), B = P^T
// v_mfma_f32_32x32x16 puts column m of the result in lane (m mod 32) of both
// half-waves, so row max / row sum / rescale are lane-local except for one
// exchange with lane+32, and the P tile that leaves the softmax is already in
// B-operand order (the contraction index n may be permuted freely as long as A
// and B agree; the V^T operand is fetched with that same permutation by
// ds_read_b64_tr_b16, which returns 4 consecutive rows of one column).
//
// Schedule.  A tile costs a wave 32 MFMAs (~1000 matrix-core cycles) and about
// as many cycles of softmax VALU work, and the two do not overlap inside one
// wave.  The 8 waves therefore run as two groups of four, one wave of each
// group per SIMD.  Between two work-group barriers (one per tile) group A runs
// its matrix phase (P.V of the previous tile, Q.K^T of the current one) and then
// its softmax; group B, one phase behind, runs the softmax of the previous tile
// and then its matrix phase, so each SIMD has one wave on the matrix pipe and
// one on the vector ALU most of the time.  The matrix phase is free of VALU
// instructions: operand addresses are kept per lane in registers, stage and row
// selection go into the instructions' immediate offsets.
#include "moa_mfma.h"

#include <atomic>
#include <mutex>

namespace moa {

constexpr int kWRows = 32;    // query rows per wave
constexpr int kKV = 64;       // keys per tile (the sparsity block)

// Work queue of one launch: next[x] = items of XCD list x handed out so far, done = work-groups that have
// left.  The queues live in a file-scope device array (every GPU the library runs on holds its own copy; in
// host code the array's name is only a handle for hipGetSymbolAddress).  A launch takes the next of the
// kQueueSlots slots in turn, so launches that overlap on one GPU do not share counters unless more than
// kQueueSlots of them are under way at once.  A slot starts at zero and is left at zero: the last
// work-group to leave a launch clears it.
struct PrefillQueue {
  unsigned next[8];
  unsigned done;
  unsigned pad[7];
};
constexpr int kQueueSlots = 256;
static __device__ __align__(256) PrefillQueue g_prefill_queues[kQueueSlots];
constexpr int kMaxSortedHeads = 512;   // kv heads the span-sorted schedule handles (else: given order)

struct Strides4 {
  int64_t b, h, n;
};

// Everything the kernel is told, as ONE kernel argument: the kernel reads the fields it needs from the
// kernel-argument segment again for every work item (through a pointer the compiler cannot see through),
// so that none of them is held in a scalar register across the item loop.
struct PrefillArgs {
  const uint16_t *q, *k, *v;
  uint16_t* o;
  Strides4 qs, ks, vs, os;
  const int64_t *sink_blocks, *local_blocks;   // spans per kv head: blocks, or tokens with span_shift = 6
  int span_shift;
  PrefillQueue* queue;
  int BH, Hq, group, N, n_qtiles;
  int per_head, Hkv;   // (BH / Hq) * group pairs per kv head in the sorted list; Hq / group
  float scale_log2_signed;
};
typedef const PrefillArgs __attribute__((address_space(4)))* PrefillArgsPtr;

// x / d and x % d for 0 <= x < 2^22, 0 < d < 2^22, through the float reciprocal and one correction step
// each way (the compiler's general 32-bit division is four times as many instructions, and wave 0 does
// a dozen of these per work item on the critical path).
struct DivMod {
  int q, r;
};
__device__ __forceinline__ DivMod divmod_small(int x, int d) {
  int q = (int)((float)x * __builtin_amdgcn_rcpf((float)d));
  int r = x - q * d;
  if (r < 0) { q -= 1; r += d; }
  if (r >= d) { q += 1; r -= d; }
  return {q, r};
}

// ---- what a wave does with a tile -----------------------------------------------------------------
// st: S^T of the current tile; oacc: O^T; pf: P^T of a tile, packed pairs, B-operand order; qf: Q fragments; k_ad, v_ad:
// operand read addresses of the lane in the stages to read.
// Matrix phase of one iteration: P.V of the previous tile and Q.K^T of the current one,
// alternating, operands fetched kAhead MFMAs ahead.  k_ad / v_ad point at the stages to read.
// Slot i: even -> P.V op i/2 (k-step (i/2)/DT, d tile (i/2)%DT), odd -> Q.K^T op i/2
// (half (i/2)%2, k-step (i/2)/2).
template <typename T, int D>
__device__ __forceinline__ void tile_matrix(f32x16 (&st)[2], f32x16 (&oacc)[D / 32], const uint32_t (&pf)[16], const u32x4 (&qf)[D / 16],
                                            const uint32_t (&k_ad)[D / 16], const uint32_t (&v_ad)[D / 32]) {
  constexpr int KS = D / 16, DT = D / 32, ROW_B = D * 2;
  constexpr int kSlots = 4 * DT + 2 * KS;
  constexpr int kAhead = 6;
  u32x4 opnd[kSlots];
  auto fetch = [&](int i) __attribute__((always_inline)) {
    const int j = i >> 1;
    if (i & 1) {
      opnd[i] = lds_load16(k_ad[j >> 1], (j & 1) * 32 * ROW_B);
    } else {
      const int tk = j / DT, dt = j % DT;
      const u32x2 lo = lds_load_tr16(v_ad[dt], (16 * tk) * ROW_B);
      const u32x2 hi = lds_load_tr16(v_ad[dt], (16 * tk + 8) * ROW_B);
      opnd[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
    }
  };
  auto op = [&](int i) __attribute__((always_inline)) {
    const int j = i >> 1;
    if (i & 1) {
      const int nt = j & 1, s = j >> 1;
      if (s == 0) {
        f32x16 z;
#pragma unroll
        for (int e = 0; e < 16; ++e) z[e] = 0.f;
        st[nt] = T::mfma(opnd[i], qf[0], z);
      } else {
        st[nt] = T::mfma(opnd[i], qf[s], st[nt]);
      }
    } else {
      const int tk = j / DT, dt = j % DT;
      const u32x4 bfrag = {pf[4 * tk], pf[4 * tk + 1], pf[4 * tk + 2], pf[4 * tk + 3]};
      oacc[dt] = T::mfma(opnd[i], bfrag, oacc[dt]);
    }
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(i);
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    if (i + kAhead < kSlots) fetch(i + kAhead);
    op(i);
    __builtin_amdgcn_sched_barrier(0);   // keeps the operand reads kAhead MFMAs ahead of their use
  }
}

// Q.K^T only (the first iteration)
template <typename T, int D>
__device__ __forceinline__ void tile_qk(f32x16 (&st)[2], const u32x4 (&qf)[D / 16], const uint32_t (&k_ad)[D / 16]) {
  constexpr int KS = D / 16, ROW_B = D * 2;
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    u32x4 kf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) kf[s] = lds_load16(k_ad[s], nt * 32 * ROW_B);
#pragma unroll
    for (int i = 0; i < 16; ++i) st[nt][i] = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) st[nt] = T::mfma(kf[s], qf[s], st[nt]);
  }
  // The next barrier lets other waves copy over this K stage.  Unlike in tile_matrix nothing else keeps the products, and
  // with them the compiler's wait for these reads, in front of it.
  wait_lds();
}

// P.V only (the last iteration)
template <typename T, int D>
__device__ __forceinline__ void tile_pv(f32x16 (&oacc)[D / 32], const uint32_t (&pf)[16], const uint32_t (&v_ad)[D / 32]) {
  constexpr int DT = D / 32, ROW_B = D * 2;
#pragma unroll
  for (int tk = 0; tk < 4; ++tk) {
    u32x4 vf[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const u32x2 lo = lds_load_tr16(v_ad[dt], (16 * tk) * ROW_B);
      const u32x2 hi = lds_load_tr16(v_ad[dt], (16 * tk + 8) * ROW_B);
      vf[dt] = u32x4{lo.x, lo.y, hi.x, hi.y};
    }
    const u32x4 bfrag = {pf[4 * tk], pf[4 * tk + 1], pf[4 * tk + 2], pf[4 * tk + 3]};
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oacc[dt] = T::mfma(vf[dt], bfrag, oacc[dt]);
  }
}

// mask + online softmax of tile j: st -> pf, updates m_run, l_run (and rescales oacc when needed;
// every P.V issued so far belongs to earlier tiles and has completed in this wave's matrix phase)
template <typename T, int D>
__device__ __forceinline__ void tile_softmax(f32x16 (&st)[2], f32x16 (&oacc)[D / 32], uint32_t (&pf)[16], float& m_run, float& l_run,
                                             bool diagonal, int thr /* row inside the 64-row block, minus the lane's column base */,
                                             bool first, float scale_log2) {
  constexpr int DT = D / 32;
  constexpr float kRescaleLimit = 256.f;   // the reference exponent is raised (and O rescaled) when a lane's 32 weights sum to more
  if (diagonal) {   // causal mask on the diagonal tile
    asm volatile("" : "+v"(thr));   // keeps the 32 compares in this branch instead of 32 hoisted lane masks
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (nt * 32 + 8 * (i >> 2) + (i & 3) > thr) st[nt][i] = -INFINITY;
  }
  // Row sums are plain fp32 adds of the unrounded weights.  (v_dot2_f32_{f16,bf16} of the packed
  // pair with a pair of ones would halve the instruction count, but those instructions stall the
  // MFMA stream of the wave that shares the SIMD: measured 20 % slower per iteration.)
  float psum[2];
  auto weights = [&]() __attribute__((always_inline)) {
    psum[0] = psum[1] = 0.f;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[nt][i], scale_log2, -m_run));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[nt][i + 1], scale_log2, -m_run));
        pf[nt * 8 + (i >> 1)] = T::pack_rne(p0, p1);
        psum[0] += p0;
        psum[1] += p1;
      }
  };
  // The common case needs no row maximum: weights are formed against the reference exponent as it
  // stands, and their sum tells whether that was good enough.  A lane's 32 weights are >= 0, so a sum of
  // at most 2^8 bounds each of them by 2^8 (the 16-bit types hold that with room to spare); a larger
  // sum, or the first live tile (the reference is still -inf and the sum is inf or NaN; the file is
  // compiled without NaN semantics, so that case is asked for by name), takes the path below.  The item's
  // first step goes there at once.
  if (!first) weights();
  if (first || __builtin_expect(__any(m_run == -INFINITY || psum[0] + psum[1] > kRescaleLimit), 0)) {
    float mx = st[0][0];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, st[nt][i]);
    mx = max_with_other_half(mx);
    const float m_cand = mx * scale_log2;   // finite: a live tile has a visible key in every row
    // The reference exponent stays an INTEGER: a weight is then 2^frac * 2^int, and its rounding to the
    // storage type does not depend on the power of two, so the rounded weights (relative to the row's
    // sum) do not depend on the tile order or on how far m_run lags behind the true maximum.
    const float m_new = __builtin_ceilf(fmaxf(m_run, m_cand));
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    l_run *= alpha;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[t][i] *= alpha;
    m_run = m_new;
    weights();
  }
  l_run += psum[0] + psum[1];
}

// A lane's pieces of its row of O, normalised: 16 bytes each, the halves of the wave having swapped 8-byte ones.
template <typename T, int D>
__device__ __forceinline__ void tile_rows(u32x4 (&rows)[D / 32][2], const f32x16 (&oacc)[D / 32], float l_run) {
  const float l_tot = l_run + other_half(l_run);
  const float inv = (l_tot > 0.f) ? 1.f / l_tot : 0.f;
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const f32x16& a = oacc[dt];
      const u32x2 lo = swap_halves(T::pack_rne(a[8 * p + 0] * inv, a[8 * p + 1] * inv), T::pack_rne(a[8 * p + 4] * inv, a[8 * p + 5] * inv));
      const u32x2 hi = swap_halves(T::pack_rne(a[8 * p + 2] * inv, a[8 * p + 3] * inv), T::pack_rne(a[8 * p + 6] * inv, a[8 * p + 7] * inv));
      rows[dt][p] = u32x4{lo.x, hi.x, lo.y, hi.y};
      asm volatile("" : "+v"(rows[dt][p]));
    }
}
// p: the lane's row, 8 elements on for the upper half of the wave
template <int D>
__device__ __forceinline__ void store_rows(uint16_t* p, const u32x4 (&rows)[D / 32][2]) {
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int h = 0; h < 2; ++h) global_store16(p + 32 * dt + 16 * h, rows[dt][h]);
}

template <typename T, int D>
__global__ __launch_bounds__(512, 1) void prefill_kernel(PrefillArgs args_in_kernarg) {
  const PrefillArgsPtr a0 = (PrefillArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();   // the argument above
  constexpr int NW = 8, S = 4;
  constexpr int KS = D / 16;          // MFMA k-steps of the QK^T product
  constexpr int DT = D / 32;          // 32-wide d tiles of the output
  constexpr int CPR = D / 8;          // 16-byte chunks per K/V row
  constexpr int kPfThreads = NW * 64;
  constexpr int kQRows = NW * kWRows; // query rows per work-group
  constexpr int kQBlocks = kQRows / kKV;   // 64-row query blocks per work-group (two waves each)
  constexpr int kStages = S;          // LDS stages per tensor
  constexpr int LPW = CPR / NW;       // async copies per wave per tile and tensor (64 chunks each)
  constexpr int TILE_B = kKV * D * 2; // bytes of one K or V stage (rows unpadded)
  constexpr int ROW_B = D * 2;
  constexpr int RSH = 16 / CPR;       // rows per 256 bytes of LDS (1 at D=128, 2 at D=64)
  constexpr uint32_t kRing = kStages * TILE_B;   // bytes of one tensor's ring (a power of two)
  static_assert(4 * DT == 2 * KS, "P.V and Q.K^T have the same number of MFMAs per tile");

  extern __shared__ __attribute__((aligned(1024))) char s_mem[];
  char* const s_k = s_mem;
  char* const s_v = s_mem + kStages * TILE_B;

  // ---- once per work-group: heads sorted by span ------------------------------------------------
  __shared__ int s_head_of_rank[kMaxSortedHeads], s_ns[kMaxSortedHeads], s_nl[kMaxSortedHeads];
  {
    const int tid = threadIdx.x;
    const int Hkv = a0->Hq / a0->group;
    const int nb = (a0->N + kKV - 1) / kKV;
    const int64_t* sink_blocks = a0->sink_blocks;
    const int64_t* local_blocks = a0->local_blocks;
    const int shift = a0->span_shift;
    if (Hkv <= kMaxSortedHeads) {
      for (int h = tid; h < Hkv; h += kPfThreads) {
        s_ns[h] = (int)max((int64_t)0, min((int64_t)nb, sink_blocks[h] >> shift));
        s_nl[h] = (int)max((int64_t)0, min((int64_t)nb, local_blocks[h] >> shift));
      }
      __syncthreads();
      for (int h = tid; h < Hkv; h += kPfThreads) {
        const int wh = min(nb, s_ns[h] + s_nl[h]);
        int rank = 0;
        for (int j = 0; j < Hkv; ++j) {
          const int wj = min(nb, s_ns[j] + s_nl[j]);
          rank += (wj > wh) || (wj == wh && j < h);
        }
        s_head_of_rank[rank] = h;
      }
    }
  }

  // ---- the LDS ring keeps turning across items ----
  uint32_t cst = (S - 1) * TILE_B;   // ring offset of the stage K(t+S-1) is copied into; V(t+S-2) goes one stage below
  uint32_t rst = 0;                  // ring offset of the stage K(t) is read from
  bool prefetched = false;           // the previous item has started this item's first copies
  u32x4 qf[KS];                      // Q rows of this wave

  // ---- the work queue ---------------------------------------------------------------------------
  // Wave 0 takes a ticket for the item after the one under way (from the own XCD's list while that has
  // items, from the other lists then), turns it into an item descriptor once and leaves it in LDS; every wave
  // reads it from there.  The ticket is taken kTakeLead iterations before the item under way ends, not at its
  // start: a ticket held through a long item starts late, behind tickets handed out after it, and the items
  // of a head then run spread over the launch instead of side by side on their XCD (start order logged per
  // item and replayed through an LRU model of the L2: 37 % of the K/V tile reads miss with tickets taken at
  // the item's start, 22 % with late ones; measured HBM reads of the launch 2.2 GB against 1.2 GB).
  //   [0] n_tiles (-1: no more items)  [1] query tile  [2] ns  [3] nl  [4] lo2  [5] n_sink  [6] n_band  [7] band_rot
  //   [8,9] K base  [10,11] V base  [12,13] Q base (row 0 of the head)  [14,15] O base
  const int my_xcd = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 7;   // XCC_ID
  __shared__ __attribute__((aligned(16))) int s_item[2][16];
  bool own_alive = true;     // wave 0: the own list still had items when last asked
  auto take = [&](int slot) __attribute__((always_inline)) {
    PrefillArgsPtr ap = a0;
    asm volatile("" : "+s"(ap));
    const int BH = ap->BH, group = ap->group, N = ap->N, n_qtiles = ap->n_qtiles;
    const int per_head = ap->per_head, Hkv = ap->Hkv;
    const int full_rounds = BH >> 3, rem = BH & 7;
    auto list_items = [&](int x) __attribute__((always_inline)) {
      const int snake = (full_rounds & 1) ? 7 - x : x;
      return (unsigned)((full_rounds + (snake < rem ? 1 : 0)) * n_qtiles);
    };
    int list = -1;
    unsigned sq = 0;
    const int lane = threadIdx.x & 63;
    int* d = s_item[slot];
    if (own_alive) {
      unsigned t = 0;
      if (lane == 0) t = atomicAdd(&ap->queue->next[my_xcd], 1u);
      sq = (unsigned)__builtin_amdgcn_readfirstlane((int)t);
      if (sq < list_items(my_xcd)) list = my_xcd; else own_alive = false;
    }
    if (list < 0) {
      // lanes 0 to 7 ask how far the lists are handed out: one round trip to memory, also where nothing is left (asking
      // the lists one after the other is seven of them, in which the whole work-group stands still at the end of its
      // last item)
      unsigned out = 0;
      if (lane < 8) out = atomicAdd(&ap->queue->next[lane], 0u);
      const unsigned long long left = __ballot(lane < 8 && out < list_items(lane & 7));
#pragma unroll 1
      for (int i = 1; i < 8; ++i) {
        const int x = (my_xcd + i) & 7;
        if (!((left >> x) & 1)) continue;
        unsigned t = 0;
        if (lane == 0) t = atomicAdd(&ap->queue->next[x], 1u);
        t = (unsigned)__builtin_amdgcn_readfirstlane((int)t);
        if (t < list_items(x)) { list = x; sq = t; break; }
      }
    }
    if (list < 0) {
      if (lane == 0) d[0] = -1;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      return;
    }
    const int nb = (N + kKV - 1) / kKV;
    const bool sorted = Hkv <= kMaxSortedHeads;
    // A list walks its pairs one after the other, late (long) query tiles first.
    const DivMod rq = divmod_small((int)sq, n_qtiles);
    const int round = rq.q;
    const int qt = n_qtiles - 1 - rq.r;
    const int pos = round * 8 + ((round & 1) ? 7 - list : list);   // position in the sorted list
    // sorted list: kv heads by rank; per kv head, batch-major, then the query heads of its group
    const DivMod ph = divmod_small(pos, per_head);   // (kv head rank, place inside the head's pairs)
    const DivMod bg = divmod_small(ph.r, group);     // (batch row, query head inside the group)
    const int hk = sorted ? s_head_of_rank[ph.q] : ph.q;
    const int b = bg.q;
    const int hq = hk * group + bg.r;
    const int ns = sorted ? s_ns[hk] : (int)max((int64_t)0, min((int64_t)nb, ap->sink_blocks[hk] >> ap->span_shift));
    const int nl = sorted ? s_nl[hk] : (int)max((int64_t)0, min((int64_t)nb, ap->local_blocks[hk] >> ap->span_shift));
    const int mb0 = kQBlocks * qt;                              // first query block of the group
    const int mbl = min(kQBlocks * qt + kQBlocks - 1, nb - 1);  // last one that exists
    // tiles of the work-group: sinks [0, hi1], then band [lo2, mbl]
    const int hi1 = min(ns - 1, mbl);
    int lo2 = max(0, mb0 + 1 - nl);
    if (lo2 <= hi1) lo2 = hi1 + 1;
    const int n_sink = hi1 + 1;
    const int n_tiles = n_sink + max(0, mbl - lo2 + 1);
    // The band is walked circularly, starting at the tile whose index is a multiple of the band
    // length: step u visits the band tile congruent to u.  Work-groups of one head whose bands
    // overlap (neighbouring query tiles, resident on the same XCD at the same time) then ask for
    // the same K/V tile at the same step and share it in L2.  The order is free: online softmax
    // does not care, liveness and the causal mask go by tile index.
    const int n_band = n_tiles - n_sink;
    int band_rot = 0;
    if (n_band > 0) {
      band_rot = n_band - divmod_small(lo2, n_band).r;   // in [1, n_band]
      if (band_rot == n_band) band_rot = 0;
    }
    if (lane != 0) return;
    d[0] = n_tiles; d[1] = qt; d[2] = ns; d[3] = nl; d[4] = lo2; d[5] = n_sink; d[6] = n_band; d[7] = band_rot;
    const uint64_t kb = (uint64_t)(ap->k + b * ap->ks.b + hk * ap->ks.h);
    const uint64_t vb = (uint64_t)(ap->v + b * ap->vs.b + hk * ap->vs.h);
    const uint64_t qb = (uint64_t)(ap->q + b * ap->qs.b + hq * ap->qs.h);
    const uint64_t ob = (uint64_t)(ap->o + b * ap->os.b + hq * ap->os.h);
    d[8] = (int)(uint32_t)kb; d[9] = (int)(uint32_t)(kb >> 32); d[10] = (int)(uint32_t)vb; d[11] = (int)(uint32_t)(vb >> 32);
    d[12] = (int)(uint32_t)qb; d[13] = (int)(uint32_t)(qb >> 32); d[14] = (int)(uint32_t)ob; d[15] = (int)(uint32_t)(ob >> 32);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // in LDS before this wave's next barrier
  };
  __syncthreads();   // the sorted heads
  if (threadIdx.x < 64) take(0);
  __syncthreads();

  // Thread 0 counts its work-group out once it has found the lists empty (it takes no ticket after that).
  unsigned left_before = ~0u;   // work-groups that were out already; ~0: not counted out yet
  auto sign_off = [&]() __attribute__((always_inline)) {
    if (threadIdx.x == 0 && left_before == ~0u) left_before = atomicAdd(&a0->queue->done, 1u);
  };

  // An item as the waves see it.
  struct Item {
    int n_tiles, qt, ns, nl, lo2, n_sink, n_band, band_rot;
    const uint16_t *kbase, *vbase, *qbase;
    uint16_t* obase;
  };
  auto read_item = [&](int slot) __attribute__((always_inline)) {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const i32x4* p = reinterpret_cast<const i32x4*>(s_item[slot]);
    const i32x4 a = p[0], b = p[1], c = p[2], e = p[3];
    auto u = [](int x) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(x); };
    Item it;
    it.n_tiles = u(a.x); it.qt = u(a.y); it.ns = u(a.z); it.nl = u(a.w);
    it.lo2 = u(b.x); it.n_sink = u(b.y); it.n_band = u(b.z); it.band_rot = u(b.w);
    auto ptr = [&](int lo, int hi) __attribute__((always_inline)) {
      return ((uint64_t)(uint32_t)u(hi) << 32) | (uint64_t)(uint32_t)u(lo);
    };
    it.kbase = (const uint16_t*)ptr(c.x, c.y);
    it.vbase = (const uint16_t*)ptr(c.z, c.w);
    it.qbase = (const uint16_t*)ptr(e.x, e.y);
    it.obase = (uint16_t*)ptr(e.z, e.w);
    return it;
  };
  // Scalar schedule.  The tile order is piecewise consecutive (sinks, then the band from its
  // rotated start, wrapping once), so the tile of the next step follows from the current one with a
  // few scalar instructions; a step past the last tile repeats the last tile.
  auto first_tile = [&](const Item& it) __attribute__((always_inline)) {
    return it.n_sink > 0 ? 0 : it.lo2 + it.band_rot;
  };
  auto next_tile_of = [&](const Item& it, int j, int t_next) __attribute__((always_inline)) {
    int jn = j + 1;
    jn = (jn > it.lo2 + it.n_band - 1) ? it.lo2 : jn;
    jn = (t_next == it.n_sink) ? it.lo2 + it.band_rot : jn;
    return (t_next >= it.n_tiles) ? j : jn;
  };
  for (int par = 0;; par ^= 1) {
  const Item it = read_item(par);
  const int n_tiles = it.n_tiles;
  if (n_tiles < 0) break;

  // what the waves need of the arguments, read again for every item (the pointer is opaque to the compiler)
  PrefillArgsPtr ap = a0;
  asm volatile("" : "+s"(ap));
  const int64_t qs_n = ap->qs.n, ks_n = ap->ks.n, vs_n = ap->vs.n, os_n = ap->os.n;
  const int N = ap->N;
  const float scale_log2_signed = ap->scale_log2_signed;
  // The row maximum is taken over the unscaled scores, which needs a scale >= 0: a negative softmax
  // scale is moved into Q (sign bits of the packed 16-bit elements flipped, exact) and its magnitude kept.
  const float scale_log2 = __builtin_fabsf(scale_log2_signed);
  const uint32_t q_sign = scale_log2_signed < 0.f ? 0x80008000u : 0u;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));   // per-lane constants are formed again per item instead of living in registers across items
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2;    // 0: group A, 1: group B (one phase behind A)
  const int mcol = lane & 31;   // query row inside the wave's 32 (the MFMA column)
  const int g = lane >> 5;      // half-wave
  const int nb = (N + kKV - 1) / kKV;

  const int mbw = kQBlocks * it.qt + (wave >> 1);             // this wave's query block
  const bool wave_has_rows = mbw < nb;
  // this wave's own live set
  const int w_hi1 = min(it.ns - 1, mbw);
  const int w_lo2 = max(0, mbw + 1 - it.nl);
  auto live_tile = [&](int j) __attribute__((always_inline)) { return wave_has_rows && (j <= w_hi1 || (j >= w_lo2 && j <= mbw)); };
  const int row0 = it.qt * kQRows + wave * kWRows;            // first query row of this wave
  const int64_t m_glob = row0 + mcol;                          // this lane's query row

  // Q fragment (B operand): Q[m][16*ks + 8*g .. +7]; rows past N repeat row N-1 (nothing of theirs is stored)
  auto load_q = [&](const Item& i) __attribute__((always_inline)) {
    const int64_t m_row = min((int64_t)i.qt * kQRows + wave * kWRows + mcol, (int64_t)N - 1);
    const uint16_t* qrow = i.qbase + m_row * qs_n + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = global_load16(qrow + 16 * s);
  };
  // the Q rows are asked for first: theirs is the longest way
  if (!prefetched && n_tiles > 0) load_q(it);
  auto pin_q = [&]() __attribute__((always_inline)) {   // the Q rows have landed: no wait of the compiler's behind this
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s]));
  };

  // ---- async tile copies: wave w, copy i fills chunks [(i*NW+w)*64, +64) of a stage --------
  const uint16_t* const kbase = it.kbase;   // uniform
  const uint16_t* const vbase = it.vbase;
  uint32_t koff[LPW], voff[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int L = (i * NW + wave) * 64 + lane;     // chunk position inside the stage
    const int row = L / CPR, pos = L % CPR;
    koff[i] = 2u * ((uint32_t)(row * ks_n) + (uint32_t)((pos ^ ((row / RSH) % CPR)) * 8));   // bytes
    voff[i] = 2u * ((uint32_t)(row * vs_n) + (uint32_t)((pos ^ (4 * ((row / RSH) % (CPR / 4)))) * 8));
  }
  // rows >= N of the ragged last tile repeat row N-1: their scores are masked, their softmax
  // weight is exactly 0, and a repeated real row is finite
  // a tile is 64 rows: its byte offset inside the head fits 32 bits (checked on the host)
  const uint32_t k_tile_bytes = (uint32_t)(2 * kKV * ks_n), v_tile_bytes = (uint32_t)(2 * kKV * vs_n);
  const int j_ragged = (N % kKV) ? nb - 1 : -1;    // the only tile with rows past N, if any
  auto issue_tile = [&](const uint16_t* base, uint32_t tile_bytes, int64_t stride_n, const uint32_t (&off)[LPW],
                        bool is_k, int j, uint32_t dst) __attribute__((always_inline)) {
    const char* src = reinterpret_cast<const char*>(base) + (uint64_t)(uint32_t)j * tile_bytes;
    if (j != j_ragged) {
#pragma unroll
      for (int i = 0; i < LPW; ++i) async_copy16(src, off[i], dst + i * NW * 1024);
    } else {
      const int last = N - 1 - j * kKV;
#pragma unroll
      for (int i = 0; i < LPW; ++i) {
        const int L = (i * NW + wave) * 64 + lane;
        const int row = L / CPR, pos = L % CPR;
        const int sw = is_k ? ((row / RSH) % CPR) : (4 * ((row / RSH) % (CPR / 4)));
        async_copy16(src, 2u * ((uint32_t)(min(row, last) * stride_n) + (uint32_t)((pos ^ sw) * 8)), dst + i * NW * 1024);
      }
    }
  };
  const uint32_t k_dst0 = lds_address(s_k) + wave * 1024;            // this wave's share of stage 0
  const uint32_t v_dst0 = lds_address(s_v) + wave * 1024;
  // Starts the first copies, K(0..S-2) and V(0..S-3), of item ni into the stages from ring offset r0 on.
  auto start_copies = [&](const Item& ni, uint32_t r0) __attribute__((always_inline)) {
    int j = first_tile(ni);
#pragma unroll
    for (int i = 0; i + 1 < S; ++i) {
      issue_tile(ni.kbase, k_tile_bytes, ks_n, koff, true, j, k_dst0 + ((r0 + i * TILE_B) & (kRing - 1)));
      if (i + 2 < S) issue_tile(ni.vbase, v_tile_bytes, vs_n, voff, false, j, v_dst0 + ((r0 + i * TILE_B) & (kRing - 1)));
      j = next_tile_of(ni, j, i + 1);
    }
  };
  // The item after this one (its descriptor is in the other slot): its Q rows and first copies are asked for now, so that
  // they arrive beside the rest of this item.  The Q registers are free: this item's last Q.K^T is behind.
  auto prefetch_next = [&](uint32_t r0) __attribute__((always_inline)) {
    const Item ni = read_item(par ^ 1);
    if (ni.n_tiles < 0) sign_off();   // the count comes back while the last item is finished
    if (ni.n_tiles <= 0) return false;
    load_q(ni);
    start_copies(ni, r0);
    return true;
  };

  // operand read addresses of this lane: LDS byte address of its row in the stage at the ring position; stage,
  // half and k-step go into the instruction's immediate offset, so the matrix phase needs no VALU work
  uint32_t k_ad[KS], v_ad[DT];
  {
    const uint32_t k_rd = (uint32_t)(mcol * ROW_B) | (uint32_t)(((g ^ ((mcol / RSH) % CPR)) & (CPR - 1)) * 16);
#pragma unroll
    for (int s = 0; s < KS; ++s) k_ad[s] = lds_address(s_k) + rst + (k_rd ^ (uint32_t)(32 * s));
    const int grp16 = lane & 15;
    const int dhalf = (lane >> 4) & 1;
    const int v_row = 4 * g + (grp16 >> 2);
    const uint32_t v_rd = (uint32_t)(v_row * ROW_B) +
                          (uint32_t)(((2 * dhalf + ((grp16 & 3) >> 1)) ^ (4 * ((v_row / RSH) % (CPR / 4)))) * 16 +
                                     8 * (grp16 & 1));
    // V trails K by one step
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_ad[dt] = lds_address(s_v) + ((rst - TILE_B) & (kRing - 1)) + (v_rd ^ (uint32_t)(64 * dt));
  }
  int kd_prev = (rst == 0) ? -(kStages - 1) * TILE_B : TILE_B;   // how far the K read addresses moved in the previous step

  if (n_tiles == 0) {   // nothing is visible from this query tile: zeros (nobody prefetches for such an item)
    if (wave == 0) take(par ^ 1);
    if (wave_has_rows && m_glob < N) {
      uint16_t* orow = it.obase + m_glob * os_n;
      u32x2 z = {0, 0};
#pragma unroll
      for (int i = 0; i < D / 8; ++i) global_store8(orow + 8 * i + 4 * g, z);
    }
    __syncthreads();   // the next descriptor, written by wave 0 above
    prefetched = false;
    continue;
  }
  if (!prefetched) start_copies(it, rst);
  // the item after this one: wave 0 works its descriptor out kTakeLead iterations before this item's last
  // one (every wave sees it after the next barrier), or here when the item is that short
  constexpr int kTakeLead = 6;
  const int t_take = n_tiles - kTakeLead;
  if (wave == 0 && t_take < 1) take(par ^ 1);

  int jt[S];   // tiles of steps t .. t+S-1
  jt[0] = first_tile(it);
#pragma unroll
  for (int i = 1; i < S; ++i) jt[i] = next_tile_of(it, jt[i - 1], i);

  // the zero the accumulators start from is formed per item (a register full of zeros that the compiler
  // keeps across items costs more than it saves)
  float zero = 0.f;
  asm volatile("" : "+v"(zero));
  f32x16 oacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[t][i] = zero;
  f32x16 st[2];              // S^T of the current tile (defined on every path: an undefined one is carried from item to item)
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int i = 0; i < 16; ++i) st[nt][i] = zero;
  uint32_t pf[16];           // P^T of the current tile, packed pairs, B-operand order
#pragma unroll
  for (int i = 0; i < 16; ++i) pf[i] = __builtin_bit_cast(uint32_t, zero);
  float m_run = -INFINITY;   // reference exponent of exp2: an integer, ceil of the row max of scale_log2 * s when it was last set; a later max may pass it by < 8
  float l_run = 0.f;         // this lane's share of the running sum (the lane+32 twin holds the rest)

  auto matrix_phase = [&]() __attribute__((always_inline)) { tile_matrix<T, D>(st, oacc, pf, qf, k_ad, v_ad); };
  auto softmax = [&](int j, bool first) __attribute__((always_inline)) {
    tile_softmax<T, D>(st, oacc, pf, m_run, l_run, j == mbw, (wave & 1) * kWRows + mcol - 4 * g, first, scale_log2);
  };

  // Iteration t: matrix phase = P.V of tile t-1 and Q.K^T of tile t, then softmax phase = tile t.
  // There is one work-group barrier per iteration; group A meets it after its softmax phase, group
  // B after its matrix phase, so B's softmax of tile t runs beside A's matrix phase of tile t+1 and
  // each SIMD holds one wave in either phase.  A wave for which tile t-1 or t is not live still
  // runs the whole matrix phase (with P = 0, or ignoring S), which keeps the loop body a single
  // straight block; it skips the phase when neither is live.  The copies started in iteration t
  // overwrite the stages of K(t-1) and V(t-2), which every wave has finished reading before
  // barrier t-1; the copies started two iterations ago (K(t+1), V(t)) are first read after barrier
  // t, and every wave waits for its own before it.  Iteration n_tiles only finishes P.V of the
  // last tile and starts the next item.
  bool lc_prev = false;        // was tile t-1 live for this wave
  constexpr int n_wait = (S - 2) * 2 * LPW;   // copies started in the last S-2 iterations may still be in flight
  auto advance = [&]() __attribute__((always_inline)) {
    // the operand addresses move to the next stages (K: t+1, V: t)
    const int kd = (rst == (kStages - 1) * TILE_B) ? -(kStages - 1) * TILE_B : TILE_B;
#pragma unroll
    for (int s = 0; s < KS; ++s) k_ad[s] += kd;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_ad[dt] += kd_prev;   // V trails K by one step
    kd_prev = kd;
    rst = (rst + TILE_B) & (kRing - 1);
    cst = (cst + TILE_B) & (kRing - 1);
  };
  auto iteration = [&](int t, auto FIRST) __attribute__((always_inline)) {
    constexpr bool kFirst = decltype(FIRST)::value != 0;
    // ---------------- matrix phase ----------------
    issue_tile(kbase, k_tile_bytes, ks_n, koff, true, jt[S - 1], k_dst0 + cst);
    issue_tile(vbase, v_tile_bytes, vs_n, voff, false, jt[S - 2], v_dst0 + ((cst - TILE_B) & (kRing - 1)));
    const bool lp = lc_prev, lc = live_tile(jt[0]);
    if (kFirst) {
      if (lc) tile_qk<T, D>(st, qf, k_ad);
    } else {
      if (lp || lc) matrix_phase();
    }
    if (grp == 1) { wait_vm(n_wait); phase_barrier(); }
    // ---------------- softmax phase ----------------
    if (lc) {
      softmax(jt[0], kFirst);
    } else if (lp) {   // the next matrix phase this wave runs must add nothing for a dead tile
#pragma unroll
      for (int i = 0; i < 16; ++i) pf[i] = 0;
    }
    advance();
    lc_prev = lc;
#pragma unroll
    for (int i = 0; i + 1 < S; ++i) jt[i] = jt[i + 1];
    jt[S - 1] = next_tile_of(it, jt[S - 1], t + S);
    if (grp == 0) { wait_vm(n_wait); phase_barrier(); }
  };
  // Q and the first copies have landed: those of an item that the one before it started were waited for there
  if (!prefetched) {
    wait_vm(0);
    pin_q();
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s] ^= u32x4{q_sign, q_sign, q_sign, q_sign};
  phase_barrier();               // K(0..2) and V(0..1) are in LDS
  iteration(0, IC<1>{});   // no P.V yet (and no V stage to read)
  for (int t = 1, stop = min(max(t_take, 1), n_tiles);;) {
    for (; t < stop; ++t) iteration(t, IC<0>{});
    if (t == t_take && wave == 0) take(par ^ 1);
    if (t >= n_tiles) break;
    stop = n_tiles;
  }

  // ---- iteration n_tiles: P.V of the last tile; the next item's first copies start here.
  // Every K stage is free by now (K(n_tiles-1) was read before the last barrier) and so are the V
  // stages other than V(n_tiles-1)'s; the next item's tile u goes where this ring position + 1 + u
  // points, which is where its iterations will look for it.  The repeated copies of the last steps
  // may still be under way into those stages: a wave's copies land in the order they were started.
  prefetched = prefetch_next((rst + TILE_B) & (kRing - 1));
  if (lc_prev) tile_pv<T, D>(oacc, pf, v_ad);
  if (grp == 1) phase_barrier();
  advance();
  if (grp == 0) phase_barrier();

  // ---- epilogue: O[m][d] = O^T[d][m] / l ---------------------------------------------------------
  // A lane holds 8-byte pieces of one row; the halves of the wave swap them so that it holds 16 bytes in a row, and two
  // lanes store 32.  Through LDS whole rows could be stored, but the way there and back costs more than the stores of
  // 32-byte pieces.  With the Q rows of the next item asked for an iteration earlier, the accesses through flat pointers
  // gone and a third of the code (every part of the queue was compiled in eight times): 4 x 8192 tokens, 32 heads of 128,
  // 1237 -> 1209 us; 8192 tokens of 64-element heads 194.9 -> 183.6; 32768 tokens, 64 heads, 8453 -> 8340.
  u32x4 rows[DT][2];
  tile_rows<T, D>(rows, oacc, l_run);
  // what the next item has been asked for lands here, before the stores: behind them it would wait for them too
  wait_vm(0);
  pin_q();
  if (m_glob < N) store_rows<D>(it.obase + m_glob * os_n + 8 * g, rows);
  }   // item loop
  // the last work-group to leave clears the queue for the next launch that uses this slot
  sign_off();
  if (threadIdx.x == 0 && left_before == gridDim.x - 1) {
    PrefillQueue* queue = a0->queue;
    for (int x = 0; x < 8; ++x) atomicExch(&queue->next[x], 0u);
    atomicExch(&queue->done, 0u);
  }
}

// ---- launches of short items ----------------------------------------------------------------------
// prefill_kernel pays about 6 us an item outside its tile loop, keeps a CU busy with one item of 256 rows, and three
// steps of an item have only some of its four query blocks live.  Where items are short (short prompts) or few, that is
// much of the launch.  Here a work-group of four waves does ONE item of 128 rows, the hardware dispatcher hands them out,
// and two of them (three at D = 64, by registers) share a CU: one starts or ends beside the other's tile loop, a long
// item runs on beside no one at the speed of a wave alone, and the code is half as long, which counts where every
// instruction is met for the first time.  Long items stay with prefill_kernel: its loop is the faster one (every tile
// read serves 256 rows, neighbours walk their bands in step: 32768 tokens, 64 heads: 8.2 ms there, 11.4 ms here).
// Tile math, layouts and results are those of prefill_kernel; tiles are taken in ascending order.
constexpr int kShortWaves = 4;
constexpr int kShortRows = kShortWaves * kWRows;
struct PrefillShortArgs {
  const uint16_t *q, *k, *v;
  uint16_t* o;
  Strides4 qs, ks, vs, os;
  const int64_t *sink_blocks, *local_blocks;
  int span_shift, BH, Hq, group, N, n_qtiles;
  int one_round;   // the chip holds all work-groups at once
  float scale_log2_signed;
};

template <typename T, int D>
__global__ __launch_bounds__(64 * kShortWaves, 2) void prefill_short_kernel(PrefillShortArgs a) {
  constexpr int NW = kShortWaves;
  constexpr int KS = D / 16, DT = D / 32;
  constexpr int CPR = D / 8;          // 16-byte chunks per K/V row
  constexpr int LPW = CPR / NW;       // async copies per wave per tile and tensor (64 chunks each)
  constexpr int ROW_B = D * 2;
  constexpr uint32_t TILE_B = kKV * ROW_B;
  constexpr int RSH = 16 / CPR;       // rows per 256 bytes of LDS
  constexpr int kCopyRows = 64 * NW / CPR;   // rows from a wave's copy of a tile to its next one
  static_assert(kCopyRows % (16 * RSH) == 0, "the copies of a wave are permuted alike");
  extern __shared__ __attribute__((aligned(1024))) char s_mem[];
  const uint32_t s_k = lds_address(s_mem), s_v = s_k + 2 * TILE_B;   // two stages each

  // ---- the item ------------------------------------------------------------------------------------
  // Work-groups go to the XCDs in turn.  Where the (batch row, head) pairs can be shared out evenly, an XCD has its pairs
  // to itself; late (long) query tiles of all of them come first.  In a launch that the chip holds as a whole (two
  // work-groups to a CU, the later half beside the earlier) the early tiles come in the opposite order, so that a CU has
  // a long item and a short one.
  const int list = blockIdx.x & 7, n_lists = a.BH % 8 == 0 ? 8 : 1;
  const int per_list = n_lists == 8 ? a.BH >> 3 : a.BH;
  const DivMod place = divmod_small((int)(n_lists == 8 ? blockIdx.x >> 3 : blockIdx.x), per_list);
  const int turn = __builtin_amdgcn_readfirstlane(place.q), pair = (n_lists == 8 ? list * per_list : 0) + __builtin_amdgcn_readfirstlane(place.r);
  const int late = (a.n_qtiles + 1) >> 1;
  const int qt = (a.one_round && turn >= late) ? turn - late : a.n_qtiles - 1 - turn;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int mcol = lane & 31;   // query row inside the wave's 32 (the MFMA column)
  const int g = lane >> 5;      // half-wave
  const int N = a.N, nb = (N + kKV - 1) / kKV;
  const DivMod bh = divmod_small(pair, a.Hq);
  const int b = __builtin_amdgcn_readfirstlane(bh.q), hq = __builtin_amdgcn_readfirstlane(bh.r);
  const int hk = __builtin_amdgcn_readfirstlane(divmod_small(hq, a.group).q);
  const int row0 = qt * kShortRows + wave * kWRows;   // first query row of this wave

  u32x4 qf[KS];              // Q fragment; rows past N repeat row N-1 (nothing of theirs is stored)
  {
    const uint16_t* qrow = a.q + b * a.qs.b + hq * a.qs.h + (int64_t)min(row0 + mcol, N - 1) * a.qs.n + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = global_load16(qrow + 16 * s);
  }
  const int ns = (int)max((int64_t)0, min((int64_t)nb, a.sink_blocks[hk] >> a.span_shift));
  const int nl = (int)max((int64_t)0, min((int64_t)nb, a.local_blocks[hk] >> a.span_shift));

  // tiles of the work-group: sinks [0, hi1], then band [lo2, mbl]; of this wave: its own live set
  const int mb0 = 2 * qt, mbl = min(mb0 + 1, nb - 1), mbw = mb0 + (wave >> 1);
  const int hi1 = min(ns - 1, mbl), n_sink = hi1 + 1;
  const int lo2 = max(max(0, mb0 + 1 - nl), n_sink);
  const int n_tiles = n_sink + max(0, mbl - lo2 + 1);
  const int w_hi1 = min(ns - 1, mbw), w_lo2 = max(0, mbw + 1 - nl);
  auto tile_of = [&](int t) __attribute__((always_inline)) { return t < n_sink ? t : lo2 + t - n_sink; };
  auto live_tile = [&](int j) __attribute__((always_inline)) { return mbw < nb && (j <= w_hi1 || (j >= w_lo2 && j <= mbw)); };

  // ---- copies: wave w, copy i fills chunks [(i*NW+w)*64, +64) of a stage -----------------------------
  uint32_t koff, voff;
  const int crow = wave * (64 / CPR) + lane / CPR, cpos = lane % CPR;
  const uint32_t ksw = (uint32_t)((cpos ^ ((crow / RSH) % CPR)) * 16), vsw = (uint32_t)((cpos ^ (4 * ((crow / RSH) % (CPR / 4)))) * 16);
  const uint32_t k_row = (uint32_t)(2 * a.ks.n), v_row_b = (uint32_t)(2 * a.vs.n);   // bytes of a row (a tile's fit 32 bits, unsigned: checked on the host)
  koff = (uint32_t)crow * k_row + ksw;
  voff = (uint32_t)crow * v_row_b + vsw;
  const char* const kbase = reinterpret_cast<const char*>(a.k + b * a.ks.b + hk * a.ks.h);
  const char* const vbase = reinterpret_cast<const char*>(a.v + b * a.vs.b + hk * a.vs.h);
  const int j_ragged = (N % kKV) ? nb - 1 : -1;    // the only tile with rows past N, if any: they repeat row N-1
  auto copy_tile = [&](const char* base, uint32_t row_bytes, uint32_t off, uint32_t swizzle, int j, uint32_t dst)
      __attribute__((always_inline)) {
    const char* src = base + (uint64_t)(uint32_t)j * (uint64_t)(kKV * row_bytes);
    if (j != j_ragged) {
#pragma unroll
      for (int i = 0; i < LPW; ++i) async_copy16(src, off + (uint32_t)(kCopyRows * i) * row_bytes, dst + i * NW * 1024);
    } else {
      const int last = N - 1 - j * kKV;
#pragma unroll
      for (int i = 0; i < LPW; ++i)
        async_copy16(src, (uint32_t)min(crow + kCopyRows * i, last) * row_bytes + swizzle, dst + i * NW * 1024);
    }
  };
  auto copy_k = [&](int t) __attribute__((always_inline)) {
    copy_tile(kbase, k_row, koff, ksw, tile_of(t), s_k + (t & 1) * TILE_B + wave * 1024);
  };
  auto copy_v = [&](int t) __attribute__((always_inline)) {
    copy_tile(vbase, v_row_b, voff, vsw, tile_of(t), s_v + (t & 1) * TILE_B + wave * 1024);
  };
  if (n_tiles > 0) {
    copy_k(0);
    if (n_tiles > 1) copy_k(1);
    copy_v(0);
  }

  // operand read addresses (see prefill_kernel)
  uint32_t k_ad[KS], v_ad[DT];
  {
    const uint32_t k_rd = (uint32_t)(mcol * ROW_B) | (uint32_t)(((g ^ ((mcol / RSH) % CPR)) & (CPR - 1)) * 16);
#pragma unroll
    for (int s = 0; s < KS; ++s) k_ad[s] = s_k + (k_rd ^ (uint32_t)(32 * s));
    const int grp16 = lane & 15, dhalf = (lane >> 4) & 1, v_row = 4 * g + (grp16 >> 2);
    const uint32_t v_rd = (uint32_t)(v_row * ROW_B) +
                          (uint32_t)(((2 * dhalf + ((grp16 & 3) >> 1)) ^ (4 * ((v_row / RSH) % (CPR / 4)))) * 16 +
                                     8 * (grp16 & 1));
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_ad[dt] = s_v + TILE_B + (v_rd ^ (uint32_t)(64 * dt));   // V trails K by one step
  }
  const float scale_log2 = __builtin_fabsf(a.scale_log2_signed);
  const int thr = (wave & 1) * kWRows + mcol - 4 * g;

  f32x16 oacc[DT], st[2];
  uint32_t pf[16];
  {
    float zero = 0.f;
    asm volatile("" : "+v"(zero));
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[t][i] = zero;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      st[0][i] = st[1][i] = zero;
      pf[i] = __builtin_bit_cast(uint32_t, zero);
    }
  }
  float m_run = -INFINITY, l_run = 0.f;
  bool lc_prev = false;

  // A stage is filled again as soon as every wave has read it: a barrier behind the matrix phase, the copies two steps
  // ahead, the softmax, a wait for the copies of the step before, a second barrier.
  auto step = [&](int t, auto FIRST) __attribute__((always_inline)) {
    constexpr bool kFirst = decltype(FIRST)::value != 0;
    const int j = tile_of(t);
    const bool lp = lc_prev, lc = live_tile(j);
    if (kFirst) {
      if (lc) tile_qk<T, D>(st, qf, k_ad);
    } else {
      if (lp || lc) tile_matrix<T, D>(st, oacc, pf, qf, k_ad, v_ad);
    }
    phase_barrier();
    const bool more_v = t + 1 < n_tiles, more_k = t + 2 < n_tiles;
    if (more_k) copy_k(t + 2);
    if (more_v) copy_v(t + 1);
    if (lc) {
      tile_softmax<T, D>(st, oacc, pf, m_run, l_run, j == mbw, thr, kFirst, scale_log2);
    } else if (lp) {   // the next matrix phase this wave runs must add nothing for a dead tile
#pragma unroll
      for (int i = 0; i < 16; ++i) pf[i] = 0;
    }
    const uint32_t flip = (t & 1) ? -TILE_B : TILE_B;   // K(t+1), V(t)
#pragma unroll
    for (int s = 0; s < KS; ++s) k_ad[s] += flip;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_ad[dt] -= flip;
    lc_prev = lc;
    if (more_k) wait_vm(2 * LPW); else if (more_v) wait_vm(LPW); else wait_vm(0);
    phase_barrier();
  };
  if (n_tiles > 0) {
    wait_vm(0);
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s]));   // no wait of the compiler's behind this
    if (a.scale_log2_signed < 0.f) {   // a negative scale goes into Q (see prefill_kernel)
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[s] ^= u32x4{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
    }
    phase_barrier();
    step(0, IC<1>{});
    for (int t = 1; t < n_tiles; ++t) step(t, IC<0>{});
    if (lc_prev) tile_pv<T, D>(oacc, pf, v_ad);
  }
  u32x4 rows[DT][2];
  tile_rows<T, D>(rows, oacc, l_run);
  const int m_row = row0 + mcol;
  if (m_row < N) store_rows<D>(a.o + b * a.os.b + hq * a.os.h + (int64_t)m_row * a.os.n + 8 * g, rows);
}

template <int D, int S>
static size_t prefill_lds_bytes() {
  return (size_t)2 * S * kKV * D * sizeof(uint16_t);   // K stages + V stages
}

// A queue slot for one launch (round robin over the slots) and the number of CUs of the current device.
static int prefill_queue(PrefillQueue** out, int* cus) {
  static PrefillQueue* base_of_device[kMaxDevices] = {};
  static int cus_of_device[kMaxDevices] = {};
  static std::atomic<unsigned> turn{0};
  static std::mutex mu;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(MOA_ERR_LAUNCH, "moa_prefill_fwd: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(MOA_ERR_UNSUPPORTED, "moa_prefill_fwd: device %d", dev);
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!base_of_device[dev]) {
      void* p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(g_prefill_queues));
      if (e != hipSuccess || !p) return fail(MOA_ERR_LAUNCH, "moa_prefill_fwd: hipGetSymbolAddress: %s", hipGetErrorString(e));
      int n = 0;
      e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
      if (e != hipSuccess || n <= 0) return fail(MOA_ERR_LAUNCH, "moa_prefill_fwd: cannot read the CU count");
      cus_of_device[dev] = n;
      base_of_device[dev] = reinterpret_cast<PrefillQueue*>(p);
    }
  }
  *out = base_of_device[dev] + (turn.fetch_add(1) % kQueueSlots);
  *cus = cus_of_device[dev];
  return MOA_OK;
}

// Which launches prefill_short_kernel takes: items are short by the prompt's length (the host does not know the spans), or
// the chip holds all of them at once.  Time against prefill_kernel's on inputs that are not cached, windows of 64-256 and
// of 64-2048 tokens + a share of the prompt, 32 to 128 (batch row, head) pairs:
//   D = 128: 1024 tokens 0.72-0.85, 2048 0.87-0.98, 3072 0.91-1.07 (4096 1.02-1.17, 6144 1.08-1.22 cached)
//   D = 64:  2048 tokens 0.71-0.89, 3072 0.82-0.84, 4096 0.82-0.98 (6144 0.98-1.08 cached)
//   up to two items to a CU: 512 tokens 0.73-0.80, 3072 0.83-0.91, 8192 0.69-0.99, 32768 (1 and 2 pairs) 0.84-0.96
// 2048 tokens, 32 heads of 64: 37.9 -> 33.2 us; 2 x 1500 tokens, 32 heads of 128: 59.5 -> 45.1; 517 tokens: 20.0 -> 15.0;
// 130 tokens: 11.9 -> 7.9.
static bool short_items(int D, int N, int64_t pairs, int cus) {
  const int64_t items = pairs * ((N + kShortRows - 1) / kShortRows);
  if (items > (1 << 21)) return false;   // divmod_small
  return N <= (D == 64 ? 4096 : 2048) || items <= 2 * (int64_t)cus;
}

template <typename T, int D>
static int launch_prefill(const void* q, const void* k, const void* v, void* o, const int64_t* qs,
                          const int64_t* ks, const int64_t* vs, const int64_t* os, int B, int Hq,
                          int Hkv, int N, const int64_t* sink_blocks, const int64_t* local_blocks,
                          int span_shift, float sm_scale, hipStream_t st) {
  constexpr int NW = 8, S = 4;
  constexpr int kQRows = NW * kWRows;
  const int n_qtiles = (N + kQRows - 1) / kQRows;
  const int64_t pairs = (int64_t)B * Hq;
  const int64_t items = pairs * n_qtiles;
  // the queue's ticket arithmetic (divmod_small) is exact below 2^22: tickets of one XCD's list (an eighth
  // of the items) and positions in the list of (batch, head) pairs
  if (items > (1LL << 25) || pairs > (1LL << 22) || N > (1 << 28))
    return fail(MOA_ERR_UNSUPPORTED, "moa_prefill_fwd: too many work items");
  const int BH = (int)pairs;
  // the async copies address a tile row through a 32-bit element offset
  if (64 * ks[2] + D >= (1ll << 31) || 64 * vs[2] + D >= (1ll << 31))
    return fail(MOA_ERR_UNSUPPORTED, "moa_prefill_fwd: k/v token stride too large");
  Strides4 sq = {qs[0], qs[1], qs[2]}, sk = {ks[0], ks[1], ks[2]}, sv = {vs[0], vs[1], vs[2]},
           so = {os[0], os[1], os[2]};
  PrefillQueue* queue = nullptr;
  int cus = 0;
  if (int rc = prefill_queue(&queue, &cus)) return rc;
  if (short_items(D, N, pairs, cus)) {
    PrefillShortArgs a;
    a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v; a.o = (uint16_t*)o;
    a.qs = sq; a.ks = sk; a.vs = sv; a.os = so;
    a.sink_blocks = sink_blocks; a.local_blocks = local_blocks; a.span_shift = span_shift;
    a.BH = BH; a.Hq = Hq; a.group = Hq / Hkv; a.N = N; a.n_qtiles = (N + kShortRows - 1) / kShortRows;
    const int64_t groups = pairs * a.n_qtiles;
    a.one_round = groups <= 2 * (int64_t)cus;
    a.scale_log2_signed = mfma_softmax_scale(sm_scale);
    hipLaunchKernelGGL((prefill_short_kernel<T, D>), dim3((unsigned)groups), dim3(64 * kShortWaves),
                       (prefill_lds_bytes<D, 2>()), st, a);
    return check_launch("moa_prefill_fwd");
  }
  const size_t lds = prefill_lds_bytes<D, S>();
  static bool lds_reserved[kMaxDevices] = {};   // per template instance
  if (int rc = reserve_lds(reinterpret_cast<const void*>(&prefill_kernel<T, D>), lds, lds_reserved, "moa_prefill_fwd"))
    return rc;
  const int64_t groups = items < cus ? items : cus;
  PrefillArgs args;
  args.q = (const uint16_t*)q; args.k = (const uint16_t*)k; args.v = (const uint16_t*)v; args.o = (uint16_t*)o;
  args.qs = sq; args.ks = sk; args.vs = sv; args.os = so;
  args.sink_blocks = sink_blocks; args.local_blocks = local_blocks; args.span_shift = span_shift; args.queue = queue;
  args.BH = BH; args.Hq = Hq; args.group = Hq / Hkv; args.N = N; args.n_qtiles = n_qtiles;
  args.per_head = B * (Hq / Hkv); args.Hkv = Hkv;
  args.scale_log2_signed = mfma_softmax_scale(sm_scale);
  hipLaunchKernelGGL((prefill_kernel<T, D>), dim3((unsigned)groups), dim3(NW * 64), lds, st, args);
  return check_launch("moa_prefill_fwd");
}

static int check_strides(const char* name, const int64_t* s, const void* p) {
  if (!s) return fail(MOA_ERR_ARG, "moa_prefill_fwd: null %s strides", name);
  if (s[3] != 1) return fail(MOA_ERR_ARG, "moa_prefill_fwd: %s must have unit stride along head_dim", name);
  for (int i = 0; i < 3; ++i)
    if (s[i] % 8 != 0)
      return fail(MOA_ERR_ARG, "moa_prefill_fwd: %s stride %d (%lld elements) breaks 16-byte row alignment",
                  name, i, (long long)s[i]);
  if (!aligned16(p)) return fail(MOA_ERR_ARG, "moa_prefill_fwd: %s must be 16-byte aligned", name);
  return MOA_OK;
}

}  // namespace moa

using namespace moa;

static int prefill_fwd(const void* q, const void* k, const void* v, void* o,
                       const int64_t* q_strides, const int64_t* k_strides,
                       const int64_t* v_strides, const int64_t* o_strides, int B, int Hq,
                       int Hkv, int N, int D, const int64_t* sink_blocks,
                       const int64_t* local_blocks, int span_shift, float sm_scale, int dtype, void* stream) {
  if (!q || !k || !v || !o || !sink_blocks || !local_blocks)
    return fail(MOA_ERR_ARG, "moa_prefill_fwd: null pointer");
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0) return fail(MOA_ERR_ARG, "moa_prefill_fwd: B, H, N must be positive");
  if (Hq % Hkv != 0) return fail(MOA_ERR_ARG, "moa_prefill_fwd: Hq=%d is not a multiple of Hkv=%d", Hq, Hkv);
  if (D != 64 && D != 128) return fail(MOA_ERR_UNSUPPORTED, "moa_prefill_fwd: head_dim %d (64 or 128)", D);
  if (dtype != MOA_DTYPE_F16 && dtype != MOA_DTYPE_BF16)
    return fail(MOA_ERR_UNSUPPORTED, "moa_prefill_fwd: dtype %d (f16 or bf16)", dtype);
  int rc;
  if ((rc = check_strides("q", q_strides, q))) return rc;
  if ((rc = check_strides("k", k_strides, k))) return rc;
  if ((rc = check_strides("v", v_strides, v))) return rc;
  if ((rc = check_strides("o", o_strides, o))) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == MOA_DTYPE_F16) {
    if (D == 128) return launch_prefill<PF16, 128>(q, k, v, o, q_strides, k_strides, v_strides, o_strides, B, Hq, Hkv, N, sink_blocks, local_blocks, span_shift, sm_scale, st);
    return launch_prefill<PF16, 64>(q, k, v, o, q_strides, k_strides, v_strides, o_strides, B, Hq, Hkv, N, sink_blocks, local_blocks, span_shift, sm_scale, st);
  }
  if (D == 128) return launch_prefill<PBF16, 128>(q, k, v, o, q_strides, k_strides, v_strides, o_strides, B, Hq, Hkv, N, sink_blocks, local_blocks, span_shift, sm_scale, st);
  return launch_prefill<PBF16, 64>(q, k, v, o, q_strides, k_strides, v_strides, o_strides, B, Hq, Hkv, N, sink_blocks, local_blocks, span_shift, sm_scale, st);
}

extern "C" int moa_prefill_fwd(const void* q, const void* k, const void* v, void* o, const int64_t* q_strides,
                               const int64_t* k_strides, const int64_t* v_strides, const int64_t* o_strides, int B,
                               int Hq, int Hkv, int N, int D, const int64_t* sink_blocks,
                               const int64_t* local_blocks, float sm_scale, int dtype, void* stream) {
  return prefill_fwd(q, k, v, o, q_strides, k_strides, v_strides, o_strides, B, Hq, Hkv, N, D, sink_blocks, local_blocks, 0,
                     sm_scale, dtype, stream);
}

extern "C" int moa_prefill_fwd_tokens(const void* q, const void* k, const void* v, void* o, const int64_t* q_strides,
                                      const int64_t* k_strides, const int64_t* v_strides, const int64_t* o_strides,
                                      int B, int Hq, int Hkv, int N, int D, const int64_t* sink_size,
                                      const int64_t* local_size, float sm_scale, int dtype, void* stream) {
  return prefill_fwd(q, k, v, o, q_strides, k_strides, v_strides, o_strides, B, Hq, Hkv, N, D, sink_size, local_size,
                     6 /* kKV = 64 tokens */, sm_scale, dtype, stream);
}
