// Rotary position embedding of the query and key projections, alone (prompt)
// and fused with the decode-step append into the circular KV cache.
//
// Replaces the step in front of the attention path in the reference's caller
// (MoA/models/llama/modeling_llama.py:238-262): apply_rotary_pos_emb(q, k,
// cos, sin) of transformers 4.44.2 (the reference's pinned dependency,
// requirements.txt:8) followed, in decode, by StaticCircularCache.update
// (MoA/attention/cache_utils.py:1020-1058).  The published formula is
//   x_embed = (x * cos) + (rotate_half(x) * sin),
//   rotate_half(x) = cat(-x[D/2:], x[:D/2]),
// evaluated by torch in the tensors' dtype, that is with one rounding after
// each of the two products and one after the sum.  The kernels round at the
// same three places, so their results are bit-identical to that evaluation.
//
// All kernels are HBM/latency bound byte work: 128-bit accesses, no LDS.  One
// thread owns a PAIR of 16-byte chunks (elements e..e+7 and e+D/2..e+D/2+7 of
// one head row), reads both and writes both, which makes in-place use safe in
// the rotation alone.
#include "moa_ring.h"

// Every product and sum below is rounded on its own, as torch does.  This file must be compiled
// with -ffp-contract=off (the build does): otherwise the compiler contracts the rounded products
// and the sum into v_fma_f16 / v_pk_fma_f16, which rounds once.

namespace moa {

template <int V>
struct IC {
  static constexpr int value = V;
};

constexpr int kRopeThreads = 256;
constexpr int kRopeRowLanes = 16;   // lanes that share one head row in the fused kernel
constexpr int kRopeRowsPerBlock = kRopeThreads / kRopeRowLanes;

struct EF16 {
  static constexpr int kPerChunk = 8;
  static __device__ __forceinline__ float get(const u32x4& c, int i) {
    const uint32_t w = c[i >> 1];
    return (float)__builtin_bit_cast(_Float16, (uint16_t)((i & 1) ? (w >> 16) : (w & 0xffffu)));
  }
  static __device__ __forceinline__ uint32_t bits(float x) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)x);
  }
  static __device__ __forceinline__ float round(float x) { return (float)(_Float16)x; }
};
struct EBF16 {
  static constexpr int kPerChunk = 8;
  static __device__ __forceinline__ float get(const u32x4& c, int i) {
    const uint32_t w = c[i >> 1];
    return __builtin_bit_cast(float, (i & 1) ? (w & 0xffff0000u) : (w << 16));
  }
  static __device__ __forceinline__ uint32_t bits(float x) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)x);
  }
  static __device__ __forceinline__ float round(float x) { return (float)(__bf16)x; }
};
struct EF32 {
  static constexpr int kPerChunk = 4;
  static __device__ __forceinline__ float get(const u32x4& c, int i) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const f32x4 f = __builtin_bit_cast(f32x4, c);
    return f[i];
  }
  static __device__ __forceinline__ uint32_t bits(float x) { return __builtin_bit_cast(uint32_t, x); }
  static __device__ __forceinline__ float round(float x) { return x; }
};

// lo/hi: chunk e..e+k-1 of the first half of a row and the chunk D/2 further; cl/sl, ch/sh: the
// cos and sin chunks at the same places.  Three roundings per element, no fused multiply-add.
template <typename E>
__device__ __forceinline__ void rope_pair(const u32x4& lo, const u32x4& hi, const u32x4& cl, const u32x4& sl,
                                          const u32x4& ch, const u32x4& sh, u32x4& out_lo, u32x4& out_hi) {
  uint32_t ol[E::kPerChunk], oh[E::kPerChunk];
#pragma unroll
  for (int i = 0; i < E::kPerChunk; ++i) {
    const float x1 = E::get(lo, i), x2 = E::get(hi, i);
    // first half: x1*cos + (-x2)*sin = x1*cos - x2*sin (rounding is symmetric, so the sign may move
    // out of the product); second half: x2*cos + x1*sin
    const float a1 = E::round(__fmul_rn(x1, E::get(cl, i)));
    const float b1 = E::round(__fmul_rn(x2, E::get(sl, i)));
    const float a2 = E::round(__fmul_rn(x2, E::get(ch, i)));
    const float b2 = E::round(__fmul_rn(x1, E::get(sh, i)));
    ol[i] = E::bits(__fsub_rn(a1, b1));
    oh[i] = E::bits(__fadd_rn(a2, b2));
  }
  if constexpr (E::kPerChunk == 8) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out_lo[i] = ol[2 * i] | (ol[2 * i + 1] << 16);
      out_hi[i] = oh[2 * i] | (oh[2 * i + 1] << 16);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out_lo[i] = ol[i];
      out_hi[i] = oh[i];
    }
  }
}

// The six chunks a pair needs.
struct PairIn {
  u32x4 lo, hi, cl, ch, sl, sh;
};
__device__ __forceinline__ PairIn load_pair(const char* src, const char* __restrict__ cos_row,
                                            const char* __restrict__ sin_row, int pair, int half_bytes) {
  const size_t o_lo = (size_t)pair * 16, o_hi = o_lo + half_bytes;
  PairIn x;
  x.lo = *reinterpret_cast<const u32x4*>(src + o_lo);
  x.hi = *reinterpret_cast<const u32x4*>(src + o_hi);
  x.cl = *reinterpret_cast<const u32x4*>(cos_row + o_lo);
  x.ch = *reinterpret_cast<const u32x4*>(cos_row + o_hi);
  x.sl = *reinterpret_cast<const u32x4*>(sin_row + o_lo);
  x.sh = *reinterpret_cast<const u32x4*>(sin_row + o_hi);
  return x;
}
template <typename E>
__device__ __forceinline__ void store_pair(const PairIn& x, char* dst, int pair, int half_bytes) {
  const size_t o_lo = (size_t)pair * 16, o_hi = o_lo + half_bytes;
  u32x4 out_lo, out_hi;
  rope_pair<E>(x.lo, x.hi, x.cl, x.sl, x.ch, x.sh, out_lo, out_hi);
  *reinterpret_cast<u32x4*>(dst + o_lo) = out_lo;
  *reinterpret_cast<u32x4*>(dst + o_hi) = out_hi;
}
template <typename E>
__device__ __forceinline__ void rope_row_pair(const char* src, char* dst,
                                              const char* __restrict__ cos_row, const char* __restrict__ sin_row,
                                              int pair, int half_bytes) {
  store_pair<E>(load_pair(src, cos_row, sin_row, pair, half_bytes), dst, pair, half_bytes);
}

struct RopeTensor {
  const char* src;
  char* dst;
  int64_t sb, sh, sn;   // source byte strides (batch, head, token)
  int64_t db, dh, dn;   // destination byte strides
};

// q and k of a whole prompt (or of one step): one thread per chunk pair.  Consecutive threads walk a row,
// then the dimension in which the SOURCE rows lie closer together (heads for views of [B, N, H, D]
// projections, tokens for [B, H, N, D] tensors), so that a wave reads one consecutive piece of memory.
template <typename E>
__global__ __launch_bounds__(kRopeThreads) void rope_kernel(RopeTensor tq, RopeTensor tk,
                                                             const char* __restrict__ cos,
                                                             const char* __restrict__ sin, int64_t cs_sb,
                                                             int64_t cs_sn, int B, int Hq, int Hkv, int N,
                                                             int pairs_per_row, int half_bytes, bool heads_inner) {
  const int64_t idx = (int64_t)blockIdx.x * kRopeThreads + threadIdx.x;
  const int64_t total = (int64_t)B * (Hq + Hkv) * N * pairs_per_row;
  if (idx >= total) return;
  const int pair = (int)(idx % pairs_per_row);
  int64_t row = idx / pairs_per_row;
  int n, hh;
  if (heads_inner) {
    hh = (int)(row % (Hq + Hkv));
    row /= (Hq + Hkv);
    n = (int)(row % N);
    row /= N;
  } else {
    n = (int)(row % N);
    row /= N;
    hh = (int)(row % (Hq + Hkv));
    row /= (Hq + Hkv);
  }
  const int b = (int)row;
  const bool is_q = hh < Hq;
  const RopeTensor& t = is_q ? tq : tk;
  const int h = is_q ? hh : hh - Hq;
  rope_row_pair<E>(t.src + b * t.sb + h * t.sh + n * t.sn, t.dst + b * t.db + h * t.dh + n * t.dn,
                   cos + b * cs_sb + n * cs_sn, sin + b * cs_sb + n * cs_sn, pair, half_bytes);
}

// Decode step: rotate q into q_out, rotate k into its ring slot, copy v into its ring slot, and
// advance the ring bookkeeping exactly as cache_append_kernel does (cache_utils.py:1020-1058).
// One group of 16 lanes per (batch row, query head) and per (batch row, kv head).
template <typename E>
__global__ __launch_bounds__(kRopeThreads) void rope_append_kernel(
    const char* __restrict__ q_new, const char* __restrict__ k_new, const char* __restrict__ v_new,
    int64_t qn_sb, int64_t qn_sh, int64_t kn_sb, int64_t kn_sh, int64_t vn_sb, int64_t vn_sh,
    const char* __restrict__ cos, const char* __restrict__ sin, int64_t cs_sb, char* __restrict__ q_out,
    char* __restrict__ kc, char* __restrict__ vc, int64_t* __restrict__ mask_cache,
    int64_t* __restrict__ update_index, int64_t* __restrict__ valid_len,
    const int64_t* __restrict__ circ_head, const int64_t* __restrict__ circ_size,
    const int64_t* __restrict__ static_size, const int64_t* __restrict__ max_len, int64_t kv_len, int B,
    int Hq, int Hkv, int row_bytes, int64_t sumC) {
  const int lane = threadIdx.x % kRopeRowLanes;
  const int64_t unit = (int64_t)blockIdx.x * kRopeRowsPerBlock + threadIdx.x / kRopeRowLanes;
  if (unit >= (int64_t)B * (Hq + Hkv)) return;
  const int b = (int)(unit / (Hq + Hkv));
  const int r = (int)(unit % (Hq + Hkv));
  const int half_bytes = row_bytes / 2;
  const int pairs = half_bytes / 16;
  const char* cos_row = cos + b * cs_sb;
  const char* sin_row = sin + b * cs_sb;
  if (r < Hq) {
    const char* src = q_new + b * qn_sb + r * qn_sh;
    char* dst = q_out + ((size_t)b * Hq + r) * row_bytes;
    for (int p = lane; p < pairs; p += kRopeRowLanes) rope_row_pair<E>(src, dst, cos_row, sin_row, p, half_bytes);
    return;
  }
  // Every load goes out before the first one is waited for: the launch is three memory latencies otherwise (the
  // slot, the rows, the bookkeeping).
  const int h = r - Hq;
  const int64_t bh = (int64_t)b * Hkv + h;
  const int units = row_bytes / 16;
  const char* const ksrc = k_new + b * kn_sb + h * kn_sh;
  const char* const vsrc = v_new + b * vn_sb + h * vn_sh;
  PairIn k0 = {};
  u32x4 v0 = {};
  if (lane < pairs) k0 = load_pair(ksrc, cos_row, sin_row, lane, half_bytes);
  if (lane < units) v0 = *reinterpret_cast<const u32x4*>(vsrc + (size_t)lane * 16);
  int64_t idx = update_index[bh], vl = valid_len[bh], ml = max_len[h], ss = static_size[h], chd = circ_head[h],
          csz = circ_size[h];
  asm volatile("" : "+v"(idx), "+v"(vl), "+v"(ml), "+v"(ss), "+v"(chd), "+v"(csz));   // keeps the loads up here
  const bool in_range = idx >= 0 && idx < sumC;
  if (lane == 0) {
    if (in_range && mask_cache != nullptr) mask_cache[(size_t)b * sumC + idx] = 1;
    valid_len[bh] = vl + (vl < ml ? 1 : 0);
    update_index[bh] = next_slot(idx, (kv_len + 1) > ss, chd, csz);
  }
  if (in_range) {
    const size_t dst = ((size_t)b * sumC + idx) * row_bytes;
    if (lane < pairs) store_pair<E>(k0, kc + dst, lane, half_bytes);
    if (lane < units) *reinterpret_cast<u32x4*>(vc + dst + (size_t)lane * 16) = v0;
    for (int p = lane + kRopeRowLanes; p < pairs; p += kRopeRowLanes)
      rope_row_pair<E>(ksrc, kc + dst, cos_row, sin_row, p, half_bytes);
    for (int u = lane + kRopeRowLanes; u < units; u += kRopeRowLanes)
      *reinterpret_cast<u32x4*>(vc + dst + (size_t)u * 16) = *reinterpret_cast<const u32x4*>(vsrc + (size_t)u * 16);
  }
}

// cos and sin chunks of one pair, and the rotation of a row's pair by them: what rope_pair computes, bit for bit, in
// the fewest instructions, for a kernel that keeps the coefficients over the heads of a token.
template <typename E>
struct Coef {
  u32x4 cl, sl, ch, sh;
  __device__ __forceinline__ void rotate(const u32x4& lo, const u32x4& hi, u32x4& out_lo, u32x4& out_hi) const {
    rope_pair<E>(lo, hi, cl, sl, ch, sh, out_lo, out_hi);
  }
};
// f16: packed f16 products and sums.  A product of two f16 is exact in fp32 and a sum of two f16 rounded to fp32 and
// then to f16 is the sum rounded once (24 >= 2 * 11 + 2 bits), so these are the fp32 evaluation's bits.
template <>
struct Coef<EF16> {
  typedef _Float16 h8 __attribute__((ext_vector_type(8)));
  u32x4 cl, sl, ch, sh;
  __device__ __forceinline__ void rotate(const u32x4& lo, const u32x4& hi, u32x4& out_lo, u32x4& out_hi) const {
    const h8 x1 = __builtin_bit_cast(h8, lo), x2 = __builtin_bit_cast(h8, hi);
    const h8 a1 = x1 * __builtin_bit_cast(h8, cl), b1 = x2 * __builtin_bit_cast(h8, sl);
    const h8 a2 = x2 * __builtin_bit_cast(h8, ch), b2 = x1 * __builtin_bit_cast(h8, sh);
    out_lo = __builtin_bit_cast(u32x4, a1 - b1);
    out_hi = __builtin_bit_cast(u32x4, a2 + b2);
  }
};
// bf16: fp32 arithmetic, two values to a conversion
template <>
struct Coef<EBF16> {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  u32x4 cl, sl, ch, sh;
  static __device__ __forceinline__ uint32_t pack(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{x, y}), b2));
  }
  static __device__ __forceinline__ float even(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
  static __device__ __forceinline__ float odd(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
  __device__ __forceinline__ void rotate(const u32x4& lo, const u32x4& hi, u32x4& out_lo, u32x4& out_hi) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p = even(lo[i]), q = odd(lo[i]), r = even(hi[i]), t = odd(hi[i]);
      const uint32_t a1 = pack(__fmul_rn(p, even(cl[i])), __fmul_rn(q, odd(cl[i])));
      const uint32_t b1 = pack(__fmul_rn(r, even(sl[i])), __fmul_rn(t, odd(sl[i])));
      const uint32_t a2 = pack(__fmul_rn(r, even(ch[i])), __fmul_rn(t, odd(ch[i])));
      const uint32_t c2 = pack(__fmul_rn(p, even(sh[i])), __fmul_rn(q, odd(sh[i])));
      out_lo[i] = pack(__fsub_rn(even(a1), even(b1)), __fsub_rn(odd(a1), odd(b1)));
      out_hi[i] = pack(__fadd_rn(even(a2), even(c2)), __fadd_rn(odd(a2), odd(c2)));
    }
  }
};

// The start of a generation in one pass over the projections: q and k of a whole prompt rotated into q_out and k_out,
// kept rows of k stored into their ring slots on the way.  HBM bound, with the vector ALU close behind it: a thread
// per chunk pair that works out its own row and slot takes 1160 us at the size below, so a wave owns a piece of a
// token here, kRopeAtOnce wave-wide loads of its q heads or of its kv heads (consecutive memory): cos and sin are
// fetched once for all of them, and in a kv piece the lanes work out the slots of all kv heads side by side.  A
// rotated row is in registers when its slot is known, so the rings of k cost their writes only.
// The first work-groups take v to the rings: in rings that have just been allocated (FRESH) they walk the rows, fetch
// the v row that belongs into each and zero the rows no token goes to, so no fill runs in front; in rings in use they
// walk the tokens that can be kept, so that a short piece of a prompt does not cost a walk over rings of any size
// (16 tokens into 32 x 8 rings of 8192 rows: 50.6 us by rows, 7.3 by tokens, 10.6 in two steps; 64 tokens into 8 x 32
// rings of 4096: 31.0, 8.0, 13.5).  What a head walks is cut into slices that are numbered head by head, and every wave
// finds its slice's head with one scan over the heads, a lane each: a grid of as many slices for every head as the
// largest has is mostly empty work-groups where heads differ (64 tokens into new rings of 8 x 16384 and 8 x 31 x 256
// rows: 151.6 us, 34.8 by slices; fill and two steps 32.7).
// Batch 8, 32 heads of 128, 16384 tokens, a third of the tokens kept (4.9 GB): 983 us (5.0 TB/s) against 743 us
// rotary + 87 us fill + 268 us insert in separate launches; 64 query heads on 8 rings, batch 1: 103 us.
struct RingArgs {
  const char* v;
  int64_t v_sb, v_sh, v_sn;   // byte strides of v
  char *kc, *vc;
  int64_t *mask_cache;
  const int64_t *update_index, *circ_head, *circ_size, *static_size;
  const int32_t *tok_of, *rank_of, *n_valid;   // with an attention mask, else null
  int64_t kv_len, sumC;
};
constexpr int kRingAtOnce = 4;      // rows a group of 16 lanes has under way
// Rows, or tokens, per work-group of the ring part: 16 KiB of them, once around at 256-byte rows.  Long slices are a chain
// of memory latencies in launches too small to hide them: 2 tokens into new rings of 32 x 512 rows 12.8 us with 256 rows
// to a slice, 9.6 with 128, 8.2 with 64 (in two steps 14); 517 tokens 13.7, 10.7, 8.9; prompt of 8 x 16384 tokens 1002, 984,
// 983; 128-byte rows lose with shorter ones (100 tokens into 32 x 32 rings of 2048: 131, 146, 171).
constexpr __host__ __device__ int ring_rows(int pairs /* chunk pairs per row */) { return pairs >= 8 ? 64 : 512 / pairs; }
// Wave-wide row loads a wave has under way, and all it does.  Measured at the two sizes above, with slices of 256 rows:
// 2: 970 and 103 us, 4: 1000 and 106 us, 8: 950 and 110 us; a whole token (q and k heads in turn) to a wave: 960 and 118.
constexpr int kRopeAtOnce = 2;
// From this many bytes of q and k on they are read, and their rotated copies written, non-temporally: the copies
// are past what the last-level cache (256 MB) could keep for the attention that reads them next, and lines held for
// them only cost (2.1 GB: 1015 -> 975 us a launch).
constexpr int64_t kRopeNtBytes = (int64_t)256 << 20;
template <bool NT>
__device__ __forceinline__ u32x4 load16(const char* p) {
  const u32x4* s = reinterpret_cast<const u32x4*>(p);
  if constexpr (NT) return __builtin_nontemporal_load(s);
  else return *s;
}
template <bool NT>
__device__ __forceinline__ void store16(char* p, u32x4 x) {
  if constexpr (NT) __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(p));
  else *reinterpret_cast<u32x4*>(p) = x;
}
template <typename E, int P /* chunk pairs per row: 64 % P == 0 */, bool FRESH, bool NT>
__global__ __launch_bounds__(kRopeThreads) void rope_insert_kernel(
    RopeTensor tq, RopeTensor tk, const char* __restrict__ cos, const char* __restrict__ sin, int64_t cs_sb,
    int64_t cs_sn, RingArgs ra, int B, int Hq, int Hkv, int N, unsigned ring_blocks,
    int row_blocks /* ring work-groups per batch row */, int64_t walked /* rows or tokens a head walks at most */,
    int pieces /* of a token's heads */) {
  constexpr int half_bytes = P * 16;
  if (blockIdx.x < ring_blocks) {
    constexpr int kRingRows = ring_rows(P);
    const int b = (int)(blockIdx.x / (unsigned)row_blocks), head_lane = threadIdx.x & 63;
    const int64_t nv = ra.n_valid ? (int64_t)ra.n_valid[b] : (int64_t)N;
    HeadRing mine = {0, 0, 0, 0, ra.kv_len};   // of head `head_lane`
    int slices = 0;
    if (head_lane < Hkv) {
      mine = load_ring(ra.update_index, ra.circ_head, ra.circ_size, ra.static_size, ra.kv_len, (int64_t)b * Hkv + head_lane,
                       head_lane);
      const int64_t count = min(FRESH ? mine.s + mine.csz : candidate_count(mine, nv), walked);
      slices = (int)((max(count, (int64_t)0) + kRingRows - 1) / kRingRows);
    }
    const int upto = wave_scan(slices);   // slices of heads 0 .. head_lane
    const int total = __builtin_amdgcn_readlane(upto, 63);
    const int lane = threadIdx.x % kRopeRowLanes;
    const int i = (int)(blockIdx.x % (unsigned)row_blocks);   // one slice to a work-group: a loop takes 130 registers more
    if (i >= total) return;
    const int h = __popcll(__ballot(upto <= i));   // heads whose slices all lie in front of i
    const int slice = i - (h > 0 ? __builtin_amdgcn_readlane(upto, h - 1) : 0);
    const HeadRing g = ring_of_lane(mine, h);
    const int64_t count = min(FRESH ? g.s + g.csz : candidate_count(g, nv), walked);
    const int64_t first = g.ch - g.s, rows = min(count, (int64_t)(slice + 1) * kRingRows);
    const int row_bytes = 2 * half_bytes, units = row_bytes / 16;
    for (int64_t r0 = (int64_t)slice * kRingRows + threadIdx.x / kRopeRowLanes; r0 < rows;
         r0 += kRopeRowsPerBlock * kRingAtOnce) {
      const char* src[kRingAtOnce];
      size_t dst[kRingAtOnce];
      bool in[kRingAtOnce], keep[kRingAtOnce];
#pragma unroll
      for (int j = 0; j < kRingAtOnce; ++j) {
        const int64_t r = r0 + j * kRopeRowsPerBlock;
        int64_t row = first + r, t = -1;
        if (FRESH) {
          in[j] = r < rows && row >= 0 && row < ra.sumC;
          if (in[j]) t = token_of_row(g, row, nv);
          keep[j] = t >= 0;
        } else {
          keep[j] = r < rows && candidate(g, r, nv, t, row) && row >= 0 && row < ra.sumC;
          in[j] = keep[j];
        }
        if (keep[j] && ra.tok_of) t = ra.tok_of[(int64_t)b * N + t];
        src[j] = ra.v + b * ra.v_sb + h * ra.v_sh + t * ra.v_sn;
        dst[j] = ((size_t)b * ra.sumC + row) * row_bytes;
        if (keep[j] && lane == 0 && ra.mask_cache != nullptr) ra.mask_cache[(size_t)b * ra.sumC + row] = 1;
      }
      for (int u = lane; u < units; u += kRopeRowLanes) {
        u32x4 x[kRingAtOnce];
#pragma unroll
        for (int j = 0; j < kRingAtOnce; ++j) {
          x[j] = u32x4{0, 0, 0, 0};
          if (keep[j]) x[j] = *reinterpret_cast<const u32x4*>(src[j] + (size_t)u * 16);
        }
#pragma unroll
        for (int j = 0; j < kRingAtOnce; ++j) {
          if (keep[j] || (FRESH && in[j])) *reinterpret_cast<u32x4*>(ra.vc + dst[j] + (size_t)u * 16) = x[j];
          if (FRESH && in[j] && !keep[j]) *reinterpret_cast<u32x4*>(ra.kc + dst[j] + (size_t)u * 16) = x[j];
        }
      }
    }
    return;
  }
  constexpr int R = 64 / P;           // rows per wave-wide load
  const int lane = threadIdx.x & 63;
  const unsigned unit = (blockIdx.x - ring_blocks) * (kRopeThreads / 64) +
                        (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned token = unit / (unsigned)pieces, piece = unit % (unsigned)pieces;
  if (token >= (unsigned)B * (unsigned)N) return;
  const int b = (int)(token / (unsigned)N), n = (int)(token % (unsigned)N);
  const int sub = lane / P;
  const size_t o_lo = (size_t)(lane % P) * 16;

  Coef<E> w;
  {
    const char* c = cos + b * cs_sb + n * cs_sn + o_lo;
    const char* s = sin + b * cs_sb + n * cs_sn + o_lo;
    w.cl = *reinterpret_cast<const u32x4*>(c);
    w.ch = *reinterpret_cast<const u32x4*>(c + half_bytes);
    w.sl = *reinterpret_cast<const u32x4*>(s);
    w.sh = *reinterpret_cast<const u32x4*>(s + half_bytes);
  }
  auto walk = [&](const RopeTensor& t, int h0, int H, auto RING) __attribute__((always_inline)) {
    const char* const src = t.src + b * t.sb + n * t.sn + o_lo;
    char* const dst = t.dst + b * t.db + n * t.dn + o_lo;
    u32x4 lo[kRopeAtOnce], hi[kRopeAtOnce];
#pragma unroll
    for (int j = 0; j < kRopeAtOnce; ++j) {
      const int h = h0 + j * R + sub;
      if (h < H) {
        const char* p = src + h * t.sh;
        lo[j] = load16<NT>(p);
        hi[j] = load16<NT>(p + half_bytes);
      }
    }
    int slot = -1;   // ring row of the token in head `lane`, -1 if it is not kept
    if (decltype(RING)::value && lane < Hkv) {
      const HeadRing g = load_ring(ra.update_index, ra.circ_head, ra.circ_size, ra.static_size, ra.kv_len,
                                   (int64_t)b * Hkv + lane, lane);
      const int64_t a = ra.rank_of ? (int64_t)ra.rank_of[token] : (int64_t)n;
      const int64_t nv = ra.n_valid ? (int64_t)ra.n_valid[b] : (int64_t)N;
      // ring tokens older than the last csz are dropped whatever their slot (:1122-1133)
      if (a >= 0 && (nv - a <= g.csz || g.kv0 + a <= g.s)) {
        const int64_t at = slot_of(g, a);
        if (keep_of(g, at, nv - a) && at >= 0 && at < ra.sumC) slot = (int)at;
      }
    }
#pragma unroll
    for (int j = 0; j < kRopeAtOnce; ++j) {
      const int h = h0 + j * R + sub;
      const int row = decltype(RING)::value ? __shfl(slot, h & 63, 64) : -1;
      if (h < H) {
        u32x4 out_lo, out_hi;
        w.rotate(lo[j], hi[j], out_lo, out_hi);
        char* p = dst + h * t.dh;
        store16<NT>(p, out_lo);
        store16<NT>(p + half_bytes, out_hi);
        if (decltype(RING)::value && row >= 0) {
          char* ring = ra.kc + ((size_t)b * ra.sumC + row) * (2 * half_bytes) + o_lo;
          *reinterpret_cast<u32x4*>(ring) = out_lo;
          *reinterpret_cast<u32x4*>(ring + half_bytes) = out_hi;
        }
      }
    }
  };
  const int first = (int)piece * (R * kRopeAtOnce), q_pieces = (Hq + R * kRopeAtOnce - 1) / (R * kRopeAtOnce);
  if ((int)piece < q_pieces) walk(tq, first, Hq, IC<0>{});
  else walk(tk, first - q_pieces * (R * kRopeAtOnce), Hkv, IC<1>{});
}

static int check_rope_rows(const char* who, const char* name, int D, int eb, const int64_t* strides, int nstr,
                           const void* p) {
  if (!p) return fail(MOA_ERR_ARG, "%s: null %s", who, name);
  if (!strides) return fail(MOA_ERR_ARG, "%s: null %s strides", who, name);
  if (strides[nstr - 1] != 1) return fail(MOA_ERR_ARG, "%s: innermost %s stride must be 1", who, name);
  for (int i = 0; i < nstr - 1; ++i)
    if ((strides[i] * eb) % 16 != 0)
      return fail(MOA_ERR_ARG, "%s: %s stride %d (%lld elements) breaks 16-byte row alignment", who, name, i,
                  (long long)strides[i]);
  if (!aligned16(p)) return fail(MOA_ERR_ARG, "%s: %s must be 16-byte aligned", who, name);
  (void)D;
  return MOA_OK;
}

static int check_head_dim(const char* who, int D, int dtype, int* eb_out) {
  const int eb = elem_bytes(dtype);
  if (eb == 0) return fail(MOA_ERR_ARG, "%s: unknown dtype %d", who, dtype);
  if (D <= 0 || (D * eb) % 32 != 0)
    return fail(MOA_ERR_UNSUPPORTED, "%s: half a head row (head_dim %d, %d-byte elements) is not a multiple of 16 bytes",
                who, D, eb);
  *eb_out = eb;
  return MOA_OK;
}

}  // namespace moa

using namespace moa;

extern "C" int moa_rope_fwd(const void* q, const void* k, void* q_out, void* k_out, const int64_t* q_strides,
                            const int64_t* k_strides, const int64_t* qo_strides, const int64_t* ko_strides,
                            const void* cos, const void* sin, const int64_t* cs_strides, int B, int Hq, int Hkv,
                            int N, int D, int dtype, void* stream) {
  const char* who = "moa_rope_fwd";
  if (B <= 0 || Hq < 0 || Hkv < 0 || Hq + Hkv <= 0 || N <= 0) return fail(MOA_ERR_ARG, "%s: B, H, N must be positive", who);
  int eb = 0, rc;
  if ((rc = check_head_dim(who, D, dtype, &eb))) return rc;
  if (Hq > 0) {
    if ((rc = check_rope_rows(who, "q", D, eb, q_strides, 4, q))) return rc;
    if ((rc = check_rope_rows(who, "q_out", D, eb, qo_strides, 4, q_out))) return rc;
  }
  if (Hkv > 0) {
    if ((rc = check_rope_rows(who, "k", D, eb, k_strides, 4, k))) return rc;
    if ((rc = check_rope_rows(who, "k_out", D, eb, ko_strides, 4, k_out))) return rc;
  }
  if ((rc = check_rope_rows(who, "cos", D, eb, cs_strides, 3, cos))) return rc;
  if ((rc = check_rope_rows(who, "sin", D, eb, cs_strides, 3, sin))) return rc;
  RopeTensor tq = {}, tk = {};
  if (Hq > 0)
    tq = {(const char*)q, (char*)q_out, q_strides[0] * eb, q_strides[1] * eb, q_strides[2] * eb,
          qo_strides[0] * eb, qo_strides[1] * eb, qo_strides[2] * eb};
  if (Hkv > 0)
    tk = {(const char*)k, (char*)k_out, k_strides[0] * eb, k_strides[1] * eb, k_strides[2] * eb,
          ko_strides[0] * eb, ko_strides[1] * eb, ko_strides[2] * eb};
  const int half_bytes = D * eb / 2;
  const int pairs = half_bytes / 16;
  const int64_t total = (int64_t)B * (Hq + Hkv) * N * pairs;
  const int64_t blocks = (total + kRopeThreads - 1) / kRopeThreads;
  if (blocks > 0x7fffffffLL) return fail(MOA_ERR_UNSUPPORTED, "%s: too many rows", who);
  hipStream_t st = (hipStream_t)stream;
  const int64_t csb = cs_strides[0] * eb, csn = cs_strides[1] * eb;
  const RopeTensor& lead = Hq > 0 ? tq : tk;
  const bool heads_inner = lead.sh < lead.sn;
#define MOA_ROPE_LAUNCH(E)                                                                                  \
  hipLaunchKernelGGL(rope_kernel<E>, dim3((unsigned)blocks), dim3(kRopeThreads), 0, st, tq, tk,             \
                     (const char*)cos, (const char*)sin, csb, csn, B, Hq, Hkv, N, pairs, half_bytes, heads_inner)
  if (dtype == MOA_DTYPE_F16) MOA_ROPE_LAUNCH(EF16);
  else if (dtype == MOA_DTYPE_BF16) MOA_ROPE_LAUNCH(EBF16);
  else MOA_ROPE_LAUNCH(EF32);
#undef MOA_ROPE_LAUNCH
  return check_launch(who);
}

extern "C" int moa_rope_cache_append(const void* q_new, const void* k_new, const void* v_new,
                                     const int64_t* qn_strides, const int64_t* kn_strides,
                                     const int64_t* vn_strides, const void* cos, const void* sin,
                                     int64_t cs_stride_b, void* q_out, void* kc, void* vc, int64_t* mask_cache,
                                     int64_t* update_index, int64_t* valid_len, const int64_t* circ_head,
                                     const int64_t* circ_size, const int64_t* static_size, const int64_t* max_len,
                                     int64_t kv_len, int B, int Hq, int Hkv, int D, int64_t sumC, int dtype,
                                     void* stream) {
  const char* who = "moa_rope_cache_append";
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || sumC <= 0) return fail(MOA_ERR_ARG, "%s: B, Hq, Hkv, sumC must be positive", who);
  if (!update_index || !valid_len || !circ_head || !circ_size || !static_size || !max_len)
    return fail(MOA_ERR_ARG, "%s: null index array", who);
  if (!kc || !vc || !q_out) return fail(MOA_ERR_ARG, "%s: null kc, vc or q_out", who);
  int eb = 0, rc;
  if ((rc = check_head_dim(who, D, dtype, &eb))) return rc;
  if ((rc = check_rope_rows(who, "q_new", D, eb, qn_strides, 3, q_new))) return rc;
  if ((rc = check_rope_rows(who, "k_new", D, eb, kn_strides, 3, k_new))) return rc;
  if ((rc = check_rope_rows(who, "v_new", D, eb, vn_strides, 3, v_new))) return rc;
  if (!cos || !sin) return fail(MOA_ERR_ARG, "%s: null cos or sin", who);
  if ((cs_stride_b * eb) % 16 != 0 || !aligned16(cos) || !aligned16(sin) || !aligned16(q_out) || !aligned16(kc) ||
      !aligned16(vc))
    return fail(MOA_ERR_ARG, "%s: cos, sin, q_out, kc, vc must be 16-byte aligned rows", who);
  const int64_t units = (int64_t)B * (Hq + Hkv);
  dim3 grid((unsigned)((units + kRopeRowsPerBlock - 1) / kRopeRowsPerBlock));
  hipStream_t st = (hipStream_t)stream;
#define MOA_ROPE_APPEND_LAUNCH(E)                                                                            \
  hipLaunchKernelGGL(rope_append_kernel<E>, grid, dim3(kRopeThreads), 0, st, (const char*)q_new,             \
                     (const char*)k_new, (const char*)v_new, qn_strides[0] * eb, qn_strides[1] * eb,         \
                     kn_strides[0] * eb, kn_strides[1] * eb, vn_strides[0] * eb, vn_strides[1] * eb,         \
                     (const char*)cos, (const char*)sin, cs_stride_b * eb, (char*)q_out, (char*)kc,          \
                     (char*)vc, mask_cache, update_index, valid_len, circ_head, circ_size, static_size,      \
                     max_len, kv_len, B, Hq, Hkv, D * eb, sumC)
  if (dtype == MOA_DTYPE_F16) MOA_ROPE_APPEND_LAUNCH(EF16);
  else if (dtype == MOA_DTYPE_BF16) MOA_ROPE_APPEND_LAUNCH(EBF16);
  else MOA_ROPE_APPEND_LAUNCH(EF32);
#undef MOA_ROPE_APPEND_LAUNCH
  return check_launch(who);
}

extern "C" int moa_rope_prefill_insert(const void* q, const void* k, const void* v, void* q_out, void* k_out,
                                       const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                       const int64_t* qo_strides, const int64_t* ko_strides, const void* cos,
                                       const void* sin, const int64_t* cs_strides, void* kc, void* vc,
                                       int64_t* mask_cache, int64_t* update_index, int64_t* valid_len,
                                       const int64_t* circ_head, const int64_t* circ_size,
                                       const int64_t* static_size, const int64_t* attention_mask, int64_t am_stride,
                                       void* workspace, size_t workspace_bytes, int64_t kv_len, int B, int Hq,
                                       int Hkv, int S, int D, int64_t sumC, int64_t max_cache_size, int zero_rest,
                                       int dtype, void* stream) {
  const char* who = "moa_rope_prefill_insert";
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || S <= 0 || sumC <= 0)
    return fail(MOA_ERR_ARG, "%s: B, Hq, Hkv, S, sumC must be positive", who);
  if (Hkv > 64 || B > 65535) return fail(MOA_ERR_UNSUPPORTED, "%s: Hkv <= 64, B <= 65535", who);
  if (sumC > 0x7fffffffLL) return fail(MOA_ERR_UNSUPPORTED, "%s: at most 2^31 - 1 cache rows per batch row", who);
  if (!update_index || !valid_len || !circ_head || !circ_size || !static_size)
    return fail(MOA_ERR_ARG, "%s: null index array", who);
  if (!kc || !vc || !aligned16(kc) || !aligned16(vc))
    return fail(MOA_ERR_ARG, "%s: kc and vc must be set and 16-byte aligned", who);
  if (max_cache_size <= 0) return fail(MOA_ERR_ARG, "%s: max_cache_size must be positive", who);
  int eb = 0, rc;
  if ((rc = check_head_dim(who, D, dtype, &eb))) return rc;
  if ((rc = check_rope_rows(who, "q", D, eb, q_strides, 4, q))) return rc;
  if ((rc = check_rope_rows(who, "k", D, eb, k_strides, 4, k))) return rc;
  if ((rc = check_rope_rows(who, "v", D, eb, v_strides, 4, v))) return rc;
  if ((rc = check_rope_rows(who, "q_out", D, eb, qo_strides, 4, q_out))) return rc;
  if ((rc = check_rope_rows(who, "k_out", D, eb, ko_strides, 4, k_out))) return rc;
  if ((rc = check_rope_rows(who, "cos", D, eb, cs_strides, 3, cos))) return rc;
  if ((rc = check_rope_rows(who, "sin", D, eb, cs_strides, 3, sin))) return rc;
  const int half_bytes = D * eb / 2;
  const int pairs = half_bytes / 16;
  if (pairs != 2 && pairs != 4 && pairs != 8 && pairs != 16)
    return fail(MOA_ERR_UNSUPPORTED, "%s: a head row of %d bytes (64, 128, 256 or 512)", who, 2 * half_bytes);
  const int64_t tokens = (int64_t)B * S;
  const int per_piece = 64 / pairs * kRopeAtOnce;   // heads a wave takes
  const int pieces = (Hq + per_piece - 1) / per_piece + (Hkv + per_piece - 1) / per_piece;
  const int64_t units = tokens * pieces;
  const int64_t unit_blocks = (units + kRopeThreads / 64 - 1) / (kRopeThreads / 64);
  // with rings in use: no more candidates than tokens, or than a head's rows + 1 (see candidate())
  const int64_t walked = zero_rest ? max_cache_size : max_cache_size < S ? max_cache_size + 1 : S;
  // slices of a batch row: of all heads alike, or where heads differ as many as their rows or tokens together make
  const int slice_rows = ring_rows(pairs);
  const int64_t slices = (int64_t)Hkv * ((walked + slice_rows - 1) / slice_rows);
  const int64_t together = (sumC + (zero_rest ? 0 : Hkv)) / slice_rows + Hkv;
  const int64_t row_blocks = slices < together ? slices : together;
  const int64_t ring_blocks = (int64_t)B * row_blocks;
  const int64_t blocks = unit_blocks + ring_blocks;
  // a launch holds less than 2^32 threads
  if (units > 0x7fffffffLL || blocks * kRopeThreads > 0xffffffffLL)
    return fail(MOA_ERR_UNSUPPORTED, "%s: too many tokens", who);
  hipStream_t st = (hipStream_t)stream;
  RingArgs ra = {(const char*)v, v_strides[0] * eb, v_strides[1] * eb, v_strides[2] * eb, (char*)kc, (char*)vc, mask_cache,
                 update_index, circ_head, circ_size, static_size, nullptr, nullptr, nullptr, kv_len, sumC};
  if (attention_mask != nullptr) {
    const size_t need = moa_cache_prefill_workspace_bytes(B, S);
    if (workspace == nullptr || workspace_bytes < need)
      return fail(MOA_ERR_WORKSPACE, "%s: workspace %zu < %zu bytes", who, workspace_bytes, need);
    int32_t* tok_of = reinterpret_cast<int32_t*>(workspace);
    int32_t* rank_of = tok_of + (size_t)B * (size_t)S;
    int32_t* n_valid = rank_of + (size_t)B * (size_t)S;
    if ((rc = launch_mask_scan(attention_mask, am_stride, B, S, tok_of, n_valid, rank_of, st))) return rc;
    ra.tok_of = tok_of;
    ra.rank_of = rank_of;
    ra.n_valid = n_valid;
  }
  const RopeTensor tq = {(const char*)q, (char*)q_out, q_strides[0] * eb, q_strides[1] * eb, q_strides[2] * eb,
                         qo_strides[0] * eb, qo_strides[1] * eb, qo_strides[2] * eb};
  const RopeTensor tk = {(const char*)k, (char*)k_out, k_strides[0] * eb, k_strides[1] * eb, k_strides[2] * eb,
                         ko_strides[0] * eb, ko_strides[1] * eb, ko_strides[2] * eb};
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kRopeThreads), 0, st, tq, tk, (const char*)cos,
                       (const char*)sin, cs_strides[0] * eb, cs_strides[1] * eb, ra, B, Hq, Hkv, S, (unsigned)ring_blocks,
                       (int)row_blocks, walked, pieces);
    return check_launch(who);
  };
  const bool nt = (int64_t)B * S * (Hq + Hkv) * D * eb >= kRopeNtBytes;
  auto by_options = [&](auto e, auto p) {
    typedef decltype(e) E;
    constexpr int P = decltype(p)::value;
    if (nt) return zero_rest ? launch(&rope_insert_kernel<E, P, true, true>) : launch(&rope_insert_kernel<E, P, false, true>);
    return zero_rest ? launch(&rope_insert_kernel<E, P, true, false>) : launch(&rope_insert_kernel<E, P, false, false>);
  };
  auto by_row = [&](auto e) {
    switch (pairs) {
      case 2: return by_options(e, IC<2>{});
      case 4: return by_options(e, IC<4>{});
      case 8: return by_options(e, IC<8>{});
      default: return by_options(e, IC<16>{});
    }
  };
  rc = dtype == MOA_DTYPE_F16 ? by_row(EF16{}) : dtype == MOA_DTYPE_BF16 ? by_row(EBF16{}) : by_row(EF32{});
  if (rc) return rc;
  // behind the copy on the same stream: it overwrites update_index, which the copy reads
  return launch_prefill_index(update_index, valid_len, circ_head, circ_size, static_size, ra.n_valid, kv_len, B, Hkv, S, st);
}
