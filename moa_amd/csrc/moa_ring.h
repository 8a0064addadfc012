// The ring arithmetic of a prompt's bulk insert (cache_utils.py:1060-1164), shared by the insert kernels.
#pragma once
#include "moa_common.h"

namespace moa {

struct HeadRing {
  int64_t upd0;   // cache_update_index before the call
  int64_t ch;     // first ring row
  int64_t csz;    // ring rows
  int64_t s;      // static_cache_size
  int64_t kv0;    // _kv_len before the call
};

__device__ __forceinline__ HeadRing load_ring(const int64_t* update_index, const int64_t* circ_head,
                                              const int64_t* circ_size, const int64_t* static_size,
                                              int64_t kv_len, int64_t bh, int h) {
  HeadRing g;
  g.upd0 = update_index[bh];
  g.ch = circ_head[h];
  g.csz = circ_size[h];
  g.s = static_size[h];
  g.kv0 = kv_len;
  return g;
}

// the ring that lane h of the wave holds (h is uniform, and kv0 the same in all lanes)
__device__ __forceinline__ int64_t value_of_lane(int64_t x, int h) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, h);
  return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), h) << 32) | lo);
}
__device__ __forceinline__ HeadRing ring_of_lane(const HeadRing& x, int h) {
  return {value_of_lane(x.upd0, h), value_of_lane(x.ch, h), value_of_lane(x.csz, h), value_of_lane(x.s, h), x.kv0};
}

// py_mod(off, csz); offsets and rings of ordinary size take the 32-bit division (a fifth of the instructions).
__device__ __forceinline__ int64_t ring_mod(int64_t off, int64_t csz) {
  if ((uint64_t)off < (1ull << 32) && (uint64_t)(csz - 1) < (1ull << 31)) return (int64_t)((uint32_t)off % (uint32_t)csz);
  return py_mod(off, csz);
}

// Slot of the token whose advancing position is `a` (:1088-1107).
__device__ __forceinline__ int64_t slot_of(const HeadRing& g, int64_t a) {
  const bool circ = (g.kv0 + a) > g.s;
  return circ ? ring_mod(g.upd0 + a - g.ch, g.csz) + g.ch : g.upd0 + a;
}

// Keep rule (:1122-1133) without the mask term.
__device__ __forceinline__ bool keep_of(const HeadRing& g, int64_t slot, int64_t rap) {
  return (rap <= g.csz) || (slot < g.ch);
}

// Candidate r -> the token with advancing position a (its index among the row's valid tokens; without a
// mask every token is valid and a is the token's position).  Only tokens that can be kept are
// enumerated: r < csz walks the valid tokens from the last one backwards (these have
// rap = r+1 <= csz); r >= csz walks the first ones (the only ones whose slot can lie in the static
// part); any other token is a ring token older than the last csz and is dropped by the keep rule.
// n_valid: valid tokens of the batch row.  Returns whether the candidate is kept, with a and its slot.
__device__ __forceinline__ bool candidate(const HeadRing& g, int64_t r, int64_t n_valid, int64_t& a, int64_t& slot) {
  if (r < g.csz) {
    a = n_valid - 1 - r;
    if (a < 0) return false;
  } else {
    a = r - g.csz;
    if (a >= n_valid - g.csz || a > g.s) return false;
  }
  const int64_t rap = n_valid - a;   // valid tokens at or after this one (:1081-1086)
  slot = slot_of(g, a);
  return keep_of(g, slot, rap);
}
// how many candidates a head has
__device__ __forceinline__ int64_t candidate_count(const HeadRing& g, int64_t n_valid) {
  return min(n_valid, g.csz + g.s + 1);
}

// The advancing position of the token that the insert of n_valid tokens leaves in `row` of the head's own segment, -1
// for none.  The inverse of slot_of and keep_of: a token in front of the ring's turn sits at upd0 + a; of the ring's
// tokens only the last csz are kept, and exactly one of those has the row's residue.
__device__ __forceinline__ int64_t token_of_row(const HeadRing& g, int64_t row, int64_t n_valid) {
  const int64_t a = row - g.upd0;
  if (a >= 0 && a < n_valid && g.kv0 + a <= g.s && keep_of(g, row, n_valid - a)) return a;
  if (row < g.ch || row >= g.ch + g.csz || n_valid <= 0) return -1;
  int64_t back = ring_mod(g.upd0 + n_valid - 1 - g.ch, g.csz) - (row - g.ch);   // rows behind the last token's
  if (back < 0) back += g.csz;
  const int64_t at = n_valid - 1 - back;
  return (at >= 0 && g.kv0 + at > g.s) ? at : -1;
}

// launches of moa_cache.hip that the fused prompt kernel needs around it (arguments are checked by the callers)
int launch_mask_scan(const int64_t* attention_mask, int64_t am_stride, int B, int S, int32_t* tok_of, int32_t* n_valid,
                     int32_t* rank_of, hipStream_t st);
int launch_prefill_index(int64_t* update_index, int64_t* valid_len, const int64_t* circ_head, const int64_t* circ_size,
                         const int64_t* static_size, const int32_t* n_valid, int64_t kv_len, int B, int H, int S,
                         hipStream_t st);

}  // namespace moa
