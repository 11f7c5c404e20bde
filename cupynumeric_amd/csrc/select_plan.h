// What one round of a selection (select.hip) hands to the next, and the step between two rounds.
// Plain C++ without device intrinsics: the last workgroup of a round runs select_advance, and so
// does a test on the host.
#pragma once

#include <stdint.h>

namespace cpn {

constexpr int SELECT_MAX_Q      = 16;
constexpr int SELECT_MAX_RANKS  = 2 * SELECT_MAX_Q;
constexpr int SELECT_BINS       = 16384;  // counters in LDS, shared by the prefixes of a round
constexpr int SELECT_FIRST_BITS = 12;
constexpr int SELECT_MAX_BITS   = 11;  // later rounds
constexpr int SELECT_MAX_ROUNDS = 8;

// Bits that a round after the first resolves for `prefixes` different prefixes.
__host__ __device__ constexpr uint32_t select_bits(uint32_t prefixes)
{
  uint32_t w = SELECT_MAX_BITS;
  while ((prefixes << w) > static_cast<uint32_t>(SELECT_BINS)) {
    --w;
  }
  return w;
}
// Rounds that resolve `bits` bits of `ranks` targets.
__host__ __device__ constexpr int select_rounds(int bits, uint32_t ranks)
{
  const int w = static_cast<int>(select_bits(ranks));
  return bits <= SELECT_FIRST_BITS ? 1 : 1 + (bits - SELECT_FIRST_BITS + w - 1) / w;
}
static_assert(select_rounds(64, SELECT_MAX_RANKS) <= SELECT_MAX_ROUNDS, "counters for every round");

constexpr uint32_t SELECT_FINISHED = ~0u;

// Device-side state, written by select_init_kernel and by the last workgroup of every round.
struct SelectPlan {
  uint64_t any[SELECT_MAX_RANKS];      // per prefix: OR of the images that have it (the round under way)
  uint64_t all[SELECT_MAX_RANKS];      // per prefix: AND of them
  uint64_t prefix[SELECT_MAX_RANKS];   // different prefixes: the resolved top bits of an image
  uint64_t image[SELECT_MAX_RANKS];    // per target, once finished
  uint32_t rank[SELECT_MAX_RANKS];     // per target: position among the keys with its prefix
  uint32_t which[SELECT_MAX_RANKS];    // per target: its prefix, or SELECT_FINISHED
  uint32_t chunk[SELECT_MAX_RANKS];    // per target: where a key that ties with other bits is found
  uint32_t n_prefix;
  uint32_t bits_left;
  uint32_t list_len;                   // keys of the list that the next round reads
  uint32_t from_copy;                  // that list is the copy, not the input
  uint32_t copy_now;                   // the next round makes the copy
  uint32_t copied;                     // keys that went to the copy, or had no room there
  uint32_t done;
  uint32_t ties;                       // float targets among the NaNs or the zeros: bit 0, bit 1
  uint32_t blocks_done[SELECT_MAX_ROUNDS + 1];
};
constexpr uint64_t SELECT_PLAN_BYTES = 2048;
static_assert(sizeof(SelectPlan) <= SELECT_PLAN_BYTES, "plan slot");

// A target after a round that resolved the bits from `shift` on: `chosen` is its prefix down to that bit,
// `any` and `all` are OR and AND of the images counted under its old prefix.  Lower bits on which all of these
// agree are known without another round: a target none of whose lower bits vary is finished, and the next
// round starts at the highest bit that varies for any target.  So a handful of values is told apart in two
// or three rounds wherever their bits are (whole numbers held as floats, small integers of either sign).  With a
// round per eleven bits, each over the whole input since no copy is small enough, five percentiles of 2^28
// zeros and ones in float64 took 4.6 ms, where the sort takes 2.5; now 1.1.
struct SelectChild {
  uint64_t image;    // right in the bits on which the keys agree
  uint64_t varying;  // bits on which they do not; 0: the image is whole
};
__host__ __device__ inline SelectChild select_child(uint64_t chosen, uint32_t shift, uint64_t any, uint64_t all)
{
  const uint64_t low = (1ull << shift) - 1;  // (the first round resolves at least one bit: shift < 64)
  return SelectChild{(chosen << shift) | (all & low), (any ^ all) & low};
}
// Bits that are left to the next round; `varying`: of all its targets.
__host__ __device__ inline uint32_t select_bits_left(uint64_t varying)
{
  return varying == 0 ? 0u : 64u - static_cast<uint32_t>(__builtin_clzll(varying));
}

// The list of the next round, which asks for `prefixes` prefixes with `total` keys in all and `left` unknown
// bits: the input, the copy, or the input while the copy is made (unless no round comes after it).  copy_now,
// from_copy: as the plan had them for this round; `copied`: keys that this round has staged for the copy.  A
// caller that writes to the input during the call may bring more of them than were counted; the result is
// undefined then, but no later round reads past the room that the copy has.
__host__ __device__ inline void select_next_list(SelectPlan* plan, bool copy_now, bool from_copy, uint32_t prefixes, uint32_t left,
                                                 uint64_t total, uint32_t copied, uint32_t copy_cap)
{
  plan->n_prefix  = prefixes;
  plan->bits_left = left;
  plan->done      = prefixes == 0 ? 1u : 0u;
  if (copy_now) {
    plan->copy_now  = 0;
    plan->from_copy = 1;
    plan->list_len  = copied < copy_cap ? copied : copy_cap;
  } else if (!from_copy && total <= copy_cap && left > select_bits(prefixes)) {
    plan->copy_now = 1;
  }
}

}  // namespace cpn
