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

// Device-side state, written by select_init_kernel and by the last workgroup of every round.
struct SelectPlan {
  uint64_t key_or, key_and;            // over all images (first round)
  uint64_t prefix[SELECT_MAX_RANKS];   // different prefixes: the resolved top bits of an image
  uint64_t image[SELECT_MAX_RANKS];    // per target, once done
  uint32_t rank[SELECT_MAX_RANKS];     // per target: position among the keys with its prefix
  uint32_t which[SELECT_MAX_RANKS];    // per target: its prefix
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

// The plan after a round.  chosen[t], count[t]: the prefix of target t down to bit `shift` and the
// keys that have it, 0 where the round counted no key at the target's rank: a caller that writes to
// the input during the call gets there.  Its result is undefined, but no later round may read
// outside the lists: list_len never exceeds copy_cap once the copy is read.
// `common`, `varying`: the bits on which all images of the input agree and differ (first round).
__host__ __device__ inline void select_advance(SelectPlan* plan, uint64_t* chosen, const uint32_t* count, uint32_t n_ranks, uint32_t shift,
                                               bool first, uint64_t common, uint64_t varying, uint32_t copied, uint32_t copy_cap)
{
  uint32_t left  = shift;
  uint64_t total = 0;
  if (first) {
    const uint32_t top = varying == 0 ? 0u : 64u - static_cast<uint32_t>(__builtin_clzll(varying));
    if (top < left) {  // every key agrees on the bits above: one bin, whose prefix takes them in
      left = top;
      for (uint32_t t = 0; t < n_ranks; ++t) {
        chosen[t] = common >> left;
      }
    }
  }
  uint32_t n = 0;
  for (uint32_t t = 0; t < n_ranks; ++t) {  // ascending targets: equal prefixes are neighbours
    if (t == 0 || chosen[t] != chosen[t - 1]) {
      plan->prefix[n++] = chosen[t];
      total += count[t];
    }
    plan->which[t] = n - 1;
  }
  plan->n_prefix  = n;
  plan->bits_left = left;
  if (plan->copy_now != 0) {
    plan->copy_now  = 0;
    plan->from_copy = 1;
    plan->list_len  = copied < copy_cap ? copied : copy_cap;
  } else if (plan->from_copy == 0 && total <= copy_cap) {
    plan->copy_now = 1;
  }
  if (left == 0) {
    plan->done = 1;
    for (uint32_t t = 0; t < n_ranks; ++t) {
      plan->image[t] = chosen[t];
    }
  }
}

}  // namespace cpn
