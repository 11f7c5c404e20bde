"""The step between two rounds of a selection (csrc/select_plan.h), run on the host: the rounds
themselves are plain loops here."""
from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parent.parent / "cupynumeric_amd" / "csrc"

ROUNDS = r"""
#include <vector>
#include "select_plan.h"
using namespace cpn;

// Rounds of a selection of `ranks` among n images of `bits` bits: the first round reads `before`, the
// later ones `after` or the copy.  Returns the rounds that ran, -1 where the plan leaves the lists.
extern "C" int run_rounds(const uint64_t* before, const uint64_t* after, uint32_t n, uint32_t bits, const uint32_t* ranks,
                          uint32_t n_ranks, uint32_t copy_cap, uint64_t* images, uint32_t* left_over, uint64_t* keys_read)
{
  SelectPlan plan{};
  std::vector<uint64_t> copy(copy_cap);
  plan.n_prefix  = 1;
  plan.bits_left = bits;
  plan.list_len  = n;
  for (uint32_t t = 0; t < n_ranks; ++t) {
    plan.rank[t] = ranks[t];
  }
  *keys_read       = 0;
  const int rounds = select_rounds(static_cast<int>(bits), n_ranks);
  int r            = 0;
  for (; r < rounds && plan.done == 0; ++r) {
    const bool first       = r == 0;
    const uint32_t np      = first ? 1u : plan.n_prefix;
    const uint32_t want    = first ? SELECT_FIRST_BITS : select_bits(np);
    const uint32_t w       = want < plan.bits_left ? want : plan.bits_left;
    const uint32_t shift   = plan.bits_left - w;
    const uint64_t* list   = plan.from_copy ? copy.data() : (first ? before : after);
    const uint32_t list_len = plan.list_len;
    if (np > SELECT_MAX_RANKS || (np << w) > static_cast<uint32_t>(SELECT_BINS) || list_len > (plan.from_copy ? copy_cap : n)) {
      return -1;
    }
    std::vector<uint32_t> hist(np << w);
    uint64_t any[SELECT_MAX_RANKS], all[SELECT_MAX_RANKS];
    for (int t = 0; t < SELECT_MAX_RANKS; ++t) {
      any[t] = 0;
      all[t] = ~0ull;
    }
    uint32_t copied = 0;
    for (uint32_t i = 0; i < list_len; ++i) {
      const uint64_t k = list[i];
      for (uint32_t t = 0; t < np; ++t) {
        if (first || (k >> plan.bits_left) == plan.prefix[t]) {
          ++hist[(t << w) + ((k >> shift) & ((1u << w) - 1))];
          any[t] |= k;
          all[t] &= k;
          if (plan.copy_now) {
            if (copied < copy_cap) {
              copy[copied] = k;
            }
            ++copied;
          }
        }
      }
    }
    *keys_read += list_len;
    uint64_t chosen[SELECT_MAX_RANKS];
    uint32_t count[SELECT_MAX_RANKS];
    for (uint32_t t = 0; t < n_ranks; ++t) {
      const uint32_t p = plan.which[t];
      uint64_t run = 0;
      chosen[t] = 0;
      count[t]  = 0;
      if (p == SELECT_FINISHED) {
        continue;
      }
      for (uint32_t b = 0; b < (1u << w); ++b) {
        const uint32_t c = hist[(p << w) + b];
        if (plan.rank[t] >= run && plan.rank[t] < run + c) {
          chosen[t] = (plan.prefix[p] << w) | b;
          count[t]  = c;
          plan.rank[t] -= static_cast<uint32_t>(run);
          break;
        }
        run += c;
      }
    }
    SelectChild child[SELECT_MAX_RANKS];
    uint64_t varying = 0;
    for (uint32_t t = 0; t < n_ranks; ++t) {
      if (plan.which[t] != SELECT_FINISHED) {
        child[t] = select_child(chosen[t], shift, any[plan.which[t]], all[plan.which[t]]);
        varying |= child[t].varying;
      }
    }
    const uint32_t left = select_bits_left(varying);
    uint32_t prefixes = 0;
    uint64_t total    = 0;
    for (uint32_t t = 0; t < n_ranks; ++t) {
      if (plan.which[t] == SELECT_FINISHED) {
        continue;
      }
      if (child[t].varying == 0) {
        plan.image[t] = child[t].image;
        plan.which[t] = SELECT_FINISHED;
        continue;
      }
      if (prefixes == 0 || plan.prefix[prefixes - 1] != child[t].image >> left) {
        plan.prefix[prefixes++] = child[t].image >> left;
        total += count[t];
      }
      plan.which[t] = prefixes - 1;
    }
    select_next_list(&plan, plan.copy_now != 0, plan.from_copy != 0, prefixes, left, total, copied, copy_cap);
  }
  for (uint32_t t = 0; t < n_ranks; ++t) {
    images[t]    = plan.image[t];
    left_over[t] = plan.rank[t];
  }
  return plan.done ? r : 0;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    folder = tmp_path_factory.mktemp("select_plan")
    (folder / "rounds.cpp").write_text(ROUNDS)
    subprocess.run(
        ["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-D__host__=", "-D__device__=", f"-I{CSRC}",
         str(folder / "rounds.cpp"), "-o", str(folder / "rounds.so")],
        check=True,
    )
    return ctypes.CDLL(str(folder / "rounds.so"))


def _run(lib, before, ranks, bits, after=None):
    after = before if after is None else after
    ranks = np.unique(ranks).astype(np.uint32)
    images, left_over = np.zeros(32, np.uint64), np.zeros(32, np.uint32)
    read = ctypes.c_uint64()
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    rounds = lib.run_rounds(p(before), p(after), before.size, bits, p(ranks), ranks.size, before.size // 4, p(images), p(left_over), ctypes.byref(read))
    return ranks, rounds, images[: ranks.size], left_over[: ranks.size], read.value


def _images(x):
    """The ordered images of key_codec.h: unsigned keys in the sort's order, NaNs all ones, zeros of either sign equal."""
    if x.dtype.kind == "u":
        return x.astype(np.uint64)
    u = np.uint32 if x.dtype.itemsize == 4 else np.uint64
    sign = u(1) << u(8 * x.dtype.itemsize - 1)
    if x.dtype.kind == "i":
        return (x.view(u) ^ sign).astype(np.uint64)
    b = np.where(x == 0, np.zeros_like(x), x).view(u)
    out = np.where(b & sign, ~b, b | sign)
    out[np.isnan(x)] = ~u(0)
    return out.astype(np.uint64)


def _data(kind, dtype, n, rng):
    dt = np.dtype(dtype)
    if kind == "equal":
        return np.full(n, 7, dtype=dt)
    if kind == "whole":
        return rng.integers(1, 6, n).astype(dt)
    if kind == "binary":
        return rng.integers(0, 2, n).astype(dt)
    if kind == "signed":
        return rng.integers(-5, 6, n).astype(np.int64).astype(dt)
    if kind == "twenty":
        return (rng.standard_normal(20) * 1e6).astype(np.int64 if dt.kind in "iu" else dt).astype(dt)[rng.integers(0, 20, n)]
    if kind == "ids":
        return rng.integers(0, 1_000_000_000, n).astype(dt)
    if dt.kind != "f":
        info = np.iinfo(dt)
        return rng.integers(info.min, info.max, n, dtype=dt, endpoint=True)
    x = rng.standard_normal(n).astype(dt)
    if kind == "specials":
        u = rng.random(n)
        x[u < 0.3] = np.nan
        x[(u >= 0.3) & (u < 0.5)] = -0.0
        x[(u >= 0.5) & (u < 0.6)] = np.inf
        x[(u >= 0.6) & (u < 0.7)] = -np.inf
    return x


@pytest.mark.parametrize("dtype", [np.int32, np.uint32, np.float32, np.int64, np.uint64, np.float64])
@pytest.mark.parametrize("kind", ["random", "equal", "whole", "binary", "signed", "twenty", "ids", "specials"])
@pytest.mark.parametrize("n", [1, 2, 7, 1000, 20_000])
def test_rounds_find_the_ranks(lib, dtype, kind, n):
    rng = np.random.default_rng(n)
    k = _images(_data(kind, dtype, n, rng))
    order = np.sort(k)
    bits = 8 * np.dtype(dtype).itemsize
    for wanted in ([n // 2], [0, n - 1], np.minimum(np.linspace(0, n, 16).astype(int), n - 1).tolist(), rng.integers(0, n, 32)):
        ranks, rounds, images, left_over, _ = _run(lib, k, wanted, bits)
        assert rounds > 0
        assert np.array_equal(images, order[ranks])
        # what is left of a rank counts the equal images before it
        assert np.array_equal(left_over, ranks - np.searchsorted(order, images))


@pytest.mark.parametrize("bits", [32, 64])
def test_no_round_leaves_the_lists_when_the_input_changes_under_way(lib, bits):
    """The first round counts keys of which few can be asked for, later rounds meet keys that all are: the
    copy has no room for them, and the next round must not read past it."""
    rng = np.random.default_rng(bits)
    n = 10_000
    before = rng.integers(0, 1 << (bits - 1), n).astype(np.uint64) << np.uint64(1)
    wanted = [n // 3, n // 2]
    middle = np.sort(before)[wanted[0]]
    for after in (np.full(n, middle), before ^ np.uint64(1 << (bits - 2)), np.zeros(n, np.uint64)):
        _, rounds, _, _, _ = _run(lib, before, wanted, bits, after=after)
        assert rounds >= 0


@pytest.mark.parametrize("dtype", [np.int64, np.float64])
@pytest.mark.parametrize("kind, reads", [("equal", 1), ("binary", 2), ("whole", 2), ("signed", 3), ("twenty", 4), ("ids", 4), ("random", 4)])
def test_few_values_take_few_passes(lib, dtype, kind, reads):
    """Vectors whose wanted values cover most of the input are never copied: every round reads all of it, so
    rounds must not be spent on bits in which the keys of a prefix agree."""
    rng = np.random.default_rng(7)
    n = 50_000
    k = _images(_data(kind, dtype, n, rng))
    for wanted in ([n // 2], np.linspace(0, n - 1, 32).astype(int)):
        _, rounds, _, _, read = _run(lib, k, wanted, 64)
        assert rounds > 0 and read <= reads * n, (rounds, read / n)
