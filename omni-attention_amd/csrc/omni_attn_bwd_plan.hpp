// What a workgroup of the dK/dV kernel keeps of its slab's metadata in LDS, beside its tiles: a bitmap of
// the list slots that name its KV block and a table of the steps to walk.  (Host arithmetic, no device code.)
#pragma once

#include <stddef.h>

namespace omni_attn {

constexpr size_t kLdsOfComputeUnit = size_t(160) * 1024;
constexpr size_t kLdsGranule = 1280;  // LDS is handed out in units of this size

// LDS of one of `n` workgroups that share a compute unit.
constexpr size_t lds_share(int n) { return kLdsOfComputeUnit / size_t(n) / kLdsGranule * kLdsGranule; }

struct DkdvPlan {
  int words;      // 64-slot words of metadata held at a time (a window)
  int steps;      // entries of the table of steps (a piece of the window's walk)
  size_t bytes;   // LDS of the workgroup
};

// Per word 12 bytes: the bitmap of its matches (8) and mode / tile index of the first (4); an odd number of
// words is rounded up, so that the table behind them lies on 8 bytes.
constexpr size_t dkdv_word_bytes(long long words) { return size_t((words + 1) / 2) * 24; }
constexpr size_t kDkdvTail = 16;       // number of steps, and where the next piece begins
constexpr int kDkdvMinTable = 128;     // a piece costs a start and end of the pipeline: two steps
constexpr int kDkdvMaxWords = 4096;

// fixed: bytes of the tiles and what goes with them; waves_fit: workgroups that a compute unit holds by
// registers; n_words: words of the slab's metadata; steps_per_block: steps of a query block.
//
// The words decide how many workgroups share a compute unit, and the table takes what that leaves, up to
// a full window's steps.  Sized for every word and 64 more it cost half the occupancy at long lists: one
// workgroup per compute unit instead of two, B H=8 S=16384 D=128, blocks 128 x 64, causal, both backward
// kernels 2480 us; without a table 2151, as it is 1995.  A walk with more steps than entries is worked
// off in pieces, a slab with more words than fit in windows of about equal size.
constexpr DkdvPlan dkdv_plan(size_t fixed, int waves_fit, long long n_words, int steps_per_block) {
  const long long held = n_words < kDkdvMaxWords ? n_words : kDkdvMaxWords;
  const size_t least = kDkdvTail + size_t(kDkdvMinTable) * 8;
  int n = waves_fit;
  while (n > 1 && (fixed + size_t(held) * 12 > lds_share(n) || fixed + dkdv_word_bytes(500) + least > lds_share(n))) --n;
  const size_t room = lds_share(n) - fixed;  // for words, table and tail
  long long words = held;
  if (held < n_words || dkdv_word_bytes(held) + least > room) {
    long long most = (long long)((room - least) / 24) * 2;
    if (most > kDkdvMaxWords) most = kDkdvMaxWords;
    const long long windows = (n_words + most - 1) / most;
    words = (n_words + windows - 1) / windows;
    if (words % 2 != 0) ++words;
  }
  const size_t left = (room - dkdv_word_bytes(words) - kDkdvTail) / 8;
  const size_t full = size_t(words) * size_t(steps_per_block);  // (a list names a block once, as a rule)
  const size_t want = full > kDkdvMinTable ? full : kDkdvMinTable;
  const size_t steps = want < left ? want : left;
  return {int(words), int(steps), fixed + dkdv_word_bytes(words) + steps * 8 + kDkdvTail};
}

}  // namespace omni_attn
