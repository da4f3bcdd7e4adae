// Finding a workgroup's piece of a packed batch from cu_seqlens on the device.
#pragma once
#include "common.h"

namespace ssla {

// Lane `from`'s value as a wavefront-uniform one (scalar registers).
__device__ __forceinline__ int64_t readlane64(int64_t x, int from) {
  const uint32_t l = __builtin_amdgcn_readlane(static_cast<int>(x), from);
  const uint32_t h = __builtin_amdgcn_readlane(static_cast<int>(x >> 32), from);
  return static_cast<int64_t>((static_cast<uint64_t>(h) << 32) | l);
}

// Sequences are cut into pieces of `unit` rows; piece j of sequence n has slot
// first(n) + j with first(n) = bos_n / unit + n, distinct for every piece of
// non-overlapping sequences (at most T / unit + n_seq + 1 slots; an empty
// sequence owns its first slot).  Finds the sequence whose slots hold `slot`
// (false: none before it); the caller checks that the piece exists.  Every
// wavefront searches the sequence starts 64 probes per round trip: one round
// for up to 64 sequences, two for 4,096.  OWN false leaves n out of first(n):
// slots that only pieces with a successor in their sequence own (at most
// (T - 1) / unit of them).
template <bool OWN = true>
__device__ __forceinline__ bool seq_of_slot(const int64_t *cu, int n_seq, int64_t T, int64_t unit, int64_t slot, int &n,
                                            int64_t &bos, int64_t &eos, int64_t &first) {
  // (32-bit division where it holds: the 64-bit one is dozens of instructions)
  auto slot_of = [&](int64_t row, int i) __attribute__((always_inline)) {
    return (T < 0x7fffffff ? static_cast<int64_t>(static_cast<uint32_t>(row) / static_cast<uint32_t>(unit))
                           : row / unit) + (OWN ? i : 0);
  };
  const int lane = threadIdx.x & 63;
  int lo = 0, hi = n_seq;
  do {
    const int step = (hi - lo + 63) >> 6;
    const int64_t i = lo + static_cast<int64_t>(lane) * step;
    const int ic = static_cast<int>(min(i, static_cast<int64_t>(hi - 1)));
    const int64_t b = min(max(cu[ic], (int64_t)0), T), e = min(max(cu[ic + 1], b), T);
    const int64_t f = slot_of(b, ic);
    const int cnt = __popcll(__ballot(i < hi && f <= slot));
    if (cnt == 0) return false;
    const int from = cnt - 1;
    lo += from * step;
    hi = min(hi, lo + step);
    bos = readlane64(b, from);
    eos = readlane64(e, from);
    first = readlane64(f, from);
  } while (hi - lo > 1);
  n = lo;
  return first <= slot;   // (always, unless the starts decrease: then no row before the sequence's is touched)
}

}  // namespace ssla
