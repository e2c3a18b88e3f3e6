// How the workgroups that share a result find out which of them arrives last, without one waiting for another: a count
// in a word of scratch memory whose content before the call does not matter.  Host and device code:
// tests/test_arrival.py compiles arrival_check.cpp, which runs it in every order.
//
// A word is a tag (upper 56 bits) and the arrivals so far (lower 8).  Every member, in this order:
//   seen = the word, at any time after the call has started;
//   arrival::begin(word, seen, tag)  makes a word with another tag (tag, 0): whoever comes first does, for the others the
//                                    word is no longer what they saw, or they saw the tag;
//   publishes its share, and waits until that and `begin` have been performed in memory;
//   arrival::arrive(word, tag, members)  counts it, and returns true for the last, which reads all shares.
// The last one leaves 0, so that a call with the same tag (a replayed graph) starts afresh.  Members of two calls that
// use a word at the same time take each other's counts: there may then be no last one in either, and the word may keep
// an unfinished count; a later call, whose tag is another, does not mind.
#pragma once

#include <cstdint>

#include "common.h"

namespace cllm {
namespace arrival {

constexpr uint64_t kCount = 0xff;

// The tag of a process's n-th call: the finaliser of Steele, Lea and Flood's SplitMix64 spreads n, so that no fill
// pattern and no other call's word is likely to carry it.
__host__ __device__ inline uint64_t tag_of(uint64_t salt, uint64_t n) {
    uint64_t z = salt + n * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return (z ^ (z >> 31)) & ~kCount;
}

template <typename Word>
__host__ __device__ inline void begin(Word word, uint64_t seen, uint64_t tag) {
    if ((seen ^ tag) & ~kCount) word.compare_exchange(seen, tag);
}

template <typename Word>
__host__ __device__ inline bool arrive(Word word, uint64_t tag, unsigned members) {
    const uint64_t old = word.add_one();
    if (((old ^ tag) & ~kCount) || (old & kCount) + 1 != members) return false;
    word.store(0);
    return true;
}

}  // namespace arrival
}  // namespace cllm
