// Entries per thread of the multiexp's bucket loops.
#pragma once
#include <stdint.h>

namespace csk {

// Sorted entries per accumulation thread, from the entries there are (digits that
// are not 0; a witness has half as many as its size allows) and the buckets K: fixed
// when the caller says so, otherwise what fills whole rounds of 2^17 threads, the two
// waves per SIMD that the bucket loops run.  One round up to 2^23 entries, two up to
// 2^26 (64 to 256 entries a thread), then as many as hold 256 entries a thread.  A
// length rounded down leaves a last round nearly empty: 2.2M G1 points, 262687 threads
// of 134 entries 4.00 ms, 3.44 by 135; 2^18 G2 points, 233017 threads of 18 entries
// 2.00 ms, 1.88 by 32.  From 64 to 256 entries a round more or less makes 1%.
//
// With K below 2^17, where the fix-up adds up to eight carries a bucket itself, a
// bucket is to span no more chunks than that (10000 G2 points, c = 11, 39 entries a
// bucket: 0.76 ms by 4, 0.60 by 8): in fewer rounds, though never less than one (2^19
// G2 points, c = 13: 4.00 ms in two rounds of 40, 3.00 in one of 80), and below a full
// round by chunks of up to 48 entries that leave 2^14 threads (tables of 300000 G1
// points, c = 15, by 48 entries 727 us, 759 by 39 and the carry rounds; of 16384 G2
// points, c = 13, by 13 and 25000 threads 543, 650 by 10).  Beyond, the chunk is what
// is waited for and the rounds, which take any chain, cost less: tables of 4095 G1
// points, c = 8, 1018 us by 158 entries (830 threads), 291 by 8; of 16383 G2 points,
// c = 11, 1212 by 60 (6550), 730 by 8; of 2^18 G2 points, c = 14, 3.10 ms by 94, 2.16
// by 39; of 2^20 G1 points, c = 8, 211 ms by 40330 (830), 3.0 by 256.
//
// Chunks below 8 entries make more carries than their threads are worth, below 4 where
// a chunk's entry takes longest (5003 G2 points in quarters: 568 us by 3, 539 by 4, 565
// by 8).
struct ChunkLen {
  uint32_t fixed, least;
  static constexpr uint32_t rounds(uint32_t entries) {
    return entries <= 1u << 23 ? 1 : entries <= 1u << 26 ? 2 : (entries + (1u << 25) - 1) >> 25;
  }
  constexpr uint32_t operator()(uint32_t entries, uint32_t K) const {
    if (fixed) return fixed;
    // entries of a chunk by which a bucket spans 6.5 of them
    const uint32_t span = K < 1u << 17 && entries / 13 * 2 > K ? (entries / 13 * 2 + K - 1) / K : 1;
    uint32_t r = rounds(entries);
    if (r > entries / span >> 17) r = entries / span >> 17;
    if (r == 0) r = 1;
    uint32_t l = (entries + (r << 17) - 1) / (r << 17);
    if (l < span && span <= 48 && span <= entries >> 14) l = span;
    if (l < least) l = least;
    return l;
  }
  // chunks of at most `entries` entries, however many there are
  constexpr uint64_t most(uint32_t entries) const {
    const uint64_t l = fixed ? fixed : least, n = (entries + l - 1) / l;
    const uint64_t r = fixed ? n : (uint64_t)rounds(entries) << 17;
    return n < r ? n : r;
  }
};

}  // namespace csk
