// Entries per thread of the multiexp's bucket loops, and how a table run is sorted.
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

// Whether a table run's windows are sorted together, as one member of Wt * n_pad
// points (a table's slices follow each other, and window w of scalar i is an
// entry for point w * n_pad + i), so that all of a bucket's entries are
// adjacent.  As members of one window each, every window has its own copy of
// the buckets, carried, fixed up and merged: at 100003 points, c = 16, 524288
// buckets of 3 entries instead of 32768 of 49, 582 -> 410 us; 500 points
// 411 -> 219, 2^20 1661 -> 1475, 2.2M (2^25 entries) 3267 -> 3002 us; G2 5000 868 ->
// 455, 2^20 4828 -> 3999 us.  A member has at most 256 second-pass workgroups, so
// larger runs keep the members: 2^22 points 5886 us joint, 5829 as members.
// So do those whose top window (254 mod c bits) is no wider than what the second
// pass sorts by (c - 9 bits): all its n_pad entries are then in one bin, and one
// workgroup's walk through them, 1.3 ns each, is waited for, while a member's top
// window has bins of its own.  The members' copies of the buckets cost 0.2 ns each
// on G1 and 0.8 on G2; the line lies at about twice that and from 2^18 points, where
// they win with wire values too (G1 2^20 points, c = 12: joint 3.66, members 2.26 ms;
// c = 14 3.31 and 2.00; c = 18 2.92 and 2.00; G2 2^20, c = 14 6.88 and 5.72).
constexpr bool table_joint(uint64_t n_pad, uint32_t c, uint32_t Wt, bool g2) {
  if (n_pad * Wt > 1ull << 25) return false;
  const bool one_bin = c > 9 && 254 % c <= c - 9;
  const uint64_t copies = (uint64_t)Wt << (c - 1);
  return !(one_bin && n_pad > 1u << 18 && 5 * n_pad > (g2 ? 3 : 2) * copies);
}

}  // namespace csk
