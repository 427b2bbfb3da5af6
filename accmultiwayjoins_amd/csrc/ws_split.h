// Arithmetic of work sharing and of unit claims, shared by the persistent AMHJ and ALFTJ engines
// and by the CPU test of the protocol (plain constexpr C++: host and device code compile the same
// lines).
//
// A wave walking the flattened children [c, c1) of a frontier level with more than split + 64
// left keeps [c, c + split) and shares the rest as k pieces of `split` children (the last one
// shorter). When the queue grants only got <= k slots, the wave publishes the LAST got pieces and
// keeps everything before them, so the kept range and the published pieces tile [c, c1) exactly.
// Reference: the split of long ranges into BUC_THRESHOLD pieces pushed to a TaskBook
// (LFTJ-GPU/ALFTJ.cuh:464-499; MHJ-GPU/Joins/AMHJ_WS.cuh:168-187).
#pragma once

#include <stdint.h>

namespace amj {

// Does a wave at child c of [c, c1) share work?
constexpr bool ws_should_split(uint64_t c, uint64_t c1, uint64_t split) {
  return split != 0 && c1 - c > split + 64;
}

// Pieces the rest [c + split, c1) is cut into (call only when ws_should_split holds).
constexpr uint64_t ws_pieces(uint64_t c, uint64_t c1, uint64_t split) {
  return (c1 - (c + split) + split - 1) / split;
}

// Piece j (0 <= j < got) of the got published ones: [*p0, *p1).
constexpr void ws_piece(uint64_t c, uint64_t c1, uint64_t split, uint64_t k, uint64_t got,
                        uint64_t j, uint64_t* p0, uint64_t* p1) {
  *p0 = c + split + (k - got + j) * split;
  *p1 = *p0 + split < c1 ? *p0 + split : c1;
}

// End of the range the wave keeps after publishing got of the k pieces (all of it when none).
constexpr uint64_t ws_keep_end(uint64_t c, uint64_t c1, uint64_t split, uint64_t k,
                               uint64_t got) {
  return got ? c + split + (k - got) * split : c1;
}

// Units are claimed from kUnitShards counters: unit u belongs to shard u % kUnitShards, and a
// shard's counter numbers its units 0, 1, .. (unit_of_shard gives them back).
constexpr uint32_t kUnitShards = 8;
constexpr uint64_t kMaxClaim = 64;  // units claimed at once by a wave
constexpr uint64_t kMinClaim = 4;   // ... and at least, in launches of many units per wave
constexpr uint64_t kManyUnits = 16; // units per wave from which a launch has many

constexpr uint64_t ws_shard_units(uint64_t units, uint32_t shard) {
  return (units + kUnitShards - 1 - shard) / kUnitShards;
}
constexpr uint64_t ws_unit_of_shard(uint64_t k, uint32_t shard) { return k * kUnitShards + shard; }

// Units a wave asks a shard for when `at` of its `size` ones are claimed (at < size), of a launch of
// `units` units and `waves` waves (max_claim 0: kMaxClaim). Guided chunks: with many units per
// wave, half of what each wave has left and at least kMinClaim, so that cheap units do not pay
// for a claim each. With fewer (the triejoin's units of many roots, heaviest first), a quarter and
// at least one: 4 units at a time took the 4-cliques of R-MAT 20 from 290 to 860 ms.
constexpr uint64_t ws_claim(uint64_t units, uint64_t size, uint64_t at, uint64_t waves,
                            uint64_t max_claim) {
  const uint64_t most = max_claim ? max_claim : kMaxClaim;
  const bool many = units >= kManyUnits * waves;
  const uint64_t least = many && most >= kMinClaim ? kMinClaim : 1;
  const uint64_t k = (size - at) * kUnitShards / ((many ? 2 : 4) * waves);
  return k < least ? least : (k > most ? most : k);
}

// Steps of 64 children (or values of a streamed list) between two progress reports of a working
// wave: idle waves then see progress while others walk long levels, whatever their units and tasks
// take. A wave's steps count over all its units, and between two of them lie a few loads: reports
// are 1 to 20 ms apart.
constexpr uint32_t kBeatSteps = 4096;

// Does a wave that has taken `before` steps report after n more?
constexpr bool ws_beat(uint32_t before, uint32_t n) {
  return (before + n) / kBeatSteps != before / kBeatSteps;
}

// What a waiting wave watches: it changes whenever a wave reports progress, starts to work or runs
// out of work.
constexpr uint64_t ws_moved(uint64_t progress, uint32_t busy) {
  return progress + ((uint64_t)busy << 40);
}

// Slots granted by one fetch-add on a counter: tail was the old value, cap the capacity (the task
// queue's, or the units of a shard).
constexpr uint64_t ws_granted(uint64_t tail, uint64_t want, uint64_t cap) {
  return tail >= cap ? 0 : (want < cap - tail ? want : cap - tail);
}

}  // namespace amj
