// What the waves of dealt::ring_walk_kernel tell each other about the key tiles of a round.  Plain arithmetic, on the host and in the kernel.
//
// A round has four tiles and a word for each.  Behind the barrier of the round every wave reads all four and finds in them which tile is the first
// to move the references; that says how many barriers follow, so all waves have to find the same.  The tile that moves says so in its
// word while others may still be on their way to reading it -- there is no barrier in between --, and so the word keeps the wish that it
// announced before: who reads early and who reads late find the same first tile.  Words of tiles behind that one are written
// again behind the next barrier only, those in front of it in the round after the next.
#pragma once
#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define RINGATTN_BOTH __host__ __device__ __forceinline__
#else
#define RINGATTN_BOTH inline
#endif

namespace ringattn {

constexpr int kNewsTiles = 4;             // of a round
constexpr int kNewsWish = 1;              // the tile wants to move the references
constexpr int kNewsMovedBit = 8;
constexpr int kNewsMoved = 1 << kNewsMovedBit | kNewsWish;  // it has done so

// Four words in one: tile i's wish at bit i; of the words shifted right by kNewsMovedBit, tile i's move.
RINGATTN_BOTH int news_of_round(int x0, int x1, int x2, int x3) { return x0 | x1 << 1 | x2 << 2 | x3 << 3; }
// which tile, from tile `from` on, is the first that wants to move the references: kNewsTiles for none
RINGATTN_BOTH int first_wish(int round, int from) {
  return from + __builtin_ctz(((round & ((1 << kNewsTiles) - 1)) | 1 << kNewsTiles) >> from);
}

}  // namespace ringattn
