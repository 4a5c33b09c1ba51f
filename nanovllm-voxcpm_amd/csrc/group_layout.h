// How the low-level ops over tiles of a slot (group.hip) are laid over a grid: who takes which tokens of a slot, and how many
// places that needs.  The kernels and the host read the same rules here.
#pragma once

#include "common.h"

namespace mlora {

// What the grid is laid over.  By slot: places are (tile of a slot, slot), then the tiles that no slot is expected to have (a
// popular adapter's), which find out from a histogram whose they are.  By token: a place is a token; the first token of every
// tile stands for it, the others leave.
constexpr int kBySlot = 0, kByToken = 1;

struct GroupPlaces {
  int T, num_slots;
  int width;   // tokens of a tile: 4, 8 or 16 (by slot: of a slot whose own tiles hold all its tokens at that width, else 16)
  int slots8;  // by slot: slot ids (and, in the shrink, one for the tokens without a slot) rounded up to eight
  int tiles;   // by slot: tiles of a slot that have a place of their own
};

// By slot: tokens of each tile of a slot that has `count` of them.  Sixteen for a slot that its own tiles do not hold at the narrow
// width: that is fewer workgroups that look for a further tile as well (255 tokens at random over 64 slots, rank 32, 1024 -> 1024, against
// narrow own tiles and wide further ones, us: shrink 5.0 / 4.3, expand 4.4 / 3.8; 256 over 32, rank 16: 4.2 / 4.2 and 3.4 / 3.4).
__host__ __device__ inline int tile_width(const GroupPlaces& p, int count) { return count > p.tiles * p.width ? MLORA_TILE_SMALL : p.width; }

// By slot: the tiles such a slot has beyond those with a place of their own.
__host__ __device__ inline int tiles_beyond(const GroupPlaces& p, int count) {
  const int n = (count + MLORA_TILE_SMALL - 1) / MLORA_TILE_SMALL - p.tiles;
  return n > 0 ? n : 0;
}

inline int groups_about(int tokens, int slots) { return tokens < slots ? tokens : slots; }  // slots with tokens, at most

// Fills in how a launch of `parts` workgroups per tile is laid out for the p.T tokens and p.num_slots slot ids that p names; returns
// its places.  extra: places for the tokens without a slot.
inline int lay_out(GroupPlaces& p, int* over, long long parts, int extra) {
  const int groups = groups_about(p.T, p.num_slots);
  // tiles of four tokens while that many workgroups find room on the chip, else eight, else sixteen
  p.width = 4;
  while (p.width < MLORA_TILE_SMALL && parts * groups * (1 + p.T / (groups * p.width)) > 256) p.width *= 2;
  // over the tokens where slots without any would be most of the places
  *over = p.T <= p.num_slots ? kByToken : kBySlot;
  p.slots8 = p.tiles = 0;
  if (*over == kByToken) return p.T;
  p.slots8 = (p.num_slots + extra + 7) & ~7;
  p.tiles = 1 + p.T / (p.num_slots * p.width);
  // All tokens on one slot need the most further places: a second slot's own tiles take at least as much as rounding up to whole
  // tiles may cost, tiles_beyond(a) + tiles_beyond(b) <= tiles_beyond(a + b).  (Own tiles that stay narrow beside wide further ones
  // would break that: many slots just above their own places' tokens need a further place each.)
  return p.slots8 * p.tiles + tiles_beyond(p, p.T);
}

}  // namespace mlora
