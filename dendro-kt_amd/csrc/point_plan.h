// Host-side layout of the point tiles (p = 1): what point_kernel.h runs.
//
// A tile is a run of SFC-consecutive traversal leaves.  Its local points are,
// in this order,
//   nodes    mesh nodes, [0, nnode);
//   rows     hanging points, each the mean of two earlier points (its row
//            word), by level: a point of level k + 1 has a parent of level k;
//   odd      hanging points that are such means too but whose transposed
//            values go to some of the nodes behind them only;
//   readers  hanging points that the stale-buffer replay writes;
//   slots    one correction slot per leaf that needs one, and a zero slot
//            (the padding of the sums).
// Every rank of every leaf is one local point (leaf_loc), hanging or not, so
// the element gather and the element scatter have no missing ranks.
#pragma once
#include <cstddef>
#include <cstdint>
#include <vector>

#include "mesh.h"

namespace dkt {

constexpr int kPtLevels = 11;       // row levels of a tile
constexpr int kPtMaxPoints = 8191;  // 13-bit point indices

// A tile's maps are two blocks of 16-byte units, which the kernel copies to LDS
// whole: one round trip to memory each.
//   A (stage and rows): nodes (int32), their output slots (int32), row words
//     (rows, odd and reader points in order), then from an 8-byte boundary the
//     replay's readers, blocks, carry weights (FP64), carry keys, chain words and
//     parent maps.
//   B (sums): steps (the nodes', then those of levels nlev - 1 .. 1), quads, pairs.
struct PtTile {
  int32_t leaf0, nleaf;  // leaves
  int32_t a0, na, b0, nb;  // blocks: first unit, units
  int32_t nnode, nlev, nrow;  // mesh nodes, row levels, first point past the rows
  uint32_t lv[kPtLevels + 1];  // per level: first point past it (lv[0]: nnode), pairs of pair steps onto it << 16
  int32_t nodd, nrdp;    // odd and reader points
  int32_t ncor;          // correction slots, after the points; then the zero slot
  int32_t nstep, nquad;  // step words (an even number), quads
  int32_t nqs;           // groups of four steps onto the nodes
  int32_t nrd, rep, ncr, ngrp, nch;  // replay: readers, blocks and carry_log() << 16, carry terms, sibling groups, chain words
  constexpr int32_t nbk() const { return rep & 0xFFFF; }
  // log2 of the lanes that sum one slot of the buffer state at the tile start: those
  // of a workgroup of the plan's leaves per tile, whatever the launch has.
  constexpr int32_t carry_log() const { return rep >> 16; }
  constexpr int32_t past(int k) const { return (int32_t)(lv[k] & 0xFFFFu); }
  constexpr int32_t npts() const { return nrow + nodd + nrdp; }
  // Byte offsets in block A and B.
  constexpr int32_t rows_at() const { return 8 * nnode; }
  constexpr int32_t readers_at() const { return (8 * nnode + 4 * (npts() - nnode) + 7) & ~7; }
  constexpr int32_t blocks_at() const { return readers_at() + 8 * nrd; }
  constexpr int32_t carry_w_at() const { return blocks_at() + 8 * nbk(); }
  constexpr int32_t carry_key_at() const { return carry_w_at() + 8 * ncr; }
  constexpr int32_t chain_at() const { return carry_key_at() + 4 * ncr; }
  constexpr int32_t gploc_at() const { return chain_at() + 4 * nch; }
  constexpr int32_t quads_at() const { return 4 * nstep; }
  constexpr int32_t pairs_at() const { return 4 * nstep + 8 * nquad; }
};

// Leaf word: bits 0-4 level, 5-8 child index, 9 has a correction slot, 16-31
// the slot (a point index).
// Chain word (uint32), one per hanging leaf the replay passes: child (4) | reader
// + 1, 0 for a leaf that is none (6) << 4 | sibling group (6) << 10 | absent parent
// ranks << 16.
// Reader (uint64): first reader point (32) | mask of missing ranks << 32.
// Row word: a (13) | b (13) << 13 | e (4) << 26: the point is (a + b) / 2; an odd
// or reader point's accumulator is scaled by 2^-e before the transposed sums.
// Pair (uint32) and quad (uint64): two and four points of 16 bits; the target
// adds half the sum of their accumulators.  Sums go by steps: a step of a target
// set covers its first n targets, one pair or quad each, from word `first` of the
// tile: first (16) | n << 16.  Steps come in groups, of four (quads) and
// two (pairs); n = 0: no step.
// Replay block (uint64): as in plan_common.h, hanging indexes counted from the
// tile's first chain word.  Carry keys: nPe + 1 slot offsets, then local nodes.

struct PointHost {
  std::vector<PtTile> tiles;
  std::vector<uint32_t> blocks;  // 16-byte units
  std::vector<int32_t> snode, soff;
  std::vector<uint16_t> lloc;
  std::vector<uint32_t> laux;
  int max_nodes = 0, max_slots = 0, max_units = 0, max_hang = 0;
  int max_terms = 0;          // ends of rows (two each)
  int max_grp = 0;            // sibling groups of a replay (0: no tile has readers)
  size_t npartial = 0;
  size_t entries = 0;         // transposed terms (without the padding)
  std::vector<double> stats;  // as dkt_plan::stats
  size_t bytes() const;
};

// Whether a mesh's tiles fit the layout (the limits above): yes, perhaps with
// fewer leaves per tile, or with none.
enum class PtFit { yes, smaller, none };

// Reference semantics over the flattened traversal, tiles of at most T leaves.  T is
// halved where the tiles (the last one aside) hold fewer than min_leaves on average.
PtFit build_points_reference(const MeshParams &mp, const Traversal &tr, size_t N, int &T, int min_leaves, PointHost &out);

// Conforming operator (sum_e C_e^T K_e C_e, build_conforming): a rank that is no
// node takes its parent cell's interpolant, whose corners do the same one level
// up, so every hanging point is a row.  Tiles of T elements, with at most
// max_terms ends of rows.
PtFit build_points_conforming(const MeshParams &mp, const Traversal &tr, const std::vector<Oct> &nodes, int T,
                              int max_terms, PointHost &out);

}  // namespace dkt
