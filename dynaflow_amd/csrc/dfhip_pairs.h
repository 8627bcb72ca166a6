// Two launches of one kernel that read the same weights, as one (not part of the C ABI; see graph_pairs.hip).
#pragma once
#include "dfhip_common.h"

// What differs between the launches of two nano-batches: everything but the weights.  A kernel that can be paired takes
// two of these and a flag in its arguments.
struct DfhipSide {
  const void* A;
  const void* R;               // residual, or null
  void* C;
  const float* a_scale;        // fp8
  float* amax;                 // fp8, fused
  float* partials;             // K in parts
  int* arrivals;
  int64_t lda, ldc;
  int M;
};

// Launches whose sides may run at once: nothing that one of them writes is the other's.
inline bool dfhip_sides_apart(const DfhipSide& a, const DfhipSide& b) {
  return a.C != b.C && (!a.partials || a.partials != b.partials) && (!a.arrivals || a.arrivals != b.arrivals) &&
         (!a.amax || a.amax != b.amax);
}

// The side of a workgroup of a launch that has those of both (DFHIP_BESIDE) and its index in the launch of that side alone:
// eight workgroups of one side, one per XCD, then the same eight of the other, so that the two readers of a weight sit on one
// XCD and start together.
DFHIP_DEVICE int pair_block(int block, int blocks, int& side) {
  const int half = blocks >> 1, full = half & ~7;
  if (block < 2 * full) {
    side = (block >> 3) & 1;
    return (block >> 4) * 8 + (block & 7);
  }
  const int rest = block - 2 * full, odd = half - full;
  side = rest >= odd;
  return full + (side ? rest - odd : rest);
}

// Rows of a launch up to which the weights, and not the products, are its time.
constexpr int DFHIP_PAIR_MAX_M = 128;

// How a launch holds two sides: in workgroups of their own (pair_block), or the rows of both in every workgroup, which then
// takes a weight once for both.
enum DfhipPaired { DFHIP_ALONE = 0, DFHIP_BESIDE = 1, DFHIP_MERGED = 2 };

// The launch that two become.
struct DfhipJoined { const void* kernel; unsigned lds; unsigned grid; };

// Makes `kernel` known to dfhip_graph_pair_launches: its arguments are one struct of `bytes` bytes, and `join` makes those
// of a paired launch of two of `grid` workgroups each (false: not the same weights).
typedef bool (*DfhipJoin)(const void* a, const void* b, unsigned grid, void* both, DfhipJoined* joined);
constexpr size_t DFHIP_PAIR_MAX_ARGS = 512;
void dfhip_pairable(const void* kernel, size_t bytes, DfhipJoin join);
// How many workgroups a launch of `kernel` may have that runs in line with paired ones (the default: SHORT_BLOCKS).
void dfhip_in_line(const void* kernel, unsigned blocks);
