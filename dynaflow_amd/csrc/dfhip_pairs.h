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
  float* amax;                 // fp8, fused: a cell, or one float per wave of the side's workgroups (fold_amax)
  float* partials;             // K in parts
  int* arrivals;
  int64_t lda, ldc;
  int M;
  bool amax_apart;             // the waves leave their maxima side by side
};

// The maximum of wave `wave` of the side's workgroup `block`, whose lanes have it in `top` (0 and more).  Side by side where there is
// room: no cell to clear first, and no queue of atomics on one address (12 ns each, of 1792 waves at 28672 columns) at the end of a
// launch.  [us, fp8 layer 8192 x 28672 of 2 x 12 tokens 142 -> 130]
DFHIP_DEVICE void fold_amax(const DfhipSide& side, int block, int wave, float top) {
  if ((threadIdx.x & 63) != 0) return;
  if (side.amax_apart) side.amax[4 * block + wave] = top;
  // non-negative floats order like their bit patterns
  else if (top > 0.0f) atomicMax(reinterpret_cast<unsigned int*>(side.amax), __float_as_uint(top));
}

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
struct DfhipJoined { const void* kernel; unsigned lds; dim3 grid; };

// Makes `kernel` known to dfhip_graph_pair_launches: its arguments are one struct, and `join` makes those of the launch that
// two of grids ga and gb become (false: they are not the same work on different rows).  `in_line`: how many workgroups a
// launch without a partner may have that runs in line with paired ones; none at all for those that read weights.
typedef bool (*DfhipJoin)(const void* a, const void* b, dim3 ga, dim3 gb, void* both, DfhipJoined* joined);
constexpr size_t DFHIP_PAIR_MAX_ARGS = 512;
constexpr unsigned DFHIP_SHORT_BLOCKS = 512;     // also that of a kernel that is not known
void dfhip_pairable(const void* kernel, DfhipJoin join, unsigned in_line = 0);
// A long kernel of which there is no launch of two: a graph that holds one stays as it is.
#define DFHIP_NOT_IN_LINE(kernel) \
  do { \
    static const bool known = (dfhip_pairable(reinterpret_cast<const void*>(kernel), nullptr), true); \
    (void)known; \
  } while (0)
inline bool dfhip_same(dim3 a, dim3 b) { return a.x == b.x && a.y == b.y && a.z == b.z; }

// A launch without weights is K::run(workgroup) of K::THREADS threads; two of them sit one behind the other.
template <class K>
struct DfhipBoth { K side[2]; unsigned blocks; };
template <class K>
__global__ void __launch_bounds__(K::THREADS) dfhip_beside_kernel(const DfhipBoth<K> p) {
  const unsigned second = blockIdx.x >= p.blocks;
  p.side[second].run(blockIdx.x - (second ? p.blocks : 0), second ? gridDim.x - p.blocks : p.blocks);
}
template <class K>
bool dfhip_join_as(const void* kernel, const void* a, const void* b, dim3 ga, dim3 gb, void* both, DfhipJoined* joined) {
  static_assert(sizeof(DfhipBoth<K>) <= DFHIP_PAIR_MAX_ARGS);
  const K &x = *static_cast<const K*>(a), &y = *static_cast<const K*>(b);
  *joined = {kernel, joined->lds, dim3(ga.x + gb.x, ga.y > gb.y ? ga.y : gb.y)};
  *static_cast<DfhipBoth<K>*>(both) = {{x, y}, ga.x};
  return x.beside(y);
}
template <class K>
bool dfhip_join_beside(const void* a, const void* b, dim3 ga, dim3 gb, void* both, DfhipJoined* joined) {
  return dfhip_join_as<K>(reinterpret_cast<const void*>(dfhip_beside_kernel<K>), a, b, ga, gb, both, joined);
}
