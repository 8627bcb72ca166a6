// GEMMs on tiles of which three slabs fit into LDS, shared by the bf16 and fp8 entry points (not part of the C ABI).
// Pointers, strides and shapes have been checked by the caller.
#pragma once

#include "dfhip_common.h"

// What a launch of tiles costs (us, to the sixth power: a sum that is close to the larger of two bounds), for a choice between
// kernels.  `share` launches of one shape side by side take their
// rounds of 256 workgroups together.  A round costs a start and an end and, per slab of K, a time that grows with the share of
// the compute units at work (the clock falls with the power they draw); parts of K cost their meeting; and the weights do
// not come in faster than `intake` (MB per us, i.e. TB/s).  Fitted to timings of the tiles below and of the kernels
// beside them at 17 .. 4096 rows, alone and in pairs, on fp8 weights 28672 x 8192, 14336 x 4096 and transposed, bf16 ones
// also 6144 x 4096, 4096 x 4096, 5632 x 2048.  Timed again, alone, on these and on 11264 x 2048 and fp8 16384 x 4096 and transposed: of the 767 timings
// within 25 % of the fastest of their shape 9 % off on average and 18 % for nine in ten; two launches in step on two streams take
// 5 - 30 % less than priced (they read their weights together).  That was before a slab's loads were spread over all of it.  With them
// spread the bf16 prices of 428 such timings are 6 % too high on average alone and level in pairs, 9 and 7 % off, 15 % for nine in ten,
// and the tile chosen takes 0.1 % more than the fastest of these alone (3.6 % at worst) and 1.5 % in pairs (10.5 %: 1100 x 2048 x 5632).  What the choices
// by it give stands at three_slabs_cheaper.
struct DfhipPrice { double slab, slab_full, round, parts, part, intake; };
inline double dfhip_price(const DfhipPrice& p, int64_t tiles, int share, double slabs, int split_k, double weight_mb) {
  const int64_t work = tiles * split_k * share;
  const double rounds = (double)((work + 255) / 256);
  const double meet = split_k > 1 ? p.parts + p.part * split_k : 0.0;
  const double compute = rounds * (slabs / split_k * (p.slab + p.slab_full * (double)work / (256.0 * rounds)) + p.round) + meet + 3.0;
  const double load = weight_mb * share / p.intake + meet + 8.0;
  const double c3 = compute * compute * compute, l3 = load * load * load;
  return c3 * c3 + l3 * l3;
}

struct DfhipRing3Tile {
  int rows, cols;             // rows of A, rows of W (gate + up: half of them each)
  DfhipPrice bf16, fp8;       // fp8: not built where zero (no shape gained from the others)
};
constexpr DfhipRing3Tile DFHIP_RING3[] = {
    {224, 192, {0.684, 0.303, 6.18, 7.73, 1.03, 4.56}, {}},
    {160, 256, {0.673, 0.289, 5.21, 7.63, 1.10, 5.00}, {0.665, 0.340, 5.46, 5.96, 1.30, 6.41}},
    {128, 256, {0.625, 0.205, 3.50, 7.59, 0.69, 4.90}, {0.586, 0.295, 4.92, 4.83, 1.02, 6.28}},
    {192, 192, {0.574, 0.289, 4.89, 7.60, 0.90, 5.40}, {}},
    {128, 192, {0.495, 0.174, 2.93, 6.59, 0.51, 4.14}, {}},
    {128, 128, {0.351, 0.143, 2.00, 5.82, 0.08, 4.40}, {0.293, 0.247, 2.65, 3.45, 0.30, 6.46}},
};
constexpr int DFHIP_RING3_TILES = sizeof(DFHIP_RING3) / sizeof(DFHIP_RING3[0]);
constexpr int DFHIP_RING3_VARIANT = 10;        // variants from here on are these tiles, in order
constexpr int DFHIP_RING3_MAX_SPLIT = 16;
inline bool dfhip_ring3_variant(int variant, bool fp8) {
  const int t = variant - DFHIP_RING3_VARIANT;
  return t >= 0 && t < DFHIP_RING3_TILES && (!fp8 || DFHIP_RING3[t].fp8.slab > 0.0);
}

struct DfhipRing3Plan { int tile, split_k; double cost; };
// The cheapest of the tiles; K in parts only if `may_split`, eight slabs a part at least, and all parts in one round.
DfhipRing3Plan dfhip_ring3_plan(bool fp8, bool gate_up, int M, int N, int K, int share, bool may_split);

// split_k > 1: `workspace` starts with the arrival counters (left zero) and holds the blocks of every part.
size_t dfhip_ring3_workspace_bytes(int M, int N, int tile, int split_k);
int dfhip_ring3_bf16(const void* A, int64_t lda, const void* W, int64_t ldw, const void* R, void* C, int64_t ldc, int M,
                     int N, int K, int tile, int split_k, void* workspace, hipStream_t stream);
int dfhip_ring3_bf16_gate_up(const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, void* C, int64_t ldc,
                             int M, int N, int K, int tile, hipStream_t stream);
int dfhip_ring3_fp8(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, const float* a_scale,
                    const float* w_scale, int M, int N, int K, int tile, int split_k, void* workspace, hipStream_t stream);
int dfhip_ring3_fp8_gate_up(const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, void* C, int64_t ldc,
                            const float* a_scale, const float* w_scale, const float* w2_scale, float* amax, bool amax_apart,
                            int M, int N, int K, int tile, hipStream_t stream);
// Workgroups of the latter; with `amax_apart` each leaves four maxima.
int dfhip_ring3_gate_up_blocks(int M, int N, int tile);
