// GEMMs for the row counts and rounds that tiles of 256 rows cut badly, bf16 and fp8 e4m3:
//   C[M,N] = A[M,K] W[N,K]^T          bf16: optional residual [M,N] added in the epilogue
//   C[M,N] = silu(A W^T) * (A W2^T)   gate and up projection in one launch (fp8: with max |C| folded into a cell)
//
// Bound: up to some 256 rows how far ahead a compute unit fetches its weights (a slab from memory takes 1 - 2 us to come,
// longer the more units ask), then the share of a round that does work, then MFMA / power.  The ring kernels keep two and a
// half slabs of 128 bytes of K in units of 32 KiB whatever the tile is, and a W half is asked for less than one slab ahead of
// its use.  Here
//   * the tile decides: LDS holds as many whole slabs as fit, three of 224 + 192 rows up to five of 128 + 128;
//   * the fragments of a slab move to registers while the slab before it is multiplied (two sets, 208 registers for the
//     largest tiles), so its LDS is free for DMA as soon as its own products start: with three slabs a fetch has 1 to 2 slabs
//     of time (the loads of a slab are spread over all of it), with five 3 to 4; one barrier a slab;
//   * the two 32-byte halves of a fragment are read from LDS slots that lie in different banks for both types;
//   * parts of K end without a wait: the part that comes last adds the blocks of all in part order, four of them in flight.
// Every tile adds in the order of K of the other kernels of its type: the same bits.
// Measured (us, weights from memory, before -> now): fp8 128 x 14336 x 4096 36 -> 27, 64 x 8192 x 28672 79 -> 53, 128 x 28672 x 8192
// 73 -> 58 (4.1 TB/s; with the weights in the memory-side cache 42); bf16 670 x 28672 x 4096 154 -> 140, 560 x 14336 x 4096 69 -> 61,
// 777 x 4096 x 14336 104 -> 93, 300 x 4096 x 14336 in pairs 126 -> 83, 1554 x 2048 x 5632 59 -> 41.
// Tried and taken back: touching the W lines of later slabs (one 4-byte DMA per line, so that they wait in L2) - 5 to 10 us
// slower everywhere; 192 x 224, 256 x 160 and 64-row tiles - never the best of those that remain by more than 2 %.
#include "dfhip_pairs.h"
#include "dfhip_ring3.h"

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));

struct Ring3Args {
  const uint8_t* W;
  const uint8_t* W2;          // up weight (FUSED)
  const float* w_scale;       // fp8: per output channel
  const float* w2_scale;
  int N, slabs;               // slabs of 128 bytes per row
  int tiles_m, tiles_n, split_k;
  int64_t ldw;                // bytes (the strides of A too; that of C in elements)
  DfhipSide side[2];          // R (residual [M, N] with the row stride of C, or null): bf16, not FUSED
};
static_assert(sizeof(Ring3Args) <= DFHIP_PAIR_MAX_ARGS);

bool sides_ring3(const void* a, const void* b, void* both) {
  const Ring3Args &x = *static_cast<const Ring3Args*>(a), &y = *static_cast<const Ring3Args*>(b);
  if (!dfhip_sides_apart(x.side[0], y.side[0]) || x.W != y.W || x.W2 != y.W2 || x.w_scale != y.w_scale ||
      x.w2_scale != y.w2_scale || x.N != y.N || x.slabs != y.slabs || x.split_k != y.split_k || x.ldw != y.ldw || x.tiles_m != y.tiles_m || x.tiles_n != y.tiles_n ||
      x.side[0].M > DFHIP_PAIR_MAX_M || y.side[0].M > DFHIP_PAIR_MAX_M)
    return false;
  Ring3Args& out = *static_cast<Ring3Args*>(both);
  out = x;
  out.side[1] = y.side[0];
  return true;
}

constexpr int GROUP_M = 4;    // tiles of one XCD are walked in panels of GROUP_M tile rows
constexpr int SLAB = 128;     // bytes of K
// Slabs of a tile that LDS holds.
constexpr int units(int tm, int tn) { const int u = 160 * 1024 / ((tm + tn) * SLAB); return u < 6 ? u : 6; }

// The chunk of K that lies in slot `s` of an LDS row (before the XOR).  The products take the chunks of a slab in the order of
// the other kernels of the type: lane quad q multiplies chunks q and 4 + q in turn (bf16), 2 q and 2 q + 1 at once (fp8).  The
// quads read slots q and 4 + q either way, which is free of bank conflicts (2 q and 2 q + 1 is not).
template <bool FP8>
DFHIP_DEVICE int chunk_of(int s) { return FP8 ? 2 * (s & 3) + (s >> 2) : s; }

template <bool FP8, bool FUSED, int TM, int TN, bool SPLIT, bool BESIDE>
__global__ void __launch_bounds__(256)
gemm_ring3_kernel(const Ring3Args p) {
  static_assert(!(FUSED && SPLIT), "the fused form keeps K whole");
  constexpr int IB = TM / 32, JB = TN / 32;    // 16-row MFMA blocks of a wave (2 x 2 waves); also its DMA instructions of 8 rows
  constexpr int OUT_N = FUSED ? TN / 2 : TN;
  constexpr int A_UNIT = TM * SLAB, W_UNIT = TN * SLAB, U = units(TM, TN), W0 = U * A_UNIT;
  static_assert(U >= 3 && TM % 32 == 0 && TN % 32 == 0, "three slabs of the tile in LDS");
  constexpr int MQ = IB * JB, D = IB + JB, READS = 2 * D;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m = wave & 1, wave_n = wave >> 1;

  int at_side = 0;
  const int block = BESIDE ? pair_block(blockIdx.x, gridDim.x, at_side) : blockIdx.x;
  const DfhipSide& my = p.side[at_side];
  const int M = my.M;
  int tile, part = 0;
  if (SPLIT) splitk_work_of(block, p.tiles_m * p.tiles_n, tile, part);
  else tile = remap_xcd(block, p.tiles_m * p.tiles_n);
  const int per_panel = GROUP_M * p.tiles_n;
  const int first_m = (tile / per_panel) * GROUP_M;
  const int rows_in_panel = (p.tiles_m - first_m) < GROUP_M ? (p.tiles_m - first_m) : GROUP_M;
  const int in_panel = tile % per_panel;
  const int m0 = (first_m + in_panel % rows_in_panel) * TM;
  const int n0 = (in_panel / rows_in_panel) * OUT_N;
  const int slab0 = SPLIT ? (int)((int64_t)p.slabs * part / p.split_k) : 0;
  const int KT = SPLIT ? (int)((int64_t)p.slabs * (part + 1) / p.split_k) - slab0 : p.slabs;

  // DMA sources: a wave-uniform base (scalar registers) plus a 32-bit byte offset per lane.  LDS rows are 128 bytes with
  // the 16-byte chunk index XOR-ed by (row / 2) % 8.  FUSED: waves 0, 1 fetch the gate rows of a slab, 2, 3 the up rows.
  uint32_t a_off[IB], w_off[JB];
#pragma unroll
  for (int t = 0; t < IB; ++t) {
    const int row = (wave * IB + t) * 8 + (lane >> 3);
    int ar = m0 + row; ar = ar < M ? ar : M - 1;
    a_off[t] = (uint32_t)((int64_t)(ar - m0) * my.lda + chunk_of<FP8>((lane & 7) ^ ((row >> 1) & 7)) * 16);
  }
#pragma unroll
  for (int t = 0; t < JB; ++t) {
    const int row = (wave * JB + t) * 8 + (lane >> 3);
    int wr = n0 + (FUSED ? row % OUT_N : row); wr = wr < p.N ? wr : p.N - 1;
    w_off[t] = (uint32_t)((int64_t)(wr - n0) * p.ldw + chunk_of<FP8>((lane & 7) ^ ((row >> 1) & 7)) * 16);
  }
  const uint8_t* const a_tile = static_cast<const uint8_t*>(my.A) + (int64_t)m0 * my.lda + (int64_t)slab0 * SLAB;
  const uint8_t* const w_tile = ((FUSED && wave >= 2) ? p.W2 : p.W) + (int64_t)n0 * p.ldw + (int64_t)slab0 * SLAB;
  auto dma = [&](int t, int slab, int unit) {  // instruction t of a slab: A first, then W
    const int64_t s = (int64_t)(slab < KT ? slab : KT - 1) * SLAB;
    if (t < IB) dma16_base(unit * A_UNIT + (wave * IB + t) * 1024, a_tile + s, a_off[t]);
    else dma16_base(W0 + unit * W_UNIT + (wave * JB + t - IB) * 1024, w_tile + s, w_off[t - IB]);
  };

  // fragment of a 16-row block for a slab: lane -> row lane % 16, slots lane / 16 and 4 + lane / 16.  bf16: one slot is the
  // operand of one 16x16x32 product; fp8: both are that of one 16x16x128 product.
  // acc[i][j] (W block j first operand, A block i second): lane holds C[16 i + lane % 16][16 j + 4 (lane / 16) + r], r = 0..3
  const int frow = lane & 15, fquad = lane >> 4, fswz = (frow >> 1) & 7;
  int a_at[2], w_at[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int k = ((4 * h + fquad) ^ fswz) * 16;
    a_at[h] = (wave_m * (16 * IB) + frow) * SLAB + k;
    w_at[h] = W0 + (wave_n * (16 * JB) + frow) * SLAB + k;
  }
  u32x4 fa[2][IB][2], fw[2][JB][2];            // [slab parity][block][chunk]
  auto read = [&](int r, int slot, int unit) { // read r of a slab's fragments: block by block, A and W in turn
    const int b = r >> 1, h = r & 1;
    constexpr int BOTH = 2 * (IB < JB ? IB : JB);
    const bool is_a = b < BOTH ? b % 2 == 1 : IB > JB;
    const int blk = b < BOTH ? b / 2 : b - BOTH / 2;
    if (is_a) fa[slot][blk][h] = *reinterpret_cast<const u32x4*>(smem + unit * A_UNIT + a_at[h] + blk * 2048);
    else fw[slot][blk][h] = *reinterpret_cast<const u32x4*>(smem + unit * W_UNIT + w_at[h] + blk * 2048);
  };

  f32x4 acc[IB][JB];
#pragma unroll
  for (int i = 0; i < IB; ++i)
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      asm volatile("" : "+a"(acc[i][j]));      // in place before the first product (whose wait states the compiler does not know)
    }
  const int unit_scale = 0x7f7f7f7f;           // e8m0 scales 2^0
  auto multiply = [&](int q, int slot) {       // snake order: odd rows walk the W blocks backwards
    const int i = q / JB, j = (i & 1) ? JB - 1 - q % JB : q % JB;
    const u32x4 a0 = fa[slot][i][0], a1 = fa[slot][i][1], w0 = fw[slot][j][0], w1 = fw[slot][j][1];
    if constexpr (FP8) {
      const i32x8 av = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
      const i32x8 wv = {(int)w0[0], (int)w0[1], (int)w0[2], (int)w0[3], (int)w1[0], (int)w1[1], (int)w1[2], (int)w1[3]};
      asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %3 op_sel_hi:[0,0,0]"
                   : "+a"(acc[i][j]) : "v"(wv), "v"(av), "v"(unit_scale));
    } else {
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\tv_mfma_f32_16x16x32_bf16 %0, %3, %4, %0"
                   : "+a"(acc[i][j]) : "v"(w0), "v"(a0), "v"(w1), "v"(a1));
    }
  };

#pragma unroll
  for (int s = 0; s < U; ++s)
#pragma unroll
    for (int t = 0; t < D; ++t) dma(t, s, s);
  wait_vmcnt<(U - 1) * D>();                         // slab 0 has landed
  workgroup_barrier();
  asm volatile("s_nop 7" ::: "memory");
#pragma unroll
  for (int r = 0; r < READS; ++r) read(r, 0, 0);
  int u = 0;                                   // unit of the slab being multiplied
  auto slab = [&](int kt, int slot) {
    // The fragments of slab kt are in registers, so its units are free; slab kt + 1 must have landed, slab kt + 2 may be
    // in flight.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    wait_vmcnt<(U - 2) * D>();
    workgroup_barrier();
    const int next = u == U - 1 ? 0 : u + 1;
    // The loads are spread over the whole slab, the reads over three quarters of it.  A compute unit has 32 KiB of loads in flight
    // whatever is asked for, so loads asked for early only make the waves wait, and what they put into LDS keeps the reads from it; half a
    // slab later is early enough.  [us, first third of a slab -> all of it, alone with weights from memory / in the memory-side cache: 670 x
    // 28672 x 4096 132 / 120 -> 128 / 113, 777 x 4096 x 14336 uncut 186 / 179 -> 183 / 156, 1554 x 28672 x 4096 300 / 294 -> 288 / 277; all at
    // the head of a slab 144 / 134, 220 / 219, 336 / 333; weights before activations 143 / 121, 211 / 176, 320 / 298]
    constexpr int RQ = (MQ * 3 + 3) / 4;
#pragma unroll
    for (int q = 0; q < MQ; ++q) {
      multiply(q, slot);
#pragma unroll
      for (int r = q * READS / RQ; r < (q + 1) * READS / RQ && r < READS; ++r) read(r, slot ^ 1, next);
#pragma unroll
      for (int t = q * D / MQ; t < (q + 1) * D / MQ; ++t) dma(t, kt + U, u);
      DFHIP_PIN;
    }
    u = next;
  };
  int kt = 0;
  for (; kt + 1 < KT; kt += 2) {
    slab(kt, 0);
    slab(kt + 1, 1);
  }
  if (kt < KT) slab(kt, 0);
  wait_vmcnt<0>();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  workgroup_barrier();                         // nobody reads or fills a unit any more
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMAs have written their accumulators
#pragma unroll
  for (int i = 0; i < IB; ++i)
#pragma unroll
    for (int j = 0; j < JB; ++j) asm volatile("" : "+a"(acc[i][j]));

  if constexpr (SPLIT) {
    // Every part leaves its fp32 block and takes a ticket; the part that comes last adds the blocks in part order (its own
    // too: the same bits whoever is last) and writes the tile.  Nobody waits.
    constexpr int BLOCK = MQ * 256;            // f32x4 of a part
    f32x4* const blocks = reinterpret_cast<f32x4*>(my.partials) + (int64_t)tile * p.split_k * BLOCK;
    f32x4* const mine = blocks + part * BLOCK + tid;
    // Row blocks of this wave that have rows: the others are not exchanged (fp8 layer 8192 x 28672 of 2 x 8 tokens 158 -> 145 us).
    const int live = (M - m0 - wave_m * (16 * IB) + 15) / 16;
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      if (i >= live) break;
#pragma unroll
      for (int j = 0; j < JB; ++j) store_f32x4_device_coherent(mine + (i * JB + j) * 256, acc[i][j]);
    }
    wait_vmcnt<0>();
    __syncthreads();
    int* const ticket_cell = reinterpret_cast<int*>(smem);
    if (tid == 0) *ticket_cell = atomicAdd(my.arrivals + tile, 1);
    __syncthreads();
    const int ticket = *ticket_cell;
    if (ticket != p.split_k - 1) return;
    if (tid == 0) atomicExch(my.arrivals + tile, 0);      // counters are left at zero
    __syncthreads();                                     // the ticket has been read before the tile is parked over it
    const auto left = coherent_blocks(blocks, p.split_k * BLOCK * 16);
    // 4 JB loads in flight (a load from the memory side takes microseconds when every tile is at it)
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      if (i >= live) break;
      f32x4 sum[JB];
#pragma unroll
      for (int j = 0; j < JB; ++j) sum[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      for (int q0 = 0; q0 < p.split_k; q0 += 4) {
        f32x4 v[4][JB];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int q = q0 + c < p.split_k ? q0 + c : p.split_k - 1;
#pragma unroll
          for (int j = 0; j < JB; ++j) v[c][j] = load_f32x4_device_coherent(left, tid * 16, q * (BLOCK * 16) + (i * JB + j) * 4096);
        }
        DFHIP_PIN;
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (q0 + c < p.split_k)
#pragma unroll
            for (int j = 0; j < JB; ++j) sum[j] += v[c][j];
      }
#pragma unroll
      for (int j = 0; j < JB; ++j) {
        acc[i][j] = sum[j];
        asm volatile("" : "+a"(acc[i][j]));
      }
    }
  }

  // round to bf16 (fp8: scale first), park the wave's block in LDS, store whole row pieces of 16 bytes
  constexpr int PROW = JB * 32 + 16, CPR = JB * 2;       // padded row of a park (bytes), pieces of a row
  const float sa = FP8 ? my.a_scale[0] : 1.0f;
  uint8_t* const park = smem + wave * (16 * IB * PROW);
#pragma unroll
  for (int j = 0; j < JB; ++j) {
    f32x4 ws = {1.0f, 1.0f, 1.0f, 1.0f};
    if constexpr (FP8) {
      int n = n0 + (FUSED ? 0 : wave_n * (16 * JB)) + j * 16 + fquad * 4;
      n = n < p.N ? n : p.N - 4;               // columns past the edge are never stored; keep the scale load in bounds
      ws = *reinterpret_cast<const f32x4*>((FUSED && wave_n ? p.w2_scale : p.w_scale) + n);
    }
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      f32x4 v = acc[i][j];
      if constexpr (FP8) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= sa * ws[e];
      }
      const u32x2 o = {pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3])};
      *reinterpret_cast<u32x2*>(park + (i * 16 + frow) * PROW + (j * 16 + fquad * 4) * 2) = o;
    }
  }
  DFHIP_PIN;
  if constexpr (FUSED) {
    // gate blocks sit in the parks of waves 0, 1 (the two halves of the rows), up blocks in those of waves 2, 3; wave w
    // combines half (w >> 1) of the rows of park w & 1
    __syncthreads();
    const uint8_t* const gpark = smem + (wave & 1) * (16 * IB * PROW);
    const uint8_t* const upark = smem + ((wave & 1) + 2) * (16 * IB * PROW);
    const int row0 = (wave >> 1) * (8 * IB);
    float vmax = 0.0f;
#pragma unroll 4
    for (int q = 0; q < (8 * IB * CPR + 63) / 64; ++q) {
      const int id = q * 64 + lane;
      const int row = row0 + id / CPR, c = id % CPR;
      const int m = m0 + (wave & 1) * (16 * IB) + row, n = n0 + c * 8;
      if (id >= 8 * IB * CPR || m >= M || n >= p.N) continue;   // N % 8 == 0: a piece is inside or outside
      const u32x4 gv = *reinterpret_cast<const u32x4*>(gpark + row * PROW + c * 16);
      const u32x4 uv = *reinterpret_cast<const u32x4*>(upark + row * PROW + c * 16);
      u32x4 o;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        float lo = silu_fast(bf16_lo_to_f32(gv[w])), hi = silu_fast(bf16_hi_to_f32(gv[w]));
        if (!FP8) {                            // bf16: silu is rounded before the product
          const uint32_t s2 = pack2_bf16(lo, hi);
          lo = bf16_lo_to_f32(s2);
          hi = bf16_hi_to_f32(s2);
        }
        o[w] = pack2_bf16(lo * bf16_lo_to_f32(uv[w]), hi * bf16_hi_to_f32(uv[w]));
        if (FP8) vmax = fmaxf(vmax, fmaxf(fabsf(bf16_lo_to_f32(o[w])), fabsf(bf16_hi_to_f32(o[w]))));
      }
      u32x4* const at = reinterpret_cast<u32x4*>(static_cast<uint16_t*>(my.C) + (int64_t)m * my.ldc + n);
      if (FP8) *at = o; else __builtin_nontemporal_store(o, at);
    }
    if constexpr (FP8) {
      fold_amax(my, block, wave, wave_max(vmax));
    }
  } else {
    const int m_base = m0 + wave_m * (16 * IB), n_base = n0 + wave_n * (16 * JB);
#pragma unroll 4
    for (int q = 0; q < (16 * IB * CPR + 63) / 64; ++q) {
      const int id = q * 64 + lane;
      const int row = id / CPR, c = id % CPR;
      const int m = m_base + row, n = n_base + c * 8;
      if (id >= 16 * IB * CPR || m >= M || n >= p.N) continue;
      u32x4 v = *reinterpret_cast<const u32x4*>(park + row * PROW + c * 16);
      u32x4* const at = reinterpret_cast<u32x4*>(static_cast<uint16_t*>(my.C) + (int64_t)m * my.ldc + n);
      if (FP8) { *at = v; continue; }
      if (my.R) {
        const u32x4 r = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(my.R) + (int64_t)m * my.ldc + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = add2_bf16(v[e], r[e]);
      }
      __builtin_nontemporal_store(v, at);
    }
  }
}

template <bool FP8, bool FUSED, bool SPLIT, int T>
bool join_ring3(const void* a, const void* b, dim3 ga, dim3 gb, void* both, DfhipJoined* joined) {
  constexpr int TM = DFHIP_RING3[T].rows, TN = DFHIP_RING3[T].cols;
  constexpr int LDS = units(TM, TN) * (TM + TN) * SLAB;
  static std::atomic<uint64_t> lds_opted_in{0};
  *joined = {reinterpret_cast<const void*>(gemm_ring3_kernel<FP8, FUSED, TM, TN, SPLIT, true>), LDS, dim3(2 * ga.x)};
  return dfhip_same(ga, gb) && sides_ring3(a, b, both) && dfhip_opt_in_lds(joined->kernel, LDS, lds_opted_in) == DFHIP_OK;
}

template <bool FP8, bool FUSED, bool SPLIT, int T>
int launch(Ring3Args p, void* workspace, hipStream_t stream) {
  constexpr int TM = DFHIP_RING3[T].rows, TN = DFHIP_RING3[T].cols, OUT_N = FUSED ? TN / 2 : TN;
  constexpr int LDS = units(TM, TN) * (TM + TN) * SLAB;
  auto kernel = gemm_ring3_kernel<FP8, FUSED, TM, TN, SPLIT, false>;
  static std::atomic<uint64_t> lds_opted_in{0};
  if (int rc = dfhip_opt_in_lds(reinterpret_cast<const void*>(kernel), LDS, lds_opted_in)) return rc;
  p.tiles_m = (p.side[0].M + TM - 1) / TM;
  p.tiles_n = (p.N + OUT_N - 1) / OUT_N;
  if (SPLIT) {
    const size_t tiles = (size_t)p.tiles_m * p.tiles_n;
    if (int rc = dfhip_clear_uncommon_counters(workspace, tiles, stream)) return rc;
    p.side[0].partials = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + dfhip_counter_area(tiles));
    p.side[0].arrivals = static_cast<int*>(workspace);
  }
  static const bool known = (dfhip_pairable(reinterpret_cast<const void*>(kernel), join_ring3<FP8, FUSED, SPLIT, T>), true);
  (void)known;
  hipLaunchKernelGGL(kernel, dim3(p.tiles_m * p.tiles_n * p.split_k), dim3(256), LDS, stream, p);
  return dfhip_check_launch();
}

template <bool FP8, bool FUSED, bool SPLIT, int T = 0>
int launch_tile(const Ring3Args& p, int tile, void* workspace, hipStream_t stream) {
  if constexpr (T < DFHIP_RING3_TILES) {
    if constexpr (!FP8 || DFHIP_RING3[T].fp8.slab > 0.0)
      if (tile == T) return launch<FP8, FUSED, SPLIT, T>(p, workspace, stream);
    return launch_tile<FP8, FUSED, SPLIT, T + 1>(p, tile, workspace, stream);
  }
  return DFHIP_ERR_BAD_ARGUMENT;
}

}  // namespace

DfhipRing3Plan dfhip_ring3_plan(bool fp8, bool gate_up, int M, int N, int K, int share, bool may_split) {
  const double slabs = K / (fp8 ? 128.0 : 64.0), weight_mb = (double)N * K * (fp8 ? 1 : 2) * (gate_up ? 2 : 1) * 1e-6;
  DfhipRing3Plan best{-1, 1, 0.0};
  for (int t = 0; t < DFHIP_RING3_TILES; ++t) {
    if (!dfhip_ring3_variant(DFHIP_RING3_VARIANT + t, fp8)) continue;
    const int cols = DFHIP_RING3[t].cols / (gate_up ? 2 : 1);
    const int64_t tiles = (int64_t)((M + DFHIP_RING3[t].rows - 1) / DFHIP_RING3[t].rows) * ((N + cols - 1) / cols);
    for (int s = 1; s <= DFHIP_RING3_MAX_SPLIT; ++s) {
      if (s > 1 && (!may_split || slabs < 8.0 * s || tiles * s * share > 256)) break;
      const DfhipPrice& price = fp8 ? DFHIP_RING3[t].fp8 : DFHIP_RING3[t].bf16;
      const double cost = dfhip_price(price, tiles, share, slabs, s, weight_mb);
      if (best.tile < 0 || cost < best.cost) best = {t, s, cost};
    }
  }
  return best;
}

size_t dfhip_ring3_workspace_bytes(int M, int N, int tile, int split_k) {
  const DfhipRing3Tile& t = DFHIP_RING3[tile];
  const size_t tiles = (size_t)((M + t.rows - 1) / t.rows) * ((N + t.cols - 1) / t.cols);
  return dfhip_counter_area(tiles) + tiles * split_k * t.rows * t.cols * sizeof(float);
}

int dfhip_ring3_bf16(const void* A, int64_t lda, const void* W, int64_t ldw, const void* R, void* C, int64_t ldc, int M,
                     int N, int K, int tile, int split_k, void* workspace, hipStream_t stream) {
  const Ring3Args p{static_cast<const uint8_t*>(W), nullptr, nullptr, nullptr, N, K / 64, 0, 0, split_k, ldw * 2,
                    {{A, R, C, nullptr, nullptr, nullptr, nullptr, lda * 2, ldc, M}, {}}};
  return split_k > 1 ? launch_tile<false, false, true>(p, tile, workspace, stream)
                     : launch_tile<false, false, false>(p, tile, nullptr, stream);
}
int dfhip_ring3_bf16_gate_up(const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, void* C, int64_t ldc,
                             int M, int N, int K, int tile, hipStream_t stream) {
  const Ring3Args p{static_cast<const uint8_t*>(W), static_cast<const uint8_t*>(W2), nullptr, nullptr, N, K / 64, 0, 0, 1,
                    ldw * 2, {{A, nullptr, C, nullptr, nullptr, nullptr, nullptr, lda * 2, ldc, M}, {}}};
  return launch_tile<false, true, false>(p, tile, nullptr, stream);
}
int dfhip_ring3_fp8(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, const float* a_scale,
                    const float* w_scale, int M, int N, int K, int tile, int split_k, void* workspace, hipStream_t stream) {
  const Ring3Args p{static_cast<const uint8_t*>(W), nullptr, w_scale, nullptr, N, K / 128, 0, 0, split_k, ldw,
                    {{A, nullptr, C, a_scale, nullptr, nullptr, nullptr, lda, ldc, M}, {}}};
  return split_k > 1 ? launch_tile<true, false, true>(p, tile, workspace, stream)
                     : launch_tile<true, false, false>(p, tile, nullptr, stream);
}
int dfhip_ring3_fp8_gate_up(const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, void* C, int64_t ldc,
                            const float* a_scale, const float* w_scale, const float* w2_scale, float* amax, bool amax_apart,
                            int M, int N, int K, int tile, hipStream_t stream) {
  const Ring3Args p{static_cast<const uint8_t*>(W), static_cast<const uint8_t*>(W2), w_scale, w2_scale, N, K / 128, 0, 0, 1,
                    ldw, {{A, nullptr, C, a_scale, amax, nullptr, nullptr, lda, ldc, M, amax_apart}, {}}};
  return launch_tile<true, true, false>(p, tile, nullptr, stream);
}
int dfhip_ring3_gate_up_blocks(int M, int N, int tile) {
  const DfhipRing3Tile& t = DFHIP_RING3[tile];
  return ((M + t.rows - 1) / t.rows) * ((N + t.cols / 2 - 1) / (t.cols / 2));
}
