// Weight-streaming GEMMs for a handful of activation rows (M <= 64), bf16 and fp8 e4m3:
//   C[M,N] = A[M,K] W[N,K]^T          bf16: optional residual [M,N] added in the epilogue
//   C[M,N] = silu(A W^T) * (A W2^T)   gate and up projection in one launch (fp8: max |C| beside it, a float a tile or one cell)
//
// Bound: HBM.  Every weight is read once and used for at most 64 rows, so the kernel is a load loop with a few
// MFMAs in it.  What it is built for is many loads in flight and nothing that makes them wait for each other:
//   * a workgroup owns 16, 32 or 64 columns (rows of W) and all of K, or one part of it; its four waves take the
//     128-byte slabs of the rows in turn (wave w: slabs w, w + 4, ...) and up to four slabs per wave are in flight;
//   * weights and activations go straight from memory to registers, no LDS and no barrier inside the loop.  A load
//     takes eight whole 128-byte lines (half a block of 16 rows), which is what lets the weights be loaded
//     non-temporally; neighbouring lanes, which share 32 bytes, then exchange a piece each (DPP), which gives the MFMA
//     operand layout;
//   * the activation rows are re-read by every workgroup from its XCD's L2; the rows of a matrix lie a multiple of
//     4 KiB apart and so on one L2 channel, hence the workgroups start at different slabs;
//   * at the end the four partial sums meet in LDS and are added in wave order.  Where K is cut into parts (a
//     caller's workspace), the part that arrives last adds them in part order: the same bits in every run.
// The order in which a column's K is summed depends on K, on the cut and on the column's tile, whose number says at which
// slab its waves start: a row of W can sum in another order in a matrix of another N, or at another place in it.  The
// fused launch has the bits of the separate, uncut ones because N, and with it the tiles, are the same.
// Measured (weights from HBM, us; M = 2 / 16 / 32 rows, against the 128-row tiles used before): gate + up + SiLU*mul
// 2 x 14336 x 4096 (235 MB) 38 / 38 / 39, before 51; down 4096 x 14336 22 / 22 / 24, before 207 / 36 / 36; q/k/v
// 6144 x 4096 11 / 12 / 16, before 62 / 22 / 22; o 4096 x 4096 8 / 10 / 11, before 61 / 21 / 21.  At 8 / 16 / 32 / 64
// rows fp8 down 8192 x 28672 (235 MB) 36 / 37 / 44 / 58, before 240 (two of 12 / 32 rows in one launch, K in parts: 40 / 49);
// fp8 gate + up 2 x 28672 x 8192 (470 MB) 77 / 76 / 84 / 96, before 113 - 117.
#include "dfhip_pairs.h"
#include "dfhip_stream.h"

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));

struct StreamArgs {
  const uint8_t* W;
  const uint8_t* W2;          // up weight (FUSED)
  const float* w_scale;       // fp8: per output channel
  const float* w2_scale;
  int N, slabs;               // slabs of 128 bytes per row
  int split_k;                // workgroups per tile along K (not FUSED)
  int64_t ldw;                // bytes (the strides of A too; that of C in elements)
  DfhipSide side[2];          // R (residual [M, N] with the row stride of C, or null): bf16, not FUSED
};
static_assert(sizeof(StreamArgs) <= DFHIP_PAIR_MAX_ARGS);

bool sides_stream(const void* a, const void* b, void* both) {
  const StreamArgs &x = *static_cast<const StreamArgs*>(a), &y = *static_cast<const StreamArgs*>(b);
  if (!dfhip_sides_apart(x.side[0], y.side[0]) || x.W != y.W || x.W2 != y.W2 || x.w_scale != y.w_scale ||
      x.w2_scale != y.w2_scale || x.N != y.N || x.slabs != y.slabs || x.split_k != y.split_k || x.ldw != y.ldw ||
      !x.side[0].R != !y.side[0].R)
    return false;
  StreamArgs& out = *static_cast<StreamArgs*>(both);
  out = x;
  out.side[1] = y.side[0];
  return true;
}

constexpr int WAVES = 4;

// Row blocks whose partial sums lie in LDS together: all of them within 64 KiB, else as many as fit.
constexpr int rows_per_round(int mb, int nb) {
  int r = mb;
  while (r > 1 && WAVES * r * nb > 64) r /= 2;
  return r;
}

// MERGED: the rows of side 1 follow those of side 0; else all are side 0.
template <bool FP8, int MB, int NB, int DEPTH, bool FUSED, bool SPLIT, bool MERGED>
__global__ void __launch_bounds__(WAVES * 64)
gemm_stream_kernel(const StreamArgs p) {
  constexpr int THREADS = WAVES * 64;
  constexpr int OB = FUSED ? NB / 2 : NB;       // 16-column blocks of the output
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = SPLIT ? blockIdx.x / p.split_k : blockIdx.x;
  const int part = SPLIT ? blockIdx.x - tile * p.split_k : 0;
  const int second = MERGED ? p.side[0].M : 16 * MB;      // the first row of side 1
  const int n0 = tile * (16 * OB);
  const int slab0 = SPLIT ? (int)((int64_t)p.slabs * part / p.split_k) : 0;
  const int slabs = SPLIT ? (int)((int64_t)p.slabs * (part + 1) / p.split_k) - slab0 : p.slabs;

  // load h of a slab takes rows h, 2 + h .. 14 + h of a block, whole 128-byte lines (lane: row 2 (lane / 2 % 8) + h, chunk
  // 2 (lane / 16) + lane % 2).  Neighbouring lanes share 32 bytes: with one row per lane (row lane % 8, chunk lane / 8) a
  // compute unit takes in 34 GB/s at most, from its L2 too and whatever is in flight, with pairs of lanes 66 (with eight
  // lanes to a line 114, but then the exchange has three stages).  [us: decode step of 40 x 4096 positions, 4 layers
  // 819 -> 771, fp8 layer 8192 x 28672 of 2 x 12 tokens 174 -> 166]
  const int lrow = lane & 14, lchunk = 2 * (lane >> 4) + (lane & 1);
  const uint8_t* w_ptr[NB][2];
  const uint8_t* a_ptr[MB][2];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int n = n0 + 16 * (FUSED ? j % OB : j) + lrow + h;
      n = n < p.N ? n : p.N - 1;                   // columns past the edge re-read the last one; never stored
      w_ptr[j][h] = (FUSED && j >= OB ? p.W2 : p.W) + (int64_t)n * p.ldw + (slab0 + wave) * 128 + lchunk * 16;
    }
#pragma unroll
  for (int i = 0; i < MB; ++i) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int m = 16 * i + lrow + h;
      const bool other = MERGED && m >= second;
      m -= other ? second : 0;
      const int M = other ? p.side[1].M : p.side[0].M;
      m = m < M ? m : M - 1;
      a_ptr[i][h] = static_cast<const uint8_t*>(other ? p.side[1].A : p.side[0].A) +
                    (int64_t)m * (other ? p.side[1].lda : p.side[0].lda) + (slab0 + wave) * 128 + lchunk * 16;
    }
  }
  const int n_slabs = (slabs - wave + WAVES - 1) / WAVES;   // >= DEPTH: a part has at least MIN_SLABS slabs

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  u32x4 wf[DEPTH][NB][2], af[DEPTH][MB][2];
  // the workgroups of an XCD start at different slabs
  const int rot = (int)((unsigned)(tile >> 3) % (unsigned)n_slabs);
  auto load = [&](int d, int s) {
    int sr = s + rot; sr = sr >= n_slabs ? sr - n_slabs : sr;
    const int64_t off = (int64_t)sr * (WAVES * 128);
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        wf[d][j][h] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w_ptr[j][h] + off));
      }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) af[d][i][h] = *reinterpret_cast<const u32x4*>(a_ptr[i][h] + off);
  };
  auto multiply = [&](int d) {
#pragma unroll
    for (int j = 0; j < NB; ++j) deal_neighbours(wf[d][j][0], wf[d][j][1]);
#pragma unroll
    for (int i = 0; i < MB; ++i) deal_neighbours(af[d][i][0], af[d][i][1]);
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        if constexpr (FP8) {
          const u32x4 a0 = af[d][i][0], a1 = af[d][i][1], w0 = wf[d][j][0], w1 = wf[d][j][1];
          const i32x8 av = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
          const i32x8 wv = {(int)w0[0], (int)w0[1], (int)w0[2], (int)w0[3], (int)w1[0], (int)w1[1], (int)w1[2], (int)w1[3]};
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wv, av, acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0,
                                                                      0x7f7f7f7f);
        } else {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[d][j][h]),
                                                                __builtin_bit_cast(bf16x8, af[d][i][h]), acc[i][j], 0,
                                                                0, 0);
        }
      }
  };

#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load(d, d);
  int s = 0;
  for (; s + 2 * DEPTH <= n_slabs; s += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      multiply(d);
      load(d, s + DEPTH + d);
      DFHIP_PIN;
    }
  }
  const int rest = n_slabs - s - DEPTH;          // 0 .. DEPTH - 1 slabs behind the ones in flight
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    multiply(d);
    if (d < rest) load(d, s + DEPTH + d);
  }
#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (d < rest) multiply(d);

  // The waves' sums meet in LDS, [wave][i][j][lane] with 16 bytes a lane; RI row blocks at a time, so that a workgroup
  // never asks for more than 64 KiB and a second one fits beside it (the launches of two nano-batches share the units).
  constexpr int RI = rows_per_round(MB, NB), ITEMS = RI * NB * 64;
  float vmax[2] = {0.0f, 0.0f};
  auto total = [&](int i, int j, int l) {
    const f32x4* at = reinterpret_cast<const f32x4*>(smem) + (i * NB + j) * 64 + l;
    f32x4 v = at[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += at[w * ITEMS];
    return v;
  };
  auto gather = [&](int i0) {
    f32x4* const mine = reinterpret_cast<f32x4*>(smem) + wave * ITEMS + lane;
#pragma unroll
    for (int i = 0; i < RI; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) mine[(i * NB + j) * 64] = acc[i0 + i][j];
    __syncthreads();
  };
  // W was the first operand: item (i, j, l) is row l % 16 of block i, columns 16 j + 4 (l / 16) .. + 3
  // (N % 8 == 0: a run of four columns is inside or outside)
  auto place = [&](int i, int j, int l, bool& other, int64_t& at) {
    int m = 16 * i + (l & 15);
    const int n = n0 + 16 * j + 4 * (l >> 4);
    other = MERGED && m >= second;
    m -= other ? second : 0;
    at = (int64_t)m * (other ? p.side[1].ldc : p.side[0].ldc) + n;
    return m < (other ? p.side[1].M : p.side[0].M) && n < p.N;
  };
  auto residual = [&](int i, int j, int l) {
    bool other;
    int64_t at;
    u32x2 r = {0, 0};
    if constexpr (!FP8 && !FUSED)
      if (p.side[0].R && place(i, j, l, other, at))
        r = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(other ? p.side[1].R : p.side[0].R) + at);
    return r;
  };
  auto finish = [&](int i, int j, int l, f32x4 v, f32x4 u, u32x2 r) {
    bool other;
    int64_t at;
    if (!place(i, j, l, other, at)) return;
    const int n = n0 + 16 * j + 4 * (l >> 4);
    const float sa = FP8 ? (other ? p.side[1].a_scale : p.side[0].a_scale)[0] : 1.0f;
    if (FP8) {
      const f32x4 ws = *reinterpret_cast<const f32x4*>(p.w_scale + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= sa * ws[e];
    }
    u32x2 o = {pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3])};
    if constexpr (FUSED) {
      if (FP8) {
        const f32x4 us = *reinterpret_cast<const f32x4*>(p.w2_scale + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] *= sa * us[e];
      }
      const u32x2 up = {pack2_bf16(u[0], u[1]), pack2_bf16(u[2], u[3])};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float lo = silu_fast(bf16_lo_to_f32(o[h])), hi = silu_fast(bf16_hi_to_f32(o[h]));
        if (!FP8) {                              // bf16: silu is rounded before the product
          const uint32_t s2 = pack2_bf16(lo, hi);
          lo = bf16_lo_to_f32(s2);
          hi = bf16_hi_to_f32(s2);
        }
        o[h] = pack2_bf16(lo * bf16_lo_to_f32(up[h]), hi * bf16_hi_to_f32(up[h]));
        if (FP8) {
          const float top = fmaxf(fabsf(bf16_lo_to_f32(o[h])), fabsf(bf16_hi_to_f32(o[h])));
          if (other) vmax[1] = fmaxf(vmax[1], top); else vmax[0] = fmaxf(vmax[0], top);
        }
      }
    } else if (!FP8 && p.side[0].R) {
      o[0] = add2_bf16(o[0], r[0]);
      o[1] = add2_bf16(o[1], r[1]);
    }
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(other ? p.side[1].C : p.side[0].C) + at) = o;
  };

  if constexpr (SPLIT) {
    // the parts of a tile meet in memory: each leaves its sums, the part that arrives last adds them in part order
    constexpr int BLOCK = MB * NB * 64 * 16;     // bytes of a part
    f32x4* const all = reinterpret_cast<f32x4*>(p.side[0].partials) + (int64_t)tile * p.split_k * (MB * NB * 64);
    f32x4* const block = all + (int64_t)part * (MB * NB * 64);
#pragma unroll
    for (int i0 = 0; i0 < MB; i0 += RI) {
      gather(i0);
#pragma unroll
      for (int item = 0; item < ITEMS; item += THREADS) {
        const int id = item + tid;
        if (ITEMS % THREADS == 0 || id < ITEMS)
          store_f32x4_device_coherent(block + i0 * NB * 64 + id, total((id >> 6) / NB, (id >> 6) % NB, id & 63));
      }
      __syncthreads();
    }
    wait_vmcnt<0>();
    __syncthreads();
    int* const ticket_cell = reinterpret_cast<int*>(smem);
    if (tid == 0) *ticket_cell = atomicAdd(p.side[0].arrivals + tile, 1);
    __syncthreads();
    if (*ticket_cell != p.split_k - 1) return;
    if (tid == 0) atomicExch(p.side[0].arrivals + tile, 0);
    const auto parts = coherent_blocks(all, p.split_k * BLOCK);
    // (items of a thread together: their loads take one latency, not one each; with the rows of a pair in as few blocks
    // as they need, 2 x 20 rows, 8B shapes: q/k/v 21.1 -> 19.1 us, o 16.5 -> 14.9, down 32.8 -> 30.6, gate + up 48 -> 45)
    constexpr int COUNT = MB * NB * 64, EACH = (COUNT + THREADS - 1) / THREADS, U = EACH < 4 ? EACH : 4;
    for (int id0 = tid; id0 < COUNT; id0 += U * THREADS) {
      f32x4 v[U];
      u32x2 r[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int id = id0 + u * THREADS < COUNT ? id0 + u * THREADS : id0;
        v[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        r[u] = residual((id >> 6) / NB, (id >> 6) % NB, id & 63);
      }
      for (int q0 = 0; q0 < p.split_k; q0 += 4) {
        f32x4 more[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int id = id0 + u * THREADS < COUNT ? id0 + u * THREADS : id0;
            const int q = q0 + c < p.split_k ? q0 + c : p.split_k - 1;
            more[u][c] = load_f32x4_device_coherent(parts, id * 16, q * BLOCK);
          }
        DFHIP_PIN;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (q0 + c < p.split_k) v[u] += more[u][c];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int id = id0 + u * THREADS;
        if (id < COUNT) finish((id >> 6) / NB, (id >> 6) % NB, id & 63, v[u], v[u], r[u]);
      }
    }
    return;
  }
#pragma unroll
  for (int i0 = 0; i0 < MB; i0 += RI) {
    constexpr int COUNT = RI * OB * 64, EACH = (COUNT + THREADS - 1) / THREADS;
    u32x2 r[EACH];                               // on their way while the sums meet
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
      const int item = tid + e * THREADS;
      r[e] = item < COUNT ? residual(i0 + (item >> 6) / OB, (item >> 6) % OB, item & 63) : u32x2{0, 0};
    }
    gather(i0);
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
      const int item = tid + e * THREADS;
      if (item >= COUNT) break;
      const int l = item & 63, i = (item >> 6) / OB, j = (item >> 6) % OB;
      const f32x4 v = total(i, j, l);
      finish(i0 + i, j, l, v, FUSED ? total(i, OB + j, l) : v, r[e]);
    }
    if (i0 + RI < MB) __syncthreads();
  }
  if constexpr (FP8 && FUSED) {
#pragma unroll
    for (int c = 0; c <= MERGED; ++c) fold_amax(p.side[c], tile, wave, wave_max(vmax[c]));
  }
}

constexpr int stream_lds(int mb, int nb) { return WAVES * rows_per_round(mb, nb) * nb * 1024; }
// Slabs in flight per wave: as many as 256 registers hold.  `width`: 16-column blocks of the output per workgroup.
constexpr int stream_depth(int mb, int width) { return width == 1 ? (mb == 4 ? 2 : 4) : width == 2 && mb == 1 ? 4 : 2; }

template <bool FP8, int MB, int WIDTH, bool FUSED, bool SPLIT, bool MERGED>
constexpr auto stream_kernel =
    gemm_stream_kernel<FP8, MB, (FUSED ? 2 : 1) * WIDTH, stream_depth(MB, WIDTH), FUSED, SPLIT, MERGED>;

template <bool FP8, int MB, int WIDTH, bool FUSED, bool SPLIT, bool MERGED>
int opt_in_stream() {
  constexpr int LDS = stream_lds(MB, (FUSED ? 2 : 1) * WIDTH);
  static std::atomic<uint64_t> lds_opted_in{0};
  return dfhip_opt_in_lds(reinterpret_cast<const void*>(stream_kernel<FP8, MB, WIDTH, FUSED, SPLIT, MERGED>), LDS, lds_opted_in);
}

// Two launches of up to 16 MB rows are one of the kernel with as many row blocks as the rows of both take, on the tiles (and
// with them the order of the sums) of the one.
template <bool FP8, int MB, int WIDTH, bool FUSED, bool SPLIT>
bool join_stream(const void* a, const void* b, dim3 ga, dim3 gb, void* both, DfhipJoined* joined) {
  if (!dfhip_same(ga, gb) || !sides_stream(a, b, both)) return false;
  const StreamArgs& p = *static_cast<const StreamArgs*>(both);
  constexpr int NB = (FUSED ? 2 : 1) * WIDTH;
  if (p.side[0].M + p.side[1].M > 16 * (2 * MB - 1)) {
    *joined = {reinterpret_cast<const void*>(stream_kernel<FP8, 2 * MB, WIDTH, FUSED, SPLIT, true>),
               (unsigned)stream_lds(2 * MB, NB), ga};
    return opt_in_stream<FP8, 2 * MB, WIDTH, FUSED, SPLIT, true>() == DFHIP_OK;
  }
  *joined = {reinterpret_cast<const void*>(stream_kernel<FP8, 2 * MB - 1, WIDTH, FUSED, SPLIT, true>),
             (unsigned)stream_lds(2 * MB - 1, NB), ga};
  return opt_in_stream<FP8, 2 * MB - 1, WIDTH, FUSED, SPLIT, true>() == DFHIP_OK;
}

template <bool FP8, int MB, int WIDTH, bool FUSED, bool SPLIT>
int launch(const StreamArgs& p, hipStream_t stream) {
  const auto kernel = stream_kernel<FP8, MB, WIDTH, FUSED, SPLIT, false>;
  if (int rc = opt_in_stream<FP8, MB, WIDTH, FUSED, SPLIT, false>()) return rc;
  if constexpr (MB <= 2) {
    static const bool known = (dfhip_pairable(reinterpret_cast<const void*>(kernel), join_stream<FP8, MB, WIDTH, FUSED, SPLIT>), true);
    (void)known;
  } else {
    DFHIP_NOT_IN_LINE(kernel);
  }
  constexpr int COLS = 16 * WIDTH;
  hipLaunchKernelGGL(kernel, dim3((p.N + COLS - 1) / COLS * p.split_k), dim3(WAVES * 64),
                     stream_lds(MB, (FUSED ? 2 : 1) * WIDTH), stream, p);
  return dfhip_check_launch();
}

// The smallest number of slabs a part of K may have: every wave has DEPTH of them (the largest depth is 4).
constexpr int MIN_SLABS = 4 * WAVES;

template <bool FP8, int MB, bool FUSED, bool SPLIT>
int launch_width(const StreamArgs& p, int width, hipStream_t stream) {
  switch (width) {
    case 1: return launch<FP8, MB, 1, FUSED, SPLIT>(p, stream);
    case 2: return launch<FP8, MB, 2, FUSED, SPLIT>(p, stream);
    default: return launch<FP8, MB, 4, FUSED, SPLIT>(p, stream);
  }
}

template <bool FP8, bool FUSED, bool SPLIT>
int launch_rows(const StreamArgs& p, int width, hipStream_t stream) {
  if (p.side[0].M <= 16) return launch_width<FP8, 1, FUSED, SPLIT>(p, width, stream);
  if (p.side[0].M <= 32) return launch_width<FP8, 2, FUSED, SPLIT>(p, width, stream);
  if constexpr (SPLIT || (!FP8 && FUSED)) return DFHIP_ERR_BAD_SHAPE;   // bf16: whole K alone, by variant
  else return launch_width<FP8, 4, FUSED, SPLIT>(p, width, stream);
}

// Columns per workgroup (in blocks of 16) when K is cut into `split_k` parts.  A wider tile re-reads the activations
// less often, but from about 160 workgroups on the launch also streams its weights at the full rate, and below that it
// does not: the widest tile that leaves 160.  [us, 8B shapes, weights from HBM: o 4096 x 4096 at 16 rows 9.7 with 256
// workgroups of 16 columns, 12.9 with 128 of 32; q/k/v 6144 x 4096 16.7 with 384 of 16, 13.3 with 192 of 32; gate +
// up + SiLU*mul 2 x 14336 x 4096 at 64 rows 88 / 64 / 49 with 16 / 32 / 64 outputs a workgroup]
int width_for(int N, int split_k) {
  for (int width = 4; width > 1; width /= 2)
    if ((int64_t)((N + 16 * width - 1) / (16 * width)) * split_k >= 160) return width;
  return 1;
}

template <bool FP8, bool FUSED>
int dispatch(const StreamArgs& p, hipStream_t stream) {
  const int width = width_for(p.N, p.split_k);
  if constexpr (!FUSED)
    if (p.split_k > 1) return launch_rows<FP8, FUSED, true>(p, width, stream);
  return launch_rows<FP8, FUSED, false>(p, width, stream);
}

}  // namespace

bool dfhip_stream_fits(int M, int N, int64_t k_bytes, int split_k) {
  return M <= DFHIP_STREAM_MAX_M && k_bytes % 128 == 0 && k_bytes / 128 / split_k >= MIN_SLABS &&
         (split_k == 1 || (N + 15) / 16 <= 1024);   // (arrival counters within the smallest counter area)
}

// Parts of K for a launch that may split.  Up to 16 rows a short K is not worth the meeting of the parts; with more
// rows two parts of twice the width are (the activations are re-read half as often), and a long K takes four: the
// partial sums weigh less against its weights.  [us: down 4096 x 14336 at 16 / 32 / 64 rows 27.7 / 40 / 65 unsplit
// with 16 columns a workgroup, 22.5 / 26.3 / 35.1 in four parts with 64; o 4096 x 4096 at 32 / 64 rows 13.1 / 20.5
// unsplit, 11.6 / 16.1 in two parts, 12.8 / 17.7 in four]
int dfhip_stream_split(int M, int N, int64_t k_bytes) {
  const int slabs = (int)(k_bytes / 128);
  const int most = slabs >= 128 ? 4 : M > 16 ? 2 : 1;
  for (int width = 4; width >= 1; width /= 2) {
    const int tiles = (N + 16 * width - 1) / (16 * width);
    int s = 256 / tiles;
    if (s > most) s = most;
    if (s < 1) s = 1;
    if (tiles * s >= 160) return dfhip_stream_fits(M, N, k_bytes, s) ? s : 1;
  }
  // narrow outputs: as many parts as fill the compute units, each with enough slabs to stream
  int s = 256 / ((N + 15) / 16);
  if (s > 8) s = 8;
  while (s > 1 && !dfhip_stream_fits(M, N, k_bytes, s)) --s;
  return s < 1 ? 1 : s;
}

int dfhip_stream_bf16(const void* A, int64_t lda, const void* W, int64_t ldw, const void* R, void* C, int64_t ldc, int M,
                      int N, int K, int split_k, void* partials, int* arrivals, hipStream_t stream) {
  const StreamArgs p{static_cast<const uint8_t*>(W), nullptr, nullptr, nullptr, N, K / 64, split_k, ldw * 2,
                     {{A, R, C, nullptr, nullptr, static_cast<float*>(partials), arrivals, lda * 2, ldc, M}, {}}};
  return dispatch<false, false>(p, stream);
}
int dfhip_stream_bf16_gate_up(const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, void* C, int64_t ldc,
                              int M, int N, int K, hipStream_t stream) {
  const StreamArgs p{static_cast<const uint8_t*>(W), static_cast<const uint8_t*>(W2), nullptr, nullptr, N, K / 64, 1, ldw * 2,
                     {{A, nullptr, C, nullptr, nullptr, nullptr, nullptr, lda * 2, ldc, M}, {}}};
  return dispatch<false, true>(p, stream);
}
int dfhip_stream_fp8(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, const float* a_scale,
                     const float* w_scale, int M, int N, int K, int split_k, void* partials, int* arrivals, hipStream_t stream) {
  const StreamArgs p{static_cast<const uint8_t*>(W), nullptr, w_scale, nullptr, N, K / 128, split_k, ldw,
                     {{A, nullptr, C, a_scale, nullptr, static_cast<float*>(partials), arrivals, lda, ldc, M}, {}}};
  return dispatch<true, false>(p, stream);
}
int dfhip_stream_fp8_gate_up(const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, void* C, int64_t ldc,
                             const float* a_scale, const float* w_scale, const float* w2_scale, float* amax, bool amax_apart,
                             int M, int N, int K, hipStream_t stream) {
  const StreamArgs p{static_cast<const uint8_t*>(W), static_cast<const uint8_t*>(W2), w_scale, w2_scale, N, K / 128, 1, ldw,
                     {{A, nullptr, C, a_scale, amax, nullptr, nullptr, lda, ldc, M, amax_apart}, {}}};
  return dispatch<true, true>(p, stream);
}
int dfhip_stream_blocks(int N) {
  const int cols = 16 * width_for(N, 1);
  return (N + cols - 1) / cols;
}
