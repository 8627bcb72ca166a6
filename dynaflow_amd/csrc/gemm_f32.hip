// fp32 GEMM for gfx950:  C[M,N] = A[M,K] * W[N,K]^T.
//
// gemm_f32_split_kernel (v_mfma_f32_16x16x4_f32, the kernel of the small fp32 configuration): a few 16 x 16 blocks of C
//   per workgroup so that a small product still has a workgroup for every compute unit; its four waves share the blocks
//   and take the 128-byte slabs of K in turn, operands go straight from memory (L2) to registers, and the four partial
//   sums meet in LDS.  Bound by the matrix pipes' fp32 rate and, at these sizes, by how evenly the blocks fall.
// gemm_f32_nt_kernel (v_mfma_f32_32x32x2_f32, any K that is a multiple of 4; many rows with a K up to about 3000): a
//   128x128 tile per workgroup, K walked in slabs of 16 through one LDS buffer.  LDS rows hold 16 floats padded to 17 so
//   that the 32 lanes of a fragment read (one float each, rows 17 words apart) hit 32 different banks.
#include "dfhip_pairs.h"

namespace {

constexpr int FBM = 128, FBN = 128, FBK = 16, FROW = FBK + 1, FTHREADS = 256;

__global__ void __launch_bounds__(FTHREADS)
gemm_f32_nt_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M,
                   int N, int K, int64_t lda, int64_t ldw, int64_t ldc) {
  __shared__ float a_lds[FBM * FROW];
  __shared__ float w_lds[FBN * FROW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wave_m = wave & 1, wave_n = wave >> 1;  // 2 x 2 waves, 64 x 64 each
  const int m0 = blockIdx.y * FBM, n0 = blockIdx.x * FBN;

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int frag_row = lane & 31, frag_k = lane >> 5;
  for (int k0 = 0; k0 < K; k0 += FBK) {
    // 128 rows x 4 float4 chunks per operand = 512 chunks, 2 per thread
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int idx = tid + p * FTHREADS;
      const int r = idx >> 2, c = (idx & 3) * 4;
      int ar = m0 + r; ar = ar < M ? ar : M - 1;
      int wr = n0 + r; wr = wr < N ? wr : N - 1;
      f32x4 av = {0.f, 0.f, 0.f, 0.f}, wv = {0.f, 0.f, 0.f, 0.f};
      if (k0 + c < K) {  // K % 4 == 0: a chunk is entirely inside or outside
        av = *reinterpret_cast<const f32x4*>(A + (int64_t)ar * lda + k0 + c);
        wv = *reinterpret_cast<const f32x4*>(W + (int64_t)wr * ldw + k0 + c);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a_lds[r * FROW + c + e] = av[e];
        w_lds[r * FROW + c + e] = wv[e];
      }
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < FBK / 2; ++ks) {
      float fa[2], fw[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = a_lds[(wave_m * 64 + i * 32 + frag_row) * FROW + ks * 2 + frag_k];
#pragma unroll
      for (int j = 0; j < 2; ++j) fw[j] = w_lds[(wave_n * 64 + j * 32 + frag_row) * FROW + ks * 2 + frag_k];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fw[j], fa[i], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }

  // W was the first MFMA operand: a lane holds row m = lane%32 and 4-wide runs of n
  const int m_lane = m0 + wave_m * 64 + frag_row;
  const int n_lane = n0 + wave_n * 64 + frag_k * 4;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m_lane + i * 32;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = n_lane + j * 32 + g * 8 + e;
          if (n < N) C[(int64_t)m * ldc + n] = acc[i][j][4 * g + e];
        }
  }
}

// A tile of MB x NB blocks of 16 x 16.  A lane multiplies eight floats of a row's slab of 32, four of each load; an MFMA takes element e
// of load h of both operands, so eight MFMAs cover the slab (each sums its own four of the floats: the same order of k for both
// operands is all that matters).
// PAIRS: neighbouring lanes load 32 bytes of a row and exchange pieces (deal_neighbours: floats 8 (lane / 16) + 4 h + e).  With a row per lane
// (floats 16 h + 4 (lane / 16) + e) a compute unit takes in 34 GB/s, which was the time of most launches; with pairs of lanes 66.  The
// exchange costs as much as a tenth of the products of 4 x 4 blocks, and registers: several workgroups on a compute unit hide the
// loads anyway.  [us, a row per lane -> pairs, alone / in pairs: 128 x 1024 x 2816 17.3 / 30.2 -> 13.7 / 20.1, 128 x 2816 x 1024 12.6 / 20.0 -> 12.1
// / 17.9, 64 x 2048 x 5632 31.7 / 59.0 -> 24.2 / 37.6, 256 x 2816 x 1024 18.1 / 37.9 -> 18.1 / 29.9; one round of 4 x 4 and 4 x 3 blocks, not taken alone: 512 x 2048
// x 5632 87 / 274 -> 98 / 196, 128 x 5632 x 2048 30.5 / 69.5 -> 31.6 / 57.0; four slabs in flight, not taken: 1000 x 2048 x 5632 178 / 353 -> 202 / 400, 256 x 5632 x 2048 62 / 116 -> 64 / 117]
constexpr int SWAVES = 4;

template <int MB, int NB, int SDEPTH, bool PAIRS>
__global__ void __launch_bounds__(SWAVES * 64)
gemm_f32_split_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N,
                      int slabs, int64_t lda, int64_t ldw, int64_t ldc, int tiles_m) {
  __shared__ f32x4 sums[SWAVES * MB * NB * 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = lane & (PAIRS ? 14 : 15), chunk = PAIRS ? 2 * (lane >> 4) + (lane & 1) : lane >> 4;
  constexpr int ROW_H = PAIRS ? 1 : 0, CHUNK_H = PAIRS ? 0 : 4;  // of load 1 behind load 0
  const int m0 = (int)(blockIdx.x % tiles_m) * (16 * MB), n0 = (int)(blockIdx.x / tiles_m) * (16 * NB);
  const float* a_ptr[MB][2];
  const float* w_ptr[NB][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      int m = m0 + 16 * i + row + ROW_H * h; m = m < M ? m : M - 1;  // rows past the edge re-read the last one; never stored
      a_ptr[i][h] = A + (int64_t)m * lda + wave * 32 + (chunk + CHUNK_H * h) * 4;
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      int n = n0 + 16 * j + row + ROW_H * h; n = n < N ? n : N - 1;
      w_ptr[j][h] = W + (int64_t)n * ldw + wave * 32 + (chunk + CHUNK_H * h) * 4;
    }
  }
  const int n_slabs = (slabs - wave + SWAVES - 1) / SWAVES;   // >= SDEPTH (checked by the launch)

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  u32x4 af[SDEPTH][MB][2], wf[SDEPTH][NB][2];
  auto load = [&](int d, int s) {
    const int off = s * (SWAVES * 32);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < MB; ++i) af[d][i][h] = *reinterpret_cast<const u32x4*>(a_ptr[i][h] + off);
#pragma unroll
      for (int j = 0; j < NB; ++j) wf[d][j][h] = *reinterpret_cast<const u32x4*>(w_ptr[j][h] + off);
    }
  };
  auto multiply = [&](int d) {
    if constexpr (PAIRS) {
#pragma unroll
      for (int i = 0; i < MB; ++i) deal_neighbours(af[d][i][0], af[d][i][1]);
#pragma unroll
      for (int j = 0; j < NB; ++j) deal_neighbours(wf[d][j][0], wf[d][j][1]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wf[d][j][h][e]), __uint_as_float(af[d][i][h][e]),
                                                             acc[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int d = 0; d < SDEPTH; ++d) load(d, d);
  int s = 0;
  for (; s + 2 * SDEPTH <= n_slabs; s += SDEPTH) {
#pragma unroll
    for (int d = 0; d < SDEPTH; ++d) {
      multiply(d);
      load(d, s + SDEPTH + d);
      DFHIP_PIN;
    }
  }
  const int rest = n_slabs - s - SDEPTH;                      // 0 .. SDEPTH - 1
#pragma unroll
  for (int d = 0; d < SDEPTH; ++d) {
    multiply(d);
    if (d < rest) load(d, s + SDEPTH + d);
  }
#pragma unroll
  for (int d = 0; d < SDEPTH - 1; ++d)
    if (d < rest) multiply(d);

#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) sums[((wave * MB + i) * NB + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  // W was the first operand: item (i, j, l) is row 16 i + l % 16, columns 16 j + 4 (l / 16) .. + 3
  const bool whole = ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15u) == 0;
  for (int item = tid; item < MB * NB * 64; item += SWAVES * 64) {
    f32x4 v = sums[item];
#pragma unroll
    for (int w = 1; w < SWAVES; ++w) v += sums[w * (MB * NB * 64) + item];
    const int l = item & 63, i = (item >> 6) / NB, j = (item >> 6) % NB;
    const int m = m0 + 16 * i + (l & 15), n = n0 + 16 * j + 4 * (l >> 4);
    if (m >= M) continue;
    float* c = C + (int64_t)m * ldc + n;
    if (whole && n + 4 <= N) {
      *reinterpret_cast<f32x4*>(c) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) c[e] = v[e];
    }
  }
}

struct F32Args {
  const float *A, *W;
  float* C;
  int M, N, K;
  int64_t lda, ldw, ldc;
};

int64_t split_tiles(const F32Args& p, int mb, int nb) {
  return (int64_t)((p.M + 16 * mb - 1) / (16 * mb)) * ((p.N + 16 * nb - 1) / (16 * nb));
}

template <int MB, int NB, int DEPTH, bool PAIRS>
int launch_split(const F32Args& p, hipStream_t stream) {
  const auto kernel = gemm_f32_split_kernel<MB, NB, DEPTH, PAIRS>;
  DFHIP_NOT_IN_LINE(kernel);
  hipLaunchKernelGGL(kernel, dim3((unsigned)split_tiles(p, MB, NB)), dim3(SWAVES * 64), 0,
                     stream, p.A, p.W, p.C, p.M, p.N, p.K / 32, p.lda, p.ldw, p.ldc, (p.M + 16 * MB - 1) / (16 * MB));
  return dfhip_check_launch();
}
// Two slabs in flight per wave while the tiles fit one round of workgroups, four beyond that (several workgroups follow
// each other on a compute unit and their loads cost more than their registers: 256 x 5632 x 2048 77 -> 62 us, 1024 x 2048
// x 5632 264 -> 178, but 256 x 2816 x 1024, one round, 18 -> 20).
template <int MB, int NB>
int launch_deep(const F32Args& p, int share, hipStream_t stream) {
  if (p.K >= 512 && split_tiles(p, MB, NB) > 256) return launch_split<MB, NB, 4, false>(p, stream);
  if (MB * NB >= 12 && share == 1) return launch_split<MB, NB, 2, false>(p, stream);
  return launch_split<MB, NB, 2, true>(p, stream);
}

// Smallest tile for which a wave's share of K has two slabs in flight.
constexpr int SPLIT_MIN_K = 32 * SWAVES * 2;

int launch_tile128(const F32Args& p, hipStream_t stream) {
  dim3 grid((p.N + FBN - 1) / FBN, (p.M + FBM - 1) / FBM);
  DFHIP_NOT_IN_LINE(gemm_f32_nt_kernel);
  hipLaunchKernelGGL(gemm_f32_nt_kernel, grid, dim3(FTHREADS), 0, stream, p.A, p.W, p.C, p.M, p.N, p.K, p.lda, p.ldw, p.ldc);
  return dfhip_check_launch();
}

// The split tile that takes the least: one round of 256 workgroups costs its blocks and about 1.5 blocks' worth of start,
// loads and meeting; of several rounds, whose workgroups overlap, each costs 0.6 of its blocks and of seven more for the
// operands (per round at K = 2048: 4 x 4 blocks 37 us, 4 x 3 31, 4 x 2 25).  [us with a row per lane, at [128 x 1024] x [2816 x 1024]^T /
// [128 x 2816] x [1024 x 2816]^T, with the workgroups in parentheses: 2 x 3 blocks 12.4 (236) / 27.5 (88), 4 x 2 14.9 (176) /
// 32.7 (64), 2 x 2 17.2 (352) / 22.2 (128), 2 x 1 18.4 (704) / 16.9 (256); the 128 x 128 tiles 105 (22) / 274 (8).  Floor at
// the fp32 rate: 4.9.]  These prices and those below were fitted with a row per lane, and not again since lanes pair up: of 54 launches
// (16 .. 1000 rows of six weights) the one chosen takes 1.7 % more than the fastest, of 54 pairs 3.9 %; it is 5 % off and more in 20 of
// these, most of several rounds, where 4 x 3 and 4 x 4 blocks are taken and 2 x 2 would be faster (1000 x 2816 x 1024 69 / 60, pairs of
// 1000 x 1408 x 512 56 / 44), and in a pair of 1000 x 5632 x 2048, on 128 x 128 tiles 581 / 422.
// Many rows and a K up to about 3000 keep the 128 x 128 tiles, which read their operands half as often: both are priced
// in us, fitted to about 190 launches (0.5 * 10^9 .. 10^12 flops, K = 288 .. 14336, alone and in pairs), the 128 x 128
// tiles by their rounds (of all launches side by side: they fill each other's units).  [us, 128 x 128 / split: 8192 x 2816
// x 512 250 / 319, 8192 x 5632 x 1024 801 / 978, 8192 x 5632 x 2048 1511 / 1623, 8192 x 4096 x 4096 2133 / 2123; a pair of
// 3000 x 2816 x 1024 337 / 402, of 1500 x 2816 x 512 126 / 140]
int launch_f32(const F32Args& p, int share, hipStream_t stream) {
  constexpr int SHAPES[8][2] = {{4, 4}, {4, 3}, {4, 2}, {2, 3}, {2, 2}, {2, 1}, {1, 2}, {1, 1}};
  int best = 0;
  double least = 0.0;
  for (int i = 0; i < 8; ++i) {
    const int64_t rounds = (split_tiles(p, SHAPES[i][0], SHAPES[i][1]) + 255) / 256;
    const int blocks = SHAPES[i][0] * SHAPES[i][1];
    const double cost = rounds == 1 ? blocks + 1.5 : 0.6 * (double)rounds * (blocks + 7);
    if (i == 0 || cost < least) { best = i; least = cost; }
  }
  const double k = p.K / 1024.0;
  const int64_t tiles128 = (int64_t)((p.M + FBM - 1) / FBM) * ((p.N + FBN - 1) / FBN);
  const double rounds128 = (double)((tiles128 * share + 255) / 256);
  const bool fits = (p.M + FBM - 1) / FBM <= 65535;          // (the rows are the grid's second dimension)
  if (fits && k * (45.0 + 58.0 * rounds128) + 8.0 * rounds128 < 1.06 * share * least * (0.52 + 1.06 * k))
    return launch_tile128(p, stream);
  switch (best) {
    case 0: return launch_deep<4, 4>(p, share, stream);
    case 1: return launch_deep<4, 3>(p, share, stream);
    case 2: return launch_deep<4, 2>(p, share, stream);
    case 3: return launch_split<2, 3, 2, true>(p, stream);
    case 4: return launch_split<2, 2, 2, true>(p, stream);
    case 5: return launch_split<2, 1, 2, true>(p, stream);
    case 6: return launch_split<1, 2, 2, true>(p, stream);
    default: return launch_split<1, 1, 2, true>(p, stream);
  }
}

}  // namespace

extern "C" int dfhip_gemm_f32_nt_shared(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
                                        int M, int N, int K, int share, dfhip_stream_t stream) {
  if (!A || !W || !C) return DFHIP_ERR_NULL_POINTER;
  if (M < 1 || N < 1 || K < 1 || K % 4 != 0) return DFHIP_ERR_BAD_SHAPE;
  if (lda < K || ldw < K || ldc < N) return DFHIP_ERR_BAD_STRIDE;
  if (lda % 4 || ldw % 4 || !dfhip_aligned16(A) || !dfhip_aligned16(W) ||
      (reinterpret_cast<uintptr_t>(C) & 3u))
    return DFHIP_ERR_BAD_ALIGNMENT;
  if (share < 1 || share > 16) return DFHIP_ERR_BAD_ARGUMENT;
  const F32Args p{static_cast<const float*>(A), static_cast<const float*>(W), static_cast<float*>(C), M, N, K, lda, ldw, ldc};
  if (K % 32 == 0 && K >= SPLIT_MIN_K) return launch_f32(p, share, static_cast<hipStream_t>(stream));
  return launch_tile128(p, static_cast<hipStream_t>(stream));
}

extern "C" int dfhip_gemm_f32_nt(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
                                 int M, int N, int K, dfhip_stream_t stream) {
  return dfhip_gemm_f32_nt_shared(A, lda, W, ldw, C, ldc, M, N, K, 1, stream);
}
