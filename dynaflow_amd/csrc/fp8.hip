// fp8 (OCP e4m3fn) path: per-tensor dynamic quantisation, SiLU*mul with amax,
// and the fp8 GEMM  C = bf16(a_scale * w_scale[n] * A[M,K] * W[N,K]^T).
//
// The GEMMs have the byte geometry of the bf16 ones (a K slab row is 128 bytes, here
// 128 fp8 values) and multiply with the scaled fp8 MFMAs (scale exponents fixed at 2^0):
// v_mfma_scale_f32_16x16x128_f8f6f4 in the ring kernels, ..._32x32x64_... in the
// register-staged one - twice the bf16 rate.  A lane feeds 32 consecutive bytes of one
// row; both operands use the same lane->k mapping, so the contraction is exact whatever
// order the hardware walks those bytes in.
//
// gemm_fp8_ring_kernel  256x256 tile, the LDS-DMA ring / pinned-schedule design of the
//                       bf16 ring kernel: five 32 KiB LDS units, 1.5 slabs in flight,
//                       XOR-swizzled 128-byte rows, one LDS read or DMA issue behind every
//                       MFMA, barrier between the two column halves of a slab, staged epilogue.
//                       Forms with 192 and 128 rows for launches of few rows (TM: 16-row blocks per wave), and
//                       with K cut into parts for few tiles: [350 x 28672] x [8192 x 28672]^T ran on 64 workgroups
//                       (230 us, 0.71 PFLOP/s), with 192 rows and four parts it takes 96.
// gemm_fp8_nt_kernel    register-staged double buffer, 128 x 128: an independent second kernel, by variant only.
#include "dfhip_pairs.h"
#include "dfhip_ring3.h"
#include "dfhip_stream.h"

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));

constexpr float FP8_MAX = 448.0f;
constexpr int QT = 256;      // threads of the elementwise fp8 kernels
constexpr int QUNROLL = 4;

DFHIP_DEVICE float silu_f32(float g) { return silu_fast(g); }   // one formula for every bf16 path

DFHIP_DEVICE void atomic_max_nonneg(float* cell, float v) {
  // non-negative floats order like their bit patterns
  atomicMax(reinterpret_cast<unsigned int*>(cell), __float_as_uint(v));
}

DFHIP_DEVICE void block_max_to(float* cell, float v) {
  __shared__ float partial[QT / 64];
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    float m = partial[0];
#pragma unroll
    for (int w = 1; w < QT / 64; ++w) m = fmaxf(m, partial[w]);
    atomic_max_nonneg(cell, m);
  }
}

// amax[0] = max(amax[0], max |x|) over a row-strided bf16 matrix; group = 8 values
__global__ void __launch_bounds__(QT)
absmax_bf16_kernel(const uint16_t* __restrict__ x, int64_t ld, uint32_t groups, uint32_t per_row,
                   float* __restrict__ amax) {
  float m = 0.0f;
  for (uint32_t gi = blockIdx.x * QT + threadIdx.x; gi < groups; gi += gridDim.x * QT) {
    const uint32_t row = gi / per_row, col = (gi - row * per_row) * 8;
    const u32x4 v = *reinterpret_cast<const u32x4*>(x + (int64_t)row * ld + col);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      m = fmaxf(m, fabsf(bf16_bits_to_f32(v[w] & 0xffffu)));
      m = fmaxf(m, fabsf(__uint_as_float(v[w] & 0xffff0000u)));
    }
  }
  block_max_to(amax, m);
}

DFHIP_DEVICE uint32_t quant4(float a, float b, float c, float d, float scale) {
  a = fminf(fmaxf(a / scale, -FP8_MAX), FP8_MAX);
  b = fminf(fmaxf(b / scale, -FP8_MAX), FP8_MAX);
  c = fminf(fmaxf(c / scale, -FP8_MAX), FP8_MAX);
  d = fminf(fmaxf(d / scale, -FP8_MAX), FP8_MAX);
  uint32_t r = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);  // bytes 0,1
  r = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, r, true);            // bytes 2,3
  return r;
}

// out = bf16(silu(g) * u) (optional store) and amax over the rounded values
__global__ void __launch_bounds__(QT)
silu_mul_absmax_kernel(const uint16_t* __restrict__ gate, int64_t ld_gate, const uint16_t* __restrict__ up,
                       int64_t ld_up, uint16_t* __restrict__ out, int64_t ld_out, uint32_t groups,
                       uint32_t per_row, float* __restrict__ amax) {
  float m = 0.0f;
  for (uint32_t gi = blockIdx.x * QT + threadIdx.x; gi < groups; gi += gridDim.x * QT) {
    const uint32_t row = gi / per_row, col = (gi - row * per_row) * 8;
    const u32x4 g = *reinterpret_cast<const u32x4*>(gate + (int64_t)row * ld_gate + col);
    const u32x4 u = *reinterpret_cast<const u32x4*>(up + (int64_t)row * ld_up + col);
    u32x4 o;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float lo = silu_f32(bf16_bits_to_f32(g[w] & 0xffffu)) * bf16_bits_to_f32(u[w] & 0xffffu);
      const float hi = silu_f32(__uint_as_float(g[w] & 0xffff0000u)) * __uint_as_float(u[w] & 0xffff0000u);
      o[w] = pack2_bf16(lo, hi);
      m = fmaxf(m, fabsf(bf16_bits_to_f32(o[w] & 0xffffu)));
      m = fmaxf(m, fabsf(__uint_as_float(o[w] & 0xffff0000u)));
    }
    if (out != nullptr) *reinterpret_cast<u32x4*>(out + (int64_t)row * ld_out + col) = o;
  }
  block_max_to(amax, m);
}

// ---- quantisation without a cell that has to be cleared first: the blocks leave their maxima in `parts`, and every block
// of the launch that quantises takes the maximum of those
constexpr int QPARTS = DFHIP_FP8_PARTS;          // blocks at most

// (address of group gi; without a gap between rows no division)
template <bool FLAT>
DFHIP_DEVICE int64_t group_at(uint32_t gi, uint32_t per_row, int64_t ld) {
  if (FLAT) return (int64_t)gi * 8;
  const uint32_t row = gi / per_row;
  return (int64_t)row * ld + (gi - row * per_row) * 8;
}
DFHIP_DEVICE float absmax8(u32x4 v) {
  float m = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; ++w) m = fmaxf(m, fmaxf(fabsf(bf16_lo_to_f32(v[w])), fabsf(bf16_hi_to_f32(v[w]))));
  return m;
}
DFHIP_DEVICE u32x2 quant8(u32x4 v, float scale) {
  return u32x2{quant4(bf16_lo_to_f32(v[0]), bf16_hi_to_f32(v[0]), bf16_lo_to_f32(v[1]), bf16_hi_to_f32(v[1]), scale),
               quant4(bf16_lo_to_f32(v[2]), bf16_hi_to_f32(v[2]), bf16_lo_to_f32(v[3]), bf16_hi_to_f32(v[3]), scale)};
}
// the block's maximum, in every thread
template <int THREADS>
DFHIP_DEVICE float block_max(float v) {
  __shared__ float partial[THREADS / 64];
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = v;
  __syncthreads();
  v = partial[0];
#pragma unroll
  for (int w = 1; w < THREADS / 64; ++w) v = fmaxf(v, partial[w]);
  return v;
}

// parts[block] = max |x| of the groups of the block; with `up`, x is first replaced by bf16(silu(x) * up), which is stored.
// Bound: HBM, or up to some MB the launch.  QUNROLL groups of a thread are loaded before the first is used, and no atomics
// queue up at one address (12 ns each): with the quantisation behind it and no launch to clear a cell, x of 12 / 350 / 2048 x
// 8192 7.6 / 12.8 / 41.6 -> 5.6 / 8.2 / 19.5 us, SiLU*mul of 350 / 2048 x 28672 32 / 106 -> 23 / 91.
template <bool FLAT, bool SILU>
DFHIP_DEVICE void absmax_part(unsigned block, unsigned blocks, const uint16_t* __restrict__ x, int64_t ld,
                              const uint16_t* __restrict__ up, int64_t ld_up, uint16_t* __restrict__ out, int64_t ld_out,
                              uint32_t groups, uint32_t per_row, float* __restrict__ parts) {
  float m = 0.0f;
  for (uint32_t g0 = block * (QT * QUNROLL) + threadIdx.x; g0 < groups; g0 += blocks * (QT * QUNROLL)) {
    u32x4 v[QUNROLL], u[QUNROLL];
#pragma unroll
    for (int k = 0; k < QUNROLL; ++k) {
      const uint32_t gi = g0 + k * QT < groups ? g0 + k * QT : g0;
      v[k] = *reinterpret_cast<const u32x4*>(x + group_at<FLAT>(gi, per_row, ld));
      if (SILU) u[k] = *reinterpret_cast<const u32x4*>(up + group_at<FLAT>(gi, per_row, ld_up));
    }
    DFHIP_PIN;
#pragma unroll
    for (int k = 0; k < QUNROLL; ++k) {
      if (SILU) {
#pragma unroll
        for (int w = 0; w < 4; ++w)
          v[k][w] = pack2_bf16(silu_f32(bf16_lo_to_f32(v[k][w])) * bf16_lo_to_f32(u[k][w]),
                               silu_f32(bf16_hi_to_f32(v[k][w])) * bf16_hi_to_f32(u[k][w]));
        if (g0 + k * QT < groups)
          *reinterpret_cast<u32x4*>(out + group_at<FLAT>(g0 + k * QT, per_row, ld_out)) = v[k];
      }
      m = fmaxf(m, absmax8(v[k]));               // (a group past the end repeats the first one)
    }
  }
  m = block_max<QT>(m);
  if (threadIdx.x == 0) parts[block] = m;
}
template <bool FLAT, bool SILU>
struct AbsmaxParts {
  static constexpr int THREADS = QT;
  const uint16_t* x;
  const uint16_t* up;
  uint16_t* out;
  float* parts;
  int64_t ld, ld_up, ld_out;
  uint32_t groups, per_row;
  DFHIP_DEVICE void run(unsigned block, unsigned blocks) const {
    absmax_part<FLAT, SILU>(block, blocks, x, ld, up, ld_up, out, ld_out, groups, per_row, parts);
  }
  bool beside(const AbsmaxParts& other) const { return parts != other.parts && (!SILU || out != other.out); }
};
template <bool FLAT, bool SILU>
__global__ void __launch_bounds__(QT) absmax_parts_kernel(const AbsmaxParts<FLAT, SILU> p) { p.run(blockIdx.x, gridDim.x); }

// q = e4m3fn(x / scale), scale = max(amax, 1e-12) / 448.  PARTS: amax is the maximum of n_parts values; else `amax` is one
// value, and with `readers` the last block to have read it clears it and the count of those that have: the cells are zero
// again for the launch that folds the next maximum into them.  The parts of a turn are asked for together.  [us, both launches, one load
// of a part after the other / together: 12 x 8192 5.7 / 5.6, 350 x 8192 7.7 / 7.3, 700 x 8192 9.5 / 8.9]
template <bool FLAT, bool PARTS>
DFHIP_DEVICE void quant_after(unsigned block, unsigned blocks, const uint16_t* __restrict__ x, int64_t ld,
                              uint8_t* __restrict__ q, int64_t ld_q, uint32_t groups, uint32_t per_row,
                              float* __restrict__ amax, int n_parts, int* __restrict__ readers,
                              float* __restrict__ scale_out) {
  const uint32_t step = blocks * (QT * QUNROLL);
  uint32_t g0 = block * (QT * QUNROLL) + threadIdx.x;
  u32x4 v[QUNROLL];
  auto load = [&]() {
#pragma unroll
    for (int k = 0; k < QUNROLL; ++k) {
      const uint32_t gi = g0 + k * QT < groups ? g0 + k * QT : groups - 1;
      v[k] = *reinterpret_cast<const u32x4*>(x + group_at<FLAT>(gi, per_row, ld));
    }
    DFHIP_PIN;
  };
  load();
  float m = 0.0f;
  if (PARTS) {
    for (int p0 = threadIdx.x; p0 < n_parts; p0 += QPARTS) {
      float part[QPARTS / QT];
#pragma unroll
      for (int p = 0; p < QPARTS / QT; ++p) part[p] = amax[p0 + p * QT < n_parts ? p0 + p * QT : p0];
      DFHIP_PIN;
#pragma unroll
      for (int p = 0; p < QPARTS / QT; ++p) m = fmaxf(m, part[p]);
    }
    m = block_max<QT>(m);
  } else {
    __shared__ float cell;
    if (threadIdx.x == 0) cell = __hip_atomic_load(amax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    m = cell;
    if (readers && threadIdx.x == 0 && atomicAdd(readers, 1) == (int)blocks - 1) {
      __hip_atomic_store(amax, 0.0f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(readers, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  const float scale = fmaxf(m, 1e-12f) / FP8_MAX;
  if (block == 0 && threadIdx.x == 0 && scale_out != nullptr) scale_out[0] = scale;
  while (g0 < groups) {
#pragma unroll
    for (int k = 0; k < QUNROLL; ++k)
      if (g0 + k * QT < groups)
        *reinterpret_cast<u32x2*>(q + group_at<FLAT>(g0 + k * QT, per_row, ld_q)) = quant8(v[k], scale);
    g0 += step;
    if (g0 < groups) load();
  }
}
template <bool FLAT, bool PARTS>
struct QuantAfter {
  static constexpr int THREADS = QT;
  const uint16_t* x;
  uint8_t* q;
  float* amax;
  int* readers;
  float* scale_out;
  int64_t ld, ld_q;
  uint32_t groups, per_row;
  int n_parts;
  DFHIP_DEVICE void run(unsigned block, unsigned blocks) const {
    quant_after<FLAT, PARTS>(block, blocks, x, ld, q, ld_q, groups, per_row, amax, n_parts, readers, scale_out);
  }
  bool beside(const QuantAfter& other) const {
    return q != other.q && amax != other.amax && (!scale_out || scale_out != other.scale_out);
  }
};
template <bool FLAT, bool PARTS>
__global__ void __launch_bounds__(QT) quant_fp8_after_kernel(const QuantAfter<FLAT, PARTS> p) { p.run(blockIdx.x, gridDim.x); }

template <bool FLAT, bool SILU>
int launch_absmax_parts(const AbsmaxParts<FLAT, SILU>& args, unsigned blocks, hipStream_t stream) {
  const auto kernel = absmax_parts_kernel<FLAT, SILU>;
  static const bool known = (dfhip_pairable(reinterpret_cast<const void*>(kernel), dfhip_join_beside<AbsmaxParts<FLAT, SILU>>,
                                            DFHIP_SHORT_BLOCKS), true);
  (void)known;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(QT), 0, stream, args);
  return dfhip_check_launch();
}
template <bool FLAT, bool PARTS>
int launch_quant_after(const QuantAfter<FLAT, PARTS>& args, unsigned blocks, hipStream_t stream) {
  const auto kernel = quant_fp8_after_kernel<FLAT, PARTS>;
  static const bool known = (dfhip_pairable(reinterpret_cast<const void*>(kernel), dfhip_join_beside<QuantAfter<FLAT, PARTS>>,
                                            DFHIP_SHORT_BLOCKS), true);
  (void)known;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(QT), 0, stream, args);
  return dfhip_check_launch();
}

// ------------------------------------------------------------------ fp8 GEMM
constexpr int FBK = 128;            // fp8 values (= bytes) per slab row
constexpr int FROW = FBK + 16;      // padded LDS row in bytes
constexpr int FCHUNKS = FBK / 16;   // 16-byte chunks per slab row

template <int BM, int BN>
__global__ void __launch_bounds__(256)
gemm_fp8_nt_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ W, uint16_t* __restrict__ C,
                   const float* __restrict__ a_scale, const float* __restrict__ w_scale, int M, int N, int K,
                   int64_t lda, int64_t ldw, int64_t ldc, int tiles_m, int tiles_n) {
  constexpr int THREADS = 256;
  constexpr int WTM = BM / 2, WTN = BN / 2, TM = WTM / 32, TN = WTN / 32;
  constexpr int A_LOADS = BM * FCHUNKS / THREADS, W_LOADS = BN * FCHUNKS / THREADS;
  constexpr int ROWS_PER_PASS = THREADS / FCHUNKS;
  constexpr int BUF_BYTES = (BM + BN) * FROW;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wave_m = wave & 1, wave_n = wave >> 1;
  const int tile = remap_xcd(blockIdx.x, tiles_m * tiles_n);
  const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;

  const int ld_row = tid / FCHUNKS, ld_chunk = tid % FCHUNKS;
  const uint8_t* a_src[A_LOADS];
  const uint8_t* w_src[W_LOADS];
#pragma unroll
  for (int p = 0; p < A_LOADS; ++p) {
    int row = m0 + ld_row + p * ROWS_PER_PASS;
    row = row < M ? row : M - 1;
    a_src[p] = A + (int64_t)row * lda + ld_chunk * 16;
  }
#pragma unroll
  for (int p = 0; p < W_LOADS; ++p) {
    int row = n0 + ld_row + p * ROWS_PER_PASS;
    row = row < N ? row : N - 1;
    w_src[p] = W + (int64_t)row * ldw + ld_chunk * 16;
  }
  u32x4 a_reg[A_LOADS], w_reg[W_LOADS];
  auto fetch = [&](int kt) {
#pragma unroll
    for (int p = 0; p < A_LOADS; ++p) a_reg[p] = *reinterpret_cast<const u32x4*>(a_src[p] + kt * FBK);
#pragma unroll
    for (int p = 0; p < W_LOADS; ++p) w_reg[p] = *reinterpret_cast<const u32x4*>(w_src[p] + kt * FBK);
  };
  auto park = [&](int buf) {
    uint8_t* a_dst = smem + buf * BUF_BYTES + ld_row * FROW + ld_chunk * 16;
    uint8_t* w_dst = a_dst + BM * FROW;
#pragma unroll
    for (int p = 0; p < A_LOADS; ++p) *reinterpret_cast<u32x4*>(a_dst + p * ROWS_PER_PASS * FROW) = a_reg[p];
#pragma unroll
    for (int p = 0; p < W_LOADS; ++p) *reinterpret_cast<u32x4*>(w_dst + p * ROWS_PER_PASS * FROW) = w_reg[p];
  };

  // lane reads 32 consecutive bytes: row lane%32, byte offset 64*ks + 32*(lane/32)
  const int frag_row = lane & 31, frag_half = lane >> 5;
  const int a_frag_off = (wave_m * WTM + frag_row) * FROW + frag_half * 32;
  const int w_frag_off = BM * FROW + (wave_n * WTN + frag_row) * FROW + frag_half * 32;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int KT = K / FBK;
  fetch(0);
  park(0);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < KT) fetch(kt + 1);
    const uint8_t* base = smem + buf * BUF_BYTES;
#pragma unroll
    for (int ks = 0; ks < FBK / 64; ++ks) {
      i32x8 fa[TM], fw[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(base + a_frag_off + i * 32 * FROW + ks * 64);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(base + a_frag_off + i * 32 * FROW + ks * 64 + 16);
        fa[i] = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(base + w_frag_off + j * 32 * FROW + ks * 64);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(base + w_frag_off + j * 32 * FROW + ks * 64 + 16);
        fw[j] = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fw[j], fa[i], acc[i][j], 0, 0, 0, 0x7f7f7f7f,
                                                                     0, 0x7f7f7f7f);
    }
    if (kt + 1 < KT) park(buf ^ 1);
    __syncthreads();
  }

  // W was the first operand: lane holds row m = lane%32, columns 8g + 4*(lane/32) + 0..3
  const float sa = a_scale[0];
  const int m_lane = m0 + wave_m * WTM + frag_row;
  const int n_lane = n0 + wave_n * WTN + frag_half * 4;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m_lane + i * 32;
    if (m >= M) continue;
    uint16_t* c_row = C + (int64_t)m * ldc;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = n_lane + j * 32 + g * 8;
        if (n < N) {
          const f32x4 ws = *reinterpret_cast<const f32x4*>(w_scale + n);
          u32x2 v;
          v[0] = pack2_bf16(acc[i][j][4 * g + 0] * (sa * ws[0]), acc[i][j][4 * g + 1] * (sa * ws[1]));
          v[1] = pack2_bf16(acc[i][j][4 * g + 2] * (sa * ws[2]), acc[i][j][4 * g + 3] * (sa * ws[3]));
          *reinterpret_cast<u32x2*>(c_row + n) = v;
        }
      }
  }
}


// ------------------------------------------------------------------ fp8 ring kernel
constexpr int F8_UNIT = 32768, F8_NUNITS = 5, F8_RING_LDS = F8_UNIT * F8_NUNITS;
constexpr int F8_GROUP_M = 4, F8_EROW = 272;

// FUSED: the W half of a slab holds 128 rows of W (gate) and the matching 128 rows of W2 (up); the tile
// then is 256 x 128 outputs, N counts those, and the epilogue writes act = bf16(silu(bf16 g) * bf16 u) -
// the roundings of the separate GEMMs and of silu_mul_absmax_kernel, so the same bits - and folds
// max |act| into amax[0].
template <bool FUSED, int TM, bool SPLIT>
__global__ void __launch_bounds__(256)
gemm_fp8_ring_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ W, const uint8_t* __restrict__ W2,
                     uint16_t* __restrict__ C, const float* __restrict__ a_scale, const float* __restrict__ w_scale,
                     const float* __restrict__ w2_scale, float* __restrict__ amax, int M, int N, int K, int64_t lda,
                     int64_t ldw, int64_t ldc, int tiles_m, int tiles_n, int split_k, float* __restrict__ partials,
                     int* __restrict__ arrivals) {
  static_assert(!(FUSED && SPLIT), "the fused form keeps K whole");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m = wave & 1, wave_n = wave >> 1;
  constexpr int TILE_M = 32 * TM;              // rows of a tile: two wave rows of TM blocks of 16
  constexpr int TILE_N = FUSED ? 128 : 256;    // output columns of a tile
  constexpr int MQ = 4 * TM;                   // MFMAs of a column half

  int tile, part = 0;
  if (SPLIT) splitk_work_of(blockIdx.x, tiles_m * tiles_n, tile, part);
  else tile = remap_xcd(blockIdx.x, tiles_m * tiles_n);
  const int per_panel = F8_GROUP_M * tiles_n;
  const int first_m = (tile / per_panel) * F8_GROUP_M;
  const int rows_in_panel = (tiles_m - first_m) < F8_GROUP_M ? (tiles_m - first_m) : F8_GROUP_M;
  const int in_panel = tile % per_panel;
  const int m0 = (first_m + in_panel % rows_in_panel) * TILE_M;
  const int n0 = (in_panel / rows_in_panel) * TILE_N;
  const int slabs = K / FBK;
  const int slab0 = SPLIT ? (int)((int64_t)slabs * part / split_k) : 0;
  const int KT = SPLIT ? (int)((int64_t)slabs * (part + 1) / split_k) - slab0 : slabs;

  // DMA addresses: a wave-uniform tile base (scalar registers, advanced per slab) plus a 32-bit byte
  // offset per lane.  FUSED: rows 0..127 of the W half come from W (waves 0, 1), rows 128..255 from W2.
  uint32_t a_off[TM], w_off[8];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int row = (wave * TM + t) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    int ar = m0 + row; ar = ar < M ? ar : M - 1;
    a_off[t] = (uint32_t)((int64_t)(ar - m0) * lda + chunk * 16);
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int row = (wave * 8 + t) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    int wr = n0 + (FUSED ? (row & 127) : row); wr = wr < N ? wr : N - 1;
    w_off[t] = (uint32_t)((int64_t)(wr - n0) * ldw + chunk * 16);
  }
  const uint8_t* const a_tile = A + (int64_t)m0 * lda + (int64_t)slab0 * FBK;
  const uint8_t* const w_tile = ((FUSED && wave >= 2) ? W2 : W) + (int64_t)n0 * ldw + (int64_t)slab0 * FBK;
  auto dma_a = [&](int t, int slab, int unit) {
    const int s = slab < KT ? slab : KT - 1;
    dma16_base(unit * F8_UNIT + (wave * TM + t) * 1024, a_tile + (int64_t)s * FBK, a_off[t]);
  };
  auto dma_w = [&](int t, int slab, int unit) {
    const int s = slab < KT ? slab : KT - 1;
    dma16_base(unit * F8_UNIT + (wave * 8 + t) * 1024, w_tile + (int64_t)s * FBK, w_off[t]);
  };

  // v_mfma_scale_f32_16x16x128_f8f6f4: one instruction covers the 128 bytes of k of a slab.  A fragment of a
  // 16-row block is 32 bytes per lane = chunks 2*(lane/16) and 2*(lane/16) + 1 of row lane%16, swizzled by
  // (row/2)%8.  acc[i][j] (W block j first operand, A block i second): lane holds
  // C[16 i + lane%16][16 j + 4 (lane/16) + r], r = 0..3.
  const int frow = lane & 15, fquad = lane >> 4, fswz = (frow >> 1) & 7;
  int koff[2];
#pragma unroll
  for (int part = 0; part < 2; ++part) koff[part] = ((2 * fquad + part) ^ fswz) * 16;
  const int a_lane = (wave_m * (16 * TM) + frow) * 128, w_lane = (wave_n * 128 + frow) * 128;

  f32x4 acc[TM][8];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

#pragma unroll
  for (int t = 0; t < TM; ++t) dma_a(t, 0, 0);
#pragma unroll
  for (int t = 0; t < 8; ++t) dma_w(t, 0, 1);
#pragma unroll
  for (int t = 0; t < TM; ++t) dma_a(t, 1, 2);
#pragma unroll
  for (int t = 0; t < 8; ++t) dma_w(t, 1, 3);
  wait_vmcnt<8 + TM>();
  workgroup_barrier();

  // A whole slab of fragments is 128 registers per operand; both operands double-buffered would not fit.
  // The slab is multiplied in two column halves instead: W blocks 0..3 (fwa), then W blocks 4..7 (fwb), both
  // against all TM A blocks.  The A blocks are double-buffered across slabs, each W half is read while the
  // other one is in use.
  u32x4 fa[2][TM][2], fwa[4][2], fwb[4][2];   // [..][block][low / high 16 bytes]
  auto read_a = [&](int half_idx, int slot, int unit_a) {   // half_idx 0..2 TM - 1: block half_idx/2, low / high half
    const int blk = half_idx >> 1, part = half_idx & 1;
    fa[slot][blk][part] = *reinterpret_cast<const u32x4*>(smem + unit_a * F8_UNIT + a_lane + koff[part] + blk * 2048);
  };
  auto read_w = [&](int half_idx, bool second, int unit_w) {   // half_idx 0..7 within the column half
    const int blk = half_idx >> 1, part = half_idx & 1;
    const u32x4 v = *reinterpret_cast<const u32x4*>(smem + unit_w * F8_UNIT + w_lane + koff[part] + ((second ? 4 : 0) + blk) * 2048);
    if (second) fwb[blk][part] = v; else fwa[blk][part] = v;
  };
  const int unit_scale = 0x7f7f7f7f;   // e8m0 scales 2^0
  auto mfma = [&](int q, int slot, bool second) {   // snake over TM A blocks x 4 W blocks
    const int i = q >> 2, jj = (i & 1) ? 3 - (q & 3) : (q & 3);
    const u32x4 (&w)[2] = second ? fwb[jj] : fwa[jj];
    const i32x8 av = {(int)fa[slot][i][0][0], (int)fa[slot][i][0][1], (int)fa[slot][i][0][2], (int)fa[slot][i][0][3],
                      (int)fa[slot][i][1][0], (int)fa[slot][i][1][1], (int)fa[slot][i][1][2], (int)fa[slot][i][1][3]};
    const i32x8 wv = {(int)w[0][0], (int)w[0][1], (int)w[0][2], (int)w[0][3], (int)w[1][0], (int)w[1][1], (int)w[1][2], (int)w[1][3]};
    // written out so that the accumulator keeps its registers
    asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %3 op_sel_hi:[0,0,0]"
                 : "+a"(acc[i][second ? 4 + jj : jj]) : "v"(wv), "v"(av), "v"(unit_scale));
  };
  // reads of the next slab in the order its first MFMAs need them: W block 0, A block 0, W blocks 1..3, then the other A blocks
  auto read_next = [&](int pos, int slot, int unit_a, int unit_w) {   // pos 0..READS - 1 (fragment halves)
    if (pos < 2) read_w(pos, false, unit_w);
    else if (pos < 4) read_a(pos - 2, slot, unit_a);
    else if (pos < 10) read_w(pos - 2, false, unit_w);
    else read_a(pos - 8, slot, unit_a);
  };

  constexpr int READS = 8 + 2 * TM;
  int ua = 0, uw = 1, ia = 4, iw = 0;
#pragma unroll
  for (int pos = 0; pos < READS; ++pos) read_next(pos, 0, ua, uw);
  // one slab; `sl` (0 / 1, a constant at each call) is the A fragment buffer this slab multiplies from
  auto slab = [&](int kt, int sl) {
    // first column half: the fragments of W blocks 4..7 behind MFMAs 0..7, the DMA of A(kt+2) behind every
    // other MFMA after that
#pragma unroll
    for (int q = 0; q < MQ; ++q) {
      mfma(q, sl, false);
      if (q < 8) read_w(q, true, uw);
      else if (q % 2 == 0 && q < 8 + 2 * TM) dma_a((q - 8) / 2, kt + 2, ia);
      DFHIP_PIN;
    }
    // every LDS read of slab kt has been issued; slab kt+1 must have landed, only A(kt+2) may be in flight
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    wait_vmcnt<TM>();
    workgroup_barrier();
    int na = ua + 2; if (na >= F8_NUNITS) na -= F8_NUNITS;
    int nw = uw + 2; if (nw >= F8_NUNITS) nw -= F8_NUNITS;
    // second column half: the DMA of W(kt+2) behind every other MFMA, the fragment halves of slab kt+1 (all of A,
    // W blocks 0..3) behind the others.  256 rows: one operation behind every MFMA; shorter tiles have fewer MFMAs
    // than operations and some carry two.
    constexpr int OPS = 8 + READS;
#pragma unroll
    for (int q = 0; q < MQ; ++q) {
      mfma(q, sl, true);
#pragma unroll
      for (int op = q * OPS / MQ; op < (q + 1) * OPS / MQ; ++op) {
        if (op < 16) { if (op % 2 == 0) dma_w(op / 2, kt + 2, iw); else read_next(op / 2, sl ^ 1, na, nw); }
        else read_next(8 + (op - 16), sl ^ 1, na, nw);
      }
      DFHIP_PIN;
    }
    ua = na; uw = nw;
    ia += 2; if (ia >= F8_NUNITS) ia -= F8_NUNITS;
    iw += 2; if (iw >= F8_NUNITS) iw -= F8_NUNITS;
  };
  int kt = 0;
  for (; kt + 1 < KT; kt += 2) {
    slab(kt, 0);
    slab(kt + 1, 1);
  }
  if (kt < KT) slab(kt, 0);
  wait_vmcnt<0>();
  workgroup_barrier();
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMAs have written their accumulators
  // (the compiler does not know that the statements above write the accumulators late: every later use
  // of an accumulator is tied behind the wait states)
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(acc[i][j]));

  if constexpr (SPLIT) {
    // Every part leaves its fp32 block in `partials` and takes a ticket; the part that comes last adds the blocks in
    // part order (its own too: the same bits whoever is last) and writes the tile.  Nobody waits.
    constexpr int BLOCK = TM * 8 * 256;
    f32x4* const blocks = reinterpret_cast<f32x4*>(partials) + (int64_t)tile * split_k * BLOCK;
    f32x4* const mine = blocks + part * BLOCK + tid;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) store_f32x4_device_coherent(mine + (i * 8 + j) * 256, acc[i][j]);
    wait_vmcnt<0>();
    __syncthreads();
    int* const ticket_cell = reinterpret_cast<int*>(smem);
    if (tid == 0) *ticket_cell = atomicAdd(arrivals + tile, 1);
    __syncthreads();
    const int ticket = *ticket_cell;
    if (ticket != split_k - 1) return;
    if (tid == 0) atomicExch(arrivals + tile, 0);     // counters are left at zero
    __syncthreads();                                  // the ticket has been read before the tile is parked over it
    const auto left = coherent_blocks(blocks, split_k * BLOCK * 16);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int p = 0; p < split_k; ++p) {
      const int base = p * (BLOCK * 16);
#pragma unroll
      for (int i = 0; i < TM; i += 2) {             // 16 loads in flight before the first is used
        f32x4 v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j)
          v[j] = load_f32x4_device_coherent(left, tid * 16, base + (i * 8 + j) * 4096);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          f32x4& sum = acc[i + j / 8][j % 8];
          sum += v[j];
          asm volatile("" : "+a"(sum));             // back to its accumulation registers
        }
      }
    }
  }

  // scale, round to bf16, park the wave's block in LDS, store whole 256-byte row pieces
  const float sa = a_scale[0];
  uint8_t* park = smem + wave * (128 * F8_EROW);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    int n = n0 + (FUSED ? 0 : wave_n * 128) + j * 16 + fquad * 4;
    n = n < N ? n : N - 4;   // columns past the edge are never stored; keep the scale load in bounds
    const f32x4 ws = *reinterpret_cast<const f32x4*>((FUSED && wave_n ? w2_scale : w_scale) + n);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      u32x2 v;
      v[0] = pack2_bf16(acc[i][j][0] * (sa * ws[0]), acc[i][j][1] * (sa * ws[1]));
      v[1] = pack2_bf16(acc[i][j][2] * (sa * ws[2]), acc[i][j][3] * (sa * ws[3]));
      *reinterpret_cast<u32x2*>(park + (i * 16 + frow) * F8_EROW + (j * 16 + fquad * 4) * 2) = v;
    }
  }
  DFHIP_PIN;
  if (FUSED) {
    // gate blocks sit in the parks of waves 0, 1 (the two halves of the rows), up blocks in those of waves 2, 3;
    // wave w combines half (w >> 1) of the rows of park w & 1
    __syncthreads();
    const uint8_t* gpark = smem + (wave & 1) * (128 * F8_EROW);
    const uint8_t* upark = smem + ((wave & 1) + 2) * (128 * F8_EROW);
    const int row0 = (wave >> 1) * (8 * TM);
    float vmax = 0.0f;
#pragma unroll 4
    for (int p = 0; p < 2 * TM; ++p) {
      const int id = p * 64 + lane;
      const int row = row0 + (id >> 4), c = id & 15;
      const u32x4 gv = *reinterpret_cast<const u32x4*>(gpark + row * F8_EROW + c * 16);
      const u32x4 uv = *reinterpret_cast<const u32x4*>(upark + row * F8_EROW + c * 16);
      u32x4 o;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float lo = silu_f32(bf16_bits_to_f32(gv[w] & 0xffffu)) * bf16_bits_to_f32(uv[w] & 0xffffu);
        const float hi = silu_f32(__uint_as_float(gv[w] & 0xffff0000u)) * __uint_as_float(uv[w] & 0xffff0000u);
        o[w] = pack2_bf16(lo, hi);
      }
      const int m = m0 + (wave & 1) * (16 * TM) + row, n = n0 + c * 8;
      if (m < M && n < N) {
        *reinterpret_cast<u32x4*>(C + (int64_t)m * ldc + n) = o;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          vmax = fmaxf(vmax, fabsf(bf16_bits_to_f32(o[w] & 0xffffu)));
          vmax = fmaxf(vmax, fabsf(__uint_as_float(o[w] & 0xffff0000u)));
        }
      }
    }
    vmax = wave_max(vmax);
    if (lane == 0) atomic_max_nonneg(amax, vmax);
    return;
  }
  const int m_base = m0 + wave_m * (16 * TM), n_base = n0 + wave_n * 128;
#pragma unroll 4
  for (int p = 0; p < 4 * TM; ++p) {
    const int id = p * 64 + lane;
    const int row = id >> 4, c = id & 15;
    const u32x4 v = *reinterpret_cast<const u32x4*>(park + row * F8_EROW + c * 16);
    const int m = m_base + row, n = n_base + c * 8;
    if (m < M && n < N) *reinterpret_cast<u32x4*>(C + (int64_t)m * ldc + n) = v;
  }
}

template <int TM, bool SPLIT>
int launch_fp8_ring(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
                    const float* a_scale, const float* w_scale, int M, int N, int K, int split_k, void* workspace,
                    hipStream_t stream) {
  auto kernel = gemm_fp8_ring_kernel<false, TM, SPLIT>;
  static std::atomic<uint64_t> lds_opted_in{0};   // per instantiation, one bit per device
  if (int rc = dfhip_opt_in_lds(reinterpret_cast<const void*>(kernel), F8_RING_LDS, lds_opted_in)) return rc;
  DFHIP_NOT_IN_LINE(kernel);
  const int tiles_m = (M + 32 * TM - 1) / (32 * TM), tiles_n = (N + 255) / 256;
  float* partials = nullptr;
  if (SPLIT) {
    const size_t tiles = (size_t)tiles_m * tiles_n;
    if (int rc = dfhip_clear_uncommon_counters(workspace, tiles, stream)) return rc;
    partials = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + dfhip_counter_area(tiles));
  }
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n * split_k), dim3(256), F8_RING_LDS, stream,
                     static_cast<const uint8_t*>(A), static_cast<const uint8_t*>(W), nullptr,
                     static_cast<uint16_t*>(C), a_scale, w_scale, nullptr, nullptr, M, N, K, lda, ldw, ldc, tiles_m,
                     tiles_n, split_k, partials, static_cast<int*>(workspace));
  return dfhip_check_launch();
}

template <int TM>
int launch_fp8_ring_fused(const void* A, int64_t lda, const void* Wg, const void* Wu, int64_t ldw, void* act,
                          int64_t ld_act, const float* a_scale, const float* wg_scale, const float* wu_scale,
                          float* amax, int M, int I, int K, hipStream_t stream) {
  auto kernel = gemm_fp8_ring_kernel<true, TM, false>;
  static std::atomic<uint64_t> lds_opted_in{0};   // per instantiation, one bit per device
  if (int rc = dfhip_opt_in_lds(reinterpret_cast<const void*>(kernel), F8_RING_LDS, lds_opted_in)) return rc;
  DFHIP_NOT_IN_LINE(kernel);
  const int tiles_m = (M + 32 * TM - 1) / (32 * TM), tiles_n = (I + 127) / 128;
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n), dim3(256), F8_RING_LDS, stream,
                     static_cast<const uint8_t*>(A), static_cast<const uint8_t*>(Wg), static_cast<const uint8_t*>(Wu),
                     static_cast<uint16_t*>(act), a_scale, wg_scale, wu_scale, amax, M, I, K, lda, ldw, ld_act,
                     tiles_m, tiles_n, 1, nullptr, nullptr);
  return dfhip_check_launch();
}


// ------------------------------------------------------------------ fp8 ring kernel, 256 x 224 tile
// The same ring with 4 waves stacked along M, each 64 x 224 = 4 x 14 MFMA blocks: column counts of
// the form 7 * 2^k (28672 = 128 * 224) then fill the rounds of 256 workgroups exactly.
constexpr int F8_TBN = 224, F8_TROW = F8_TBN * 2 + 16;

__global__ void __launch_bounds__(256)
gemm_fp8_ring224_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ W, uint16_t* __restrict__ C,
                        const float* __restrict__ a_scale, const float* __restrict__ w_scale, int M, int N, int K,
                        int64_t lda, int64_t ldw, int64_t ldc, int tiles_m, int tiles_n) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const int tile = remap_xcd(blockIdx.x, tiles_m * tiles_n);
  const int per_panel = F8_GROUP_M * tiles_n;
  const int first_m = (tile / per_panel) * F8_GROUP_M;
  const int rows_in_panel = (tiles_m - first_m) < F8_GROUP_M ? (tiles_m - first_m) : F8_GROUP_M;
  const int in_panel = tile % per_panel;
  const int m0 = (first_m + in_panel % rows_in_panel) * 256;
  const int n0 = (in_panel / rows_in_panel) * F8_TBN;
  const int KT = K / FBK;

  uint32_t a_off[8], w_off[7];   // byte offsets from the tile's first row; the tile base sits in scalar registers
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int row = (wave * 8 + t) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    int ar = m0 + row; ar = ar < M ? ar : M - 1;
    a_off[t] = (uint32_t)((int64_t)(ar - m0) * lda + chunk * 16);
  }
#pragma unroll
  for (int t = 0; t < 7; ++t) {
    const int row = (wave * 7 + t) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    int wr = n0 + row; wr = wr < N ? wr : N - 1;
    w_off[t] = (uint32_t)((int64_t)(wr - n0) * ldw + chunk * 16);
  }
  const uint8_t* const a_tile = A + (int64_t)m0 * lda;
  const uint8_t* const w_tile = W + (int64_t)n0 * ldw;
  auto dma_a = [&](int t, int slab, int unit) {
    const int s = slab < KT ? slab : KT - 1;
    dma16_base(unit * F8_UNIT + (wave * 8 + t) * 1024, a_tile + (int64_t)s * FBK, a_off[t]);
  };
  auto dma_w = [&](int t, int slab, int unit) {
    const int s = slab < KT ? slab : KT - 1;
    dma16_base(unit * F8_UNIT + (wave * 7 + t) * 1024, w_tile + (int64_t)s * FBK, w_off[t]);
  };

  // fragments and accumulators as in gemm_fp8_ring_kernel (16x16x128 instruction); the slab is multiplied in
  // two column halves of 7 W blocks against the wave's 4 A blocks
  const int frow = lane & 15, fquad = lane >> 4, fswz = (frow >> 1) & 7;
  int koff[2];
#pragma unroll
  for (int part = 0; part < 2; ++part) koff[part] = ((2 * fquad + part) ^ fswz) * 16;
  const int a_lane = (wave * 64 + frow) * 128, w_lane = frow * 128;

  f32x4 acc[4][14];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 14; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

#pragma unroll
  for (int t = 0; t < 8; ++t) dma_a(t, 0, 0);
#pragma unroll
  for (int t = 0; t < 7; ++t) dma_w(t, 0, 1);
#pragma unroll
  for (int t = 0; t < 8; ++t) dma_a(t, 1, 2);
#pragma unroll
  for (int t = 0; t < 7; ++t) dma_w(t, 1, 3);
  wait_vmcnt<15>();
  workgroup_barrier();

  u32x4 fa[2][4][2], fwa[7][2], fwb[7][2];   // [..][block][low / high 16 bytes]
  auto read_a = [&](int half_idx, int slot, int unit_a) {
    const int blk = half_idx >> 1, part = half_idx & 1;
    fa[slot][blk][part] = *reinterpret_cast<const u32x4*>(smem + unit_a * F8_UNIT + a_lane + koff[part] + blk * 2048);
  };
  auto read_w = [&](int half_idx, bool second, int unit_w) {   // half_idx 0..13 within the column half
    const int blk = half_idx >> 1, part = half_idx & 1;
    const u32x4 v = *reinterpret_cast<const u32x4*>(smem + unit_w * F8_UNIT + w_lane + koff[part] + ((second ? 7 : 0) + blk) * 2048);
    if (second) fwb[blk][part] = v; else fwa[blk][part] = v;
  };
  const int unit_scale = 0x7f7f7f7f;   // e8m0 scales 2^0
  auto mfma = [&](int q, int slot, bool second) {   // snake over 4 A blocks x 7 W blocks
    const int i = q / 7, jj = (i & 1) ? 6 - q % 7 : q % 7;
    const u32x4 (&w)[2] = second ? fwb[jj] : fwa[jj];
    const i32x8 av = {(int)fa[slot][i][0][0], (int)fa[slot][i][0][1], (int)fa[slot][i][0][2], (int)fa[slot][i][0][3],
                      (int)fa[slot][i][1][0], (int)fa[slot][i][1][1], (int)fa[slot][i][1][2], (int)fa[slot][i][1][3]};
    const i32x8 wv = {(int)w[0][0], (int)w[0][1], (int)w[0][2], (int)w[0][3], (int)w[1][0], (int)w[1][1], (int)w[1][2], (int)w[1][3]};
    asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %3 op_sel_hi:[0,0,0]"
                 : "+a"(acc[i][second ? 7 + jj : jj]) : "v"(wv), "v"(av), "v"(unit_scale));
  };
  // reads of the next slab in the order its first MFMAs need them: W block 0, A block 0, W blocks 1..6, A 1..3
  auto read_next = [&](int pos, int slot, int unit_a, int unit_w) {   // pos 0..21 (fragment halves)
    if (pos < 2) read_w(pos, false, unit_w);
    else if (pos < 4) read_a(pos - 2, slot, unit_a);
    else if (pos < 16) read_w(pos - 2, false, unit_w);
    else read_a(pos - 14, slot, unit_a);
  };

  int ua = 0, uw = 1, ia = 4, iw = 0;
#pragma unroll
  for (int pos = 0; pos < 22; ++pos) read_next(pos, 0, ua, uw);
  auto slab = [&](int kt, int sl) {
    // first column half: the 14 fragment halves of W blocks 7..13 and the 8 DMA instructions of A(kt+2)
#pragma unroll
    for (int q = 0; q < 28; ++q) {
      mfma(q, sl, false);
      if (q < 14) read_w(q, true, uw);
      if (q % 2 == 1 && q < 16) dma_a(q / 2, kt + 2, ia);
      DFHIP_PIN;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    wait_vmcnt<8>();
    workgroup_barrier();
    int na = ua + 2; if (na >= F8_NUNITS) na -= F8_NUNITS;
    int nw = uw + 2; if (nw >= F8_NUNITS) nw -= F8_NUNITS;
    // second column half: the 7 DMA instructions of W(kt+2), then the 22 fragment halves of slab kt+1
#pragma unroll
    for (int q = 0; q < 28; ++q) {
      mfma(q, sl, true);
      if (q % 2 == 0 && q < 14) dma_w(q / 2, kt + 2, iw);
      if (q >= 6) read_next(q - 6, sl ^ 1, na, nw);
      DFHIP_PIN;
    }
    ua = na; uw = nw;
    ia += 2; if (ia >= F8_NUNITS) ia -= F8_NUNITS;
    iw += 2; if (iw >= F8_NUNITS) iw -= F8_NUNITS;
  };
  int kt = 0;
  for (; kt + 1 < KT; kt += 2) {
    slab(kt, 0);
    slab(kt + 1, 1);
  }
  if (kt < KT) slab(kt, 0);
  wait_vmcnt<0>();
  workgroup_barrier();
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMAs have written their accumulators
  // (the compiler does not know that the statements above write the accumulators late: every later use
  // of an accumulator is tied behind the wait states)
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 14; ++j) asm volatile("" : "+a"(acc[i][j]));

  const float sa = a_scale[0];
  uint8_t* park = smem + wave * (64 * F8_TROW);
#pragma unroll
  for (int j = 0; j < 14; ++j) {
    int n = n0 + j * 16 + fquad * 4;
    n = n < N ? n : N - 4;
    const f32x4 ws = *reinterpret_cast<const f32x4*>(w_scale + n);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u32x2 v;
      v[0] = pack2_bf16(acc[i][j][0] * (sa * ws[0]), acc[i][j][1] * (sa * ws[1]));
      v[1] = pack2_bf16(acc[i][j][2] * (sa * ws[2]), acc[i][j][3] * (sa * ws[3]));
      *reinterpret_cast<u32x2*>(park + (i * 16 + frow) * F8_TROW + (j * 16 + fquad * 4) * 2) = v;
    }
  }
  DFHIP_PIN;
  const int m_base = m0 + wave * 64;
#pragma unroll 4
  for (int p = 0; p < 28; ++p) {
    const int id = p * 64 + lane;
    const int row = id / 28, c = id - row * 28;
    const u32x4 v = *reinterpret_cast<const u32x4*>(park + row * F8_TROW + c * 16);
    const int m = m_base + row, n = n0 + c * 8;
    if (m < M && n < N) *reinterpret_cast<u32x4*>(C + (int64_t)m * ldc + n) = v;
  }
}

int launch_fp8_ring224(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
                       const float* a_scale, const float* w_scale, int M, int N, int K, hipStream_t stream) {
  static std::atomic<uint64_t> lds_opted_in{0};   // per instantiation, one bit per device
  if (int rc = dfhip_opt_in_lds(reinterpret_cast<const void*>(gemm_fp8_ring224_kernel), F8_RING_LDS, lds_opted_in)) return rc;
  DFHIP_NOT_IN_LINE(gemm_fp8_ring224_kernel);
  const int tiles_m = (M + 255) / 256, tiles_n = (N + F8_TBN - 1) / F8_TBN;
  hipLaunchKernelGGL(gemm_fp8_ring224_kernel, dim3(tiles_m * tiles_n), dim3(256), F8_RING_LDS, stream,
                     static_cast<const uint8_t*>(A), static_cast<const uint8_t*>(W), static_cast<uint16_t*>(C),
                     a_scale, w_scale, M, N, K, lda, ldw, ldc, tiles_m, tiles_n);
  return dfhip_check_launch();
}

template <int BM, int BN>
int launch_fp8(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, const float* a_scale,
               const float* w_scale, int M, int N, int K, hipStream_t stream) {
  constexpr int LDS_BYTES = 2 * (BM + BN) * FROW;
  auto kernel = gemm_fp8_nt_kernel<BM, BN>;
  static std::atomic<uint64_t> lds_opted_in{0};   // per instantiation, one bit per device
  if (int rc = dfhip_opt_in_lds(reinterpret_cast<const void*>(kernel), LDS_BYTES, lds_opted_in)) return rc;
  DFHIP_NOT_IN_LINE(kernel);
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n), dim3(256), LDS_BYTES, stream, static_cast<const uint8_t*>(A),
                     static_cast<const uint8_t*>(W), static_cast<uint16_t*>(C), a_scale, w_scale, M, N, K, lda, ldw,
                     ldc, tiles_m, tiles_n);
  return dfhip_check_launch();
}

constexpr int F8_MAX_SPLIT = 16;
constexpr int F8_STREAM = 8;          // the streaming kernel with K in parts, as a variant (up to 32 rows)

// 16-row blocks per wave of a ring tile (256 columns), 0 for the other kernels
int ring_blocks(int variant) { return variant == 0 ? 8 : variant == 3 ? 6 : variant == 4 ? 4 : 0; }

struct TilePlan { int variant, split_k; double cost; };

// What one launch (or `share` of one shape side by side) costs in us: rounds of 256 workgroups, each the slabs of a
// part at the kernel's time per slab and a fixed start and end, plus the hand-over of the fp32 blocks of a split, whose
// reader takes split_k blocks one after the other.  A shorter tile is hardly faster per slab (the loads bound it), so
// it pays where it saves a round or leaves tiles to split; the 224-column kernel enters with a rate of its own.  The
// register-staged 128 x 128 kernel is never faster than the 128-row ring (17 .. 300 rows, 256 .. 8192 columns and K: 6
// against 6 us at the smallest, 51 against 40 at K = 8192).  The prices are good to about 15 %: 8192 x 28672 takes seven
// parts up to 128 rows, 77 us, where eight take 64.
double tile_cost(int64_t tiles, int split_k, int share, int K, double per_slab, int tm) {
  const double rounds = (double)((tiles * split_k * share + 255) / 256);
  return rounds * ((double)(K / FBK) / split_k * per_slab + 6.0) + (split_k > 1 ? 0.9 * tm * split_k + 4.0 : 0.0);
}
struct RingTile { int variant, tm; double per_slab; };
constexpr RingTile F8_RINGS[3] = {{0, 8, 1.07}, {3, 6, 0.97}, {4, 4, 0.85}};

// The tile shape and the parts of K.  K is only cut where the caller allows it, for the projection back to the model
// width, and where K > N: few tiles and a long K (8192 x 28672, us at 128 / 350 / 1024 rows: 245 / 236 / 242 before,
// 78 / 90 / 183 now).  At least eight slabs a part.
TilePlan plan_tile(int M, int N, int K, int share, bool may_split) {
  TilePlan best{2, 1, tile_cost((int64_t)((M + 255) / 256) * ((N + F8_TBN - 1) / F8_TBN), 1, share, K, 1.0, 0)};
  for (const RingTile& ring : F8_RINGS) {
    const int64_t tiles = (int64_t)((M + 32 * ring.tm - 1) / (32 * ring.tm)) * ((N + 255) / 256);
    for (int s = 1; s <= F8_MAX_SPLIT; ++s) {
      if (s > 1 && (!may_split || K <= N || K / FBK < 8 * s || tiles * s * share > 256)) break;
      const TilePlan plan{ring.variant, s, tile_cost(tiles, s, share, K, ring.per_slab, ring.tm)};
      if (plan.cost < best.cost) best = plan;
    }
  }
  return best;
}

// Prices of the ring kernels as those of the three-slab tiles (dfhip_ring3.h), by variant.
constexpr DfhipPrice F8_RING_PRICE[3] = {{0.774, 0.642, 7.45, 17.5, 2.35, 5.6}, {0.100, 1.010, 8.73, 5.24, 2.14, 5.6},
                                         {0.566, 0.620, 2.00, 1.00, 1.96, 6.01}};   // of F8_RINGS
constexpr DfhipPrice F8_RING224_PRICE = {0.861, 0.401, 8.58, 0.0, 0.0, 6.0};

// Whether a three-slab tile takes the place of the planned kernel, and which: where it is 4 % cheaper, 7 % above 256 rows and
// for gate + up, whose pairs above 128 rows need 15 % (192 rows of 2 x 28672 x 8192 in pairs, priced 8 % lower, took 228 us
// on 224 x 192 tiles where the 192-row ones take 195).  At 25 counts of rows of six
// weights (those of dfhip_price), alone and in pairs, 136 launches change their kernel: 19 % less on the geometric mean, at best 49 %
// (33 x 4096 x 14336 alone: 40 -> 20.5 us), at worst 7 % more (350 x 4096 x 16384 alone: 42 -> 45), the only one that stays above 3 %
// in every run.
DfhipRing3Plan three_slabs_cheaper(bool gate_up, int M, int N, int K, int share, int variant, int split_k, bool may_split) {
  const int tm = ring_blocks(variant);
  const int rows = tm ? 32 * tm : 256, cols = !tm ? F8_TBN : gate_up ? 128 : 256;
  const DfhipPrice& price = tm == 8 ? F8_RING_PRICE[0] : tm == 6 ? F8_RING_PRICE[1] : tm == 4 ? F8_RING_PRICE[2]
                                                                                            : F8_RING224_PRICE;
  const int64_t tiles = (int64_t)((M + rows - 1) / rows) * ((N + cols - 1) / cols);
  const double now = dfhip_price(price, tiles, share, K / FBK, split_k, (double)N * K * (gate_up ? 2e-6 : 1e-6));
  const DfhipRing3Plan best = dfhip_ring3_plan(true, gate_up, M, N, K, share, may_split);
  // (side by side and up to 128 rows also where it is priced 5 % higher, which only gate + up is: two of these launches can become
  // one, dfhip_pairs.h, and where they do not it is faster or within 1 %.  [us a pair on two streams at 33 / 64 / 100 / 128 rows against the
  // 128-row ring: 28672 x 8192 152 / 153 / 160 / 168 and 154 / 154 / 158 / 166, 14336 x 4096 40.9 / 42.1 / 44.6 / 45.5 and 42.7 / 43.1 /
  // 44.4 / 45.1, 13824 x 5120 50 / 52 / 55 / 57 and 58 / 59 / 59 / 60])
  const double clearly = share > 1 && M <= DFHIP_PAIR_MAX_M ? 1.05
                         : gate_up && share > 1 ? 0.85 : M > 256 || gate_up ? 0.93 : 0.96;
  const double cube = clearly * clearly * clearly;
  return best.cost < cube * cube * now ? best : DfhipRing3Plan{-1, 1, 0.0};
}

// Activations of a few rows: the kernel that streams W past LDS (gemm_stream.hip); with 16 rows and more from K = 4096
// on, as for bf16 rows of the same bytes.  From 33 rows on every workgroup re-reads the activations four times as wide as
// up to 16, which a tile shares: there the 128 x 128 tiles take over, unless the launch is alone and its weights few.  [us at 33 / 64
// rows, streamed against 128 x 128: alone 28672 x 8192 47 / 52 against 52 / 54, with gate + up + SiLU*mul 96 / 96 against 91 / 90,
// 14336 x 4096 15 / 16 against 24 / 25, with gate + up 34 / 35 against 33 / 34; in pairs 28672 x 8192 94 / 110 against 89 / 92,
// 14336 x 4096 34 / 37 against 30 / 30.  The first goes with its gate + up.]  A product that may be cut along K goes there alone from 33
// rows on; in pairs it is streamed in parts of K from 9 to 32 rows (few_rows_parts) and goes there above.  [8192 x 28672 alone at 17 / 24
// / 33 / 64 rows: 38 / 41 / 47 / 58 against 46 / 46 / 48 / 50, in pairs at 33 / 64 100 / 122 against 80 / 84; 4096 x 14336 alone 13 / 14 / 18
// / 23 against 19 / 19 / 20 / 22, in pairs at 33 / 64 42 / 53 against 32 / 35.  Fewer than 2^25 weights stay: 1536 x 7168 alone at 40
// rows 10 against 13, in pairs at 12 rows level.]
bool few_rows_streamed(int M, int N, int K, int share, bool may_split) {
  if (!dfhip_stream_fits(M, N, K, 1) || (M >= 16 && K < 4096)) return false;
  const int64_t weights = (int64_t)N * K;
  if (!may_split || K <= N) return M <= 32 || (share == 1 && weights < (int64_t)1 << 27);
  if (weights < (int64_t)1 << 25) return M <= 32 || share == 1;
  return M <= (share == 1 ? 32 : weights < (int64_t)1 << 27 ? 16 : 8);
}

// Parts of K for 9 .. 32 rows beside as many of another nano-batch, where K may be cut (down to the model width): the fewest that give
// 160 workgroups of 32 columns and more, as a whole K does with fewer columns each, for which the activations are read again.
// Two such launches in a captured schedule become one, whose workgroups take each weight once for the rows of both; on
// 128 x 128 tiles they read it twice, and 128 rows of activations with it.  [us a pair in one launch, whole K up to 16 (8192 x 28672:
// 8) rows or 128 x 128 tiles -> in parts, at 12 / 17 / 24 / 32 rows: 8192 x 28672 60 / 62 / 64 / 64 -> 40 / 42 / 45 / 49, 4096 x 14336
// 15.4 / 21.4 / 21.5 / 21.9 -> 14.3 / 16.3 / 17.6 / 19.8, 2048 x 16384 14.4 / 17.0 / 17.3 / 17.4 -> 10.0 / 11.3 / 12.1 / 13.5, 8192 x 16384 39
// / 41 / 39 / 40 -> 31 / 33 / 33 / 35; at 2 rows 4096 x 14336 11.9 -> 13.5; layer 8192 x 28672 of 2 x 12 tokens 163 -> 142.
// Launches that stay two (DFHIP_SPLIT_APART) read their weights twice either way.  They take four parts and more, which fill the chip,
// and two where whole K would be streamed with fewer than 160 workgroups; two parts of anything wider, or instead of tiles, are
// slower.  [us a pair on two streams in a graph, without parts -> in parts, at 9 / 12 / 16 / 17 / 24 / 32 rows: taken 1280 x 16384 25.8 / 27.4 / 29.4
// / 31.3 / 33.9 / 36.9 -> 20.1 / 20.3 / 20.4 / 21.8 / 22.1 / 23.0, 2048 x 16384 27.1 / 27.4 / 29.0 / 26.0 / 26.2 / 26.3 -> 21.9 / 21.9 / 22.0 / 23.1 /
// 22.9 / 24.2, from 12 rows 3072 x 8192 20.1 / 20.8 / 22.0 / 23.2 / 24.4 / 26.2 -> 20.9 / 20.8 / 21.6 / 22.1 / 23.3 / 23.7, at 12 and 16 4096 x 14336
// 29.2 / 30.4 / 32.9 / 31.0 / 31.4 / 31.5 -> 29.9 / 30.2 / 30.6 / 31.1 / 32.6 / 33.5, 4608 x 18432 50 / 46 / 49 / 39 / 39 / 40 -> 43 / 44 / 45 / 46 / 48
// / 50; not taken 5120 x 25600 64 / 64 / 67 / 52 / 52 / 53 -> 64 / 63 / 64 / 65 / 67 / 70, 6144 x 16384 47 / 48 / 48 / 45 / 45 / 46 -> 50 / 50 / 50 / 51 / 51
// / 52, 8192 x 16384 50 / 51 / 50 / 51 / 52 / 52 -> 59 / 59 / 59 / 60 / 61 / 61, 8192 x 28672 78 / 76 / 76 / 77 / 77 / 78 -> 84 / 82 / 82 / 84 / 85 / 88]
int few_rows_parts(int M, int N, int K, int share, int may_split, bool streamed) {
  if (!may_split || share < 2 || K <= N || M < 9 || M > 32) return 1;
  const int64_t tiles = (N + 31) / 32;
  for (int s = 2; s <= 8; s *= 2) {
    if (tiles * s < 160) continue;
    if (may_split == DFHIP_SPLIT_APART && s < 4 && !(streamed && M >= 12 && tiles < 160)) return 1;
    return dfhip_stream_fits(M, N, K, s) ? s : 1;
  }
  return 1;
}

// The plan of a launch: -1 for the streaming kernel (F8_STREAM for counts of rows that have a tile as well), or a tile, and the parts of K.
TilePlan plan_launch(int M, int N, int K, int share, int may_split) {
  const bool streamed = few_rows_streamed(M, N, K, share, may_split);
  const int parts = few_rows_parts(M, N, K, share, may_split, streamed);
  if (streamed || parts > 1) return {streamed ? -1 : F8_STREAM, parts, 0.0};
  const TilePlan plan = plan_tile(M, N, K, share, may_split);
  const DfhipRing3Plan tiles = three_slabs_cheaper(false, M, N, K, share, plan.variant, plan.split_k, may_split && K > N);
  return tiles.tile < 0 ? plan : TilePlan{DFHIP_RING3_VARIANT + tiles.tile, tiles.split_k, tiles.cost};
}

int check_gemm(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, const float* a_scale,
               const float* w_scale, int M, int N, int K) {
  if (!A || !W || !C || !a_scale || !w_scale) return DFHIP_ERR_NULL_POINTER;
  if (M < 1 || N < 1 || K < 1 || K % FBK != 0 || N % 8 != 0) return DFHIP_ERR_BAD_SHAPE;
  if (lda < K || ldw < K || ldc < N) return DFHIP_ERR_BAD_STRIDE;
  if (lda >= (1 << 23) || ldw >= (1 << 23)) return DFHIP_ERR_BAD_STRIDE;   // 256 rows of a tile within 32-bit byte offsets
  if (lda % 16 || ldw % 16 || ldc % 8 || !dfhip_aligned16(A) || !dfhip_aligned16(W) || !dfhip_aligned16(C) ||
      !dfhip_aligned16(w_scale))
    return DFHIP_ERR_BAD_ALIGNMENT;
  return DFHIP_OK;
}

int check_q(const void* x, int64_t ld, int M, int D) {
  if (!x) return DFHIP_ERR_NULL_POINTER;
  if (M < 1 || D < 8 || D % 8 != 0 || (int64_t)M * (D / 8) >= (int64_t)1 << 31) return DFHIP_ERR_BAD_SHAPE;
  if (ld < D) return DFHIP_ERR_BAD_STRIDE;
  if (ld % 8 || !dfhip_aligned16(x)) return DFHIP_ERR_BAD_ALIGNMENT;
  return DFHIP_OK;
}

unsigned grid_for(uint32_t groups) {
  uint32_t blocks = (groups + QT * QUNROLL - 1) / (QT * QUNROLL);
  return blocks < 1 ? 1 : (blocks > 4096 ? 4096 : blocks);
}

}  // namespace

extern "C" int dfhip_absmax_bf16(const void* x, int64_t ld, int M, int D, float* amax, dfhip_stream_t stream) {
  if (int rc = check_q(x, ld, M, D)) return rc;
  if (!amax) return DFHIP_ERR_NULL_POINTER;
  const uint32_t per_row = D / 8, groups = (uint32_t)M * per_row;
  hipLaunchKernelGGL(absmax_bf16_kernel, dim3(grid_for(groups)), dim3(QT), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint16_t*>(x), ld, groups, per_row, amax);
  return dfhip_check_launch();
}

namespace {
unsigned parts_for(uint32_t groups) {
  const uint32_t blocks = (groups + QT * QUNROLL - 1) / (QT * QUNROLL);
  return blocks > QPARTS ? QPARTS : blocks;
}
int check_q_out(const void* q, int64_t ld_q, int D) {
  if (!q) return DFHIP_ERR_NULL_POINTER;
  if (ld_q < D) return DFHIP_ERR_BAD_STRIDE;
  return ld_q % 8 || (reinterpret_cast<uintptr_t>(q) & 7u) ? DFHIP_ERR_BAD_ALIGNMENT : DFHIP_OK;
}
template <bool PARTS>
int launch_quant_after(const void* x, int64_t ld, void* q, int64_t ld_q, int M, int D, float* amax, int n_parts, int* readers,
                       float* scale_out, hipStream_t stream) {
  const uint32_t per_row = D / 8, groups = (uint32_t)M * per_row;
  const QuantAfter<false, PARTS> args{static_cast<const uint16_t*>(x), static_cast<uint8_t*>(q), amax, readers, scale_out, ld,
                                      ld_q, groups, per_row, n_parts};
  if (ld != D || ld_q != D) return launch_quant_after(args, parts_for(groups), stream);
  return launch_quant_after(QuantAfter<true, PARTS>{args.x, args.q, amax, readers, scale_out, ld, ld_q, groups, per_row, n_parts},
                            parts_for(groups), stream);
}
template <bool SILU>
int launch_absmax_parts(const void* x, int64_t ld, const void* up, int64_t ld_up, void* out, int64_t ld_out, int M, int D,
                        bool flat, float* parts, hipStream_t stream) {
  const uint32_t per_row = D / 8, groups = (uint32_t)M * per_row;
  const AbsmaxParts<false, SILU> args{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(up),
                                      static_cast<uint16_t*>(out), parts, ld, ld_up, ld_out, groups, per_row};
  if (!flat) return launch_absmax_parts(args, parts_for(groups), stream);
  return launch_absmax_parts(AbsmaxParts<true, SILU>{args.x, args.up, args.out, parts, ld, ld_up, ld_out, groups, per_row},
                             parts_for(groups), stream);
}
}  // namespace

extern "C" int dfhip_quant_fp8_bf16(const void* x, int64_t ld, void* q, int64_t ld_q, int M, int D,
                                    const float* amax, float* scale_out, dfhip_stream_t stream) {
  if (int rc = check_q(x, ld, M, D)) return rc;
  if (!amax) return DFHIP_ERR_NULL_POINTER;
  if (int rc = check_q_out(q, ld_q, D)) return rc;
  return launch_quant_after<false>(x, ld, q, ld_q, M, D, const_cast<float*>(amax), 0, nullptr, scale_out,
                                   static_cast<hipStream_t>(stream));
}

extern "C" int dfhip_quant_fp8_dynamic_bf16(const void* x, int64_t ld, void* q, int64_t ld_q, int M, int D, float* parts,
                                            float* scale_out, dfhip_stream_t stream) {
  if (int rc = check_q(x, ld, M, D)) return rc;
  if (int rc = check_q_out(q, ld_q, D)) return rc;
  if (!parts) return DFHIP_ERR_NULL_POINTER;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (int rc = launch_absmax_parts<false>(x, ld, nullptr, 0, nullptr, 0, M, D, ld == D, parts, s)) return rc;
  return launch_quant_after<true>(x, ld, q, ld_q, M, D, parts, (int)parts_for((uint32_t)M * (D / 8)), nullptr, scale_out, s);
}

extern "C" int dfhip_silu_mul_quant_fp8_bf16(const void* gate, int64_t ld_gate, const void* up, int64_t ld_up, void* act,
                                             int64_t ld_act, void* q, int64_t ld_q, int M, int D, float* parts,
                                             float* scale_out, dfhip_stream_t stream) {
  if (int rc = check_q(gate, ld_gate, M, D)) return rc;
  if (int rc = check_q(up, ld_up, M, D)) return rc;
  if (int rc = check_q(act, ld_act, M, D)) return rc;
  if (int rc = check_q_out(q, ld_q, D)) return rc;
  if (!parts) return DFHIP_ERR_NULL_POINTER;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const bool flat = ld_gate == D && ld_up == D && ld_act == D;
  if (int rc = launch_absmax_parts<true>(gate, ld_gate, up, ld_up, act, ld_act, M, D, flat, parts, s)) return rc;
  return launch_quant_after<true>(act, ld_act, q, ld_q, M, D, parts, (int)parts_for((uint32_t)M * (D / 8)), nullptr, scale_out,
                                  s);
}

extern "C" int dfhip_requant_fp8_bf16(const void* x, int64_t ld, void* q, int64_t ld_q, int M, int D, void* cells,
                                      float* scale_out, dfhip_stream_t stream) {
  if (int rc = check_q(x, ld, M, D)) return rc;
  if (int rc = check_q_out(q, ld_q, D)) return rc;
  if (!cells) return DFHIP_ERR_NULL_POINTER;
  // counting readers costs 12 ns a block (350 x 28672: 21 us with 1024 of them, 11 with the launch that clears): up to 128
  if (parts_for((uint32_t)M * (D / 8)) > 128) {
    if (int rc = dfhip_quant_fp8_bf16(x, ld, q, ld_q, M, D, static_cast<float*>(cells), scale_out, stream)) return rc;
    return dfhip_fill_u32(cells, 0u, 1, stream);
  }
  return launch_quant_after<false>(x, ld, q, ld_q, M, D, static_cast<float*>(cells), 0, static_cast<int*>(cells) + 1,
                                   scale_out, static_cast<hipStream_t>(stream));
}

extern "C" int dfhip_silu_mul_absmax_bf16(const void* gate, int64_t ld_gate, const void* up, int64_t ld_up,
                                          void* out, int64_t ld_out, int M, int D, float* amax,
                                          dfhip_stream_t stream) {
  if (int rc = check_q(gate, ld_gate, M, D)) return rc;
  if (int rc = check_q(up, ld_up, M, D)) return rc;
  if (!amax) return DFHIP_ERR_NULL_POINTER;
  if (out) {
    if (ld_out < D) return DFHIP_ERR_BAD_STRIDE;
    if (ld_out % 8 || !dfhip_aligned16(out)) return DFHIP_ERR_BAD_ALIGNMENT;
  }
  const uint32_t per_row = D / 8, groups = (uint32_t)M * per_row;
  hipLaunchKernelGGL(silu_mul_absmax_kernel, dim3(grid_for(groups)), dim3(QT), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint16_t*>(gate), ld_gate, static_cast<const uint16_t*>(up), ld_up,
                     static_cast<uint16_t*>(out), ld_out, groups, per_row, amax);
  return dfhip_check_launch();
}

extern "C" int dfhip_gemm_fp8_nt_variant(const void* A, int64_t lda, const void* W, int64_t ldw, void* C,
                                         int64_t ldc, const float* a_scale, const float* w_scale, int M, int N,
                                         int K, int variant, dfhip_stream_t stream) {
  if (int rc = check_gemm(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (variant < 0) return dfhip_gemm_fp8_nt_shared(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, 1, stream);
  switch (variant) {
    case 0: return launch_fp8_ring<8, false>(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, 1, nullptr, s);
    case 1: return launch_fp8<128, 128>(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, s);
    case 2: return launch_fp8_ring224(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, s);
    case 3: return launch_fp8_ring<6, false>(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, 1, nullptr, s);
    case 4: return launch_fp8_ring<4, false>(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, 1, nullptr, s);
    default:
      if (!dfhip_ring3_variant(variant, true)) return DFHIP_ERR_BAD_ARGUMENT;
      return dfhip_ring3_fp8(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, variant - DFHIP_RING3_VARIANT, 1, nullptr, s);
  }
}

extern "C" int dfhip_gemm_fp8_nt_shared(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
                                        const float* a_scale, const float* w_scale, int M, int N, int K, int share,
                                        dfhip_stream_t stream) {
  if (int rc = check_gemm(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K)) return rc;
  if (share < 1 || share > 16) return DFHIP_ERR_BAD_ARGUMENT;
  const TilePlan plan = plan_launch(M, N, K, share, false);
  if (plan.variant < 0)
    return dfhip_stream_fp8(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, 1, nullptr, nullptr, static_cast<hipStream_t>(stream));
  return dfhip_gemm_fp8_nt_variant(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, plan.variant, stream);
}

extern "C" int dfhip_gemm_fp8_plan_shared(int M, int N, int K, int share, int* variant, int* split_k) {
  if (!variant || !split_k) return DFHIP_ERR_NULL_POINTER;
  if (M < 1 || N < 1 || K < 1) return DFHIP_ERR_BAD_SHAPE;
  if (share < 1 || share > 16) return DFHIP_ERR_BAD_ARGUMENT;
  *variant = -1;
  *split_k = 1;
  if (few_rows_streamed(M, N, K, share, true)) return DFHIP_OK;
  const TilePlan plan = plan_tile(M, N, K, share, true);
  *variant = plan.variant;
  *split_k = plan.split_k;
  return DFHIP_OK;
}

extern "C" int dfhip_gemm_fp8_plan_tiles(int M, int N, int K, int share, int may_split, int* variant, int* split_k) {
  if (!variant || !split_k) return DFHIP_ERR_NULL_POINTER;
  if (M < 1 || N < 1 || K < 1) return DFHIP_ERR_BAD_SHAPE;
  if (share < 1 || share > 16) return DFHIP_ERR_BAD_ARGUMENT;
  const TilePlan plan = plan_launch(M, N, K, share, may_split);
  *variant = plan.variant;
  *split_k = plan.split_k;
  return DFHIP_OK;
}

extern "C" size_t dfhip_gemm_fp8_splitk_workspace_bytes(int M, int N, int variant, int split_k) {
  const int tm = ring_blocks(variant);
  if (M >= 1 && N >= 1 && (variant < 0 || variant == F8_STREAM) && split_k >= 2 && split_k <= F8_MAX_SPLIT)
    return DFHIP_COMMON_COUNTERS + (size_t)((N + 63) / 64) * 64 * split_k * 64 * sizeof(float);
  if (M >= 1 && N >= 1 && split_k >= 2 && split_k <= DFHIP_RING3_MAX_SPLIT && dfhip_ring3_variant(variant, true))
    return dfhip_ring3_workspace_bytes(M, N, variant - DFHIP_RING3_VARIANT, split_k);
  if (M < 1 || N < 1 || split_k < 2 || split_k > F8_MAX_SPLIT || !tm) return 0;
  const size_t tiles = (size_t)((M + 32 * tm - 1) / (32 * tm)) * ((N + 255) / 256);
  return dfhip_counter_area(tiles) + tiles * split_k * (size_t)(32 * tm) * 256 * sizeof(float);
}

extern "C" int dfhip_gemm_fp8_nt_splitk(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
                                        const float* a_scale, const float* w_scale, int M, int N, int K, int variant,
                                        int split_k, void* workspace, size_t workspace_bytes, dfhip_stream_t stream) {
  if (int rc = check_gemm(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K)) return rc;
  const int tm = ring_blocks(variant);
  const bool three_slabs = dfhip_ring3_variant(variant, true), streamed = variant < 0 || variant == F8_STREAM;
  if (streamed && (M > 32 || split_k < 2 || !dfhip_stream_fits(M, N, K, split_k))) return DFHIP_ERR_BAD_ARGUMENT;
  if ((!tm && !three_slabs && !streamed) || split_k < 2 || split_k > F8_MAX_SPLIT || K / FBK < 2 * split_k) return DFHIP_ERR_BAD_ARGUMENT;
  if (!workspace) return DFHIP_ERR_NULL_POINTER;
  if (!dfhip_aligned16(workspace)) return DFHIP_ERR_BAD_ALIGNMENT;
  if (workspace_bytes < dfhip_gemm_fp8_splitk_workspace_bytes(M, N, variant, split_k)) return DFHIP_ERR_BAD_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (streamed)
    return dfhip_stream_fp8(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, split_k,
                            static_cast<uint8_t*>(workspace) + DFHIP_COMMON_COUNTERS, static_cast<int*>(workspace), s);
  if (three_slabs)
    return dfhip_ring3_fp8(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, variant - DFHIP_RING3_VARIANT, split_k,
                           workspace, s);
  switch (tm) {
    case 8: return launch_fp8_ring<8, true>(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, split_k, workspace, s);
    case 6: return launch_fp8_ring<6, true>(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, split_k, workspace, s);
    default: return launch_fp8_ring<4, true>(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, split_k, workspace, s);
  }
}

namespace {
// The kernel of a gate + up + SiLU*mul launch: a three-slab tile, the streaming kernel (both -1), or a ring tile of 32 `tm` rows.
struct GateUpPlan { int three_slabs, tm; };
GateUpPlan plan_gate_up(int M, int I, int K, int share) {
  if (few_rows_streamed(M, I, K, share, false)) return {-1, -1};
  // the height of the tile that costs least in rounds (see tile_cost); every height adds in the same order.  A pair of
  // 2 x 14336 x 4096 at 192 / 256 rows: one round of 192 and 256-row tiles 53 / 59 us, two of 128-row ones 66 / 68.  (Of a
  // pair the last round runs beside the other launch, and can cost less than it is priced at: 2 x 12288 x 6144 at 700
  // rows takes 192-row tiles and 181 us where 256-row ones take 167.)
  const RingTile* ring = &F8_RINGS[0];
  double least = 0.0;
  for (const RingTile& r : F8_RINGS) {
    const int64_t tiles = (int64_t)((M + 32 * r.tm - 1) / (32 * r.tm)) * ((I + 127) / 128);
    const double cost = tile_cost(tiles, 1, share, K, r.per_slab, r.tm);
    if (&r == &F8_RINGS[0] || cost < least) { ring = &r; least = cost; }
  }
  const DfhipRing3Plan three = three_slabs_cheaper(true, M, I, K, share, ring->variant, 1, false);
  return three.tile >= 0 ? GateUpPlan{three.tile, 0} : GateUpPlan{-1, ring->tm};
}
int check_gate_up(const void* A, int64_t lda, const void* W_gate, const void* W_up, int64_t ldw, const void* act, int64_t ld_act,
                  const float* a_scale, const float* w_gate_scale, const float* w_up_scale, const float* amax, int M, int I, int K,
                  int share) {
  if (!A || !W_gate || !W_up || !act || !a_scale || !w_gate_scale || !w_up_scale || !amax)
    return DFHIP_ERR_NULL_POINTER;
  if (M < 1 || I < 8 || K < 1 || K % FBK != 0 || I % 8 != 0) return DFHIP_ERR_BAD_SHAPE;
  if (lda < K || ldw < K || ld_act < I) return DFHIP_ERR_BAD_STRIDE;
  if (lda >= (1 << 23) || ldw >= (1 << 23)) return DFHIP_ERR_BAD_STRIDE;
  if (lda % 16 || ldw % 16 || ld_act % 8 || !dfhip_aligned16(A) || !dfhip_aligned16(W_gate) ||
      !dfhip_aligned16(W_up) || !dfhip_aligned16(act) || !dfhip_aligned16(w_gate_scale) ||
      !dfhip_aligned16(w_up_scale))
    return DFHIP_ERR_BAD_ALIGNMENT;
  if (share < 1 || share > 16) return DFHIP_ERR_BAD_ARGUMENT;
  return DFHIP_OK;
}
int launch_gate_up(const GateUpPlan& plan, const void* A, int64_t lda, const void* W_gate, const void* W_up, int64_t ldw, void* act,
                   int64_t ld_act, const float* a_scale, const float* w_gate_scale, const float* w_up_scale, float* amax,
                   bool amax_apart, int M, int I, int K, hipStream_t s) {
  if (plan.three_slabs >= 0)
    return dfhip_ring3_fp8_gate_up(A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale, w_up_scale, amax, amax_apart, M, I,
                                   K, plan.three_slabs, s);
  switch (plan.tm) {
    case -1: return dfhip_stream_fp8_gate_up(A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale, w_up_scale, amax,
                                             amax_apart, M, I, K, s);
    case 8: return launch_fp8_ring_fused<8>(A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale, w_up_scale, amax,
                                            M, I, K, s);
    case 6: return launch_fp8_ring_fused<6>(A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale, w_up_scale, amax,
                                            M, I, K, s);
    default: return launch_fp8_ring_fused<4>(A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale, w_up_scale,
                                             amax, M, I, K, s);
  }
}
}  // namespace

extern "C" int dfhip_gemm_fp8_gate_up_silu_absmax_shared(const void* A, int64_t lda, const void* W_gate,
                                                         const void* W_up, int64_t ldw, void* act, int64_t ld_act,
                                                         const float* a_scale, const float* w_gate_scale,
                                                         const float* w_up_scale, float* amax, int M, int I, int K,
                                                         int share, dfhip_stream_t stream) {
  if (int rc = check_gate_up(A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale, w_up_scale, amax, M, I, K, share)) return rc;
  return launch_gate_up(plan_gate_up(M, I, K, share), A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale, w_up_scale, amax,
                        false, M, I, K, static_cast<hipStream_t>(stream));
}

extern "C" int dfhip_gemm_fp8_gate_up_silu_quant_shared(const void* A, int64_t lda, const void* W_gate, const void* W_up, int64_t ldw,
                                                        void* act, int64_t ld_act, void* q, int64_t ld_q, const float* a_scale,
                                                        const float* w_gate_scale, const float* w_up_scale, float* parts,
                                                        float* scale_out, int M, int I, int K, int share, dfhip_stream_t stream) {
  if (int rc = check_gate_up(A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale, w_up_scale, parts, M, I, K, share)) return rc;
  if (int rc = check_q(act, ld_act, M, I)) return rc;
  if (int rc = check_q_out(q, ld_q, I)) return rc;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const GateUpPlan plan = plan_gate_up(M, I, K, share);
  const int64_t blocks = plan.three_slabs >= 0 ? dfhip_ring3_gate_up_blocks(M, I, plan.three_slabs)
                                               : plan.tm < 0 ? dfhip_stream_blocks(I) : DFHIP_FP8_GEMM_PARTS;
  const bool apart = 4 * blocks <= DFHIP_FP8_GEMM_PARTS;
  if (!apart)
    if (int rc = dfhip_fill_u32(parts, 0u, 1, stream)) return rc;
  if (int rc = launch_gate_up(plan, A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale, w_up_scale, parts, apart, M, I, K, s))
    return rc;
  return apart ? launch_quant_after<true>(act, ld_act, q, ld_q, M, I, parts, 4 * (int)blocks, nullptr, scale_out, s)
               : launch_quant_after<false>(act, ld_act, q, ld_q, M, I, parts, 0, nullptr, scale_out, s);
}

extern "C" int dfhip_gemm_fp8_gate_up_silu_absmax(const void* A, int64_t lda, const void* W_gate, const void* W_up,
                                                  int64_t ldw, void* act, int64_t ld_act, const float* a_scale,
                                                  const float* w_gate_scale, const float* w_up_scale, float* amax,
                                                  int M, int I, int K, dfhip_stream_t stream) {
  return dfhip_gemm_fp8_gate_up_silu_absmax_shared(A, lda, W_gate, W_up, ldw, act, ld_act, a_scale, w_gate_scale,
                                                   w_up_scale, amax, M, I, K, 1, stream);
}

extern "C" int dfhip_gemm_fp8_nt(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
                                 const float* a_scale, const float* w_scale, int M, int N, int K,
                                 dfhip_stream_t stream) {
  return dfhip_gemm_fp8_nt_variant(A, lda, W, ldw, C, ldc, a_scale, w_scale, M, N, K, -1, stream);
}
