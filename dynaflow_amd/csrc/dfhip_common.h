// Internal helpers shared by the kernel sources (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "../../include/dynaflow_hip.h"

typedef __bf16 bf16_t;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define DFHIP_DEVICE __device__ __forceinline__

static inline bool dfhip_aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Opt a kernel in to `bytes` of dynamic LDS.  The attribute belongs to the (function, device) pair, so `done`
// - one word per kernel instantiation - carries one bit per device; setting the attribute twice from two
// threads is harmless, reading a torn flag is not, hence the atomic.
static inline int dfhip_opt_in_lds(const void* kernel, int bytes, std::atomic<uint64_t>& done) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return DFHIP_ERR_NO_DEVICE;
  const uint64_t bit = 1ull << (device & 63);
  if (done.load(std::memory_order_acquire) & bit) return DFHIP_OK;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)
    return DFHIP_ERR_LAUNCH;
  done.fetch_or(bit, std::memory_order_release);
  return DFHIP_OK;
}

static inline int dfhip_check_launch() {
  return hipGetLastError() == hipSuccess ? DFHIP_OK : DFHIP_ERR_LAUNCH;
}

// Split-K workspaces start with the arrival counters.  All split-K kernels, bf16 and fp8, use the same size of
// counter area up to 1024 tiles (4 KiB), so that the fp32 blocks one of them leaves behind do not lie where another
// expects counters that are zero.  A launch of more tiles has counters where smaller ones leave blocks, and clears
// those first (a fill kernel, legal inside a captured graph).
constexpr size_t DFHIP_COMMON_COUNTERS = 4096;
static inline size_t dfhip_counter_area(size_t tiles) {
  const size_t need = ((tiles * sizeof(int)) + 255) & ~(size_t)255;
  return need > DFHIP_COMMON_COUNTERS ? need : DFHIP_COMMON_COUNTERS;
}
static inline int dfhip_clear_uncommon_counters(void* workspace, size_t tiles, hipStream_t stream) {
  const size_t area = dfhip_counter_area(tiles);
  if (area == DFHIP_COMMON_COUNTERS) return DFHIP_OK;
  return dfhip_fill_u32(static_cast<uint8_t*>(workspace) + DFHIP_COMMON_COUNTERS, 0u,
                        (int64_t)((area - DFHIP_COMMON_COUNTERS) / 4), stream);
}

// bf16 <-> fp32 on raw 16-bit storage
DFHIP_DEVICE float bf16_bits_to_f32(uint32_t bits16) { return __uint_as_float(bits16 << 16); }

// round-to-nearest-even fp32 -> bf16 (quiet NaN preserved)
DFHIP_DEVICE uint32_t f32_to_bf16_bits(float f) {
  bf16_t h = static_cast<bf16_t>(f);
  return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, h));
}

// two values rounded and packed by one v_cvt_pk_bf16_f32 (same rounding as f32_to_bf16_bits, lo in bits 0..15)
DFHIP_DEVICE uint32_t pack2_bf16(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
// the two bf16 values of a packed pair, as fp32
DFHIP_DEVICE float bf16_lo_to_f32(uint32_t pair) { return __uint_as_float(pair << 16); }
DFHIP_DEVICE float bf16_hi_to_f32(uint32_t pair) { return __uint_as_float(pair & 0xffff0000u); }

// bf16(x + r) on packed pairs: the product is rounded to bf16 first (x is such a rounded value), the
// sum is rounded again - the roundings of a GEMM followed by a separate bf16 addition.
DFHIP_DEVICE uint32_t add2_bf16(uint32_t x, uint32_t r) {
  return pack2_bf16(bf16_lo_to_f32(x) + bf16_lo_to_f32(r),
                    bf16_hi_to_f32(x) + bf16_hi_to_f32(r));
}

// silu(g) = g / (1 + e^-g) on the hardware exponential and reciprocal (a few fp32 ulp; the bf16 paths
// round the result to 8 bits of mantissa right after).  -inf gives NaN like the exact quotient.
DFHIP_DEVICE float silu_fast(float g) {
  return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * g));
}

// 64-lane reductions through DPP-free shuffles (wave64)
DFHIP_DEVICE float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
DFHIP_DEVICE float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// Two loads of 16 rows of 128 bytes, in which neighbouring lanes share 32 bytes of a row (load h, lane: row 2 (lane / 2 % 8) + h, chunk
// 2 (lane / 16) + lane % 2 of 16 bytes) -> two MFMA fragments (lane: row lane % 16, chunks 2 (lane / 16) and + 1): neighbours
// exchange one of their two pieces.
// Written out: a selection whose one operand comes from the neighbour is one instruction, of which the compiler makes two.  It does
// not see the registers being read and written in here, so the block waits for them itself, two states each: in front between the
// write of a register and its read by another lane, behind between the last write and an MFMA that reads it (an fp8 one reads all
// eight registers at once).
DFHIP_DEVICE void deal_neighbours(u32x4& first, u32x4& second) {
  uint32_t a0, a1, a2, a3, b0, b1, b2, b3;
  asm("s_mov_b32 vcc_lo, 0x55555555\n\ts_mov_b32 vcc_hi, 0x55555555\n\ts_nop 1\n\t"       // even lanes keep their own
      "v_cndmask_b32_dpp %0, %12, %8, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %1, %13, %9, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %2, %14, %10, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %3, %15, %11, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "s_not_b64 vcc, vcc\n\t"                                                            // odd ones
      "v_cndmask_b32_dpp %4, %8, %12, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %5, %9, %13, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %6, %10, %14, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %7, %11, %15, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1"
      : "=&v"(a0), "=&v"(a1), "=&v"(a2), "=&v"(a3), "=&v"(b0), "=&v"(b1), "=&v"(b2), "=&v"(b3)
      : "v"(first[0]), "v"(first[1]), "v"(first[2]), "v"(first[3]), "v"(second[0]), "v"(second[1]), "v"(second[2]), "v"(second[3])
      : "vcc", "scc");
  first = u32x4{a0, a1, a2, a3};
  second = u32x4{b0, b1, b2, b3};
}

// The 8 XCDs of the chip take workgroups round-robin (workgroup i runs on XCD
// i % 8) and each XCD has a private L2.  remap_xcd turns the launch index into
// a tile index such that every XCD walks one contiguous range of tiles, so the
// tiles that are resident together on an XCD are neighbours and share operand
// rows/columns in that XCD's L2.  (Also compiled for the host: the mapping is
// replayed by CPU tests.)
__host__ __device__ __forceinline__ int remap_xcd(int pid, int total) {
  constexpr int XCDS = 8;
  const int xcd = pid % XCDS;
  const int local = pid / XCDS;
  const int base = total / XCDS;
  const int rem = total % XCDS;
  const int start = xcd * base + (xcd < rem ? xcd : rem);
  return start + local;
}

// Work item of a workgroup of the 256 x 256 split-K launch (`tiles` tiles, K of every tile cut into
// `split_k` parts): the launch is part-major - launch indices [p * tiles, (p + 1) * tiles) are part p of
// every tile, dealt to the XCDs like the tiles of an unsplit launch.  The last part of a tile, which waits
// for the others, therefore has the highest launch index of that tile for every tile count, and the parts
// it waits for were dispatched before it.
__host__ __device__ __forceinline__ void splitk_work_of(int pid, int tiles, int& tile, int& part) {
  part = pid / tiles;
  tile = remap_xcd(pid - part * tiles, tiles);
}

// ---- hand-ordered memory operations of the LDS-DMA GEMM kernels ------------------------------
// One LDS-DMA instruction: 64 lanes x 16 bytes from per-lane global addresses to
// LDS[lds_addr + 16*lane].  The compiler does not see the memory effect; ordering is kept by
// hand with wait_vmcnt / workgroup_barrier.
DFHIP_DEVICE void dma16(uint32_t lds_addr, const void* g) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_addr), "v"(g)
               : "memory", "m0");
}
// The same for what is read once: non-temporal, past what the caches keep.
DFHIP_DEVICE void dma16_once(uint32_t lds_addr, const void* g) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds_addr), "v"(g)
               : "memory", "m0");
}
// The same with a wave-uniform base (scalar registers) and a 32-bit per-lane byte offset.
DFHIP_DEVICE void dma16_base(uint32_t lds_addr, const void* base, uint32_t offset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(offset), "s"(base)
               : "memory", "m0");
}
template <int N>
DFHIP_DEVICE void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// 16-byte store / load that is coherent across the XCDs (sc1: written through to, and read
// from, the memory side instead of the XCD-private L2).  Used for split-K partial blocks so
// that no L2-wide write-back or invalidate is needed to hand them from one XCD to another.
// A load is a builtin and not inline assembly: the compiler takes an asm output as written at once, so it
// may copy or reuse the registers of a load that is still on its way, and it places no wait for it.
// A store of more than 8 bytes reads its data registers for a few cycles after issue and the compiler
// cannot see that this statement is one: the wait states keep the next write to those registers away.
DFHIP_DEVICE void store_f32x4_device_coherent(f32x4* p, f32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}
// The blocks that the parts of one tile left: `base` is the same for the whole wave.
DFHIP_DEVICE __amdgpu_buffer_rsrc_t coherent_blocks(const void* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00027000);
}
// `at` bytes (of the lane) + `uniform` bytes (of the wave) into them
DFHIP_DEVICE f32x4 load_f32x4_device_coherent(__amdgpu_buffer_rsrc_t blocks, int at, int uniform) {
  constexpr int SC1 = 16;
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(blocks, at, uniform, SC1));
}
DFHIP_DEVICE void workgroup_barrier() { asm volatile("s_barrier" ::: "memory"); }
#define DFHIP_PIN __builtin_amdgcn_sched_barrier(0)
