// Weight-streaming launches for a handful of rows, shared by the bf16 and fp8 entry points (not part of the C ABI).
// Pointers, strides and shapes have been checked by the caller.
#pragma once
#include "dfhip_common.h"

constexpr int DFHIP_STREAM_MAX_M = 64;

// Whether the kernel takes M rows, N columns and rows of k_bytes with K cut into split_k parts.
bool dfhip_stream_fits(int M, int N, int64_t k_bytes, int split_k);
// The parts K should be cut into by a caller with a workspace.
int dfhip_stream_split(int M, int N, int64_t k_bytes);

// split_k > 1 (up to 32 rows): `partials` holds ceil(N / 64) * 64 * split_k * 64 floats, `arrivals` one zero per 16 columns (left zero).
int dfhip_stream_bf16(const void* A, int64_t lda, const void* W, int64_t ldw, const void* R, void* C, int64_t ldc, int M,
                      int N, int K, int split_k, void* partials, int* arrivals, hipStream_t stream);
int dfhip_stream_bf16_gate_up(const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, void* C, int64_t ldc,
                              int M, int N, int K, hipStream_t stream);
int dfhip_stream_fp8(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, const float* a_scale,
                     const float* w_scale, int M, int N, int K, int split_k, void* partials, int* arrivals, hipStream_t stream);
int dfhip_stream_fp8_gate_up(const void* A, int64_t lda, const void* W, const void* W2, int64_t ldw, void* C, int64_t ldc,
                             const float* a_scale, const float* w_scale, const float* w2_scale, float* amax, bool amax_apart,
                             int M, int N, int K, hipStream_t stream);
// Workgroups of a launch with whole K; with `amax_apart` each leaves four maxima.
int dfhip_stream_blocks(int N);
