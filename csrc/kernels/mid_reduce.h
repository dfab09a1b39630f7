// The sums that close split projections (mid_gemm.hip holds the kernels): partial sums ws [S, M, N] in 32 bits, added in fixed order.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// y [M, N] = sum (+ bias), or with pair silu(gate) * up [M, N / 2]; rows of stride ys (a multiple of 4, y on 8 bytes).
int mid_reduce(const void* ws, const void* bias, void* y, long ys, int M, int N, int S, int pair, hipStream_t stream);

// residual [M, N] += sum, y [M, N] = rms norm of the new rows * weight.
bool mid_reduce_norm_takes(const void* residual, const void* weight, const void* y, int N);
int mid_reduce_norm(const void* ws, void* residual, const void* weight, void* y, int M, int N, int S, float eps, hipStream_t stream);

// q | k | v of one token per sequence: q rotated to q_out [M, n_q * 128], k rotated and v to the cache (slots < 0: nowhere).
bool mid_reduce_qkv_takes(const void* q_out, const void* bias, const void* cos_sin);
int mid_reduce_qkv(const void* ws, const void* bias, void* q_out, const int* positions, const long* slots, const float* cos_sin,
                   void* cache, long page_stride, long v_offset, int M, int n_q, int n_kv, int S, hipStream_t stream);
