// Mixture-of-experts routing kernels for gfx950 (Mixtral-style top-k softmax routing).
//   1. moe_topk_softmax: router logits -> top-k expert ids + renormalised weights
//   2. moe_align:        counting sort of the (token, k) pairs by expert -> per-expert
//                        contiguous row ranges for the expert GEMMs
//   3. moe_permute:      gather activation rows into expert-sorted order
//   4. moe_combine:      out[t] = sum_k w[t,k] * y[pos[t,k]]  (gather form: no atomics, so
//                        the result is bitwise reproducible)
// The experts' products on those row ranges: mid_experts_kernel (mid_gemm.hip) up to 48 rows an expert on average, the
// grouped form of tile_gemm.hip above, per-pair kernels for a single token.
#include <type_traits>

#include "common.h"

#define MAX_EXPERTS 64        // top-k softmax: a lane per expert
#define ALIGN_MAX_EXPERTS 1024  // the counting sort keeps its counters in LDS
#define MAX_TOPK 8

// The router's product, logits[t, e] = x[t] . w[e] rounded to bf16, for up to 64 experts: a workgroup takes 16 tokens, its waves quarters of
// the reduction (a token's row is read once, 64 bytes of 16 rows an instruction, 16 on their way), and their sums meet in LDS.  What
// bounds it is the way of the rows to too few CUs; the library's tile of 16 x 16 walks the whole reduction with one wave: 1531 tokens of
// 4096 channels, 8 experts 16.6 -> 10.7 us in a step (the loads one at a time, as the compiler puts them by itself: 15).  ops.moe_router_takes
// has the sizes where it is the better choice.
template <int ET>
__global__ __launch_bounds__(256) void moe_router_kernel(const uint16_t* __restrict__ x, long x_stride, const uint16_t* __restrict__ w,
                                                         uint16_t* __restrict__ logits, int tokens, int n_experts, int hidden) {
  __shared__ f32x4 part[3][ET][64];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * 16, row = min(t0 + c, tokens - 1), steps = hidden / 128;  // of 32 channels, a wave's
  const uint16_t* xp = x + (long)row * x_stride + wave * steps * 32 + 8 * g;
  const uint16_t* wp[ET];
#pragma unroll
  for (int i = 0; i < ET; ++i) wp[i] = w + (long)min(16 * i + c, n_experts - 1) * hidden + wave * steps * 32 + 8 * g;
  f32x4 acc[ET];
#pragma unroll
  for (int i = 0; i < ET; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto go = [&](auto batch, int k) {
    constexpr int B = decltype(batch)::value;
    bf16x8 xf[B], wf[ET][B];
#pragma unroll
    for (int j = 0; j < B; ++j) {
      xf[j] = *reinterpret_cast<const bf16x8*>(xp + (k + j) * 32);
#pragma unroll
      for (int i = 0; i < ET; ++i) wf[i][j] = *reinterpret_cast<const bf16x8*>(wp[i] + (k + j) * 32);
    }
    __builtin_amdgcn_sched_barrier(0);  // all of them are on their way before the first is waited for
#pragma unroll
    for (int j = 0; j < B; ++j)
#pragma unroll
      for (int i = 0; i < ET; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][j], xf[j], acc[i], 0, 0, 0);
  };
  int k = 0;
  for (; k + 16 / ET <= steps; k += 16 / ET) go(std::integral_constant<int, 16 / ET>(), k);
  for (; k < steps; ++k) go(std::integral_constant<int, 1>(), k);
  if (wave) {
#pragma unroll
    for (int i = 0; i < ET; ++i) part[wave - 1][i][lane] = acc[i];
  }
  __syncthreads();
  if (wave || t0 + c >= tokens) return;
#pragma unroll
  for (int i = 0; i < ET; ++i) {
    const f32x4 sum = (acc[i] + part[0][i][lane]) + (part[1][i][lane] + part[2][i][lane]);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = 16 * i + 4 * g + q;
      if (e < n_experts) logits[(long)(t0 + c) * n_experts + e] = (uint16_t)(pack_bf16x2(sum[q], 0.f) & 0xffff);
    }
  }
}

// A lane per expert, G = 8, 16, 32 or 64 lanes per token.  (One thread per token kept the scores in an array that it indexes: scratch memory,
// 18 us for 1531 tokens of 8 experts, 5 here.)  An expert whose score is not a number is never chosen; where nothing is left
// to choose the choice is expert 0.
template <int G>
__global__ __launch_bounds__(256) void moe_topk_softmax_kernel(const uint16_t* __restrict__ logits,
                                                               float* __restrict__ weights,
                                                               int* __restrict__ ids, int tokens,
                                                               int n_experts, int topk,
                                                               int renorm) {
  const int t = (blockIdx.x * 256 + threadIdx.x) / G, e = threadIdx.x % G;
  const bool in = t < tokens && e < n_experts;
  float v = in ? bf16_bits_to_f32(logits[(long)t * n_experts + e]) : -INFINITY;
  float mx = v;
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  v = in ? __expf(v - mx) : 0.f;
  float den = v;
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) den += __shfl_xor(den, off, 64);
  float key = in && v >= 0.f ? v : -1.f, wsum = 0.f, mine_w = 0.f;
  int mine = 0;  // lane k < topk keeps choice k
  for (int k = 0; k < topk; ++k) {
    float best = key;
    int bi = key < 0.f ? 0 : e;
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, 64);
      const int oi = __shfl_xor(bi, off, 64);
      if (ob > best || (ob == best && oi < bi)) best = ob, bi = oi;
    }
    if (e == bi) key = -1.f;
    const float wk = best / den;
    wsum += wk;
    if (e == k) mine = bi, mine_w = wk;
  }
  if (t < tokens && e < topk) {
    weights[(long)t * topk + e] = renorm ? mine_w / wsum : mine_w;
    ids[(long)t * topk + e] = mine;
  }
}

// Single-workgroup counting sort.  offsets has n_experts + 1 entries; pos[i] is the sorted
// row of pair i = t*topk + k; sorted_tok[row] = token of that row, sorted_w[row] (optional) its pair's weight.  Pairs of
// one expert keep their token order (stable), so results do not depend on scheduling.
// Each of the 16 waves owns a contiguous run of pairs: it counts its run's pairs per expert, the counts turn into the
// run's first row per expert (expert by expert, run by run), and the wave walks its run 64 pairs at a time, a pair's
// rank among the 64 being its place among the lanes with the same expert (one ballot per bit of the expert's number).
#define ALIGN_WAVES 16
__global__ __launch_bounds__(1024) void moe_align_kernel(const int* __restrict__ ids,
                                                         int* __restrict__ offsets,
                                                         int* __restrict__ pos,
                                                         int* __restrict__ sorted_tok,
                                                         const float* __restrict__ weights,
                                                         float* __restrict__ sorted_w, int n_pairs,
                                                         int n_experts, int topk, int id_bits) {
  extern __shared__ int cnt[];  // [ALIGN_WAVES][n_experts]: counts, then next free rows; [n_experts]: totals
  int* const total = cnt + ALIGN_WAVES * n_experts;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int e = tid; e < ALIGN_WAVES * n_experts; e += 1024) cnt[e] = 0;
  __syncthreads();
  const int run = ((n_pairs + ALIGN_WAVES - 1) / ALIGN_WAVES + 63) & ~63;
  const int i_lo = wave * run, i_hi = min(n_pairs, i_lo + run);
  int* const mine = cnt + wave * n_experts;
  for (int i = i_lo + lane; i < i_hi; i += 64) {
    const int e = ids[i];
    if (e >= 0 && e < n_experts) atomicAdd(&mine[e], 1);
  }
  __syncthreads();
  for (int e = tid; e < n_experts; e += 1024) {
    int sum = 0;
    for (int w = 0; w < ALIGN_WAVES; ++w) sum += cnt[w * n_experts + e];
    total[e] = sum;
  }
  __syncthreads();
  if (wave == 0) {  // exclusive prefix over the experts, 64 at a time
    int base = 0;
    for (int e0 = 0; e0 < n_experts; e0 += 64) {
      const int e = e0 + lane;
      const int v = e < n_experts ? total[e] : 0;
      int incl = v;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
      }
      if (e < n_experts) {
        total[e] = base + incl - v;
        offsets[e] = base + incl - v;
      }
      base += __shfl(incl, 63, 64);
    }
    if (lane == 0) offsets[n_experts] = base;
  }
  __syncthreads();
  for (int e = tid; e < n_experts; e += 1024) {
    int at = total[e];
    for (int w = 0; w < ALIGN_WAVES; ++w) {
      const int c = cnt[w * n_experts + e];
      cnt[w * n_experts + e] = at;
      at += c;
    }
  }
  __syncthreads();
  for (int i0 = i_lo; i0 < i_hi; i0 += 64) {
    const int i = i0 + lane;
    const int e = i < i_hi ? ids[i] : -1;
    const bool ok = e >= 0 && e < n_experts;
    unsigned long long same = __ballot(ok);
    for (int b = 0; b < id_bits; ++b) {
      const unsigned long long set = __ballot(ok && ((e >> b) & 1));
      same &= ((e >> b) & 1) ? set : ~set;
    }
    if (ok) {
      const unsigned long long below = same & ((1ull << lane) - 1ull);
      const int row = mine[e] + __popcll(below);
      pos[i] = row;
      sorted_tok[row] = i / topk;
      if (sorted_w) sorted_w[row] = weights[i];
      // the wave runs in lockstep: every lane has read mine[e] before the last lane of its expert moves it on
      __builtin_amdgcn_wave_barrier();
      if ((same >> lane) == 1ull) mine[e] = row + 1;
      __builtin_amdgcn_wave_barrier();
    }
  }
}

__global__ __launch_bounds__(256) void moe_permute_kernel(const u32x4* __restrict__ x,
                                                          const int* __restrict__ sorted_tok,
                                                          u32x4* __restrict__ xs, int vec_per_row) {
  const int row = blockIdx.x;
  const int tok = sorted_tok[row];
  for (int i = threadIdx.x; i < vec_per_row; i += 256)
    xs[(long)row * vec_per_row + i] = x[(long)tok * vec_per_row + i];
}

__global__ __launch_bounds__(256) void moe_combine_kernel(const uint16_t* __restrict__ y,
                                                          const float* __restrict__ weights,
                                                          const int* __restrict__ pos,
                                                          uint16_t* __restrict__ out, int hidden,
                                                          int topk) {
  const int t = blockIdx.x;
  for (int i = threadIdx.x * 8; i < hidden; i += 256 * 8) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < topk; ++k) {
      const float w = weights[(long)t * topk + k];
      if (w == 0.f) continue;  // a pair of an expert held by another rank: its row was never written
      const long row = pos[(long)t * topk + k];
      const u32x4 a = *reinterpret_cast<const u32x4*>(y + row * hidden + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[2 * j] += w * bf16lo(a[j]);
        acc[2 * j + 1] += w * bf16hi(a[j]);
      }
    }
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = pack_bf16x2(acc[2 * j], acc[2 * j + 1]);
    *reinterpret_cast<u32x4*>(out + (long)t * hidden + i) = o;
  }
}

VPSA_EXPORT int vpsa_moe_topk_softmax(const void* logits, float* weights, int* ids, int tokens,
                                      int n_experts, int topk, int renorm, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (n_experts > MAX_EXPERTS || topk > MAX_TOPK || topk > n_experts) return -1;
#define TOPK(G)                                                                                                            \
  moe_topk_softmax_kernel<G><<<dim3((unsigned)(((long)tokens * G + 255) / 256)), dim3(256), 0, stream>>>(                  \
      (const uint16_t*)logits, weights, ids, tokens, n_experts, topk, renorm)
  if (n_experts <= 8) TOPK(8);
  else if (n_experts <= 16) TOPK(16);
  else if (n_experts <= 32) TOPK(32);
  else TOPK(64);
#undef TOPK
  return 0;
}

// x bf16 [tokens, hidden] (row stride elements), w bf16 [n_experts, hidden] contiguous, both on 16 bytes; hidden a multiple of 128, up to 64
// experts.  Nonzero for what the kernel does not take.
VPSA_EXPORT int vpsa_moe_router(const void* x, long x_stride, const void* w, void* logits, int tokens, int n_experts, int hidden,
                                hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (n_experts < 1 || n_experts > MAX_EXPERTS || hidden <= 0 || hidden % 128 != 0 || (x_stride & 7) || (((uintptr_t)x | (uintptr_t)w) & 15))
    return -1;
  const dim3 grid((tokens + 15) / 16);
#define ROUTER(ET) \
  moe_router_kernel<ET><<<grid, 256, 0, stream>>>((const uint16_t*)x, x_stride, (const uint16_t*)w, (uint16_t*)logits, tokens, n_experts, hidden)
  if (n_experts <= 16) ROUTER(1);
  else if (n_experts <= 32) ROUTER(2);
  else ROUTER(4);
#undef ROUTER
  return 0;
}

VPSA_EXPORT int vpsa_moe_align(const int* ids, int* offsets, int* pos, int* sorted_tok,
                               const float* weights, float* sorted_w, int n_pairs, int n_experts, int topk, hipStream_t stream) {
  if (n_experts < 1 || n_experts > ALIGN_MAX_EXPERTS || (sorted_w && !weights)) return -1;
  const size_t lds = (size_t)(ALIGN_WAVES + 1) * n_experts * sizeof(int);  // 68 KiB at the most
  static bool attr_set = false;
  if (lds > 48 * 1024 && !attr_set) {
    if (hipFuncSetAttribute((const void*)moe_align_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (ALIGN_WAVES + 1) * ALIGN_MAX_EXPERTS * (int)sizeof(int)) != hipSuccess)
      return -2;
    attr_set = true;
  }
  int id_bits = 0;
  while ((1 << id_bits) < n_experts) ++id_bits;
  hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(1024), lds, stream, ids, offsets, pos,
                     sorted_tok, weights, sorted_w, n_pairs, n_experts, topk, id_bits);
  return 0;
}

VPSA_EXPORT int vpsa_moe_permute(const void* x, const int* sorted_tok, void* xs, int rows,
                                 int hidden, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (hidden % 8 != 0) return -1;
  hipLaunchKernelGGL(moe_permute_kernel, dim3(rows), dim3(256), 0, stream, (const u32x4*)x,
                     sorted_tok, (u32x4*)xs, hidden / 8);
  return 0;
}

VPSA_EXPORT int vpsa_moe_combine(const void* y, const float* weights, const int* pos, void* out,
                                 int tokens, int hidden, int topk, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (hidden % 8 != 0) return -1;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(tokens), dim3(256), 0, stream, (const uint16_t*)y,
                     weights, pos, (uint16_t*)out, hidden, topk);
  return 0;
}

// ---------------------------------------------------------------------------------
// Small-batch expert MLP (decode): only the experts a token was routed to are read.
// Pair p = t * topk + k uses expert e = ids[p] on token t.  Both kernels are weight-streaming
// GEMVs: a wave owns ROWS output rows, every lane walks the reduction dimension in 16-byte
// chunks (ROWS (x2 for gate/up) independent 16-byte loads in flight per step), partial sums
// are combined with wave shuffles.  No host sync and no data-dependent launch shape, so the
// step stays capturable in a HIP graph.
//   gate_up: act[p, n] = silu(W13[e][n, :] . x[t]) * (W13[e][I + n, :] . x[t])     n < I
//   down:    y[p, h]   = W2[e][h, :] . act[p, :]                                    h < H
// grid = (ceil(rows / (4 * ROWS)), pairs), block = 256.
// ---------------------------------------------------------------------------------
#define GEMV_ROWS 4

__device__ __forceinline__ float dot8(u32x4 w, u32x4 a) {
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    s += bf16lo(w[j]) * bf16lo(a[j]);
    s += bf16hi(w[j]) * bf16hi(a[j]);
  }
  return s;
}

__global__ __launch_bounds__(256) void moe_gemv_gate_up_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w13, const int* __restrict__ ids,
    uint16_t* __restrict__ act, int hidden, int inter, int topk) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int p = blockIdx.y;
  const int t = p / topk;
  const int e = ids[p];
  const int n0 = (blockIdx.x * 4 + wave) * GEMV_ROWS;
  if (n0 >= inter) return;
  const int chunks = hidden >> 3;
  const u32x4* xv = reinterpret_cast<const u32x4*>(x + (long)t * hidden);
  const uint16_t* wbase = w13 + (long)e * 2 * inter * hidden;
  float g[GEMV_ROWS], u[GEMV_ROWS];
#pragma unroll
  for (int r = 0; r < GEMV_ROWS; ++r) g[r] = u[r] = 0.f;
  for (int c = lane; c < chunks; c += 64) {
    const u32x4 a = xv[c];
    u32x4 wg[GEMV_ROWS], wu[GEMV_ROWS];
#pragma unroll
    for (int r = 0; r < GEMV_ROWS; ++r) {
      const int n = n0 + r < inter ? n0 + r : inter - 1;
      // whole lines, read once per step: streaming loads (the matrix-core kernels below read half
      // lines per step and need the cache to hold the other half: plain loads there, measured)
      wg[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wbase + (long)n * hidden) + c);
      wu[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wbase + (long)(inter + n) * hidden) + c);
    }
#pragma unroll
    for (int r = 0; r < GEMV_ROWS; ++r) {
      g[r] += dot8(wg[r], a);
      u[r] += dot8(wu[r], a);
    }
  }
#pragma unroll
  for (int r = 0; r < GEMV_ROWS; ++r) {
    g[r] = wave_reduce_sum(g[r]);
    u[r] = wave_reduce_sum(u[r]);
  }
  if (lane < GEMV_ROWS && n0 + lane < inter) {
    float gv = 0.f, uv = 0.f;
#pragma unroll
    for (int r = 0; r < GEMV_ROWS; ++r)
      if (r == lane) { gv = g[r]; uv = u[r]; }
    // the library path rounds gate/up to bf16 before the activation: do the same
    gv = bf16_bits_to_f32(__builtin_bit_cast(uint16_t, (bf16_t)gv));
    uv = bf16_bits_to_f32(__builtin_bit_cast(uint16_t, (bf16_t)uv));
    const float s = gv / (1.f + __expf(-gv)) * uv;
    act[(long)p * inter + n0 + lane] = __builtin_bit_cast(uint16_t, (bf16_t)s);
  }
}

__global__ __launch_bounds__(256) void moe_gemv_down_kernel(
    const uint16_t* __restrict__ act, const uint16_t* __restrict__ w2, const int* __restrict__ ids,
    uint16_t* __restrict__ y, int hidden, int inter) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int p = blockIdx.y;
  const int e = ids[p];
  const int h0 = (blockIdx.x * 4 + wave) * GEMV_ROWS;
  if (h0 >= hidden) return;
  const int chunks = inter >> 3;
  const u32x4* av = reinterpret_cast<const u32x4*>(act + (long)p * inter);
  const uint16_t* wbase = w2 + (long)e * hidden * inter;
  float acc[GEMV_ROWS];
#pragma unroll
  for (int r = 0; r < GEMV_ROWS; ++r) acc[r] = 0.f;
  for (int c = lane; c < chunks; c += 64) {
    const u32x4 a = av[c];
    u32x4 w[GEMV_ROWS];
#pragma unroll
    for (int r = 0; r < GEMV_ROWS; ++r) {
      const int h = h0 + r < hidden ? h0 + r : hidden - 1;
      w[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wbase + (long)h * inter) + c);
    }
#pragma unroll
    for (int r = 0; r < GEMV_ROWS; ++r) acc[r] += dot8(w[r], a);
  }
#pragma unroll
  for (int r = 0; r < GEMV_ROWS; ++r) acc[r] = wave_reduce_sum(acc[r]);
  if (lane < GEMV_ROWS && h0 + lane < hidden) {
    float v = 0.f;
#pragma unroll
    for (int r = 0; r < GEMV_ROWS; ++r)
      if (r == lane) v = acc[r];
    y[(long)p * hidden + h0 + lane] = __builtin_bit_cast(uint16_t, (bf16_t)v);
  }
}

// x [tokens, hidden], w13 [E, 2*inter, hidden], w2 [E, hidden, inter], ids [tokens*topk]
// act [tokens*topk, inter] and y [tokens*topk, hidden] are caller-provided workspaces.
VPSA_EXPORT int vpsa_moe_gemv(const void* x, const void* w13, const void* w2, const int* ids,
                              void* act, void* y, int tokens, int topk, int hidden, int inter,
                              hipStream_t stream) {
  const int pairs = tokens * topk;
  if (pairs <= 0) return 0;
  if (hidden % 8 != 0 || inter % 8 != 0) return -1;
  const int per_block = 4 * GEMV_ROWS;
  hipLaunchKernelGGL(moe_gemv_gate_up_kernel, dim3((inter + per_block - 1) / per_block, pairs),
                     dim3(256), 0, stream, (const uint16_t*)x, (const uint16_t*)w13, ids,
                     (uint16_t*)act, hidden, inter, topk);
  hipLaunchKernelGGL(moe_gemv_down_kernel, dim3((hidden + per_block - 1) / per_block, pairs),
                     dim3(256), 0, stream, (const uint16_t*)act, (const uint16_t*)w2, ids,
                     (uint16_t*)y, hidden, inter);
  return 0;
}
