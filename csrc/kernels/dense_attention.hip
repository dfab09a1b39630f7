// Single-query attention over dense (unpaged) K/V for 64-channel heads: the decoder of a
// speech model attends with ONE new query per window to its own few hundred earlier positions
// and to the 1500 encoder positions of the window (cross-attention), both held as plain
// [window][position][head * 64] tensors.
//
// The work is a GEMV pair per (window, head): 2 x T x 64 bf16 values read once, no reuse, so the
// kernel is a streaming reduction, not an MFMA kernel.  One workgroup per (head, window); eight
// lanes share a key (16 bytes of the key row each: one 128-byte line per key and group), every
// group keeps four keys in flight, and each group runs its own online softmax (running maximum,
// denominator, 8 output channels per lane).  Groups are merged at the end, inside a wave with
// cross-lane moves, between waves through 2.5 KB of LDS.  Scores, probabilities and the output
// stay in fp32 registers; nothing but Q, K, V and the 64 outputs touches memory, where the same
// step written with library calls is five launches with [window, head, T] fp32 round trips.
//
// The number of valid positions is read from device memory (position counter + 1), so a captured
// HIP graph replays the same launch for every decode step.
#include <type_traits>

#include "common.h"

#define DA_KEYS 4  // keys in flight per 8-lane group

__device__ __forceinline__ void da_merge(float& m, float& l, float (&acc)[8], float m2, float l2,
                                         const float (&acc2)[8]) {
  const float mn = fmaxf(m, m2);
  const float a = __builtin_amdgcn_exp2f(m - mn), b = __builtin_amdgcn_exp2f(m2 - mn);
  l = l * a + l2 * b;
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = acc[i] * a + acc2[i] * b;
  m = mn;
}

template <int THREADS>
__global__ __launch_bounds__(THREADS) void dense_decode_attn_kernel(
    const uint16_t* __restrict__ q, long q_bs, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, long kv_bs, long kv_ts, const long* __restrict__ pos, int T,
    uint16_t* __restrict__ out, long o_bs, float scale_log2e) {
  constexpr int SLOTS = THREADS / 8, WAVES = THREADS / 64;
  __shared__ float merge[WAVES][8][10];
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const int c8 = tid & 7, slot = tid >> 3;
  int n = T;
  if (pos != nullptr) {
    const long p = pos[0] + 1;
    n = p < T ? (int)p : T;
  }
  float qf[8];
  {
    const u32x4 qw = *(const u32x4*)(q + b * q_bs + h * 64 + c8 * 8);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      qf[2 * i] = bf16lo(qw[i]) * scale_log2e;
      qf[2 * i + 1] = bf16hi(qw[i]) * scale_log2e;
    }
  }
  const uint16_t* kb = k + b * kv_bs + h * 64 + c8 * 8;
  const uint16_t* vb = v + b * kv_bs + h * 64 + c8 * 8;
  float m = -1e30f, l = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int base = 0; base < n; base += SLOTS * DA_KEYS) {
    u32x4 kk[DA_KEYS], vv[DA_KEYS];
    bool ok[DA_KEYS];
#pragma unroll
    for (int j = 0; j < DA_KEYS; ++j) {
      const int key = base + j * SLOTS + slot;
      ok[j] = key < n;
      const long off = (long)(ok[j] ? key : n - 1) * kv_ts;
      kk[j] = *(const u32x4*)(kb + off);
      vv[j] = *(const u32x4*)(vb + off);
    }
#pragma unroll
    for (int j = 0; j < DA_KEYS; ++j) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s = fmaf(qf[2 * i], bf16lo(kk[j][i]), s);
        s = fmaf(qf[2 * i + 1], bf16hi(kk[j][i]), s);
      }
      s += __shfl_xor(s, 1, 64);
      s += __shfl_xor(s, 2, 64);
      s += __shfl_xor(s, 4, 64);
      if (ok[j]) {
        const float mn = fmaxf(m, s);
        const float a = __builtin_amdgcn_exp2f(m - mn), p = __builtin_amdgcn_exp2f(s - mn);
        l = l * a + p;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[2 * i] = acc[2 * i] * a + p * bf16lo(vv[j][i]);
          acc[2 * i + 1] = acc[2 * i + 1] * a + p * bf16hi(vv[j][i]);
        }
        m = mn;
      }
    }
  }
  // the 8 groups of a wave: lanes that differ in bits 3..5 hold the same channels
#pragma unroll
  for (int off = 8; off < 64; off <<= 1) {
    const float m2 = __shfl_xor(m, off, 64), l2 = __shfl_xor(l, off, 64);
    float acc2[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc2[i] = __shfl_xor(acc[i], off, 64);
    da_merge(m, l, acc, m2, l2, acc2);
  }
  const int wave = tid >> 6, lane = tid & 63;
  if (lane < 8) {
    merge[wave][lane][0] = m;
    merge[wave][lane][1] = l;
#pragma unroll
    for (int i = 0; i < 8; ++i) merge[wave][lane][2 + i] = acc[i];
  }
  __syncthreads();
  if (tid < 8) {
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      float acc2[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc2[i] = merge[w][tid][2 + i];
      da_merge(m, l, acc, merge[w][tid][0], merge[w][tid][1], acc2);
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = pack_bf16x2(acc[2 * i] * inv, acc[2 * i + 1] * inv);
    *(u32x4*)(out + b * o_bs + h * 64 + tid * 8) = o;
  }
}

// q [B][heads * 64] (row stride q_bs elements), k / v [B][T][heads * 64] (strides kv_bs, kv_ts),
// out [B][heads * 64] (row stride o_bs); every row start 16-byte aligned.  pos: device pointer to
// the index of the newest valid position (positions 0..pos[0] are attended), or null for all T.
// Returns -1 for arguments the kernel does not cover.
VPSA_EXPORT int vpsa_dense_decode_attention(const void* q, long q_bs, const void* k, const void* v,
                                            long kv_bs, long kv_ts, const void* pos, int B, int heads,
                                            int T, void* out, long o_bs, float scale,
                                            hipStream_t stream) {
  if (B <= 0 || heads <= 0) return 0;
  if (T <= 0 || B > 65535 || (q_bs & 7) || (kv_bs & 7) || (kv_ts & 7) || (o_bs & 7)) return -1;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) return -1;
  const float sl = scale * 1.4426950408889634f;
  hipLaunchKernelGGL((dense_decode_attn_kernel<512>), dim3(heads, B), dim3(512), 0, stream,
                     (const uint16_t*)q, q_bs, (const uint16_t*)k, (const uint16_t*)v, kv_bs, kv_ts,
                     (const long*)pos, T, (uint16_t*)out, o_bs, sl);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

// ---------------------------------------------------------------------------------------------
// Bidirectional attention over dense Q/K/V for 64-channel heads (speech encoder: 1500 positions
// attending to each other; decoder prompt rows attending to the encoder output).
//
// One workgroup = 4 waves x 32 query rows (or 2 pairs of waves, below) against 64-key tiles staged through LDS (double
// buffered: the next tile is on its way to LDS during the current tile's math, one
// barrier per tile).  Per wave and tile:
//   S^T[64 keys x 32 queries] = K_tile . Q^T        8 x v_mfma_f32_32x32x16_bf16, K rows from LDS
//                                                   (ds_read_b128), Q^T fragments kept in registers
//   online softmax down each lane's column          lane (query, half) holds 32 of the 64 keys; one
//                                                   cross-half exchange per tile for the maximum
//   O^T[64 ch x 32 queries] += V_tile^T . P^T       8 MFMAs; P^T is the packed score registers as
//                                                   they are; V stays row-major in LDS and is read
//                                                   through the transposing ds_read_b64_tr_b16, whose
//                                                   4-key blocks are exactly the accumulator's key order
// A wave and tile cost 512 cycles of matrix instructions, 512 of exponentials and 640 of other vector work, in 1500 where the chip
// is full (32 windows x 12 heads), so vector work bounds this.  Rows of 128 B without padding (K's 16-byte chunks are swapped by key
// bits 1..3, V's halves by key bit 1: both kinds of read stay free of bank conflicts) and tiles that go to LDS without passing
// through registers (122 instead of 138) let four workgroups share a CU.  Of 8 windows x 12 heads 128 of 1152 workgroups are left behind
// the first 1024 (74.0 us by themselves); started behind them they come to lie on few CUs.  So they are cut in two (dense_attn_rows<true>: half the
// rows, a pair of waves shares them and takes every other tile, K's and V's two tiles loaded in turn) and 256 of the first 1024, one
// on each CU, go on with them: 84.2 -> 80.8 us, 88 pairs 79.9 -> 74.8, 22 windows x 8 heads 140.3 -> 135.4; with 256 or 512 left the halves share
// CUs and gain nothing (89.4 / 89.6, 106 / 111), so they stay whole.  Calls of up to 256 workgroups are cut as well where that pays (dense_blocks_cut): eight pairs 23.6 ->
// 15.8, 12 and 16 pairs 23.9 -> 22.3 (half of the halves share a CU; 24 pairs 34.2 / 34.2), four query rows of 64 pairs 21.9 -> 14.2.  (The
// two waves with 32 keys of every tile: 18.7 where this takes 17.7.)  (The next tile's scores under this one's exponentials need 182
// registers: two workgroups a CU, 23.4 us for one window instead of 26.5 but 91 for 8 and 305 for 32.)  The scale goes into the
// exponent's fused multiply, the mask only touches the last tile, and a window's query blocks run on one XCD.  Measured: 8
// windows x 12 heads x 1500 positions 153 -> 97 us, 2 windows 55.5 -> 41, 32 windows x 8 heads 324 -> 225.  Then, with the queries waited for before the loop, K read two products ahead, the mask in a tile of its
// own and a slice's products under the next slice's exponentials: 97.3 -> 94.1 (0.59 PFLOP/s), one window 31.0 -> 28.9, four
// query rows 32 -> 26, 32 windows x 8 heads 225 -> 219.  Then, with tiles straight into LDS and four workgroups instead of three:
// 93.1 -> 87.7, 32 windows x 12 heads 303 -> 284, two 38.7 -> 36.9, one 27.5 -> 26.5.  Then, with the maximum's halves exchanged by a
// lane swap instead of through LDS: 89.9 -> 88.2, 32 windows 308.8 -> 305.5, one 26.5 -> 24.3, four query rows 24.9 -> 22.9.  A
// maximum that follows only in steps of 2^8 is no faster and rounds the largest probability: error 1.9e-3 -> 2.3e-3.
// The [B, heads, Tq, Tk] score matrix never exists in memory.
#define DF_KT 64

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bf16x8 lds_tr_pair(const uint16_t* lo, const uint16_t* hi) {
  typedef __attribute__((address_space(3))) s16x4* lds_ptr;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)lo);
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)hi);
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// 16 bytes a lane from global memory into LDS, in lane order from `to`.  In assembly because the compiler waits for all loads of the builtin
// in front of any read from LDS; whoever reads what is loaded waits for it.  (A scalar register that a vector instruction wrote may be read
// five states later.)
__device__ __forceinline__ void load_to_lds(const void* src, uint32_t to) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(to) : "m0", "memory");
}
__device__ __forceinline__ uint32_t lds_address(const uint16_t* at) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint16_t*)at;
}

// The rows from row_of_block on of head h in window b.  PAIRS false: 128 rows, a wave takes 32 of them with all keys.  true: 64 rows, two
// waves share 32 of them, one takes the tiles of even number, the other those of odd number, and they meet in LDS at the end.
template <bool PAIRS>
__device__ __forceinline__ void dense_attn_rows(
    const uint16_t* __restrict__ q, long q_bs, long q_ts, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, long kv_bs, long kv_ts, uint16_t* __restrict__ out, long o_bs,
    long o_ts, int Tq, int Tk, int h, int b, int row_of_block, float scale_log2e, uint16_t (*lds_k)[DF_KT * 64], uint16_t (*lds_v)[DF_KT * 64]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 31, hf = lane >> 5;
  const int part = wave & 1;  // PAIRS
  const int qrow = row_of_block + (PAIRS ? wave >> 1 : wave) * 32 + r;
  const int qc = qrow < Tq ? qrow : Tq - 1;
  const uint16_t* qp = q + b * q_bs + (long)qc * q_ts + h * 64;
  bf16x8 qf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) qf[ks] = *(const bf16x8*)(qp + 16 * ks + 8 * hf);

  const uint16_t* kbase_p = k + b * kv_bs + h * 64;
  const uint16_t* vbase_p = v + b * kv_bs + h * 64;
  const int n_tiles = (Tk + DF_KT - 1) / DF_KT;
  // A wave's load is eight keys' rows: keys 8 wave .. and 32 further of a tile.  LDS is filled in lane order, so the chunks are swapped
  // on the way there: the source of chunk c of key j is K's c ^ (j / 2 % 8), V's c ^ (j % 4 / 2 * 4).
  const int row0 = 8 * wave + (lane >> 3);
  const int kc = 8 * ((lane & 7) ^ ((row0 >> 1) & 7)), vc = 8 * ((lane & 7) ^ ((row0 & 2) << 1));
  const long row_step = kv_ts * 32;
  const uint16_t *ksrc = kbase_p + row0 * kv_ts + kc, *vsrc = vbase_p + row0 * kv_ts + vc;
  auto stage = [&](int t) {
    const int buf = t & 1;
    const uint16_t *k1 = ksrc + row_step, *v1 = vsrc + row_step;
    if (t == n_tiles - 1) {  // keys past the last read the last one
      const long back0 = max(0, t * DF_KT + row0 - (Tk - 1)) * kv_ts, back1 = max(0, t * DF_KT + row0 + 32 - (Tk - 1)) * kv_ts;
      ksrc -= back0, vsrc -= back0, k1 -= back1, v1 -= back1;
    }
    const uint32_t kd = lds_address(&lds_k[buf][512 * wave]), vd = lds_address(&lds_v[buf][512 * wave]);
    load_to_lds(ksrc, kd);
    load_to_lds(vsrc, vd);
    load_to_lds(k1, kd + 4096);
    load_to_lds(v1, vd + 4096);
    ksrc = k1 + row_step, vsrc = v1 + row_step;
  };
  // PAIRS: tiles 2 i and 2 i + 1 of one operand
  auto stage_two = [&](int i, const uint16_t*& src, const uint16_t* base, int c, uint16_t (*to)[DF_KT * 64]) {
    const uint32_t at = lds_address(&to[0][512 * wave]);
    if (2 * i + 2 < n_tiles) {
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        load_to_lds(src, at + 4096 * x);
        src += row_step;
      }
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x) load_to_lds(base + min(128 * i + 32 * x + row0, Tk - 1) * kv_ts + c, at + 4096 * x);
    }
  };
  if constexpr (PAIRS) stage_two(0, ksrc, kbase_p, kc, lds_k);
  else stage(0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  // The queries have arrived before the loop: waited for at their first use inside it, every tile would wait there, and with them
  // for the tile that is being loaded.
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(qf[ks]));

  f32x16 o_acc[2];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb)
#pragma unroll
    for (int i = 0; i < 16; ++i) o_acc[cb][i] = 0.f;
  float m_run = -1e30f, l_run = 0.f;
  // transposed read: lane 4q + p of a 16-lane group points at row q, columns 4p..4p+3 of its block
  const int tr_row = (lane >> 2) & 3;
  const int tr_off = (4 * hf + tr_row) * 64 + ((16 * ((lane >> 4) & 1) + 4 * (lane & 3)) ^ ((tr_row & 2) << 4));
  const int k_off = r * 64, k_swz = (r >> 1) & 7;

  f32x16 s_acc[2];
  // scores of a tile at kt, its first key t * 64 where some are masked; returns what the sums so far have to be multiplied with
  auto scores = [&](const uint16_t* kt, int t, auto masked) {
    bf16x8 kf[8];  // the products follow the reads at a distance of two
    auto read_k = [&](int j) { kf[j] = *(const bf16x8*)(kt + 32 * (j >> 2) * 64 + k_off + 8 * ((2 * (j & 3) + hf) ^ k_swz)); };
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s_acc[kb][i] = 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j) read_k(j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j + 2 < 8) read_k(j + 2);
      __builtin_amdgcn_sched_barrier(0);
      s_acc[j >> 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[j], qf[j & 3], s_acc[j >> 2], 0, 0, 0);
    }
    // accumulator register i of block kb, half hf = key 64 t + 32 kb + 8 (i >> 2) + 4 hf + (i & 3)
    if (masked.value) {
      const int kbase = t * DF_KT;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (kbase + 32 * kb + 8 * (i >> 2) + 4 * hf + (i & 3) >= Tk) s_acc[kb][i] = -INFINITY;
    }
    float mx = -1e30f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s_acc[kb][i]);
    const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
    mx = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1])) * scale_log2e;
    const float m_new = fmaxf(m_run, mx);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    return alpha;
  };
  auto values = [&](const uint16_t* vt, float alpha) {
    bf16x8 vf[4][2];
    auto read_v = [&](int s4) {
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        const uint16_t* blk = vt + 16 * s4 * 64 + (tr_off ^ (32 * cb));
        vf[s4][cb] = lds_tr_pair(blk, blk + 8 * 64);
      }
    };
    float psum = 0.f;
    read_v(0);
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int i = 0; i < 16; ++i) o_acc[cb][i] *= alpha;
    // a slice's products run under the next one's exponentials
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      if (s4 + 1 < 4) read_v(s4 + 1);
      u32x4 pk;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(s_acc[s4 >> 1][8 * (s4 & 1) + 2 * jj], scale_log2e, -m_run));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(s_acc[s4 >> 1][8 * (s4 & 1) + 2 * jj + 1], scale_log2e, -m_run));
        psum += p0 + p1;
        pk[jj] = pack_bf16x2(p0, p1);
      }
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
        o_acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[s4][cb], __builtin_bit_cast(bf16x8, pk), o_acc[cb], 0, 0, 0);
    }
    l_run = l_run * alpha + psum;
  };
  if constexpr (PAIRS) {
    // V's two tiles are on their way during the scores, K's next two during the exponentials: each barrier ends the reads of the one
    // and shows that the other has landed.
    auto two = [&](int i, auto masked) {
      stage_two(i, vsrc, vbase_p, vc, lds_v);
      const float alpha = scores(lds_k[part], 2 * i + part, masked);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (!masked.value) stage_two(i + 1, ksrc, kbase_p, kc, lds_k);
      // (of an odd number of tiles the last one has no partner: its place holds repeats of the last key, whose values may be infinite)
      if (!masked.value || 2 * i + part < n_tiles) values(lds_v[part], alpha);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    };
    const int n = (n_tiles + 1) >> 1;
    for (int i = 0; i + 1 < n; ++i) two(i, std::false_type{});
    two(n - 1, std::true_type{});
  } else {
    auto tile = [&](int t, auto masked) {
      const int buf = t & 1;
      if (!masked.value) stage(t + 1);
      const float alpha = scores(lds_k[buf], t, masked);
      values(lds_v[buf], alpha);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next tile has landed
      __syncthreads();
    };
    for (int t = 0; t + 1 < n_tiles; ++t) tile(t, std::false_type{});
    tile(n_tiles - 1, std::true_type{});
  }
  // O^T accumulator register i of block cb, half hf = channel 32 cb + 8 (i >> 2) + 4 hf + (i & 3)
  float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  if constexpr (PAIRS) {  // (the tiles' places are free behind the last barrier: 34 values of 64 lanes, twice)
    float* const ex = reinterpret_cast<float*>(&lds_k[0][0]) + (wave >> 1) * (34 * 64) + lane;
    if (part) {
      ex[0] = m_run;
      ex[64] = l_tot;
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int i = 0; i < 16; ++i) ex[(2 + 16 * cb + i) * 64] = o_acc[cb][i];
    }
    __syncthreads();
    if (part) return;
    const float m = fmaxf(m_run, ex[0]), a0 = __builtin_amdgcn_exp2f(m_run - m), a1 = __builtin_amdgcn_exp2f(ex[0] - m);
    l_tot = l_tot * a0 + ex[64] * a1;
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int i = 0; i < 16; ++i) o_acc[cb][i] = o_acc[cb][i] * a0 + ex[(2 + 16 * cb + i) * 64] * a1;
  }
  if (qrow < Tq) {
    const float inv = 1.f / l_tot;
    uint16_t* op = out + b * o_bs + (long)qrow * o_ts + h * 64;
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        u32x2 w;
        w[0] = pack_bf16x2(o_acc[cb][4 * g4] * inv, o_acc[cb][4 * g4 + 1] * inv);
        w[1] = pack_bf16x2(o_acc[cb][4 * g4 + 2] * inv, o_acc[cb][4 * g4 + 3] * inv);
        *(u32x2*)(op + 32 * cb + 8 * g4 + 4 * hf) = w;
      }
  }
}

// Blocks of 128 rows, by `whole` workgroups (a multiple of 8); `left` blocks more in two of 64 each, by those workgroups from `first` on
// when they are done with theirs (whole 0: by workgroups of their own).  WHOLE, CUT: whether there are such.  (In one kernel with the other
// path the loop over whole tiles is scheduled otherwise: 200 keys, 288 workgroups 9.55 -> 10.4.)
template <bool WHOLE, bool CUT>
__global__ __launch_bounds__(256, 4) void dense_attn_fwd_kernel(
    const uint16_t* __restrict__ q, long q_bs, long q_ts, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, long kv_bs, long kv_ts, uint16_t* __restrict__ out, long o_bs,
    long o_ts, int Tq, int Tk, int heads, int pairs, int q_blocks, int whole, int first, int left, float scale_log2e) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[4][DF_KT * 64];
  // workgroups go round the eight XCDs: one pair's query blocks follow each other on one of them and share its L2
  const int xcd = blockIdx.x & 7;
  auto rows = [&](auto pairs_of_waves, int at, int row) {
    const int pair = at / q_blocks * 8 + xcd;
    row += at % q_blocks * 128;
    if (pair < pairs && row < Tq)
      dense_attn_rows<decltype(pairs_of_waves)::value>(q, q_bs, q_ts, k, v, kv_bs, kv_ts, out, o_bs, o_ts, Tq, Tk, pair % heads, pair / heads,
                                                       row, scale_log2e, lds, lds + 2);
  };
  if constexpr (WHOLE) rows(std::false_type{}, blockIdx.x >> 3, 0);  // (as many workgroups as there are)
  const int past = (int)blockIdx.x - first;
  if (CUT && past >= 0 && past < 2 * left) rows(std::true_type{}, (whole >> 3) + (past >> 4), (past >> 3 & 1) * 64);
}

// Blocks of 128 rows that are cut in two (microseconds whole / cut).  Behind whole rounds of four a CU: up to 128 of them, see above.  In calls
// that the chip holds at once a pair of waves spares half of the tiles and costs a wave's exchange.  Where every half has a CU to itself that pays from
// two tiles on with more than 64 rows (32 workgroups, 65 keys 5.43 / 5.00, 129 6.23 / 5.99, 1500 22.8 / 14.9), from four on with fewer, whose second half is
// empty (64 rows, 65 keys 4.80 / 4.97, 129 5.58 / 5.89, 200 6.34 / 6.03, 1500 22.0 / 14.7).  Up to 256 workgroups, whose halves share CUs, it does from 15
// tiles on (192 workgroups, 129 keys 6.6 / 7.6, 300 8.2 / 9.3, 700 13.0 / 13.6, 800 14.3 / 14.2 to 14.6, 1000 16.9 / 15.9, 1500 23.5 / 21.7; 256, 700 keys 13.4 / 14.2,
// 1000 17.4 / 16.5).
static int dense_blocks_cut(long pairs, int Tq, int Tk) {
  const long columns = (pairs + 7) / 8 * 8, groups = columns * ((Tq + 127) / 128), halves = columns * ((Tq + 63) / 64), left = groups % 1024;
  if (Tk <= DF_KT) return 0;
  if (groups >= 1024) return left <= 128 ? (int)left : 0;
  if (halves <= 256) return Tk > (Tq > 64 ? 1 : 3) * DF_KT ? (int)left : 0;
  return groups <= 256 && Tk > 14 * DF_KT ? (int)left : 0;
}
VPSA_EXPORT int vpsa_dense_attention_cut(int B, int heads, int Tq, int Tk) { return dense_blocks_cut((long)B * heads, Tq, Tk); }

// q [B][Tq][heads * 64], k / v [B][Tk][heads * 64], out [B][Tq][heads * 64]; strides in elements
// (batch, position), unit stride over channels, every row start 16-byte aligned (out: 8-byte).
// Every query attends to every key.  Returns -1 for arguments the kernel does not cover.
VPSA_EXPORT int vpsa_dense_attention(const void* q, long q_bs, long q_ts, const void* k, const void* v,
                                     long kv_bs, long kv_ts, void* out, long o_bs, long o_ts, int B,
                                     int heads, int Tq, int Tk, float scale, hipStream_t stream) {
  if (B <= 0 || heads <= 0 || Tq <= 0) return 0;
  if (Tk <= 0 || B > 65535 || heads > 65535) return -1;
  if ((q_bs & 7) || (q_ts & 7) || (kv_bs & 7) || (kv_ts & 7) || (o_bs & 3) || (o_ts & 3)) return -1;
  if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15) || ((uintptr_t)out & 7)) return -1;
  const int q_blocks = (Tq + 127) / 128;
  const long pairs = (long)B * heads, groups = (pairs + 7) / 8 * 8 * q_blocks;
  if (groups >= (1L << 31)) return -1;
  const int left = dense_blocks_cut(pairs, Tq, Tk);
  const int whole = (int)groups - left;
  auto* const kernel = left == 0 ? dense_attn_fwd_kernel<true, false> : whole == 0 ? dense_attn_fwd_kernel<false, true> : dense_attn_fwd_kernel<true, true>;
  hipLaunchKernelGGL(kernel, dim3(whole ? whole : 2 * left), dim3(256), 0, stream, (const uint16_t*)q, q_bs, q_ts, (const uint16_t*)k,
                     (const uint16_t*)v, kv_bs, kv_ts, (uint16_t*)out, o_bs, o_ts, Tq, Tk, heads, (int)pairs, q_blocks, whole, whole ? whole - 1024 : 0, left,
                     scale * 1.4426950408889634f);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}
