// Projections of a decode batch of up to 16 rows for gfx950, without partial sums in memory: y[M, N] = x[M, K] . W[N, K]^T.
// What bounds such a step is W's way through HBM and, beside it, launches that wait for each other: a split product needs another one to
// close it.  Here a workgroup's eight waves share the reduction among themselves, so that the product is whole in one launch, and what
// stands behind it (the stream's update; rotation and cache) is made in the same one.  The norm between two of them is taken apart: the product that
// updates the stream leaves the new rows times the norm's weights and the squares' sums of 16 channels each, and the next product
// applies a row's factor to its own sums.
//   * Weight rows go out in octets, two octets a tile; a workgroup takes a tile and goes on to its next one (at most one workgroup a CU).
//     Wave j multiplies chunks of 64 elements from its eighth of the row; the waves' sums meet in LDS, where one wave a tile adds them.
//   * A wave's weight rows come straight into a ring in LDS of its own (rows of 128 bytes, 16-byte chunk j of row r at j ^ (r ^ r / 8) % 8): no
//     barrier between load and use, 64 to 128 KiB a CU on their way, also across tiles and while the rows are normed.
//   * Token rows come through the ring beside the weights.  (Kept in registers as fragments, which are there before the first weights, 4096 x 4096
//     took 9.5 us with 1 row instead of 9.2, with 16 11.6 instead of 10.3; multiplied with the norm's weights on their way, 6144 x 4096 14.3
//     instead of 12.4.)
//   * Workgroups begin at different chunks of their eighths: rows whose length is a power of two put a chunk of all of them on the
//     same few memory channels.
// Beside mid_gemm.hip's split products and their reductions, figures at the dispatch in ops/__init__.py.
#include "common.h"

namespace {

constexpr int BK = 64, ROWB = BK * 2, WAVES = 8, CUS = 256;
constexpr int depth(int ai) { return ai == 2 ? 4 : 5; }  // stages of a wave's ring
constexpr int RED = WAVES * 1024;                        // the waves' sums of a tile
enum { ADD, QKV };

struct RowArgs {
  const uint16_t* x;
  long x_stride;
  const uint16_t* w;
  uint16_t* y;  // ADD: the residual stream [M, N]; QKV: the query rows
  int M, N, K;
  const uint16_t* norm;  // ADD: weight of the norm that follows, or null
  uint16_t* normed;      //      the new rows times it
  float* squares;        //      sums of the new rows' squares [M, N / 16]; QKV: of its own rows [M, K / 16]
  float eps;
  const uint16_t* bias;
  const int* positions;
  const long* slots;
  const float* cos_sin;
  uint16_t* cache;
  long page_stride, v_offset;
  int n_q, n_kv;
};

__device__ __forceinline__ int swz(int r) { return (r ^ (r >> 3)) & 7; }

// reads: -1, or 0 for loads that find nothing.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(const void* p, int reads) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, __builtin_amdgcn_readfirstlane(reads), 0x00020000);
}
__device__ __forceinline__ int positive(int v) { return ~((v - 1) >> 31); }  // -1 or 0, without a condition that would move to vector registers

// 16 bytes a lane from the resource's base + off + at straight to LDS, lane after lane.  Buffer loads: with global ones on their way the
// compiler has every load into a register wait for all of them.  POLICY: 2 = non-temporal.
template <int POLICY>
__device__ __forceinline__ void to_lds(__amdgpu_buffer_rsrc_t src, uint32_t off, uint32_t at, char* lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (__attribute__((address_space(3))) void*)lds, 16, off, at, 0, POLICY);
}

// AI: token rows in groups of 8.
template <int EPI, int AI>
__global__ __launch_bounds__(512, 1) void row_gemm_kernel(RowArgs a) {
  constexpr int STAGE = 2048 + AI * 1024, NL = 2 + AI, DEPTH = depth(AI);
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  char* ring = lds + wave * DEPTH * STAGE;
  char* sums = lds + WAVES * DEPTH * STAGE;
  const uint32_t row_bytes = a.K * 2, x_bytes = (uint32_t)a.x_stride * 2;
  const int chunks = a.K / BK, per = chunks / WAVES, extra = chunks % WAVES;
  const int n = per + (wave < extra ? 1 : 0), c0 = min(wave * per + min(wave, extra), chunks - 1);
  const int first = n > 0 ? (int)(blockIdx.x >> 3) % n : 0;
  const int row = min(c16, a.M - 1);  // rows past the last repeat it
  // An octet: 8 weight rows, or 4 channels and their 4 rotation partners.  Rounds of whole tiles over all workgroups, then what is left: single
  // octets where every workgroup can have one (not ADD: squares are summed by tiles).
  const int octets = a.N / 8, grid = gridDim.x, b = blockIdx.x, rounds = octets / (2 * grid), rest = octets - 2 * grid * rounds;
  const int step = EPI == QKV && rest <= grid ? 1 : 2, mine = rounds + (step * b < rest ? 1 : 0);
  auto octet_of = [&](int it) { return it < rounds ? 2 * (b + it * grid) : 2 * grid * rounds + step * b; };
  auto whole = [&](int it) { return positive(rounds - it) | (positive(step - 1) & positive(rest - 2 * b - 1)); };  // -1 or 0
  auto base_of = [&](int octet) {
    const long r = EPI == ADD ? (long)octet * 8 : (long)(octet >> 4) * HEAD_DIM + (octet & 15) * 4;
    return reinterpret_cast<const char*>(a.w) + r * row_bytes + c0 * ROWB;
  };

  // what the epilogue needs, before the ring's first loads: what is asked for first is here first
  int pos = 0;
  long slot = 0;
  f32x4 sq[2][2];
  if (EPI == QKV) {
    pos = a.positions[min(lane >> 2, a.M - 1)], slot = a.slots[row];
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // 256 sums of a row at a time, nothing past them
      const auto src = __builtin_amdgcn_make_buffer_rsrc(a.squares + (long)min(2 * wave + i, a.M - 1) * (a.K / 16), 0, a.K / 16 * 4, 0x00020000);
#pragma unroll
      for (int j = 0; j < 2; ++j) sq[i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(src, 16 * lane + 1024 * j, 0, 0));
    }
  }
  char* const beside_lds = sums + 2 * RED;
  float* const factor = reinterpret_cast<float*>(beside_lds + 4096);  // [16]

  uint32_t w_lane[2], x_lane[AI];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = lane >> 3;
    w_lane[i] = (EPI == ADD ? r + 8 * i : (r & 3) + 4 * i + (r >> 2) * 64) * row_bytes + (((lane & 7) ^ swz(8 * i + r)) << 4);
  }
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int r = 8 * i + (lane >> 3);
    x_lane[i] = (uint32_t)min(r, a.M - 1) * x_bytes + (((lane & 7) ^ swz(r)) << 4);
  }
  // The ring's loads: every step asks for one stage, past the last one for nothing, so that what is on its way always counts the same.
  int in_it = 0, in_at = first, in_slot = 0, in_left = mine * n;
  const char* in_base = base_of(octet_of(0));
  int in_whole = whole(0);
  auto load = [&]() {
    char* st = ring + in_slot;
    const int reads = positive(in_left);
    to_lds<2>(resource(in_base, reads), w_lane[0], in_at * ROWB, st);
    to_lds<2>(resource(in_base, reads & in_whole), w_lane[1], in_at * ROWB, st + 1024);
#pragma unroll
    for (int i = 0; i < AI; ++i)
      to_lds<0>(resource(reinterpret_cast<const char*>(a.x) + c0 * ROWB, reads), x_lane[i], in_at * ROWB, st + 2048 + i * 1024);
    --in_left;
    in_slot = in_slot == (DEPTH - 1) * STAGE ? 0 : in_slot + STAGE;
    in_at = in_at + 1 >= n ? 0 : in_at + 1;
    if (in_at == first) {
      ++in_it;
      in_base = base_of(octet_of(in_it));
      in_whole = whole(in_it);
    }
  };
#pragma unroll
  for (int i = 0; i < DEPTH; ++i) load();
  __builtin_amdgcn_sched_barrier(0);

  if (EPI == QKV) {  // a row's factor is there behind the first tile's barrier
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float tot = wave_reduce_sum(sq[i][0][0] + sq[i][0][1] + sq[i][0][2] + sq[i][0][3] + sq[i][1][0] + sq[i][1][1] + sq[i][1][2] + sq[i][1][3]);
      if (lane == 0) factor[2 * wave + i] = rsqrtf(tot / (float)a.K + a.eps);
    }
    asm volatile("" : "+v"(pos), "+v"(slot));  // (waited for here, where the loads behind them are counted)
  }
  const int fr = c16 * ROWB, f2[2] = {(g ^ swz(c16)) << 4, ((4 + g) ^ swz(c16)) << 4};
  const int rx = AI == 1 ? c16 & 7 : c16;  // (rows past the groups of 8 that were loaded repeat the group's)
  int out_slot = 0;
  f32x4 acc;
  auto multiply = [&]() {
    // my oldest stage has landed: all loads but those of the stages behind it
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * NL) : "memory");
    const char* st = ring + out_slot;
    bf16x8 wf[2], xf[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      wf[s] = *reinterpret_cast<const bf16x8*>(st + fr + f2[s]);
      xf[s] = *reinterpret_cast<const bf16x8*>(st + 2048 + rx * ROWB + (((4 * s + g) ^ swz(rx)) << 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    load();
#pragma unroll
    for (int s = 0; s < 2; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s], xf[s], acc, 0, 0, 0);
    out_slot = out_slot == (DEPTH - 1) * STAGE ? 0 : out_slot + STAGE;
  };

  for (int it = 0; it < mine; ++it) {
    const int octet = octet_of(it);
    const bool two = whole(it) != 0;
    const int oct = octet + (two ? g >> 1 : 0);                      // this lane's octet,
    const int head = oct >> 4, ch = (oct & 15) * 4 + (g & 1) * 64;  // and, QKV, its head and channels: lanes 16 away hold the rotation partners
    acc = (f32x4){0.f, 0.f, 0.f, 0.f};
    // What the sums meet, a piece of 16 bytes a lane, comes straight to LDS as well, asked for by the wave that will add: of token row l / 4 the
    // cosines and sines of its octets' channels; of row l / 2 of the residual stream the octets, and of the norm's weights.  (A load into registers
    // would have to be waited for behind all of the next tile's.)
    char* const beside = beside_lds + (it & 1) * 2048;
    if (wave == (it & (WAVES - 1))) {
      if (EPI == QKV) {
        const int o = min(octet + (lane & 1), octets - 1) & 15;
        to_lds<0>(resource(a.cos_sin, -1), (uint32_t)pos * (HEAD_DIM * 4) + (lane & 2) * 128 + o * 16, 0, beside);
      } else {
        to_lds<0>(resource(a.y, -1), (uint32_t)((min(lane >> 1, a.M - 1) * (long)a.N + min(octet + (lane & 1), octets - 1) * 8) * 2), 0, beside);
        if (a.norm != nullptr) to_lds<0>(resource(a.norm, -1), (uint32_t)min(octet + (lane & 1), octets - 1) * 16, 0, beside + 1024);
      }
    }
    for (int f = 0; f < n; ++f) multiply();
    f32x4* red = reinterpret_cast<f32x4*>(sums + (it & 1) * RED);
    red[wave * 64 + lane] = acc;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // one wave a tile adds: it is done with the buffer before the next barrier, and others write to it behind that one
    if (wave != (it & (WAVES - 1))) continue;
    if (n < DEPTH) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (else the loads behind those beside the sums have been waited for)
    f32x4 s = red[lane];
#pragma unroll
    for (int j = 1; j < WAVES; ++j) s += red[j * 64 + lane];
    const bool mine_too = c16 < a.M && (two || g < 2);
    if (EPI == ADD) {
      const u32x2 old = *reinterpret_cast<const u32x2*>(beside + c16 * 32 + g * 8);
      const u32x2 h = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
      const u32x2 r = {pack_bf16x2(bf16lo(h[0]) + bf16lo(old[0]), bf16hi(h[0]) + bf16hi(old[0])),
                       pack_bf16x2(bf16lo(h[1]) + bf16lo(old[1]), bf16hi(h[1]) + bf16hi(old[1]))};
      const long at = (long)c16 * a.N + oct * 8 + 4 * (g & 1);
      if (mine_too) *reinterpret_cast<u32x2*>(a.y + at) = r;
      if (a.norm == nullptr) continue;
      const u32x2 nw = *reinterpret_cast<const u32x2*>(beside + 1024 + g * 8);
      const float v[4] = {bf16lo(r[0]), bf16hi(r[0]), bf16lo(r[1]), bf16hi(r[1])};
      if (mine_too)
        *reinterpret_cast<u32x2*>(a.normed + at) = (u32x2){pack_bf16x2(v[0] * bf16lo(nw[0]), v[1] * bf16hi(nw[0])),
                                                           pack_bf16x2(v[2] * bf16lo(nw[1]), v[3] * bf16hi(nw[1]))};
      float ss = v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
      const auto far = __builtin_amdgcn_permlane32_swap(__float_as_uint(ss), __float_as_uint(ss), false, false);
      ss = __uint_as_float(far[0]) + __uint_as_float(far[1]);
      const auto near = __builtin_amdgcn_permlane16_swap(__float_as_uint(ss), __float_as_uint(ss), false, false);
      ss = __uint_as_float(near[0]) + __uint_as_float(near[1]);
      if (g == 0 && c16 < a.M) a.squares[(long)c16 * (a.N / 16) + octet / 2] = ss;
      continue;
    }
    s *= factor[c16];
    if (a.bias != nullptr) {
      const u32x2 bb = *reinterpret_cast<const u32x2*>(a.bias + head * HEAD_DIM + ch);
      s += (f32x4){bf16lo(bb[0]), bf16hi(bb[0]), bf16lo(bb[1]), bf16hi(bb[1])};
    }
    u32x2 v = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])}, p;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const auto sw = __builtin_amdgcn_permlane16_swap(v[r], v[r], false, false);
      p[r] = g & 1 ? sw[0] : sw[1];
    }
    if (!mine_too) continue;
    if (head < a.n_q + a.n_kv) {
      const f32x4 cs = *reinterpret_cast<const f32x4*>(beside + c16 * 64 + (g >> 1) * 16), sn = *reinterpret_cast<const f32x4*>(beside + c16 * 64 + 32 + (g >> 1) * 16);
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float me = r & 1 ? bf16hi(v[r >> 1]) : bf16lo(v[r >> 1]), other = r & 1 ? bf16hi(p[r >> 1]) : bf16lo(p[r >> 1]);
        o[r] = g & 1 ? rope_hi(other, me, cs[r], sn[r]) : rope_lo(me, other, cs[r], sn[r]);
      }
      v = (u32x2){pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
    }
    if (head < a.n_q) {
      *reinterpret_cast<u32x2*>(a.y + ((long)c16 * a.n_q + head) * HEAD_DIM + ch) = v;
      continue;
    }
    if (slot < 0) continue;
    uint16_t* page = a.cache + slot / PAGE * a.page_stride;
    const int off = (int)(slot % PAGE);
    if (head < a.n_q + a.n_kv) {
      *reinterpret_cast<u32x2*>(page + (long)(head - a.n_q) * PAGE * HEAD_DIM + k_elem_off(off, ch)) = v;
    } else {
      uint16_t* vd = page + a.v_offset + (long)(head - a.n_q - a.n_kv) * HEAD_DIM * PAGE;
#pragma unroll
      for (int r = 0; r < 4; ++r) vd[v_elem_off(ch + r, off)] = (uint16_t)(v[r >> 1] >> (16 * (r & 1)));
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing is on its way to LDS when the wave ends
}

template <int EPI, int AI>
int launch(const RowArgs& a, hipStream_t stream) {
  constexpr int LDS = WAVES * depth(AI) * (2048 + AI * 1024) + 2 * RED + 4096 + 64;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)row_gemm_kernel<EPI, AI>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return -2;
    attr_set = true;
  }
  const int tiles = a.N / 16;
  return launched(row_gemm_kernel<EPI, AI>, dim3(tiles < CUS ? tiles : CUS), 512, LDS, stream, a);
}

// Shapes that the kernels take (offsets within the weights have 32 bits).
bool takes(int M, int N, int K) { return M >= 1 && M <= 16 && N >= 16 && N % 16 == 0 && K >= BK && K % BK == 0 && (long)N * K * 2 < (1L << 32); }

bool reads(const RowArgs& a) {
  return a.x_stride >= a.K && !(a.x_stride & 7) && a.x_stride < (1L << 26) && !(((uintptr_t)a.x | (uintptr_t)a.w | (uintptr_t)a.y) & 15);
}

}  // namespace

VPSA_EXPORT int vpsa_row_gemm_takes(int M, int N, int K) { return takes(M, N, K); }

// residual [M, N] += x W^T: x [M, K] (row stride xs elements), w [N, K] contiguous; the product is rounded to 16 bits before the sum.  norm [N]
// or null: also normed [M, N] = the new rows * norm, and squares [M, N / 16], sums of 16 of the new rows' squares.
VPSA_EXPORT int vpsa_row_add(const void* x, long xs, const void* w, void* residual, const void* norm, void* normed, float* squares, int M,
                             int N, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  RowArgs a{};
  a.x = (const uint16_t*)x, a.x_stride = xs, a.w = (const uint16_t*)w, a.y = (uint16_t*)residual, a.M = M, a.N = N, a.K = K;
  a.norm = (const uint16_t*)norm, a.normed = (uint16_t*)normed, a.squares = squares;
  if (!takes(M, N, K) || !reads(a) || (((uintptr_t)norm | (uintptr_t)normed) & 15) || ((uintptr_t)squares & 3)) return -1;
  return M <= 8 ? launch<ADD, 1>(a, stream) : launch<ADD, 2>(a, stream);
}

// q | k | v = h W^T (+ bias) of one token per sequence, h = x times its rows' factors 1 / sqrt(sum of squares / K + eps), squares [M, K / 16], K up
// to 8192: q rotated to q_out [M, n_q * 128], k rotated and v to the cache (layer base `cache`; slots < 0: nowhere).
VPSA_EXPORT int vpsa_row_qkv(const void* x, long xs, const float* squares, float eps, const void* w, const void* bias, void* q_out, int M, int K,
                             const int* positions, const long* slots, const float* cos_sin, void* cache, long page_stride, long v_offset,
                             int n_q, int n_kv, hipStream_t stream) {
  if (M <= 0) return 0;
  RowArgs a{};
  a.x = (const uint16_t*)x, a.x_stride = xs, a.w = (const uint16_t*)w, a.squares = const_cast<float*>(squares), a.eps = eps, a.y = (uint16_t*)q_out;
  a.M = M, a.N = (n_q + 2 * n_kv) * HEAD_DIM, a.K = K, a.bias = (const uint16_t*)bias, a.positions = positions, a.slots = slots;
  a.cos_sin = cos_sin, a.cache = (uint16_t*)cache, a.page_stride = page_stride, a.v_offset = v_offset, a.n_q = n_q, a.n_kv = n_kv;
  if (!takes(M, a.N, K) || K > 8192 || !reads(a) || (((uintptr_t)bias | (uintptr_t)cache) & 7) || (((uintptr_t)cos_sin | (uintptr_t)squares) & 15) ||
      ((page_stride | v_offset) & 3))
    return -1;
  return M <= 8 ? launch<QKV, 1>(a, stream) : launch<QKV, 2>(a, stream);
}
