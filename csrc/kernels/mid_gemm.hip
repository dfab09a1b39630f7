// Projections of up to a few hundred token rows for gfx950: y[M, N] = x[M, K] . W[N, K]^T, the sizes of decode batches and of a new
// turn's prompt.  Too few rows for 256 x 256 tiles (a tile would be mostly padding and too few CUs would stream the weights):
// the job is to pull W through HBM once at full rate, with the token rows beside it.
//   * A workgroup owns 128 weight rows (PAIR: 64 gate and the 64 matching up rows) and up to 128 token rows; the reduction is
//     split over workgroups until about every CU has one (splits of whole 64-element chunks, not necessarily equal).
//   * Both operands go from memory straight into LDS (rows of 128 bytes, 16-byte chunk j of row r at j ^ (r ^ r / 8) % 8, so that
//     the 16 rows of a fragment cover all banks), four stages of which three are on their way: 54 to 96 KiB a CU in flight.
//   * One barrier a chunk, counted waits.  A wave multiplies 32 weight rows with all token tiles on v_mfma_f32_16x16x32_bf16;
//     its accumulators hold four consecutive outputs of a token, as in the streaming kernel of gemm.hip, whose reduction
//     (partial sums in 32 bits, fixed order) closes a split product.
//   * Workgroups start at different chunks of their range (see `first`).
//   * What bounds it: HBM up to 64 rows.  Beyond, LDS: with eight token tiles a chunk is 32 KiB in and 80 KiB out beside 512 cycles of
//     products, in 1700 to 1900 cycles (activations that a CU's first-level cache holds are no faster).
// 28672 x 4096 with the gated unit: 8 rows 45.2 -> 37.5 us (6.26 TB/s of weights), 64 rows 57.2 -> 40.1, 97 rows 60.6 -> 48.2; 128256 x
// 4096, 8 rows: 191 -> 161 (6.5 TB/s); 4096 x 14336, 88 rows: 50.1 -> 31.  The whole range stands at the dispatch in ops/__init__.py.
#include "common.h"
#include "mid_reduce.h"

namespace {

constexpr int BN = 128, BK = 64, STAGES = 4, ROWB = BK * 2;

__device__ __forceinline__ int swz(int r) { return (r ^ (r >> 3)) & 7; }

// The chunk of its n that a workgroup begins with: those of the XCDs an eighth of the row apart, and within an XCD, whose workgroups'
// numbers are eight apart, three.  With 3 * block an XCD's workgroups meet on the eighths of a row of 64 chunks (28672 x 4096, 1 to
// 40 rows, 39.3 -> 38.5 us), all of them on one chunk of a range of eight (4096 x 4096 in eight ranges, 1 / 64 rows 10.3 -> 10.0 / 14.4 -> 13.8),
// and beyond 48 rows ranges are far slower (8192 x 28672, 128 rows 135 -> 109; 3584 x 18944 49.3 -> 40.3).  But it stays where it is the
// better one.  `whole`: unsplit products with rows of 128 chunks and more, where it spreads an XCD over all of the row (28672 x 8192,
// 8 / 64 rows 74 / 77 against 83 / 84), or of more than a round of workgroups, which get out of step by themselves (57344 x 8192 145 / 149
// against 166 / 176; 128256 x 4096, 96 rows 195 against 200).  And ranges of fewer than 16 chunks that have no whole eighths (2560 x 9728 in
// twelve, 128 rows 22.8 against 23.4).
__host__ __device__ __forceinline__ int first_chunk(int block, int n, bool whole) {
  const int eighth = n / 8;
  if (whole || (n < 16 && (n & 7))) return block * 3 % n;
  return ((block >> 3) * 3 + (block & 7) * (eighth - (eighth % 3 == 0))) % n;  // (threes and a multiple of three would meet)
}

// acc[i][t] += W tile i of the wave x token tile t over chunks [0, n) of both operands: NA * 64 weight rows and MT * 16 token rows a
// chunk, all of it in LDS stages.  The weight rows lie w_row bytes apart from wp on, those from the 64th on w_half further; xrow(r): bytes
// from xp to row r's first chunk; arow: the wave's weight tiles (rows within the workgroup's).  POLICY of the weight loads: 2 =
// non-temporal.  Nothing is on its way or read any more on return.
template <int MT, int NA, int POLICY, typename XRow>
__device__ __forceinline__ void stream_product(const char* __restrict__ wp, uint32_t w_row, long w_half, const char* __restrict__ xp,
                                               XRow xrow, int n, int first, char* lds, const int (&arow)[NA],
                                               f32x4 (&acc)[NA][MT]) {
  constexpr int WI = 2 * NA;        // KiB of weight rows that a wave loads of a stage
  constexpr int XI = (MT + 1) / 2;  // and of token rows (the last ones twice where MT is odd)
  constexpr int NL = WI + XI;       // loads of a stage
  constexpr int BN = 64 * NA, STAGE = (BN + 16 * MT) * ROWB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  // what this lane loads: 8 rows of 8 chunks a KiB
  uint32_t woff[WI], xoff[XI];
  int xlds[XI];
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = 8 * (4 * i + wave) + (lane >> 3);
    woff[i] = (r & 63) * w_row + (((lane & 7) ^ swz(r)) << 4);
  }
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int kib = min(4 * i + wave, 2 * MT - 1), r = 8 * kib + (lane >> 3);
    xoff[i] = xrow(r) + (((lane & 7) ^ swz(r)) << 4);
    xlds[i] = BN * ROWB + kib * 1024;
  }
  auto load = [&](int i_c) {
    char* st = lds + (i_c & (STAGES - 1)) * STAGE;
    const int c = i_c + first < n ? i_c + first : i_c + first - n;
#pragma unroll
    for (int i = 0; i < WI; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wp + (i >> 1) * w_half + (long)c * ROWB + woff[i]),
                                       (__attribute__((address_space(3))) void*)(st + (4 * i + wave) * 1024), 16, 0, POLICY);
#pragma unroll
    for (int i = 0; i < XI; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(xp + (long)c * ROWB + xoff[i]),
                                       (__attribute__((address_space(3))) void*)(st + xlds[i]), 16, 0, 0);
  };
  // fragments: row c16 of a 16-row tile, chunk 4 ks + g; swz(16 m + c16) = swz(c16) ^ (2 m) % 8: a tile's number moves its chunks
  // by an even step
  const int fr = c16 * ROWB, f[2] = {(g ^ swz(c16)) << 4, ((4 + g) ^ swz(c16)) << 4};
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[i][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int c = 0; c < STAGES - 1 && c < n; ++c) load(c);
  for (int c = 0; c < n; ++c) {
    // chunk c has landed (mine: all but the loads of the two chunks behind it) and my reads of chunk c - 1 are done;
    // everyone's: the barrier
    if (c + 2 < n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * NL) : "memory");
    else if (c + 1 < n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NL) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (c + STAGES - 1 < n) load(c + STAGES - 1);
    __builtin_amdgcn_sched_barrier(0);
    // The products follow the reads at a distance of two token tiles.  Left to itself the compiler reads two tiles and waits for both
    // (28672 x 4096 with 97 rows, eight tiles 55 us, seven 58); all of the chunk's reads before its products: 54 with seven, 57 with eight;
    // at two or four tiles' distance 48 and 51.
    const char* st = lds + (c & (STAGES - 1)) * STAGE;
    bf16x8 a[2][NA], b[2 * MT];
    auto read_a = [&](int ks) {
#pragma unroll
      for (int i = 0; i < NA; ++i)
        a[ks][i] = *reinterpret_cast<const bf16x8*>(st + arow[i] * ROWB + fr + (f[ks] ^ ((2 * (arow[i] >> 4) & 7) << 4)));
    };
    auto read_b = [&](int j) {  // token tile j % MT of the chunk's half j / MT
      b[j] = *reinterpret_cast<const bf16x8*>(st + (BN + 16 * (j % MT)) * ROWB + fr + (f[j / MT] ^ ((2 * (j % MT) & 7) << 4)));
    };
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (j % MT == 0) read_a(j / MT);
      read_b(j);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j) {
      if (j + 2 < 2 * MT) {
        if (j + 2 == MT) read_a(1);
        read_b(j + 2);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < NA; ++i)
        acc[i][j % MT] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j / MT][i], b[j], acc[i][j % MT], 0, 0, 0);
    }
  }
  __syncthreads();
}

// FACTORS (unsplit, one token tile): squares are sums of 16 squares of the rows behind x [M, K / 16], K up to 8192; a row's factor 1 /
// sqrt(their sum / K + eps) is applied to its outputs.
template <int MT, bool PAIR, bool FACTORS = false>
__global__ __launch_bounds__(256, 1) void mid_gemm_kernel(const uint16_t* __restrict__ x, long x_stride,
                                                          const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias,
                                                          uint16_t* __restrict__ y, long y_stride, float* __restrict__ ws, int M,
                                                          int N, int K, int S, const float* __restrict__ squares, float eps) {
  // weights are read once: non-temporal loads, except where the partial sums of many rows want the memory-side cache as well
  constexpr int POLICY = PAIR || MT <= 3 ? 2 : 0;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  const int n_out = PAIR ? N >> 1 : N;
  const int n0 = blockIdx.x * (PAIR ? BN / 2 : BN), m0 = blockIdx.z * 128;
  const int chunks = K / BK, per = chunks / S, extra = chunks % S, sp = blockIdx.y;
  const int c0 = sp * per + min(sp, extra), n = per + (sp < extra ? 1 : 0);
  const int mrows = min(M - m0, 16 * MT);
  const int arow[2] = {PAIR ? 16 * wave : 32 * wave, PAIR ? 64 + 16 * wave : 32 * wave + 16};
  f32x4 acc[2][MT];
  // a wave sums four rows' squares; asked for before the stream, used behind it
  f32x4 sq[4][2];
  if constexpr (FACTORS)
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // 256 sums of a row at a time, nothing past them
      const auto src = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(squares) + (long)min(4 * wave + i, M - 1) * (K / 16), 0, K / 16 * 4, 0x00020000);
#pragma unroll
      for (int j = 0; j < 2; ++j) sq[i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(src, 16 * lane + 1024 * j, 0, 0));
    }
  // Workgroups walk their chunks from different ones on (first_chunk): rows whose length is a power of two put a chunk of all 128 rows on
  // the same few memory channels, and workgroups in step would meet there (28672 x 4096: 44.7 -> 39.5 us, 128256 x 4096: 205 -> 160).
  stream_product<MT, 2, POLICY>(
      reinterpret_cast<const char*>(w + (long)n0 * K) + (long)c0 * ROWB, (uint32_t)(K * 2), (PAIR ? n_out : 64) * (long)(K * 2),
      reinterpret_cast<const char*>(x + (long)m0 * x_stride) + (long)c0 * ROWB,
      [&](int r) { return (uint32_t)(min(r, mrows - 1) * (int)(x_stride * 2)); },  // rows past the last repeat it
      n, n > 0 ? first_chunk(blockIdx.x, n, S == 1 && (n >= 128 || gridDim.x > 256)) : 0, lds, arow, acc);
  if constexpr (FACTORS) {
    float* const factor = reinterpret_cast<float*>(lds);  // (nothing reads or loads there any more)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float tot = wave_reduce_sum(sq[i][0][0] + sq[i][0][1] + sq[i][0][2] + sq[i][0][3] + sq[i][1][0] + sq[i][1][1] + sq[i][1][2] + sq[i][1][3]);
      if (lane == 0) factor[4 * wave + i] = rsqrtf(tot / (float)K + eps);
    }
    __syncthreads();
    acc[0][0] *= factor[c16], acc[1][0] *= factor[c16];
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int j = 16 * t + c16;
    if (j >= mrows) continue;
    if (S > 1) {
      float* p = ws + ((long)sp * M + m0 + j) * N;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        *reinterpret_cast<f32x4*>(p + n0 + (PAIR ? 16 * wave + i * n_out : arow[i]) + 4 * g) = acc[i][t];
    } else if (PAIR) {
      f32x4 s = acc[0][t];
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = s[r] / (1.f + __expf(-s[r])) * acc[1][t][r];
      const u32x2 o = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
      *reinterpret_cast<u32x2*>(y + (long)(m0 + j) * y_stride + n0 + 16 * wave + 4 * g) = o;
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int col = n0 + arow[i] + 4 * g;
        f32x4 s = acc[i][t];
        if (bias != nullptr) {
          const u32x2 bb = *reinterpret_cast<const u32x2*>(bias + col);
          s[0] += bf16lo(bb[0]);
          s[1] += bf16hi(bb[0]);
          s[2] += bf16lo(bb[1]);
          s[3] += bf16hi(bb[1]);
        }
        const u32x2 o = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
        *reinterpret_cast<u32x2*>(y + (long)(m0 + j) * y_stride + col) = o;
      }
    }
  }
}

// The experts of a decode-sized batch: every routed expert's weights are streamed once against its rows (more than 16 MT rows: once
// for each 16 MT).  UNIT: grid (inter / 64, experts), act[row] = unit(gate, up) of x[sorted_tok[row]], rows sorted by expert; act_limit >
// 0: min(g, limit) * sigmoid(alpha g) * (clamp(u) + bias), else silu(g) * u; row_scale: factors of gate and up.  Else grid
// (hidden / 64, experts), y[row] = W2 act[row] (64 weight rows a workgroup: with 128 a layer's 4096 rows leave one workgroup per CU
// and no slack for experts without rows).
// Against 16-row tiles that went from memory into registers, 64 bytes a row and load, 8 experts of 28672 x 4096 and 4096 x
// 14336: 540 -> 435 us a mixture of 16 tokens, 283 -> 248 of 4; a decode step of two layers, 8 tokens 1105 -> 921, 48 tokens 1420 -> 1116.
template <int MT, bool UNIT>
__global__ __launch_bounds__(256, 1) void mid_experts_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                             const int* __restrict__ offsets, const int* __restrict__ sorted_tok,
                                                             uint16_t* __restrict__ y, int N, int K, float act_limit,
                                                             float act_alpha, float act_bias, const float* __restrict__ row_scale) {
  constexpr int NA = UNIT ? 2 : 1;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int e = blockIdx.y, r0 = offsets[e], n_e = offsets[e + 1] - r0;
  if (n_e <= 0) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  const int n_out = UNIT ? N >> 1 : N, n0 = blockIdx.x * 64, n = K / BK;
  int arow[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) arow[i] = 64 * i + 16 * wave;
  for (int m0 = 0; m0 < n_e; m0 += 16 * MT) {
    const int last = min(n_e - m0, 16 * MT) - 1;
    f32x4 acc[NA][MT];
    stream_product<MT, NA, 2>(
        reinterpret_cast<const char*>(w + ((long)e * N + n0) * K), (uint32_t)(K * 2), n_out * (long)(K * 2),
        reinterpret_cast<const char*>(UNIT ? x : x + (long)(r0 + m0) * K),
        [&](int r) { return (uint32_t)(UNIT ? sorted_tok[r0 + m0 + min(r, last)] : min(r, last)) * (uint32_t)(K * 2); },
        n, (first_chunk(blockIdx.x, n, false) + e) % n, lds, arow, acc);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int j = 16 * t + c16;
      if (j > last) continue;
      const long row = r0 + m0 + j;
      f32x4 s = acc[0][t];
      if (UNIT) {
        const float rs = row_scale ? row_scale[row] : 1.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float gt = s[r] * rs, up = acc[NA - 1][t][r] * rs;
          if (act_limit > 0.f) {
            gt = fminf(gt, act_limit);
            up = fminf(fmaxf(up, -act_limit), act_limit) + act_bias;
            s[r] = gt / (1.f + __expf(-act_alpha * gt)) * up;
          } else {
            s[r] = gt / (1.f + __expf(-gt)) * up;
          }
        }
      }
      const u32x2 o = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
      *reinterpret_cast<u32x2*>(y + row * n_out + n0 + 16 * wave + 4 * g) = o;
    }
  }
}

// out[m, n .. n + 3] = epilogue(sum_s ws[s, m, n .. n + 3]); one thread per 4 output columns, eight partials in flight.
template <bool PAIR>
__global__ __launch_bounds__(256) void mid_reduce_kernel(const float* __restrict__ ws, const uint16_t* __restrict__ bias,
                                                         uint16_t* __restrict__ y, long y_stride, int M, int N, int S) {
  const int n_out = PAIR ? N >> 1 : N;
  const int col = (blockIdx.x * 256 + threadIdx.x) * 4, m = blockIdx.y;
  if (col >= n_out) return;
  const float* p = ws + (long)m * N + col;
  const long step = (long)M * N;
  f32x4 s = {0.f, 0.f, 0.f, 0.f}, s2 = s;
  for (int i0 = 0; i0 < S; i0 += 8) {
    f32x4 v[8], v2[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const long at = (long)min(i0 + i, S - 1) * step;
      v[i] = *reinterpret_cast<const f32x4*>(p + at);
      if (PAIR) v2[i] = *reinterpret_cast<const f32x4*>(p + at + n_out);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i0 + i < S) {
        s += v[i];
        if (PAIR) s2 += v2[i];
      }
  }
  if (PAIR) {
#pragma unroll
    for (int r = 0; r < 4; ++r) s[r] = s[r] / (1.f + __expf(-s[r])) * s2[r];
  } else if (bias != nullptr) {
    const u32x2 bb = *reinterpret_cast<const u32x2*>(bias + col);
    s[0] += bf16lo(bb[0]);
    s[1] += bf16hi(bb[0]);
    s[2] += bf16lo(bb[1]);
    s[3] += bf16hi(bb[1]);
  }
  const u32x2 o = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
  *reinterpret_cast<u32x2*>(y + (long)m * y_stride + col) = o;
}

// The reduction of a split product that closes a sublayer: residual[m] += sum_s ws[s, m], y[m] = rms norm of the new row * weight.  One
// workgroup per row, CH runs of four channels a thread; the sum, the new row and the result are rounded to 16 bits where the
// separate passes round them.  A launch of a few workgroups is latency: the pass of its own that it saves took 4.7 us of a
// decode step's layer, twice (16 layers, hidden size 4096, 14336 wide: one sequence 1769 -> 1724 us, 12 sequences 2137 -> 2088, 97 rows 3393 ->
// 3384).
template <int CH>
__global__ __launch_bounds__(1024) void mid_reduce_norm_kernel(const float* __restrict__ ws, uint16_t* __restrict__ residual,
                                                               const uint16_t* __restrict__ weight, uint16_t* __restrict__ y, int M,
                                                               int N, int S, float eps) {
  __shared__ float red[16];
  const int m = blockIdx.x, tid = threadIdx.x;
  const long step = (long)M * N;
  f32x4 v[CH];
  u32x2 ww[CH];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int col = (c * (int)blockDim.x + tid) * 4;
    v[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
    ww[c] = (u32x2){0, 0};
    if (col >= N) continue;
    uint16_t* rr = residual + (long)m * N + col;
    const u32x2 old = *reinterpret_cast<const u32x2*>(rr);
    ww[c] = *reinterpret_cast<const u32x2*>(weight + col);
    const float* p = ws + (long)m * N + col;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < S; i0 += 8) {
      f32x4 part[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) part[i] = *reinterpret_cast<const f32x4*>(p + (long)min(i0 + i, S - 1) * step);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i0 + i < S) s += part[i];
    }
    const u32x2 h = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
    const u32x2 o = {pack_bf16x2(bf16lo(h[0]) + bf16lo(old[0]), bf16hi(h[0]) + bf16hi(old[0])),
                     pack_bf16x2(bf16lo(h[1]) + bf16lo(old[1]), bf16hi(h[1]) + bf16hi(old[1]))};
    *reinterpret_cast<u32x2*>(rr) = o;
    v[c] = (f32x4){bf16lo(o[0]), bf16hi(o[0]), bf16lo(o[1]), bf16hi(o[1])};
    ss += v[c][0] * v[c][0] + v[c][1] * v[c][1] + v[c][2] * v[c][2] + v[c][3] * v[c][3];
  }
  ss = wave_reduce_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) tot += red[i];
  const float inv = rsqrtf(tot / (float)N + eps);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int col = (c * (int)blockDim.x + tid) * 4;
    if (col >= N) continue;
    const u32x2 o = {pack_bf16x2(v[c][0] * inv * bf16lo(ww[c][0]), v[c][1] * inv * bf16hi(ww[c][0])),
                     pack_bf16x2(v[c][2] * inv * bf16lo(ww[c][1]), v[c][3] * inv * bf16hi(ww[c][1]))};
    *reinterpret_cast<u32x2*>(y + (long)m * N + col) = o;
  }
}

// The reduction of a decode step's or short prompts' q | k | v projection, heads of 128 channels: q rotated to `q_out` [M, n_q * 128], k rotated and v to the
// token's slot of the paged cache.  Grid (M, head groups of 8), 32 lanes a head: lane j holds channels 2 j, 2 j + 1 and their
// rotation partners 64 further on.  Rounded to 16 bits before and after the rotation, as the separate passes do: what it saves
// is their two launches (the same steps: one sequence 1724 -> 1677 us, 12 sequences 2088 -> 2028, 40 sequences of 21.5k tokens, 8 layers, 5134 -> 5103).
__global__ __launch_bounds__(256) void mid_reduce_qkv_kernel(const float* __restrict__ ws, const uint16_t* __restrict__ bias,
                                                             uint16_t* __restrict__ q_out, const int* __restrict__ positions,
                                                             const long* __restrict__ slots, const float* __restrict__ cos_sin,
                                                             uint16_t* __restrict__ cache, long page_stride, long v_offset, int M,
                                                             int n_q, int n_kv, int S) {
  const int m = blockIdx.x, j = threadIdx.x & 31, h = blockIdx.y * 8 + (threadIdx.x >> 5);
  const int heads = n_q + 2 * n_kv;
  if (h >= heads) return;
  const int N = heads * HEAD_DIM, col = h * HEAD_DIM + 2 * j;
  const long step = (long)M * N;
  const float* p = ws + (long)m * N + col;
  const int pos = positions[m];
  const long slot = slots[m];
  const float2 c = *reinterpret_cast<const float2*>(cos_sin + (long)pos * HEAD_DIM + 2 * j);
  const float2 s = *reinterpret_cast<const float2*>(cos_sin + (long)pos * HEAD_DIM + 64 + 2 * j);
  float2 a = {0.f, 0.f}, b = {0.f, 0.f};
  for (int i0 = 0; i0 < S; i0 += 8) {
    float2 va[8], vb[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float* q = p + (long)min(i0 + i, S - 1) * step;
      va[i] = *reinterpret_cast<const float2*>(q);
      vb[i] = *reinterpret_cast<const float2*>(q + 64);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i0 + i < S) {
        a.x += va[i].x;
        a.y += va[i].y;
        b.x += vb[i].x;
        b.y += vb[i].y;
      }
  }
  if (bias != nullptr) {
    const uint32_t ba = *reinterpret_cast<const uint32_t*>(bias + col), bb = *reinterpret_cast<const uint32_t*>(bias + col + 64);
    a.x += bf16lo(ba);
    a.y += bf16hi(ba);
    b.x += bf16lo(bb);
    b.y += bf16hi(bb);
  }
  uint32_t lo = pack_bf16x2(a.x, a.y), hi = pack_bf16x2(b.x, b.y);
  if (h < n_q + n_kv) {
    const float x0 = bf16lo(lo), x1 = bf16hi(lo), y0 = bf16lo(hi), y1 = bf16hi(hi);
    lo = pack_bf16x2(rope_lo(x0, y0, c.x, s.x), rope_lo(x1, y1, c.y, s.y));
    hi = pack_bf16x2(rope_hi(x0, y0, c.x, s.x), rope_hi(x1, y1, c.y, s.y));
  }
  if (h < n_q) {
    uint16_t* q = q_out + ((long)m * n_q + h) * HEAD_DIM + 2 * j;
    *reinterpret_cast<uint32_t*>(q) = lo;
    *reinterpret_cast<uint32_t*>(q + 64) = hi;
    return;
  }
  if (slot < 0) return;
  uint16_t* page = cache + slot / PAGE * page_stride;
  const int off = (int)(slot % PAGE);
  if (h < n_q + n_kv) {
    uint16_t* kd = page + (long)(h - n_q) * PAGE * HEAD_DIM;
    *reinterpret_cast<uint32_t*>(kd + k_elem_off(off, 2 * j)) = lo;
    *reinterpret_cast<uint32_t*>(kd + k_elem_off(off, 64 + 2 * j)) = hi;
  } else {
    uint16_t* vd = page + v_offset + (long)(h - n_q - n_kv) * HEAD_DIM * PAGE;
    vd[v_elem_off(2 * j, off)] = (uint16_t)(lo & 0xffff);
    vd[v_elem_off(2 * j + 1, off)] = (uint16_t)(lo >> 16);
    vd[v_elem_off(64 + 2 * j, off)] = (uint16_t)(hi & 0xffff);
    vd[v_elem_off(65 + 2 * j, off)] = (uint16_t)(hi >> 16);
  }
}

template <int MT, bool PAIR, bool FACTORS = false>
int launch_mid(const void* x, long xs, const void* w, const void* bias, void* y, long ys, float* ws, int M, int N, int K, int S,
               hipStream_t stream, const float* squares = nullptr, float eps = 0.f) {
  constexpr int LDS = STAGES * (BN + 16 * MT) * ROWB;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)mid_gemm_kernel<MT, PAIR, FACTORS>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess)
      return -2;
    attr_set = true;
  }
  const int n_out = PAIR ? N / 2 : N;
  return launched(mid_gemm_kernel<MT, PAIR, FACTORS>, dim3(n_out / (PAIR ? BN / 2 : BN), S, (M + 127) / 128), 256, LDS, stream, (const uint16_t*)x, xs,
                  (const uint16_t*)w, (const uint16_t*)bias, (uint16_t*)y, ys, ws, M, N, K, S, squares, eps);
}

template <int MT>
int launch_experts(const void* x, const void* w13, const void* w2, const int* offsets, const int* sorted_tok, void* act, void* y,
                   int n_experts, int hidden, int inter, float act_limit, float act_alpha, float act_bias, const float* row_scale,
                   hipStream_t stream) {
  constexpr int UNIT_LDS = STAGES * (128 + 16 * MT) * ROWB, DOWN_LDS = STAGES * (64 + 16 * MT) * ROWB;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)mid_experts_kernel<MT, true>, hipFuncAttributeMaxDynamicSharedMemorySize, UNIT_LDS) != hipSuccess ||
        hipFuncSetAttribute((const void*)mid_experts_kernel<MT, false>, hipFuncAttributeMaxDynamicSharedMemorySize, DOWN_LDS) != hipSuccess)
      return -2;
    attr_set = true;
  }
  mid_experts_kernel<MT, true><<<dim3(inter / 64, n_experts), 256, UNIT_LDS, stream>>>(
      (const uint16_t*)x, (const uint16_t*)w13, offsets, sorted_tok, (uint16_t*)act, 2 * inter, hidden, act_limit, act_alpha, act_bias,
      row_scale);
  mid_experts_kernel<MT, false><<<dim3(hidden / 64, n_experts), 256, DOWN_LDS, stream>>>(
      (const uint16_t*)act, (const uint16_t*)w2, offsets, nullptr, (uint16_t*)y, hidden, inter, 0.f, 1.f, 0.f, nullptr);
  return 0;
}

}  // namespace

// x [tokens, hidden]; w13 [E, 2*inter, hidden]; w2 [E, hidden, inter]; offsets [E+1] and sorted_tok [tokens*topk] from
// vpsa_moe_align; act [tokens*topk, inter] and y [tokens*topk, hidden] are workspaces in expert-sorted row order.  No host
// synchronisation and a launch shape that does not depend on the routing: HIP-graph capturable.  act_limit > 0: the clamped gated
// unit (limit, alpha, bias) instead of SwiGLU.  row_scale (sorted order, or null): gate and up of a row are multiplied by it before
// the activation (a factor on the row's input).
VPSA_EXPORT int vpsa_moe_mfma_act(const void* x, const void* w13, const void* w2, const int* offsets, const int* sorted_tok,
                                  void* act, void* y, int tokens, int topk, int n_experts, int hidden, int inter, float act_limit,
                                  float act_alpha, float act_bias, const float* row_scale, hipStream_t stream) {
  if (tokens * topk <= 0) return 0;
  if (n_experts < 1 || n_experts > 65535 || hidden % 128 != 0 || inter % 512 != 0) return -1;
  if (((uintptr_t)x | (uintptr_t)w13 | (uintptr_t)w2 | (uintptr_t)act) & 15) return -1;
  if ((long)tokens * hidden * 2 >= (1L << 32) || (hidden > inter ? hidden : inter) >= (1 << 24)) return -1;  // offsets of 32 bits
  // an expert sees each token at most once: tokens bounds its row count
#define EXPERTS(MT)                                                                                                         \
  return launch_experts<MT>(x, w13, w2, offsets, sorted_tok, act, y, n_experts, hidden, inter, act_limit, act_alpha, act_bias, \
                            row_scale, stream)
  if (tokens <= 16) EXPERTS(1);
  if (tokens <= 32) EXPERTS(2);
  if (tokens <= 48) EXPERTS(3);
  EXPERTS(4);
#undef EXPERTS
}

VPSA_EXPORT int vpsa_moe_mfma(const void* x, const void* w13, const void* w2, const int* offsets, const int* sorted_tok, void* act,
                              void* y, int tokens, int topk, int n_experts, int hidden, int inter, hipStream_t stream) {
  return vpsa_moe_mfma_act(x, w13, w2, offsets, sorted_tok, act, y, tokens, topk, n_experts, hidden, inter, 0.f, 1.f, 0.f, nullptr,
                           stream);
}

// Workgroups along the reduction for a shape, 0 where the kernel does not tile it: as many as fill the chip's 256 CUs once, none
// shorter than eight chunks (the three on their way at the start are a third of it).
VPSA_EXPORT int vpsa_mid_gemm_splits(int M, int N, int K, int pair) {
  const int n_out = pair ? N / 2 : N, bn = pair ? BN / 2 : BN;
  if (M <= 0 || n_out <= 0 || (pair && (N & 1)) || n_out % bn != 0 || K % BK != 0 || (long)N * K * 2 >= (1L << 32)) return 0;
  const int blocks = n_out / bn * ((M + 127) / 128);
  int s = 256 / blocks;
  const int most = K / BK / 8;
  if (s > most) s = most;
  return s < 1 ? 1 : s;
}

// The product itself: y when S == 1, else partial sums in ws.
static int mid_product(const void* x, long xs, const void* w, const void* bias, void* y, long ys, void* ws, int M, int N, int K,
                       int pair, int S, hipStream_t stream) {
  if ((xs & 7) || (((uintptr_t)x | (uintptr_t)w) & 15) || xs * 256 >= (1L << 31)) return -1;
  if (S <= 0 || S != vpsa_mid_gemm_splits(M, N, K, pair) || (S > 1 && !ws) || M > 65535) return -1;
#define MID(MT)                                                                                             \
  return pair ? launch_mid<MT, true>(x, xs, w, bias, y, ys, (float*)ws, M, N, K, S, stream)                 \
              : launch_mid<MT, false>(x, xs, w, bias, y, ys, (float*)ws, M, N, K, S, stream)
  switch ((M + 15) / 16) {
    case 1: MID(1);
    case 2: MID(2);
    case 3: MID(3);
    case 4: MID(4);
    case 5: MID(5);
    case 6: MID(6);
    case 7: MID(7);
    default: MID(8);
  }
#undef MID
}

int mid_reduce(const void* ws, const void* bias, void* y, long ys, int M, int N, int S, int pair, hipStream_t stream) {
  const int n_out = pair ? N / 2 : N;
  const dim3 grid((n_out / 4 + 255) / 256, M);
  if (pair) mid_reduce_kernel<true><<<grid, 256, 0, stream>>>((const float*)ws, (const uint16_t*)bias, (uint16_t*)y, ys, M, N, S);
  else mid_reduce_kernel<false><<<grid, 256, 0, stream>>>((const float*)ws, (const uint16_t*)bias, (uint16_t*)y, ys, M, N, S);
  return 0;
}

bool mid_reduce_norm_takes(const void* residual, const void* weight, const void* y, int N) {
  return N % 4 == 0 && N <= 8192 && (((uintptr_t)residual | (uintptr_t)weight | (uintptr_t)y) & 7) == 0;
}

int mid_reduce_norm(const void* ws, void* residual, const void* weight, void* y, int M, int N, int S, float eps, hipStream_t stream) {
  const int threads = N >= 4096 ? 1024 : (N / 4 + 63) / 64 * 64;
  if (N <= 4096)
    mid_reduce_norm_kernel<1><<<M, threads, 0, stream>>>((const float*)ws, (uint16_t*)residual, (const uint16_t*)weight, (uint16_t*)y, M,
                                                         N, S, eps);
  else
    mid_reduce_norm_kernel<2><<<M, threads, 0, stream>>>((const float*)ws, (uint16_t*)residual, (const uint16_t*)weight, (uint16_t*)y, M,
                                                         N, S, eps);
  return 0;
}

bool mid_reduce_qkv_takes(const void* q_out, const void* bias, const void* cos_sin) {
  return !((uintptr_t)q_out & 3) && !((uintptr_t)bias & 3) && !((uintptr_t)cos_sin & 7);
}

int mid_reduce_qkv(const void* ws, const void* bias, void* q_out, const int* positions, const long* slots, const float* cos_sin,
                   void* cache, long page_stride, long v_offset, int M, int n_q, int n_kv, int S, hipStream_t stream) {
  mid_reduce_qkv_kernel<<<dim3(M, (n_q + 2 * n_kv + 7) / 8), 256, 0, stream>>>(
      (const float*)ws, (const uint16_t*)bias, (uint16_t*)q_out, positions, slots, cos_sin, (uint16_t*)cache, page_stride, v_offset, M,
      n_q, n_kv, S);
  return 0;
}

// x [M, K] (row stride xs elements, 16-byte aligned rows), w [N, K] contiguous, bias [N] or null, y [M, N] (or [M, N / 2] when
// pair != 0; row stride ys).  ws: fp32 workspace of S * M * N elements (unused when S == 1).
VPSA_EXPORT int vpsa_mid_gemm(const void* x, long xs, const void* w, const void* bias, void* y, long ys, void* ws, int M, int N,
                              int K, int pair, int S, hipStream_t stream) {
  if (M <= 0) return 0;
  if ((ys & 3) || ((uintptr_t)y & 7) || (pair && bias)) return -1;
  const int rc = mid_product(x, xs, w, bias, y, ys, ws, M, N, K, pair, S, stream);
  return rc || S == 1 ? rc : mid_reduce(ws, bias, y, ys, M, N, S, pair, stream);
}

// y [M, N / 2] = silu(gate) * up, gate | up = x W^T times the rows' factors 1 / sqrt(sum of squares / K + eps), squares [M, K / 16]: M up to 16,
// K up to 8192, an unsplit shape.
VPSA_EXPORT int vpsa_mid_unit_factors(const void* x, long xs, const float* squares, float eps, const void* w, void* y, long ys, int M, int N,
                                      int K, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 16 || K > 8192 || vpsa_mid_gemm_splits(M, N, K, 1) != 1 || (ys & 3) || ((uintptr_t)y & 7)) return -1;
  if ((xs & 7) || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)squares) & 15) || xs * 256 >= (1L << 31)) return -1;
  return launch_mid<1, true, true>(x, xs, w, nullptr, y, ys, nullptr, M, N, K, 1, stream, squares, eps);
}

// residual [M, N] += x W^T, y [M, N] = rms norm of the new rows * weight; a split product (S > 1), N a multiple of 4 up to 8192.
VPSA_EXPORT int vpsa_mid_gemm_norm(const void* x, long xs, const void* w, void* residual, const void* weight, void* y, void* ws, int M,
                                   int N, int K, int S, float eps, hipStream_t stream) {
  if (M <= 0) return 0;
  if (S < 2 || !mid_reduce_norm_takes(residual, weight, y, N)) return -1;
  const int rc = mid_product(x, xs, w, nullptr, nullptr, 0, ws, M, N, K, 0, S, stream);
  return rc ? rc : mid_reduce_norm(ws, residual, weight, y, M, N, S, eps, stream);
}

// q | k | v = x W^T (+ bias) of one token per sequence: q rotated to q_out [M, n_q * 128], k rotated and v to the cache (layer base
// `cache`; slots < 0: nowhere); a split product (S > 1), N = (n_q + 2 n_kv) * 128.
VPSA_EXPORT int vpsa_mid_gemm_qkv(const void* x, long xs, const void* w, const void* bias, void* q_out, void* ws, int M, int K, int S,
                                  const int* positions, const long* slots, const float* cos_sin, void* cache, long page_stride,
                                  long v_offset, int n_q, int n_kv, hipStream_t stream) {
  if (M <= 0) return 0;
  if (S < 2 || !mid_reduce_qkv_takes(q_out, bias, cos_sin)) return -1;
  const int rc = mid_product(x, xs, w, nullptr, nullptr, 0, ws, M, (n_q + 2 * n_kv) * HEAD_DIM, K, 0, S, stream);
  return rc ? rc : mid_reduce_qkv(ws, bias, q_out, positions, slots, cos_sin, cache, page_stride, v_offset, M, n_q, n_kv, S, stream);
}

// Where a workgroup of a product begins (tests).
VPSA_EXPORT int vpsa_mid_first_chunk(int block, int n, int whole) { return n > 0 ? first_chunk(block, n, whole != 0) : -1; }
