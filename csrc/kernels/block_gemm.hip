// Products of a few hundred to some ten thousand token rows for gfx950 whose 256 x 256 tiles would not fill the chip's 256 CUs in whole
// rounds, or whose reductions are short: y[M, N] = epilogue(x[M, K] . W[N, K]^T + bias), tiles of several shapes on one scheme.
//   * 256 threads, waves as 2 (rows) x 2 (columns); a wave multiplies 16 TM token rows with 16 TN weight rows on
//     v_mfma_f32_16x16x32_bf16, a workgroup BM = 32 TM rows with BN = 32 TN columns.
//   * Both operands go from memory straight into LDS in chunks of 64 along K (rows of 128 bytes, 16-byte piece j of row r at
//     j ^ (r / 2) % 8: the 16 rows of a fragment cover every bank), S chunks in a ring.
//   * One barrier a chunk, in its middle: the fragments of the chunk's second half and of the next chunk's first half are read while
//     the matrix cores work on the half before, so that a lone wave on a SIMD keeps them busy; the chunk's place in the ring is
//     requested again right behind that barrier, S - 1/2 chunks ahead of its use.
//   * The weight rows are the MFMA's A operand and are ordered so that a lane ends with eight consecutive columns of a token row.
//   * Where there are more tiles than the chip holds at once, as many workgroups as it holds make several each: the ring goes on with the next
//     tile's chunks while the last ones of a tile are multiplied and its epilogue runs.
// What bounds it: LDS, which carries (reads and the loads' writes) 128 bytes for every 64 x 96 x 96 of products in the largest shape, as many
// cycles as the matrix cores need; with short reductions the time until a tile's first chunk is there and its epilogue (gelu 75
// cycles of vector work a wave and value).  12000 rows in a loop over the same operands, library with the activation's pass / this: 3072 x
// 768 with gelu 107 / 70 us, 768 x 3072 57 / 48 (+ residual), three of 768 x 768 62 / 48, 768 x 2304 with gelu 50 / 42; 1500 rows, 2048 x 512 with
// gelu 26 / 11.  Over operands that no cache holds, a workgroup for every tile / several tiles a workgroup with the costs below: the first
// 78.9 / 72.7, the second 62.4 / 62.4, the third 53.5 / 45.7, one 768 x 768 with a residual 25.6 / 22.6, 395 products of 1500 to 48000 rows 5.7 %; an encoder
// of 12 layers, 8 windows 3733 / 3565, 2 1746 / 1640, 32 13.66 / 12.97 ms, none of 1 to 32 windows slower.
#include <type_traits>

#include "common.h"
#include "mid_reduce.h"

namespace {

constexpr int BK = 64, ROWB = BK * 2;

enum { ACT_NONE = 0, ACT_GELU = 1, ACT_SILU = 2 };  // SILU: w is [gate rows | up rows], silu(gate) * up

// Row r of an operand lies at (r / batch_rows) * bs + (r % batch_rows) * ld elements.
struct Rows {
  long ld, bs;
};

struct BlockArgs {
  const uint16_t* a;
  const uint16_t* w[3];     // the products of several weights of one shape stand side by side in c
  const uint16_t* bias[3];  // or null
  const uint16_t* res;      // added behind the activation, or null
  uint16_t* c;
  Rows ar, cr, rr;
  int batch_rows, M, N, K, n_tiles;  // N: rows of one weight; n_tiles: column tiles of one weight
  int parts;
  float* ws;  // splits > 1: partial sums [splits, M, N]
  int splits;
  uint32_t a_bytes, w_bytes;  // ends of the operands, for loads past the reduction's end
};

// x Phi(x).  Phi(-|x|) = exp(-x^2 / 2) t P(t), t = 1 / (1 + 0.31 |x|), P of degree 5 fitted here to the smallest relative error over
// 0 <= |x| <= 14: 5e-6, also far out on the negative side.
__device__ __forceinline__ float gelu(float x) {
  const float ax = fabsf(x), t = __builtin_amdgcn_rcpf(fmaf(0.31f, ax, 1.f));
  float p = -0.0739278644f;
  p = fmaf(p, t, 0.1804467738f);
  p = fmaf(p, t, 0.0157485195f);
  p = fmaf(p, t, 0.1334278733f);
  p = fmaf(p, t, 0.1204417273f);
  p = fmaf(p, t, 0.1238606647f);
  const float h = p * t * __builtin_amdgcn_exp2f(x * x * -0.72134752044448170f);
  return x * (x >= 0.f ? 1.f - h : h);
}

// STREAM: few row tiles, weights read about once, by non-temporal loads and from another chunk on for every column tile.  MANY: a workgroup
// makes several tiles.
template <int TM, int TN, int S, int ACT, bool STREAM, bool MANY>
__global__ __launch_bounds__(256, (TM + TN) * S * 4096 <= 81920 ? 2 : 1) void block_gemm_kernel(const BlockArgs args) {
  constexpr bool PAIR = ACT == ACT_SILU;
  constexpr int BM = 32 * TM, BN = 32 * TN, STAGE = (BM + BN) * ROWB, NL = TM + TN;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g = lane >> 4, wr = wave >> 1, wc = wave & 1;
  const int M = args.M, N = args.N, K = args.K;

  // Tiles in blocks of an eighth of the row tiles (up to eight), column by column inside a block, cut in eight runs, one per XCD
  // (workgroups go round them): those that share an L2 at any time are about a square of tiles.
  const int m_tiles = (M + BM - 1) / BM, cols = args.n_tiles * args.parts, tiles = m_tiles * cols, total = STREAM ? tiles * args.splits : tiles;
  const int xcd = blockIdx.x & 7, run = (total >> 3) + (xcd < (total & 7)), run0 = xcd * (total >> 3) + min(xcd, total & 7);
  int at = blockIdx.x >> 3;  // in the run; then every (gridDim.x + 7) / 8-th
  int split = 0, c0 = 0, n = K / BK, first = 0;  // chunks c0 .. c0 + n - 1 of the reduction, from c0 + first round
  int m0, n0, part;                              // the tile whose chunks are loaded
  auto place = [&]() {
    int t = run0 + at;
    if (STREAM) {
      split = t / tiles;
      t -= split * tiles;
    }
    const int blk = min(8, (m_tiles + 7) / 8), block = t / (blk * cols), rem = t - block * blk * cols, rows = min(blk, m_tiles - blk * block);
    const int col = rem / rows;
    m0 = (blk * block + rem - col * rows) * BM;
    part = col / args.n_tiles;
    n0 = (col - part * args.n_tiles) * BN;
    if (STREAM) {
      const int per = n / args.splits, extra = n - per * args.splits;
      c0 = split * per + min(split, extra);
      n = per + (split < extra);
      first = col * 3 % n;
    }
  };
  place();

  // what this lane loads of a chunk: 8 rows of 8 pieces a KiB; rows past the last repeat it
  uint32_t aoff[TM], woff[TN];
  const int lrow = lane >> 3;
  auto rows_of_tile = [&]() {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r = 8 * (4 * i + wave) + lrow, row = min(m0 + r, M - 1);
      const int b = row / args.batch_rows;
      aoff[i] = (uint32_t)((b * args.ar.bs + (row - b * args.batch_rows) * args.ar.ld) * 2) + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int r = 8 * (4 * i + wave) + lrow, rr = r % (16 * TN), j = rr & 15, perm = 8 * (j >> 2) + 4 * ((rr >> 4) & 1) + (j & 3);
      // PAIR: tiles 2 b, 2 b + 1 of a wave are 16 gate rows and the up rows beside them
      const int col = PAIR ? n0 / 2 + r / (16 * TN) * (8 * TN) + 16 * (rr >> 5) + j : n0 + r / (16 * TN) * (16 * TN) + 32 * (rr >> 5) + perm;
      const int row = PAIR ? min(col, N / 2 - 1) + ((rr >> 4) & 1 ? N / 2 : 0) : min(col, N - 1);
      woff[i] = (uint32_t)row * (uint32_t)(K * 2) + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
  };
  rows_of_tile();
  bool more = false;  // behind the last chunk come those of the next tile
  auto load = [&](int c, char* st, int i) {  // the i-th KiB of this wave; nothing past the last tile's last chunk (a buffer of no bytes)
    const bool x = i < TM;
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(x ? args.a : args.w[part]), 0, c < n || (MANY && more) ? (int)(x ? args.a_bytes : args.w_bytes) : 0, 0x00020000);
    const auto to = (__attribute__((address_space(3))) void*)(st + (4 * i + wave) * 1024);
    const int off = (int)(x ? aoff[i % TM] : woff[(i - TM + TN) % TN]);
    const int from = c >= n ? (MANY && more ? (c - n) * ROWB : 0) : STREAM ? (c0 + (c + first < n ? c + first : c + first - n)) * ROWB : c * ROWB;
    if (STREAM && !x) __builtin_amdgcn_raw_ptr_buffer_load_lds(src, to, 16, off, from, 0, 2);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(src, to, 16, off, from, 0, 0);
  };

  // fragments: row c16 of a 16-row tile, piece 4 ks + g
  const int fr = c16 * ROWB + ((g ^ (c16 >> 1)) << 4);
  const int a_rd = wr * 16 * TM * ROWB, w_rd = (BM + wc * 16 * TN) * ROWB;
  bf16x8 wf[2][TN], xf[2][TM];
  auto read = [&](const char* st, int ks, int i) {
    const int f = fr ^ (ks << 6);
    if (i < TM) xf[ks][i % TM] = *reinterpret_cast<const bf16x8*>(st + a_rd + i * 2048 + f);
    else wf[ks][(i - TM + TN) % TN] = *reinterpret_cast<const bf16x8*>(st + w_rd + (i - TM) * 2048 + f);
  };
  f32x4 acc[TN][TM];
  // Half a chunk: its matrix instructions, between the first two thirds of them the reads of the half that follows (from `from`) and
  // between all of them the requests [lo, hi) of a later chunk c (into `to`).  The order is written out: left alone, the compiler puts
  // all loads in front.
  auto half = [&](int ks, const char* from, int lo, int hi, int c, char* to) {
    constexpr int MMA = TM * TN, R = TM + TN, PER = MMA * 2 / (3 * R) > 0 ? MMA * 2 / (3 * R) : 1;
#pragma unroll
    for (int m = 0; m < MMA; ++m) {
      acc[m / TM][m % TM] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[ks][m / TM], xf[ks][m % TM], acc[m / TM][m % TM], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (m % PER == 0 && m / PER < R) read(from, ks ^ 1, m / PER);
#pragma unroll
      for (int q = m * (hi - lo) / MMA; q < (m + 1) * (hi - lo) / MMA; ++q) load(c, to, lo + q);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = (MMA - 1) / PER + 1; i < R; ++i) read(from, ks ^ 1, i);
  };
  // A chunk's place is free from the middle of the chunk on.  Three places and more: the requests into it are spread over a whole
  // chunk's time; with two they all go out in the half that follows.
  constexpr int L0 = S > 2 ? NL / 2 : NL;

#pragma unroll
  for (int c = 0; c < S; ++c) {
#pragma unroll
    for (int i = 0; i < (c < S - 1 ? NL : L0); ++i) load(c, lds + c * STAGE, i);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * NL + L0) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  char *st = lds, *prev = lds + (S - 1) * STAGE;
#pragma unroll
  for (int i = 0; i < NL; ++i) read(st, 0, i);
  for (;;) {  // a tile
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int tm0 = m0, tn0 = n0, tpart = part;  // the tile that is multiplied
    for (int c = 0; c < n; ++c) {
      half(0, st, L0, NL, c + S - 1, prev);
      // chunk c + 1 has landed (mine: all but the loads of the chunks behind it) and my reads of chunk c are done; everyone's: the barrier
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * NL) : "memory");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      prev = st;
      st = st + STAGE == lds + S * STAGE ? lds : st + STAGE;
      if (MANY && c + S == n) {
        at += (gridDim.x + 7) >> 3;
        more = at < run;
        if (more) {
          asm volatile("" ::: "memory");  // a branch: without it the compiler works the places out in every chunk and selects
          place();
          rows_of_tile();
          asm volatile("" ::: "memory");
        }
      }
      half(1, st, 0, L0, c + S, prev);
    }
    if (!MANY || !more) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still write to LDS when the wave ends

    // accumulator [i][j]: token row 16 j + c16 of the wave's; registers of tiles 2 b, 2 b + 1: columns 8 g .. 8 g + 7 of the 32 of pair b
    constexpr int NB = TN / 2;
    if (STREAM && args.splits > 1) {
      float* const ws = args.ws + (long)split * M * N;
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int row = tm0 + wr * 16 * TM + 16 * j + c16;
        if (row >= M) continue;
#pragma unroll
        for (int i = 0; i < TN; ++i) {
          const int col = PAIR ? tn0 / 2 + wc * 8 * TN + 16 * (i >> 1) + 4 * g : tn0 + wc * 16 * TN + 32 * (i >> 1) + 8 * g + 4 * (i & 1);
          if (col < (PAIR ? N / 2 : N)) *reinterpret_cast<f32x4*>(ws + (long)row * N + col + (PAIR && (i & 1) ? N / 2 : 0)) = acc[i][j];
        }
      }
      return;
    }
    if constexpr (PAIR) {
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int row = tm0 + wr * 16 * TM + 16 * j + c16;
        if (row >= M) continue;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int col = tn0 / 2 + wc * 8 * TN + 16 * b + 4 * g;
          if (col >= N / 2) continue;
          f32x4 s = acc[2 * b][j];
#pragma unroll
          for (int e = 0; e < 4; ++e) s[e] = s[e] / (1.f + __expf(-s[e])) * acc[2 * b + 1][j][e];
          *reinterpret_cast<u32x2*>(args.c + row * args.cr.ld + col) = (u32x2){pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
        }
      }
      return;
    }
    const int col0 = tn0 + wc * 16 * TN + 8 * g;
    u32x4 bias[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      bias[b] = (u32x4){0, 0, 0, 0};
      if (args.bias[tpart] != nullptr && col0 + 32 * b < N)
        bias[b] = *reinterpret_cast<const u32x4*>(args.bias[tpart] + col0 + 32 * b);
    }
    // waited for here: on its way into the next tile, past rows that are not there, it would be waited for among the first reads of every chunk
    if (MANY) {
#pragma unroll
      for (int b = 0; b < NB; ++b) asm volatile("" : "+v"(bias[b]));
    }
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int row = tm0 + wr * 16 * TM + 16 * j + c16;
      if (row >= M) continue;
      const int bt = row / args.batch_rows, tr = row - bt * args.batch_rows;
      uint16_t* const cp = args.c + bt * args.cr.bs + tr * args.cr.ld + (long)tpart * N;
      const uint16_t* const rp = args.res + bt * args.rr.bs + tr * args.rr.ld;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int col = col0 + 32 * b;
        if (col >= N) continue;
        float v[8];
#pragma unroll
        for (int p = 0; p < 8; ++p) {
          v[p] = acc[2 * b + (p >> 2)][j][p & 3] + (p & 1 ? bf16hi(bias[b][p >> 1]) : bf16lo(bias[b][p >> 1]));
          if (ACT == ACT_GELU) v[p] = gelu(v[p]);
        }
        if (args.res != nullptr) {
          const u32x4 r = *reinterpret_cast<const u32x4*>(rp + col);
#pragma unroll
          for (int p = 0; p < 8; ++p) v[p] += p & 1 ? bf16hi(r[p >> 1]) : bf16lo(r[p >> 1]);
        }
        const u32x4 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
        *reinterpret_cast<u32x4*>(cp + col) = o;
      }
    }
    if (!MANY || !more) return;
    more = false;
  }
}

template <int TM, int TN, int S, int ACT, bool STREAM, bool MANY>
int start(const BlockArgs& args, long blocks, hipStream_t stream) {
  constexpr int LDS = (TM + TN) * S * 4096;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)block_gemm_kernel<TM, TN, S, ACT, STREAM, MANY>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) !=
        hipSuccess)
      return -2;
    attr_set = true;
  }
  block_gemm_kernel<TM, TN, S, ACT, STREAM, MANY><<<dim3((unsigned)blocks), 256, LDS, stream>>>(args);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// Whether workgroups make several of the tiles: more than the chip holds, and reductions that a ring of so many places does not outrun.
bool several(long tiles, int K, int round, int ring) { return tiles > round && K / BK >= ring; }

template <int TM, int TN, int S, int ACT, bool STREAM = false>
int launch(BlockArgs& args, hipStream_t stream) {
  args.n_tiles = (args.N + 32 * TN - 1) / (32 * TN);
  const long blocks = (long)args.n_tiles * args.parts * args.splits * ((args.M + 32 * TM - 1) / (32 * TM));
  if (blocks >= (1L << 31)) return -1;
  constexpr int ROUND = (TM + TN) * S * 4096 <= 81920 ? 512 : 256;  // what the chip holds
  if constexpr (!STREAM)
    if (several(blocks, args.K, ROUND, S)) return start<TM, TN, S, ACT, false, true>(args, ROUND, stream);
  return start<TM, TN, S, ACT, STREAM, false>(args, blocks, stream);
}

// The tile shapes, and what they cost in microseconds: a chunk and what stands beside a tile's chunks (epilogue) in a round of one
// workgroup a CU, or, where two share a CU, of two (up to half of such a round has a CU to each workgroup and a pair of numbers of its
// own); more of the epilogue with gelu and with a residual; a launch's start.  A round that is not full is shorter, for its workgroups share memory and
// power with fewer: `least` is the share of its time that it keeps with next to none, `over` where it stands between a half and a full round when the first
// CUs have two.  Counted as whole beyond a half, 7500 rows of 768 x 3072 went to 192 x 128 (240 of 512 places, 60.5 us over operands from memory, 45.6 from
// the caches) instead of 128 x 128 (354 of 512: 55.6 / 43.6), three 1280 x 1280 with 1500 rows took 26.9 / 26.4 instead of 23.1 / 23.3.  Fitted to 395 products of a
// speech encoder (N, K of 384 to 5120, 1500 to 48000 rows), each over operands from memory and from the caches, and drawn towards the best choice:
// in the mean of the two 0.3 % off the best shape on average, at the most 7 (with whole rounds 1.5 and 16).  Where the two disagree, the mean decides: 3000 rows of 768
// x 3072 take 128 x 128 by itself on a CU, 35.9 / 24.5, 64 x 128 would 32.0 / 31.0.
struct Shape {
  int bm, bn, per_cu;
  float chunk, fixed, chunk1, fixed1, gelu, res, start, least, over;
};
constexpr Shape SHAPES[] = {{192, 192, 1, 0.82f, 3.68f, 0.f, 0.f, 5.50f, 8.76f, 6.85f, 0.73f, 1.00f}, {128, 128, 1, 0.52f, 1.87f, 0.f, 0.f, 2.43f, 3.19f, 3.12f, 0.67f, 1.00f},
                            {128, 128, 2, 0.98f, 2.80f, 0.71f, 0.00f, 2.30f, 5.42f, 4.14f, 0.91f, 0.33f}, {64, 128, 2, 0.70f, 1.31f, 0.41f, 0.15f, 0.63f, 2.24f, 2.54f, 0.48f, 0.72f},
                            {192, 128, 2, 1.26f, 2.21f, 0.95f, 0.34f, 3.86f, 8.20f, 6.63f, 0.66f, 0.55f}, {96, 192, 2, 1.19f, 1.94f, 0.93f, 0.00f, 2.42f, 6.76f, 4.92f, 0.60f, 0.17f}};

int choose(int M, int N, int K, int parts, int act, bool res) {
  int best = 0;
  double best_t = 0;
  for (int i = 0; i < (int)(sizeof(SHAPES) / sizeof(SHAPES[0])); ++i) {
    const Shape& s = SHAPES[i];
    const long tiles = (long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn) * parts, round = 256 * s.per_cu;
    const double more = (act == ACT_GELU ? s.gelu : 0) + (res ? s.res : 0), full = K / BK * s.chunk + s.fixed + more, fill = (double)(tiles % round) / round;
    const double half = K / BK * s.chunk1 + s.fixed1 + more / 2;
    const double left = fill == 0         ? 0
                        : s.per_cu == 1   ? full * (s.least + (1 - s.least) * fill)
                        : fill <= 0.5     ? half * (s.least + (1 - s.least) * 2 * fill)
                                          : half + (full - half) * (s.over + (1 - s.over) * (2 * fill - 1));
    const double t = s.start + tiles / round * full + left;
    if (i == 0 || t < best_t) best = i, best_t = t;
  }
  return best;
}

}  // namespace

// The tile shape of a product (its place in SHAPES), plus 16 where workgroups make several tiles each.
VPSA_EXPORT int vpsa_block_gemm_shape(int M, int N, int K, int parts, int act, int res) {
  constexpr int RING[] = {3, 4, 2, 3, 2, 2};
  const int i = choose(M, N, K, parts, act, res != 0);
  const Shape& s = SHAPES[i];
  return i + (several((long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn) * parts, K, 256 * s.per_cu, RING[i]) ? 16 : 0);
}

// c[r] = act(x[r] W_p^T + bias_p) + res[r], the columns of weights p = 0 .. parts - 1 (N rows of K each) side by side.  Rows r = 0 .. M - 1
// in batches of batch_rows (one batch: M): strides of a row and of a batch in elements for x, c and res (c may be res).  act: 0 none,
// 1 gelu (erf form).  Pieces of 16 bytes: N and strides multiples of 8, bases on 16 bytes; K a multiple of 64.  Returns 0, or a negative
// number for what the kernel does not take.
VPSA_EXPORT int vpsa_block_gemm(const void* x, long ld, long bs, const void* w0, const void* w1, const void* w2, const void* b0,
                                const void* b1, const void* b2, int parts, void* c, long ldc, long cbs, const void* res, long ldr,
                                long rbs, int batch_rows, int M, int N, int K, int act, hipStream_t stream) {
  if (M <= 0) return 0;
  if (N <= 0 || N % 8 != 0 || K <= 0 || K % BK != 0 || batch_rows <= 0 || parts < 1 || parts > 3 || act < 0 || act > 1) return -1;
  if (((ld | bs | ldc | cbs | ldr | rbs) & 7) != 0 || ld < 0 || bs < 0 ||
      (((uintptr_t)x | (uintptr_t)w0 | (uintptr_t)w1 | (uintptr_t)w2 | (uintptr_t)b0 | (uintptr_t)b1 | (uintptr_t)b2 | (uintptr_t)c |
        (uintptr_t)res) & 15) != 0)
    return -1;
  const int last = batch_rows < M ? batch_rows - 1 : M - 1;
  const double a_bytes = 2. * ((double)((M - 1) / batch_rows) * bs + (double)last * ld + K), w_bytes = 2. * N * K;
  if (a_bytes >= 4294967296. || w_bytes >= 4294967296.) return -1;  // offsets of 32 bits
  BlockArgs args = {(const uint16_t*)x,
                    {(const uint16_t*)w0, (const uint16_t*)w1, (const uint16_t*)w2},
                    {(const uint16_t*)b0, (const uint16_t*)b1, (const uint16_t*)b2},
                    (const uint16_t*)res, (uint16_t*)c, {ld, bs}, {ldc, cbs}, {ldr, rbs}, batch_rows, M, N, K, 0, parts, nullptr, 1,
                    (uint32_t)a_bytes, (uint32_t)w_bytes};
#define SHAPE(TM, TN, S) return act == ACT_GELU ? launch<TM, TN, S, ACT_GELU>(args, stream) : launch<TM, TN, S, ACT_NONE>(args, stream)
  switch (choose(M, N, K, parts, act, res != nullptr)) {
    case 0: SHAPE(6, 6, 3);
    case 1: SHAPE(4, 4, 4);
    case 2: SHAPE(4, 4, 2);
    case 3: SHAPE(2, 4, 3);
    case 4: SHAPE(6, 4, 2);
    default: SHAPE(3, 6, 2);
  }
#undef SHAPE
}

// Projections of 97 to 512 rows: up to 256 in one row tile of the smallest height that holds them, beyond in two; 128 weight rows a
// workgroup, the reduction split until about every CU has one (ranges of six chunks at least), as in mid_gemm.hip, whose reductions close it.
// Against mid_gemm's two blocks of 128 rows the weights pass through LDS once, and a wave multiplies 64 weight rows with half of the
// token rows instead of 32 with all (a third less to read from LDS).  What bounds it: with all operands in the caches 28672 x 4096 takes 35 us
// with 128 rows and 54 with 256 (1.1 PFLOP/s), with weights from memory 48 and 58: the two do not quite overlap.  More
// chunks on their way (five stages), 64 weight rows a workgroup and two workgroups a CU changed nothing or were slower; non-temporal
// loads of the weights take 5 % off, other start chunks for every column tile 1 to 2 %.
// Library with its activation or norm pass / this: 28672 x 4096 with the gated unit, 129 rows 61.6 / 49.3 us, 256 rows 72.0 / 58.3; 4096 x 14336 with
// the norm, 129 rows 58.4 / 38.1, 512 rows 93.1 / 68.2.  A step of 8 layers: 150 rows behind 3000 tokens 1938 -> 1610, 256 sequences 2578 -> 2243.
static int block_splits(int M, int N, int K) {
  const int blocks = (N + 127) / 128 * ((M + 255) / 256), most = K / BK / 6, s = 256 / (blocks > 0 ? blocks : 1);
  return s > most ? (most > 0 ? most : 1) : s < 1 ? 1 : s;
}

// Workgroups along the reduction, 0 where the kernel does not tile the shape.
VPSA_EXPORT int vpsa_block_proj_splits(int M, int N, int K, int pair) {
  if (M <= 0 || M > 512 || N <= 0 || N % (pair ? 16 : 8) != 0 || K <= 0 || K % BK != 0 || (long)N * K * 2 >= (1L << 32)) return 0;
  return block_splits(M, N, K);
}

static int block_product(const void* x, long xs, const void* w, const void* bias, void* y, long ys, void* ws, int M, int N, int K, int pair,
                         int S, hipStream_t stream) {
  if (M <= 0 || S <= 0 || S != vpsa_block_proj_splits(M, N, K, pair) || (S > 1 && !ws)) return -1;
  if (xs < K || (xs & 7) || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)ws) & 15) || (double)M * xs * 2 >= 4294967296.) return -1;
  if (S == 1 && ((ys & 7) || ((uintptr_t)y & 15) || ((uintptr_t)bias & 15))) return -1;
  BlockArgs args = {(const uint16_t*)x, {(const uint16_t*)w, nullptr, nullptr}, {S == 1 ? (const uint16_t*)bias : nullptr, nullptr, nullptr},
                    nullptr, (uint16_t*)y, {xs, 0}, {ys, 0}, {0, 0}, M, M, N, K, 0, 1, (float*)ws, S,
                    (uint32_t)(2 * ((M - 1) * xs + K)), (uint32_t)(2L * N * K)};
#define SHAPE(TM, S) return pair ? launch<TM, 4, S, ACT_SILU, true>(args, stream) : launch<TM, 4, S, ACT_NONE, true>(args, stream)
  switch ((M + 32 * ((M + 255) / 256) - 1) / (32 * ((M + 255) / 256))) {
    case 5: SHAPE(5, 4);
    case 6: SHAPE(6, 3);
    case 7: SHAPE(7, 3);
    case 8: SHAPE(8, 3);
    default: SHAPE(4, 4);
  }
#undef SHAPE
}

// y [M, N] = x W^T (+ bias), or silu(gate) * up [M, N / 2] with pair (w = [gate rows | up rows]).  x rows of stride xs, y rows of stride ys;
// ws: fp32 workspace of S * M * N elements (unused when S == 1).
VPSA_EXPORT int vpsa_block_proj(const void* x, long xs, const void* w, const void* bias, void* y, long ys, void* ws, int M, int N, int K,
                                int pair, int S, hipStream_t stream) {
  if ((ys & 3) || ((uintptr_t)y & 7) || (pair && bias)) return -1;
  const int rc = block_product(x, xs, w, bias, y, ys, ws, M, N, K, pair, S, stream);
  return rc || S == 1 ? rc : mid_reduce(ws, bias, y, ys, M, N, S, pair, stream);
}

// residual [M, N] += x W^T, y [M, N] = rms norm of the new rows * weight; S > 1.
VPSA_EXPORT int vpsa_block_proj_norm(const void* x, long xs, const void* w, void* residual, const void* weight, void* y, void* ws, int M,
                                     int N, int K, int S, float eps, hipStream_t stream) {
  if (S < 2 || !mid_reduce_norm_takes(residual, weight, y, N)) return -1;
  const int rc = block_product(x, xs, w, nullptr, nullptr, 0, ws, M, N, K, 0, S, stream);
  return rc ? rc : mid_reduce_norm(ws, residual, weight, y, M, N, S, eps, stream);
}

// One token per sequence: q rotated to q_out, k rotated and v to the cache, as vpsa_mid_gemm_qkv; S > 1.
VPSA_EXPORT int vpsa_block_proj_qkv(const void* x, long xs, const void* w, const void* bias, void* q_out, void* ws, int M, int K, int S,
                                    const int* positions, const long* slots, const float* cos_sin, void* cache, long page_stride,
                                    long v_offset, int n_q, int n_kv, hipStream_t stream) {
  if (S < 2 || !mid_reduce_qkv_takes(q_out, bias, cos_sin)) return -1;
  const int rc = block_product(x, xs, w, nullptr, nullptr, 0, ws, M, (n_q + 2 * n_kv) * HEAD_DIM, K, 0, S, stream);
  return rc ? rc : mid_reduce_qkv(ws, bias, q_out, positions, slots, cos_sin, cache, page_stride, v_offset, M, n_q, n_kv, S, stream);
}
