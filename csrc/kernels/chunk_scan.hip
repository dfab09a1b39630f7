// The recurrences S <- a_t (.) S + k_t v_t^T, o_t = S^T q_t over prompt chunks, on the matrix cores: a fixed decay per head (q and
// k rotated, or through silu), or a gate per key channel (a = lo + (1 - lo) sigmoid(z + b), k = 1 - a, q = silu(q)).
//
// Token by token (seqmix.hip) every token costs two or three vector operations per state element.  Here blocks of up to 32 tokens are
// contractions.  With R_j = a_(j+1) .. a_(n-1) (per channel; n tokens, R_(n-1) = 1), A = a_0 .. a_(n-1) and S0 the state before:
//     S' = A S0    q^_i = q_i / R_i    k^_j = k_j R_j       o_i = S'^T q^_i + sum_(j <= i) (q^_i . k^_j) v_j       S = S' + sum_j k^_j v_j^T
// Operands stay at 32 bits: each is cut into three bf16 parts of 8 bits (exactly: hi + mid + lo), v is one part as
// it comes (three behind silu), and products of parts down to 2^-24 of the largest go through v_mfma_f32_16x16x32_bf16 (three instructions
// for k^ v and the scores' product with v, six for S'^T q^ and the scores; sums in 32 bits, those of the small products apart).  A 32-bit
// instruction does a sixteenth of that work per cycle.  Error against 64 bits, fixed decay: 1.1e-7 (64 rows) to 1.7e-7 (8192 rows), on
// 32-bit matrix instructions 1.7e-7 to 3.0e-7; gated, whose 1 - a comes from the exponential: 0.9e-7, token by token in seqmix.hip 1.2e-7; gates
// around a half 0.7e-7 against 0.5e-7, gates that forget (token by token here as well) 0.5e-7 both.
//   * What bounds it: vector work (a block costs a wave 1000 instructions, half of them to cut the state up, and a SIMD's two waves
//     2 x 166 matrix instructions) and the barriers between staging, scores and products; HBM has a third of its traffic.
//   * Measured, token by token or on 32-bit matrix instructions / here: 8192 rows of two sequences, 32 heads: gated 128 x 128 1559 / 296 us,
//     fixed 128 x 256, rotated, 702 / 347; 1000 rows: gated (16 heads, three sequences) 229 / 55, fixed (one) 154 / 84; 200 rows of two 199 / 37.
//   * 1 / R must stay in range: a block in which some |R| leaves 2^-60 .. 2^60 is taken again with half its tokens (a block of one token
//     divides by nothing); fixed decays know their longest block beforehand, and those that need shorter ones go to retention.hip.
//   * A workgroup holds a head's whole 128 x VD state in accumulators, 32 columns a wave, so q, k and the scores are made once for all
//     columns.  S' is cut into parts as it lies in the accumulators: register r of lane (c, g) is row 4 g + r of
//     a 16-row tile, and two tiles are one operand of 32 channels.  The outputs come out transposed: four columns of a token a lane.
//   * LDS images of q^, k^ and v are rows of tokens whose 16-byte chunks are XORed with bits of the row: k^ and v so that 8 rows x 32 bytes of
//     a transposing read cover every bank, q^ so that 16 rows of a fragment do beside their neighbouring chunks.
//   * 128 columns: two workgroups share a CU, and while one cuts and stages, the other multiplies.  256: one of eight waves (four waves of
//     64 columns spill 250 registers).
// A block with a value that is not finite, and all after it in the run, go token by token on vector arithmetic, for zero times infinity.
// Gates that forget too fast for blocks of more than eight tokens (a quarter and less a token, or now and then all at once) take the
// rest of their run token by token as well, 16 tokens in 32 bits in LDS at a time: 1.8 us a token of both phases with two workgroups a
// CU, where blocks of eight cost 16, and of one the same.  8192 rows, 32 heads, 128 x 128, in blocks down to one token / so, by the mean
// logit behind a lower bound of 0: 0 546 / 527, -2 1064 / 942, -6 2095 / 979, -14 4146 / 994, -40 8252 / 994; token by token out of memory 1559.
// 200 rows 64 / 69, 111 / 119, 199 / 123, 371 / 123, 712 / 123; 206.  The loop stands behind the blocks' and not inside: shared by turns, its
// registers and theirs spilled (302 -> 338 where no gate forgets).
// Pieces: the step's list is walked in runs of `group` pieces of one sequence.  Phase 1 makes the runs' end states from zero,
// chain_kernel turns them into start states, phase 2 computes the outputs; phase 0 walks whole sequences from slot to slot.
#include "common.h"

namespace {

constexpr int RT = 32;     // tokens of a block
constexpr int RD = 128;    // state rows (key channels)
constexpr int TN = 2;      // tiles of 16 value columns a wave holds
constexpr int IMG = RT * RD * 2;  // one part of q^ or k^
constexpr int WALK = 8;    // blocks of so few tokens cost more than the tokens one by one

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
// 1 / x, x and 1 / x normal: the instruction's result (one unit in the last place) with one Newton step
__device__ __forceinline__ float reciprocal(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.f), r, r);
}
// exp(-|x|) = 2^h (1 + e ln 2) with h + e = -|x| / ln 2, h rounded.
__device__ __forceinline__ float exp_minus(float x) {
  const float y = -fabsf(x), h = y * 1.44269504f, e = fmaf(y, 1.44269504f, -h) + y * 1.92596299e-8f;
  const float t2 = __builtin_amdgcn_exp2f(h);
  return h < -200.f ? 0.f : fmaf(t2, e * 0.693147181f, t2);
}
// sigmoid(x) and sigmoid(-x) from t = exp(-|x|): 1 / (1 + t) and t / (1 + t).  The Newton step takes 1 - r (1 + t) without rounding 1 + t
// (1 - r is exact), so that a quotient has its own rounding and little else.
__device__ __forceinline__ void sigmoids(float x, float* s, float* rest) {
  const float t = exp_minus(x), r0 = __builtin_amdgcn_rcpf(1.f + t), r = fmaf(fmaf(-t, r0, 1.f - r0), r0, r0);
  *s = x >= 0.f ? r : t * r;
  *rest = x >= 0.f ? t * r : r;
}
__device__ __forceinline__ float silu(float x) {
  const float t = exp_minus(x), r = __builtin_amdgcn_rcpf(1.f + t), n = x >= 0.f ? x : x * t, q = n * r;
  return fabsf(q) < __builtin_inff() ? fmaf(fmaf(-t, q, n - q), r, q) : q;  // (n - q is exact: n / 2 <= q <= n)
}
__device__ __forceinline__ bool finite(float x) { return fabsf(x) < __builtin_inff(); }

// Two values' parts, packed: x = p0 + p1 + p2, each rounded to the nearest (what is left of 24 bits after two parts fits the third).
// The dot product takes the part off without unpacking it first: x - p0 is exact.
__device__ __forceinline__ void cut2(float x, float y, uint32_t* p) {
  uint32_t lo = 0xbf80u, hi = 0xbf800000u;  // -1 in one half, in registers: as an inline constant the second would mean the first
  asm("" : "+s"(lo), "+s"(hi));
  const bf16x2 first = __builtin_bit_cast(bf16x2, lo), second = __builtin_bit_cast(bf16x2, hi);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    p[i] = pack_bf16x2(x, y);
    if (i == 2) break;
    const bf16x2 part = __builtin_bit_cast(bf16x2, p[i]);
    x = __builtin_amdgcn_fdot2_f32_bf16(part, first, x, false);
    y = __builtin_amdgcn_fdot2_f32_bf16(part, second, y, false);
  }
}

// 16-byte chunk j of row r lies at j ^ swz(r)
__device__ __forceinline__ int swz(int r) { return ((r & 7) << 1) | ((r >> 3) & 1); }

// the same for q^, whose rows are read 16 at a time by four lane groups with neighbouring chunks, and never transposed
__device__ __forceinline__ int swz_q(int r) { return ((r & 1) << 3) | ((r >> 1) & 7); }

__device__ __forceinline__ bf16x8 read_tr(const char* lo, const char* hi) {
  typedef __attribute__((address_space(3))) s16x4* lds_ptr;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)lo);
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)hi);
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// The runs of `group` pieces: how many lie before sequence `want` (or, want < 0, which sequence run `z` belongs to).
// Lanes take a sequence each; every wave computes the same.
struct Run { int seq, first, count; };  // first run of the sequence, its runs
__device__ __forceinline__ Run find_run(const int* __restrict__ seq_pieces, int n_seqs, int group, int z, int want) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int s0 = 0; s0 < n_seqs; s0 += 64) {
    const int s = s0 + lane;
    const int cnt = s < n_seqs ? (seq_pieces[s + 1] - seq_pieces[s] + group - 1) / group : 0;
    int incl = cnt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    int at = -1;
    if (want >= 0) {
      if (want < s0 + 64) at = want - s0;
    } else {
      const unsigned long long hit = __ballot(z < before + incl);
      if (hit) at = __ffsll(hit) - 1;
    }
    if (at >= 0) {
      const int c = __shfl(cnt, at, 64);
      return {s0 + at, before + __shfl(incl, at, 64) - c, c};
    }
    before += __shfl(incl, 63, 64);
  }
  return {-1, 0, 0};
}

// Rows [r0, r1) of run `k` of a sequence.
__device__ __forceinline__ void run_rows(const int* __restrict__ pieces, const int* __restrict__ seq_pieces, int seq, int k, int group,
                                         int* r0, int* r1) {
  const int p0 = seq_pieces[seq] + k * group, p1 = min(p0 + group, seq_pieces[seq + 1]) - 1;
  *r0 = pieces[3 * p0 + 1];
  *r1 = pieces[3 * p1 + 1] + pieces[3 * p1 + 2];
}

struct ScanArgs {
  const uint16_t* proj;
  long p_stride;
  int q_col, k_col, v_col, heads;
  const int* positions;
  const float *decay, *cos_sin;              // fixed decay
  int rot_dims, layout;
  float k_scale;
  const float *gate_bias, *gate_lower;       // gated
  float* state;
  long state_stride;
  const int *seq_cu, *seq_state;
  int n_seqs;
  const int *pieces, *seq_pieces;
  int group;
  float *ws_state, *ws_decay, *out;
};

constexpr float R_MIN = 8.6736174e-19f, R_MAX = 1.1529215e18f;  // 2^-60, 2^60

// LDS: q^ (three parts), k^ (three), v (VT), scores (three) | tables
constexpr int lds_bytes(int nw, int vt, int phase, bool gated) {
  return (phase == 1 ? 1 : 2) * 3 * IMG + vt * RT * nw * 64 + 3 * RT * 64 + (gated ? 2 * nw * RD * 4 : 0) + RD * 4 + 3 * 36 * 4 + 64;
}

// VT: parts of a value (3: q, k and v pass through silu).
template <int NW, bool GATED, int VT, int PHASE>
__global__ __launch_bounds__(NW * 64, 2) void chunk_scan_kernel(const ScanArgs args) {
  constexpr int NT = NW * 64, VD = NW * 32, VROW = VD * 2, VIMG = RT * VROW;
  // what a thread stages: VU 16-byte pieces of v, QU groups of four channels of q and of k
  constexpr int VU = RT * VD / 8 / NT, QU = RT * RD / 4 / NT, GROUPS = RT / QU;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  char* const ks = lds;
  char* const qs = ks + 3 * IMG;                             // not in phase 1
  char* const vs = qs + (PHASE == 1 ? 0 : 3 * IMG);
  char* const ps = vs + VT * VIMG;                           // scores: 32 rows i of 32 tokens, a lane's piece of 8 in its order
  float* const tot = reinterpret_cast<float*>(ps + 3 * RT * 64);   // gated: products of QU rows each
  float* const pn = tot + (GATED ? GROUPS * RD : 0);              // A
  float* const dpow = pn + RD;                               // fixed: d^n, 1 / d^n
  float* const dinv = dpow + 36;
  float* const kpow = dinv + 36;                             // k_scale d^n
  int* const flags = reinterpret_cast<int*>(kpow + 36);
  float* const one = reinterpret_cast<float*>(ps);           // a single token's q, k and v in 32 bits

  const int head = blockIdx.x, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, g = lane >> 4;
  int seq, r0, r1;
  if (PHASE == 0) {
    seq = blockIdx.y, r0 = args.seq_cu[seq], r1 = args.seq_cu[seq + 1];
  } else {
    const Run run = find_run(args.seq_pieces, args.n_seqs, args.group, blockIdx.y, -1);
    if (run.seq < 0) return;
    seq = run.seq;
    run_rows(args.pieces, args.seq_pieces, seq, blockIdx.y - run.first, args.group, &r0, &r1);
  }
  // (the same for all lanes, and said so: bounds, branches and the positions' addresses stay in scalar registers)
  r0 = __builtin_amdgcn_readfirstlane(r0), r1 = __builtin_amdgcn_readfirstlane(r1);
  if (r1 <= r0) return;
  const int slot = __builtin_amdgcn_readfirstlane(args.seq_state[seq]), heads = args.heads;
  float* const out = args.out;
  if (slot < 0) {  // rows of no sequence: their output is zero
    if (PHASE != 1)
      for (int r = r0; r < r1; ++r)
        for (int i = tid; i < VD; i += NT) out[((long)r * heads + head) * VD + i] = 0.f;
    return;
  }
  float* const st = PHASE == 0 ? args.state + (long)slot * args.state_stride + (long)head * RD * VD
                               : args.ws_state + ((long)blockIdx.y * heads + head) * RD * VD;
  const int col0 = wave * 16 * TN;
  f32x4 S[8][TN];
  const bool from_zero = PHASE == 1 || (PHASE == 0 && args.positions[r0] == 0);
  int odd = 0;
#pragma unroll
  for (int t = 0; t < 8; ++t)
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        S[t][n][r] = from_zero ? 0.f : st[(16 * t + 4 * g + r) * VD + col0 + 16 * n + c];
        odd |= !finite(S[t][n][r]);
      }

  // fixed decay: its powers from 64 bits, and the longest block that they allow
  int longest = RT;
  if (!GATED) {
    const double d = args.decay[head];
    if (tid <= RT) {
      double p = 1.0;
      for (int i = 0; i < tid; ++i) p *= d;
      dpow[tid] = (float)p;
      dinv[tid] = (float)(1.0 / p);
      kpow[tid] = (float)(p * args.k_scale);
    }
    const float a = fabsf((float)d);
    float p = 1.f;
    longest = 1;
    while (longest < RT && (p *= a) >= R_MIN && p <= R_MAX) ++longest;
    longest = __builtin_amdgcn_readfirstlane(longest);
  }
  float pgate[GATED ? 4 : 1];  // gated, phase 1: the run's total decay of this thread's channels
  if (GATED)
#pragma unroll
    for (int i = 0; i < 4; ++i) pgate[i] = 1.f;

  auto fresh = [](int x) {  // hides a value: the compiler would keep every address made from it in a register throughout
    asm volatile("" : "+v"(x));
    return x;
  };
  // ---- staging.  Fixed: a thread takes two groups of four channels (a rotation's partners) of QU / 2 rows.  Gated: four channels of
  // QU neighbouring rows.  A group of four channels is half a 16-byte chunk of a row.
  u32x2 rq[QU], rk[QU];
  u32x4 rv[VU];
  f32x4 co[QU / 2], si[QU / 2];
#pragma unroll
  for (int u = 0; u < QU / 2; ++u) co[u] = si[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
  constexpr bool EARLY = NW == 8;  // table rows are asked for a block ahead (four waves have no registers for them)
  const int half = args.rot_dims >> 1, layout = args.layout;
  int ch0, ch1;  // gated: ch0 alone
  if (GATED) {
    ch0 = ch1 = (tid & 31) * 4;
  } else {
    const int a = tid & 15;
    if (layout == 1 || args.rot_dims == 0) {
      ch0 = 8 * a;
      ch1 = 8 * a + 4;
    } else if (4 * a < half) {
      ch0 = 4 * a;
      ch1 = half + 4 * a;
    } else {
      ch0 = args.rot_dims + 8 * (a - half / 4);
      ch1 = ch0 + 4;
    }
  }
  const bool turn = !GATED && args.rot_dims && ch1 < args.rot_dims;
  auto row_of = [&](int u) { return GATED ? (tid >> 5) * QU + u : (tid >> 4) + (u >> 1) * (NT / 16); };
  const int vrow = tid / (VD / 8), vch = (tid % (VD / 8)) * 8;  // of v: row vrow + 8 u
  static_assert(NT / (VD / 8) == 16, "rows a round of v");
  auto fetch = [&](int r) {  // up to 32 rows from r on; rows past the run's are zero
    const int nr = r1 - r;
    const uint16_t* const base = args.proj + (long)r * args.p_stride + head * RD;
    const uint16_t* const vbase = args.proj + (long)r * args.p_stride + args.v_col + head * VD;
#pragma unroll
    for (int u = 0; u < QU; ++u) {
      const int row = row_of(u);
      const uint32_t at = (uint32_t)row * (uint32_t)args.p_stride + (!GATED && (u & 1) ? ch1 : ch0);
      rk[u] = rq[u] = (u32x2){0, 0};
      if (row < nr) {
        rk[u] = *reinterpret_cast<const u32x2*>(base + args.k_col + at);
        if (PHASE != 1) rq[u] = *reinterpret_cast<const u32x2*>(base + args.q_col + at);
      }
    }
#pragma unroll
    for (int u = 0; u < VU; ++u) {
      const int row = vrow + 16 * u;
      rv[u] = (u32x4){0, 0, 0, 0};
      if (row < nr) rv[u] = *reinterpret_cast<const u32x4*>(vbase + (uint32_t)row * (uint32_t)args.p_stride + vch);
    }
  };
  // The table rows of what `fetch` has asked for.  A wave's positions come as scalars, four rows in a row: as vector loads they would
  // have to be waited for, and with them all that was asked for before.
  typedef __attribute__((address_space(4))) const int* scalar_ptr;
  const scalar_ptr positions = (scalar_ptr)(uintptr_t)args.positions;
  i32x4 spos[QU / 2];
  auto fetch_positions = [&](int r) {
    if (GATED || args.rot_dims == 0) return;
#pragma unroll
    for (int u = 0; u < QU / 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) spos[u][i] = positions[min(r + 4 * wave + u * (NT / 16) + i, r1 - 1)];
  };
  auto fetch_turns = [&]() {
    if (!turn) return;
#pragma unroll
    for (int u = 0; u < QU / 2; ++u) {
      const int pos = g & 2 ? (g & 1 ? spos[u][3] : spos[u][2]) : (g & 1 ? spos[u][1] : spos[u][0]);
      const float* cs = args.cos_sin + (long)pos * args.rot_dims + 4 * (tid & 15);
      co[u] = *reinterpret_cast<const f32x4*>(cs);
      si[u] = *reinterpret_cast<const f32x4*>(cs + half);
    }
  };
  auto put_k = [&](int row, int ch, const float* x) {  // four channels in their parts
    uint32_t a[3], b[3];
    cut2(x[0], x[1], a);
    cut2(x[2], x[3], b);
    char* const p = ks + row * 256 + (((ch >> 3) ^ swz(row)) << 4) + (ch & 4) * 2;
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x2*>(p + i * IMG) = (u32x2){a[i], b[i]};
  };
  auto put_q = [&](int row, int ch, const float* x) {  // in the order of the state's registers: chunk 4 u + g: channels 32 u + 4 g and 32 u + 16 + 4 g
    uint32_t a[3], b[3];
    cut2(x[0], x[1], a);
    cut2(x[2], x[3], b);
    char* const p = qs + row * 256 + ((((ch >> 5) * 4 + ((ch >> 2) & 3)) ^ swz_q(row)) << 4) + ((ch >> 4) & 1) * 8;
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x2*>(p + i * IMG) = (u32x2){a[i], b[i]};
  };
  // gated: s = sigmoid(x) and 1 - s of a fetched logit, from one exponential: 1 - a would lose what a near 1 rounds away
  auto gate = [&](int u, int i, f32x4 bias, float* s, float* rest) {
    sigmoids((i & 1 ? bf16hi(rk[u][i >> 1]) : bf16lo(rk[u][i >> 1])) + bias[i], s, rest);
  };
  // registers -> LDS for the first nb rows; bit 0: a value is not finite, bit 1: out of range.  Rows past them: k^ is zero, q^ and v
  // are never used with anything else.
  auto stage = [&](int nb) {
    u16x2 top = {0, 0};          // largest exponents of what came in
    float sum = 0.f;             // becomes NaN with anything that is not finite
    float least = 1.f, most = 1.f;
    auto check = [&](uint32_t w) { top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, w & 0x7fff7fffu)); };
    if (GATED) {
      float a[QU][4], k[QU][4], R[QU][4];
      const f32x4 bias = *reinterpret_cast<const f32x4*>(args.gate_bias + head * RD + ch0);
      const f32x4 low = *reinterpret_cast<const f32x4*>(args.gate_lower + head * RD + ch0);
#pragma unroll
      for (int u = 0; u < QU; ++u) {
        const bool in = row_of(u) < nb;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float s, rest;
          gate(u, i, bias, &s, &rest);
          a[u][i] = in ? low[i] + (1.f - low[i]) * s : 1.f;
          k[u][i] = in ? (1.f - low[i]) * rest : 0.f;
          sum = fmaf(a[u][i], 0.f, sum);
        }
      }
      float p[4] = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
      for (int u = QU - 1; u >= 0; --u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          R[u][i] = p[i];
          p[i] *= a[u][i];
        }
      *reinterpret_cast<f32x4*>(tot + (tid >> 5) * RD + ch0) = (f32x4){p[0], p[1], p[2], p[3]};
      __syncthreads();
      f32x4 later = {1.f, 1.f, 1.f, 1.f};
      for (int w = GROUPS - 1; w > (tid >> 5); --w) later *= *reinterpret_cast<const f32x4*>(tot + w * RD + ch0);
      if (tid < 32) *reinterpret_cast<f32x4*>(pn + ch0) = later * (f32x4){p[0], p[1], p[2], p[3]};
#pragma unroll
      for (int u = 0; u < QU; ++u) {
        float q[4];
        if (PHASE != 1) check(rq[u][0]), check(rq[u][1]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float Rr = R[u][i] * later[i];
          least = fminf(least, fabsf(Rr));
          most = fmaxf(most, fabsf(Rr));
          k[u][i] *= Rr;
          if (PHASE != 1) {
            q[i] = silu(i & 1 ? bf16hi(rq[u][i >> 1]) : bf16lo(rq[u][i >> 1])) * reciprocal(Rr);
            most = fmaxf(most, fabsf(q[i]) * 1e-16f);
          }
        }
        const int ch = fresh(ch0);
        put_k(row_of(u), ch, k[u]);
        if (PHASE != 1) put_q(row_of(u), ch, q);
      }
    } else {
#pragma unroll
      for (int u = 0; u < QU / 2; ++u) {
        const int row = row_of(2 * u);
        auto turned = [&](const u32x2* w, float factor, float* raw, auto put) {
          float x0[4] = {bf16lo(w[0][0]), bf16hi(w[0][0]), bf16lo(w[0][1]), bf16hi(w[0][1])};
          float x1[4] = {bf16lo(w[1][0]), bf16hi(w[1][0]), bf16lo(w[1][1]), bf16hi(w[1][1])};
#pragma unroll
          for (int i = 0; i < 4; ++i) check(w[i >> 1][i & 1]);
          if (VT == 3) {
#pragma unroll
            for (int i = 0; i < 4; ++i) x0[i] = silu(x0[i]), x1[i] = silu(x1[i]);
          }
          if (turn) {
            if (layout == 0) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float p = x0[i], q = x1[i];
                x0[i] = p * co[u][i] - q * si[u][i];
                x1[i] = q * co[u][i] + p * si[u][i];
              }
            } else {
#pragma unroll
              for (int i = 0; i < 4; i += 2) {
                const float p = x0[i], q = x0[i + 1], p1 = x1[i], q1 = x1[i + 1];
                x0[i] = p * co[u][i >> 1] - q * si[u][i >> 1];
                x0[i + 1] = q * co[u][i >> 1] + p * si[u][i >> 1];
                x1[i] = p1 * co[u][2 + (i >> 1)] - q1 * si[u][2 + (i >> 1)];
                x1[i + 1] = q1 * co[u][2 + (i >> 1)] + p1 * si[u][2 + (i >> 1)];
              }
            }
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            x0[i] *= factor;
            x1[i] *= factor;
            most = fmaxf(most, fmaxf(fabsf(x0[i]), fabsf(x1[i])) * 1e-16f);
            if (nb == 1 && row == 0) raw[ch0 + i] = x0[i], raw[ch1 + i] = x1[i];  // (a block's last token has factors of one)
          }
          put(row, fresh(ch0), x0);
          put(row, fresh(ch1), x1);
        };
        const int back = max(nb - 1 - row, 0);
        turned(rk + 2 * u, row < nb ? kpow[back] : 0.f, one + RD, put_k);
        if (PHASE != 1) turned(rq + 2 * u, dinv[back], one, put_q);
      }
    }
#pragma unroll
    for (int u = 0; u < VU; ++u) {
      const int row = vrow + 16 * u;
      const u32x4 w = rv[u];
      char* const to = vs + row * VROW + (((vch >> 3) ^ swz(row)) << 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) check(w[i]);
      if (VT == 3) {
        u32x4 part[3];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t p[3];
          cut2(silu(bf16lo(w[i])), silu(bf16hi(w[i])), p);
          part[0][i] = p[0], part[1][i] = p[1], part[2][i] = p[2];
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4*>(to + p * VIMG) = part[p];
      } else {
        *reinterpret_cast<u32x4*>(to) = w;
      }
      if (!GATED && nb == 1 && row == 0)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          one[2 * RD + vch + 2 * i] = VT == 3 ? silu(bf16lo(w[i])) : bf16lo(w[i]);
          one[2 * RD + vch + 2 * i + 1] = VT == 3 ? silu(bf16hi(w[i])) : bf16hi(w[i]);
        }
    }
    const bool odd_in = top[0] >= 0x7f80 || top[1] >= 0x7f80 || !(sum == 0.f);
    const bool wide = !(least >= R_MIN) || !(most <= R_MAX);
    const int any = (__ballot(odd_in) != 0 ? 1 : 0) | (__ballot(wide) != 0 ? 2 : 0);
    if (lane == 0) flags[wave] = any;
  };

  // gated: 16 tokens (from the 16 * h-th fetched row on) for the walk token by token: k | a | q in 32 bits, and with the first all of v
  float* const walk_k = reinterpret_cast<float*>(ks);
  float* const walk_a = walk_k + 16 * RD;
  float* const walk_q = reinterpret_cast<float*>(qs);
  static_assert(2 * 16 * RD * 4 <= 3 * IMG && 16 * RD * 4 <= 3 * IMG, "place of the walk's operands");
  auto stage_walk = [&](int h) {
    const f32x4 bias = *reinterpret_cast<const f32x4*>(args.gate_bias + head * RD + ch0);
    const f32x4 low = *reinterpret_cast<const f32x4*>(args.gate_lower + head * RD + ch0);
#pragma unroll
    for (int u = 0; u < QU; ++u) {
      if (row_of(u) >> 4 != h) continue;
      f32x4 a, k, q;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float s, rest;
        gate(u, i, bias, &s, &rest);
        a[i] = low[i] + (1.f - low[i]) * s;
        k[i] = (1.f - low[i]) * rest;
        q[i] = silu(i & 1 ? bf16hi(rq[u][i >> 1]) : bf16lo(rq[u][i >> 1]));
      }
      const int at = fresh((row_of(u) & 15) * RD + ch0);
      *reinterpret_cast<f32x4*>(walk_k + at) = k;
      *reinterpret_cast<f32x4*>(walk_a + at) = a;
      if (PHASE != 1) *reinterpret_cast<f32x4*>(walk_q + at) = q;
    }
#pragma unroll
    for (int u = 0; u < VU; ++u)
      if (h == 0) *reinterpret_cast<u32x4*>(vs + (vrow + 16 * u) * VROW + (((vch >> 3) ^ swz(vrow + 16 * u)) << 4)) = rv[u];
  };

  // fragment addresses within an image; a tile further is an XOR away
  const int row16 = c * 256 + ((g >> 1) ^ swz(c)) * 16 + (g & 1) * 8;  // k^ for the scores: channels 4 g .. of tile 0
  const int row_q = c * 256 + (g ^ swz_q(c)) * 16;
  const int tr_row = 4 * g + (c >> 2);                                  // transposing reads: rows 4 g .. 4 g + 3 and 16 more
  const int tr_chunk = (((c >> 1) & 1) ^ swz(tr_row)) * 16 + (c & 1) * 8;  // four channels 4 (c % 4) of sixteen

  __syncthreads();
  odd = __builtin_amdgcn_readfirstlane(__syncthreads_or(odd));
  int r = r0, cap = longest, good = 0;
  int wait = 1;   // good blocks of 16 tokens and more before a longer one is tried: doubled where that failed
  // gated: blocks of WALK tokens and fewer, and tries that end with one, before the rest of the run goes token by token (one token that
  // forgets all takes eight of them; in a run of few tokens they would be most of its time)
  int left = max(1, min(12, (r1 - r0) / 32));
  bool walk = false;
  fetch(r);
  fetch_positions(r);
  if (EARLY) fetch_turns();
  while (r < r1) {
    if (!EARLY) fetch_turns();
    int nb = min(odd && !GATED ? 1 : cap, r1 - r);
    walk = GATED && (odd || left <= 0);
    while (!walk) {
      __syncthreads();  // the block before is done with LDS
      stage(nb);
      __syncthreads();
      int any = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) any |= flags[w];
      any = __builtin_amdgcn_readfirstlane(any);
      if (any & 1) {
        odd = 1;
        if (nb == 1) break;
        nb = 1;
      } else if ((any & 2) && nb > 1) {
        nb = cap = nb >> 1;
        good = 0;
        if (nb > WALK) wait = min(2 * wait, 16);
        else --left;
      } else {
        break;
      }
      walk = GATED && (odd || left <= 0);
    }
    if (walk) break;
    if (nb <= WALK) --left;
    if (nb == longest) wait = 1;
    if (nb == cap && cap < longest && ++good >= (cap > WALK ? wait : 1)) cap = min(2 * cap, longest), good = 0;
    const int nx = r + nb;
    if (nx < r1) {
      fetch(nx);
      fetch_positions(nx);
    }

    // S' = A S0
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      f32x4 A;
      if (GATED) A = *reinterpret_cast<const f32x4*>(pn + 16 * t + 4 * g);
      else A = dpow[nb] * (f32x4){1.f, 1.f, 1.f, 1.f};
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) S[t][n][q] *= A[q];
    }
    if (GATED && PHASE == 1 && tid < 32)
#pragma unroll
      for (int i = 0; i < 4; ++i) pgate[i] *= pn[ch0 + i];
    if (!GATED && odd) {  // one token on vector arithmetic
      float o[TN];
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const float v = one[2 * RD + col0 + 16 * n + c];
        o[n] = 0.f;
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            S[t][n][q] = fmaf(one[RD + 16 * t + 4 * g + q], v, S[t][n][q]);
            if (PHASE != 1) o[n] = fmaf(S[t][n][q], one[16 * t + 4 * g + q], o[n]);
          }
        if (PHASE != 1) {
          o[n] += __shfl_xor(o[n], 16, 64);
          o[n] += __shfl_xor(o[n], 32, 64);
          if (g == 0) out[((long)r * heads + head) * VD + col0 + 16 * n + c] = o[n];
        }
      }
      if (EARLY && nx < r1) fetch_turns();
      r = nx;
      continue;
    }
    const bool two = nb > 16;
    const int at_q = fresh(row_q), at_k = fresh(row16);
    f32x4 O[2][TN], small[2][TN];  // small: products of the parts below the first, whose sums round finer
    if (PHASE != 1) {
      // scores, transposed (tile im of rows i, jm of tokens j); the three tiles go to waves 0 to 2
      if (wave < 3 && (wave == 0 || two)) {
        const int im = wave > 0, jm = wave > 1;
        f32x4 P = {0.f, 0.f, 0.f, 0.f}, small = P, small2 = P;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          bf16x8 kf[3], qf[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            const char* k = ks + p * IMG + jm * 4096;
            const u32x2 lo = *reinterpret_cast<const u32x2*>(k + (at_k ^ (u << 6)));
            const u32x2 hi = *reinterpret_cast<const u32x2*>(k + (at_k ^ (u << 6) ^ 32));
            kf[p] = __builtin_bit_cast(bf16x8, (u32x4){lo[0], lo[1], hi[0], hi[1]});
            qf[p] = *reinterpret_cast<const bf16x8*>(qs + p * IMG + im * 4096 + (at_q ^ (u << 6)));
          }
          small = mma(kf[0], qf[2], small);
          small2 = mma(kf[1], qf[1], small2);
          P = mma(kf[0], qf[0], P);
          small = mma(kf[2], qf[0], small);
          small2 = mma(kf[0], qf[1], small2);
          small = mma(kf[1], qf[0], small);
        }
        P += small + small2;
        const int i = 16 * im + c;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (16 * jm + 4 * g + q > i) P[q] = 0.f;
        uint32_t a[3], b[3];
        cut2(P[0], P[1], a);
        cut2(P[2], P[3], b);
        char* const to = ps + i * 64 + ((g ^ ((c >> 2) & 3)) << 4) + jm * 8;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          *reinterpret_cast<u32x2*>(to + p * RT * 64) = (u32x2){a[p], b[p]};
          if (im == 0) *reinterpret_cast<u32x2*>(to + p * RT * 64 + 8) = (u32x2){0, 0};  // tokens 16 .. 31 of rows 0 .. 15
        }
      }
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) O[m][n] = small[m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
      // the next tiles of the state are cut up between the matrix instructions of the ones before
      bf16x8 sf[2][3];
      auto cut_state = [&](int x, bf16x8* to) {  // tiles 2 u, 2 u + 1 of column tile n, x = TN u + n
        const int u = x / TN, n = x % TN;
        u32x4 w[3];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t p[3];
          cut2(S[2 * u + (i >> 1)][n][2 * (i & 1)], S[2 * u + (i >> 1)][n][2 * (i & 1) + 1], p);
          w[0][i] = p[0], w[1][i] = p[1], w[2][i] = p[2];
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) to[p] = __builtin_bit_cast(bf16x8, w[p]);
      };
      cut_state(0, sf[0]);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        bf16x8 qf[2][3];
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int p = 0; p < 3; ++p)
            qf[m][p] = *reinterpret_cast<const bf16x8*>(qs + p * IMG + m * 4096 + (at_q ^ (u << 6)));
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          const int x = TN * u + n;
          if (x + 1 < 4 * TN) cut_state(x + 1, sf[(x + 1) & 1]);
          const bf16x8* f = sf[x & 1];
          small[0][n] = mma(f[0], qf[0][2], small[0][n]);
          small[1][n] = mma(f[0], qf[1][2], small[1][n]);
          O[0][n] = mma(f[0], qf[0][0], O[0][n]);
          O[1][n] = mma(f[0], qf[1][0], O[1][n]);
          small[0][n] = mma(f[1], qf[0][1], small[0][n]);
          small[1][n] = mma(f[1], qf[1][1], small[1][n]);
          small[0][n] = mma(f[2], qf[0][0], small[0][n]);
          small[1][n] = mma(f[2], qf[1][0], small[1][n]);
          small[0][n] = mma(f[0], qf[0][1], small[0][n]);
          small[1][n] = mma(f[0], qf[1][1], small[1][n]);
          small[0][n] = mma(f[1], qf[0][0], small[0][n]);
          small[1][n] = mma(f[1], qf[1][0], small[1][n]);
#pragma unroll
          for (int i = 0; NW == 4 && i < 12; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
          }
        }
      }
      __syncthreads();  // the scores are there
    }
    if (EARLY && nx < r1) fetch_turns();
    bf16x8 vf[VT][TN];
    const int at_v = fresh(tr_row * VROW + (tr_chunk ^ (wave * TN << 5))), at_t = fresh(tr_row * 256 + tr_chunk);
#pragma unroll
    for (int p = 0; p < VT; ++p)
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const char* v = vs + p * VIMG + (at_v ^ (n << 5));
        vf[p][n] = read_tr(v, v + 16 * VROW);
      }
    if (PHASE != 1) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if (m && !two) break;
        bf16x8 pf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          pf[p] = *reinterpret_cast<const bf16x8*>(ps + p * RT * 64 + (16 * m + c) * 64 + ((g ^ ((c >> 2) & 3)) << 4));
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int vp = min(VT - 1, 2 - p); vp >= 0; --vp)
#pragma unroll
            for (int n = 0; n < TN; ++n) {
              if (p + vp) small[m][n] = mma(vf[vp][n], pf[p], small[m][n]);
              else O[m][n] = mma(vf[0][n], pf[0], O[m][n]);
            }
        const int i = 16 * m + c;
        if (i < nb) {
          float* const to = out + ((long)r * heads + head) * VD + ((uint32_t)i * (uint32_t)(heads * VD) + col0 + 4 * g);
#pragma unroll
          for (int n = 0; n < TN; ++n) *reinterpret_cast<f32x4*>(to + 16 * n) = O[m][n] + small[m][n];
        }
      }
    }
    // a tile's operands are read while the tile before is multiplied (left alone the compiler waits for every read by itself; with the
    // positions as scalars, 4 % gated, 3 % fixed)
    bf16x8 kf[2][3];
    auto read_k = [&](int t) {
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const char* k = ks + p * IMG + (at_t ^ (t << 5));
        kf[t & 1][p] = read_tr(k, k + 16 * 256);
      }
    };
    read_k(0);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      if (t + 1 < 8) read_k(t + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int vp = min(VT - 1, 2 - p); vp >= 0; --vp)
#pragma unroll
          for (int n = 0; n < TN; ++n) S[t][n] = mma(kf[t & 1][p], vf[vp][n], S[t][n]);
      __builtin_amdgcn_sched_barrier(0);
    }
    r = nx;
  }
  // token by token, the same channels and columns a lane
  while (GATED && r < r1) {
    const int rows = min(RT, r1 - r), nx = r + rows;
    for (int h = 0; 16 * h < rows; ++h) {
      const int m = min(rows - 16 * h, 16);
      __syncthreads();  // what was there before has been read
      stage_walk(h);
      if (16 * h + m == rows && nx < r1) fetch(nx);
      __syncthreads();
      if (PHASE == 1 && tid < 32) {
#pragma unroll 4
        for (int i = 0; i < m; ++i) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(walk_a + i * RD + ch0);
#pragma unroll
          for (int j = 0; j < 4; ++j) pgate[j] *= a[j];
        }
      }
      for (int i = 0; i < m; ++i) {
        float v[TN], o[TN][2];  // two sums a column: a row's channels in one chain of 32 round more than the sums of before
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          const int col = fresh(col0 + 16 * n + c), row = 16 * h + i;
          v[n] = bf16_bits_to_f32(*reinterpret_cast<const uint16_t*>(vs + row * VROW + (((col >> 3) ^ swz(row)) << 4) + (col & 7) * 2));
          o[n][0] = o[n][1] = 0.f;
        }
        f32x4 a[2], k[2], q[2];  // a tile's are read while the tile before is computed
        const int at = fresh(i * RD + 4 * g);
        auto read = [&](int t) {
          a[t & 1] = *reinterpret_cast<const f32x4*>(walk_a + at + 16 * t);
          k[t & 1] = *reinterpret_cast<const f32x4*>(walk_k + at + 16 * t);
          if (PHASE != 1) q[t & 1] = *reinterpret_cast<const f32x4*>(walk_q + at + 16 * t);
        };
        read(0);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          if (t + 1 < 8) read(t + 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              S[t][n][j] = fmaf(k[t & 1][j], v[n], S[t][n][j] * a[t & 1][j]);
              if (PHASE != 1) o[n][t & 1] = fmaf(S[t][n][j], q[t & 1][j], o[n][t & 1]);
            }
          __builtin_amdgcn_sched_barrier(0);
        }
        if (PHASE != 1)
#pragma unroll
          for (int n = 0; n < TN; ++n) {
            float sum = o[n][0] + o[n][1];
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            if (g == 0) out[((long)(r + 16 * h + i) * heads + head) * VD + col0 + 16 * n + c] = sum;
          }
      }
    }
    r = nx;
  }
  if (PHASE != 2) {
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) st[(16 * t + 4 * g + q) * VD + col0 + 16 * n + c] = S[t][n][q];
    if (GATED && PHASE == 1 && tid < 32)
      *reinterpret_cast<f32x4*>(args.ws_decay + ((long)blockIdx.y * heads + head) * RD + ch0) = (f32x4){pgate[0], pgate[1], pgate[2], pgate[3]};
  }
}

// Walks a sequence's runs in order: ws_state[run] (its end state from zero) becomes its start state, the sequence's slot
// gets the end state.  Four state elements a thread; the loads of four runs are in flight together.
template <bool GATED>
__global__ __launch_bounds__(256) void chain_kernel(const ScanArgs args, int vdim) {
  const int seq = blockIdx.z, head = blockIdx.y, e = (blockIdx.x * 256 + threadIdx.x) * 4, elems = RD * vdim;
  const int slot = args.seq_state[seq], heads = args.heads;
  if (slot < 0 || args.seq_cu[seq + 1] <= args.seq_cu[seq]) return;
  const Run run = find_run(args.seq_pieces, args.n_seqs, args.group, 0, seq);
  float* const st = args.state + (long)slot * args.state_stride + (long)head * elems + e;
  const double d = GATED ? 0.0 : args.decay[head];
  const bool fresh = args.positions[args.seq_cu[seq]] == 0;
  f32x4 S;
#pragma unroll
  for (int i = 0; i < 4; ++i) S[i] = fresh ? 0.f : st[i];
  const long step = (long)heads * elems;
  float* const w = args.ws_state + ((long)run.first * heads + head) * elems + e;
  for (int k0 = 0; k0 < run.count; k0 += 4) {
    f32x4 end[4];
    float f[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k0 + k >= run.count) continue;
      end[k] = *reinterpret_cast<const f32x4*>(w + (k0 + k) * step);
      if (GATED) {
        f[k] = args.ws_decay[((long)(run.first + k0 + k) * heads + head) * RD + e / vdim];
      } else {
        int r0, r1;
        run_rows(args.pieces, args.seq_pieces, seq, k0 + k, args.group, &r0, &r1);
        double p = 1.0, b = d;
        for (int n = r1 - r0; n; n >>= 1, b *= b)
          if (n & 1) p *= b;
        f[k] = (float)p;
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k0 + k >= run.count) break;
      *reinterpret_cast<f32x4*>(w + (k0 + k) * step) = S;
#pragma unroll
      for (int i = 0; i < 4; ++i) S[i] = fmaf(f[k], S[i], end[k][i]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) st[i] = S[i];
}

template <int NW, bool GATED, int VT, int PHASE>
int launch(const ScanArgs& args, int units, hipStream_t stream) {
  constexpr int LDS = lds_bytes(NW, VT, PHASE, GATED);
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)chunk_scan_kernel<NW, GATED, VT, PHASE>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess)
      return -2;
    attr_set = true;
  }
  chunk_scan_kernel<NW, GATED, VT, PHASE><<<dim3(args.heads, units), NW * 64, LDS, stream>>>(args);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

template <int NW, bool GATED, int VT>
int scan(ScanArgs& args, int n_pieces, hipStream_t stream) {
  if (n_pieces <= 0) return launch<NW, GATED, VT, 0>(args, args.n_seqs, stream);
  constexpr int PLACES = NW == 8 ? 256 : 512;  // workgroups that the chip holds at once
  args.group = (n_pieces * args.heads + PLACES - 1) / PLACES;
  const int runs = n_pieces / args.group + args.n_seqs;
  int rc = launch<NW, GATED, VT, 1>(args, runs, stream);
  if (rc) return rc;
  chain_kernel<GATED><<<dim3(RD * NW * 32 / 1024, args.heads, args.n_seqs), 256, 0, stream>>>(args, NW * 32);
  return launch<NW, GATED, VT, 2>(args, runs, stream);
}

}  // namespace

// proj bf16 [rows, p_stride] with q, k (or gate logits; heads of 128 channels) and v (heads of vdim channels) at their columns; state:
// the slots of this layer; out fp32 [rows, heads, vdim].  Fixed decay: decay [heads], rot_dims a multiple of 8 (layout 0 or 1) or 0; act:
// q, k and v pass through silu (no rotation then).  Gated (decay null): gate_bias, gate_lower [heads, 128].  pieces / seq_pieces as in
// vpsa_recurrent_scan with ws_state fp32 [n_pieces, heads, 128, vdim] and, gated, ws_decay fp32 [n_pieces, heads, 128]; n_pieces 0: whole
// sequences.  vdim 128 or 256; every row and column start on 16-byte boundaries.
VPSA_EXPORT int vpsa_chunk_scan(const void* proj, long p_stride, int q_col, int k_col, int v_col, int heads, int vdim, float* state,
                                long state_stride, const int* seq_cu, const int* seq_state, int n_seqs, const int* positions,
                                const float* decay, const float* cos_sin, int rot_dims, int layout, float k_scale, int act,
                                const float* gate_bias, const float* gate_lower, float* out, const int* pieces,
                                const int* seq_pieces, int n_pieces, float* ws_state, float* ws_decay, hipStream_t stream) {
  if (n_seqs <= 0 || heads <= 0) return 0;
  if ((vdim != 128 && vdim != 256) || (rot_dims & 7) || rot_dims > RD || (act && rot_dims) || n_seqs > 65535) return 1;
  if (((uintptr_t)proj & 15) || (p_stride & 7) || ((q_col | k_col | v_col) & 7)) return 2;
  if (rot_dims && ((uintptr_t)cos_sin & 15)) return 2;
  if (!decay && (((uintptr_t)gate_bias | (uintptr_t)gate_lower) & 15)) return 2;
  ScanArgs args = {(const uint16_t*)proj, p_stride, q_col, k_col, v_col, heads, positions, decay, cos_sin, rot_dims, layout, k_scale,
                   gate_bias, gate_lower, state, state_stride, seq_cu, seq_state, n_seqs, pieces, seq_pieces, 1, ws_state, ws_decay, out};
  if (!decay) return vdim == 256 ? scan<8, true, 1>(args, n_pieces, stream) : scan<4, true, 1>(args, n_pieces, stream);
  if (act) return vdim == 256 ? scan<8, false, 3>(args, n_pieces, stream) : scan<4, false, 3>(args, n_pieces, stream);
  return vdim == 256 ? scan<8, false, 1>(args, n_pieces, stream) : scan<4, false, 1>(args, n_pieces, stream);
}
