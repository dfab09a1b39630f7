// The fixed-decay recurrence S <- d S + k_t v_t^T, o_t = S^T q_t over prompt chunks, on the matrix cores in 32-bit.
//
// For decays that the blocks of chunk_scan.hip would have to be short for, or that the host does not know: those divide by products of
// decays, which has to stay in range over a block's 32 tokens (0.26 a token).  Here nothing is divided, and every decay takes the same
// time: 8192 rows, 32 heads, 128 x 128 / 128 x 256: 360 / 672 us, chunk_scan.hip 229 / 335 with decays of 0.97, 357 / 506 of 0.1, 604 / 894 of
// 0.01, 1447 / 2179 of 1e-6; 200 rows 48 / 64, there 43 / 48, 57 / 62, 78 / 85, 143 / 158.  Token by token (seqmix.hip) every token costs two
// vector operations per state element: 2.29 ms for 128 x 256.  Blocks of RT = 32 tokens
// are contractions (d^n: the n-th power, S0: the state before the block, n: its tokens)
//     o_i = d^(i+1) S0^T q_i + sum_(j <= i) d^(i-j) (q_i . k_j) v_j        S = d^n S0 + sum_j d^(n-1-j) k_j v_j^T
// on v_mfma_f32_16x16x4 (32-bit operands and sums: nothing is rounded to 16 bits; 154 TFLOP/s in a large product here).
// The powers come from a table made in 64 bits, so decays need no lower bound.
//   * A workgroup holds a head's whole 128 x (32 per wave) state in accumulators, so q, k and the 32 x 32 scores are made
//     once for all value columns.  A wave owns 32 columns: 64 accumulators.
//   * The accumulator layout of S (lane (c, g): rows 4 g + r of a 16-row tile, column c) is used as the B operand of
//     S0^T q as it is: step r contracts rows {4 g + r}, and A reads channels 4 g .. 4 g + 3 of q in one 16-byte LDS read.
//     The same order over tokens lets one set of value operands serve scores x V and K^T V.
//   * LDS rows are padded by four floats: four lane groups that read rows 4 apart then fall on different banks.
//   * q and k are rotated (or pass through silu) on their way into LDS: no prepared copy in memory.
// Pieces: the step's list is walked in runs of `group` pieces of one sequence, enough runs for two rounds of workgroups (8192
// rows, 32 heads: 512 of 576 rows; runs of 96 rows moved 1.4 GB of piece states).  Phase 1 makes the runs' end states from
// zero, retention_chain_kernel turns them into start states, phase 2 computes the outputs.
// Measured: 8192 rows of two sequences, 32 heads, 128 x 256, rotated: 2.29 -> 0.70 ms (phases 0.22 and 0.43 ms with the matrix
// cores busy for half of it, the chain 0.05); 300 rows of 16 heads 183 -> 62 us.  Two waves per SIMD: four (128 registers)
// spill 79 of them and take 0.90 ms.
#include "common.h"

namespace {

constexpr int RT = 32;          // tokens of a block
constexpr int RD = 128;         // state rows (key channels)
constexpr int QS = RD + 4;      // LDS row of q, k
constexpr int PS = RT + 4;      // LDS row of the scores

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float silu(float x) { return x * (1.f / (1.f + expf(-x))); }

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

template <int NW, int PHASE>
__global__ __launch_bounds__(NW * 64, 2) void retention_kernel(
    const uint16_t* __restrict__ proj, long p_stride, int q_col, int k_col, int v_col, int heads,
    const int* __restrict__ positions, const float* __restrict__ decay, const float* __restrict__ cos_sin, int rot_dims,
    int layout, float k_scale, int act, const int* __restrict__ seq_state, int n_seqs, const int* __restrict__ pieces,
    const int* __restrict__ seq_pieces, int group, float* __restrict__ ws_state, float* __restrict__ out) {
  constexpr int VD = NW * 32, VS = VD + 4, NT = NW * 64, UNITS = RT * 16 / NT;
  __shared__ __attribute__((aligned(16))) float qs[PHASE == 2 ? RT * QS : 4];
  __shared__ __attribute__((aligned(16))) float ks[RT * QS];
  __shared__ __attribute__((aligned(16))) float vs[RT * VS];
  __shared__ __attribute__((aligned(16))) float ps[PHASE == 2 ? RT * PS : 4];
  __shared__ float pw[RT + 1];
  const int head = blockIdx.x, z = blockIdx.y;
  const Run run = find_run(seq_pieces, n_seqs, group, z, -1);
  if (run.seq < 0) return;
  int r0, r1;
  run_rows(pieces, seq_pieces, run.seq, z - run.first, group, &r0, &r1);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int col0 = wave * 32 + c;
  if (seq_state[run.seq] < 0) {  // rows of no sequence: their output is zero
    if (PHASE == 2)
      for (int r = r0; r < r1; ++r)
        for (int i = tid; i < VD; i += NT) out[((long)r * heads + head) * VD + i] = 0.f;
    return;
  }
  if (tid <= RT) {
    double p = 1.0;
    const double d = decay[head];
    for (int i = 0; i < tid; ++i) p *= d;
    pw[tid] = (float)p;
  }
  float* st = ws_state + ((long)z * heads + head) * RD * VD;
  f32x4 S[8][2];
#pragma unroll
  for (int t = 0; t < 8; ++t)
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[t][n][r] = PHASE == 2 ? st[(16 * t + 4 * g + r) * VD + col0 + 16 * n] : 0.f;

  // A unit is two groups of four channels of one row of q and k; a rotation's partners lie in the same unit.
  const int half = rot_dims >> 1;
  u32x2 rq[UNITS][2], rk[UNITS][2];
  u32x4 rv[2];
  int rpos[UNITS];
  auto chans = [&](int a, int* g0, int* g1) {
    if (layout == 1 || rot_dims == 0) {
      *g0 = 8 * a;
      *g1 = 8 * a + 4;
    } else if (4 * a < half) {
      *g0 = 4 * a;
      *g1 = half + 4 * a;
    } else {
      *g0 = rot_dims + 8 * (a - half / 4);
      *g1 = *g0 + 4;
    }
  };
  auto fetch = [&](int r, int nb) {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int e = tid + u * NT, row = e >> 4;
      int g0, g1;
      chans(e & 15, &g0, &g1);
      if (row < nb) {
        const uint16_t* p = proj + (long)(r + row) * p_stride + (long)head * RD;
        rk[u][0] = *reinterpret_cast<const u32x2*>(p + k_col + g0);
        rk[u][1] = *reinterpret_cast<const u32x2*>(p + k_col + g1);
        if (PHASE == 2) {
          rq[u][0] = *reinterpret_cast<const u32x2*>(p + q_col + g0);
          rq[u][1] = *reinterpret_cast<const u32x2*>(p + q_col + g1);
        }
        rpos[u] = rot_dims ? positions[r + row] : 0;
      } else {
        rk[u][0] = rk[u][1] = rq[u][0] = rq[u][1] = (u32x2){0, 0};
        rpos[u] = 0;
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = tid + u * NT, row = e / (VD / 8), ch = (e % (VD / 8)) * 8;
      rv[u] = row < nb ? *reinterpret_cast<const u32x4*>(proj + (long)(r + row) * p_stride + v_col + (long)head * VD + ch)
                       : (u32x4){0, 0, 0, 0};
    }
  };
  // registers -> LDS; tells whether a value is not finite
  auto stage = [&]() {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int e = tid + u * NT, row = e >> 4, a = e & 15;
      int g0, g1;
      chans(a, &g0, &g1);
      const bool turn = rot_dims && g1 < rot_dims;
      f32x4 co = {1.f, 1.f, 1.f, 1.f}, si = {0.f, 0.f, 0.f, 0.f};
      if (turn) {
        const float* cs = cos_sin + (long)rpos[u] * rot_dims + 4 * a;
        co = *reinterpret_cast<const f32x4*>(cs);
        si = *reinterpret_cast<const f32x4*>(cs + half);
      }
      auto put = [&](const u32x2* w, float* dst, float scale) {
        f32x4 x0 = {bf16lo(w[0][0]), bf16hi(w[0][0]), bf16lo(w[0][1]), bf16hi(w[0][1])};
        f32x4 x1 = {bf16lo(w[1][0]), bf16hi(w[1][0]), bf16lo(w[1][1]), bf16hi(w[1][1])};
        if (act) {
#pragma unroll
          for (int i = 0; i < 4; ++i) x0[i] = silu(x0[i]), x1[i] = silu(x1[i]);
        }
        if (turn) {
          if (layout == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float p = x0[i], q = x1[i];
              x0[i] = p * co[i] - q * si[i];
              x1[i] = q * co[i] + p * si[i];
            }
          } else {
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
              const float p = x0[i], q = x0[i + 1], p1 = x1[i], q1 = x1[i + 1];
              x0[i] = p * co[i >> 1] - q * si[i >> 1];
              x0[i + 1] = q * co[i >> 1] + p * si[i >> 1];
              x1[i] = p1 * co[2 + (i >> 1)] - q1 * si[2 + (i >> 1)];
              x1[i + 1] = q1 * co[2 + (i >> 1)] + p1 * si[2 + (i >> 1)];
            }
          }
        }
        *reinterpret_cast<f32x4*>(dst + row * QS + g0) = x0 * scale;
        *reinterpret_cast<f32x4*>(dst + row * QS + g1) = x1 * scale;
      };
      if (PHASE == 2) put(rq[u], qs, 1.f);
      put(rk[u], ks, k_scale);
    }
    int odd = 0;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = tid + u * NT, row = e / (VD / 8), ch = (e % (VD / 8)) * 8;
      float x[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[2 * i] = bf16lo(rv[u][i]), x[2 * i + 1] = bf16hi(rv[u][i]);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (act) x[i] = silu(x[i]);
        odd |= !(fabsf(x[i]) < __builtin_inff());
      }
      *reinterpret_cast<f32x4*>(vs + row * VS + ch) = (f32x4){x[0], x[1], x[2], x[3]};
      *reinterpret_cast<f32x4*>(vs + row * VS + ch + 4) = (f32x4){x[4], x[5], x[6], x[7]};
    }
    return odd;
  };

  int turn_no = 0, one_by_one = r0;  // rows before one_by_one are walked a token at a time
  int r = r0;
  fetch(r, min(RT, r1 - r));
  while (r < r1) {
    const int nb = r < one_by_one ? 1 : min(RT, r1 - r);
    __syncthreads();  // the block before is done with LDS
    const int odd = stage();
    // A score of a later token is zero, and zero times an infinite value is not: a block that holds one goes token by
    // token (the rows of a one-token block past it are zeros).
    if (__syncthreads_or(odd) && nb > 1) {
      one_by_one = r + nb;
      fetch(r, 1);
      continue;
    }
    const int nx = r + nb;
    const bool two = nb > 16;
    f32x4 O[2][2];
    if (PHASE == 2) {
      const int job = (wave + turn_no) % NW;  // the three score tiles go round the waves
      if (job < 3 && (job == 0 || two)) {
        const int im = job > 0, jm = job > 1;
        f32x4 P = {0.f, 0.f, 0.f, 0.f}, P2 = P;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(qs + (16 * im + c) * QS + 16 * t + 4 * g);
          const f32x4 b = *reinterpret_cast<const f32x4*>(ks + (16 * jm + c) * QS + 16 * t + 4 * g);
          P = mfma4(a[0], b[0], P);
          P2 = mfma4(a[1], b[1], P2);
          P = mfma4(a[2], b[2], P);
          P2 = mfma4(a[3], b[3], P2);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = 16 * im + 4 * g + q, j = 16 * jm + c;
          ps[i * PS + j] = j <= i ? (P[q] + P2[q]) * pw[i - j] : 0.f;
        }
      }
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n) O[m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const f32x4 a0 = *reinterpret_cast<const f32x4*>(qs + c * QS + 16 * t + 4 * g);
        const f32x4 a1 = *reinterpret_cast<const f32x4*>(qs + (16 + c) * QS + 16 * t + 4 * g);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          O[0][0] = mfma4(a0[q], S[t][0][q], O[0][0]);
          O[0][1] = mfma4(a0[q], S[t][1][q], O[0][1]);
          O[1][0] = mfma4(a1[q], S[t][0][q], O[1][0]);
          O[1][1] = mfma4(a1[q], S[t][1][q], O[1][1]);
        }
      }
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float w = pw[16 * m + 4 * g + q + 1];
          O[m][0][q] *= w;
          O[m][1][q] *= w;
        }
      __syncthreads();  // the scores are there
    }
    f32x4 vb[2][2];  // [token tile][column tile], register r: token 16 tile + 4 g + r
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) vb[t][n][q] = vs[(16 * t + 4 * g + q) * VS + col0 + 16 * n];
    if (PHASE == 2) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if (m && !two) break;
#pragma unroll
        for (int t = 0; t <= m; ++t) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(ps + (16 * m + c) * PS + 16 * t + 4 * g);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            O[m][0] = mfma4(a[q], vb[t][0][q], O[m][0]);
            O[m][1] = mfma4(a[q], vb[t][1][q], O[m][1]);
          }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = 16 * m + 4 * g + q;
          if (i < nb) {
            float* op = out + ((long)(r + i) * heads + head) * VD + col0;
            op[0] = O[m][0][q];
            op[16] = O[m][1][q];
          }
        }
      }
    }
    if (nx < r1) fetch(nx, nx < one_by_one ? 1 : min(RT, r1 - nx));  // under the state's update: earlier costs registers
    const float pn = pw[nb];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = 16 * t + 4 * g + q;
        const float w = j < nb ? pw[nb - 1 - j] : 0.f;
        vb[t][0][q] *= w;
        vb[t][1][q] *= w;
      }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      S[i][0] *= pn;
      S[i][1] *= pn;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (t && !two) break;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float a = ks[(16 * t + 4 * g + q) * QS + 16 * i + c];
          S[i][0] = mfma4(a, vb[t][0][q], S[i][0]);
          S[i][1] = mfma4(a, vb[t][1][q], S[i][1]);
        }
      }
    }
    r = nx;
    ++turn_no;
  }
  if (PHASE == 1) {
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) st[(16 * t + 4 * g + q) * VD + col0 + 16 * n] = S[t][n][q];
  }
}

// Walks a sequence's runs in order: ws_state[run] (its end state from zero) becomes its start state, the sequence's slot
// gets the end state.  One thread per state element; the loads of four runs are in flight together.
__global__ __launch_bounds__(256) void retention_chain_kernel(float* __restrict__ ws_state, const float* __restrict__ decay,
                                                              float* __restrict__ state, long state_stride,
                                                              const int* __restrict__ seq_cu, const int* __restrict__ seq_state,
                                                              int n_seqs, const int* __restrict__ pieces,
                                                              const int* __restrict__ seq_pieces, int group,
                                                              const int* __restrict__ positions, int heads, int elems) {
  const int seq = blockIdx.z, head = blockIdx.y, e = blockIdx.x * 256 + threadIdx.x;
  const int slot = seq_state[seq];
  if (slot < 0 || seq_cu[seq + 1] <= seq_cu[seq]) return;
  const Run run = find_run(seq_pieces, n_seqs, group, 0, seq);
  if (e >= elems) return;
  float* st = state + (long)slot * state_stride + (long)head * elems + e;
  const double d = decay[head];
  float S = positions[seq_cu[seq]] == 0 ? 0.f : *st;
  const long step = (long)heads * elems;
  float* w = ws_state + ((long)run.first * heads + head) * elems + e;
  for (int k0 = 0; k0 < run.count; k0 += 4) {
    float end[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) end[k] = k0 + k < run.count ? w[(k0 + k) * step] : 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k0 + k >= run.count) break;
      int r0, r1;
      run_rows(pieces, seq_pieces, seq, k0 + k, group, &r0, &r1);
      double p = 1.0, b = d;
      for (int n = r1 - r0; n; n >>= 1, b *= b)
        if (n & 1) p *= b;
      w[(k0 + k) * step] = S;
      S = fmaf((float)p, S, end[k]);
    }
  }
  *st = S;
}

}  // namespace

// proj bf16 [rows, p_stride] with q, k (heads of 128 channels) and v (heads of vdim channels) at their columns; state: the
// slots of this layer; out fp32 [rows, heads, vdim]; pieces / seq_pieces as in vpsa_recurrent_scan, ws_state fp32
// [n_pieces, heads, 128, vdim].  vdim 128 or 256 (a wave per 32 columns); every row and column start on 16-byte
// boundaries; rot_dims a multiple of 8 (layout 0 or 1) or 0.  act: q, k and v pass through silu (no rotation then).
VPSA_EXPORT int vpsa_retention_scan(const void* proj, long p_stride, int q_col, int k_col, int v_col, int heads, int vdim,
                                    float* state, long state_stride, const int* seq_cu, const int* seq_state, int n_seqs,
                                    const int* positions, const float* decay, const float* cos_sin, int rot_dims, int layout,
                                    float k_scale, int act, float* out, const int* pieces, const int* seq_pieces, int n_pieces,
                                    float* ws_state, hipStream_t stream) {
  if (n_seqs <= 0 || n_pieces <= 0) return 0;
  if ((vdim != 128 && vdim != 256) || (rot_dims & 7) || rot_dims > RD || (act && rot_dims)) return 1;
  if (((uintptr_t)proj & 15) || (p_stride & 7) || ((q_col | k_col | v_col) & 7)) return 2;
  if (rot_dims && ((uintptr_t)cos_sin & 15)) return 2;
  const int group = (n_pieces * heads + 511) / 512;
  const dim3 grid(heads, n_pieces / group + n_seqs);
#define RETENTION(NW, PH)                                                                                              \
  retention_kernel<NW, PH><<<grid, NW * 64, 0, stream>>>((const uint16_t*)proj, p_stride, q_col, k_col, v_col, heads,  \
                                                         positions, decay, cos_sin, rot_dims, layout, k_scale, act,    \
                                                         seq_state, n_seqs, pieces, seq_pieces, group, ws_state, out)
  if (vdim == 256) RETENTION(8, 1);
  else RETENTION(4, 1);
  retention_chain_kernel<<<dim3(RD * vdim / 256, heads, n_seqs), 256, 0, stream>>>(
      ws_state, decay, state, state_stride, seq_cu, seq_state, n_seqs, pieces, seq_pieces, group, positions, heads, RD * vdim);
  if (vdim == 256) RETENTION(8, 2);
  else RETENTION(4, 2);
#undef RETENTION
  return 0;
}
