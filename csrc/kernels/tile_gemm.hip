// Prefill-sized bf16 GEMM for gfx950 (CDNA4), dense or grouped, with fused epilogues.
//
//   for every group g:  C[rows(g), :] = epilogue( A[arows(g), :] . W[g]^T )      W[g] is [N, K], K-contiguous
//
// rows(g) = offsets[g] .. offsets[g+1] read on the DEVICE (a mixture-of-experts layer is one launch
// whatever the routing, no host synchronisation, HIP-graph capturable); offsets == null is one group
// of max_rows rows (a dense projection).
//
// Structure: 256 x 256 output tile per workgroup, K in steps of 64, 512 threads = 8 waves as
// 2 (rows) x 4 (columns), each wave 128 x 64 of the tile in 32 accumulators of
// v_mfma_f32_16x16x32_bf16 (the chip holds a higher clock on this shape than on 32x32x16 for the
// same FLOPs).  The two wave rows run half a phase apart ("ping-pong"): the SIMD's two waves are
// one of each row, so while one multiplies 16 MFMAs the other reads its next fragments from LDS and
// issues the direct-to-LDS loads of later K tiles; every phase ends in a workgroup barrier, so the
// alternation is exact.  A K tile is four phases (one 64 x 32 quadrant of the wave's block each);
// its operand tiles are cut in four half tiles of 16 KiB (rows of the first / second quadrant row,
// columns of the first / second quadrant column) so that a half tile is free for re-use as early as
// one phase after the only phase that reads it; one half tile is requested per phase, three are in
// flight behind a COUNTED vmcnt at the end of each K tile (never 0 inside the loop), two LDS buffers
// of 64 KiB.
//
// The MFMA takes the weight rows as its A operand and the activation rows as B, so an accumulator
// holds C transposed: lane = one output row, registers = consecutive output columns.  The weight
// rows of a 32-column quadrant are ordered in LDS so that the two accumulators of a lane are 8
// consecutive columns: the epilogue writes 16 bytes per lane with no shuffle.
//
// LDS image of a half tile: 128 rows of 128 B, the eight 16-byte slots of a row XOR-swizzled with
// (row >> 1) & 7: conflict-free for the 16-row x 64-byte fragment reads (ds_read_b128).  Direct-to-
// LDS loads write LDS linearly (lane x 16 B), so the swizzle is applied to the per-lane SOURCE
// address; per-lane sources also make the row gather (arow_idx) free.
//
// Epilogues: bf16 store; SwiGLU (W = [gate rows | up rows], the first quadrant column of a wave is
// gate and the second the matching up columns: silu(gate) * up, [rows, N / 2]); bf16 store of
// accumulator + residual (the residual stream update of the o / down projections).
//
// Tail: tiles that would fill less than half of a last round of workgroups (or of the only one) have their reduction cut until they fill it,
// their accumulators go to a workspace in 32 bits, and a pass behind the product adds them in fixed order and makes the
// epilogue (tile_tail.h: which tiles, how many ranges; tail_finish_kernel, tail_norm_kernel, moe_combine_parts_kernel).
// 4096 x 14336 with the norm, 512 rows 261 us whole / 71 cut, 1000 rows 259 / 107, 5300 rows 562 / 482; the experts' last products, 8 of 4096 x 14336,
// 800 tokens 310 / 206; a step of four layers of 5300 rows 9087 -> 7694, of 4300 8535 -> 6846 (with library products before).
#include <type_traits>

#include "common.h"
#include "tile_tail.h"

#define TG_BK 64
#define TG_HT 16384          // half tile
#define TG_BUF (4 * TG_HT)   // X-h0, X-h1, W-h0, W-h1
#define TG_LDS (2 * TG_BUF)

#define TG_EPI_PLAIN 0
#define TG_EPI_SWIGLU 1
#define TG_EPI_RESIDUAL 2
#define TG_EPI_GLU_CLAMP 3  // paired like SwiGLU: min(g, limit) * sigmoid(alpha * min(g, limit)) * (clamp(u, +-limit) + bias)
#define TG_EPI_RELU_SQ 4    // relu(product)^2
#define TG_EPI_XIELU 5      // z > 0: act_alpha z^2 + z / 2, else act_bias (exp(z) - 1 - z) + z / 2
#define TG_EPI_GELU_GLU 6   // paired like SwiGLU: gelu(g) * u with gelu in its tanh form
#define TG_PAIRED(E) ((E) == TG_EPI_SWIGLU || (E) == TG_EPI_GLU_CLAMP || (E) == TG_EPI_GELU_GLU)

typedef __attribute__((address_space(3))) void* tg_lds_ptr_t;

__device__ __forceinline__ void tg_glds16(const char* gptr, char* lds_dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)gptr, (tg_lds_ptr_t)lds_dst, 16, 0, 0);
}

// DBG: timing experiments with WRONG results (bit 0: no loads inside the K loop, bit 1: no fragment
// reads inside the K loop, bit 2: every load inside the K loop re-requests K tile 0, i.e. hits in
// cache); 0 in every production launch.
// RAGGED: tiles of fewer than 193 rows go through with one, two or three of a quadrant's four 16-row tiles.  A group's rows are dealt
// out evenly in units of 64, so that its last tile is not mostly padding: eight experts of 350 to 410 rows, 28672 x 4096 764 -> 714 us
// and 4096 x 14336 360 -> 348; of 50 to 100 rows 436 -> 376 and 267 -> 243.  The instance without keeps its registers and its
// instruction cache for the one form (1500 dense rows 0.9 % faster).
// TAIL: with a workspace for the tail's partial sums (256 slots of 256 x 256).
template <int EPI, int DBG, bool RAGGED, bool TAIL>
__global__ __launch_bounds__(512, 2) void tile_gemm_kernel(
    const uint16_t* __restrict__ a, long lda, const int* __restrict__ arow_idx,
    const uint16_t* __restrict__ w, long w_group_stride, const int* __restrict__ offsets, int n_groups, int max_rows,
    uint16_t* __restrict__ c, long ldc, const uint16_t* __restrict__ resid, long ldr,
    int n_total, int k_total, int n_tiles, float act_limit, float act_alpha, float act_bias,
    const float* __restrict__ row_scale, float* __restrict__ ws) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- which tile is mine (wave-uniform scalar work).  Tile order: group by group; inside a group
  // bands of TG_BAND column tiles; inside a band row tile by row tile.  The order is cut in 8
  // contiguous runs, one per XCD (workgroups go to XCDs round robin), so the workgroups that share
  // an XCD's L2 at any time are (row tiles of one group) x (one band).
  const TileRows rows_of = {offsets, n_groups, max_rows, n_tiles, RAGGED};
  const int total = TAIL ? rows_of.tiles_by_wave() : rows_of.tiles();  // (with a tail the grid has 256 workgroups more that may have nothing to do)
  const TileTail tail = TAIL ? tile_tail(total, k_total / TG_BK) : TileTail{total, 1};
  const int bid = blockIdx.x, units_all = tail.cut + (total - tail.cut) * tail.splits;
  if (bid >= units_all) return;
  int t, split = 0;
  {
    const bool whole = !TAIL || bid < tail.cut;  // (whole tiles before a tail: a multiple of 256)
    const int n = whole ? tail.cut : units_all - tail.cut, u = whole ? bid : bid - tail.cut;
    const int xcd = u & 7, q = n >> 3, r = n & 7;
    t = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (u >> 3);
    if (!whole) {
      split = t / (total - tail.cut);
      t = tail.cut + t - split * (total - tail.cut);
    }
  }
  const TileAt at = rows_of.at(t);
  const int g = at.group, row0 = at.row0, row_end = at.row_end, n_idx = at.n_idx, units = at.units;  // units: 64 rows each that the tile holds
  const char* const a_base = reinterpret_cast<const char*>(a);
  const char* const w_base = reinterpret_cast<const char*>(w + (long)g * w_group_stride);
  const int inter = n_total >> 1;  // SwiGLU: gate rows 0..inter-1, up rows inter..2*inter-1

  const int wr = wave >> 2, wc = wave & 3;

  // A tile of 64 MI rows: the same steps with MI of the four 16-row tiles in every quadrant.
  auto body = [&](auto tag) {
  constexpr int MI = decltype(tag)::value;
  // ---- per-lane source offsets (bytes) of the direct-to-LDS loads.  One wave instruction fills 8
  // LDS rows: lane -> (row = lane / 8, slot = lane % 8); instruction j (0, 1) of a half tile: wave
  // `wave` fills rows 64 j + 8 wave + lane / 8.  Slot s of LDS row r receives the 16-byte chunk
  // s ^ ((r >> 1) & 7) of the source row.
  //   X half tile h, LDS row r:  tile row 32 MI (r / 64) + 16 MI h + r % 64
  //   W half tile h, LDS row r:  wave column block r / 32, MFMA tile (r % 32) / 16, MFMA row i = r % 16
  //                              -> column 64 (r / 32) + 32 h + 8 (i / 4) + 4 tile + i % 4
  uint32_t src_off[4][2];
  {
    const int lrow = lane >> 3, lslot = lane & 7;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = 64 * j + 8 * wave + lrow;
      const int chunk = lslot ^ ((r >> 1) & 7);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int in_half = (r & 63) < 16 * MI ? r & 63 : 16 * MI - 1;  // (places past the tile's rows repeat one: never read)
        int arow = row0 + 32 * MI * (r >> 6) + 16 * MI * h + in_half;
        if (arow >= row_end) arow = row_end - 1;  // rows past the group's end repeat its last row (never stored)
        const long src_row = arow_idx ? (long)arow_idx[arow] : (long)arow;
        src_off[h][j] = (uint32_t)((src_row * lda + chunk * 8) * 2);
        const int cb = r >> 5, ti = (r >> 4) & 1, i = r & 15;
        const int nloc = 8 * (i >> 2) + 4 * ti + (i & 3);
        int wrow;
        if (TG_PAIRED(EPI)) {
          int col = n_idx * 128 + cb * 32 + nloc;
          if (col >= inter) col = inter - 1;
          wrow = h == 0 ? col : inter + col;
        } else {
          wrow = n_idx * TG_BN + cb * 64 + 32 * h + nloc;
          if (wrow >= n_total) wrow = n_total - 1;
        }
        src_off[2 + h][j] = (uint32_t)(((long)wrow * k_total + chunk * 8) * 2);
      }
    }
  }
  int k_first = 0, k_tiles = k_total / TG_BK;
  const bool part = TAIL && t >= tail.cut;
  if (part) {
    const int per = k_tiles / tail.splits, more = k_tiles - per * tail.splits;
    k_first = split * per + (split < more ? split : more);
    k_tiles = per + (split < more);
  }
  char* const fill_base = lds + wave * 1024;
  bool in_loop = false;
  auto stage = [&](int which, int buf, int kt) {
    if ((DBG & 1) && in_loop) return;
    int ktc = kt < k_tiles ? kt : k_tiles - 1;  // past the end: re-request the last tile into a free slot
    if ((DBG & 4) && in_loop) ktc = 0;
    const char* base = (which < 2 ? a_base : w_base) + (long)(k_first + ktc) * (TG_BK * 2);
    tg_glds16(base + src_off[which][0], fill_base + buf * TG_BUF + which * TG_HT);
    tg_glds16(base + src_off[which][1], fill_base + buf * TG_BUF + which * TG_HT + 8192);
  };

  // ---- fragment read offsets.  MFMA operand lane -> (row = lane % 16, k quarter = lane / 16); all
  // fragment rows start at a multiple of 16, so the row's swizzle is (lane % 16) / 2
  const int fr = lane & 15, fq = lane >> 4;
  const int sl0 = ((fq) ^ (fr >> 1)) << 4, sl1 = ((4 + fq) ^ (fr >> 1)) << 4;
  const int x_rd = (wr * 64 + fr) * 128;
  const int w_rd = 2 * TG_HT + (wc * 32 + fr) * 128;

  f32x4 acc[2][2][MI][2];  // [quadrant row][quadrant column][row tile][column tile]
#pragma unroll
  for (int i0 = 0; i0 < 2; ++i0)
#pragma unroll
    for (int i1 = 0; i1 < 2; ++i1)
#pragma unroll
      for (int i2 = 0; i2 < MI; ++i2)
#pragma unroll
        for (int i3 = 0; i3 < 2; ++i3) acc[i0][i1][i2][i3] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 xa[MI][2];      // activation fragments of the current quadrant row: [row tile][k step]
  bf16x8 wb[2][2][2];   // weight fragments of both quadrant columns: [quadrant column][column tile][k step]

  auto read_w = [&](int buf, int nh) {
    if ((DBG & 2) && in_loop) return;
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
      wb[nh][ni][0] = *reinterpret_cast<const bf16x8*>(lds + buf * TG_BUF + nh * TG_HT + ni * 2048 + w_rd + sl0);
      wb[nh][ni][1] = *reinterpret_cast<const bf16x8*>(lds + buf * TG_BUF + nh * TG_HT + ni * 2048 + w_rd + sl1);
    }
  };
  auto read_x = [&](int buf, int mh) {
    if ((DBG & 2) && in_loop) return;
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      xa[mi][0] = *reinterpret_cast<const bf16x8*>(lds + buf * TG_BUF + mh * TG_HT + mi * 2048 + x_rd + sl0);
      xa[mi][1] = *reinterpret_cast<const bf16x8*>(lds + buf * TG_BUF + mh * TG_HT + mi * 2048 + x_rd + sl1);
    }
  };
  auto mma = [&](int mh, int nh) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
          acc[mh][nh][mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[nh][ni][s], xa[mi][s], acc[mh][nh][mi][ni], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };

#define TG_SB() __builtin_amdgcn_sched_barrier(0)
#define TG_BAR()                    \
  do {                              \
    TG_SB();                        \
    __builtin_amdgcn_s_barrier();   \
    TG_SB();                        \
  } while (0)
#define TG_LGKM0()                                        \
  do {                                                    \
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    \
    TG_SB();                                              \
  } while (0)

  // ---- prologue: K tile 0 whole, then the first three half tiles of K tile 1 (the order the loop
  // keeps: W-h0, X-h0, W-h1; X-h1 follows in the first phase)
  stage(0, 0, 0);
  stage(1, 0, 0);
  stage(2, 0, 0);
  stage(3, 0, 0);
  stage(2, 1, 1);
  stage(0, 1, 1);
  stage(3, 1, 1);
  stage(1, 1, 1);
  asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  TG_BAR();
  if (wr == 1) TG_BAR();  // the second wave row runs one barrier behind the first

  // One K tile (LDS buffer B, tile index KT).  Phase = {fragment reads, one half-tile request,
  // barrier, 16 MFMAs, barrier}.  Requests: X-h1 of tile KT+1 (its slot was last read two phases
  // ago), then W-h0, X-h0, W-h1 of tile KT+2 into THIS buffer: W-h0 is read in phase 1 only and
  // those reads are retired (a counted wait: the four W reads are issued first) before phase 1's first
  // barrier, so it may be overwritten from phase 2 on; X-h0 (read in phase 1) from phase 3; W-h1
  // (phase 2) from phase 4; X-h1 (phase 3) from the next tile's phase 1.  The counted wait of phase
  // 4 leaves the three youngest half tiles in flight: everything of tile KT+1 has landed before the
  // barrier that precedes its first read.
#define TG_TILE(B, KT)                                          \
  do {                                                          \
    read_w(B, 0);                                               \
    TG_SB();                                                    \
    read_x(B, 0);                                               \
    TG_SB();                                                    \
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(2 * MI) : "memory");          \
    TG_BAR();                                                   \
    TG_LGKM0();                                                 \
    mma(0, 0);                                                  \
    TG_BAR();                                                   \
    read_w(B, 1);                                               \
    TG_SB();                                                    \
    stage(2, B, (KT) + 2);                                      \
    TG_BAR();                                                   \
    TG_LGKM0();                                                 \
    mma(0, 1);                                                  \
    TG_BAR();                                                   \
    read_x(B, 1);                                               \
    TG_SB();                                                    \
    stage(0, B, (KT) + 2);                                      \
    TG_SB();                                                    \
    TG_LGKM0();                                                 \
    TG_BAR();                                                   \
    mma(1, 1);                                                  \
    TG_BAR();                                                   \
    stage(3, B, (KT) + 2);                                      \
    stage(1, B, (KT) + 2);                                      \
    TG_SB();                                                    \
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");            \
    TG_BAR();                                                   \
    mma(1, 0);                                                  \
    TG_BAR();                                                   \
  } while (0)

  if (DBG) {
    read_w(0, 0); read_w(0, 1); read_x(0, 0);
    in_loop = true;
  }
  int kt = 0;
  for (; kt + 1 < k_tiles; kt += 2) {
    TG_TILE(0, kt);
    TG_TILE(1, kt + 1);
  }
  if (kt < k_tiles) TG_TILE(0, kt);
#undef TG_TILE
  if (wr == 0) TG_BAR();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be writing LDS when the wave ends

  // ---- epilogue.  Accumulator [mh][nh][mi][ni]: lane -> output row 32 MI wr + 16 MI mh + 16 mi + lane % 16,
  // register e -> column 64 wc + 32 nh + 8 (lane / 16) + 4 ni + e.
  if (part) {  // 16 lanes write a row's 128 bytes of two column tiles
    float* const slot = ws + ((long)(t - tail.cut) * tail.splits + split) * (TG_BM * TG_BN);
#pragma unroll
    for (int mh = 0; mh < 2; ++mh)
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const int r = 32 * MI * wr + 16 * MI * mh + 16 * mi + fr;
        if (row0 + r >= row_end) continue;
#pragma unroll
        for (int nh = 0; nh < 2; ++nh)
#pragma unroll
          for (int ni = 0; ni < 2; ++ni)
            *reinterpret_cast<f32x4*>(slot + r * TG_BN + (TG_PAIRED(EPI) ? 128 * nh + 32 * wc : 64 * wc + 32 * nh) + 8 * fq + 4 * ni) =
                acc[mh][nh][mi][ni];
      }
    return;
  }
  float rs[2][MI];  // the rows' factors, all loads in flight
  if (EPI == TG_EPI_GLU_CLAMP) {
#pragma unroll
    for (int mh = 0; mh < 2; ++mh)
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const int row = row0 + 32 * MI * wr + 16 * MI * mh + 16 * mi + fr;
        rs[mh][mi] = row_scale ? row_scale[row < row_end ? row : row_end - 1] : 1.f;
      }
  }
#pragma unroll
  for (int mh = 0; mh < 2; ++mh) {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      const int row = row0 + 32 * MI * wr + 16 * MI * mh + 16 * mi + fr;
      if (TG_PAIRED(EPI)) {
        const int col = n_idx * 128 + wc * 32 + 8 * fq;
        float v[8];
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float gt = acc[mh][0][mi][ni][e], up = acc[mh][1][mi][ni][e];
            if (EPI == TG_EPI_GLU_CLAMP) {
              gt = fminf(gt * rs[mh][mi], act_limit);
              up = fminf(fmaxf(up * rs[mh][mi], -act_limit), act_limit) + act_bias;
              v[4 * ni + e] = gt / (1.f + __expf(-act_alpha * gt)) * up;
            } else if (EPI == TG_EPI_GELU_GLU) {
              // 0.5 g (1 + tanh(y)) = g / (1 + exp(-2 y)),  y = sqrt(2 / pi) (g + 0.044715 g^3)
              const float y2 = 1.5957691216057308f * (gt + 0.044715f * gt * gt * gt);
              v[4 * ni + e] = gt / (1.f + __expf(-y2)) * up;
            } else {
              v[4 * ni + e] = gt / (1.f + __expf(-gt)) * up;
            }
          }
        if (row < row_end && col < inter) {
          u32x4 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
          *reinterpret_cast<u32x4*>(c + (long)row * ldc + col) = o;
        }
      } else {
#pragma unroll
        for (int nh = 0; nh < 2; ++nh) {
          const int col = n_idx * TG_BN + wc * 64 + 32 * nh + 8 * fq;
          if (row < row_end && col < n_total) {
            float v[8];
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
#pragma unroll
              for (int e = 0; e < 4; ++e) v[4 * ni + e] = acc[mh][nh][mi][ni][e];
            if (EPI == TG_EPI_RELU_SQ) {
#pragma unroll
              for (int p = 0; p < 8; ++p) {
                const float r = fmaxf(v[p], 0.f);
                v[p] = r * r;
              }
            }
            if (EPI == TG_EPI_XIELU) {
#pragma unroll
              for (int p = 0; p < 8; ++p) {
                const float z = v[p];
                v[p] = z > 0.f ? fmaf(act_alpha * z, z, 0.5f * z) : fmaf(act_bias, expm1f(z) - z, 0.5f * z);
              }
            }
            if (EPI == TG_EPI_RESIDUAL) {
              const u32x4 rr = *reinterpret_cast<const u32x4*>(resid + (long)row * ldr + col);
#pragma unroll
              for (int p = 0; p < 4; ++p) {
                v[2 * p] += bf16lo(rr[p]);
                v[2 * p + 1] += bf16hi(rr[p]);
              }
            }
            u32x4 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
            *reinterpret_cast<u32x4*>(c + (long)row * ldc + col) = o;
          }
        }
      }
    }
  }
  };
  if constexpr (!RAGGED) return body(std::integral_constant<int, 4>());
  switch (units) {
    case 1: return body(std::integral_constant<int, 1>());
    case 2: return body(std::integral_constant<int, 2>());
    case 3: return body(std::integral_constant<int, 3>());
    default: return body(std::integral_constant<int, 4>());
  }
}

static int g_tg_debug = 0;
VPSA_EXPORT int vpsa_tile_gemm_debug(int v) {
  int old = g_tg_debug;
  g_tg_debug = v;
  return old;
}

// a [*, K] bf16 (row stride lda elements, 16-byte aligned rows); arow_idx [rows] int32 or null (null:
// output row r reads A row r); w [G, N, K] contiguous; offsets [G + 1] int32 on the device with
// offsets[G] <= max_rows, or null (one group of max_rows rows); c [max_rows, N] (SwiGLU: N / 2
// columns), row stride ldc; epi: 0 store, 1 SwiGLU, 2 store of product + resid (row stride ldr; may
// alias c), 6 gated gelu unit (tanh form, paired like SwiGLU), 3 clamped gated unit (paired like SwiGLU, constants act_*), 4 squared ReLU, 5 xIELU (act_alpha, act_bias: its two curvatures).  Every byte offset into a and into one group of w must fit 32 bits.
// row_scale fp32 [max_rows] or null (epi 3 only): gate and up of output row r are multiplied by row_scale[r] before the
// clamps, i.e. the row's input carries that factor.
// ws (epi 0, 1, 2; or null): workspace of 256 x 256 x 256 fp32 for the tail; its tiles' outputs are then left to one of the passes below.
// Returns 0, or a negative number when the shape is outside what the kernel tiles.
VPSA_EXPORT int vpsa_tile_gemm(const void* a, long lda, const void* arow_idx, const void* w, const void* offsets,
                               int n_groups, void* c, long ldc, int max_rows, int n, int k, int epi, const void* resid,
                               long ldr, long a_rows, float act_limit, float act_alpha, float act_bias,
                               const void* row_scale, void* ws, hipStream_t stream) {
  if (k % TG_BK != 0 || k <= 0 || n <= 0 || max_rows <= 0 || n_groups <= 0 || lda % 8 != 0 || ldc % 8 != 0) return -1;
  if (!offsets && n_groups != 1) return -1;
  if (TG_PAIRED(epi) && (n % 2 != 0 || (n / 2) % 32 != 0)) return -1;
  if (!TG_PAIRED(epi) && n % 8 != 0) return -1;
  if (epi == TG_EPI_RESIDUAL && (!resid || ldr % 8 != 0)) return -1;
  if (epi < 0 || epi > 6 || (row_scale && epi != TG_EPI_GLU_CLAMP)) return -1;
  if ((double)a_rows * (double)lda * 2.0 >= 4294967296.0 || (double)n * (double)k * 2.0 >= 4294967296.0) return -1;
  const int n_tiles = TG_PAIRED(epi) ? (n / 2 + 127) / 128 : (n + TG_BN - 1) / TG_BN;
  const int m_tiles_max = offsets ? max_rows / TG_BM + n_groups : (max_rows + TG_BM - 1) / TG_BM;
  if (ws && (((uintptr_t)ws & 15) || (epi != TG_EPI_PLAIN && epi != TG_EPI_SWIGLU && epi != TG_EPI_RESIDUAL))) return -1;
  const long blocks = (long)n_tiles * m_tiles_max + (ws ? TG_CUS : 0);  // (more than one round of tail workgroups there is never)
  if (blocks > 0x7fffffffL) return -1;
  const long wstride = (long)n * k;
  // (an even deal gives every tile four units exactly when the rows' units are four times the tiles)
  const bool ragged = offsets || (max_rows + 63) / 64 != 4 * m_tiles_max;
#define TG_RUN(KERNEL)                                                                                                 \
  do {                                                                                                                 \
    static bool attr_set = false;                                                                                      \
    const auto kernel = KERNEL;                                                                                        \
    if (!attr_set) {                                                                                                   \
      if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS) != hipSuccess)  \
        return -2;                                                                                                     \
      attr_set = true;                                                                                                 \
    }                                                                                                                  \
    kernel<<<dim3((unsigned)blocks), dim3(512), TG_LDS, stream>>>(                                                     \
        (const uint16_t*)a, lda, (const int*)arow_idx, (const uint16_t*)w, wstride, (const int*)offsets, n_groups,     \
        max_rows, (uint16_t*)c, ldc, (const uint16_t*)resid, ldr, n, k, n_tiles, act_limit, act_alpha, act_bias,       \
        (const float*)row_scale, (float*)ws);                                                                          \
  } while (0)
#define TG_LAUNCH(E, D)                                            \
  do {                                                             \
    if (D == 0 && ragged) TG_RUN((tile_gemm_kernel<E, D, D == 0, false>)); \
    else TG_RUN((tile_gemm_kernel<E, D, false, false>));           \
  } while (0)
#define TG_LAUNCH_TAIL(E)                                          \
  do {                                                             \
    if (ragged) TG_RUN((tile_gemm_kernel<E, 0, true, true>));      \
    else TG_RUN((tile_gemm_kernel<E, 0, false, true>));            \
  } while (0)
  if (ws && epi == TG_EPI_SWIGLU) TG_LAUNCH_TAIL(TG_EPI_SWIGLU);
  else if (ws && epi == TG_EPI_RESIDUAL) TG_LAUNCH_TAIL(TG_EPI_RESIDUAL);
  else if (ws) TG_LAUNCH_TAIL(TG_EPI_PLAIN);
  else if (epi == TG_EPI_SWIGLU) TG_LAUNCH(TG_EPI_SWIGLU, 0);
  else if (epi == TG_EPI_RESIDUAL) TG_LAUNCH(TG_EPI_RESIDUAL, 0);
  else if (epi == TG_EPI_GLU_CLAMP) TG_LAUNCH(TG_EPI_GLU_CLAMP, 0);
  else if (epi == TG_EPI_RELU_SQ) TG_LAUNCH(TG_EPI_RELU_SQ, 0);
  else if (epi == TG_EPI_XIELU) TG_LAUNCH(TG_EPI_XIELU, 0);
  else if (epi == TG_EPI_GELU_GLU) TG_LAUNCH(TG_EPI_GELU_GLU, 0);
  else if (g_tg_debug == 1) TG_LAUNCH(TG_EPI_PLAIN, 1);
  else if (g_tg_debug == 2) TG_LAUNCH(TG_EPI_PLAIN, 2);
  else if (g_tg_debug == 3) TG_LAUNCH(TG_EPI_PLAIN, 3);
  else if (g_tg_debug == 4) TG_LAUNCH(TG_EPI_PLAIN, 4);
  else TG_LAUNCH(TG_EPI_PLAIN, 0);
#undef TG_LAUNCH_TAIL
#undef TG_LAUNCH
#undef TG_RUN
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

namespace {

// Four outputs from a tail tile's partial sums: slot-local row and column.
__device__ __forceinline__ f32x4 tail_sum(const float* __restrict__ p, int splits) {
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < splits; i0 += 4) {
    f32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const f32x4*>(p + (long)min(i0 + i, splits - 1) * (TG_BM * TG_BN));
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i0 + i < splits) s += v[i];
  }
  return s;
}

// A dense product's tail: sums, epilogue, 16-bit outputs.  Grid (tail tiles, 32): eight rows a workgroup, 64 threads a row of 256 columns (32 of
// 128 pairs).  Bound by the launch and the sums' way from the memory-side cache.
template <int EPI>
__global__ __launch_bounds__(256) void tail_finish_kernel(const float* __restrict__ ws, const TileRows rows_of, int k_total, int n_total,
                                                          uint16_t* __restrict__ c, long ldc, const uint16_t* __restrict__ resid, long ldr) {
  const int total = rows_of.tiles();
  const TileTail tail = tile_tail(total, k_total / TG_BK);
  const int t = tail.cut + (int)blockIdx.x;
  if (t >= total) return;
  const TileAt at = rows_of.at(t);
  const float* const slot = ws + (long)blockIdx.x * tail.splits * (TG_BM * TG_BN);
  constexpr int LANES = EPI == TG_EPI_SWIGLU ? 32 : 64, STEP = 256 / LANES;
  const int lc = (threadIdx.x % LANES) * 4, width = EPI == TG_EPI_SWIGLU ? 128 : TG_BN, limit = EPI == TG_EPI_SWIGLU ? n_total / 2 : n_total;
  const int col = at.n_idx * width + lc, end = min(at.row_end - at.row0, 64 * at.units);
  if (col >= limit) return;
#pragma unroll
  for (int r = blockIdx.y * 8 + threadIdx.x / LANES; r < (int)blockIdx.y * 8 + 8; r += STEP) {
    if (r >= end) break;
    f32x4 v = tail_sum(slot + r * TG_BN + lc, tail.splits);
    if (EPI == TG_EPI_SWIGLU) {
      const f32x4 up = tail_sum(slot + r * TG_BN + 128 + lc, tail.splits);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] / (1.f + __expf(-v[e])) * up[e];
    }
    if (EPI == TG_EPI_RESIDUAL) {
      const u32x2 o = *reinterpret_cast<const u32x2*>(resid + (long)(at.row0 + r) * ldr + col);
      v += (f32x4){bf16lo(o[0]), bf16hi(o[0]), bf16lo(o[1]), bf16hi(o[1])};
    }
    *reinterpret_cast<u32x2*>(c + (long)(at.row0 + r) * ldc + col) = (u32x2){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
}

// The rest of a residual update and the norm behind it: residual (whole tiles: updated by the product's epilogue) += the tail's sums, y = rms
// norm of the rows * weight.  A workgroup a row, CH runs of four channels a thread.
template <int CH>
__global__ __launch_bounds__(1024) void tail_norm_kernel(const float* __restrict__ ws, const TileRows rows_of, int k_total, int N,
                                                         uint16_t* __restrict__ residual, const uint16_t* __restrict__ weight,
                                                         uint16_t* __restrict__ y, float eps) {
  __shared__ float red[16];
  const int m = blockIdx.x, tid = threadIdx.x, total = rows_of.tiles();
  const TileTail tail = tile_tail(total, k_total / TG_BK);
  int m_idx, row0;
  rows_of.row_tile(0, rows_of.max_rows, m, m_idx, row0);
  f32x4 v[CH];
  u32x2 ww[CH];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int col = (c * (int)blockDim.x + tid) * 4;
    v[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
    ww[c] = (u32x2){0, 0};
    if (col >= N) continue;
    uint16_t* const rr = residual + (long)m * N + col;
    u32x2 o = *reinterpret_cast<const u32x2*>(rr);
    ww[c] = *reinterpret_cast<const u32x2*>(weight + col);
    v[c] = (f32x4){bf16lo(o[0]), bf16hi(o[0]), bf16lo(o[1]), bf16hi(o[1])};
    const int t = rows_of.tile_index(rows_of.m_tiles(0, rows_of.max_rows), m_idx, col / TG_BN);
    if (t >= tail.cut) {
      v[c] += tail_sum(ws + (long)(t - tail.cut) * tail.splits * (TG_BM * TG_BN) + (m - row0) * TG_BN + col % TG_BN, tail.splits);
      o = (u32x2){pack_bf16x2(v[c][0], v[c][1]), pack_bf16x2(v[c][2], v[c][3])};
      *reinterpret_cast<u32x2*>(rr) = o;
      v[c] = (f32x4){bf16lo(o[0]), bf16hi(o[0]), bf16lo(o[1]), bf16hi(o[1])};
    }
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
    *reinterpret_cast<u32x2*>(y + (long)m * N + col) =
        (u32x2){pack_bf16x2(v[c][0] * inv * bf16lo(ww[c][0]), v[c][1] * inv * bf16hi(ww[c][0])),
                pack_bf16x2(v[c][2] * inv * bf16lo(ww[c][1]), v[c][3] * inv * bf16hi(ww[c][1]))};
  }
}

// out[t] = sum over a token's pairs of weight * expert output, read from y (whole tiles) or summed from the tail's partial sums.
__global__ __launch_bounds__(256) void moe_combine_parts_kernel(const float* __restrict__ ws, const TileRows rows_of, int k_total,
                                                                const uint16_t* __restrict__ y, const float* __restrict__ weights,
                                                                const int* __restrict__ pos, uint16_t* __restrict__ out, int hidden, int topk) {
  const int tok = blockIdx.x, total = rows_of.tiles_by_wave();
  const TileTail tail = tile_tail(total, k_total / TG_BK);
  if (tail.splits == 1) {  // (a routing without a tail: wider reads, no search)
    for (int i = threadIdx.x * 8; i < hidden; i += 256 * 8) {
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int k = 0; k < topk; ++k) {
        const float w = weights[(long)tok * topk + k];
        if (w == 0.f) continue;  // a pair of an expert held by another rank: its row was never written
        const u32x4 a = *reinterpret_cast<const u32x4*>(y + (long)pos[(long)tok * topk + k] * hidden + i);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[2 * j] += w * bf16lo(a[j]);
          acc[2 * j + 1] += w * bf16hi(a[j]);
        }
      }
      *reinterpret_cast<u32x4*>(out + (long)tok * hidden + i) =
          (u32x4){pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]), pack_bf16x2(acc[4], acc[5]), pack_bf16x2(acc[6], acc[7])};
    }
    return;
  }
  // what a pair's row needs, found once by a lane of its own
  __shared__ struct {
    int first, m, m_idx, row, in_slot;
    float w;
  } pair[256];
  if ((int)threadIdx.x < topk) {
    const long p = (long)tok * topk + threadIdx.x;
    auto& mine = pair[threadIdx.x];
    mine.w = weights[p];
    if (mine.w != 0.f) {  // (0: a pair of an expert held by another rank, its row was never written)
      int lo, hi, row0;
      mine.row = pos[p];
      rows_of.group_of(mine.row, mine.first, lo, hi);
      rows_of.row_tile(lo, hi, mine.row, mine.m_idx, row0);
      mine.m = TileRows::m_tiles(lo, hi);
      mine.in_slot = (mine.row - row0) * TG_BN;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x * 4; i < hidden; i += 256 * 4) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < topk; ++k) {
      const auto& p = pair[k];
      if (p.w == 0.f) continue;
      const int t = p.first + rows_of.tile_index(p.m, p.m_idx, i / TG_BN);
      f32x4 v;
      if (t >= tail.cut) {
        v = tail_sum(ws + (long)(t - tail.cut) * tail.splits * (TG_BM * TG_BN) + p.in_slot + i % TG_BN, tail.splits);
      } else {
        const u32x2 o = *reinterpret_cast<const u32x2*>(y + (long)p.row * hidden + i);
        v = (f32x4){bf16lo(o[0]), bf16hi(o[0]), bf16lo(o[1]), bf16hi(o[1])};
      }
      acc += p.w * v;
    }
    *reinterpret_cast<u32x2*>(out + (long)tok * hidden + i) = (u32x2){pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3])};
  }
}

TileRows tile_rows_of(const void* offsets, int n_groups, int max_rows, int n, bool paired) {
  const int n_tiles = paired ? (n / 2 + 127) / 128 : (n + TG_BN - 1) / TG_BN;
  return {(const int*)offsets, n_groups, max_rows, n_tiles, offsets || (max_rows + 63) / 64 != 4 * ((max_rows + TG_BM - 1) / TG_BM)};
}

}  // namespace

// Ranges that the tail's tiles of a product are cut in, 1 where there is no tail: `tiles` tiles, reductions of k.
VPSA_EXPORT int vpsa_tile_tail(int tiles, int k) { return tile_tail(tiles, k / TG_BK).splits; }

// The passes behind vpsa_tile_gemm with a workspace: the tail's outputs of a dense product (epi 0, 1, 2 and its arguments as there) ...
VPSA_EXPORT int vpsa_tile_tail_finish(const void* ws, void* c, long ldc, int rows, int n, int k, int epi, const void* resid, long ldr,
                                      hipStream_t stream) {
  const TileRows rows_of = tile_rows_of(nullptr, 1, rows, n, epi == TG_EPI_SWIGLU);
  const dim3 grid(TG_CUS / 2, TG_BM / 8);  // (a tail has up to half a round of tiles)
#define FINISH(E)                                                                                                                  \
  tail_finish_kernel<E><<<grid, 256, 0, stream>>>((const float*)ws, rows_of, k, n, (uint16_t*)c, ldc, (const uint16_t*)resid, ldr)
  if (epi == TG_EPI_SWIGLU) FINISH(TG_EPI_SWIGLU);
  else if (epi == TG_EPI_RESIDUAL) FINISH(TG_EPI_RESIDUAL);
  else FINISH(TG_EPI_PLAIN);
#undef FINISH
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// ... of a dense product with epi 2 into residual [rows, n], with the norm of the rows; n a multiple of 4 up to 8192 ...
VPSA_EXPORT int vpsa_tile_tail_norm(const void* ws, void* residual, const void* weight, void* y, int rows, int n, int k, float eps,
                                    hipStream_t stream) {
  if (n % 4 != 0 || n > 8192 || (((uintptr_t)residual | (uintptr_t)weight | (uintptr_t)y) & 7)) return -1;
  const TileRows rows_of = tile_rows_of(nullptr, 1, rows, n, false);
  const int threads = n >= 4096 ? 1024 : (n / 4 + 63) / 64 * 64;
  if (n <= 4096) tail_norm_kernel<1><<<rows, threads, 0, stream>>>((const float*)ws, rows_of, k, n, (uint16_t*)residual, (const uint16_t*)weight, (uint16_t*)y, eps);
  else tail_norm_kernel<2><<<rows, threads, 0, stream>>>((const float*)ws, rows_of, k, n, (uint16_t*)residual, (const uint16_t*)weight, (uint16_t*)y, eps);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// ... or of a grouped product with epi 0 into y, with the weighted sum of a token's pairs (pos: the row of a pair).
VPSA_EXPORT int vpsa_moe_combine_parts(const void* ws, const void* offsets, int n_groups, int max_rows, int k, const void* y, const void* weights,
                                       const void* pos, void* out, int tokens, int hidden, int topk, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (hidden % 8 != 0 || topk > 256) return -1;
  moe_combine_parts_kernel<<<tokens, 256, 0, stream>>>((const float*)ws, tile_rows_of(offsets, n_groups, max_rows, hidden, false), k,
                                                      (const uint16_t*)y, (const float*)weights, (const int*)pos, (uint16_t*)out, hidden, topk);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
