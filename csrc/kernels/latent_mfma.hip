// Latent attention on the matrix cores (gfx950, bf16): prefill tiles and decode rows.
//
// In latent space every head of a token attends over the SAME entries (latent | rotated key part,
// RANK + ROT values per token), so a work item is a tile of up to 64 query slots = (token, head) pairs
// of one sequence, token-major: consecutive tokens x all heads for prefill chunks (heads <= 64), one
// token's heads (in runs of 64) for decode rows.  The tile walks its sequence's pages; a page is
// exactly one key tile (64 entries, contiguous in the pool).
//
// Workgroup = 4 waves; wave w owns slots 16 w .. 16 w + 15 end to end (its queries stay in registers
// as MFMA B operands, its output accumulators [16 slots x RANK] too), so the waves share nothing but
// the staged page:
//   K image  [64 keys][RANK + ROT]  (+16 B row padding): A operand of  S^T = K Q^T
//   V^T image [RANK][64 keys]       (+16 B row padding): A operand of  O^T = V^T P^T
// The V^T image is made while staging: a thread loads a 4-key x 8-channel block (coalesced 16-byte
// loads), stores its rows into the K image and the 4 x 8 transpose into the V^T image.  The keys of
// the V^T image are permuted so that the 8 keys a lane owns in the S^T accumulators (v_mfma 16x16x32:
// lane = query l % 16, keys 4 (l / 16) + e of four 16-key tiles) are 16 contiguous bytes: P goes from
// the S accumulators into the second product without leaving the lane.  (The 16-byte chunks of a V^T row
// are XOR-swizzled with (row / 8) % 8: the transposing stores of neighbouring lanes lie 8 rows apart.)
// The next page's global loads are issued before the current page is multiplied.
//
// With a sliding window of `window` positions (a query at position p sees keys p - window + 1 .. p) the walk starts
// at the page of the first key that the tile's earliest query sees; only pages that hold a key some slot does not
// see are masked key by key.
//
// Without q_lat (ROT_ONLY) the scores come from the entries' last ROT channels alone and the first RANK are values
// only: the expanded per-head entries of a prefill, value | key.
//
// Softmax state (running max, sum) is fp32 per slot, scores in powers of two; an optional per-head sink logit starts the state
// (max = sink, sum = 1).  With key-range splits every split writes unnormalised partial outputs and
// (max, sum) to a workspace and a merge kernel adds the sink and normalises.
#include <float.h>

#include "common.h"

namespace {

constexpr int MERGE_MAX = 64;  // key-range splits the merge kernel takes

struct LatTile {
  int seq, row0, n_tok, pos0, head0, hcount;
};

__device__ __forceinline__ u32x4 ld16(const uint16_t* p) { return *reinterpret_cast<const u32x4*>(p); }

constexpr float LOG2E = 1.4426950408889634f, LN2 = 0.6931471805599453f;

// (entries of up to 256 values leave registers for three waves per SIMD; at 320 they would spill and lose)
template <int RANK, int ROT, bool ROT_ONLY>
__global__ __launch_bounds__(256, RANK + ROT <= 256 && RANK <= 128 ? 3 : 1) void latent_mfma_kernel(
    const uint16_t* __restrict__ q_lat, long ql_row, long ql_head, const uint16_t* __restrict__ q_rot, long qr_row,
    long qr_head, const uint16_t* __restrict__ cache, long page_stride, const int* __restrict__ block_tables,
    int bt_stride, const int* __restrict__ tiles, const int* __restrict__ positions, int heads,
    const float* __restrict__ sink, uint16_t* __restrict__ out, long o_row, long o_head, float scale, int window,
    int splits, float* __restrict__ ws_o, float* __restrict__ ws_ml) {
  constexpr int ENTRY = RANK + ROT;
  constexpr int K0 = ROT_ONLY ? RANK : 0;     // first channel that scores read
  constexpr int KC = ENTRY - K0;
  constexpr int KS = KC / 32;
  constexpr int DT = RANK / 16;
  constexpr int PK = KC * 2 + 16;
  constexpr int PV = 64 * 2 + 16;
  constexpr int NBLK = 2 * RANK;              // 4-key x 8-channel blocks of the latent part: 16 key quads x RANK / 8
  constexpr int RB = (NBLK + 255) / 256;      // of which a thread takes this many
  constexpr int CB = ROT / 32;    // 16-byte chunks of the rotated part per thread
  extern __shared__ __attribute__((aligned(16))) char lds[];
  char* kimg = lds;
  char* vimg = lds + 64 * PK;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  LatTile t;
  if (tiles) {
    const int* e = tiles + 6 * blockIdx.x;
    t = {e[0], e[1], e[2], e[3], e[4], e[5]};
  } else {  // decode rows: row r is sequence r, one token, its heads in runs of 64
    const int runs = (heads + 63) >> 6;
    const int row = blockIdx.x / runs, h0 = (blockIdx.x % runs) << 6;
    t = {row, row, 1, positions[row], h0, min(64, heads - h0)};
  }
  if (t.seq < 0) return;
  const int slot = wave * 16 + c16;
  const bool valid = slot < t.n_tok * t.hcount;
  const bool wave_active = wave * 16 < t.n_tok * t.hcount;  // wave-uniform
  const float scale2 = scale * LOG2E;
  const int tok = valid ? slot / t.hcount : 0;
  const int head = t.head0 + (valid ? slot % t.hcount : 0);
  const long row = t.row0 + tok;
  const int my_pos = valid ? t.pos0 + tok : -1;
  const int n_pages = (t.pos0 + t.n_tok + PAGE - 1) / PAGE;
  const int p_first = max(0, t.pos0 - window + 1) / PAGE;
  const int per = (n_pages - p_first + splits - 1) / splits;
  const int p_begin = p_first + blockIdx.y * per, p_end = min(n_pages, p_begin + per);
  const int my_first = my_pos - window;  // keys beyond it, up to my_pos, are seen
  const int* bt = block_tables + (long)t.seq * bt_stride;

  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d = K0 + 32 * ks + 8 * g;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (valid)
      v = d < RANK ? ld16(q_lat + row * ql_row + head * ql_head + d) : ld16(q_rot + row * qr_row + head * qr_head + (d - RANK));
    qf[ks] = __builtin_bit_cast(bf16x8, v);
  }
  const bool seeded = splits == 1 && sink != nullptr && valid;
  float m = seeded ? sink[head] * LOG2E : -INFINITY;
  float l = seeded ? 1.f : 0.f;
  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // staging registers: the page's latent part in 4-key x 8-channel blocks, its rotated part in chunks
  u32x4 rb[RB][4];
  u32x4 cb[CB > 0 ? CB : 1];
  auto fetch = [&](int p) {
    const uint16_t* src = cache + (long)bt[p] * page_stride;
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int id = tid + 256 * b, dc = id % (RANK / 8), kq = id / (RANK / 8);
      if (id < NBLK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) rb[b][i] = ld16(src + (long)(4 * kq + i) * ENTRY + 8 * dc);
      }
    }
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int id = tid + 256 * b, dc = id % (ROT / 8), key = id / (ROT / 8);
      cb[b] = ld16(src + (long)key * ENTRY + RANK + 8 * dc);
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int id = tid + 256 * b, dc = id % (RANK / 8), kq = id / (RANK / 8);
      if (id >= NBLK) continue;
      if constexpr (!ROT_ONLY) {
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(kimg + (4 * kq + i) * PK + 16 * dc) = rb[b][i];
      }
      // keys 4 kq .. 4 kq + 3 = 16 n + 4 gg + e  ->  image position (n / 2) * 32 + gg * 8 + (n % 2) * 4 + e
      // = 16-byte chunk (n / 2) * 4 + gg, half n % 2.  Rows 8 dc .. 8 dc + 7 are written by one lane and
      // consecutive lanes hold consecutive dc, 8 rows = 1152 B apart: the chunk index is XORed with dc % 8
      // (= (row / 8) % 8, which the reader undoes) so that those lanes spread over the banks.
      const int n = kq >> 2, gg = kq & 3;
      const int koff = ((((n >> 1) * 4 + gg) ^ (dc & 7)) << 4) + ((n & 1) << 3);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t a0 = rb[b][0][w], a1 = rb[b][1][w], a2 = rb[b][2][w], a3 = rb[b][3][w];
        u32x2 even = {(a0 & 0xffffu) | (a1 << 16), (a2 & 0xffffu) | (a3 << 16)};
        u32x2 odd = {(a0 >> 16) | (a1 & 0xffff0000u), (a2 >> 16) | (a3 & 0xffff0000u)};
        *reinterpret_cast<u32x2*>(vimg + (8 * dc + 2 * w) * PV + koff) = even;
        *reinterpret_cast<u32x2*>(vimg + (8 * dc + 2 * w + 1) * PV + koff) = odd;
      }
    }
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int id = tid + 256 * b, dc = id % (ROT / 8), key = id / (ROT / 8);
      *reinterpret_cast<u32x4*>(kimg + key * PK + 2 * (RANK - K0) + 16 * dc) = cb[b];
    }
  };

  // V^T fragment of (d tile dt, key half kk): row 16 dt + c16, chunk (4 kk + g) ^ ((row / 8) % 8); the row's
  // share of the swizzle is (2 dt) % 8 | c16 / 8, so eight lane offsets cover every dt
  int voff[2][4];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int j = 0; j < 4; ++j) voff[kk][j] = c16 * PV + (((kk * 4 + g) ^ (c16 >> 3) ^ (2 * j)) << 4);

  if (p_begin < p_end) fetch(p_begin);
  for (int p = p_begin; p < p_end; ++p) {
    __syncthreads();  // the previous page's fragment reads are done
    stash();
    __syncthreads();
    if (p + 1 < p_end) fetch(p + 1);  // in flight while this page is multiplied
    if (!wave_active) continue;       // a wave without slots (decode rows of few heads) only helps staging

    f32x4 s[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) s[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(kimg + (16 * nt + c16) * PK + (32 * ks + 8 * g) * 2);
        s[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[ks], s[nt], 0, 0, 0);
      }
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) s[nt] *= scale2;
    // (where every slot of the tile sees the whole page there is nothing to mask)
    if (p * PAGE + PAGE - 1 > t.pos0 || p * PAGE <= t.pos0 + t.n_tok - 1 - window) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = p * PAGE + 16 * nt + 4 * g + e;
          if (key > my_pos || key <= my_first) s[nt][e] = -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[nt][e]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);
    const bool dead = mn == -INFINITY;   // nothing seen so far and nothing visible here:
    const float mref = dead ? 0.f : mn;  // every score is -inf and weighs 0
    const float corr = dead ? 1.f : __builtin_amdgcn_exp2f(m - mref);
    float ps = 0.f;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float pv = __builtin_amdgcn_exp2f(s[nt][e] - mref);
        s[nt][e] = pv;
        ps += pv;
      }
    ps += __shfl_xor(ps, 16, 64);
    ps += __shfl_xor(ps, 32, 64);
    l = l * corr + ps;
    m = mn;
    bf16x8 pf[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      u32x4 w = {pack_bf16x2(s[2 * kk][0], s[2 * kk][1]), pack_bf16x2(s[2 * kk][2], s[2 * kk][3]),
                 pack_bf16x2(s[2 * kk + 1][0], s[2 * kk + 1][1]), pack_bf16x2(s[2 * kk + 1][2], s[2 * kk + 1][3])};
      pf[kk] = __builtin_bit_cast(bf16x8, w);
    }
    if (!__all(corr == 1.f)) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= corr;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(vimg + voff[kk][dt & 3] + dt * 16 * PV);
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pf[kk], o[dt], 0, 0, 0);
      }
    }
  }

  if (!valid) return;
  if (splits == 1) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t* dst = out + row * o_row + head * o_head + 4 * g;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      u32x2 w = {pack_bf16x2(o[dt][0] * inv, o[dt][1] * inv), pack_bf16x2(o[dt][2] * inv, o[dt][3] * inv)};
      *reinterpret_cast<u32x2*>(dst + 16 * dt) = w;
    }
  } else {
    const long rec = ((long)blockIdx.x * splits + blockIdx.y) * 64 + slot;
    float* dst = ws_o + rec * RANK + 4 * g;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(dst + 16 * dt) = o[dt];
    if (g == 0) {
      ws_ml[2 * rec] = m * LN2;
      ws_ml[2 * rec + 1] = l;
    }
  }
}

// The same walk for wide entries (512 + 64), decode rows here and tiles of 64 slots in the kernel behind it: pages go straight
// into LDS, two of them, and the second product reads its transposed operand from the K image through the transposing LDS read.
// What it replaces was bound by staging: a page passed through 128 registers into a K and a V^T image (137 KB of LDS writes with
// 4 x 4 transposes) between two barriers, and a decode tile of 32 heads left two of the four waves idle meanwhile.
//   * Image: 64 rows of ENTRY values without padding; a row's 16-byte chunk j lies at j ^ f(row), f = (row / 2 % 4) * 2 +
//     row / 8 % 2 (applied to the source address: a wave's load fills 1 KiB of LDS in lane order).  The 16 rows of a K fragment
//     then cover all banks, and so do the 8 rows x 32 bytes that half a wave reads transposed.
//   * ds_read_b64_tr_b16 gives lane (c, g) the keys 4 g .. 4 g + 3 of channel c: the order in which the S accumulators hold them.
//   * Two pages are on their way except while one is read: the page after next is asked for as soon as its buffer is free, before
//     the next one is waited for (a counted wait).  Waiting for each page before asking for another left 4.5 TB/s.
//   * Decode rows of at most 32 heads: eight waves, four of which share 16 slots.  Each scores 16 keys of a page, the
//     four exchange scores through 8 KB of LDS, keep the same softmax state and sum a quarter of the channels over all 64 keys.
//     (With keys and states of its own a wave held all channels, and joining the four moved 130 KB through LDS at the end: 4 to 5 us
//     that ranges of one or two pages could not hide.)  A quarter of a page's values fits into registers beside the rest, so the
//     page is read whole before the scores go round: that barrier frees its buffer, and softmax and second product run with two
//     pages on their way (one sequence of 26k entries 52 -> 49 us, 200 of 2k 115 -> 104).
//     The weights enter as two parts of 16 bits, a matrix instruction more for every value fragment that is read: with one part and
//     one maximum for all 64 keys the error against 64 bits was 2.03e-3 on average over batches and contexts, with a maximum for
//     each quarter 1.97e-3, with two parts it is 1.66e-3, the rounding of the result.
//   * Decode rows read a page once: non-temporal loads (5.6 against 4.5 TB/s without the arithmetic).
//     The exchange, softmax and second product of a page stand between its last read and the next one's first: maxima over lane groups
//     by lane swaps instead of through LDS, sums kept by lane until the end, scores scaled where they are weighed (32 heads, one sequence of
//     26k entries 44.7 -> 40.8 us, 200 of 2k 98.6 -> 93.5, 32 of 4k 35.4 -> 34.3; 16 heads, one of 26k 34.5 -> 30.4).
// Decode rows with their merge, pages from memory, staged through registers / this: 32 heads, 32 sequences of 4k entries in 8 ranges
// 65 / 34 us, 8 of 8k in 32 42 / 26, one of 26k in 32 86 / 41.

// o[dt] += V^T fragment of d tile dt x P^T.  In assembly because the compiler makes the builtin wait for the pages that are on
// their way into LDS; the reads are waited for in the block that issues them.  32 keys: two transposed reads of 4 keys x 16
// channels a tile, keys 16 apart, eight tiles a block.
template <int ROW>
__device__ __forceinline__ void read_transposed(u32x2 (&r)[16], const uint32_t (&at)[4]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %16 offset:%20\n\tds_read_b64_tr_b16 %1, %16 offset:%21\n\t"
      "ds_read_b64_tr_b16 %2, %17 offset:%20\n\tds_read_b64_tr_b16 %3, %17 offset:%21\n\t"
      "ds_read_b64_tr_b16 %4, %18 offset:%20\n\tds_read_b64_tr_b16 %5, %18 offset:%21\n\t"
      "ds_read_b64_tr_b16 %6, %19 offset:%20\n\tds_read_b64_tr_b16 %7, %19 offset:%21\n\t"
      "ds_read_b64_tr_b16 %8, %16 offset:%22\n\tds_read_b64_tr_b16 %9, %16 offset:%23\n\t"
      "ds_read_b64_tr_b16 %10, %17 offset:%22\n\tds_read_b64_tr_b16 %11, %17 offset:%23\n\t"
      "ds_read_b64_tr_b16 %12, %18 offset:%22\n\tds_read_b64_tr_b16 %13, %18 offset:%23\n\t"
      "ds_read_b64_tr_b16 %14, %19 offset:%22\n\tds_read_b64_tr_b16 %15, %19 offset:%23\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7]), "=&v"(r[8]),
        "=&v"(r[9]), "=&v"(r[10]), "=&v"(r[11]), "=&v"(r[12]), "=&v"(r[13]), "=&v"(r[14]), "=&v"(r[15])
      : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(0), "n"(16 * ROW), "n"(128), "n"(128 + 16 * ROW)
      : "memory");
}

// The weights in two parts of 16 bits, high and low.
__device__ __forceinline__ void multiply_tiles(f32x4* o, const u32x2 (&r)[16], const bf16x8 (&pf)[2]) {
#pragma unroll
  for (int part = 0; part < 2; ++part)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, (u32x4){r[2 * i][0], r[2 * i][1], r[2 * i + 1][0], r[2 * i + 1][1]}),
                                                     pf[part], o[i], 0, 0, 0);
}
// How many of `splits` key ranges a decode row of `pages` pages is cut into.  A workgroup fills a CU (two pages in LDS) and what it
// does once - queries, the first page's way, a partial result of 64 KB - takes about as long as four pages (two or three give the
// same times), so more workgroups than a round of 256 only pay if their ranges are long: 100 sequences of 1000 entries in 8 ranges
// of two pages were four rounds.  In a graph with the merge, all ranges / those used: 100 x 1000 entries 74 / 43 us, 40 x 3000 (7 / 6) 56 / 42,
// 33 x 12000 (8 / 7) 139 / 97; 128 x 100, where a row has two pages, 23 / 24.5.
// `rows` are those of the step's batch bucket, not of the launch: a row's ranges, and with them the order of its sums, are the same
// in a captured step that is padded to the bucket and in an eager one that is not.
constexpr int WIDE_ONCE = 4;
// A prefill tile's ranges are no shorter than this (the launch's count is chosen from the widest table).  A tile of one range finishes its
// rows itself, and the merge passes over it (300 rows of 32 heads behind a table of 512 pages, two ranges a tile: 44 -> 32 us; 28 uncut).
constexpr int TILE_RANGE_PAGES = 4;
__device__ __forceinline__ int tile_ranges(int pos0, int n_tok, int window, int splits) {
  const int pages = (pos0 + n_tok + PAGE - 1) / PAGE - max(0, pos0 - window + 1) / PAGE;
  return min(splits, max(1, pages / TILE_RANGE_PAGES));
}
__device__ __forceinline__ int wide_splits(int pages, int rows, int splits) {
  int best = 1 << 30, used = splits;
  for (int r = 1; rows * splits > 256; ++r) {
    const int e = min(splits, max(1, r * 256 / rows)), cost = (rows * e + 255) / 256 * ((pages + e - 1) / e + WIDE_ONCE);
    if (cost < best) best = cost, used = e;
    if (e == splits) break;
  }
  return used;
}

// (In assembly where a value comes from another lane or from LDS: the compiler would quieten it first, two instructions more for one.)
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float max_of_swapped(uint32_t a, uint32_t b) {  // (two states before a swap reads what a vector instruction wrote)
  float r;
  asm("v_max_f32 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// The maximum over the lanes c, c + 16, c + 32, c + 48.
__device__ __forceinline__ float max_of_groups(float x) {
  const auto far = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const uint32_t half = __float_as_uint(max_of_swapped(far[0], far[1]));
  const auto near = __builtin_amdgcn_permlane16_swap(half, half, false, false);
  return max_of_swapped(near[0], near[1]);
}
// Lane group g: the maximum of x[g] over the four groups' lanes of one number.  Swapping halves of two values leaves two of their four
// parts in each half, and then swapping groups of 16 lanes the four values in the four groups.
__device__ __forceinline__ float max_of_groups(const float (&x)[4]) {
  const auto half = [](float a, float b) {
    const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return max_of_swapped(both[0], both[1]);
  };
  const float even = half(x[0], x[2]), odd = half(x[1], x[3]);
  const auto both = __builtin_amdgcn_permlane16_swap(__float_as_uint(even), __float_as_uint(odd), false, false);
  return max_of_swapped(both[0], both[1]);
}

// Scores are scaled behind their masks and maxima: by a positive number, their sign turned before where the scale is negative.  (Comparisons
// and not fmaxf, which would drop a NaN that has to reach the result; the same for a sink, at which the running maximum starts.)
__device__ __forceinline__ float positive_scale(float scale) {
  const float x = fabsf(scale) * LOG2E;
  return x < FLT_MIN ? FLT_MIN : x;
}
__device__ __forceinline__ float finite_seed(float sink) {
  const float x = sink * LOG2E;
  return x < -FLT_MAX ? -FLT_MAX : x;
}

// Decode rows of at most 32 heads.
template <int RANK, int ROT>
__global__ __launch_bounds__(512, 2) void latent_wide_kernel(
    const uint16_t* __restrict__ q_lat, long ql_row, long ql_head, const uint16_t* __restrict__ q_rot, long qr_row,
    long qr_head, const uint16_t* __restrict__ cache, long page_stride, const int* __restrict__ block_tables,
    int bt_stride, const int* __restrict__ positions, int heads, const float* __restrict__ sink, uint16_t* __restrict__ out,
    long o_row, long o_head, float scale, int window, int splits, float* __restrict__ ws_o, float* __restrict__ ws_ml, int bucket) {
  constexpr int ENTRY = RANK + ROT, KS = ENTRY / 32, DT = RANK / 16, ROW = ENTRY * 2, PAGE_BYTES = 64 * ROW;
  constexpr int WAVES = 8, SHARE = 4;              // waves that share 16 slots
  constexpr int NI = PAGE_BYTES / (1024 * WAVES);  // KiB of a page that a wave loads
  constexpr int DW = DT / SHARE;                   // 16-channel tiles that it sums
  static_assert(ENTRY % 64 == 0 && DW == 8, "chunks are exchanged within groups of eight; eight tiles a block of reads");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  const int sg = wave / SHARE, part = wave % SHARE;  // slots; keys and channels
  const int row = blockIdx.x, slot = sg * 16 + c16;
  const int pos = positions[row];
  const bool valid = slot < heads;
  const bool wave_active = sg * 16 < heads;  // wave-uniform
  const float scale2 = positive_scale(scale);
  const int head = valid ? slot : 0;
  // The queries come through LDS, where the second page will lie: latent parts of 1 KiB, then rotated parts of 128 bytes, 16-byte chunks
  // exchanged so that a fragment's rows lie on different banks.  (Four waves read the same 16 rows, and a fragment read from memory takes
  // half of every line; with the second page asked for only behind these reads, 32 sequences of 4k entries, 32 heads, still take 38.7 ->
  // 35.3 us, 100 of 1000 40.1 -> 36.7, one of 26k 48.4 -> 44.9; 16 heads 31.4 -> 29.1, 30.0 -> 27.3, 37.0 -> 34.5.)  In a single round
  // every range may be used, and the queries are on their way while the row's position and page are looked up (one sequence of 2k
  // entries 18.6 -> 17.7 us); with more, most of the workgroups have nothing to do (100 x 400 entries 37 -> 31 if they don't load them).
  static_assert(RANK == 512 && ROT == 64, "a wave's load is a query's latent part or eight rotated ones");
  char* const queries = lds + PAGE_BYTES;
  auto load_q = [&]() {
    const uint16_t* const ql = q_lat + (long)row * ql_row;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int of = 4 * wave + i;
      if (of < heads)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)(ql + of * ql_head), 0, RANK * 2, 0x00020000),
                                                 (__attribute__((address_space(3))) void*)(queries + of * 1024), 16, (lane ^ (of & 15)) * 16, 0, 0, 0);
    }
    if (wave < 4) {
      const int at = 8 * wave + (lane >> 3);
      const uint16_t* const q = q_rot + (long)row * qr_row + (at < heads ? at : 0) * qr_head + ((lane ^ (at >> 1)) & 7) * 8;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)q,
                                       (__attribute__((address_space(3))) void*)(queries + 32 * 1024 + wave * 1024), 16, 0, 0);
    }
  };
  const bool all_used = bucket * splits <= 256;
  if (all_used) load_q();
  const int n_pages = (pos + PAGE) / PAGE, p_first = max(0, pos - window + 1) / PAGE;
  const int used = wide_splits(n_pages - p_first, bucket, splits);
  const int per = (n_pages - p_first + used - 1) / used;
  const int p_begin = p_first + blockIdx.y * per, p_end = min(n_pages, p_begin + per);
  if (splits > 1 && p_begin >= p_end) {  // nothing to see: the merge passes over the record
    if (tid < heads) {
      const long rec = ((long)blockIdx.x * splits + blockIdx.y) * 64 + tid;
      ws_ml[2 * rec] = -INFINITY;
      ws_ml[2 * rec + 1] = 0.f;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (nothing may still be on its way to LDS)
    return;
  }
  if (!all_used) load_q();
  const int* bt = block_tables + (long)row * bt_stride;

  int src_off[NI];  // bytes into a page of what this lane loads into byte (WAVES i + wave) * 1024 + lane * 16 of the image
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int o = (WAVES * i + wave) * 1024 + lane * 16, r = o / ROW, ch = (o % ROW) >> 4;
    src_off[i] = r * ROW + ((ch ^ (((r >> 1) & 3) << 1 | ((r >> 3) & 1))) << 4);
  }
  auto load_page = [&](int p, int buf) {
    const char* src = reinterpret_cast<const char*>(cache + (long)bt[p] * page_stride);
#pragma unroll
    for (int i = 0; i < NI; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + src_off[i]),
                                       (__attribute__((address_space(3))) void*)(lds + buf * PAGE_BYTES + (WAVES * i + wave) * 1024),
                                       16, 0, 2);  // 2: non-temporal
  };
  const bool seeded = splits == 1 && sink != nullptr && valid;
  float m = seeded ? finite_seed(sink[head]) : -FLT_MAX;
  float l = seeded && g == 0 ? 1.f : 0.f;  // of this lane's keys alone
  f32x4 o[DW];
#pragma unroll
  for (int dt = 0; dt < DW; ++dt) o[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // K fragment of (this wave's key tile, step ks): row 16 part + c16, chunk 4 ks + g; V^T fragment of (d tile dt, 16 keys from 16 n):
  // the lane points at row 16 n + 4 g + lane / 4 % 4, channels 16 dt + 4 (lane % 4)
  const int fk = ((c16 >> 1) & 3) << 1 | (c16 >> 3);
  int koff[2], voff[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) koff[i] = (16 * part + c16) * ROW + (((i * 4 + g) ^ fk) << 4);
  const int vr = 4 * g + ((lane >> 2) & 3), fv = ((vr >> 1) & 3) << 1 | (vr >> 3);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    voff[i] = vr * ROW + (((2 * i + ((lane & 3) >> 1)) ^ fv) << 4) + (lane & 1) * 8 + part * DW * 32;

  bf16x8 qf[KS];
  f32x4 s[4];  // scores, then weights, of a page's keys
  auto score = [&](int buf) {
    const char* img = lds + buf * PAGE_BYTES;
    s[0] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      s[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(img + koff[ks & 1] + (ks >> 1) * 128), qf[ks], s[0], 0, 0, 0);
  };
  auto weigh = [&](int p) {
    if (scale < 0.f || p * PAGE + PAGE - 1 > pos || p * PAGE <= pos - window) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (scale < 0.f) s[nt][e] = -s[nt][e];
          const int key = p * PAGE + 16 * nt + 4 * g + e;
          if (key > pos || key <= pos - window) s[nt][e] = -INFINITY;
        }
    }
    float mx = max3(s[0][0], s[0][1], s[0][2]);
    mx = max3(mx, s[0][3], s[1][0]);
    mx = max3(mx, s[1][1], s[1][2]);
    mx = max3(mx, s[1][3], s[2][0]);
    mx = max3(mx, s[2][1], s[2][2]);
    mx = max3(mx, s[2][3], s[3][0]);
    mx = max3(mx, s[3][1], s[3][2]);
    const float mn = fmaxf(m, max_of_groups(max3(mx, s[3][3], s[3][3])) * scale2);
    const float corr = __builtin_amdgcn_exp2f(m - mn);
    float ps[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
#pragma unroll
      for (int e = 0; e < 4; ++e) s[nt][e] = __builtin_amdgcn_exp2f(fmaf(s[nt][e], scale2, -mn));
      ps[nt] = (s[nt][0] + s[nt][1]) + (s[nt][2] + s[nt][3]);
    }
    l = l * corr + ((ps[0] + ps[1]) + (ps[2] + ps[3]));
    m = mn;
    if (!__all(corr == 1.f)) {
#pragma unroll
      for (int dt = 0; dt < DW; ++dt) o[dt] *= corr;
    }
  };
  auto weights = [&](int kk, bf16x8 (&pf)[2]) {  // of keys 32 kk ..
    u32x4 w, low;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p0 = s[2 * kk + (i >> 1)][2 * (i & 1)], p1 = s[2 * kk + (i >> 1)][2 * (i & 1) + 1];
      w[i] = pack_bf16x2(p0, p1);
      low[i] = pack_bf16x2(p0 - bf16lo(w[i]), p1 - bf16hi(w[i]));
    }
    pf[0] = __builtin_bit_cast(bf16x8, w);
    pf[1] = __builtin_bit_cast(bf16x8, low);
  };
  auto everyone = [&]() {  // (not __syncthreads, which would wait for the pages on their way)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  if (p_begin < p_end) {
    load_page(p_begin, 0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");  // the queries have landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int of = valid ? slot : 0, lat = of * 1024 + ((g ^ (of & 3)) << 4 | (of & 12) << 4);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = *reinterpret_cast<const bf16x8*>(queries + (32 * ks < RANK ? (lat ^ ((ks & 3) << 6)) + (ks >> 2) * 256
                                                                          : 32 * 1024 + of * 128 + (((4 * ks + g) ^ (of >> 1)) & 7) * 16));
    everyone();
    if (p_begin + 1 < p_end) load_page(p_begin + 1, 1);
  }
  for (int p = p_begin; p < p_end; ++p) {
    const int buf = (p - p_begin) & 1;
    const uint32_t page = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds + buf * PAGE_BYTES;
    // this page has landed (mine: all but the NI loads of the page behind it; everyone's: the barrier)
    if (p + 1 < p_end) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // a page is read whole before its scores go round: the barrier of that exchange frees its buffer as well
    f32x4* round = reinterpret_cast<f32x4*>(lds + 2 * PAGE_BYTES) + sg * 256 + lane;  // of four key quarters
    u32x2 v0[16], v1[16];
    if (wave_active) {
      score(buf);
      round[part * 64] = s[0];
      const uint32_t at0[4] = {page + voff[0], page + voff[1], page + voff[2], page + voff[3]};
      read_transposed<ROW>(v0, at0);
      const uint32_t at1[4] = {at0[0] + 32 * ROW, at0[1] + 32 * ROW, at0[2] + 32 * ROW, at0[3] + 32 * ROW};
      read_transposed<ROW>(v1, at1);
    }
    everyone();
    if (p + 2 < p_end) load_page(p + 2, buf);
    if (wave_active) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) s[nt] = round[nt * 64];
      weigh(p);
      bf16x8 pf[2];
      weights(0, pf);
      multiply_tiles(o, v0, pf);
      weights(1, pf);
      multiply_tiles(o, v1, pf);
    }
  }

  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (!valid) return;
  if (splits == 1) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t* dst = out + (long)row * o_row + head * o_head + part * DW * 16 + 4 * g;
#pragma unroll
    for (int dt = 0; dt < DW; ++dt) {
      u32x2 w = {pack_bf16x2(o[dt][0] * inv, o[dt][1] * inv), pack_bf16x2(o[dt][2] * inv, o[dt][3] * inv)};
      *reinterpret_cast<u32x2*>(dst + 16 * dt) = w;
    }
  } else {
    const long rec = ((long)blockIdx.x * splits + blockIdx.y) * 64 + slot;
    float* dst = ws_o + rec * RANK + part * DW * 16 + 4 * g;
#pragma unroll
    for (int dt = 0; dt < DW; ++dt) *reinterpret_cast<f32x4*>(dst + 16 * dt) = o[dt];
    if (g == 0 && part == 0) {
      ws_ml[2 * rec] = m * LN2;
      ws_ml[2 * rec + 1] = l;
    }
  }
}

// Tiles of 64 slots (prefill chunks, decode rows of more than 32 heads), images and pages as above.  What bounds a tile is reading a
// page's fragments from LDS.  Eight waves, two of which shared 16 slots, read every fragment four times, 550 KB a page, and took 3.1 us
// for it; waves of 32 slots read half of that, but two on a SIMD spill (143 to 285 registers of 256, 0.79x).  So four waves with all 64
// slots, one on a SIMD, whose queries take the 256 accumulator registers:
//   * A wave scores 16 of a page's keys for all slots and sums a quarter of the channels over all keys: each K and V^T fragment is read
//     once and multiplied with four tiles of slots.  The waves exchange their keys' maxima by slot, then the weights in 16 bits (9 KB
//     instead of 16 KB of scores).  A lane adds up its own keys' weights; the sums meet at the end.
//   * Nothing but the order of instructions hides a wait: reads run three fragments in front of their products, the next page's loads
//     go out one a step of the scores (all at once, they held those up), and rows past the list's last page load no bytes.
//   * Queries come through LDS (below): 5 us a workgroup less than as fragments from memory.
//   * Nothing runs beside a lone wave's vector instructions, so those between the two products count in full, 1 % of the time for
//     every 20: the four slot tiles' maxima over lane groups take three swaps together, scores are scaled where they are weighed, one
//     branch holds masks and negative scales, the state starts at a finite number, a wave's weights lie as the second product reads them
//     (2000 rows behind 6000 entries 1070 -> 919 us, 60 behind 7940 59.6 -> 54.7).  Reads of the next page's keys or of the values further
//     ahead, and the page's loads in the first half of the scores, are slower by 0 to 2 %.
// 2.1 us a page.  32 heads: 2000 rows behind 6000 entries 1399 -> 919 us, 2000 of one sequence 248 -> 178, 600 behind 7400 565 -> 390,
// 200 behind 3800 122 -> 88, 20 behind 1980 32.7 -> 27.6; 16 heads, 60 behind 7940 47.0 -> 38.4; decode rows, 32 sequences of 4k
// entries, 64 heads 49.7 -> 41, 128 heads 76.6 -> 61.  Errors against 64 bits are what they were, to four digits.
// Lists of few tiles are cut along the keys (ops/latent.py).
__device__ __forceinline__ bf16x8 read_transposed_pair(const char* lo, const char* hi) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* lds_ptr;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)lo);
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)hi);
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int RANK, int ROT>
__global__ __launch_bounds__(256, 1) void latent_tile_kernel(
    const uint16_t* __restrict__ q_lat, long ql_row, long ql_head, const uint16_t* __restrict__ q_rot, long qr_row,
    long qr_head, const uint16_t* __restrict__ cache, long page_stride, const int* __restrict__ block_tables,
    int bt_stride, const int* __restrict__ tiles, const int* __restrict__ positions, int heads,
    const float* __restrict__ sink, uint16_t* __restrict__ out, long o_row, long o_head, float scale, int window,
    int splits, float* __restrict__ ws_o, float* __restrict__ ws_ml, int bucket) {
  constexpr int ENTRY = RANK + ROT, KS = ENTRY / 32, ROW = ENTRY * 2, PAGE_BYTES = 64 * ROW, NS = 4;
  constexpr int NI = PAGE_BYTES / 4096;  // KiB of a page that a wave loads
  constexpr int DW = RANK / 64;          // 16-channel tiles that a wave sums
  static_assert(ENTRY % 64 == 0 && NI <= 20, "chunks are exchanged within groups of eight; three bits a load");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, part = __builtin_amdgcn_readfirstlane(tid >> 6);  // keys and channels
  const int c16 = lane & 15, g = lane >> 4;
  LatTile t;
  if (tiles) {
    const int* e = tiles + 6 * blockIdx.x;
    t = {e[0], e[1], e[2], e[3], e[4], e[5]};
  } else {
    const int runs = (heads + 63) >> 6;
    const int row = blockIdx.x / runs, h0 = (blockIdx.x % runs) << 6;
    t = {row, row, 1, positions[row], h0, min(64, heads - h0)};
  }
  if (t.seq < 0) return;
  const int n_slots = t.n_tok * t.hcount;
  const int n_pages = (t.pos0 + t.n_tok + PAGE - 1) / PAGE;
  const int p_first = max(0, t.pos0 - window + 1) / PAGE;
  const int used = tiles ? tile_ranges(t.pos0, t.n_tok, window, splits) : wide_splits(n_pages - p_first, bucket, splits);
  const bool whole = splits == 1 || (tiles && used == 1);
  const int per = (n_pages - p_first + used - 1) / used;
  const int p_begin = p_first + blockIdx.y * per, p_end = min(n_pages, p_begin + per);
  if (splits > 1 && p_begin >= p_end) {  // nothing to see: the merge passes over the record
    if (!whole && tid < n_slots) {
      const long rec = ((long)blockIdx.x * splits + blockIdx.y) * 64 + tid;
      ws_ml[2 * rec] = -INFINITY;
      ws_ml[2 * rec + 1] = 0.f;
    }
    return;
  }
  const int* bt = block_tables + (long)t.seq * bt_stride;
  // chunk (4 i + part) * 64 + lane of the image comes from the chunk whose low three bits are those of lane ^ f(row): three bits a load
  uint32_t swizzle[2] = {0, 0};
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = ((4 * i + part) * 64 + lane) / (ROW / 16);
    swizzle[i / 10] |= (uint32_t)(((r >> 1) & 3) << 1 | ((r >> 3) & 1)) << (3 * (i % 10));
  }
  // the i-th KiB of this wave of page p (past the last: of no bytes)
  auto load = [&](int p, int buf, int i) {
    const __amdgpu_buffer_rsrc_t src =
        __builtin_amdgcn_make_buffer_rsrc((void*)(cache + (long)bt[min(p, p_end - 1)] * page_stride), 0, p < p_end ? PAGE_BYTES : 0, 0x00020000);
    uint32_t f = swizzle[i / 10];
    asm volatile("" : "+v"(f));  // (or the compiler keeps all the addresses)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (__attribute__((address_space(3))) void*)(lds + buf * PAGE_BYTES + (4 * i + part) * 1024), 16,
                                             (int)((lane ^ ((f >> (3 * (i % 10))) & 7)) * 16), (4 * i + part) * 1024, 0, 0);
  };
  static_assert(NI == KS, "a load a step");
  // The queries come through LDS, where the second page will lie: read as fragments from memory, by every wave, they were lines used by
  // half, and took as long as two pages.  Latent parts of 1 KiB a slot, then rotated parts of 128 bytes, 16-byte chunks exchanged so that
  // a fragment's rows lie on different banks.  (A slot past the tile reads the tile's first query, and nothing of it is stored.)
  static_assert(RANK == 512 && ROT == 64, "a wave's load is a query's latent part or eight rotated ones");
  char* const queries = lds + PAGE_BYTES;
  const bool seeded = whole && sink != nullptr;
  float seed[NS] = {0.f, 0.f, 0.f, 0.f};
  if (seeded)  // (asked for before the rest, that nothing of it is waited for)
#pragma unroll
    for (int j = 0; j < NS; ++j) seed[j] = sink[t.head0 + (16 * j + c16) % t.hcount];
  {
    int tok = 16 * part / t.hcount, head = 16 * part - tok * t.hcount;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const bool valid = 16 * part + i < n_slots;
      const uint16_t* const q = q_lat + (t.row0 + (valid ? tok : 0)) * ql_row + (t.head0 + (valid ? head : 0)) * ql_head;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)q, 0, RANK * 2, 0x00020000),
                                               (__attribute__((address_space(3))) void*)(queries + (16 * part + i) * 1024), 16, (lane ^ i) * 16, 0, 0, 0);
      if (++head == t.hcount) ++tok, head = 0;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int at = 16 * part + 8 * i + (lane >> 3), slot = at < n_slots ? at : 0, of = slot / t.hcount;
      const uint16_t* const q = q_rot + (t.row0 + of) * qr_row + (t.head0 + slot - of * t.hcount) * qr_head + ((lane ^ (at >> 1)) & 7) * 8;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)q,
                                       (__attribute__((address_space(3))) void*)(queries + 64 * 1024 + (2 * part + i) * 1024), 16, 0, 0);
    }
  }
  if (p_begin < p_end)
#pragma unroll
    for (int i = 0; i < NI; ++i) load(p_begin, 0, i);

  const float scale2 = positive_scale(scale);
  bf16x8 qf[NS][KS];
  int* const last_seen = reinterpret_cast<int*>(lds + 2 * PAGE_BYTES + 9 * 1024) + c16;  // by slot
  float m[NS], l[NS];  // l: of this lane's keys alone
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int slot = 16 * j + c16;
    const bool valid = slot < n_slots;
    m[j] = seeded && valid ? finite_seed(seed[j]) : -FLT_MAX;  // (finite: a page of which a slot sees nothing needs no care)
    l[j] = seeded && valid && part == 0 && g == 0 ? 1.f : 0.f;
    if (part == 0 && g == 0) last_seen[16 * j] = valid ? t.pos0 + slot / t.hcount : -1;  // (read behind the first page's barrier)
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NI) : "memory");  // the queries have landed (a tile sees a page)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int row = 16 * j + c16, lat = row * 1024 + ((g ^ (c16 & 3)) << 4 | (c16 & 12) << 4);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qf[j][ks] = *reinterpret_cast<const bf16x8*>(queries + (32 * ks < RANK ? (lat ^ ((ks & 3) << 6)) + (ks >> 2) * 256
                                                                             : 64 * 1024 + row * 128 + (((4 * ks + g) ^ (row >> 1)) & 7) * 16));
    }
#pragma unroll
    for (int ks = 0; ks < RANK / 32; ++ks) asm volatile("" : "+a"(qf[j][ks]));  // in accumulator registers: the others are taken
  }
  f32x4 o[NS][DW];
#pragma unroll
  for (int j = 0; j < NS; ++j)
#pragma unroll
    for (int dt = 0; dt < DW; ++dt) o[j][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // K fragment of (this wave's key tile, step ks): row 16 part + c16, chunk 4 ks + g; V^T fragments: see latent_wide_kernel
  const int fk = ((c16 >> 1) & 3) << 1 | (c16 >> 3);
  const int koff = (16 * part + c16) * ROW + ((g ^ fk) << 4);
  const int vr = 4 * g + ((lane >> 2) & 3), fv = ((vr >> 1) & 3) << 1 | (vr >> 3);
  const int voff = vr * ROW + ((((lane & 3) >> 1) ^ fv) << 4) + (lane & 1) * 8 + part * DW * 32;
  float* const maxima = reinterpret_cast<float*>(lds + 2 * PAGE_BYTES);                // [slot][key tile]
  u32x4* const weights = reinterpret_cast<u32x4*>(lds + 2 * PAGE_BYTES + 1024) + lane;  // [keys 32 ..][slot tile][lane][16 of the keys]
  auto everyone = [&]() {  // (not __syncthreads, which would wait for the page on its way)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  for (int p = p_begin; p < p_end; ++p) {
    const int buf = (p - p_begin) & 1;
    const char* const img = lds + buf * PAGE_BYTES;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this page has landed; behind the barrier nobody reads the other any more
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    f32x4 s[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) s[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    {
      constexpr int AHEAD = 3;  // the products follow the reads
      bf16x8 kf[KS];
      auto read_k = [&](int ks) { kf[ks] = *reinterpret_cast<const bf16x8*>(img + (koff ^ ((ks & 1) << 6)) + (ks >> 1) * 128); };
#pragma unroll
      for (int ks = 0; ks < AHEAD; ++ks) read_k(ks);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + AHEAD < KS) read_k(ks + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NS; ++j) s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], qf[j][ks], s[j], 0, 0, 0);
        load(p + 1, buf ^ 1, ks);  // (all of them in front of the scores would hold those up)
      }
    }
    const bool masked = p * PAGE + PAGE - 1 > t.pos0 || p * PAGE <= t.pos0 + t.n_tok - 1 - window;
    if (masked || scale < 0.f) {
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        if (scale < 0.f) s[j] = -s[j];
        const int my_pos = last_seen[16 * j];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = p * PAGE + 16 * part + 4 * g + e;
          if (key > my_pos || key <= my_pos - window) s[j][e] = -INFINITY;
        }
      }
    }
    float top[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) top[j] = fmaxf(fmaxf(s[j][0], s[j][1]), fmaxf(s[j][2], s[j][3]));
    maxima[lane * 4 + part] = max_of_groups(top) * scale2;
    everyone();
    f32x4 mx[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) mx[j] = *reinterpret_cast<const f32x4*>(maxima + (16 * j + c16) * 4);
    float corr[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const float mn = max3(max3(m[j], mx[j][0], mx[j][1]), mx[j][2], mx[j][3]);
      corr[j] = __builtin_amdgcn_exp2f(m[j] - mn);
      float w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = __builtin_amdgcn_exp2f(fmaf(s[j][e], scale2, -mn));
      reinterpret_cast<u32x2*>(weights + ((part >> 1) * NS + j) * 64)[part & 1] = (u32x2){pack_bf16x2(w[0], w[1]), pack_bf16x2(w[2], w[3])};
      l[j] = l[j] * corr[j] + ((w[0] + w[1]) + (w[2] + w[3]));
      m[j] = mn;
    }
#pragma unroll
    for (int j = 0; j < NS; ++j)
      if (!__all(corr[j] == 1.f)) {
#pragma unroll
        for (int dt = 0; dt < DW; ++dt) o[j][dt] *= corr[j];
      }
    {
      constexpr int AHEAD = 3;
      bf16x8 vf[2 * DW], pf[2][NS];
      auto read_v = [&](int x) {  // keys 32 (x / DW) .., channel tile x % DW
        const char* const at = img + (voff ^ ((x & 3) << 5)) + (x % DW >> 2) * 128 + x / DW * 32 * ROW;
        vf[x] = read_transposed_pair(at, at + 16 * ROW);
      };
      auto read_p = [&](int kk) {
#pragma unroll
        for (int j = 0; j < NS; ++j) pf[kk][j] = __builtin_bit_cast(bf16x8, weights[(kk * NS + j) * 64]);
      };
#pragma unroll
      for (int x = 0; x < AHEAD; ++x) read_v(x);
      everyone();
      read_p(0);
#pragma unroll
      for (int x = 0; x < 2 * DW; ++x) {
        if (x + AHEAD < 2 * DW) read_v(x + AHEAD);
        if (x == DW - 2) read_p(1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NS; ++j) o[j][x % DW] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[x], pf[x / DW][j], o[j][x % DW], 0, 0, 0);
      }
    }
  }

  // the waves' and lanes' shares of the sums (nothing may still write to LDS)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    l[j] += __shfl_xor(l[j], 16, 64);
    l[j] += __shfl_xor(l[j], 32, 64);
    if (g == 0) maxima[(16 * j + c16) * 4 + part] = l[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int slot = 16 * j + c16;
    if (slot >= n_slots) continue;
    const f32x4 all = *reinterpret_cast<const f32x4*>(maxima + (16 * j + c16) * 4);
    const float sum = (all[0] + all[1]) + (all[2] + all[3]);
    if (whole) {
      const float inv = sum > 0.f ? 1.f / sum : 0.f;
      uint16_t* dst = out + (long)(t.row0 + slot / t.hcount) * o_row + (t.head0 + slot % t.hcount) * o_head + part * DW * 16 + 4 * g;
#pragma unroll
      for (int dt = 0; dt < DW; ++dt)
        *reinterpret_cast<u32x2*>(dst + 16 * dt) = (u32x2){pack_bf16x2(o[j][dt][0] * inv, o[j][dt][1] * inv),
                                                          pack_bf16x2(o[j][dt][2] * inv, o[j][dt][3] * inv)};
    } else {
      const long rec = ((long)blockIdx.x * splits + blockIdx.y) * 64 + slot;
      float* dst = ws_o + rec * RANK + part * DW * 16 + 4 * g;
#pragma unroll
      for (int dt = 0; dt < DW; ++dt) *reinterpret_cast<f32x4*>(dst + 16 * dt) = o[j][dt];
      if (g == 0 && part == 0) {
        ws_ml[2 * rec] = m[j] * LN2;
        ws_ml[2 * rec + 1] = sum;
      }
    }
  }
}

// One workgroup per (tile, slot): out = sum_s o_s exp(m_s - M) / (sum_s l_s exp(m_s - M) + exp(sink - M)).  The splits'
// factors are made once, by a wave with a split per lane; a thread then owns runs of 4 channels, all loads of a run in
// flight together.
__global__ __launch_bounds__(128) void latent_merge_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml,
                                                           const int* __restrict__ tiles, int heads,
                                                           const float* __restrict__ sink, uint16_t* __restrict__ out,
                                                           long o_row, long o_head, int splits, int rank, int window) {
  const int tile = blockIdx.x, slot = blockIdx.y;
  int row0, n_tok, head0, hcount;
  if (tiles) {
    const int* e = tiles + 6 * tile;
    if (e[0] < 0 || (window && tile_ranges(e[3], e[2], window, splits) == 1)) return;
    row0 = e[1], n_tok = e[2], head0 = e[4], hcount = e[5];
  } else {
    const int runs = (heads + 63) >> 6;
    row0 = tile / runs, n_tok = 1, head0 = (tile % runs) << 6, hcount = min(64, heads - head0);
  }
  if (slot >= n_tok * hcount) return;
  const long row = row0 + slot / hcount;
  const int head = head0 + slot % hcount;
  __shared__ float fac[MERGE_MAX];  // 0: nothing was seen in the split (its record may hold anything)
  const long rec0 = (long)tile * splits * 64 + slot;
  if (threadIdx.x < 64) {
    const int s = threadIdx.x;
    const float ms = s < splits ? ws_ml[2 * (rec0 + 64L * s)] : -INFINITY;
    const float ls = s < splits ? ws_ml[2 * (rec0 + 64L * s) + 1] : 0.f;
    float big = wave_reduce_max(ms);
    if (sink) big = fmaxf(big, sink[head]);
    const float f = ms == -INFINITY ? 0.f : __expf(ms - big);
    // (a sum that is no number counts whatever its factor: the maximum of a row of NaN is the lowest finite number, below any sink.  A NaN
    // denominator passes the comparison and every factor becomes one.)
    float den = wave_reduce_sum(f == 0.f && ls == ls ? 0.f : ls * f);
    if (sink) den += sink[head] == big ? 1.f : __expf(sink[head] - big);  // (1 also for an infinite sink, which leaves the entries nothing)
    fac[s] = den == 0.f ? 0.f : f / den;
  }
  __syncthreads();
  for (int d = threadIdx.x * 4; d < rank; d += 512) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < splits; s0 += 8) {
      f32x4 v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[i] = s0 + i < splits && fac[s0 + i] != 0.f
                   ? *reinterpret_cast<const f32x4*>(ws_o + (rec0 + 64L * (s0 + i)) * rank + d)
                   : (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float f = s0 + i < splits ? fac[s0 + i] : 0.f;
        if (f != 0.f) a += v[i] * f;
      }
    }
    u32x2 w = {pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3])};
    *reinterpret_cast<u32x2*>(out + row * o_row + head * o_head + d) = w;
  }
}

template <int RANK, int ROT, bool ROT_ONLY>
int launch(const void* q_lat, long ql_row, long ql_head, const void* q_rot, long qr_row, long qr_head,
           const void* cache, long page_stride, const int* block_tables, int bt_stride, const int* tiles,
           const int* positions, int n_tiles, int heads, const float* sink, void* out, long o_row, long o_head,
           float scale, int window, int splits, float* ws_o, float* ws_ml, int bucket, hipStream_t st) {
  // entries of 512 + 64 values: pages straight into LDS.  (A quarter of the channels has to be a block of eight 16-channel tiles, which
  // leaves 512; of the others, those of up to 256 values have three waves per SIMD in the kernel above to hide their staging.)
  static bool attr_set[2] = {false, false};
  auto ready = [](const void* kernel, int lds, bool* done) {
    if (!*done) *done = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
    return *done;
  };
  if constexpr (!ROT_ONLY && RANK == 512 && ROT == 64) {
    constexpr int PAGES = 2 * 64 * (RANK + ROT) * 2;
    if (!tiles && heads <= 32) {  // (a prefill tile fills its 64 slots)
      const auto kernel = latent_wide_kernel<RANK, ROT>;
      if (!ready((const void*)kernel, PAGES + 8 * 1024, &attr_set[1])) return -2;
      kernel<<<dim3(n_tiles, splits), dim3(512), PAGES + 8 * 1024, st>>>(
          (const uint16_t*)q_lat, ql_row, ql_head, (const uint16_t*)q_rot, qr_row, qr_head, (const uint16_t*)cache,
          page_stride, block_tables, bt_stride, positions, heads, sink, (uint16_t*)out, o_row, o_head, scale, window,
          splits, ws_o, ws_ml, bucket);
    } else {
      const auto kernel = latent_tile_kernel<RANK, ROT>;
      if (!ready((const void*)kernel, PAGES + 9 * 1024 + 256, &attr_set[0])) return -2;
      kernel<<<dim3(n_tiles, splits), dim3(256), PAGES + 9 * 1024 + 256, st>>>(
          (const uint16_t*)q_lat, ql_row, ql_head, (const uint16_t*)q_rot, qr_row, qr_head, (const uint16_t*)cache,
          page_stride, block_tables, bt_stride, tiles, positions, heads, sink, (uint16_t*)out, o_row, o_head, scale,
          window, splits, ws_o, ws_ml, bucket);
    }
  } else {
    constexpr int LDS = 64 * ((ROT_ONLY ? ROT : RANK + ROT) * 2 + 16) + RANK * (64 * 2 + 16);
    const auto kernel = latent_mfma_kernel<RANK, ROT, ROT_ONLY>;
    if (!ready((const void*)kernel, LDS, &attr_set[0])) return -2;
    kernel<<<dim3(n_tiles, splits), dim3(256), LDS, st>>>(
        (const uint16_t*)q_lat, ql_row, ql_head, (const uint16_t*)q_rot, qr_row, qr_head, (const uint16_t*)cache,
        page_stride, block_tables, bt_stride, tiles, positions, heads, sink, (uint16_t*)out, o_row, o_head, scale,
        window, splits, ws_o, ws_ml);
  }
  if (splits > 1)
    latent_merge_kernel<<<dim3(n_tiles, tiles ? 64 : min(heads, 64)), dim3(128), 0, st>>>(
        ws_o, ws_ml, tiles, heads, sink, (uint16_t*)out, o_row, o_head, splits, RANK, !ROT_ONLY && RANK == 512 && ROT == 64 ? window : 0);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace

// 1 when the matrix-core kernel tiles entries of this shape
// (latent entries: rank + rot; expanded per-head entries of a prefill: value | unrotated key | rotated key part,
// rank = value channels, rot = the key's channels)
#define LAT_SHAPES(X) \
  X(64, 32) X(64, 64) X(128, 32) X(128, 64) X(256, 32) X(256, 64) X(512, 32) X(512, 64) LAT_EXPANDED(X)
#define LAT_EXPANDED(X) X(32, 64) X(64, 96) X(64, 128) X(128, 128) X(128, 192)

VPSA_EXPORT int vpsa_latent_mfma_supported(int rank, int rot) {
#define LAT_IS(R, C) if (rank == R && rot == C) return 1;
  LAT_SHAPES(LAT_IS)
#undef LAT_IS
  return 0;
}

// 1 when it also has the shape as value | key entries (no q_lat)
VPSA_EXPORT int vpsa_latent_mfma_expanded(int rank, int rot) {
#define LAT_IS(R, C) if (rank == R && rot == C) return 1;
  LAT_EXPANDED(LAT_IS)
#undef LAT_IS
  return 0;
}

// tiles: int32 [n_tiles, 6] = (sequence, first query row, tokens, position of the first token, first head,
// heads per token) with tokens * heads <= 64 and sequence < 0 for an unused entry; null = decode rows
// (n_tiles = rows * ceil(heads / 64), positions [rows]).  Row and head strides in elements; every query
// and output vector 16-byte / 8-byte aligned.  q_lat null: see ROT_ONLY above.  window >= 1 (a query sees itself and the window - 1 entries before
// it; any window of at least the context length is plain causal attention).  splits > 1 needs ws_o [n_tiles * splits * 64 * rank] and
// ws_ml [n_tiles * splits * 64 * 2] floats.  bucket: the n_tiles that the choice of a decode row's key ranges goes by, where that is
// more than this launch's.
VPSA_EXPORT int vpsa_latent_attention_mfma(const void* q_lat, long ql_row, long ql_head, const void* q_rot,
                                           long qr_row, long qr_head, const void* cache, long page_stride,
                                           const int* block_tables, int bt_stride, const int* tiles,
                                           const int* positions, int n_tiles, int heads, const float* sink, void* out,
                                           long o_row, long o_head, int rank, int rot, float scale, int window,
                                           int splits, float* ws_o, float* ws_ml, int bucket, hipStream_t st) {
  if (n_tiles <= 0) return 0;
  if (bucket < n_tiles) bucket = n_tiles;
  if (window < 1 || splits > MERGE_MAX) return -1;
  if (splits < 1 || splits > 65535 || (splits > 1 && (!ws_o || !ws_ml)) || (!tiles && !positions)) return -1;
  if (((ql_row | ql_head | qr_row | qr_head) & 7) || ((o_row | o_head) & 3) || (page_stride & 7)) return -1;
#define LAT_ONLY(R, C)                                                                                              \
  if (!q_lat && rank == R && rot == C)                                                                              \
    return launch<R, C, true>(q_lat, ql_row, ql_head, q_rot, qr_row, qr_head, cache, page_stride, block_tables,      \
                              bt_stride, tiles, positions, n_tiles, heads, sink, out, o_row, o_head, scale, window,   \
                              splits, ws_o, ws_ml, bucket, st);
  LAT_EXPANDED(LAT_ONLY)
#undef LAT_ONLY
  if (!q_lat) return -1;
#define LAT_CASE(R, C)                                                                                              \
  if (rank == R && rot == C)                                                                                        \
    return launch<R, C, false>(q_lat, ql_row, ql_head, q_rot, qr_row, qr_head, cache, page_stride, block_tables, bt_stride, \
                        tiles, positions, n_tiles, heads, sink, out, o_row, o_head, scale, window, splits, ws_o,      \
                        ws_ml, bucket, st);
  LAT_SHAPES(LAT_CASE)
#undef LAT_CASE
  return -1;
}
