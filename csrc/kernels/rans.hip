// Entropy stage of the CacheGen-style KV codec on the GPU: interleaved rANS (range asymmetric
// numeral systems) over the int8 symbols that the quantiser (kvcache.hip) produces.
//
// Why rANS here: an adaptive binary range coder is a serial dependency chain per symbol (the
// host coder manages ~30 M symbols/s, 0.13 s per 8 MiB page); rANS with a static table is a
// handful of integer operations per symbol and thousands of independent streams can run side
// by side, so a page is coded in tens of microseconds next to the quantiser and the
// compressed bytes are what crosses PCIe.
//
// Layout.  The symbols of a page fall into contexts (one per layer: K and V deltas of a layer
// share statistics), ctx_len symbols each.  A context is cut into spc streams; stream j owns
// symbols j, j + spc, j + 2 spc, ... so that at every step the 64 lanes of a wave touch 64
// consecutive bytes (coalesced loads in the encoder, coalesced stores in the decoder).
// One thread codes one stream; a workgroup has 64 streams, so that a page's 16384 streams reach every CU: what bounds
// both directions is a stream's chain of dependent steps, not arithmetic or bytes.  The chain is kept short:
//   encoder  symbols and their table entries are read a batch of eight ahead, the division by a symbol's frequency is a
//            multiplication, coded bytes leave four at a time;
//   decoder  one table entry per step (symbol, frequency and offset within it), the streams' coded bytes staged in LDS and read
//            two at a time, at most two bytes a step without a loop.
// Page of a 32-layer cache with 8 KV heads (4.2 M symbols): coding loop 107 -> 25 us, with tables and gathering 150 -> 47; decoding
// 118 -> 24 us, 29 beside the copy of the next page (before: 64 workgroups, symbols and coded bytes read and written one at a time from memory, divisions).
// Per context: a 256-entry frequency table normalised to 2^12,
// built from a histogram of that very page (it travels with the blob: 512 B per context).
// Coder: 32-bit state, byte-wise renormalisation, lower bound 2^23.  The encoder runs over its
// symbols backwards and writes its bytes backwards into a private scratch slot, so the decoder
// reads forwards; the slots are then gathered into one dense byte string at the prefix sum of the sizes.
#include <string.h>

#include <atomic>

#include "common.h"
#include "host_copies.h"

#define RANS_BITS 12
#define RANS_M (1u << RANS_BITS)
#define RANS_LOW (1u << 23)
#define RANS_HIST_BLOCKS 64

// grid (blocks_per_ctx, n_ctx), block 256: a block's own histogram -> part[ctx][block][256].
__global__ __launch_bounds__(256) void rans_hist_kernel(const uint8_t* __restrict__ sym, uint32_t* __restrict__ part,
                                                        long ctx_len) {
  __shared__ uint32_t h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const uint8_t* p = sym + (long)blockIdx.y * ctx_len;
  const long stride = (long)gridDim.x * 256 * 4;
  for (long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4; i + 3 < ctx_len; i += stride) {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(p + i);
    atomicAdd(&h[w & 0xff], 1u);
    atomicAdd(&h[(w >> 8) & 0xff], 1u);
    atomicAdd(&h[(w >> 16) & 0xff], 1u);
    atomicAdd(&h[w >> 24], 1u);
  }
  __syncthreads();
  part[((long)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x] = h[threadIdx.x];
}

// What the encoder needs of a symbol of frequency f and start c: the published reciprocal form of the byte-wise rANS encoder
// (F. Giesen's ryg_rans, after R. Alverson, "Integer Division Using Reciprocals").  With s = ceil(log2 f) and m = ceil(2^(31 + s) / f) the
// quotient x / f of x < 2^31 is floor(x m / 2^(31 + s)): the product is off by less than x f / (f 2^(31 + s)) < 1 / f.  The new
// state (x / f) 4096 + x % f + c is x + (x / f) (4096 - f) + c.  f = 1 would need m = 2^31 and a shift to the left; m = 2^32 - 1
// gives x - 1 instead (x >= 1), and c + 4095 makes up for it.
// Words: m | f 2^19 | f 2^27 (or what no state reaches) | s - 1 (5 bits), 4096 - f (13), start (14).
__device__ __forceinline__ u32x4 rans_enc_entry(uint32_t f, uint32_t c) {
  if (f == 0) return (u32x4){0, 0, 0, 0};
  const uint32_t one = f << 19, two = f < 16 ? f << 27 : 0xffffffffu;
  if (f == 1) return (u32x4){0xffffffffu, one, two, 4095u << 5 | (c + 4095u) << 18};
  const uint32_t s = 32 - __clz(f - 1);
  const uint64_t m = ((1ull << (31 + s)) + f - 1) / f;
  return (u32x4){(uint32_t)m, one, two, (s - 1) | (RANS_M - f) << 5 | c << 18};
}

// grid n_ctx, block 256.  freq[s] = max(1, round(count * 4096 / total)) for symbols that occur,
// then the entry with the largest frequency (lowest index on ties) absorbs the rounding error
// so that the table sums to exactly 4096.  err[ctx]: that entry would drop below 1.
__global__ __launch_bounds__(256) void rans_normalize_kernel(const uint32_t* __restrict__ part, int parts,
                                                             uint16_t* __restrict__ freq, u32x4* __restrict__ table,
                                                             long ctx_len, int* __restrict__ err) {
  __shared__ int sf[256];
  __shared__ int si[256];
  __shared__ int scan[256];
  const int t = threadIdx.x;
  uint32_t c = 0;
#pragma unroll 8
  for (int i = 0; i < parts; ++i) c += part[((long)blockIdx.x * parts + i) * 256 + t];
  int f = 0;
  if (c) {
    f = (int)(((unsigned long long)c * RANS_M + (unsigned long long)(ctx_len / 2)) /
              (unsigned long long)ctx_len);
    if (f < 1) f = 1;
  }
  // sum and arg-max in one tree
  scan[t] = f;
  sf[t] = f;
  si[t] = t;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (t < off) {
      scan[t] += scan[t + off];
      const int a = sf[t], b = sf[t + off];
      if (b > a || (b == a && si[t + off] < si[t])) {
        sf[t] = b;
        si[t] = si[t + off];
      }
    }
    __syncthreads();
  }
  const int diff = (int)RANS_M - scan[0];
  const int imax = si[0];
  __syncthreads();
  if (t == imax) {
    f += diff;
    err[blockIdx.x] = f < 1;
    if (f < 1) f = 1;
  }
  // exclusive scan of the final frequencies
  scan[t] = f;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const int v = t >= off ? scan[t - off] : 0;
    __syncthreads();
    scan[t] += v;
    __syncthreads();
  }
  freq[blockIdx.x * 256 + t] = (uint16_t)f;
  table[blockIdx.x * 256 + t] = rans_enc_entry((uint32_t)f, (uint32_t)(scan[t] - f));
}

// grid (spc / 64, n_ctx), block 64.  slot = scratch bytes per stream (2 * symbols per stream, up to a multiple of 4).
// Symbols come through LDS and coded bytes leave through it, RANS_TILE symbols at a time: a load from memory in the loop would
// wait for the stores before it.  Every step writes the two bytes it could emit below the position and moves it by those that
// it does emit, without a branch; byte p of the 64 streams lies side by side, so that moving is all the address takes.
// The table entries of a batch are read while the batch before is coded.  (A word at a time gathered in registers and stored to
// the slot in the loop took 37 us a page, this 25.)
#define RANS_TILE 256
__global__ __launch_bounds__(64) void rans_encode_kernel(const uint8_t* __restrict__ sym, const u32x4* __restrict__ table,
                                                         uint8_t* __restrict__ scratch, uint32_t* __restrict__ states,
                                                         uint16_t* __restrict__ sizes, uint32_t* __restrict__ group_bytes,
                                                         long ctx_len, int spc, int slot) {
  constexpr int B = 8, WORDS = RANS_TILE / 2 + 1;  // two bytes a symbol, and a word begun in the tile before
  __shared__ u32x4 tab[256];
  __shared__ __attribute__((aligned(16))) uint8_t rows[RANS_TILE * 64];
  __shared__ uint8_t bytes[WORDS * 4 * 64];
  const int ctx = blockIdx.y, t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) tab[t + 64 * i] = table[ctx * 256 + t + 64 * i];
  const long gs = (long)ctx * spc + blockIdx.x * 64 + t;
  const uint8_t* p = sym + (long)ctx * ctx_len + blockIdx.x * 64;
  const bool wide = ((uintptr_t)sym & 15) == 0;  // every row of 64 streams starts a multiple of 64 further on
  uint32_t* out = reinterpret_cast<uint32_t*>(scratch + gs * slot + slot);  // the end of what is still to be written
  uint32_t x = RANS_LOW;
  int pos = WORDS * 4, done = 0;  // in the tile's bytes, counted down; bytes of earlier tiles
  for (int k1 = (int)(ctx_len / spc); k1 > 0; k1 -= RANS_TILE) {
    const int k0 = max(k1 - RANS_TILE, 0), n = k1 - k0;
    __syncthreads();
    if (wide) {
#pragma unroll
      for (int i = 0; i < RANS_TILE / 16; ++i) {
        const int r = i * 16 + (t >> 2);
        if (r < n) *reinterpret_cast<u32x4*>(rows + r * 64 + (t & 3) * 16) =
            *reinterpret_cast<const u32x4*>(p + (long)(k0 + r) * spc + (t & 3) * 16);
      }
    } else {
#pragma unroll 16
      for (int r = t >> 4; r < n; r += 4)
        *reinterpret_cast<uint32_t*>(rows + r * 64 + (t & 15) * 4) =
            *reinterpret_cast<const uint32_t*>(p + (long)(k0 + r) * spc + (t & 15) * 4);
    }
    __syncthreads();
    u32x4 nx[B];
#pragma unroll
    for (int i = 0; i < B; ++i) nx[i] = tab[rows[max(n - 1 - i, 0) * 64 + t]];
    int at = (pos - 2) * 64 + t;
    for (int k = n - 1; k >= 0; k -= B) {
      u32x4 e[B];
#pragma unroll
      for (int i = 0; i < B; ++i) e[i] = nx[i];
#pragma unroll
      for (int i = 0; i < B; ++i) nx[i] = tab[rows[max(k - B - i, 0) * 64 + t]];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        if (k - i < 0) break;
        const uint32_t w = e[i][3];
        bytes[at + 64] = (uint8_t)x;
        bytes[at] = (uint8_t)(x >> 8);
        const int n8 = (x >= e[i][1] ? 8 : 0) + (x >= e[i][2] ? 8 : 0);  // x < 2^31 and f 2^19 >= 2^19: never more than two
        x >>= n8;
        at -= n8 * 8;
        // x < f 2^19 now: the quotient has 19 bits
        x += __umul24(__umulhi(x, e[i][0]) >> (w & 31), (w >> 5) & 0x1fff) + (w >> 18);
      }
    }
    pos = ((at - t) >> 6) + 2;
    // whole words to the slot, the word begun goes on in the next tile
    const bool last = k0 == 0;
    const int w_lo = last ? pos >> 2 : (pos + 3) >> 2, n_w = WORDS - w_lo;
#pragma unroll 8
    for (int w = WORDS - 1; w >= w_lo; --w) {
      const uint8_t* b = bytes + w * 256 + t;
      out[w - WORDS] = b[0] | b[64] << 8 | b[128] << 16 | (uint32_t)b[192] << 24;
    }
    if (last) {
      done += WORDS * 4 - pos;
    } else {
      done += n_w * 4;
      out -= n_w;
      const int part = w_lo * 4 - pos;  // bytes of a begun word
      if (part)
        for (int i = 0; i < 4; ++i) bytes[((WORDS - 1) * 4 + i) * 64 + t] = bytes[((w_lo - 1) * 4 + i) * 64 + t];
      pos = WORDS * 4 - part;
    }
  }
  states[gs] = x;
  sizes[gs] = (uint16_t)done;
  int sum = done;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if (t == 0) group_bytes[ctx * gridDim.x + blockIdx.x] = (uint32_t)sum;
}

// Exclusive prefix of one value per lane.
__device__ __forceinline__ int wave_before(int v) {
  const int lane = threadIdx.x & 63;
  int incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int u = __shfl_up(incl, off, 64);
    if (lane >= off) incl += u;
  }
  return incl - v;
}

// Block 256, one workgroup per 64 streams: their bytes from the scratch slots to the dense output.  The group's place is the sum
// of the groups before it (a few hundred values: cheaper than a scan of its own).  The last workgroup leaves
// meta = coded bytes | contexts whose table could not be normalised.
__global__ __launch_bounds__(256) void rans_pack_kernel(const uint8_t* __restrict__ scratch,
                                                        const uint16_t* __restrict__ sizes,
                                                        const uint32_t* __restrict__ group_bytes,
                                                        uint8_t* __restrict__ out, int slot, const int* __restrict__ err,
                                                        int n_ctx, long* __restrict__ meta) {
  __shared__ long part[4];
  __shared__ int at[64], len[64];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, group = blockIdx.x;
  long sum = 0;
  for (int i = t; i < group; i += 256) sum += group_bytes[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if (lane == 0) part[wave] = sum;
  if (wave == 0) {
    const int n = sizes[(long)group * 64 + lane];
    at[lane] = wave_before(n);
    len[lane] = n;
  }
  __syncthreads();
  const long base = part[0] + part[1] + part[2] + part[3];
#pragma unroll 8
  for (int i = 0; i < 16; ++i) {
    const int s = wave * 16 + i, n = len[s];
    const uint8_t* src = scratch + ((long)group * 64 + s) * slot + (slot - n);
    uint8_t* dst = out + base + at[s];
    uint8_t v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = lane + 64 * q < n ? src[lane + 64 * q] : 0;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (lane + 64 * q < n) dst[lane + 64 * q] = v[q];
    for (int q = lane + 256; q < n; q += 64) dst[q] = src[q];
  }
  if (group == (int)gridDim.x - 1) {
    int bad = 0;
    for (int i = t; i < n_ctx; i += 256) bad += err[i];
    bad = __syncthreads_count(bad != 0);
    if (t == 0) {
      meta[0] = base + group_bytes[group];
      meta[1] = bad;
    }
  }
}

// A stream's symbols; `pair` gives the two bytes at a place of the wave's coded bytes, the first one higher, from LDS or (streams too
// long for it) from memory.  Two copies of the loop: one that may load from memory waits for its own stores at every step.  DIR: which way the
// places run.  What bounds it is the chain from a state to the next, and every instruction of a wave that has its SIMD to itself stands in
// it: an entry of two words, f | symbol << 24 and the offset, makes the new state one instruction (a 24-bit product takes the first as it is),
// the bytes come in by one funnel shift, a row's place is a scalar, places are bounded once in 16 steps.  15 instructions a step instead
// of 27; left alone, the compiler moves the second read behind a branch where no byte is due, and the shift behind another: 35 us a page
// instead of 24.
template <int DIR, typename F>
__device__ __forceinline__ void rans_decode_stream(F pair, int at, uint32_t x, const u32x2* tab, uint8_t* __restrict__ out, int lane, int len,
                                                   int spc) {
  auto step = [&](__amdgpu_buffer_rsrc_t to, uint32_t row) {  // (a row's place is a scalar beside the lane's)
    const uint32_t q = x >> RANS_BITS;
    u32x2 e = tab[x & (RANS_M - 1)];
    uint32_t p = pair(at);
    asm volatile("" : "+v"(p), "+v"(e));  // both reads are under way before anything of either is used (not behind a branch where no byte is due)
    x = __umul24(e[0], q) + e[1];  // (a state the encoder leaves has 19 bits in q)
    const bool one = x < RANS_LOW, two = x < (RANS_LOW >> 8);
    uint32_t in = __builtin_amdgcn_alignbit(x, p << 16, two ? 16 : 24);
    asm volatile("" : "+v"(in));
    x = one ? in : x;
    at += one ? DIR : 0;
    at += two ? DIR : 0;
    __builtin_amdgcn_raw_buffer_store_b8((uint8_t)(e[0] >> 24), to, lane, row, 0);
  };
  constexpr int RUN = 16;
  for (; len >= RUN; len -= RUN, out += (long)RUN * spc) {
    if (DIR < 0) at = max(at, 2 * RUN);  // (an undamaged stream's places are past DECODE_SLACK)
    const auto to = __builtin_amdgcn_make_buffer_rsrc(out, 0, -1, 0x00020000);
#pragma unroll
    for (int k = 0; k < RUN; ++k) step(to, (uint32_t)k * (uint32_t)spc);
  }
  if (DIR < 0) at = max(at, 2 * RUN);
  for (; len > 0; --len, out += spc) step(__builtin_amdgcn_make_buffer_rsrc(out, 0, -1, 0x00020000), 0);
}

#define DECODE_THREADS 256
#define DECODE_SLACK 64  // bytes below any that a stream reads: places are bounded once in so many steps that they move by less
// grid (spc / 64, n_ctx).  The workgroup makes the context's 4096 table entries and brings in the coded bytes of its 64 streams, which lie side
// by side behind those of all streams before them; then every wave decodes 16 streams, a lane each.  The bytes are staged when they fit (a stream's
// share is 320, a symbol rarely takes one), last byte first, so that a pair is one read.  coded_len bounds every read (a damaged blob
// decodes to garbage, never out of bounds: a damaged table gives entries of some symbol, every field masked to its width), and a step takes
// at most two bytes whatever the state is.  A page of 16384 streams of 256 symbols: tables in a launch of their own 4 us and one wave for all 64
// streams 33; in one launch 32 with one wave (which waited for memory ten times in a row before its first step), 28 with four (fewer lanes meet
// in a bank of LDS; eight waves 32), 24 with the loop above.  (53 KB of LDS: three a CU; with two, 80 contexts took two rounds, 49.6 us for 39.3.)
__global__ __launch_bounds__(DECODE_THREADS) void rans_decode_kernel(const uint8_t* __restrict__ coded, long coded_len, const uint16_t* __restrict__ freq,
                                                          const uint16_t* __restrict__ sizes, const uint32_t* __restrict__ states,
                                                          uint8_t* __restrict__ sym, long ctx_len, int spc) {
  typedef uint16_t any_u16 __attribute__((aligned(1)));
  constexpr int LDS_WORDS = 64 * 80 + DECODE_SLACK / 4, LDS_BYTES = LDS_WORDS * 4;
  __shared__ __attribute__((aligned(16))) u32x2 tab[RANS_M];
  __shared__ __attribute__((aligned(16))) uint32_t bytes[LDS_WORDS];
  constexpr int NT = DECODE_THREADS, WAVES = NT / 64, EACH = 64 / WAVES;  // streams of a wave
  __shared__ uint32_t in_wave[4];
  __shared__ long part[WAVES];
  uint32_t *const cum = bytes, *const fr = bytes + 256;  // (until the bytes come)
  const int ctx = blockIdx.y, t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const uint32_t f = t < 256 ? freq[ctx * 256 + t] : 0;
  const long stream0 = (long)ctx * spc + blockIdx.x * 64;
  const int n = sizes[stream0 + lane];  // (every wave: the bytes of the workgroup's streams)
  const uint32_t x0 = states[stream0 + lane];
  // bytes before the workgroup's first stream
  long first = 0;
  if (((uintptr_t)sizes & 15) == 0) {
    const u32x4* const sz = reinterpret_cast<const u32x4*>(sizes);
    const long pieces = stream0 / 8;  // (whole: stream0 is a multiple of 64)
    for (long i0 = 0; i0 < pieces; i0 += NT * 8) {
      u32x4 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const long i = i0 + t + NT * j;
        v[j] = sz[i < pieces ? i : 0];
        if (i >= pieces) v[j] = (u32x4){0, 0, 0, 0};
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int w = 0; w < 4; ++w) first += (v[j][w] & 0xffff) + (v[j][w] >> 16);
    }
  } else {
    for (long i = t; i < stream0; i += NT) first += sizes[i];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) first += __shfl_xor(first, off, 64);
  const int cum0 = wave_before((int)f), before = wave_before(n), all = __shfl(before + n, 63, 64);
  if (t < 256) fr[t] = f;
  if (lane == 63) {
    if (wave < 4) in_wave[wave] = (uint32_t)cum0 + f;
    part[wave] = first;
  }
  __syncthreads();
  if (t < 256) {
    uint32_t c = (uint32_t)cum0;
    for (int w = 0; w < wave; ++w) c += in_wave[w];
    cum[t] = c;
  }
  first = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) first += part[w];
  // words of the coded bytes, counted from the aligned word that holds byte 0
  const int lead = (int)((uintptr_t)coded & 3);
  const uint32_t* cw = reinterpret_cast<const uint32_t*>(coded - lead);
  const long n_words = (coded_len + lead + 3) >> 2;
  const long w0 = (first + lead) >> 2, w1 = min((first + all + lead + 3) >> 2, n_words);
  const bool staged = w1 - w0 < LDS_WORDS - DECODE_SLACK / 4;
  const int held = staged ? max((int)(w1 - w0), 0) : 0;
  constexpr int AHEAD = 3584 / NT;  // words that a thread asks for before it waits: a page's usual share at once
  uint32_t v[AHEAD];
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) v[j] = t + NT * j < held ? cw[w0 + t + NT * j] : 0u;
  __syncthreads();
  // the last symbol that starts at or before the slot (those before it with the same start do not occur)
#pragma unroll 4
  for (int i = 0; i < (int)RANS_M / NT; ++i) {
    const uint32_t slot = t + NT * i;
    int s = 0;
#pragma unroll
    for (int step = 128; step > 0; step >>= 1)
      if (cum[s + step] <= slot) s += step;
    tab[slot] = (u32x2){((fr[s] - 1) & 0xfff) + 1 | (uint32_t)s << 24, (slot - cum[s]) & 0xfff};
  }
  if (held > LDS_WORDS - 512) __syncthreads();  // (the same for all threads; else nobody writes where the table was made from)
#pragma unroll
  for (int j = 0; j < AHEAD; ++j)
    if (t + NT * j < held) bytes[LDS_WORDS - 1 - (t + NT * j)] = __builtin_bswap32(v[j]);
  for (int i = t + NT * AHEAD; i < held; i += NT) bytes[LDS_WORDS - 1 - i] = __builtin_bswap32(cw[w0 + i]);
  __syncthreads();
  uint8_t* out = sym + (long)ctx * ctx_len + blockIdx.x * 64 + EACH * wave;
  const int len = (int)(ctx_len / spc);
  const uint32_t rp = __shfl((uint32_t)((first + lead) & 3) + (uint32_t)before, (EACH * wave + lane) & 63, 64);
  const uint32_t x = __shfl(x0, (EACH * wave + lane) & 63, 64);
  if (lane >= EACH) return;
  if (staged)
    rans_decode_stream<-1>([&](int i) {
      return (uint32_t)*reinterpret_cast<const any_u16*>(reinterpret_cast<const char*>(bytes) + i);
    }, LDS_BYTES - 2 - (int)rp, x, tab, out, lane, len, spc);
  else
    rans_decode_stream<1>([&](uint32_t i) {
      const uint32_t lo = w0 + (i >> 2) < n_words ? cw[w0 + (i >> 2)] : 0u, hi = w0 + (i >> 2) + 1 < n_words ? cw[w0 + (i >> 2) + 1] : 0u;
      const uint32_t b = __builtin_amdgcn_alignbyte(hi, lo, i & 3);  // the next byte lowest
      return (b & 0xff) << 8 | ((b >> 8) & 0xff);
    }, (int)rp, x, tab, out, lane, len, spc);
}

// More workgroups than the chip holds (three a CU, by their LDS) stand in each other's way: four waves for 64 streams are four times the instructions, every one
// makes its context's table and sums the sizes before it.  Those calls take two launches, one for tables and sums, one of a wave for 64
// streams, four of them a CU: 80 contexts of 512 streams of 256 symbols 39.3 us by the kernel above, 41.3 by these, 126 contexts 61.0 / 50.2; of 16 symbols 17.1 / 14.6, 512
// contexts 70.5 / 43.3, 2048 contexts 634 / 168.
constexpr long DECODE_TOGETHER = 3 * 256;
// grid n_ctx, block 1024: a context's 4096 decoder entries, symbol | (freq - 1) << 8 | (slot - cum) << 20, and the bytes of its
// streams.  (A damaged table gives entries of some symbol; every field is masked to its width.)
__global__ __launch_bounds__(1024) void rans_decode_tables_kernel(const uint16_t* __restrict__ freq, uint32_t* __restrict__ table,
                                                                  const uint16_t* __restrict__ sizes, int spc,
                                                                  long* __restrict__ ctx_bytes) {
  __shared__ uint32_t cum[256], fr[256];
  __shared__ long part[16];
  const int t = threadIdx.x;
  uint32_t f = 0;
  if (t < 256) {
    f = freq[blockIdx.x * 256 + t];
    fr[t] = f;
  }
  long sum = 0;
  for (int i = t; i < spc; i += 1024) sum += sizes[(long)blockIdx.x * spc + i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if ((t & 63) == 0) part[t >> 6] = sum;
  const int before = wave_before((int)f);  // (of the wave's 64 symbols)
  if (t < 256) cum[t] = before;
  __syncthreads();
  if (t == 0) {
    long s = 0;
    for (int w = 0; w < 16; ++w) s += part[w];
    ctx_bytes[blockIdx.x] = s;
  }
  if (t < 256) {
    uint32_t c = cum[t];
    for (int w = 0; w < (t >> 6); ++w) c += cum[w * 64 + 63] + fr[w * 64 + 63];
    f = c;
  }
  __syncthreads();
  if (t < 256) cum[t] = f;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t slot = t + 1024 * i;
    int s = 0;  // the last symbol that starts at or before the slot (those before it with the same start do not occur)
#pragma unroll
    for (int step = 128; step > 0; step >>= 1)
      if (cum[s + step] <= slot) s += step;
    table[blockIdx.x * (long)RANS_M + slot] = (uint32_t)s | ((fr[s] - 1) & 0xfff) << 8 | ((slot - cum[s]) & 0xfff) << 20;
  }
}

// A stream's symbols; `word` reads words i and i + 1 of the wave's coded bytes, from LDS or (streams too long for it) from memory.
// Two copies of the loop: one that may load from memory waits for its own stores at every step.  The words around the next
// byte are read in the same wait as the state's table entry.
template <typename F>
__device__ __forceinline__ void rans_decode_many_stream(F word, uint32_t rp, uint32_t x, const uint32_t* tab,
                                                   uint8_t* __restrict__ out, int len, int spc) {
  for (int k = 0; k < len; ++k) {
    const uint32_t e = tab[x & (RANS_M - 1)];
    const uint64_t w = word(rp >> 2);
    const uint32_t lo = (uint32_t)w, hi = (uint32_t)(w >> 32);
    *out = (uint8_t)e;
    out += spc;
    const uint32_t q = x >> RANS_BITS;  // 20 bits (19 of a state the encoder leaves)
    x = __umul24((e >> 8) & 0xfff, q) + (q + (e >> 20));
    const uint32_t b = __builtin_amdgcn_alignbyte(hi, lo, rp & 3);  // the next byte lowest
    const uint32_t x1 = (x << 8) | (b & 0xff), x2 = (x1 << 8) | ((b >> 8) & 0xff);
    const bool one = x < RANS_LOW, two = x < (RANS_LOW >> 8);
    x = two ? x2 : one ? x1 : x;
    rp += one + two;
  }
}

// grid (spc / 64, n_ctx), block 64.  The wave's coded bytes lie side by side, behind those of the contexts and of the context's
// streams before it; they are staged when they fit (a stream's share of LDS_WORDS is 320 bytes, a symbol rarely takes one).
// coded_len bounds every read (a damaged blob decodes to garbage, never out of bounds), and a step takes at most two bytes
// whatever the state is.
__global__ __launch_bounds__(64) void rans_decode_many_kernel(const uint8_t* __restrict__ coded, long coded_len,
                                                         const long* __restrict__ ctx_bytes, const uint16_t* __restrict__ sizes,
                                                         const uint32_t* __restrict__ states, const uint32_t* __restrict__ table,
                                                         uint8_t* __restrict__ sym, long ctx_len, int spc) {
  constexpr int LDS_WORDS = 64 * 80;
  __shared__ __attribute__((aligned(16))) uint32_t tab[RANS_M];
  __shared__ uint32_t bytes[LDS_WORDS];
  const int ctx = blockIdx.y, t = threadIdx.x;
  const u32x4* tp = reinterpret_cast<const u32x4*>(table + (long)ctx * RANS_M);
#pragma unroll
  for (int i = 0; i < RANS_M / 256; ++i) reinterpret_cast<u32x4*>(tab)[t + 64 * i] = tp[t + 64 * i];
  const uint16_t* sz = sizes + (long)ctx * spc;
  long first = 0;  // byte of the wave's first stream
  for (int i = t; i < ctx; i += 64) first += ctx_bytes[i];
  for (int i = t; i < (int)blockIdx.x * 64; i += 64) first += sz[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) first += __shfl_xor(first, off, 64);
  const int n = sz[blockIdx.x * 64 + t], before = wave_before(n), all = __shfl(before + n, 63, 64);
  const uint32_t x = states[(long)ctx * spc + blockIdx.x * 64 + t];
  // words of the coded bytes, counted from the aligned word that holds byte 0
  const int lead = (int)((uintptr_t)coded & 3);
  const uint32_t* cw = reinterpret_cast<const uint32_t*>(coded - lead);
  const long n_words = (coded_len + lead + 3) >> 2;
  const long w0 = (first + lead) >> 2, w1 = min((first + all + lead + 3) >> 2, n_words);
  const bool staged = w1 - w0 < LDS_WORDS;
  const int held = staged ? max((int)(w1 - w0), 0) : 0;
#pragma unroll 8
  for (int i = t; i < held; i += 64) bytes[i] = cw[w0 + i];
  __syncthreads();
  uint8_t* out = sym + (long)ctx * ctx_len + blockIdx.x * 64 + t;
  const int len = (int)(ctx_len / spc);
  const uint32_t rp = (uint32_t)((first + lead) & 3) + (uint32_t)before;
  if (staged)
    rans_decode_many_stream([&](uint32_t i) {
      const uint32_t at = min(i, (uint32_t)LDS_WORDS - 2);
      return (uint64_t)bytes[at + 1] << 32 | bytes[at];
    }, rp, x, tab, out, len, spc);
  else
    rans_decode_many_stream([&](uint32_t i) {
      const uint32_t lo = w0 + i < n_words ? cw[w0 + i] : 0u, hi = w0 + i + 1 < n_words ? cw[w0 + i + 1] : 0u;
      return (uint64_t)hi << 32 | lo;
    }, rp, x, tab, out, len, spc);
}

static bool rans_shape_ok(long n, int n_ctx, int spc) {
  if (n <= 0 || n_ctx <= 0 || spc <= 0 || spc % 256 != 0 || n % n_ctx != 0) return false;
  const long ctx_len = n / n_ctx;
  if (ctx_len % spc != 0 || ctx_len % 4 != 0) return false;
  const long len = ctx_len / spc;
  return len >= 1 && 2 * len <= 65535;
}

static int rans_slot(long n, int n_ctx, int spc) { return (int)((2 * (n / n_ctx / spc) + 3) & ~3L); }

// Bytes of the encoder's workspace (0: the shape is not taken): histograms | table | errors | bytes per 64 streams | slots.
VPSA_EXPORT long vpsa_rans_workspace(long n, int n_ctx, int spc) {
  if (!rans_shape_ok(n, n_ctx, spc)) return 0;
  return (long)n_ctx * (RANS_HIST_BLOCKS * 1024 + 4096 + 16) + (long)n_ctx * spc * (4 + rans_slot(n, n_ctx, spc));
}

// Histogram -> table -> per-stream coding -> dense bytes.  freq u16 [n_ctx * 256], states u32 and sizes u16 [n_ctx * spc], coded
// with room for 2 n bytes, meta i64 [2] = coded bytes, contexts that could not be normalised; ws 16-byte aligned.
VPSA_EXPORT int vpsa_rans_encode(const void* sym, long n, int n_ctx, int spc, void* ws, void* freq, void* states, void* sizes,
                                 void* coded, long* meta, hipStream_t stream) {
  if (!rans_shape_ok(n, n_ctx, spc)) return -1;
  const long ctx_len = n / n_ctx, groups = (long)n_ctx * spc / 64;
  const int slot = rans_slot(n, n_ctx, spc);
  const long per_block = (ctx_len / 4 + 255) / 256;
  const int hb = (int)(per_block > RANS_HIST_BLOCKS ? RANS_HIST_BLOCKS : per_block);
  uint32_t* part = (uint32_t*)ws;
  u32x4* table = (u32x4*)((char*)ws + (long)n_ctx * RANS_HIST_BLOCKS * 1024);
  int* err = (int*)(table + (long)n_ctx * 256);
  uint32_t* group_bytes = (uint32_t*)((char*)err + (long)n_ctx * 16);
  uint8_t* scratch = (uint8_t*)(group_bytes + (long)n_ctx * spc);
  hipLaunchKernelGGL(rans_hist_kernel, dim3(hb, n_ctx), dim3(256), 0, stream, (const uint8_t*)sym, part, ctx_len);
  hipLaunchKernelGGL(rans_normalize_kernel, dim3(n_ctx), dim3(256), 0, stream, part, hb, (uint16_t*)freq, table, ctx_len, err);
  hipLaunchKernelGGL(rans_encode_kernel, dim3(spc / 64, n_ctx), dim3(64), 0, stream, (const uint8_t*)sym, table, scratch,
                     (uint32_t*)states, (uint16_t*)sizes, group_bytes, ctx_len, spc, slot);
  hipLaunchKernelGGL(rans_pack_kernel, dim3((unsigned)groups), dim3(256), 0, stream, scratch, (const uint16_t*)sizes, group_bytes,
                     (uint8_t*)coded, slot, err, n_ctx, meta);
  return 0;
}

// Bytes of the decoder's workspace (calls of many contexts: tables | bytes per context), 0: none.
VPSA_EXPORT long vpsa_rans_decode_workspace(long n, int n_ctx, int spc) {
  return rans_shape_ok(n, n_ctx, spc) && (long)n_ctx * spc / 64 > DECODE_TOGETHER ? (long)n_ctx * (RANS_M * 4 + 8) : 0;
}

// Only freq, states and sizes travel beside the coded bytes; ws 16-byte aligned, or null where none is needed.
VPSA_EXPORT int vpsa_rans_decode(const void* coded, long coded_len, const void* states, const void* freq, const void* sizes, void* ws, void* sym,
                                 long n, int n_ctx, int spc, hipStream_t stream) {
  if (!rans_shape_ok(n, n_ctx, spc)) return -1;
  const long ctx_len = n / n_ctx;
  if (vpsa_rans_decode_workspace(n, n_ctx, spc) == 0)
    return launched(rans_decode_kernel, dim3(spc / 64, n_ctx), DECODE_THREADS, 0, stream, (const uint8_t*)coded, coded_len, (const uint16_t*)freq,
                    (const uint16_t*)sizes, (const uint32_t*)states, (uint8_t*)sym, ctx_len, spc);
  if (ws == nullptr || ((uintptr_t)ws & 15)) return -1;
  uint32_t* table = (uint32_t*)ws;
  long* ctx_bytes = (long*)(table + (long)n_ctx * RANS_M);
  const int rc = launched(rans_decode_tables_kernel, dim3(n_ctx), 1024, 0, stream, (const uint16_t*)freq, table, (const uint16_t*)sizes, spc, ctx_bytes);
  return rc ? rc : launched(rans_decode_many_kernel, dim3(spc / 64, n_ctx), 64, 0, stream, (const uint8_t*)coded, coded_len, ctx_bytes,
                            (const uint16_t*)sizes, (const uint32_t*)states, table, (uint8_t*)sym, ctx_len, spc);
}

// ---------------------------------------------------------------------------------
// What a KV page's stored form needs of the host in one call each way.  A call spends its host time beside the copy of 3.5 MB (45 us from
// cache, 60 to 90 from memory) on launches, buffers and views: coming back a page took 178 us of host time for 117 of kernels and copies.
extern "C" int vpsa_cachegen_decode(const void* symbols, const float* scales, void* staging, long n_elems, long unit_elems,
                                    hipStream_t stream);

struct PageParts {
  char *scales, *freq, *states, *sizes, *coded;
};
static PageParts page_parts(void* body, long n, int n_ctx, int spc) {
  char* p = (char*)body;
  const long groups = n / 64 * 4, freq = 512L * n_ctx, streams = (long)n_ctx * spc;
  return {p, p + groups, p + groups + freq, p + groups + freq + 4 * streams, p + groups + freq + 6 * streams};
}
static long page_symbols(long n) { return (n + 255) & ~255L; }

// A page's parts, scales fp32 [n / 64] | freq | states | sizes | coded bytes, lie side by side in `body` on the device.
// Bytes of the workspace of vpsa_page_decode (symbols | the coder's), 0: the shape is not taken.
VPSA_EXPORT long vpsa_page_workspace(long n, int n_ctx, int spc) {
  return rans_shape_ok(n, n_ctx, spc) && n % 64 == 0 ? page_symbols(n) + vpsa_rans_decode_workspace(n, n_ctx, spc) : 0;
}

VPSA_EXPORT int vpsa_copy_parts(long size) { return copy_parts(size); }

// `size` bytes from the device to `to` by way of a pinned buffer.  Over on return.  (Four parts, each leaving the buffer while the next is on
// its way, were no faster, 158 us a page against 162, and on the way back they cost the device 50 us a page: a copy's start is 10 to 15.
// A kernel that stores the coded bytes into pinned memory right behind the coder spares the host one of its two waits, 201 us a page against 213 to 220,
// but it gathers them in LDS, and its workgroups lie on the CUs as long as the link takes: products whose workgroups want most of a CU's LDS find no
// place beside them.  A decode step of 12 sequences on another stream took 2830 us beside one thread that encodes pages and 4170 to 4520 beside two,
// with the runtime's copy, which holds no LDS, 2100 to 2160 and 2350; 1920 by itself.)
VPSA_EXPORT int vpsa_fetch(const void* from, void* pinned, void* to, long size, hipStream_t stream) {
  const bool sent = hipMemcpyAsync(pinned, from, size, hipMemcpyDeviceToHost, stream) == hipSuccess;
  if (hipStreamSynchronize(stream) != hipSuccess || !sent) return -3;
  copy_in_parts((char*)to, (const char*)pinned, size);
  return 0;
}

// The stream of the current device that pages' bytes come in on, this library's own: a stream out of torch's pool may be handed to someone
// else, who queues on it or captures it.  Made on the first call, one a device, and kept; null where none can be had.
VPSA_EXPORT hipStream_t vpsa_page_copy_stream() {
  static std::atomic<hipStream_t> streams[64];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return nullptr;
  hipStream_t mine = streams[device].load(std::memory_order_acquire);
  if (mine != nullptr) return mine;
  hipStream_t made = nullptr;
  if (hipStreamCreateWithFlags(&made, hipStreamNonBlocking) != hipSuccess) return nullptr;
  if (streams[device].compare_exchange_strong(mine, made)) return made;
  (void)hipStreamDestroy(made);
  return mine;
}

// The copy of a page on that stream, so that it runs beside the kernels of the page before it (3.5 MB: 67 us of copy, 30 of kernels by themselves and
// 34 beside it); `stream` waits for it, and it for nothing but the copies before it: all callers share it.  fresh: `body` is new to the caller, and what
// `stream` still has to do may touch its memory; the copy then stands in `stream`, where nobody else waits for it.  Below 2 MB the
// events cost the host, which is behind there anyway, what the copy takes (a page of 1.5 MB of many, one stream / two: 87 / 91 us; of 3.5 MB
// 143 / 115, of 8 MB 238 / 196; with helpers that wait).
constexpr long COPY_AHEAD = 2 << 20;
static int page_copy(void* body, const void* pinned, long size, int fresh, hipStream_t stream) {
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  const bool ahead = !fresh && size >= COPY_AHEAD && hipStreamIsCapturing(stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone;
  const hipStream_t copies = ahead ? vpsa_page_copy_stream() : nullptr;
  if (copies == nullptr) return hipMemcpyAsync(body, pinned, size, hipMemcpyHostToDevice, stream) == hipSuccess ? 0 : -3;
  hipEvent_t event;
  if (hipEventCreateWithFlags(&event, hipEventDisableTiming) != hipSuccess) return -3;
  const bool sent = hipMemcpyAsync(body, pinned, size, hipMemcpyHostToDevice, copies) == hipSuccess;
  const bool ok = sent && hipEventRecord(event, copies) == hipSuccess && hipStreamWaitEvent(stream, event, 0) == hipSuccess;
  if (sent && !ok) (void)hipStreamSynchronize(copies);  // nothing may read the buffer that the caller does not know of
  (void)hipEventDestroy(event);  // (released when it has passed)
  return ok ? 0 : -3;
}

// `size` host bytes at `from` (a page's parts) through the pinned buffer into `body`, then symbols and values.  Not waited
// for: pinned buffer and body are in use until `stream` has come past this call.
VPSA_EXPORT int vpsa_page_decode(const void* from, void* pinned, void* body, long size, long n, int n_ctx, int spc, long unit_elems, void* ws,
                                 void* out, int fresh, hipStream_t stream) {
  if (vpsa_page_workspace(n, n_ctx, spc) <= 0) return -1;
  const PageParts at = page_parts(body, n, n_ctx, spc);
  const long coded = size - (at.coded - (char*)body);
  if (coded < 0) return -1;
  copy_in_parts((char*)pinned, (const char*)from, size);
  if (const int rc = page_copy(body, pinned, size, fresh, stream)) return rc;
  const int rc = vpsa_rans_decode(at.coded, coded, at.states, at.freq, at.sizes, (char*)ws + page_symbols(n), ws, n, n_ctx, spc, stream);
  return rc ? rc : vpsa_cachegen_decode(ws, (const float*)at.scales, out, n, unit_elems, stream);
}
