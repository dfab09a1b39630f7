"""The entropy decoder's kernel built for the host, a thread for every lane, under AddressSanitizer: whole pages come back, and damaged sizes, tables,
states and coded bytes decode to something without a read or write outside of what the call was given."""

import os
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from vllm_production_stack_amd.ops import reference as ref

ROOT = Path(__file__).resolve().parents[1]
HOST = r"""
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <algorithm>
#include <barrier>
#include <thread>
#include <vector>
using std::max;
using std::min;
#define RANS_BITS 12
#define RANS_M (1u << RANS_BITS)
#define RANS_LOW (1u << 23)
#define __global__
#define __device__
#define __forceinline__ inline
#define __launch_bounds__(n)
#define __shared__ static
#define asm
#define volatile(...)
typedef uint32_t u32x2 __attribute__((vector_size(8)));
typedef uint32_t u32x4 __attribute__((vector_size(16)));
struct Place { int x, y; };
static thread_local Place threadIdx;
static Place blockIdx;
static std::barrier<>* everyone;
static std::barrier<>* of_wave[4];
static long lanes[4][64];
static void __syncthreads() { everyone->arrive_and_wait(); }
template <typename T>
static T __shfl(T v, int from, int) {
  const int wave = threadIdx.x >> 6;
  lanes[wave][threadIdx.x & 63] = (long)v;
  of_wave[wave]->arrive_and_wait();
  const T got = (T)lanes[wave][from & 63];
  of_wave[wave]->arrive_and_wait();
  return got;
}
template <typename T>
static T __shfl_xor(T v, int off, int) { return __shfl(v, (threadIdx.x & 63) ^ off, 64); }
static int wave_before(int v) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  lanes[wave][lane] = v;
  of_wave[wave]->arrive_and_wait();
  int sum = 0;
  for (int i = 0; i < lane; ++i) sum += (int)lanes[wave][i];
  of_wave[wave]->arrive_and_wait();
  return sum;
}
static uint32_t __umul24(uint32_t a, uint32_t b) { return (a & 0xffffff) * (b & 0xffffff); }
struct Out { uint8_t* at; };
#define __amdgpu_buffer_rsrc_t Out
#define __builtin_amdgcn_make_buffer_rsrc(p, stride, size, flags) Out{p}
#define __builtin_amdgcn_raw_buffer_store_b8(v, to, lane, row, policy) ((to).at[(uint32_t)(lane) + (row)] = (v))
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_alignbit(hi, lo, s) ((uint32_t)(((uint64_t)(hi) << 32 | (lo)) >> ((s) & 31)))
#define __builtin_amdgcn_alignbyte(hi, lo, s) ((uint32_t)(((uint64_t)(hi) << 32 | (lo)) >> (8 * ((s) & 3))))
"""
MAIN = r"""
template <typename T>
static T* take(const char* name, long bytes, int shift = 0) {  // exactly as large, `shift` bytes past 16
  uint8_t* p = (uint8_t*)aligned_alloc(16, (bytes + shift + 15) / 16 * 16) + shift;
  FILE* f = fopen(name, "rb");
  if (!f || (long)fread(p, 1, bytes, f) != bytes) exit(3);
  fclose(f);
  return (T*)p;
}
int main(int, char** v) {  // coded's length and alignment, contexts, streams, symbols of a stream
  const long coded_len = atol(v[1]);
  const int lead = atoi(v[2]), n_ctx = atoi(v[3]), spc = atoi(v[4]), len = atoi(v[5]);
  const long n = (long)n_ctx * spc * len;
  // (whole words are read)
  uint8_t* coded = take<uint8_t>("coded", (coded_len + lead + 3) / 4 * 4 - lead, lead);
  auto *freq = take<uint16_t>("freq", 512L * n_ctx), *sizes = take<uint16_t>("sizes", 2L * n_ctx * spc);
  auto* states = take<uint32_t>("states", 4L * n_ctx * spc);
  uint8_t* sym = (uint8_t*)malloc(n);
  for (int ctx = 0; ctx < n_ctx; ++ctx)
    for (int group = 0; group < spc / 64; ++group) {
      blockIdx = {group, ctx};
      std::barrier<> all(DECODE_THREADS);
      everyone = &all;
      for (auto& w : of_wave) w = new std::barrier<>(64);
      std::vector<std::thread> threads;
      for (int t = 0; t < DECODE_THREADS; ++t)
        threads.emplace_back([=] {
          threadIdx = {t, 0};
          rans_decode_kernel(coded, coded_len, freq, sizes, states, sym, (long)spc * len, spc);
        });
      for (auto& t : threads) t.join();
      for (auto& w : of_wave) delete w;
    }
  FILE* f = fopen("sym", "wb");
  return fwrite(sym, 1, n, f) == (size_t)n && fclose(f) == 0 ? 0 : 4;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    text = (ROOT / "csrc/kernels/rans.hip").read_text()
    begin = text.index("template <int DIR, typename F>")
    end = text.index("\n}\n", text.index("void rans_decode_kernel(")) + 3
    at = tmp_path_factory.mktemp("rans")
    (at / "decode.cpp").write_text(HOST + text[begin:end] + MAIN)
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-w", "-pthread", "-fsanitize=address", "decode.cpp", "-o", "decode"], cwd=at, check=True, timeout=120)
    return at


def _decode(at, freq, states, sizes, coded, n_ctx, spc, length, lead=0):
    whole = (coded.size + lead + 3) // 4 * 4 - lead
    (at / "coded").write_bytes(coded.tobytes() + bytes(whole - coded.size))
    for name, a in (("freq", freq), ("states", states), ("sizes", sizes)):
        (at / name).write_bytes(np.ascontiguousarray(a).tobytes())
    run = subprocess.run(["./decode", *map(str, (coded.size, lead, n_ctx, spc, length))], cwd=at, capture_output=True, text=True, timeout=100,
                         env={**os.environ, "ASAN_OPTIONS": "detect_leaks=0"})
    assert run.returncode == 0, run.stderr[-3000:]
    return np.fromfile(at / "sym", dtype=np.int8)


# less than a run of 16, whole runs, a remainder; bytes of 64 streams that a thread asks for at once, more, as much as where the table is made, and too much to stage
@pytest.mark.parametrize("length,spread,lead", [(1, 64, 0), (15, 64, 1), (16, 2, 2), (17, 64, 3), (262, 64, 0), (345, 64, 1), (372, 64, 3)])
def test_pages_come_back(program, length, spread, lead):
    n_ctx, spc = 2, 128
    sym = np.random.default_rng(length).integers(-spread, spread, n_ctx * spc * length, dtype=np.int8)
    sym[: spc * length] = np.where(np.arange(spc * length) % 7 == 0, sym[: spc * length], 5)
    freq, states, sizes, coded = ref.rans_encode(sym, n_ctx, spc)
    assert np.array_equal(_decode(program, freq, states, sizes, coded, n_ctx, spc, length, lead), sym)


@pytest.mark.parametrize("what,length", [(w, n) for w in ("sizes", "small sizes", "tables", "states", "bytes", "short") for n in (1, 17)]
                         + [("everything", n) for n in (1, 15, 16, 17, 300)])
def test_damage_stays_inside(program, what, length):
    n_ctx, spc = 2, 128
    g = np.random.default_rng(length)
    sym = g.integers(-64, 64, n_ctx * spc * length, dtype=np.int8)
    freq, states, sizes, coded = ref.rans_encode(sym, n_ctx, spc)
    if what in ("sizes", "everything"):
        sizes = g.integers(0, 1 << 16, sizes.size, dtype=np.uint16)  # their sum is past the coded bytes, and a group's past what is staged
    if what == "small sizes":
        sizes = g.integers(0, 4, sizes.size, dtype=np.uint16)
    if what in ("tables", "everything"):
        freq = g.integers(0, 1 << 16, freq.size, dtype=np.uint16)
        freq[::3] = 0
    if what in ("states", "everything"):
        states = g.integers(0, 1 << 32, states.size, dtype=np.uint32)
        states[::5] = 0  # two bytes a step to the end
    if what in ("bytes", "everything"):
        coded = g.integers(0, 256, coded.size, dtype=np.uint8)
    if what == "short":
        coded = coded[: coded.size // 3]
    assert _decode(program, freq, states, sizes, coded, n_ctx, spc, length, length % 4).size == n_ctx * spc * length
