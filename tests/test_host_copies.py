"""Copies from host memory to host memory by several threads (``csrc/kernels/host_copies.h``), built for the host alone: sizes round the pieces, many
callers, no memory for anything of its own, a fork; under ThreadSanitizer and AddressSanitizer too."""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
SOURCE = r"""
#ifdef __SANITIZE_THREAD__  // gcc 11's does not know the wait by another clock and takes the mutex for held meanwhile
#include <cstddef>
#undef _GLIBCXX_USE_PTHREAD_COND_CLOCKWAIT
#endif
#include "host_copies.h"
#include <stdio.h>
#include <stdlib.h>
#include <sys/wait.h>
#include <unistd.h>
#include <vector>

static std::atomic<bool> poor{false};  // no memory for `new`
static void* take(size_t n) { return poor ? nullptr : malloc(n ? n : 1); }
void* operator new(size_t n) { if (void* p = take(n)) return p; throw std::bad_alloc(); }
void* operator new(size_t n, const std::nothrow_t&) noexcept { return take(n); }
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

static bool copy(long n, unsigned seed) {
  char *from = (char*)malloc(n + 1), *to = (char*)malloc(n + 1);
  for (long i = 0; i < n; ++i) from[i] = (char)(i * 2654435761u + seed >> 13);
  to[n] = 77;
  copy_in_parts(to, from, n);
  const bool same = memcmp(from, to, n) == 0 && to[n] == 77;
  free(from), free(to);
  return same;
}

int main(int argc, char**) {
  const long sizes[] = {0, 1, COPY_PART - 1, COPY_PART, 2 * COPY_PART - 1, 2 * COPY_PART, 3 * COPY_PART + 5, 4 * COPY_PART + 4095, 9 * COPY_PART};
  poor = true;  // before there is a helper
  for (long n : sizes) if (!copy(n, 1)) return 1;
  poor = false;
  for (long n : sizes) if (!copy(n, 2)) return 2;
  poor = true;
  for (int i = 0; i < 20; ++i) if (!copy(4 * COPY_PART + i, 3)) return 3;
  poor = false;
  std::atomic<int> bad{0};
  std::vector<std::thread> callers;
  for (int t = 0; t < 6; ++t)
    callers.emplace_back([&, t] { for (int i = 0; i < 12; ++i) bad += !copy(sizes[(t + i) % 9] + t, t + i); });
  for (auto& c : callers) c.join();
  if (bad) return 4;
  if (argc == 1) {  // (a sanitizer's own threads do not live through a fork)
    const pid_t child = fork();
    if (child == 0) _exit(copy(5 * COPY_PART, 9) ? 0 : 1);
    int status = 1;
    if (waitpid(child, &status, 0) != child || status != 0) return 5;
  }
  puts("copies ok");
  return 0;
}
"""


@pytest.mark.parametrize("flags", [[], ["-fsanitize=thread"], ["-fsanitize=address,undefined"]], ids=["plain", "threads", "addresses"])
def test_copies(tmp_path, flags):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    src, exe = tmp_path / "copies.cpp", tmp_path / "copies"
    src.write_text(SOURCE)
    build = subprocess.run([gxx, "-std=c++17", "-O1", "-g", *flags, "-I", str(ROOT / "csrc/kernels"), str(src), "-o", str(exe), "-lpthread"],
                           capture_output=True, text=True)
    if build.returncode != 0 and "cannot find" in build.stderr:
        pytest.skip(f"sanitizer runtime not installed: {build.stderr.splitlines()[-1]}")
    assert build.returncode == 0, build.stderr
    env = {"ASAN_OPTIONS": "alloc_dealloc_mismatch=0:detect_leaks=0", "TSAN_OPTIONS": "halt_on_error=1"}
    run = subprocess.run([str(exe), *(["-"] if flags else [])], capture_output=True, text=True, timeout=120, env=env)
    assert run.returncode == 0 and "copies ok" in run.stdout, (run.returncode, run.stdout + run.stderr)
