"""A mesh's bounding box (init_mesh, j3d_amd/csrc/j3dg.hip, compiled from the
source): the sequential std::min / std::max fold over the vertices on any
number of threads, no more of them than the caller allows, and also when a
thread cannot be had."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEAD = r"""
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <random>
#include <thread>
#include <vector>

static std::atomic<int> g_made{0}, g_left{1 << 30};
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
  using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Fn real = (Fn)dlsym(RTLD_NEXT, "pthread_create");
  if (g_left.fetch_sub(1) <= 0) return EAGAIN;
  g_made++;
  return real(t, a, f, arg);
}
struct Mesh {
  bool live = false;
  uint32_t db_id = 0;
  float cs[16], inv_cs[16];
  struct { uint64_t n_vertices, n_triangles; float bb_min[3], bb_max[3]; } info;
};
static void invert_orthonormal(const float*, float*) {}
"""

MAIN = r"""
int main() {
  int bad = 0;
  std::mt19937 rng(3);
  std::uniform_real_distribution<float> U(-5.f, 5.f);
  for (uint64_t n : {1ull, 2ull, 65535ull, 65536ull, 65537ull, 300001ull})
    for (int kind = 0; kind < 3; ++kind) {
      std::vector<float> v(3 * n);
      for (auto& x : v) x = U(rng);
      if (kind) for (uint64_t i = kind == 1 ? 0 : 1; i < 3 * n; i += 37) v[i] = NAN;
      float lo[3], hi[3];
      for (int k = 0; k < 3; ++k) lo[k] = hi[k] = v[k];
      for (uint64_t i = 0; i < n; ++i)
        for (int k = 0; k < 3; ++k) lo[k] = std::min(lo[k], v[3 * i + k]), hi[k] = std::max(hi[k], v[3 * i + k]);
      for (int threads : {0, 1, 2, 64})
        for (int left : {1 << 30, 0, 1}) {
          Mesh m;
          g_made = 0, g_left = left;
          init_mesh(m, 1, nullptr, v.data(), n, 0, threads);
          const int limit = threads ? threads - 1 : 1 << 30;
          if (std::memcmp(m.info.bb_min, lo, 12) || std::memcmp(m.info.bb_max, hi, 12) || g_made > limit || g_made > left)
            ++bad, printf("n %llu kind %d threads %d left %d: %d threads made\n", (unsigned long long)n, kind, threads,
                          left, g_made.load());
        }
    }
  printf(bad ? "BAD %d\n" : "BOX OK\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_box_on_any_number_of_threads(tmp_path):
    s = open(os.path.join(ROOT, "j3d_amd", "csrc", "j3dg.hip")).read()
    body = s[s.index("static void init_mesh("):s.index("static uint32_t insert_mesh(")]
    src = tmp_path / "box.cpp"
    src.write_text(HEAD + body + MAIN)
    exe = tmp_path / "box"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-o", str(exe), str(src), "-ldl"], check=True, timeout=120)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0 and "BOX OK" in r.stdout, r.stdout[-2000:]
