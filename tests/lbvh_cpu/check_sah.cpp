// The host SAH over the top levels of a device-built tree
// (lbvh::sah_build, j3d_amd/csrc/bvh_gpu.hip, cut out by the test) with its
// threads: random, equal, NaN and nested clusters around the sizes where a
// subtree gets a thread.  Arguments:
//   trees      the threaded build gives the tree that one thread builds, and
//              every cluster is in it once (built with ThreadSanitizer too)
//   threads N  the same with every thread creation after the first N refused
//   memory     every allocation of the build fails in turn: the exception
//              reaches the caller, with every thread at its end
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <atomic>
#include <map>
#include <new>
#include <random>
#include <string>
#include <vector>

#include "shim.h"

static std::atomic<long> g_fail_at{-1};    // the allocation that fails, counted down; -1: none
static std::atomic<long> g_threads_left{1L << 40};

#ifdef CHECK_MEMORY
void* operator new(size_t n) {
  if (g_fail_at.load() >= 0 && g_fail_at.fetch_sub(1) == 0) throw std::bad_alloc();
  if (void* p = malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
#endif
#ifdef CHECK_THREADS
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
  using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Fn real = (Fn)dlsym(RTLD_NEXT, "pthread_create");
  if (g_threads_left.fetch_sub(1) <= 0) return EAGAIN;
  return real(t, a, f, arg);
}
#endif

namespace j3d {
#include "lbvh_body.inc"
}
using namespace j3d;
using namespace j3d::lbvh;

static std::vector<Cluster> clusters(uint32_t m, int kind) {
  std::mt19937 rng(m * 7 + kind);
  std::uniform_real_distribution<float> U(-1.f, 1.f);
  std::vector<Cluster> cl(m);
  for (uint32_t i = 0; i < m; ++i) {
    Cluster& c = cl[i];
    c.ref = i;
    c.count = 1 + i % 5;
    const float nested = std::exp2(100.f * (float)i / (float)m - 50.f);
    for (int a = 0; a < 3; ++a) {
      const float x = U(rng), w = 0.05f * std::fabs(U(rng));
      c.lo[a] = kind == 1 ? -1.f : kind == 3 ? -nested : x - w;
      c.hi[a] = kind == 1 ? 1.f : kind == 3 ? 1.01f * nested : x + w;
      if (kind == 2 && i % 11 == (uint32_t)a) c.hi[a] = NAN;
      c.c[a] = 0.5f * c.lo[a] + 0.5f * c.hi[a];
    }
  }
  return cl;
}

// the tree below r as text, children in order
static void walk(const std::vector<SahNode>& n, uint32_t r, std::string& out, std::vector<int>& seen) {
  std::vector<uint32_t> todo = {r};
  while (!todo.empty()) {
    const uint32_t x = todo.back();
    todo.pop_back();
    if (x & kSahTag) {
      const SahNode& s = n[x & ~kSahTag];
      out += '(';
      out.append((const char*)&s.count, sizeof(s) - offsetof(SahNode, count));
      todo.push_back(s.right);
      todo.push_back(s.left);
    } else {
      seen[x]++;
      out += std::to_string(x) + ' ';
    }
  }
}

static std::string tree(std::vector<Cluster> cl, bool threaded, int& bad) {
  const uint32_t m = (uint32_t)cl.size();
  std::vector<SahNode> n;
  std::vector<float> area(m + 1);
  uint32_t root;
  if (threaded) {
    root = sah_build(cl, 0, m, n, area);
  } else {
    SahSpace sp(m, area);
    for (int a = 0; a < 3; ++a) sah_sort(cl, sp, a, 0, m);
    root = sah_range(cl, sp, 0, m, n);
  }
  std::string s;
  std::vector<int> seen(m, 0);
  walk(n, kSahTag | root, s, seen);
  bad += root != 0 || n.size() != m - 1;
  for (int k : seen) bad += k != 1;
  return s;
}

int main(int argc, char** argv) {
  const std::string what = argv[1];
  int bad = 0;
  if (what == "memory") {
    const std::vector<Cluster> cl = clusters(3 * kSahTask, 0);
    const uint32_t m = (uint32_t)cl.size();
    long thrown = 0, at = 0;
    for (;; ++at) {
      std::vector<Cluster> c = cl;
      std::vector<SahNode> n;
      std::vector<float> area(m + 1);
      n.reserve(m);
      g_fail_at = at;
      bool failed = false;
      try {
        sah_build(c, 0, m, n, area);
      } catch (const std::bad_alloc&) {
        failed = true;
      }
      const bool reached = g_fail_at.load() < 0;
      g_fail_at = -1;
      thrown += failed;
      if (reached && !failed) ++bad;
      if (!reached) break;  // the build makes no more than `at` allocations
    }
    printf("%ld allocations, %ld failures thrown\n", at, thrown);
    bad += thrown < 10;
  } else {
    if (argc > 2) g_threads_left = atol(argv[2]);
    for (uint32_t m : {2u, 3u, 100u, kSahTask - 1, kSahTask, kSahTask + 1, 2 * kSahTask + 1, 20000u})
      for (int kind = 0; kind < 4; ++kind) {
        const std::vector<Cluster> cl = clusters(m, kind);
        if (tree(cl, true, bad) != tree(cl, false, bad)) ++bad, printf("m %u kind %d: other tree\n", m, kind);
      }
  }
  printf(bad ? "FAILED %d\n" : "SAH OK\n", bad);
  return bad != 0;
}
