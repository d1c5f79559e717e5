// block_add (j3d_amd/csrc/bvh_gpu.hip, cut out by the test as the GPU compiles
// it) on the emulated HIP runtime: every thread of a block gets a range of its
// own, in thread order, and the counter the block's sum, with one atomic per
// block; several calls in a row, counts of 0 to 3, blocks of 1 to 16 waves.
#include <hip/hip_runtime.h>

// the calling lane's value from `d` lanes below; its own in the first d lanes
#define __shfl_up(v, d, w) \
  __shfl((v), ((threadIdx.x & 63u) >= (d) ? (threadIdx.x & 63u) - (d) : (threadIdx.x & 63u)), 64)

static uint64_t g_atomics = 0;
inline uint32_t counted_add(uint32_t* p, uint32_t v) {
  ++g_atomics;
  return atomicAdd(p, v);
}
#define __HIPCC__
#define atomicAdd counted_add
#include "block_add.inc"
#undef atomicAdd

struct Out {
  uint32_t at[2], n[2];
};

static void k_check(Out* out, uint32_t* counters, uint32_t seed) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  for (uint32_t c = 0; c < 2; ++c) {
    uint32_t h = (i * 2654435761u) ^ (seed * 40503u) ^ (c << 7);
    h ^= h >> 15, h *= 2246822519u, h ^= h >> 13;
    const uint32_t n = seed == 0 ? 0u : seed == 1 ? 1u : h & 3u;
    out[i].n[c] = n;
    out[i].at[c] = block_add(counters + c, n);
  }
}

int main() {
  int bad = 0;
  for (uint32_t block : {64u, 128u, 256u, 1024u})
    for (uint32_t seed = 0; seed < 5; ++seed) {
      const uint32_t blocks = 3, total = block * blocks;
      std::vector<Out> out(total);
      uint32_t counters[2] = {5, 0};
      g_atomics = 0;
      emu::launch("k_check", k_check, dim3(blocks), dim3(block), 0, out.data(), counters, seed);
      for (uint32_t c = 0; c < 2; ++c) {
        uint32_t at = c == 0 ? 5 : 0;  // blocks run one after the other
        for (uint32_t i = 0; i < total; ++i) {
          if (out[i].n[c] && out[i].at[c] != at) ++bad;
          at += out[i].n[c];
        }
        if (counters[c] != at) ++bad;
      }
      if (g_atomics > 2 * blocks) ++bad;
      if (bad) printf("block %u seed %u\n", block, seed);
    }
  printf(bad ? "FAILED %d\n" : "BLOCK ADD OK\n", bad);
  return bad != 0;
}
