// allhits.hip -- the second query of the reference's BVH: every hit of a ray
// in one mesh (jtk::qbvh::find_all_triangles, called at j3d/vox.cpp:333), and
// the voxel grid write_vox builds from it (j3d/vox.cpp:278-376), on the GPU.
//
// The query: one ray per lane, one launch: the lane walks the mesh's BVH with
// the frame kernel's node decode and stack (top entries in LDS, older ones
// spilled), and keeps its hits in a list in global memory sorted by (t,
// triangle id), the first `cap` of them (an insertion per accepted hit).  The
// result does not depend on the visiting order.
//
// The voxel grid: a group of eight lanes per ray, each walking parts of the
// tree with a stack of its own; the hits go to the ray's list in any order and
// their ranks in (t, triangle id) order are counted afterwards.  Where several
// hits land in one voxel, the reference's sequential order decides (axis, row,
// column, hit): each write is a 64-bit key (that position, then the palette
// index) merged with atomicMax, so the largest key -- the sequentially last
// write -- survives.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <vector>

#include "bvh_build.h"
#include "j3dg.h"
#include "j3dg_internal.h"
#include "rt_math.h"
#include "traverse.h"

namespace j3d {
namespace {

constexpr int kAllD = 16;             // LDS stack entries per lane
constexpr uint32_t kAllBlock = 256;
constexpr uint32_t kMaxVoxDim = 1024;  // voxel grid side (the key holds 12 bits per row / column index)
constexpr uint32_t kMaxVoxHits = 1u << 24;  // hits per voxel ray (24 bits of the key)

struct HitRec {
  float t;
  uint32_t tri;
  float u, v;
};

struct AllHitsArgs {
  const float4* nodes;
  const float4* tris;
  float inv_cs[16];         // world -> object for query rays
  const float* rays;        // n x 8 world rays (the query)
  uint32_t n;
  uint32_t axis_first[3];   // voxel rays: first ray of the x, y and z axis (x rays start at 0)
  uint32_t dim[3];
  float bmin[3], bmax[3];
  uint32_t cap;             // stored hits per ray
  HitRec* hits;             // cap per ray (the query) or per group of the grid (voxel rays)
  uint32_t* counts;         // the query: hits per ray (all of them, stored or not)
  uint32_t* max_count;      // voxel rays: largest count over the rays that did not fit
  uint2* spill;
  uint32_t spill_cap;
  unsigned long long* keys;  // voxel grid, 0 = empty
  const float* verts;
  const uint32_t* idx;
  const float* vcol;
  const float* uv;
  const uint32_t* tex;
  uint32_t tex_w, tex_h;
  uint32_t color_mode;      // 0 white, 1 vertex colours, 2 texture
};

__device__ inline bool hit_less(float t, uint32_t id, float t2, uint32_t id2) {
  return t < t2 || (t == t2 && id < id2);
}

// Keeps list[0 .. min(count, cap)) the smallest hits by (t, id), sorted.
__device__ inline void insert_hit(HitRec* list, uint32_t& count, uint32_t cap, float t, uint32_t id, float u,
                                  float v) {
  uint32_t stored = count < cap ? count : cap;
  ++count;
  if (stored == cap) {
    if (cap == 0) return;
    const HitRec last = list[cap - 1];
    if (!hit_less(t, id, last.t, last.tri)) return;
    --stored;
  }
  uint32_t j = stored;
  while (j > 0) {
    const HitRec p = list[j - 1];
    if (!hit_less(t, id, p.t, p.tri)) break;
    list[j] = p;
    --j;
  }
  list[j] = HitRec{t, id, u, v};
}

// (uint32_t)x for a coordinate that should lie in [0, n): truncation toward
// zero, saturated into [0, n - 1], NaN -> 0 (the reference's casts are
// undefined outside the range).
__device__ inline uint32_t vox_index(float x, uint32_t n) {
  if (!(x > 0.f)) return 0u;
  if (x >= (float)n) return n - 1u;
  const uint32_t i = (uint32_t)x;
  return i < n ? i : n - 1u;
}

// color_to_index (j3d/vox.cpp:154-171)
__device__ inline uint32_t vox_color_index(uint32_t r, uint32_t g, uint32_t b) {
  r = r < 16u ? 0u : r - 16u;
  g = g < 16u ? 0u : g - 16u;
  b = b < 32u ? 0u : b - 32u;
  const uint32_t ret = ((r >> 5) << 5) | ((g >> 5) << 2) | (b >> 6);
  return ret ? ret : 1u;
}

template <int W>
__global__ void __launch_bounds__(kAllBlock) k_all_hits(AllHitsArgs a) {
  extern __shared__ uint2 lds_stack[];
  StackArea area;
  area.init(lds_stack, a.spill, a.spill_cap);
  Stack<kAllD> st(area);
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  Trav s;
  const float* q = a.rays + 8 * (size_t)i;
  const f4 o = {q[0], q[1], q[2], 1.f}, d = {q[3], q[4], q[5], 0.f};
  s.r = make_object_ray(a.inv_cs, o, d, q[6], q[7]);
  s.nodes = a.nodes;
  s.tris = a.tris;
  s.thi = s.r.t_far * kSlackUp;
  s.tmax = s.r.t_far;
  s.cur = ray_finite(o, d) ? 0u : kNone;  // the root, an internal node; a ray that is not finite hits nothing
  s.obj = 0;
  s.base = 0;
  s.any = false;
  Counters c = {0, 0, 0};
  HitRec* list = a.hits + (size_t)i * a.cap;
  uint32_t count = 0;
  for (;;) {
    if (s.cur != kNone) {
      if (s.cur & kLeafBit) {
        const uint32_t first = s.cur & kLeafIndexMask;
        const uint32_t cnt = ((s.cur >> kLeafCountShift) & 3u) + 1u;
        for (uint32_t k = 0; k < cnt; ++k) {
          const float4* tp = s.tris + (size_t)(first + k) * 3;
          const float4 v0 = gload4(tp), e1 = gload4(tp + 1), e2 = gload4(tp + 2);
          float t, u, v;
          if (intersect_triangle(s.r.ox, s.r.oy, s.r.oz, s.r.dx, s.r.dy, s.r.dz, v0.x, v0.y, v0.z, e1.x, e1.y, e1.z,
                                 e2.x, e2.y, e2.z, s.r.t_near, s.r.t_far, t, u, v))
            insert_hit(list, count, a.cap, t, __float_as_uint(v0.w), u, v);
        }
        s.cur = kNone;
      } else {
        s.cur = visit_node<W, kAllD, false>(s.nodes, s.cur, s.r, s.thi, st, c);
      }
    }
    if (s.cur == kNone && pop_next<kAllD>(s, st)) break;
  }
  a.counts[i] = count;
}

// A hit of a voxel ray to its voxel (j3d/vox.cpp:335-375); rank: its position
// among the ray's hits.
__device__ inline void write_voxel(const AllHitsArgs& a, const HitRec& h, uint32_t rank, uint32_t ax, uint32_t d1,
                                   uint32_t d2) {
  const uint32_t* tr = a.idx + 3 * (size_t)h.tri;
  const float* p0 = a.verts + 3 * (size_t)tr[0];
  const float* p1 = a.verts + 3 * (size_t)tr[1];
  const float* p2 = a.verts + 3 * (size_t)tr[2];
  const float w = 1.f - h.u - h.v;
  float pos[3], clr[3] = {1.f, 1.f, 1.f};
  for (int j = 0; j < 3; ++j) pos[j] = p0[j] * w + h.u * p1[j] + h.v * p2[j];
  if (a.color_mode == 2) {
    const float* uvc = a.uv + 6 * (size_t)h.tri;
    float cc[2];
    for (int j = 0; j < 2; ++j) {
      cc[j] = w * uvc[j] + h.u * uvc[2 + j] + h.v * uvc[4 + j];
      // std::max(std::min(c, 1.f), 0.f), NaN kept (vox.cpp:345-346)
      const float lo = 1.f < cc[j] ? 1.f : cc[j];
      cc[j] = lo < 0.f ? 0.f : lo;
    }
    const uint32_t x = vox_index(cc[0] * (float)(a.tex_w - 1), a.tex_w);
    const uint32_t y = vox_index(cc[1] * (float)(a.tex_h - 1), a.tex_h);
    const uint32_t col = a.tex[(size_t)y * a.tex_w + x];
    clr[0] = (float)(col & 255u) / 255.f;
    clr[1] = (float)((col >> 8) & 255u) / 255.f;
    clr[2] = (float)((col >> 16) & 255u) / 255.f;
  } else if (a.color_mode == 1) {
    const float* c0 = a.vcol + 3 * (size_t)tr[0];
    const float* c1 = a.vcol + 3 * (size_t)tr[1];
    const float* c2 = a.vcol + 3 * (size_t)tr[2];
    for (int j = 0; j < 3; ++j) clr[j] = c0[j] * w + h.u * c1[j] + h.v * c2[j];
  }
  uint32_t X[3];
  for (int j = 0; j < 3; ++j)
    X[j] = vox_index((pos[j] - a.bmin[j]) / (a.bmax[j] - a.bmin[j]) * (float)a.dim[j], a.dim[j]);
  const uint32_t ci = vox_color_index(color_byte(clr[0]), color_byte(clr[1]), color_byte(clr[2]));
  unsigned long long key = ax;
  key = (key << 12) | d1;
  key = (key << 12) | d2;
  key = (key << 24) | rank;
  key = (key << 8) | ci;
  atomicMax(a.keys + X[0] + ((size_t)X[1] + (size_t)X[2] * a.dim[1]) * a.dim[0], key);
}

// The voxel rays of all three axes.  A ray along an axis crosses the whole
// mesh, hundreds of dependent node fetches where it grazes the surface, and a
// grid has few of them (256 x 224 x 128: 118,000, two waves per SIMD with one
// ray per lane, each as long as its longest ray).  So a group of
// kVoxLanes lanes takes a ray: each walks its own part of the tree, and idle
// lanes take entries from the others' stacks after every step.  Order does not
// matter here, so nodes are not sorted.  Waves take rounds of 64 / kVoxLanes
// rays, a round's lists being the waves' own.  One lane / eight lanes per ray, us:
//   2M triangles      256 per side  605 /  121   512   826 /  340   1024 1935 / 1144
//   28M triangles                  1032 /  187        1294 /  508        3081 / 1530
//   100,000 triangles               376 /   77         512 /  249        1135 /  873
//   20,000, a dense soup            812 /  347        2094 / 1211
//   1,280 triangles                  97 /   82         265 /  292         790 / 1131
// Only a coarse mesh on a large grid has rays too short to share; its call
// (13.5 and 105 ms) is the grid's copy to the host.
constexpr uint32_t kVoxLanes = 8;
constexpr uint32_t kVoxGroups = kAllBlock / kVoxLanes;
// Hits of a ray ranked by counting (k^2 / 8 reads per lane); more are sorted.
constexpr uint32_t kRankMax = 128;

// Sorts a ray's hits by (t, id): bitonic, in memory, by the group's lanes.  The
// list's capacity is a power of two, so there is room for the padding.
__device__ inline void sort_list(HitRec* list, uint32_t count, uint32_t lane) {
  uint32_t p2 = kRankMax;
  while (p2 < count) p2 *= 2;
  for (uint32_t k = count + lane; k < p2; k += kVoxLanes) list[k] = HitRec{INFINITY, kMiss, 0.f, 0.f};
  for (uint32_t size = 2; size <= p2; size *= 2)
    for (uint32_t step = size / 2; step >= 1; step /= 2) {
      __threadfence_block();  // the other lanes' exchanges of the last step are in memory
      for (uint32_t m = lane; m < p2 / 2; m += kVoxLanes) {
        const uint32_t i = m / step * step * 2 + m % step, j = i + step;
        const HitRec x = list[i], y = list[j];
        const bool up = (i & size) == 0;
        if (up ? hit_less(y.t, y.tri, x.t, x.tri) : hit_less(x.t, x.tri, y.t, y.tri)) list[i] = y, list[j] = x;
      }
    }
  __threadfence_block();
}

template <int W>
__global__ void __launch_bounds__(kAllBlock, 4) k_vox_rays(AllHitsArgs a) {
  extern __shared__ uint2 lds_stack[];
  __shared__ uint32_t hit_count[kVoxGroups];
  StackArea area;
  area.init(lds_stack, a.spill, a.spill_cap);
  Stack<kAllD> st(area);
  const uint32_t group = threadIdx.x / kVoxLanes, lane = threadIdx.x % kVoxLanes;
  HitRec* list = a.hits + ((size_t)blockIdx.x * kVoxGroups + group) * a.cap;
  // waves of consecutive blocks take consecutive octets of rays
  constexpr uint32_t kWaveRays = 64u / kVoxLanes;
  const uint32_t n_waves = gridDim.x * (kAllBlock / 64u);
  for (uint32_t r0 = ((threadIdx.x >> 6) * gridDim.x + blockIdx.x) * kWaveRays; r0 < a.n; r0 += n_waves * kWaveRays) {
    const uint32_t i = r0 + (threadIdx.x & 63u) / kVoxLanes;
    uint32_t d1 = 0, d2 = 0, ax = 0;
    bool finite = false;
    Trav s;
    s.r = Ray{0.f, 0.f, 0.f, 1.f, 0.f, 0.f, 1.f, 1.f, 1.f, 0.f, 0.f};
    if (i < a.n) {
      // write_vox's ray of row d1, column d2 along axis ax (j3d/vox.cpp:317-330)
      ax = i >= a.axis_first[2] ? 2u : (i >= a.axis_first[1] ? 1u : 0u);
      const uint32_t ax1 = (ax + 1) % 3, ax2 = (ax + 2) % 3, r = i - a.axis_first[ax];
      d1 = r / a.dim[ax2];
      d2 = r % a.dim[ax2];
      float o[3], d[3] = {0.f, 0.f, 0.f};
      o[ax] = a.bmin[ax];
      o[ax1] = (((float)d1 + 0.5f) / (float)a.dim[ax1]) * (a.bmax[ax1] - a.bmin[ax1]) + a.bmin[ax1];
      o[ax2] = (((float)d2 + 0.5f) / (float)a.dim[ax2]) * (a.bmax[ax2] - a.bmin[ax2]) + a.bmin[ax2];
      d[ax] = ax == 2 ? 2.f : 1.f;
      const f4 oo = {o[0], o[1], o[2], 1.f}, dd = {d[0], d[1], d[2], 0.f};
      finite = ray_finite(oo, dd);  // a NaN or infinite mesh box gives rays that hit nothing
      s.r = world_ray(oo, dd, 0.f, FLT_MAX);
    }
    s.nodes = a.nodes;
    s.tris = a.tris;
    s.thi = FLT_MAX * kSlackUp;
    s.tmax = FLT_MAX;
    s.cur = finite && lane == 0 ? 0u : kNone;  // lane 0 starts at the root, an internal node
    s.obj = 0;
    s.base = 0;
    s.any = true;  // no order
    st.sp = 0;
    if (lane == 0) hit_count[group] = 0;
    __builtin_amdgcn_wave_barrier();
    Counters c = {0, 0, 0};
    while (__ballot(s.cur != kNone)) {
      if (s.cur != kNone) {
        if (s.cur & kLeafBit) {
          const uint32_t first = s.cur & kLeafIndexMask;
          const uint32_t cnt = ((s.cur >> kLeafCountShift) & 3u) + 1u;
          for (uint32_t k = 0; k < cnt; ++k) {
            const float4* tp = s.tris + (size_t)(first + k) * 3;
            const float4 v0 = gload4(tp), e1 = gload4(tp + 1), e2 = gload4(tp + 2);
            float t, u, v;
            if (intersect_triangle(s.r.ox, s.r.oy, s.r.oz, s.r.dx, s.r.dy, s.r.dz, v0.x, v0.y, v0.z, e1.x, e1.y, e1.z,
                                   e2.x, e2.y, e2.z, s.r.t_near, s.r.t_far, t, u, v)) {
              const uint32_t at = atomicAdd(&hit_count[group], 1u);
              if (at < a.cap) list[at] = HitRec{t, __float_as_uint(v0.w), u, v};
            }
          }
          s.cur = kNone;
        } else {
          constexpr int kVec = W == 8 ? 6 : 4;
          const float4* np = s.nodes + (size_t)s.cur * kVec;
          float4 v[kVec];
#pragma unroll
          for (int k = 0; k < kVec; ++k) v[k] = gload4(np + k);
          s.cur = decode_node<W, kAllD, false>(v, s.r, s.thi, st, c, false);
        }
        if (s.cur == kNone && pop_next<kAllD>(s, st)) s.cur = kNone;
      }
      const bool busy = s.cur != kNone;
      const uint32_t idle = split_mask(__ballot(!busy), kVoxLanes);
      const uint32_t donors = split_mask(__ballot(busy && st.sp > 0u), kVoxLanes);
      j3d_u32x2 got = {kNone, 0u};
      int src;
      uint32_t pos;
      if (idle && donors && deal_work<kAllD>(st, busy, idle, donors, kVoxLanes, got, src, pos)) s.cur = got.x;
    }
    // the group's hits are in memory before its lanes read them
    __threadfence_block();
    const uint32_t count = *(volatile uint32_t*)&hit_count[group];
    if (count > a.cap) {  // the host grows the lists and runs the launch again
      if (lane == 0) atomicMax(a.max_count, count);
      continue;
    }
    const bool sorted = count > kRankMax;
    if (sorted) sort_list(list, count, lane);
    for (uint32_t k = lane; k < count; k += kVoxLanes) {
      const HitRec h = list[k];
      uint32_t rank = k;
      if (!sorted) {
        rank = 0;
        for (uint32_t m = 0; m < count; ++m) rank += hit_less(list[m].t, list[m].tri, h.t, h.tri) ? 1u : 0u;
      }
      write_voxel(a, h, rank, ax, d1, d2);
    }
  }
}

__global__ void k_vox_final(const unsigned long long* __restrict__ keys, uint64_t n, uint8_t* __restrict__ data) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    data[i] = (uint8_t)(keys[i] & 255ull);
}

// write_vox's grid size (j3d/vox.cpp:284-297), in float: dim_k = max_dim *
// extent_k / largest extent, at least 1; a NaN ratio counts as 0.
void vox_dims(const float* mn, const float* mx, uint32_t max_dim, uint32_t dim[3]) {
  int L = 0;
  if ((mx[1] - mn[1]) > (mx[L] - mn[L])) L = 1;
  if ((mx[2] - mn[2]) > (mx[L] - mn[L])) L = 2;
  for (int j = 0; j < 3; ++j) {
    const float q = (float)max_dim * (mx[j] - mn[j]) / (mx[L] - mn[L]);
    uint32_t d = 0;
    if (q > 0.f) d = q >= (float)max_dim ? max_dim : (uint32_t)q;
    dim[j] = d ? d : 1u;
  }
}

void fill_mesh_args(const Mesh& m, AllHitsArgs& a) {
  std::memset(&a, 0, sizeof(a));
  a.nodes = m.d_nodes;
  a.tris = m.d_tris;
  std::memcpy(a.inv_cs, m.inv_cs, sizeof(a.inv_cs));
  a.verts = m.d_verts;
  a.idx = m.d_idx;
}

// Launches the query (grid: a lane per ray) or the voxel rays.
int launch_all_hits(Ctx* ctx, const Mesh& m, AllHitsArgs& a, uint32_t grid, bool vox) {
  const uint32_t cap = m.max_stack > (uint32_t)kAllD ? m.max_stack - kAllD + 1 : 1;
  int rc = ctx->ensure_spill((uint64_t)grid * kAllBlock, cap);
  if (rc) return rc;
  a.spill = ctx->spill;
  a.spill_cap = cap;
  const size_t lds = (size_t)kAllD * kAllBlock * sizeof(uint2);
  const bool w8 = m.info.width == 8;
  void (*fn)(AllHitsArgs) = vox ? (w8 ? k_vox_rays<8> : k_vox_rays<4>) : (w8 ? k_all_hits<8> : k_all_hits<4>);
  hipLaunchKernelGGL(fn, dim3(grid), dim3(kAllBlock), lds, ctx->stream, a);
  HIP_TRY(hipGetLastError(), J3DG_ERR_LAUNCH);
  return J3DG_OK;
}

// Blocks of a voxel launch: those the GPU holds at once (four per CU, by the
// kernel's register bound and by LDS: 32,896 bytes a block), or fewer for few rays.
uint32_t vox_grid(uint32_t n, int n_cus) {
  return std::max(1u, std::min((n + kVoxGroups - 1) / kVoxGroups, (uint32_t)n_cus * 4u));
}

}  // namespace
}  // namespace j3d

using j3d::Ctx;
using j3d::Mesh;

extern "C" {

int j3dg_all_hits(j3dg_ctx* h, uint32_t slot, const float* rays, uint64_t n, uint32_t max_hits, uint32_t* counts,
                  uint32_t* tri, float* t, float* u, float* v) {
  Ctx* ctx = reinterpret_cast<Ctx*>(h);
  CHECK_CTX();
  if ((!rays || !counts) && n) return ctx->fail(J3DG_ERR_INVALID_ARG, "null rays or counts");
  if (slot >= ctx->meshes.size() || !ctx->meshes[slot].live) return ctx->fail(J3DG_ERR_NOT_FOUND, "unknown mesh slot");
  if (n > (1ull << 31)) return ctx->fail(J3DG_ERR_INVALID_ARG, "too many rays in one call");
  if (max_hits > 65536 || n * (uint64_t)max_hits > (1ull << 28))
    return ctx->fail(J3DG_ERR_INVALID_ARG, "n * max_hits exceeds 2^28 stored hits");
  if (n == 0) return J3DG_OK;
  HIP_CALL(hipSetDevice(ctx->device), J3DG_ERR_NO_DEVICE);
  const Mesh& m = ctx->meshes[slot];
  void* d_rays = ctx->scratch_buffer(0, n * 8 * sizeof(float));
  void* d_hits = ctx->scratch_buffer(1, n * max_hits * sizeof(j3d::HitRec));
  void* d_counts = ctx->scratch_buffer(2, n * sizeof(uint32_t));
  if (!d_rays || !d_hits || !d_counts) return ctx->fail(J3DG_ERR_OUT_OF_MEMORY, "all-hits buffers");
  HIP_CALL(hipMemcpyAsync(d_rays, rays, n * 8 * sizeof(float), hipMemcpyHostToDevice, ctx->stream),
           J3DG_ERR_LAUNCH);
  j3d::AllHitsArgs a;
  j3d::fill_mesh_args(m, a);
  a.rays = static_cast<const float*>(d_rays);
  a.n = (uint32_t)n;
  a.cap = max_hits;
  a.hits = static_cast<j3d::HitRec*>(d_hits);
  a.counts = static_cast<uint32_t*>(d_counts);
  int rc = j3d::launch_all_hits(ctx, m, a, (a.n + j3d::kAllBlock - 1) / j3d::kAllBlock, false);
  if (rc) return rc;
  HIP_CALL(hipMemcpyAsync(counts, d_counts, n * sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream),
           J3DG_ERR_LAUNCH);
  std::vector<j3d::HitRec> hits((size_t)n * max_hits);
  if (max_hits)
    HIP_CALL(hipMemcpyAsync(hits.data(), d_hits, hits.size() * sizeof(j3d::HitRec), hipMemcpyDeviceToHost,
                            ctx->stream),
             J3DG_ERR_LAUNCH);
  HIP_CALL(hipStreamSynchronize(ctx->stream), J3DG_ERR_LAUNCH);
  for (uint64_t i = 0; i < n; ++i)
    for (uint32_t k = 0; k < max_hits; ++k) {
      const size_t o = (size_t)i * max_hits + k;
      const bool has = k < counts[i];
      if (tri) tri[o] = has ? hits[o].tri : 0xFFFFFFFFu;
      if (t) t[o] = has ? hits[o].t : 0.f;
      if (u) u[o] = has ? hits[o].u : 0.f;
      if (v) v[o] = has ? hits[o].v : 0.f;
    }
  return J3DG_OK;
}

int j3dg_voxelize(j3dg_ctx* h, uint32_t slot, uint32_t max_dim, uint32_t dim[3], uint8_t* data, uint64_t capacity) {
  Ctx* ctx = reinterpret_cast<Ctx*>(h);
  CHECK_CTX();
  if (!dim) return ctx->fail(J3DG_ERR_INVALID_ARG, "null dim");
  if (slot >= ctx->meshes.size() || !ctx->meshes[slot].live) return ctx->fail(J3DG_ERR_NOT_FOUND, "unknown mesh slot");
  if (max_dim == 0 || max_dim > j3d::kMaxVoxDim) return ctx->fail(J3DG_ERR_INVALID_ARG, "max_dim must be 1 .. 1024");
  const Mesh& m = ctx->meshes[slot];
  j3d::vox_dims(m.info.bb_min, m.info.bb_max, max_dim, dim);
  const uint64_t nvox = (uint64_t)dim[0] * dim[1] * dim[2];
  if (!data) return J3DG_OK;
  if (capacity < nvox) return ctx->fail(J3DG_ERR_INVALID_ARG, "voxel buffer smaller than dim[0] * dim[1] * dim[2]");
  HIP_CALL(hipSetDevice(ctx->device), J3DG_ERR_NO_DEVICE);
  // scratch 0: keys, then the uint8 grid after them; 1: hit lists; 2: the overflow count
  void* d_keys = ctx->scratch_buffer(0, nvox * sizeof(unsigned long long) + nvox);
  void* d_max = ctx->scratch_buffer(2, sizeof(uint32_t));
  if (!d_keys || !d_max) return ctx->fail(J3DG_ERR_OUT_OF_MEMORY, "voxel buffers");
  uint8_t* d_data = static_cast<uint8_t*>(d_keys) + nvox * sizeof(unsigned long long);
  HIP_CALL(hipMemsetAsync(d_keys, 0, nvox * sizeof(unsigned long long), ctx->stream), J3DG_ERR_LAUNCH);
  j3d::AllHitsArgs a;
  j3d::fill_mesh_args(m, a);
  for (int k = 0; k < 3; ++k) a.dim[k] = dim[k], a.bmin[k] = m.info.bb_min[k], a.bmax[k] = m.info.bb_max[k];
  a.keys = static_cast<unsigned long long*>(d_keys);
  a.max_count = static_cast<uint32_t*>(d_max);
  // texture over vertex colours over white (j3d/vox.cpp:301-304)
  if (m.d_uv && m.d_tex && m.tex_w && m.tex_h) {
    a.color_mode = 2, a.uv = m.d_uv, a.tex = m.d_tex, a.tex_w = m.tex_w, a.tex_h = m.tex_h;
  } else if (m.d_vcol) {
    a.color_mode = 1, a.vcol = m.d_vcol;
  }
  // the three axes' rays in one launch: x rays, then y, then z
  a.axis_first[0] = 0;
  a.axis_first[1] = dim[1] * dim[2];
  a.axis_first[2] = a.axis_first[1] + dim[2] * dim[0];
  const uint32_t n = a.axis_first[2] + dim[0] * dim[1];
  const uint32_t grid = j3d::vox_grid(n, ctx->n_cus);
  uint32_t cap = 32;  // a power of two (sort_list pads to one)
  for (;;) {
    void* d_hits = ctx->scratch_buffer(1, (size_t)grid * j3d::kVoxGroups * cap * sizeof(j3d::HitRec));
    if (!d_hits) return ctx->fail(J3DG_ERR_OUT_OF_MEMORY, "voxel hit lists");
    HIP_CALL(hipMemsetAsync(d_max, 0, sizeof(uint32_t), ctx->stream), J3DG_ERR_LAUNCH);
    a.n = n;
    a.cap = cap;
    a.hits = static_cast<j3d::HitRec*>(d_hits);
    int rc = j3d::launch_all_hits(ctx, m, a, grid, true);
    if (rc) return rc;
    uint32_t mc = 0;
    HIP_CALL(hipMemcpyAsync(&mc, d_max, sizeof(mc), hipMemcpyDeviceToHost, ctx->stream), J3DG_ERR_LAUNCH);
    HIP_CALL(hipStreamSynchronize(ctx->stream), J3DG_ERR_LAUNCH);
    if (mc <= cap) break;
    if (mc > j3d::kMaxVoxHits) return ctx->fail(J3DG_ERR_UNSUPPORTED, "more than 2^24 hits on one voxel ray");
    while (cap < mc) cap *= 2;  // the rays that fitted wrote their voxels already; writing them again is harmless
  }
  const uint32_t blocks = (uint32_t)std::min<uint64_t>((nvox + 255) / 256, 65536);
  hipLaunchKernelGGL(j3d::k_vox_final, dim3(blocks), dim3(256), 0, ctx->stream,
                     (const unsigned long long*)d_keys, nvox, d_data);
  HIP_CALL(hipGetLastError(), J3DG_ERR_LAUNCH);
  HIP_CALL(hipMemcpyAsync(data, d_data, nvox, hipMemcpyDeviceToHost, ctx->stream), J3DG_ERR_LAUNCH);
  HIP_CALL(hipStreamSynchronize(ctx->stream), J3DG_ERR_LAUNCH);
  return J3DG_OK;
}

}  // extern "C"
