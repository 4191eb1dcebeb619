// Closest-point queries of librmh: for a batch of query points, the nearest point of the
// map strictly within max_distance.  Replaces EmbreeMap::closestPoint / EmbreeScene::closestPoint
// (src/rmagine_embree/src/map/EmbreeMap.cpp:33-37, src/rmagine_embree/src/map/embree/EmbreeScene.cpp:292-315)
// and its point-query callback (EmbreeMesh.cpp:22-131: closest point of a triangle,
// result {d, p, n, primID, geomID}, updated while d < the query radius).
//
// One lane per query.  A bound first (one descent to the nearer child at every level and
// that leaf's triangles), then a depth-first BVH walk, nearer child first; a subtree is
// skipped when its (outward padded) box lies farther than the bound.  Everything in the walk
// is FP32 with proven margins (rmh_closest_bounds.hpp): a triangle gives a lower and an upper
// bound of its distance, the upper ones shrink the search, and the triangles whose lower
// bound does not exceed it are listed.  The list (6 slots per lane in LDS, emptied when a
// closer triangle outdates all of it) is evaluated in FP64 at the end, when all lanes are
// there, or when a triangle is to be listed and it is full or ends with a degenerate triangle or
// sliver, which have no bounds: the triangle's closest point (Ericson, Real-Time Collision
// Detection, 5.1.5: Voronoi regions of the vertices, edges and face) and its distance, so the
// result is the FP64 nearest triangle; equal distances go to the lower global face index.
// Evaluated in the leaves, the FP64 code ran for nearly every triangle, for one or two lanes
// of the wave each time (44 triangles per query on the terrain, 6.7 of them closer than what
// was known; 1.6 evaluations now).  Outputs per query (each pointer may be NULL): distance
// (FLT_MAX when nothing lies within max_distance), closest point, unit face normal (not
// flipped), face id within its mesh, geom id, object id (0xFFFFFFFF for none; point and
// normal NaN).
//
// The lanes of a wave walk nodes together until half of those still searching hold a leaf,
// then test their leaves together (terrain, 1M queries, FP64 evaluation still in the leaves:
// 1.95 ms; waiting for a third 2.03, a quarter 2.12, an eighth 2.38, for all of them 3.19;
// node and leaf steps mixed in one loop, as at first, 2.93).  The walk is bound by its chain of
// dependent node and triangle loads and by the spread of the work between the lanes (on the
// terrain 72 nodes per query, 146 for a wave's slowest): 4M queries now take 4.4 ms instead
// of 8.0, 1M 1.73 instead of 2.93, 1M between scattered objects 1.22 instead of 1.72.  The
// walk's stack is the ray kernels' (rmh_trace.hpp): the top rows in LDS, deeper entries in
// private memory.
//
// Lanes of a wave that walk unrelated parts of the tree fetch its nodes separately: random
// query sets fetch about 3x the node bytes of the same points in spatial order.  Batches of
// at least kSortQueries queries are therefore sorted by the Morton code of their positions in
// the map's bounding box (30-bit codes, on the device, in stream-ordered scratch), and walked
// in that order when a sample of their waves spans kSpreadRatio times less space in it than
// in the caller's order (the walk then reads queries and writes results scattered, which
// costs a walk in an already coherent order more than it gains).  Each lane reads and writes
// its own query's slots, so the results do not depend on the order.  Under stream capture,
// or when the scratch cannot be had, the batch is walked in the caller's order.  The scratch
// (17 B per query) comes from the library's pool (scratch_pool).
#include "rmh_closest_bounds.hpp"
#include "rmh_trace.hpp"

#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <cfloat>

namespace {

using namespace rmh;

struct CPArgs {
  MapData map;
  const rmh_vec3* q;
  const uint32_t* order;  // lane i takes query order[i] when the spread test below holds
  const float* spread;    // summed wave extents of a sample: [0] caller's order, [1] sorted
  uint32_t n;
  uint32_t per_wave;      // queries per wave, one lane each
  double best0;  // max_distance^2: a result needs d^2 < best0
  rmh_closest_outputs out;
};

// 12 LDS stack rows and 6 candidate slots (7.5 KB per wave) keep the five waves per SIMD that
// the registers allow (terrain, 1M queries: 1.70 ms; 10 rows 1.79, 16 rows and four waves 1.98;
// 4 slots 1.72 there but 1.48 instead of 1.29 ms between scattered objects, where the list
// overflows more often; 8 slots 1.77).
constexpr int kClosestLds = 12;
constexpr uint32_t kCand = 6;
// Waves of consecutive queries are dealt to the XCDs 64 at a time, so that an XCD's L2 keeps a
// region's nodes and triangles (contiguous ranges per XCD: terrain 1.70 ms against 1.73, but a
// room, whose regions differ in cost, 0.43 ms against 0.39; round-robin waves 1.87 and 0.39).
constexpr uint32_t kDealt = 64;
// One lane per query, 64 queries per wave, or fewer while that leaves at most 3 waves per
// SIMD: with the chip that empty, a wave's walk is as long as its slowest query's and its
// loads touch fewer lines (1,000 queries on the terrain: 64 per wave 366 us, 1 per wave 290;
// 16,000: 574, 8 per wave 496; 60,000: 551, 32 per wave 541; at 4 waves per SIMD 60,000
// queries in a room took 112 us instead of 102).
constexpr uint32_t kSparseWaves = 3072;
constexpr float kSpreadRatio = 4.0f;

// FP32 value at least the squared distance d2 (infinite for those beyond FP32).
__device__ __forceinline__ float upper_f32(double d2) { return __double2float_ru(d2); }

template <int STACK>
__global__ __launch_bounds__(64, 5) void k_closest(const CPArgs a) {
  __shared__ int2 stk[kClosestLds][64];
  __shared__ uint32_t cand[kCand][64];
  const uint32_t lane_q = xcd_dealt<kDealt>(blockIdx.x, gridDim.x) * a.per_wave + threadIdx.x;
  if (threadIdx.x >= a.per_wave || lane_q >= a.n) return;
  const bool reorder = a.order && a.spread[1] * kSpreadRatio < a.spread[0];
  const uint32_t i = reorder ? a.order[lane_q] : lane_q;
  const rmh_vec3 qv = a.q[i];
  const F3 qf{qv.x, qv.y, qv.z};
  // The walk runs on FP32 bounds: `upper` is at least the smallest squared distance met so
  // far (and at most about best0), and the triangles that may hold it are listed in LDS
  // (`cand`), to be evaluated in FP64 together at the end, or when the list is full.  A
  // triangle is dropped only when its lower bound exceeds `upper`, which only triangles shrink
  // whose FP64 distance does not exceed it, so every triangle at the smallest FP64 distance is
  // evaluated.
  double best = a.best0;
  uint32_t best_slot = 0xFFFFFFFFu, best_face = 0xFFFFFFFFu;
  float upper = upper_f32(best);
  float bound = walk_bound(upper);      // boxes beyond it hold nothing nearer
  float least = __builtin_inff();       // least lower bound of the listed triangles
  uint32_t n_cand = 0;
  bool thin = false;                    // the last listed triangle has no upper bound
  auto evaluate = [&]() {
    const D3 q = d3(qv.x, qv.y, qv.z);
    for (uint32_t k = 0; k < n_cand; k++) {
      const uint32_t slot = cand[k][threadIdx.x];
      const size_t s = static_cast<size_t>(slot) * 3;
      const float4 v0 = a.map.tris[s], v1 = a.map.tris[s + 1], v2 = a.map.tris[s + 2];
      const D3 p = closest_on_triangle(q, d3(v0.x, v0.y, v0.z), d3(v1.x, v1.y, v1.z), d3(v2.x, v2.y, v2.z));
      const D3 dv = sub(p, q);
      const double d2 = ddot(dv, dv);
      const uint32_t face = __float_as_uint(v2.w);
      if (d2 < best || (d2 == best && best_slot != 0xFFFFFFFFu && face < best_face)) {
        best = d2;
        best_slot = slot;
        best_face = face;
      }
    }
    n_cand = 0;
    least = __builtin_inff();
  };
  volatile int spill_mem[STACK > kClosestLds ? 2 * (STACK - kClosestLds) : 2];
  PrivInt* spill = (PrivInt*)spill_mem;
  int sp = 0;
  // the triangles of leaf reference `leaf` against the query
  auto leaf_test = [&](int leaf) {
    const uint32_t e = ~static_cast<uint32_t>(leaf);
    const uint32_t first = e >> 3, cnt = (e & 7u) + 1u;
    for (uint32_t k = 0; k < cnt; k++) {
      const size_t s = static_cast<size_t>(first + k) * 3;
      const float4 v0 = a.map.tris[s], v1 = a.map.tris[s + 1], v2 = a.map.tris[s + 2];
      const D2Bounds d = triangle_bounds(fsub(F3{v0.x, v0.y, v0.z}, qf), fsub(F3{v1.x, v1.y, v1.z}, qf),
                                         fsub(F3{v2.x, v2.y, v2.z}, qf));
      if (d.lo > upper) continue;
      if (d.hi < upper) {
        upper = d.hi;
        if (upper < least) { n_cand = 0; least = __builtin_inff(); }
      }
      // A triangle without an upper bound shrinks the search by its FP64 distance when the next
      // one is listed; left in the list, it did so only when the list overflowed, lane by lane
      // (200,000 queries around a fan of 3,000 thin triangles 13.5 ms, 7.9 so, 7.4 with every
      // triangle in FP64; a fan of 100,000 529, 313 and 313; 50,000 needles 0.21, 0.22 and 0.23).
      // Evaluated as it is listed, which fills the list at six: fan 8.2 ms, but 200,000 to
      // 600,000 queries in a room of 50k triangles 8 % slower; at the end of the leaf, in code of
      // its own: small batches 2-5 % slower; with the shape asked for before the bounds are
      // formed: fan 6.8 ms, but 1M terrain queries 3-6 % slower.
      if (n_cand == kCand || thin) {
        evaluate();
        upper = fminf(upper, upper_f32(best));
      }
      cand[n_cand][threadIdx.x] = first + k;
      n_cand++;
      least = fminf(least, d.lo);
      thin = !(d.hi < __builtin_inff());
    }
    bound = walk_bound(upper);
  };
  int ref = kDone;
  if (a.map.n_faces) {
    // a bound before the walk: one descent to the nearer child at every level, then that
    // leaf's triangles.  Without it the walk starts unbounded and pushes the farther child
    // at every level of its first descent, deeper than the LDS rows hold.  The walk tests
    // that leaf again, which changes nothing (same distance, same face).
    int g = a.map.root;
    while (g >= 0) {
      const Node2 nd = a.map.nodes[g];
      const float b0 = box_d2(qf, nd.a.x, nd.a.y, nd.a.z, nd.a.w, nd.c.x, nd.c.y);
      const float b1 = box_d2(qf, nd.b.x, nd.b.y, nd.b.z, nd.b.w, nd.c.z, nd.c.w);
      g = b0 <= b1 ? nd.d.x : nd.d.y;
    }
    leaf_test(g);
    if (thin) {  // a bound from slivers too: without it 50,000 needles take 0.27 ms
      evaluate();
      upper = fminf(upper, upper_f32(best));
      bound = walk_bound(upper);
      thin = false;
    }
    n_cand = 0;  // the walk meets that leaf again
    least = __builtin_inff();
    ref = a.map.root;
  }
  for (;;) {
    for (;;) {
      const uint64_t walking = __ballot(ref >= 0 && ref != kDone), holding = __ballot(ref < 0);
      if (walking == 0 || 2 * __popcll(holding) >= __popcll(walking | holding)) break;
      if (ref >= 0 && ref != kDone) {
        const Node2 nd = a.map.nodes[ref];
        const float b0 = box_d2(qf, nd.a.x, nd.a.y, nd.a.z, nd.a.w, nd.c.x, nd.c.y);
        const float b1 = box_d2(qf, nd.b.x, nd.b.y, nd.b.z, nd.b.w, nd.c.z, nd.c.w);
        const bool h0 = b0 <= bound, h1 = b1 <= bound;
        if (h0 && h1) {
          // one entry per level: the host picks STACK >= tree depth
          const bool first0 = b0 <= b1;
          push_ref<STACK, 64, kClosestLds, true>(stk, spill, sp, first0 ? nd.d.y : nd.d.x, first0 ? b1 : b0);
          ref = first0 ? nd.d.x : nd.d.y;
        } else if (h0) {
          ref = nd.d.x;
        } else if (h1) {
          ref = nd.d.y;
        } else {
          ref = pop_ref<STACK, 64, kClosestLds, true>(stk, spill, sp, bound);
        }
      }
    }
    if (__ballot(ref < 0) == 0) break;
    if (ref < 0) {
      leaf_test(ref);
      ref = pop_ref<STACK, 64, kClosestLds, true>(stk, spill, sp, bound);
    }
  }
  evaluate();
  const rmh_closest_outputs& o = a.out;
  if (best_slot != 0xFFFFFFFFu) {
    const size_t s = static_cast<size_t>(best_slot) * 3;
    const float4 nn = a.map.normals[best_slot];
    D3 best_p = d3(0, 0, 0);
    if (o.points) {  // evaluated again rather than held through the walk
      const float4 v0 = a.map.tris[s], v1 = a.map.tris[s + 1], v2 = a.map.tris[s + 2];
      best_p = closest_on_triangle(d3(qv.x, qv.y, qv.z), d3(v0.x, v0.y, v0.z), d3(v1.x, v1.y, v1.z), d3(v2.x, v2.y, v2.z));
    }
    if (o.dist) o.dist[i] = static_cast<float>(sqrt(best));
    if (o.points) { rmh_vec3 v; v.x = (float)best_p.x; v.y = (float)best_p.y; v.z = (float)best_p.z; o.points[i] = v; }
    if (o.normals) { rmh_vec3 v; v.x = nn.x; v.y = nn.y; v.z = nn.z; o.normals[i] = v; }
    if (o.face_ids) o.face_ids[i] = __float_as_uint(a.map.tris[s].w);
    if (o.geom_ids) o.geom_ids[i] = __float_as_uint(a.map.tris[s + 1].w);
    if (o.object_ids) o.object_ids[i] = __float_as_uint(nn.w);
  } else {
    const float qnan = __builtin_nanf("");
    rmh_vec3 v; v.x = qnan; v.y = qnan; v.z = qnan;
    if (o.dist) o.dist[i] = FLT_MAX;
    if (o.points) o.points[i] = v;
    if (o.normals) o.normals[i] = v;
    if (o.face_ids) o.face_ids[i] = 0xFFFFFFFFu;
    if (o.geom_ids) o.geom_ids[i] = 0xFFFFFFFFu;
    if (o.object_ids) o.object_ids[i] = 0xFFFFFFFFu;
  }
}

constexpr uint32_t kSortQueries = 1u << 16;

// Spreads the low 10 bits of v to every third bit.
__device__ __forceinline__ uint32_t spread3(uint32_t v) {
  v &= 0x3FFu;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

// 30-bit Morton code of each query's cell in a grid of cubic cells, 1024 along the longest
// side of the root's box (queries outside it clamp to the border cells; cubic cells keep a
// wave's queries in a compact region of a flat map, not a thin slab), and the identity
// permutation beside it.
__global__ __launch_bounds__(256) void k_query_keys(const Node2* nodes, int root, const rmh_vec3* q, uint32_t n,
                                                   uint32_t* keys, uint32_t* idx, float* spread) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i == 0) { spread[0] = 0.0f; spread[1] = 0.0f; }
  if (i >= n) return;
  const Node2 r = nodes[root];
  const float lx = fminf(r.a.x, r.b.x), hx = fmaxf(r.a.y, r.b.y);
  const float ly = fminf(r.a.z, r.b.z), hy = fmaxf(r.a.w, r.b.w);
  const float lz = fminf(r.c.x, r.c.z), hz = fmaxf(r.c.y, r.c.w);
  const float scale = 1024.0f / fmaxf(fmaxf(fmaxf(hx - lx, hy - ly), hz - lz), 1e-30f);
  const rmh_vec3 p = q[i];
  auto cell = [scale](float v, float lo) {
    return static_cast<uint32_t>(fminf(fmaxf((v - lo) * scale, 0.0f), 1023.0f));  // NaN -> 0
  };
  keys[i] = spread3(cell(p.x, lx)) | (spread3(cell(p.y, ly)) << 1) | (spread3(cell(p.z, lz)) << 2);
  idx[i] = i;
}

constexpr uint32_t kSpreadWaves = 4096;

// Extent (x + y + z) of the queries of sampled waves, in the caller's order and in the
// sorted one, summed into spread[0] and spread[1].  Wave k of the grid takes the 64 queries
// from (k * stride) * 64; lanes past n repeat query n - 1, which belongs to the same wave.
__global__ __launch_bounds__(256) void k_order_spread(const rmh_vec3* q, const uint32_t* order, uint32_t n,
                                                     uint32_t stride, float* spread) {
  __shared__ float part[2][4];
  const uint32_t wave = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x & 63u;
  const uint64_t first = static_cast<uint64_t>(wave) * stride * 64;
  float ext[2] = {0.0f, 0.0f};
  if (first < n) {
    const uint32_t j = first + lane < n ? static_cast<uint32_t>(first + lane) : n - 1;
    const rmh_vec3 pts[2] = {q[j], q[order[j]]};
    for (int o = 0; o < 2; o++) {
      float lo[3] = {pts[o].x, pts[o].y, pts[o].z}, hi[3] = {pts[o].x, pts[o].y, pts[o].z};
      for (int m = 32; m >= 1; m >>= 1)
        for (int c = 0; c < 3; c++) {
          lo[c] = fminf(lo[c], __shfl_xor(lo[c], m, 64));
          hi[c] = fmaxf(hi[c], __shfl_xor(hi[c], m, 64));
        }
      ext[o] = (hi[0] - lo[0]) + (hi[1] - lo[1]) + (hi[2] - lo[2]);
      if (!(ext[o] <= FLT_MAX)) ext[o] = FLT_MAX;  // NaN or overflow
    }
  }
  if (lane == 0) { part[0][threadIdx.x / 64] = ext[0]; part[1][threadIdx.x / 64] = ext[1]; }
  __syncthreads();
  if (threadIdx.x < 2) {
    const float v = part[threadIdx.x][0] + part[threadIdx.x][1] + part[threadIdx.x][2] + part[threadIdx.x][3];
    atomicAdd(&spread[threadIdx.x], v);
  }
}

// Morton order of the queries in `scratch` (stream-ordered; freed by the caller after the
// walk) and the spread sums that decide whether the walk takes it, or NULL when the batch is
// walked in the caller's order.
uint32_t* query_order(const rmh_map* map, const rmh_vec3* q, uint32_t n, hipStream_t s, void** scratch,
                      const float** spread_out) {
  *scratch = nullptr;
  if (n < kSortQueries || map->root < 0 || map->n_faces == 0) return nullptr;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return nullptr;
  }
  size_t tmp_bytes = 0;
  if (rocprim::radix_sort_pairs(nullptr, tmp_bytes, static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr),
                                static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr), n, 0u, 30u,
                                s) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  const size_t arr = (static_cast<size_t>(n) * sizeof(uint32_t) + 255) & ~static_cast<size_t>(255);
  hipMemPool_t pool = scratch_pool(map->device);
  if (!pool || hipMallocFromPoolAsync(scratch, 4 * arr + 256 + tmp_bytes, pool, s) != hipSuccess) {
    (void)hipGetLastError();
    *scratch = nullptr;
    return nullptr;
  }
  char* base = static_cast<char*>(*scratch);
  uint32_t* keys = reinterpret_cast<uint32_t*>(base);
  uint32_t* keys2 = reinterpret_cast<uint32_t*>(base + arr);
  uint32_t* idx = reinterpret_cast<uint32_t*>(base + 2 * arr);
  uint32_t* order = reinterpret_cast<uint32_t*>(base + 3 * arr);
  float* spread = reinterpret_cast<float*>(base + 4 * arr);
  const uint32_t waves = (n + 63) / 64, sampled = std::min(waves, kSpreadWaves);
  const uint32_t stride = waves / sampled;  // >= 1; sampled * stride <= waves
  k_query_keys<<<(n + 255) / 256, 256, 0, s>>>(map->nodes, map->root, q, n, keys, idx, spread);
  bool ok = hipGetLastError() == hipSuccess &&
            rocprim::radix_sort_pairs(base + 4 * arr + 256, tmp_bytes, keys, keys2, idx, order, n, 0u, 30u, s) ==
                hipSuccess;
  if (ok) {
    k_order_spread<<<(sampled + 3) / 4, 256, 0, s>>>(q, order, n, stride, spread);
    ok = hipGetLastError() == hipSuccess;
  }
  if (!ok) {
    (void)hipGetLastError();
    (void)hipFreeAsync(*scratch, s);
    *scratch = nullptr;
    return nullptr;
  }
  *spread_out = spread;
  return order;
}

}  // namespace

extern "C" int rmh_closest_points(const rmh_map* map, const rmh_vec3* queries, uint32_t n, float max_distance,
                                  const rmh_closest_outputs* out, void* stream) {
  if (!map) return fail(RMH_ERR_NOMAP, "rmh_closest_points: no map set");
  if (!out) return fail(RMH_ERR_INVALID, "rmh_closest_points: NULL outputs");
  if (n == 0) return RMH_OK;
  if (!queries) return fail(RMH_ERR_INVALID, "rmh_closest_points: NULL queries");
  if (!(max_distance >= 0.0f)) return fail(RMH_ERR_INVALID, "rmh_closest_points: max_distance must be >= 0");
  if (map->info.max_depth > 128) return fail(RMH_ERR_UNSUPPORTED, "rmh_closest_points: BVH deeper than 128 levels");
  CPArgs a;
  a.map.tris = map->tris;
  a.map.normals = map->normals;
  a.map.nodes = map->nodes;
  a.map.root = map->root;
  a.map.n_faces = map->n_faces;
  a.q = queries;
  a.n = n;
  a.best0 = static_cast<double>(max_distance) * static_cast<double>(max_distance);
  a.out = *out;
  a.per_wave = 64;
  while (a.per_wave > 1 && (n + a.per_wave / 2 - 1) / (a.per_wave / 2) <= kSparseWaves) a.per_wave /= 2;
  const uint32_t blocks = (n + a.per_wave - 1) / a.per_wave;
  hipStream_t s = static_cast<hipStream_t>(stream);
  void* scratch = nullptr;
  a.spread = nullptr;
  a.order = query_order(map, queries, n, s, &scratch, &a.spread);
  const uint32_t depth = map->info.max_depth;
  if (depth <= 32) k_closest<32><<<blocks, 64, 0, s>>>(a);
  else if (depth <= 64) k_closest<64><<<blocks, 64, 0, s>>>(a);
  else k_closest<128><<<blocks, 64, 0, s>>>(a);
  const hipError_t e = hipGetLastError();
  if (scratch) RMH_HIP_TRY(hipFreeAsync(scratch, s));
  RMH_HIP_TRY(e);
  return RMH_OK;
}
