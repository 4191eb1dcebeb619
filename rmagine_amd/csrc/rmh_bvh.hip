// GPU BVH builder of librmh: the role of OptixScene's GAS build
// (src/rmagine_optix/src/map/optix/OptixScene.cpp:230-379) and EmbreeScene::commit
// (src/rmagine_embree/src/map/embree/EmbreeScene.cpp:187-191).
//
// Steps, all on the device:
//   1. per face: bounds, centroid, scene centroid bounds (wave64 shuffle + one atomic
//      per block), face-index validation;
//   2. 63-bit Morton codes of the centroids;
//   3. radix sort of (code, face) pairs (rocPRIM);
//   4. Karras 2012 radix tree over the sorted codes (index-augmented for duplicates);
//   4b. SAH refinement: three bottom-up rounds of treelet restructuring (Karras and Aila,
//      HPG 2013; rmh_treelet.hpp), then depth-first renumbering of the leaves so that
//      every subtree is one range of the triangle array again;
//   5. bottom-up pass: node boxes, primitive counts and the area-weighted SAH cost; a
//      subtree of at most max_leaf_size triangles becomes a leaf when that is cheaper
//      under SAH.  The bottom-up passes (4b, 5) run one launch per tree depth, deepest
//      first, over the interior nodes sorted by depth (make_levels);
//   6. layout: 64-byte binary nodes that hold both child boxes (padded outward), plus
//      depth statistics of the reachable tree;
//   7. gather of the triangles in Morton order (3 x float4 per triangle with the face,
//      geometry and global ids in the w lanes) and of FP64-derived unit face normals.
// The normals play the part of EmbreeMesh::computeFaceNormals
// (src/rmagine_embree/src/map/embree/EmbreeMesh.cpp:275-295) and of
// computeFaceNormals_kernel (src/rmagine_cuda/src/map/mesh_preprocessing.cu:6-20).
#include "rmh_internal.hpp"
#include "rmh_treelet.hpp"

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <new>
#include <utility>
#include <vector>

namespace {

using namespace rmh;

constexpr int kBlock = 256;
constexpr uint32_t kWideBlocks = 2048;  // grid-stride passes: eight blocks per CU
constexpr uint32_t kLeafBit = kTreeLeafBit;
constexpr int kTreeletRounds = 3;
// largest map: node references must stay below 2^26 (32-bit node byte offsets in the ray kernels)
constexpr uint32_t kMaxFaces = 1u << 26;

__device__ inline void atomic_min_float(float* addr, float v) {
  if (v >= 0.0f) atomicMin(reinterpret_cast<int*>(addr), __float_as_int(v));
  else atomicMax(reinterpret_cast<unsigned int*>(addr), __float_as_uint(v));
}

__device__ inline void atomic_max_float(float* addr, float v) {
  if (v >= 0.0f) atomicMax(reinterpret_cast<int*>(addr), __float_as_int(v));
  else atomicMin(reinterpret_cast<unsigned int*>(addr), __float_as_uint(v));
}

__device__ inline float wave_min(float v) {
  for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off, 64));
  return v;
}

__device__ inline float wave_max(float v) {
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

__global__ void k_init(float* bounds, uint32_t* err) {
  if (threadIdx.x < 3) bounds[threadIdx.x] = FLT_MAX;
  else if (threadIdx.x < 6) bounds[threadIdx.x] = -FLT_MAX;
  else if (threadIdx.x == 6) *err = 0u;
}

// Step 1.  At most kWideBlocks blocks: the bounds' atomics go to six addresses, and with a
// block per 256 faces they took most of its 0.33 ms on the 2.1M-triangle terrain.
__global__ __launch_bounds__(kBlock) void k_prep(const float* __restrict__ V, uint32_t nv,
                                                 const uint32_t* __restrict__ F, uint32_t nf,
                                                 float4* __restrict__ lo, float4* __restrict__ hi,
                                                 float* bounds, uint32_t* err) {
  float cmin[3] = {FLT_MAX, FLT_MAX, FLT_MAX};
  float cmax[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
  uint32_t bad = 0;
  for (uint32_t f = blockIdx.x * kBlock + threadIdx.x; f < nf; f += gridDim.x * kBlock) {
    uint32_t idx[3] = {F[3 * f + 0], F[3 * f + 1], F[3 * f + 2]};
    for (int k = 0; k < 3; k++) {
      if (idx[k] >= nv) { bad |= 1u; idx[k] = 0; }
    }
    float b0[3], b1[3];
    for (int a = 0; a < 3; a++) {
      const float x0 = V[3 * idx[0] + a], x1 = V[3 * idx[1] + a], x2 = V[3 * idx[2] + a];
      b0[a] = fminf(x0, fminf(x1, x2));
      b1[a] = fmaxf(x0, fmaxf(x1, x2));
      if (!(isfinite(x0) && isfinite(x1) && isfinite(x2))) bad |= 2u;
      const float c = 0.5f * b0[a] + 0.5f * b1[a];
      cmin[a] = fminf(cmin[a], c);
      cmax[a] = fmaxf(cmax[a], c);
    }
    lo[f] = make_float4(b0[0], b0[1], b0[2], 0.0f);
    hi[f] = make_float4(b1[0], b1[1], b1[2], 0.0f);
  }
  if (bad) atomicOr(err, bad);
  __shared__ float red[2][3][kBlock / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int a = 0; a < 3; a++) {
    const float mn = wave_min(cmin[a]), mx = wave_max(cmax[a]);
    if (lane == 0) { red[0][a][wid] = mn; red[1][a][wid] = mx; }
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int a = threadIdx.x;
    float mn = red[0][a][0], mx = red[1][a][0];
    for (int w = 1; w < kBlock / 64; w++) { mn = fminf(mn, red[0][a][w]); mx = fmaxf(mx, red[1][a][w]); }
    atomic_min_float(&bounds[a], mn);
    atomic_max_float(&bounds[3 + a], mx);
  }
}

// Step 2.
__global__ __launch_bounds__(kBlock) void k_morton(const float4* __restrict__ lo, const float4* __restrict__ hi,
                                                   uint32_t nf, const float* __restrict__ bounds,
                                                   uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
  if (f >= nf) return;
  const float4 a = lo[f], b = hi[f];
  const float l[3] = {a.x, a.y, a.z}, h[3] = {b.x, b.y, b.z};
  const float bmin[3] = {bounds[0], bounds[1], bounds[2]};
  const float ext = fmaxf(fmaxf(bounds[3] - bounds[0], bounds[4] - bounds[1]), bounds[5] - bounds[2]);
  keys[f] = morton_key(l, h, bmin, ext);
  vals[f] = f;
}

// Step 4 (karras_node: Karras 2012, Fig. 4).
__global__ __launch_bounds__(kBlock) void k_karras(const uint64_t* __restrict__ keys, int n,
                                                   uint32_t* __restrict__ child, uint32_t* __restrict__ range,
                                                   int* __restrict__ parent_int, int* __restrict__ parent_leaf) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n - 1) return;
  karras_node(keys, n, i, child, range, parent_int, parent_leaf);
}

__device__ inline float half_area(float4 a, float4 b) {
  const float dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z;
  return dx * dy + dy * dz + dz * dx;
}

// Step 5.  node_lo.w = SAH cost (area weighted), node_hi.w = primitive count.  One launch
// per depth of the radix tree, deepest first (make_levels): every node of the level reads
// its children, which earlier launches finished, so no arrival counters are needed (an
// agent-scope acquire-release atomic writes back and invalidates the L2 of an XCD each time,
// which made the counter-driven pass 7 ms on the 2.1M-triangle terrain).
__global__ __launch_bounds__(kBlock) void k_bottom_up_level(const uint32_t* __restrict__ order, uint32_t lo, uint32_t hi,
                                                            const uint32_t* __restrict__ vals,
                                                            const float4* __restrict__ flo, const float4* __restrict__ fhi,
                                                            const uint32_t* __restrict__ child,
                                                            float4* node_lo, float4* node_hi,
                                                            uint8_t* collapse, uint32_t* subtree,
                                                            uint32_t max_leaf, float c_node, float c_tri) {
  const uint32_t k = lo + blockIdx.x * kBlock + threadIdx.x;
  if (k >= hi) return;
  const uint32_t p = order[k];
  float4 lo2[2], hi2[2];
  float cost[2], cnt[2];
  uint32_t below = 0;  // interior nodes of the final tree in the children's subtrees
  for (int c = 0; c < 2; c++) {
    const uint32_t ch = child[2 * p + c];
    if (ch & kLeafBit) {
      const uint32_t f = vals[ch & ~kLeafBit];
      lo2[c] = flo[f];
      hi2[c] = fhi[f];
      cnt[c] = 1.0f;
      cost[c] = c_tri * half_area(lo2[c], hi2[c]);
    } else {
      lo2[c] = node_lo[ch];
      hi2[c] = node_hi[ch];
      cost[c] = lo2[c].w;
      cnt[c] = hi2[c].w;
      below += subtree[ch];
    }
  }
  float4 L = make_float4(fminf(lo2[0].x, lo2[1].x), fminf(lo2[0].y, lo2[1].y), fminf(lo2[0].z, lo2[1].z), 0.0f);
  float4 H = make_float4(fmaxf(hi2[0].x, hi2[1].x), fmaxf(hi2[0].y, hi2[1].y), fmaxf(hi2[0].z, hi2[1].z), 0.0f);
  const float count = cnt[0] + cnt[1];
  const float area = half_area(L, H);
  const float split_cost = c_node * area + cost[0] + cost[1];
  float node_cost = split_cost;
  uint8_t col = 0;
  if (count <= static_cast<float>(max_leaf)) {
    const float leaf_cost = c_tri * area * count;
    if (leaf_cost <= split_cost) { node_cost = leaf_cost; col = 1; }
  }
  L.w = node_cost;
  H.w = count;
  node_lo[p] = L;
  node_hi[p] = H;
  collapse[p] = col;
  subtree[p] = col ? 0u : 1u + below;  // a collapsed node becomes a leaf of the final tree
}

// Sort key of every interior node of the radix tree for the level-by-level passes: its
// depth (the root, node 0, has parent -1), deepest first, and within a depth the nodes
// that get a treelet (count >= gamma; none when count is NULL) before the others.  A parent
// chain that leaves the node range or runs longer than kMaxTreeWalk steps (a cycle) sets err
// bit 8.
__global__ __launch_bounds__(kBlock) void k_level_keys(int n, const int* __restrict__ parent_int,
                                                       const uint32_t* __restrict__ count, uint32_t gamma,
                                                       uint32_t* __restrict__ keys, uint32_t* __restrict__ idx,
                                                       uint32_t* err) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n - 1) return;
  uint32_t d = 0;
  for (int p = parent_int[i]; p >= 0; p = parent_int[p]) {
    if (++d > static_cast<uint32_t>(kMaxTreeWalk) || p >= n - 1) { atomicOr(err, 8u); d = 0; break; }
  }
  const bool need = count && count[i] >= gamma;
  keys[i] = 2u * (static_cast<uint32_t>(kMaxTreeWalk) - d) + (need ? 0u : 1u);
  idx[i] = static_cast<uint32_t>(i);
}

// start[key] = first position of `key` in the sorted keys (untouched for absent keys)
__global__ __launch_bounds__(kBlock) void k_level_starts(uint32_t ni, const uint32_t* __restrict__ skeys,
                                                         uint32_t* __restrict__ start) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= ni) return;
  if (i == 0 || skeys[i] != skeys[i - 1]) start[skeys[i]] = i;
}

// Triangles below every interior node of the radix tree: its range of sorted leaves.
__global__ __launch_bounds__(kBlock) void k_range_counts(uint32_t ni, const uint32_t* __restrict__ range,
                                                         uint32_t* __restrict__ count) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < ni) count[i] = range[2 * i + 1] - range[2 * i] + 1u;
}

// Outward padding so that the FP32 slab test stays conservative for boxes of zero
// thickness and for values that are not exactly representable after subtraction.
__device__ inline float pad_lo(float x) { return x - fabsf(x) * 2.4e-7f - 1e-30f; }
__device__ inline float pad_hi(float x) { return x + fabsf(x) * 2.4e-7f + 1e-30f; }

// Step 6.  Grid-stride, so that the node count and depth take two atomics per block of at most
// kWideBlocks (two per reachable node took most of its 0.78 ms).
__global__ __launch_bounds__(kBlock) void k_layout(int n, const uint32_t* __restrict__ vals,
                                                   const float4* __restrict__ flo, const float4* __restrict__ fhi,
                                                   const uint32_t* __restrict__ child, const uint32_t* __restrict__ range,
                                                   const int* __restrict__ parent_int,
                                                   const float4* __restrict__ node_lo, const float4* __restrict__ node_hi,
                                                   const uint8_t* __restrict__ collapse, Node2* __restrict__ nodes,
                                                   uint32_t* stats /* [0]=reachable interior, [1]=max depth */,
                                                   uint8_t* __restrict__ reach) {
  uint32_t found = 0, deepest = 0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n - 1; i += gridDim.x * kBlock) {
    float4 lo[2], hi[2];
    int ref[2];
    for (int c = 0; c < 2; c++) {
      const uint32_t ch = child[2 * i + c];
      if (ch & kLeafBit) {
        const uint32_t k = ch & ~kLeafBit;
        const uint32_t f = vals[k];
        lo[c] = flo[f];
        hi[c] = fhi[f];
        ref[c] = make_leaf_ref(k, 1u);
      } else {
        lo[c] = node_lo[ch];
        hi[c] = node_hi[ch];
        if (collapse[ch]) {
          const uint32_t first = range[2 * ch], last = range[2 * ch + 1];
          ref[c] = make_leaf_ref(first, last - first + 1u);
        } else {
          ref[c] = static_cast<int>(ch);
        }
      }
    }
    Node2 nd;
    nd.a = make_float4(pad_lo(lo[0].x), pad_hi(hi[0].x), pad_lo(lo[0].y), pad_hi(hi[0].y));
    nd.b = make_float4(pad_lo(lo[1].x), pad_hi(hi[1].x), pad_lo(lo[1].y), pad_hi(hi[1].y));
    nd.c = make_float4(pad_lo(lo[0].z), pad_hi(hi[0].z), pad_lo(lo[1].z), pad_hi(hi[1].z));
    nd.d = make_int4(ref[0], ref[1], 0, 0);
    nodes[i] = nd;
    // reachable iff neither this node nor an ancestor became a leaf
    bool reachable = collapse[i] == 0;
    uint32_t depth = 0;
    int p = i;
    while (reachable && p != 0) {
      p = parent_int[p];
      depth++;
      if (collapse[p]) reachable = false;
    }
    reach[i] = reachable ? 1 : 0;
    if (reachable) {
      found++;
      deepest = max(deepest, depth + 1u);
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    found += __shfl_xor(found, off, 64);
    deepest = max(deepest, static_cast<uint32_t>(__shfl_xor(deepest, off, 64)));
  }
  __shared__ uint32_t red[2][kBlock / 64];
  if ((threadIdx.x & 63) == 0) { red[0][threadIdx.x >> 6] = found; red[1][threadIdx.x >> 6] = deepest; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kBlock / 64; w++) { found += red[0][w]; deepest = max(deepest, red[1][w]); }
    if (found > 0) {
      atomicAdd(&stats[0], found);
      atomicMax(&stats[1], deepest);
    }
  }
}

// Step 8: node order.  Interior indices of the radix tree follow split positions, and the
// subtrees collapsed into leaves leave about half of them unused, so the nodes a ray visits
// one after another lie far apart.  The final tree is rewritten in depth-first preorder
// (a node, its first child's subtree, its second child's subtree): a descent through first
// children reads consecutive 64-B nodes, every subtree is one contiguous range, and the
// array holds only reachable nodes.  The interior-node count of every subtree of the final
// tree (size) comes from the bottom-up pass of step 5.
// 8a: preorder position = sum over the path from the root of 1 per step, plus the size
// of the first child's subtree wherever the path takes the second child.
__global__ __launch_bounds__(kBlock) void k_preorder_rank(uint32_t ni, const uint8_t* __restrict__ reach,
                                                          const int* __restrict__ parent, const Node2* __restrict__ nodes,
                                                          const uint32_t* __restrict__ size, uint32_t* __restrict__ rank,
                                                          uint32_t* err) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= ni || !reach[i]) return;
  uint32_t r = 0;
  int j = static_cast<int>(i);
  for (int steps = 0; j != 0; steps++) {
    if (steps >= kMaxTreeWalk) { atomicOr(err, 1u); return; }
    const int p = parent[j];
    const int first = nodes[p].d.x;
    r += 1u + ((first != j && first >= 0) ? size[first] : 0u);
    j = p;
  }
  rank[i] = r;
}

// 8b: move every reachable node to its preorder slot, with its child references and parent link
// renumbered.
__global__ __launch_bounds__(kBlock) void k_preorder_scatter(uint32_t ni, uint32_t n_out, const uint8_t* __restrict__ reach,
                                                             const int* __restrict__ parent, const Node2* __restrict__ nodes,
                                                             const uint32_t* __restrict__ rank, Node2* __restrict__ out,
                                                             int* __restrict__ out_parent, uint32_t* err) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= ni || !reach[i]) return;
  const uint32_t s = rank[i];
  if (s >= n_out) { atomicOr(err, 1u); return; }
  Node2 nd = nodes[i];
  if (nd.d.x >= 0) nd.d.x = static_cast<int>(rank[nd.d.x]);
  if (nd.d.y >= 0) nd.d.y = static_cast<int>(rank[nd.d.y]);
  out[s] = nd;
  out_parent[s] = i == 0 ? -1 : static_cast<int>(rank[parent[i]]);
}

// Step 7.
__global__ __launch_bounds__(kBlock) void k_gather(uint32_t nf, const uint32_t* __restrict__ vals,
                                                   const float* __restrict__ V, const uint32_t* __restrict__ F,
                                                   const uint32_t* __restrict__ mesh_off, uint32_t n_meshes,
                                                   float4* __restrict__ tris, float4* __restrict__ normals) {
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= nf) return;
  const uint32_t f = vals[k];
  // geometry of face f: largest g with mesh_off[g] <= f
  uint32_t lo = 0, hi = n_meshes;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (mesh_off[mid] <= f) lo = mid; else hi = mid;
  }
  const uint32_t g = lo, local = f - mesh_off[lo];
  const uint32_t i0 = F[3 * f], i1 = F[3 * f + 1], i2 = F[3 * f + 2];  // validated in k_prep
  const float x0 = V[3 * i0], y0 = V[3 * i0 + 1], z0 = V[3 * i0 + 2];
  const float x1 = V[3 * i1], y1 = V[3 * i1 + 1], z1 = V[3 * i1 + 2];
  const float x2 = V[3 * i2], y2 = V[3 * i2 + 1], z2 = V[3 * i2 + 2];
  tris[3 * static_cast<size_t>(k) + 0] = make_float4(x0, y0, z0, __uint_as_float(local));
  tris[3 * static_cast<size_t>(k) + 1] = make_float4(x1, y1, z1, __uint_as_float(g));
  tris[3 * static_cast<size_t>(k) + 2] = make_float4(x2, y2, z2, __uint_as_float(f));
  const double ax = (double)x1 - (double)x0, ay = (double)y1 - (double)y0, az = (double)z1 - (double)z0;
  const double bx = (double)x2 - (double)x0, by = (double)y2 - (double)y0, bz = (double)z2 - (double)z0;
  const double nx = ay * bz - az * by, ny = az * bx - ax * bz, nz = ax * by - ay * bx;
  const double len = sqrt(nx * nx + ny * ny + nz * nz);
  // w: object id of the face (the mesh index until rmh_map_set_mesh_ids says otherwise)
  float4 nrm = make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(g));
  if (len > 0.0) nrm = make_float4((float)(nx / len), (float)(ny / len), (float)(nz / len), __uint_as_float(g));
  normals[k] = nrm;
}

// Per-mesh geom / object ids: for every Morton slot, the mesh of its global face (v2.w)
// selects the ids (NULL table = keep).
__global__ __launch_bounds__(kBlock) void k_set_ids(uint32_t nf, const uint32_t* __restrict__ mesh_off, uint32_t n_meshes,
                                                    const uint32_t* __restrict__ geom, const uint32_t* __restrict__ obj,
                                                    float4* __restrict__ tris, float4* __restrict__ normals) {
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= nf) return;
  const uint32_t f = __float_as_uint(tris[3 * static_cast<size_t>(k) + 2].w);
  uint32_t lo = 0, hi = n_meshes;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (mesh_off[mid] <= f) lo = mid; else hi = mid;
  }
  if (geom) tris[3 * static_cast<size_t>(k) + 1].w = __uint_as_float(geom[lo]);
  if (obj) normals[k].w = __uint_as_float(obj[lo]);
}

// ---- SAH refinement: treelet restructuring (rmh_treelet.hpp) ------------------------------------

__global__ __launch_bounds__(kBlock) void k_leaf_boxes(uint32_t nf, const uint32_t* __restrict__ vals,
                                                       const float4* __restrict__ flo, const float4* __restrict__ fhi,
                                                       float* __restrict__ leaf_box) {
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= nf) return;
  const uint32_t f = vals[k];
  const float4 a = flo[f], b = fhi[f];
  float* o = leaf_box + 6 * static_cast<size_t>(k);
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = b.x; o[4] = b.y; o[5] = b.z;
}

// One bottom-up treelet pass runs level by level over the current tree, deepest first
// (make_levels): at each depth, the box, count and cost of the nodes with fewer than `gamma`
// triangles below are set from their children (thread per node), and those of the others
// too, each of which one wave then restructures.  One launch does both (k_treelet_nodes);
// k_refresh_nodes serves depths without treelets.  Children are final when their parent's
// level runs (earlier launches), a treelet only involves nodes of its subtree, and the nodes
// of one depth have disjoint subtrees, so no counters or fences are needed.  Which nodes get
// a treelet is known in advance: a node's triangle count depends only on its leaf set, which
// restructuring below it does not change.
__global__ __launch_bounds__(kBlock) void k_refresh_nodes(const uint32_t* __restrict__ order, uint32_t lo, uint32_t hi,
                                                          TreeArrays t, float c_node, float c_tri) {
  const uint32_t k = lo + blockIdx.x * kBlock + threadIdx.x;
  if (k < hi) refresh_node(t, static_cast<int>(order[k]), c_node, c_tri);
}

// One treelet leaf, held by one lane.
struct TreeletLeaf {
  uint32_t ref;
  uint32_t ch0, ch1;  // children of an interior leaf
  float b[6];
  float area;         // half area of an interior leaf, -1 for a triangle: what to open next
  float cost;
  uint32_t count;
};

__device__ __forceinline__ float half_area_of(const float* b) {
  const float dx = b[3] - b[0], dy = b[4] - b[1], dz = b[5] - b[2];
  return dx * dy + dy * dz + dz * dx;
}

__device__ __forceinline__ void load_treelet_leaf(const TreeArrays& t, uint32_t ref, float c_tri, TreeletLeaf& l) {
  const bool tri = (ref & kTreeLeafBit) != 0;
  const uint32_t i = ref & ~kTreeLeafBit;
  const float2* b = reinterpret_cast<const float2*>((tri ? t.leaf_box : t.box) + 6 * static_cast<size_t>(i));
  uint2 ch = make_uint2(0u, 0u);
  float cost = 0.0f;
  uint32_t count = 1u;
  if (!tri) {
    ch = *reinterpret_cast<const uint2*>(t.child + 2 * static_cast<size_t>(i));
    cost = t.cost[i];
    count = t.count[i];
  }
  const float2 b0 = b[0], b1 = b[1], b2 = b[2];
  l.ref = ref;
  l.ch0 = ch.x;
  l.ch1 = ch.y;
  l.b[0] = b0.x; l.b[1] = b0.y; l.b[2] = b1.x; l.b[3] = b1.y; l.b[4] = b2.x; l.b[5] = b2.y;
  const float area = half_area_of(l.b);
  l.area = tri ? -1.0f : area;
  l.cost = tri ? c_tri * area : cost;
  l.count = count;
}

__device__ __forceinline__ uint32_t lane_u32(uint32_t v, uint32_t lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float lane_f32(float v, uint32_t lane) {
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}

// The seven-leaf treelet below every node of order[lo, mid), one wave each: box, count
// and cost of the node from its children, then treelet_form, the dynamic program and
// treelet_rebuild of rmh_treelet.hpp with the same choices and the same arithmetic (the trees
// are those of the serial treelet_optimize()).  A node that gets a treelet has at least seven
// triangles below it, so it always has seven leaves.
//
// What bounds it is the length of one treelet's chain, so nothing in it is serial that need
// not be: lane j holds leaf j of the growing treelet with its box, cost and children, so
// opening a leaf is one dependent load round; the 127 subset areas take two subsets per lane
// (S and S + 64, whose boxes differ by leaf 6); subsets of up to five leaves have their splits
// walked by one lane each (at most 15), the 7 subsets of six are shared by 8 lanes each (4
// splits per lane) and the 63 splits of the whole treelet by all lanes; the new topology is
// built in registers and its six nodes are written by six lanes.  With the treelet formed and
// rebuilt by lane 0 through memory, and every subset's splits walked by one lane (126 steps
// for the whole treelet), three rounds on the 2.1M-triangle terrain took 11.2 ms, 3.1 ms now.
//
// The workgroups after those refresh the nodes order[mid, hi) of the same depth, 64 each: in a
// launch of their own they took 8 us a depth and a gap (builds of 2.1M, 500k and 79k
// triangles 5.64, 3.29 and 1.64 ms, now 5.43, 3.08 and 1.54).
__global__ __launch_bounds__(64) void k_treelet_nodes(const uint32_t* __restrict__ order, uint32_t lo, uint32_t mid,
                                                      uint32_t hi, TreeArrays t, float c_node, float c_tri) {
  static_assert(kTreeletLeaves == 7, "lanes are laid out for seven leaves");
  __shared__ float s_copt[128];
  __shared__ uint8_t s_part[128];
  const uint32_t lane = threadIdx.x;
  if (blockIdx.x >= mid - lo) {
    const uint32_t k = mid + (blockIdx.x - (mid - lo)) * 64u + lane;
    if (k < hi) refresh_node(t, static_cast<int>(order[k]), c_node, c_tri);
    return;
  }
  const uint32_t root = __builtin_amdgcn_readfirstlane(order[lo + blockIdx.x]);

  // the treelet: lanes 0 and 1 start with the root's children; the interior leaf of largest
  // area (the first of equals) is opened, its children go to its lane and to the next one
  TreeletLeaf leaf;
  leaf.area = -1.0f;
  const uint2 rc = *reinterpret_cast<const uint2*>(t.child + 2 * static_cast<size_t>(root));
  if (lane < 2) load_treelet_leaf(t, lane == 0 ? rc.x : rc.y, c_tri, leaf);
  float root_box[6];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float a0 = lane_f32(leaf.b[k], 0), a1 = lane_f32(leaf.b[k], 1);
    const float h0 = lane_f32(leaf.b[3 + k], 0), h1 = lane_f32(leaf.b[3 + k], 1);
    root_box[k] = a0 < a1 ? a0 : a1;
    root_box[3 + k] = h0 > h1 ? h0 : h1;
  }
  const float root_cost = c_node * half_area_of(root_box) + lane_f32(leaf.cost, 0) + lane_f32(leaf.cost, 1);
  const uint32_t root_count = lane_u32(leaf.count, 0) + lane_u32(leaf.count, 1);
  uint32_t inner = root;  // lane i: the i-th interior node of the treelet
#pragma unroll
  for (uint32_t nl = 2; nl < 7; nl++) {
    float a = leaf.area;
    uint32_t best = lane;
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) {
      const float oa = __shfl_xor(a, off, 8);
      const uint32_t ob = __shfl_xor(best, off, 8);
      const bool take = oa > a || (oa == a && ob < best);
      a = take ? oa : a;
      best = take ? ob : best;
    }
    best = __builtin_amdgcn_readfirstlane(best);
    const uint32_t x = lane_u32(leaf.ref, best), c0 = lane_u32(leaf.ch0, best), c1 = lane_u32(leaf.ch1, best);
    if (lane == nl - 1) inner = x;
    if (lane == best || lane == nl) load_treelet_leaf(t, lane == best ? c0 : c1, c_tri, leaf);
  }

  // areas of the subsets lane (leaves 0-5) and lane + 64 (with leaf 6)
  float bx[6] = {3.0e38f, 3.0e38f, 3.0e38f, -3.0e38f, -3.0e38f, -3.0e38f};
#pragma unroll
  for (uint32_t j = 0; j < 6; j++) {
    const bool in = (lane >> j) & 1u;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float l = lane_f32(leaf.b[k], j), h = lane_f32(leaf.b[3 + k], j);
      bx[k] = in && l < bx[k] ? l : bx[k];
      bx[3 + k] = in && h > bx[3 + k] ? h : bx[3 + k];
    }
  }
  const float area_lo = half_area_of(bx);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float l = lane_f32(leaf.b[k], 6), h = lane_f32(leaf.b[3 + k], 6);
    bx[k] = l < bx[k] ? l : bx[k];
    bx[3 + k] = h > bx[3 + k] ? h : bx[3 + k];
  }
  const float area_hi = half_area_of(bx);

  // least costs and splits, subset size by subset size: a split is the part P that holds the
  // lowest member, P's other members a proper subset r of the rest, in descending order, the
  // first of equals kept
  if (lane < 7) s_copt[1u << lane] = leaf.cost;
  __syncthreads();
  const uint32_t members = __popc(lane);
#pragma unroll
  for (uint32_t size = 2; size <= 5; size++) {
    const bool high = members == size - 1;
    if (high || members == size) {
      const uint32_t S = high ? lane + 64u : lane;
      const uint32_t low = S & (0u - S), rest = S ^ low;
      float best = 3.0e38f;
      uint32_t bp = low;
      uint32_t r = rest;
#pragma unroll
      for (uint32_t k = 0; k < (1u << (size - 1)) - 1u; k++) {
        r = (r - 1u) & rest;
        const float c = s_copt[low | r] + s_copt[rest ^ r];
        if (c < best) { best = c; bp = low | r; }
      }
      s_copt[S] = c_node * (high ? area_hi : area_lo) + best;
      s_part[S] = static_cast<uint8_t>(bp);
    }
    __syncthreads();
  }
  {
    // six leaves: subset 127 without leaf m, 8 lanes each; split j (of 31) in the compressed
    // index of its five other members, the larger of equals
    const uint32_t m = lane >> 3, S = 127u ^ (1u << m);
    float best = 3.0e38f;
    uint32_t bj = 0;
    if (m < 7) {
#pragma unroll
      for (uint32_t q = 0; q < 4; q++) {
        const uint32_t j = (lane & 7u) + 8u * q;
        if (j < 31u) {
          const uint32_t x = 1u | (j << 1);
          const uint32_t P = ((x >> m) << (m + 1)) | (x & ((1u << m) - 1u));
          const float c = s_copt[P] + s_copt[S ^ P];
          if (c <= best) { best = c; bj = j; }
        }
      }
    }
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) {
      const float oc = __shfl_xor(best, off, 8);
      const uint32_t oj = __shfl_xor(bj, off, 8);
      const bool take = oc < best || (oc == best && oj > bj);
      best = take ? oc : best;
      bj = take ? oj : bj;
    }
    const float area_m = __shfl(area_hi, static_cast<int>(63u ^ (1u << m)) & 63, 64);  // by all lanes
    const float area = m == 6 ? lane_f32(area_lo, 63) : area_m;
    if (m < 7 && (lane & 7u) == 0) {
      const uint32_t x = 1u | (bj << 1);
      s_copt[S] = c_node * area + best;
      s_part[S] = static_cast<uint8_t>(((x >> m) << (m + 1)) | (x & ((1u << m) - 1u)));
    }
  }
  __syncthreads();
  float best = 3.0e38f;
  uint32_t bj = 0;
  if (lane < 63) {
    const uint32_t P = 1u | (lane << 1);
    const float c = s_copt[P] + s_copt[127u ^ P];
    if (c < best) { best = c; bj = lane; }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float oc = __shfl_xor(best, off, 64);
    const uint32_t oj = __shfl_xor(bj, off, 64);
    const bool take = oc < best || (oc == best && oj > bj);
    best = take ? oc : best;
    bj = take ? oj : bj;
  }
  best = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(best)));
  const uint32_t part_all = 1u | (__builtin_amdgcn_readfirstlane(bj) << 1);
  const float copt_all = c_node * lane_f32(area_hi, 63) + best;
  if (!(copt_all < root_cost * (1.0f - 1e-6f))) {
    // the topology stays: the node's own box, count and cost
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < 6; k++) t.box[6 * static_cast<size_t>(root) + k] = root_box[k];
      t.count[root] = root_count;
      t.cost[root] = root_cost;
    }
    return;
  }

  // the new topology, built by all lanes alike: slot i (lane i) is the i-th interior node;
  // subsets still to be split wait on a stack (lane = position)
  uint32_t st_set = 127u, st_slot = 0u;                       // the stack
  uint32_t n_set = 0u, n_ref0 = 0u, n_ref1 = 0u;              // lane i: slot i
  uint32_t n_c0 = 0u, n_c1 = 0u;                              // its children: leaf j, or 8 + slot
  uint32_t made = 0u;                                         // slots in the order they were made, 4 bits each
  uint32_t sp = 1u, next = 1u;
#pragma unroll
  for (uint32_t k = 0; k < 6; k++) {
    sp--;
    const uint32_t S = lane_u32(st_set, sp), slot = lane_u32(st_slot, sp);
    made |= slot << (4 * k);
    const uint32_t P = S == 127u ? part_all : __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s_part[S]));
    uint32_t refs[2], kids[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const uint32_t sub = c ? S ^ P : P;
      if ((sub & (sub - 1u)) == 0u) {
        kids[c] = __builtin_ctz(sub);
        refs[c] = lane_u32(leaf.ref, kids[c]);
      } else {
        kids[c] = 8u + next;
        refs[c] = lane_u32(inner, next);
        if (lane == sp) { st_set = sub; st_slot = next; }
        sp++;
        next++;
      }
    }
    if (lane == slot) { n_set = S; n_ref0 = refs[0]; n_ref1 = refs[1]; n_c0 = kids[0]; n_c1 = kids[1]; }
  }
  // costs bottom-up in reverse order of making
  float n_cost = 0.0f;
#pragma unroll
  for (int k = 5; k >= 0; k--) {
    const uint32_t slot = (made >> (4 * k)) & 15u;
    const uint32_t S = lane_u32(n_set, slot), k0 = lane_u32(n_c0, slot), k1 = lane_u32(n_c1, slot);
    const float area = S >= 64u ? lane_f32(area_hi, S - 64u) : lane_f32(area_lo, S);
    const float cost0 = k0 < 8u ? lane_f32(leaf.cost, k0) : lane_f32(n_cost, k0 - 8u);
    const float cost1 = k1 < 8u ? lane_f32(leaf.cost, k1) : lane_f32(n_cost, k1 - 8u);
    const float cost = c_node * area + cost0 + cost1;
    if (lane == slot) n_cost = cost;
  }
  float nb[6] = {3.0e38f, 3.0e38f, 3.0e38f, -3.0e38f, -3.0e38f, -3.0e38f};
  uint32_t n_count = 0u;
#pragma unroll
  for (uint32_t j = 0; j < 7; j++) {
    const bool in = (n_set >> j) & 1u;
    n_count += in ? lane_u32(leaf.count, j) : 0u;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float l = lane_f32(leaf.b[k], j), h = lane_f32(leaf.b[3 + k], j);
      nb[k] = in && l < nb[k] ? l : nb[k];
      nb[3 + k] = in && h > nb[3 + k] ? h : nb[3 + k];
    }
  }
  if (lane < 6) {
    *reinterpret_cast<uint2*>(t.child + 2 * static_cast<size_t>(inner)) = make_uint2(n_ref0, n_ref1);
    float2* b = reinterpret_cast<float2*>(t.box + 6 * static_cast<size_t>(inner));
    b[0] = make_float2(nb[0], nb[1]);
    b[1] = make_float2(nb[2], nb[3]);
    b[2] = make_float2(nb[4], nb[5]);
    t.count[inner] = n_count;
    t.cost[inner] = n_cost;
    set_parent(t, n_ref0, static_cast<int>(inner));
    set_parent(t, n_ref1, static_cast<int>(inner));
  }
}

// Structure check of the refined tree before anything walks it: every child slot points
// into range at a node whose parent link names the slot's owner, no node is referenced
// twice (refs[] counts references), and every node reaches the root by parent links within
// kMaxTreeWalk steps (no cycle).  Any failure sets *err.
__global__ __launch_bounds__(kBlock) void k_check_tree(int n, TreeArrays t, uint32_t* refs, uint32_t* err) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n - 1) {
    const uint32_t c0 = t.child[2 * i], c1 = t.child[2 * i + 1];
    if (c0 == c1) atomicOr(err, 4u);
    for (int c = 0; c < 2; c++) {
      const uint32_t r = c ? c1 : c0;
      if (r & kTreeLeafBit) {
        const uint32_t k = r & ~kTreeLeafBit;
        if (k >= static_cast<uint32_t>(n) || t.parent_leaf[k] != i) { atomicOr(err, 4u); continue; }
        atomicAdd(&refs[n - 1 + k], 1u);
      } else {
        if (r == 0u || r >= static_cast<uint32_t>(n - 1) || t.parent_int[r] != i) { atomicOr(err, 4u); continue; }
        atomicAdd(&refs[r], 1u);
      }
    }
  }
  if (i < n) {
    int p = t.parent_leaf[i];
    int steps = 0;
    while (p >= 0 && steps < kMaxTreeWalk) {
      if (p >= n - 1) { p = -2; break; }
      p = t.parent_int[p];
      steps++;
    }
    if (p != -1) atomicOr(err, 4u);
  }
}

__global__ __launch_bounds__(kBlock) void k_check_refs(int n, const uint32_t* refs, uint32_t* err) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= 2 * n - 1) return;
  const uint32_t want = i == 0 ? 0u : 1u;  // the root has no parent slot
  if (refs[i] != want) atomicOr(err, 4u);
}

// Depth-first position of every leaf and of the first leaf below every interior node.
__global__ __launch_bounds__(kBlock) void k_dfs_positions(int n, TreeArrays t, uint32_t* __restrict__ pos,
                                                          uint32_t* __restrict__ off) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) pos[i] = dfs_offset(t, static_cast<uint32_t>(i) | kTreeLeafBit);
  if (i < n - 1) off[i] = dfs_offset(t, static_cast<uint32_t>(i));
}

// Leaves renumbered depth-first: the sorted face list, the leaf parents and the leaf
// references follow, and every interior node covers the range [off, off + count - 1].
__global__ __launch_bounds__(kBlock) void k_apply_order(int n, TreeArrays t, const uint32_t* __restrict__ pos,
                                                        const uint32_t* __restrict__ off, const uint32_t* __restrict__ vals,
                                                        uint32_t* __restrict__ vals_out, int* __restrict__ pleaf_out,
                                                        uint32_t* __restrict__ range) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) {
    vals_out[pos[i]] = vals[i];
    pleaf_out[pos[i]] = t.parent_leaf[i];
  }
  if (i < n - 1) {
    for (int c = 0; c < 2; c++) {
      const uint32_t r = t.child[2 * i + c];
      if (r & kTreeLeafBit) t.child[2 * i + c] = pos[r & ~kTreeLeafBit] | kTreeLeafBit;
    }
    range[2 * i] = off[i];
    range[2 * i + 1] = off[i] + t.count[i] - 1u;
  }
}

// ---- 4-wide quantised tree ------------------------------------------------------------------
//
// Collapsed top-down from the binary tree, one launch pair per level: a wide node made
// from binary node b starts with b's two children and repeatedly opens the interior
// candidate of largest surface area until it has four children or only leaves.  A
// level's children are numbered by an exclusive scan of the per-node interior-child
// counts, so the build is deterministic and each level lies in memory in the order of its
// parents (Morton order of the binary tree).

constexpr int kEmptyRef = 0x7fffffff;  // unused child slot (masked by the child count)

struct Cand {
  int ref;
  float lo[3], hi[3];
};

__device__ inline Cand child_cand(const Node2& nd, int c) {
  Cand k;
  if (c == 0) {
    k.ref = nd.d.x;
    k.lo[0] = nd.a.x; k.hi[0] = nd.a.y; k.lo[1] = nd.a.z; k.hi[1] = nd.a.w; k.lo[2] = nd.c.x; k.hi[2] = nd.c.y;
  } else {
    k.ref = nd.d.y;
    k.lo[0] = nd.b.x; k.hi[0] = nd.b.y; k.lo[1] = nd.b.z; k.hi[1] = nd.b.w; k.lo[2] = nd.c.z; k.hi[2] = nd.c.w;
  }
  return k;
}

__device__ inline float cand_area(const Cand& c) {
  const float dx = c.hi[0] - c.lo[0], dy = c.hi[1] - c.lo[1], dz = c.hi[2] - c.lo[2];
  return dx * dy + dy * dz + dz * dx;
}

// Children of the wide node made from binary node b, in left-to-right order.
__device__ inline int select_children(const Node2* __restrict__ nodes, int b, Cand c[4]) {
  const Node2 nd = nodes[b];
  c[0] = child_cand(nd, 0);
  c[1] = child_cand(nd, 1);
  int n = 2;
  while (n < 4) {
    int best = -1;
    float best_area = -1.0f;
    for (int k = 0; k < n; k++)
      if (c[k].ref >= 0 && cand_area(c[k]) > best_area) { best_area = cand_area(c[k]); best = k; }
    if (best < 0) break;
    const Node2 cn = nodes[c[best].ref];
    for (int k = n; k > best + 1; k--) c[k] = c[k - 1];
    c[best] = child_cand(cn, 0);
    c[best + 1] = child_cand(cn, 1);
    n++;
  }
  return n;
}

// Grid of one axis for the planes in [lo, hi]: the smallest exponent e >= -126 with an
// origin o = floor(lo / 2^e) 2^e such that o + 255 2^e >= hi and every o + q 2^e
// (q = 0..255) is an FP32 number (|o| and |o + 255 2^e| below 2^(24+e) and FLT_MAX).
// All of it is exact in FP64.  False when no exponent up to 127 fits.
__device__ inline bool quant_frame(float lo, float hi, int& e_out, double& origin_out) {
  const double L = lo, H = hi;
  int e = 0;
  (void)frexp((H - L) / 255.0, &e);
  e = max(e - 1, -126);
  for (; e <= 127; e++) {
    const double s = ldexp(1.0, e);
    const double o = floor(L / s) * s;
    const double top = o + 255.0 * s;
    if (top < H) continue;
    const double lim = fmin(ldexp(1.0, 24 + e), static_cast<double>(FLT_MAX));
    if (fabs(o) >= lim || fabs(top) >= lim) continue;
    e_out = e;
    origin_out = o;
    return true;
  }
  return false;
}

// Largest grid plane <= x and smallest grid plane >= x (x inside [o, o + 255 s]); the
// checks are exact FP64 comparisons, so a rounded quotient cannot move a plane inward.
__device__ inline uint32_t quant_lo(float x, double o, double s) {
  double q = fmin(fmax(floor((static_cast<double>(x) - o) / s), 0.0), 255.0);
  while (q > 0.0 && o + q * s > static_cast<double>(x)) q -= 1.0;
  return static_cast<uint32_t>(q);
}

__device__ inline uint32_t quant_hi(float x, double o, double s) {
  double q = fmin(fmax(ceil((static_cast<double>(x) - o) / s), 0.0), 255.0);
  while (q < 255.0 && o + q * s < static_cast<double>(x)) q += 1.0;
  return static_cast<uint32_t>(q);
}

__global__ __launch_bounds__(kBlock) void k_wide_count(const Node2* __restrict__ nodes, const int* __restrict__ front,
                                                       uint32_t n, uint32_t* __restrict__ counts) {
  const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
  if (j >= n) return;
  Cand c[4];
  const int k = select_children(nodes, front[j], c);
  uint32_t cnt = 0;
  for (int i = 0; i < k; i++) cnt += c[i].ref >= 0 ? 1u : 0u;
  counts[j] = cnt;
}

// Writes the wide nodes of one level (slots base .. base + n - 1) and the binary indices
// of the next level's nodes (slot next_base + offsets[j] + t for the t-th interior child).
__global__ __launch_bounds__(kBlock) void k_wide_emit(const Node2* __restrict__ nodes, const int* __restrict__ front,
                                                      uint32_t n, uint32_t base, uint32_t next_base, uint32_t cap,
                                                      const uint32_t* __restrict__ offsets, Node4* __restrict__ out,
                                                      int* __restrict__ next_front, uint32_t* err) {
  const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
  if (j >= n) return;
  if (base + j >= cap) { atomicOr(err, 2u); return; }
  Cand c[4];
  const int k = select_children(nodes, front[j], c);
  Node4 nd;
  for (int i = 0; i < 16; i++) nd.w[i] = 0u;
  uint32_t meta = static_cast<uint32_t>(k) << 24;
  for (int a = 0; a < 3; a++) {
    float lo = c[0].lo[a], hi = c[0].hi[a];
    for (int i = 1; i < k; i++) { lo = fminf(lo, c[i].lo[a]); hi = fmaxf(hi, c[i].hi[a]); }
    int e;
    double o;
    if (!quant_frame(lo, hi, e, o)) { atomicOr(err, 1u); return; }
    const double s = ldexp(1.0, e);
    nd.w[a] = __float_as_uint(static_cast<float>(o));  // exact: o is an FP32 number
    meta |= static_cast<uint32_t>(e + 127) << (8 * a);
    for (int i = 0; i < k; i++) {
      nd.w[4 + 2 * a] |= quant_lo(c[i].lo[a], o, s) << (8 * i);
      nd.w[5 + 2 * a] |= quant_hi(c[i].hi[a], o, s) << (8 * i);
    }
  }
  nd.w[3] = meta;
  uint32_t slot = offsets[j];
  for (int i = 0; i < 4; i++) {
    int ref = kEmptyRef;
    if (i < k) {
      ref = c[i].ref;
      if (ref >= 0) {
        if (next_base + slot >= cap) { atomicOr(err, 2u); return; }
        next_front[slot] = ref;
        ref = static_cast<int>(next_base + slot);
        slot++;
      }
    }
    nd.w[10 + i] = static_cast<uint32_t>(ref);
  }
  out[base + j] = nd;
}

// Arrays laid out one after another in one block, 256-byte aligned: with base NULL only the
// size is counted.
struct Carve {
  char* base = nullptr;
  size_t size = 0;
  template <class T>
  T* take(size_t n) {
    T* p = reinterpret_cast<T*>(base ? base + size : nullptr);
    size += (n * sizeof(T) + 255) & ~static_cast<size_t>(255);
    return p;
  }
};

// One block of scratch from the library's pool (from hipMalloc when the pool cannot give it),
// handed back in stream order.
struct Scratch {
  void* p = nullptr;
  bool pooled = false;
  hipStream_t stream = nullptr;
  hipError_t alloc(int device, size_t bytes, hipStream_t s) {
    stream = s;
    const hipMemPool_t pool = scratch_pool(device);
    if (pool && hipMallocFromPoolAsync(&p, bytes, pool, s) == hipSuccess) {
      pooled = true;
      return hipSuccess;
    }
    (void)hipGetLastError();
    p = nullptr;
    return hipMalloc(&p, bytes);
  }
  ~Scratch() {
    if (!p) return;
    if (pooled) (void)hipFreeAsync(p, stream);
    else (void)hipFree(p);
  }
};

struct DevBuf {
  void* p = nullptr;
  ~DevBuf() { if (p) (void)hipFree(p); }
  template <class T> T* as() { return static_cast<T*>(p); }
};

inline uint32_t blocks_for(uint64_t n) { return static_cast<uint32_t>((n + kBlock - 1) / kBlock); }

// One depth of the level-by-level passes: order[lo, mid) are its nodes with a treelet,
// order[mid, hi) the others.
struct LevelClass {
  uint32_t lo, mid, hi;
};

constexpr uint32_t kLevelKeys = 2u * (static_cast<uint32_t>(kMaxTreeWalk) + 1u);

// Scratch of make_levels for a tree of ni interior nodes.
struct LevelBufs {
  uint32_t *keys = nullptr, *keys2 = nullptr, *idx = nullptr, *order = nullptr, *start = nullptr;
  char* tmp = nullptr;
  size_t tmp_bytes = 0;

  hipError_t sort(uint32_t ni, hipStream_t stream) {
    return rocprim::radix_sort_pairs(tmp, tmp_bytes, keys, keys2, idx, order, ni, 0u, 14u, stream);
  }
  void carve(Carve& c, uint32_t ni) {
    keys = c.take<uint32_t>(ni);
    keys2 = c.take<uint32_t>(ni);
    idx = c.take<uint32_t>(ni);
    order = c.take<uint32_t>(ni);
    start = c.take<uint32_t>(kLevelKeys);
    tmp = c.take<char>(tmp_bytes);
  }
};

// Interior nodes of the radix tree (n leaves, n - 1 interior nodes) grouped by depth,
// deepest first, into b.order; `classes` receives the launch ranges in that order (within a
// depth the treelet nodes first).  count = NULL: no treelets.  Synchronous: the range sizes
// size the launches.  A broken tree sets err bit 8.
hipError_t make_levels(int n, const int* parent_int, const uint32_t* count, uint32_t gamma, LevelBufs& b,
                       uint32_t* err, hipStream_t stream, std::vector<LevelClass>& classes) {
  const uint32_t ni = static_cast<uint32_t>(n - 1);
  hipError_t e;
  k_level_keys<<<blocks_for(ni), kBlock, 0, stream>>>(n, parent_int, count, gamma, b.keys,
                                                      b.idx, err);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if ((e = b.sort(ni, stream)) != hipSuccess) return e;
  if ((e = hipMemsetAsync(b.start, 0xFF, sizeof(uint32_t) * kLevelKeys, stream)) != hipSuccess) return e;
  k_level_starts<<<blocks_for(ni), kBlock, 0, stream>>>(ni, b.keys2, b.start);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  std::vector<uint32_t> st(kLevelKeys);
  if ((e = hipMemcpyAsync(st.data(), b.start, sizeof(uint32_t) * kLevelKeys, hipMemcpyDeviceToHost, stream)) !=
      hipSuccess)
    return e;
  if ((e = hipStreamSynchronize(stream)) != hipSuccess) return e;
  classes.clear();
  uint32_t end = ni;
  for (uint32_t d = kLevelKeys / 2u; d-- > 0;) {  // the keys are depth-major, so ranges end where the next begins
    const uint32_t lo = st[2u * d], mid = st[2u * d + 1u];
    if (lo == 0xFFFFFFFFu && mid == 0xFFFFFFFFu) continue;
    const LevelClass c{lo != 0xFFFFFFFFu ? lo : mid, mid != 0xFFFFFFFFu ? mid : end, end};
    classes.push_back(c);
    end = c.lo;
  }
  std::reverse(classes.begin(), classes.end());
  return hipSuccess;
}

void map_free(rmh_map* m) {
  if (!m) return;
  if (m->mesh_block) (void)hipFree(m->mesh_block);
  if (m->tree_block) (void)hipFree(m->tree_block);
  if (m->nodes4) (void)hipFree(m->nodes4);
  for (const RefitPass& r : m->refit_passes)
    if (r.nodes) (void)hipFree(r.nodes);
  delete m;
}

// Most levels of the 4-wide tree the ray kernels accept: a lane's stack holds at most 3
// entries per level, and the largest stack template has 128.
constexpr uint32_t kMaxWideLevels = 42;

void free_wide(rmh_map* m) {
  if (m->nodes4) (void)hipFree(m->nodes4);
  m->nodes4 = nullptr;
  m->wide_capacity = 0;
  m->root4 = m->root;
  m->info.n_wide_nodes = 0;
  m->info.wide_levels = 0;
}

// (Re)builds the 4-wide tree of m from its binary tree, in place when the existing buffer
// is large enough (a refit keeps the node count, so the buffer address stays the same).
// Frees it (the ray kernels then use the binary tree) for a single-leaf tree, for a tree
// of more than kMaxWideLevels wide levels, and for coordinates no 8-bit grid can hold.
hipError_t build_wide(rmh_map* m, hipStream_t stream) {
  const uint32_t cap = m->info.n_nodes;  // one wide node per binary node at most
  if (m->root < 0 || cap == 0 || m->n_internal == 0) { free_wide(m); return hipSuccess; }
  DevBuf fa, fb, counts, offsets, err, tmp;
  hipError_t e;
  if (!m->nodes4 || m->wide_capacity < cap) {
    free_wide(m);
    if ((e = hipMalloc(&m->nodes4, sizeof(Node4) * cap)) != hipSuccess) { m->nodes4 = nullptr; return e; }
    m->wide_capacity = cap;
  }
  if ((e = hipMalloc(&fa.p, sizeof(int) * cap)) != hipSuccess) return e;
  if ((e = hipMalloc(&fb.p, sizeof(int) * cap)) != hipSuccess) return e;
  if ((e = hipMalloc(&counts.p, sizeof(uint32_t) * cap)) != hipSuccess) return e;
  if ((e = hipMalloc(&offsets.p, sizeof(uint32_t) * cap)) != hipSuccess) return e;
  if ((e = hipMalloc(&err.p, sizeof(uint32_t))) != hipSuccess) return e;
  size_t tmp_bytes = 0;
  if ((e = rocprim::exclusive_scan(nullptr, tmp_bytes, counts.as<uint32_t>(), offsets.as<uint32_t>(), 0u, cap,
                                   rocprim::plus<uint32_t>(), stream)) != hipSuccess) return e;
  if ((e = hipMalloc(&tmp.p, tmp_bytes)) != hipSuccess) return e;
  if ((e = hipMemsetAsync(err.p, 0, sizeof(uint32_t), stream)) != hipSuccess) return e;
  const int root = 0;
  if ((e = hipMemcpyAsync(fa.p, &root, sizeof(int), hipMemcpyHostToDevice, stream)) != hipSuccess) return e;
  int* front = fa.as<int>();
  int* next = fb.as<int>();
  uint32_t n = 1, base = 0, levels = 0;
  bool ok = true;
  while (n > 0) {
    const uint32_t next_base = base + n;
    k_wide_count<<<blocks_for(n), kBlock, 0, stream>>>(m->nodes, front, n, counts.as<uint32_t>());
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = rocprim::exclusive_scan(tmp.p, tmp_bytes, counts.as<uint32_t>(), offsets.as<uint32_t>(), 0u, n,
                                     rocprim::plus<uint32_t>(), stream)) != hipSuccess) return e;
    k_wide_emit<<<blocks_for(n), kBlock, 0, stream>>>(m->nodes, front, n, base, next_base, cap, offsets.as<uint32_t>(),
                                                      m->nodes4, next, err.as<uint32_t>());
    if ((e = hipGetLastError()) != hipSuccess) return e;
    uint32_t h[3] = {0, 0, 0};
    if ((e = hipMemcpyAsync(&h[0], offsets.as<uint32_t>() + (n - 1), sizeof(uint32_t), hipMemcpyDeviceToHost,
                            stream)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(&h[1], counts.as<uint32_t>() + (n - 1), sizeof(uint32_t), hipMemcpyDeviceToHost,
                            stream)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(&h[2], err.p, sizeof(uint32_t), hipMemcpyDeviceToHost, stream)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(stream)) != hipSuccess) return e;
    levels++;
    const uint64_t children = static_cast<uint64_t>(h[0]) + h[1];
    if (h[2] != 0u || next_base + children > cap || levels > kMaxWideLevels) { ok = false; break; }
    base = next_base;
    n = static_cast<uint32_t>(children);
    std::swap(front, next);
  }
  if (!ok) {
    free_wide(m);
    return hipSuccess;
  }
  m->root4 = 0;
  m->info.n_wide_nodes = base;
  m->info.wide_levels = levels;
  return hipSuccess;
}

#define BUILD_TRY(expr)                                             \
  do {                                                              \
    hipError_t _e = (expr);                                         \
    if (_e != hipSuccess) { map_free(m); return hip_fail(_e, #expr); } \
  } while (0)

}  // namespace

// Writes the n_reach reachable nodes of the ni radix-tree slots (root at slot 0; size =
// interior nodes of the final tree per subtree) and their parents in preorder
// into the map's tree block.  rank and err are scratch.
static hipError_t preorder_nodes(rmh_map* m, uint32_t ni, uint32_t n_reach, const Node2* nodes, const int* parent,
                                 const uint8_t* reach, const uint32_t* size, uint32_t* rank, uint32_t* err,
                                 hipStream_t stream) {
  Carve c;
  for (int pass = 0; pass < 2; pass++) {
    c.size = 0;
    m->nodes = c.take<Node2>(n_reach);
    m->parent = c.take<int>(n_reach);
    if (pass == 0) {
      const hipError_t e = hipMalloc(&m->tree_block, c.size);
      if (e != hipSuccess) { m->tree_block = nullptr; return e; }
      c.base = static_cast<char*>(m->tree_block);
    }
  }
  hipError_t e = hipMemsetAsync(err, 0, sizeof(uint32_t), stream);
  if (e == hipSuccess) {
    k_preorder_rank<<<blocks_for(ni), kBlock, 0, stream>>>(ni, reach, parent, nodes, size, rank, err);
    e = hipGetLastError();
  }
  if (e == hipSuccess) {
    k_preorder_scatter<<<blocks_for(ni), kBlock, 0, stream>>>(ni, n_reach, reach, parent, nodes, rank, m->nodes,
                                                              m->parent, err);
    e = hipGetLastError();
  }
  uint32_t herr = 0, root_size = 0;
  if (e == hipSuccess) e = hipMemcpyAsync(&herr, err, sizeof(uint32_t), hipMemcpyDeviceToHost, stream);
  if (e == hipSuccess) e = hipMemcpyAsync(&root_size, size, sizeof(uint32_t), hipMemcpyDeviceToHost, stream);
  if (e == hipSuccess) e = hipStreamSynchronize(stream);
  // a walk that did not end at the root, or a count that differs from the reachable
  // nodes, means the links do not form one tree: the build fails
  if (e == hipSuccess && (herr != 0 || root_size != n_reach)) e = hipErrorInvalidValue;
  if (e != hipSuccess) return e;
  m->n_internal = n_reach;
  return hipSuccess;
}

static int map_build(const float* vertices, uint32_t nv, const uint32_t* faces, uint32_t nf,
                     const uint32_t* mesh_face_offsets, uint32_t n_meshes, const rmh_bvh_params* params,
                     void* stream_, rmh_map** out);

// The ray kernels hold one stack entry per tree level, at most 128.  The radix tree is at
// most 95 levels deep (63 key bits, then at most 32 levels of index bits among equal keys),
// but treelet restructuring may lengthen paths; a refined tree deeper than 128 levels is
// replaced by the unrefined one, so every map the build accepts can be traced.
extern "C" int rmh_map_build(const float* vertices, uint32_t nv, const uint32_t* faces, uint32_t nf,
                             const uint32_t* mesh_face_offsets, uint32_t n_meshes,
                             const rmh_bvh_params* params, void* stream_, rmh_map** out) {
  const int rc = map_build(vertices, nv, faces, nf, mesh_face_offsets, n_meshes, params, stream_, out);
  if (rc != RMH_OK || (*out)->info.max_depth <= kMaxBinaryDepth) return rc;
  if (params && (params->flags & RMH_BVH_NO_REFINE)) return rc;  // not reached, by the bound above
  map_free(*out);
  *out = nullptr;
  rmh_bvh_params prm{4u, 1.0f, 1.5f, 0u};
  if (params) prm = *params;
  prm.flags |= RMH_BVH_NO_REFINE;
  return map_build(vertices, nv, faces, nf, mesh_face_offsets, n_meshes, &prm, stream_, out);
}

static int map_build(const float* vertices, uint32_t nv, const uint32_t* faces, uint32_t nf,
                     const uint32_t* mesh_face_offsets, uint32_t n_meshes, const rmh_bvh_params* params,
                     void* stream_, rmh_map** out) {
  if (!out) return fail(RMH_ERR_INVALID, "rmh_map_build: out is NULL");
  *out = nullptr;
  if (nf > 0 && (!vertices || !faces || nv == 0))
    return fail(RMH_ERR_INVALID, "rmh_map_build: faces given without vertices");
  // The ray kernels address a node as a 32-bit byte offset (index << 6, 64-byte nodes), so
  // every tree must have fewer than 2^26 interior nodes; a binary tree over n_faces leaves
  // has at most n_faces - 1 of them (and the 4-wide tree fewer still).
  if (nf > kMaxFaces)
    return fail(RMH_ERR_UNSUPPORTED, "rmh_map_build: at most 2^26 faces (BVH node offsets are 32-bit)");
  rmh_bvh_params prm{4u, 1.0f, 1.5f, 0u};
  if (params) prm = *params;
  if (prm.max_leaf_size < 1 || prm.max_leaf_size > static_cast<uint32_t>(kMaxLeaf))
    return fail(RMH_ERR_INVALID, "rmh_map_build: max_leaf_size must be in [1, 8]");
  std::vector<uint32_t> off;
  if (mesh_face_offsets && n_meshes > 0) {
    off.assign(mesh_face_offsets, mesh_face_offsets + n_meshes + 1);
    if (off.front() != 0 || off.back() != nf)
      return fail(RMH_ERR_INVALID, "rmh_map_build: mesh_face_offsets must start at 0 and end at n_faces");
    for (uint32_t g = 0; g < n_meshes; g++)
      if (off[g] > off[g + 1]) return fail(RMH_ERR_INVALID, "rmh_map_build: mesh_face_offsets not sorted");
  } else {
    n_meshes = 1;
    off = {0u, nf};
  }
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  rmh_map* m = new (std::nothrow) rmh_map();
  if (!m) return fail(RMH_ERR_ALLOC, "rmh_map_build: out of host memory");
  m->n_vertices = nv;
  m->n_faces = nf;
  m->n_meshes = n_meshes;
  (void)hipGetDevice(&m->device);
  m->info.n_vertices = nv;
  m->info.n_faces = nf;
  m->info.n_meshes = n_meshes;
  m->mesh_offsets = off;
  if (nf == 0) {  // empty map: every ray misses
    m->root = 0;
    *out = m;
    return RMH_OK;
  }

  hipEvent_t ev0, ev1;
  BUILD_TRY(hipEventCreate(&ev0));
  BUILD_TRY(hipEventCreate(&ev1));
  struct EvGuard { hipEvent_t a, b; ~EvGuard() { (void)hipEventDestroy(a); (void)hipEventDestroy(b); } } evg{ev0, ev1};

  Carve mc;
  for (int pass = 0; pass < 2; pass++) {
    mc.size = 0;
    m->vertices = mc.take<float>(3 * static_cast<size_t>(nv));
    m->faces = mc.take<uint32_t>(3 * static_cast<size_t>(nf));
    m->tris = mc.take<float4>(3 * static_cast<size_t>(nf));
    m->normals = mc.take<float4>(nf);
    if (pass == 0) {
      BUILD_TRY(hipMalloc(&m->mesh_block, mc.size));
      mc.base = static_cast<char*>(m->mesh_block);
    }
  }
  BUILD_TRY(hipMemcpyAsync(m->vertices, vertices, sizeof(float) * 3 * nv, hipMemcpyDeviceToDevice, stream));
  BUILD_TRY(hipMemcpyAsync(m->faces, faces, sizeof(uint32_t) * 3 * nf, hipMemcpyDeviceToDevice, stream));

  // All scratch is one block of the pool: 32 arrays allocated and freed one by one took 7 of
  // the 14.5 ms of a 2.1M-triangle build.
  const int n = static_cast<int>(nf);
  const uint32_t ni = nf > 1 ? nf - 1 : 0;
  const bool refine = !(prm.flags & RMH_BVH_NO_REFINE) && n >= kTreeletLeaves;
  float4 *flo, *fhi, *nlo, *nhi;
  float *bounds, *lbox = nullptr, *tbox = nullptr, *tcost = nullptr;
  uint32_t *err, *vals, *vals2, *child, *range, *stats, *moff, *subtree, *rank;
  uint32_t *tcount = nullptr, *pos = nullptr, *offs = nullptr, *vals3 = nullptr, *refs = nullptr;
  uint64_t *keys, *keys2;
  int *pint, *pleaf, *pleaf2 = nullptr;
  uint8_t *coll, *reach;
  Node2* slots;  // nodes in radix-tree order
  char* sort_tmp;
  size_t sort_bytes = 0;
  LevelBufs lb;                    // scratch of the level-by-level passes (make_levels)
  std::vector<LevelClass> levels;  // their launch ranges
  BUILD_TRY(rocprim::radix_sort_pairs(nullptr, sort_bytes, static_cast<uint64_t*>(nullptr), static_cast<uint64_t*>(nullptr),
                                      static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr), nf, 0u, 63u, stream));
  if (ni > 0) BUILD_TRY(lb.sort(ni, stream));  // with tmp NULL: the size of its scratch
  Scratch scratch;
  Carve sc;
  for (int pass = 0; pass < 2; pass++) {
    sc.size = 0;
    flo = sc.take<float4>(nf);
    fhi = sc.take<float4>(nf);
    bounds = sc.take<float>(8);
    err = sc.take<uint32_t>(4);
    stats = sc.take<uint32_t>(4);
    moff = sc.take<uint32_t>(n_meshes + 1);
    keys = sc.take<uint64_t>(nf);
    keys2 = sc.take<uint64_t>(nf);
    vals = sc.take<uint32_t>(nf);
    vals2 = sc.take<uint32_t>(nf);
    sort_tmp = sc.take<char>(sort_bytes);
    child = sc.take<uint32_t>(2 * static_cast<size_t>(ni + 1));
    range = sc.take<uint32_t>(2 * static_cast<size_t>(ni + 1));
    pint = sc.take<int>(ni + 1);
    pleaf = sc.take<int>(nf);
    nlo = sc.take<float4>(ni + 1);
    nhi = sc.take<float4>(ni + 1);
    coll = sc.take<uint8_t>(ni + 1);
    subtree = sc.take<uint32_t>(ni + 1);
    slots = sc.take<Node2>(ni + 1);
    reach = sc.take<uint8_t>(ni + 1);
    rank = sc.take<uint32_t>(ni + 1);
    if (ni > 0) lb.carve(sc, ni);
    if (refine) {
      lbox = sc.take<float>(6 * static_cast<size_t>(nf));
      tbox = sc.take<float>(6 * static_cast<size_t>(ni));
      tcost = sc.take<float>(ni);
      tcount = sc.take<uint32_t>(ni);
      pos = sc.take<uint32_t>(nf);
      offs = sc.take<uint32_t>(ni);
      vals3 = sc.take<uint32_t>(nf);
      pleaf2 = sc.take<int>(nf);
      refs = sc.take<uint32_t>(2 * static_cast<size_t>(nf) - 1);
    }
    if (pass == 0) {
      BUILD_TRY(scratch.alloc(m->device, sc.size, stream));
      sc.base = static_cast<char*>(scratch.p);
    }
  }
  BUILD_TRY(hipMemcpyAsync(moff, off.data(), sizeof(uint32_t) * (n_meshes + 1), hipMemcpyHostToDevice, stream));

  BUILD_TRY(hipEventRecord(ev0, stream));
  k_init<<<1, 64, 0, stream>>>(bounds, err);
  k_prep<<<std::min(blocks_for(nf), kWideBlocks), kBlock, 0, stream>>>(m->vertices, nv, m->faces, nf, flo, fhi,
                                                bounds, err);
  BUILD_TRY(hipGetLastError());
  uint32_t herr = 0;
  BUILD_TRY(hipMemcpyAsync(&herr, err, sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
  BUILD_TRY(hipStreamSynchronize(stream));
  if (herr & 1u) { map_free(m); return fail(RMH_ERR_INVALID, "rmh_map_build: face index >= n_vertices"); }
  if (herr & 2u) { map_free(m); return fail(RMH_ERR_INVALID, "rmh_map_build: non-finite vertex coordinate"); }

  k_morton<<<blocks_for(nf), kBlock, 0, stream>>>(flo, fhi, nf, bounds,
                                                  keys, vals);
  BUILD_TRY(hipGetLastError());
  BUILD_TRY(rocprim::radix_sort_pairs(sort_tmp, sort_bytes, keys, keys2,
                                      vals, vals2, nf, 0u, 63u, stream));
  uint64_t* skeys = keys2;
  uint32_t* svals = vals2;

  BUILD_TRY(hipMemsetAsync(stats, 0, sizeof(uint32_t) * 4, stream));
  if (n >= 2) {
    k_karras<<<blocks_for(ni), kBlock, 0, stream>>>(skeys, n, child, range,
                                                    pint, pleaf);
    BUILD_TRY(hipGetLastError());
    if (refine) {
      // SAH refinement of the radix tree, then depth-first leaf order so that every
      // subtree is again one range of the triangle array
      TreeArrays ta;
      ta.child = child;
      ta.parent_int = pint;
      ta.parent_leaf = pleaf;
      ta.box = tbox;
      ta.cost = tcost;
      ta.count = tcount;
      ta.leaf_box = lbox;
      k_leaf_boxes<<<blocks_for(nf), kBlock, 0, stream>>>(nf, svals, flo, fhi, lbox);
      BUILD_TRY(hipGetLastError());
      BUILD_TRY(hipMemsetAsync(err, 0, sizeof(uint32_t), stream));
      // triangle counts of the radix tree decide the first round's treelets; each round
      // leaves every count current for the next
      k_range_counts<<<blocks_for(ni), kBlock, 0, stream>>>(ni, range, ta.count);
      BUILD_TRY(hipGetLastError());
      for (int r = 0; r < kTreeletRounds; r++) {
        // the depths change with every round's restructuring
        BUILD_TRY(make_levels(n, pint, ta.count, static_cast<uint32_t>(kTreeletLeaves), lb, err,
                              stream, levels));
        for (const LevelClass& c : levels) {
          if (c.mid > c.lo)
            k_treelet_nodes<<<c.mid - c.lo + (c.hi - c.mid + 63u) / 64u, 64, 0, stream>>>(
                lb.order, c.lo, c.mid, c.hi, ta, prm.sah_cost_node, prm.sah_cost_tri);
          else
            k_refresh_nodes<<<blocks_for(c.hi - c.lo), kBlock, 0, stream>>>(lb.order, c.lo, c.hi, ta,
                                                                             prm.sah_cost_node, prm.sah_cost_tri);
          BUILD_TRY(hipGetLastError());
        }
      }
      {
        BUILD_TRY(hipMemsetAsync(refs, 0, sizeof(uint32_t) * (2 * static_cast<size_t>(nf) - 1), stream));
        k_check_tree<<<blocks_for(nf), kBlock, 0, stream>>>(n, ta, refs, err);
        BUILD_TRY(hipGetLastError());
        k_check_refs<<<blocks_for(2 * static_cast<uint64_t>(nf)), kBlock, 0, stream>>>(n, refs,
                                                                                       err);
        BUILD_TRY(hipGetLastError());
        uint32_t terr = 0;
        BUILD_TRY(hipMemcpyAsync(&terr, err, sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
        BUILD_TRY(hipStreamSynchronize(stream));
        if (terr) { map_free(m); return fail(RMH_ERR_UNSUPPORTED, "rmh_map_build: BVH refinement produced an invalid tree"); }
      }
      k_dfs_positions<<<blocks_for(nf), kBlock, 0, stream>>>(n, ta, pos, offs);
      BUILD_TRY(hipGetLastError());
      k_apply_order<<<blocks_for(nf), kBlock, 0, stream>>>(n, ta, pos, offs, svals,
                                                           vals3, pleaf2, range);
      BUILD_TRY(hipGetLastError());
      svals = vals3;
      std::swap(pleaf, pleaf2);
    }
    BUILD_TRY(make_levels(n, pint, nullptr, 0u, lb, err, stream, levels));
    for (const LevelClass& c : levels) {
      const uint32_t cnt = c.hi - c.lo;
      k_bottom_up_level<<<blocks_for(cnt), kBlock, 0, stream>>>(lb.order, c.lo, c.hi, svals,
                                                                flo, fhi, child,
                                                                nlo, nhi, coll,
                                                                subtree, prm.max_leaf_size,
                                                                prm.sah_cost_node, prm.sah_cost_tri);
      BUILD_TRY(hipGetLastError());
    }
    k_layout<<<std::min(blocks_for(ni), kWideBlocks), kBlock, 0, stream>>>(n, svals, flo, fhi, child,
                                                    range, pint, nlo,
                                                    nhi, coll, slots, stats,
                                                    reach);
    BUILD_TRY(hipGetLastError());
  }
  k_gather<<<blocks_for(nf), kBlock, 0, stream>>>(nf, svals, m->vertices, m->faces, moff, n_meshes,
                                                  m->tris, m->normals);
  BUILD_TRY(hipGetLastError());
  BUILD_TRY(hipEventRecord(ev1, stream));
  BUILD_TRY(hipStreamSynchronize(stream));
  float ms = 0.0f;
  BUILD_TRY(hipEventElapsedTime(&ms, ev0, ev1));

  uint32_t hstats[4] = {0, 0, 0, 0};
  uint8_t root_collapsed = 0;
  float4 root_lo = make_float4(0, 0, 0, 0), root_hi = make_float4(0, 0, 0, 0);
  if (n >= 2) {
    BUILD_TRY(hipMemcpy(hstats, stats, sizeof(hstats), hipMemcpyDeviceToHost));
    BUILD_TRY(hipMemcpy(&root_collapsed, coll, 1, hipMemcpyDeviceToHost));
    BUILD_TRY(hipMemcpy(&root_lo, nlo, sizeof(float4), hipMemcpyDeviceToHost));
    BUILD_TRY(hipMemcpy(&root_hi, nhi, sizeof(float4), hipMemcpyDeviceToHost));
  }
  m->n_internal = ni;
  if (n == 1 || root_collapsed) {
    m->root = make_leaf_ref(0u, nf);
    m->info.n_nodes = 0;
    m->info.n_leaves = 1;
    m->info.max_depth = 0;
  } else {
    m->root = 0;
    m->info.n_nodes = hstats[0];
    m->info.n_leaves = hstats[0] + 1;
    m->info.max_depth = hstats[1];
  }
  {
    const float dx = root_hi.x - root_lo.x, dy = root_hi.y - root_lo.y, dz = root_hi.z - root_lo.z;
    const float area = dx * dy + dy * dz + dz * dx;
    m->info.sah_cost = (n >= 2 && area > 0.0f) ? root_lo.w / area : 0.0f;
  }
  if (m->root == 0 && hstats[0] > 0) {
    BUILD_TRY(hipEventRecord(ev0, stream));
    BUILD_TRY(preorder_nodes(m, ni, hstats[0], slots, pint, reach, subtree, rank, err, stream));
    BUILD_TRY(hipEventRecord(ev1, stream));
    BUILD_TRY(hipStreamSynchronize(stream));
    float order_ms = 0.0f;
    BUILD_TRY(hipEventElapsedTime(&order_ms, ev0, ev1));
    ms += order_ms;
  } else {
    m->n_internal = 0;
  }
  m->root4 = m->root;
  if (prm.flags & RMH_BVH_WIDE) {
    BUILD_TRY(hipEventRecord(ev0, stream));
    BUILD_TRY(build_wide(m, stream));
    BUILD_TRY(hipEventRecord(ev1, stream));
    BUILD_TRY(hipStreamSynchronize(stream));
    float wide_ms = 0.0f;
    BUILD_TRY(hipEventElapsedTime(&wide_ms, ev0, ev1));
    ms += wide_ms;
  }
  m->info.build_ms = ms;
  m->info.device_bytes = sizeof(float4) * 4 * static_cast<uint64_t>(nf) + sizeof(Node2) * static_cast<uint64_t>(m->n_internal) +
                         sizeof(Node4) * static_cast<uint64_t>(m->info.n_wide_nodes);
  *out = m;
  return RMH_OK;
}

extern "C" int rmh_map_destroy(rmh_map* map) {
  map_free(map);
  return RMH_OK;
}

extern "C" int rmh_map_set_mesh_ids(rmh_map* map, const uint32_t* geom_ids, const uint32_t* object_ids,
                                    uint32_t n_meshes) {
  if (!map) return fail(RMH_ERR_INVALID, "rmh_map_set_mesh_ids: NULL map");
  if (n_meshes != map->n_meshes)
    return fail(RMH_ERR_INVALID, "rmh_map_set_mesh_ids: n_meshes differs from the map's mesh count");
  if (map->n_faces == 0 || (!geom_ids && !object_ids)) return RMH_OK;
  const uint32_t n = map->n_meshes;
  std::vector<uint32_t> host;
  host.reserve(3 * static_cast<size_t>(n) + 1);
  host.insert(host.end(), map->mesh_offsets.begin(), map->mesh_offsets.end());      // n + 1
  if (geom_ids) host.insert(host.end(), geom_ids, geom_ids + n);
  if (object_ids) host.insert(host.end(), object_ids, object_ids + n);
  uint32_t* dev = nullptr;
  RMH_HIP_TRY(hipMalloc(&dev, sizeof(uint32_t) * host.size()));
  hipError_t e = hipMemcpy(dev, host.data(), sizeof(uint32_t) * host.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    const uint32_t* g = geom_ids ? dev + n + 1 : nullptr;
    const uint32_t* o = object_ids ? dev + n + 1 + (geom_ids ? n : 0) : nullptr;
    k_set_ids<<<blocks_for(map->n_faces), kBlock>>>(map->n_faces, dev, n, g, o, map->tris, map->normals);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  (void)hipFree(dev);
  if (e != hipSuccess) return hip_fail(e, "rmh_map_set_mesh_ids");
  return RMH_OK;
}

// ---- refit: new vertex positions, same topology -------------------------------------------------

__global__ __launch_bounds__(kBlock) void k_refit_tris(uint32_t nf, const float* __restrict__ V, const uint32_t* __restrict__ F,
                                                       float4* __restrict__ tris, float4* __restrict__ normals) {
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= nf) return;
  float4 t0 = tris[3 * static_cast<size_t>(k)], t1 = tris[3 * static_cast<size_t>(k) + 1], t2 = tris[3 * static_cast<size_t>(k) + 2];
  const uint32_t f = __float_as_uint(t2.w);
  const uint32_t i0 = F[3 * f], i1 = F[3 * f + 1], i2 = F[3 * f + 2];
  t0.x = V[3 * i0]; t0.y = V[3 * i0 + 1]; t0.z = V[3 * i0 + 2];
  t1.x = V[3 * i1]; t1.y = V[3 * i1 + 1]; t1.z = V[3 * i1 + 2];
  t2.x = V[3 * i2]; t2.y = V[3 * i2 + 1]; t2.z = V[3 * i2 + 2];
  tris[3 * static_cast<size_t>(k)] = t0;
  tris[3 * static_cast<size_t>(k) + 1] = t1;
  tris[3 * static_cast<size_t>(k) + 2] = t2;
  const double ax = (double)t1.x - (double)t0.x, ay = (double)t1.y - (double)t0.y, az = (double)t1.z - (double)t0.z;
  const double bx = (double)t2.x - (double)t0.x, by = (double)t2.y - (double)t0.y, bz = (double)t2.z - (double)t0.z;
  const double nx = ay * bz - az * by, ny = az * bx - ax * bz, nz = ax * by - ay * bx;
  const double len = sqrt(nx * nx + ny * ny + nz * nz);
  float4 nrm = normals[k];
  nrm.x = len > 0.0 ? (float)(nx / len) : 0.0f;
  nrm.y = len > 0.0 ? (float)(ny / len) : 0.0f;
  nrm.z = len > 0.0 ? (float)(nz / len) : 0.0f;
  normals[k] = nrm;
}

__device__ inline void set_child_box(Node2& nd, int c, float4 lo, float4 hi) {
  if (c == 0) {
    nd.a.x = pad_lo(lo.x); nd.a.y = pad_hi(hi.x); nd.a.z = pad_lo(lo.y); nd.a.w = pad_hi(hi.y);
    nd.c.x = pad_lo(lo.z); nd.c.y = pad_hi(hi.z);
  } else {
    nd.b.x = pad_lo(lo.x); nd.b.y = pad_hi(hi.x); nd.b.z = pad_lo(lo.y); nd.b.w = pad_hi(hi.y);
    nd.c.z = pad_lo(lo.z); nd.c.w = pad_hi(hi.z);
  }
}

// Box updates go bottom-up through the tree in a few passes.  Nodes lie in preorder, so of a
// window of kWindow consecutive ones only the ancestors of the next window's first node have
// anything below them outside the window: a chain of at most one node per level.  A pass gives
// each window to one workgroup, which settles all its other nodes through the LDS; the
// chains, a few per cent of the nodes and again a tree in preorder, are the next pass's
// nodes.  1,048,576 vertices (one launch per level of the tree, 23 of them at 6.6 us, took
// 150 us): see k_refit_window.
constexpr uint32_t kWindow = 512;

// Lengths of the chains of a pass's windows, or (nodes given) the chains themselves, written at
// the windows' offsets in preorder.  up[k]: position in the pass of node k's parent.
__global__ __launch_bounds__(kBlock) void k_refit_chains(uint32_t n, const int* __restrict__ up, uint32_t* __restrict__ count,
                                                         const uint32_t* __restrict__ offset,
                                                         const uint32_t* __restrict__ from, uint32_t* __restrict__ nodes) {
  const uint32_t w = blockIdx.x * kBlock + threadIdx.x;
  if (static_cast<uint64_t>(w + 1) * kWindow >= n) return;  // nothing follows the last window
  const int lo = static_cast<int>(w * kWindow);
  uint32_t c = 0;
  for (int p = up[lo + kWindow]; p >= lo; p = up[p]) {
    if (nodes) nodes[offset[w + 1] - 1 - c] = from ? from[p] : static_cast<uint32_t>(p);
    c++;
  }
  if (count) count[w] = c;
}

// Position of x in the ascending list, -1 if it is not there.
__device__ __forceinline__ int list_position(const uint32_t* __restrict__ list, uint32_t n, uint32_t x) {
  uint32_t lo = 0, hi = n;  // the first position whose value is >= x
  while (lo < hi) {
    const uint32_t mid = (lo + hi) / 2;
    if (list[mid] < x) lo = mid + 1; else hi = mid;
  }
  return lo < n && list[lo] == x ? static_cast<int>(lo) : -1;
}

// Children and parents of a pass's nodes as positions in the pass.
__global__ __launch_bounds__(kBlock) void k_refit_links(uint32_t n, const uint32_t* __restrict__ list,
                                                        const Node2* __restrict__ nodes, const int* __restrict__ parent,
                                                        int* __restrict__ kids, int* __restrict__ up) {
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= n) return;
  const int4 d = nodes[list[k]].d;
  kids[2 * k] = d.x < 0 ? -1 : list_position(list, n, static_cast<uint32_t>(d.x));
  kids[2 * k + 1] = d.y < 0 ? -1 : list_position(list, n, static_cast<uint32_t>(d.y));
  const int p = parent[list[k]];
  up[k] = p < 0 ? -1 : list_position(list, n, static_cast<uint32_t>(p));
}

// Bounds of a leaf's triangles.
__device__ __forceinline__ void leaf_box(const float4* __restrict__ tris, int ref, float4& lo, float4& hi) {
  const uint32_t e = ~static_cast<uint32_t>(ref);
  const uint32_t first = e >> 3, cnt = (e & 7u) + 1u;
  lo = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
  hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
  for (uint32_t t = first; t < first + cnt; t++)
    for (int v = 0; v < 3; v++) {
      const float4 p = tris[3 * static_cast<size_t>(t) + v];
      lo.x = fminf(lo.x, p.x); lo.y = fminf(lo.y, p.y); lo.z = fminf(lo.z, p.z);
      hi.x = fmaxf(hi.x, p.x); hi.y = fmaxf(hi.y, p.y); hi.z = fmaxf(hi.z, p.z);
    }
}

// Union of a node's two (already padded) boxes.
__device__ __forceinline__ void union_box(const Node2& n, float4& lo, float4& hi) {
  lo = make_float4(fminf(n.a.x, n.b.x), fminf(n.a.z, n.b.z), fminf(n.c.x, n.c.z), 0.0f);
  hi = make_float4(fmaxf(n.a.y, n.b.y), fmaxf(n.a.w, n.b.w), fmaxf(n.c.y, n.c.w), 0.0f);
}

// One pass: a workgroup per window, a thread per node.  Leaf slots are boxed by the first pass
// (FIRST) from their triangles; a child of an earlier pass is read from its node; the other
// children are threads of the same workgroup, whose boxes go through the LDS round by round
// until a round settles nothing.  Nodes left then have a child beyond the window: the next
// pass holds exactly those.  The rounds cost barriers and LDS reads, not the memory latency
// and launch that a level of the whole tree costs.
template <bool FIRST>
__global__ __launch_bounds__(kWindow) void k_refit_window(uint32_t n, const uint32_t* __restrict__ list,
                                                          const int* __restrict__ kids, const float4* __restrict__ tris,
                                                          Node2* nodes) {
  __shared__ float box[6][kWindow];
  __shared__ uint8_t ready[kWindow];
  const uint32_t t = threadIdx.x, base = blockIdx.x * kWindow, k = base + t;
  const uint32_t size = n - base < kWindow ? n - base : kWindow;
  const bool mine = t < size;
  ready[t] = 0;
  Node2 nd;
  uint32_t i = 0;
  int wait[2] = {-1, -1};  // window positions of the children still to come
  bool beyond = false;
  if (mine) {
    i = FIRST ? k : list[k];
    nd = nodes[i];
    for (int c = 0; c < 2; c++) {
      const int ref = c ? nd.d.y : nd.d.x;
      float4 lo, hi;
      if (ref < 0) {
        if constexpr (FIRST) {
          leaf_box(tris, ref, lo, hi);
          set_child_box(nd, c, lo, hi);
        }
        continue;
      }
      const int kid = FIRST ? ref : kids[2 * k + c];
      if (kid < 0) {
        union_box(nodes[ref], lo, hi);
        set_child_box(nd, c, lo, hi);
      } else if (static_cast<uint32_t>(kid) - base < size) {
        wait[c] = kid - static_cast<int>(base);
      } else {
        beyond = true;
      }
    }
  }
  bool todo = mine && !beyond;
  __syncthreads();
  for (;;) {
    if (todo) {
      for (int c = 0; c < 2; c++)
        if (wait[c] >= 0 && ready[wait[c]]) {
          const int j = wait[c];
          set_child_box(nd, c, make_float4(box[0][j], box[1][j], box[2][j], 0.0f),
                        make_float4(box[3][j], box[4][j], box[5][j], 0.0f));
          wait[c] = -1;
        }
    }
    const bool settled = todo && wait[0] < 0 && wait[1] < 0;
    if (!__syncthreads_or(settled)) break;  // also: every thread is done reading this round
    if (settled) {
      float4 lo, hi;
      union_box(nd, lo, hi);
      box[0][t] = lo.x; box[1][t] = lo.y; box[2][t] = lo.z;
      box[3][t] = hi.x; box[4][t] = hi.y; box[5][t] = hi.z;
      ready[t] = 1;
      todo = false;
    }
    __syncthreads();
  }
  if (mine && (FIRST || (!todo && !beyond))) {
    nodes[i].a = nd.a;
    nodes[i].b = nd.b;
    nodes[i].c = nd.c;
  }
}

// The passes of a map (once: the tree's topology never changes after the build).
hipError_t make_refit_passes(rmh_map* m, hipStream_t stream) {
  std::vector<RefitPass> passes(1);
  passes[0].n = m->n_internal;
  int* up = nullptr;  // parent positions of the current pass; the first pass uses m->parent
  uint32_t* lens = nullptr;
  hipError_t e = hipMalloc(&lens, sizeof(uint32_t) * (2 * (m->n_internal / kWindow + 1) + 2));
  while (e == hipSuccess && passes.back().n > kWindow) {
    const RefitPass cur = passes.back();
    const uint32_t nw = (cur.n + kWindow - 1) / kWindow;  // windows; the last has no chain
    uint32_t* offs = lens + nw;
    const int* cur_up = cur.nodes ? up : m->parent;
    std::vector<uint32_t> h(nw), off(nw + 1, 0);
    k_refit_chains<<<blocks_for(nw), kBlock, 0, stream>>>(cur.n, cur_up, lens, nullptr, cur.nodes, nullptr);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(h.data(), lens, sizeof(uint32_t) * (nw - 1), hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess) break;
    for (uint32_t w = 0; w + 1 < nw; w++) off[w + 1] = off[w] + h[w];
    RefitPass next;
    next.n = off[nw - 1];
    if (next.n == 0 || next.n >= cur.n) { e = hipErrorInvalidValue; break; }  // a tree deeper than a window is wide
    uint32_t* mem = nullptr;
    int* next_up = nullptr;
    e = hipMalloc(&mem, sizeof(uint32_t) * 3 * next.n);
    if (e == hipSuccess) {
      next.nodes = mem;
      next.kids = reinterpret_cast<int*>(mem + next.n);
      passes.push_back(next);
      e = hipMalloc(&next_up, sizeof(int) * next.n);
    }
    if (e == hipSuccess) e = hipMemcpyAsync(offs, off.data(), sizeof(uint32_t) * nw, hipMemcpyHostToDevice, stream);
    if (e == hipSuccess) {
      k_refit_chains<<<blocks_for(nw), kBlock, 0, stream>>>(cur.n, cur_up, nullptr, offs, cur.nodes, next.nodes);
      k_refit_links<<<blocks_for(next.n), kBlock, 0, stream>>>(next.n, next.nodes, m->nodes, m->parent, next.kids, next_up);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (up) (void)hipFree(up);
    up = next_up;
  }
  if (up) (void)hipFree(up);
  if (lens) (void)hipFree(lens);
  if (e != hipSuccess) {
    for (const RefitPass& r : passes)
      if (r.nodes) (void)hipFree(r.nodes);
    return e;
  }
  m->refit_passes = std::move(passes);
  return hipSuccess;
}

extern "C" int rmh_map_refit(rmh_map* map, const float* vertices, void* stream_) {
  if (!map) return fail(RMH_ERR_INVALID, "rmh_map_refit: NULL map");
  if (map->n_faces == 0) return RMH_OK;
  if (!vertices) return fail(RMH_ERR_INVALID, "rmh_map_refit: NULL vertices");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  RMH_HIP_TRY(hipMemcpyAsync(map->vertices, vertices, sizeof(float) * 3 * static_cast<size_t>(map->n_vertices),
                             hipMemcpyDeviceToDevice, stream));
  k_refit_tris<<<blocks_for(map->n_faces), kBlock, 0, stream>>>(map->n_faces, map->vertices, map->faces, map->tris,
                                                                 map->normals);
  RMH_HIP_TRY(hipGetLastError());
  if (map->root >= 0 && map->n_internal > 0) {
    if (map->refit_passes.empty()) {
      const hipError_t e = make_refit_passes(map, stream);
      if (e != hipSuccess) return hip_fail(e, "rmh_map_refit: passes");
    }
    // a pass reads only what earlier launches wrote, and its own window through the LDS
    hipError_t e = hipSuccess;
    for (const RefitPass& r : map->refit_passes) {
      const uint32_t blocks = (r.n + kWindow - 1) / kWindow;
      if (!r.nodes) k_refit_window<true><<<blocks, kWindow, 0, stream>>>(r.n, nullptr, nullptr, map->tris, map->nodes);
      else k_refit_window<false><<<blocks, kWindow, 0, stream>>>(r.n, r.nodes, r.kids, map->tris, map->nodes);
      if ((e = hipGetLastError()) != hipSuccess) break;
    }
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return hip_fail(e, "rmh_map_refit");
    // the 4-wide tree is collapsed again from the refitted binary boxes
    if (map->nodes4) {
      const uint64_t before = sizeof(Node4) * static_cast<uint64_t>(map->info.n_wide_nodes);
      e = build_wide(map, stream);
      if (e != hipSuccess) {
        free_wide(map);  // never leave a half-written tree for the ray kernels
        return hip_fail(e, "rmh_map_refit: 4-wide tree");
      }
      map->info.device_bytes = map->info.device_bytes - before + sizeof(Node4) * static_cast<uint64_t>(map->info.n_wide_nodes);
    }
  }
  return RMH_OK;
}

extern "C" int rmh_map_set_layout(rmh_map* map, int wide, void* stream_) {
  if (!map) return fail(RMH_ERR_INVALID, "rmh_map_set_layout: NULL map");
  const uint64_t before = sizeof(Node4) * static_cast<uint64_t>(map->info.n_wide_nodes);
  if (wide) {
    if (!map->nodes4) {
      const hipError_t e = build_wide(map, static_cast<hipStream_t>(stream_));
      if (e != hipSuccess) {
        free_wide(map);
        return hip_fail(e, "rmh_map_set_layout");
      }
    }
  } else if (map->nodes4) {
    RMH_HIP_TRY(hipDeviceSynchronize());
    free_wide(map);
  }
  map->info.device_bytes = map->info.device_bytes - before + sizeof(Node4) * static_cast<uint64_t>(map->info.n_wide_nodes);
  return RMH_OK;
}

extern "C" int rmh_map_get_info(const rmh_map* map, rmh_map_info* info) {
  if (!map || !info) return fail(RMH_ERR_INVALID, "rmh_map_get_info: NULL argument");
  *info = map->info;
  return RMH_OK;
}
