// Pose adjoint of librmh: gradients of a Huber range-residual loss with respect to 6-DoF
// sensor poses, through the hit triangle's plane.  The reference has no differentiable
// path; the closest pieces are its point-to-plane Jacobian
// (src/rmagine_core/include/rmagine/math/optimization.h:113-137) and the SE(3)
// exponential / SO(3) left Jacobian (src/rmagine_core/include/rmagine/math/lie.tcc:252-277).
//
// For pose p (base -> map transform Tbm = (R, t)) and ray k the forward pass is the same
// closest-hit query as simulate() (FP64 distance r to the hit triangle with unit world
// normal n, ray origin o and direction d in the map frame).  With a target range r*_k the
// loss is L_p = sum_k rho(r_k - r*_k), rho the Huber function with threshold delta, over
// rays that hit (r >= range.min) and whose target is valid.  The pose is perturbed on the
// left in the map frame, t -> t + tau, R -> Exp(omega) R; then
//   dr/dtau   = g,                      g = -n / (n . d)
//   dr/domega = (o + r d - t) x g       (lever arm from the base origin to the hit point)
// and dL/d(tau, omega) = sum_k rho'(e_k) dr_k/d(tau, omega).  Per ray in FP64, reduced per
// pose in FP64 (wave shuffles within each 64-ray tile, then the tiles of a pose in a fixed
// order).
//
// Output per pose: 8 doubles {L, dL/dtau (3), dL/domega (3), number of rays used}.
#include "rmh_trace.hpp"
#include "rmh_wave_sum.hpp"

#include <algorithm>

namespace {

using namespace rmh;

struct GradArgs {
  MapData map;
  RayGen g;
  Tf Tsb;
  const rmh_transform* Tbm;
  uint32_t pose_offset;
  const float* target;
  const uint8_t* target_mask;
  uint32_t target_stride;     // 0: one target scan shared by all poses; else ray_count
  double delta;
  Tiling tl;                  // one 64-ray tile per workgroup; chunks = tiles per pose
  double* partial;            // (pose, tile) -> 8 doubles
};

constexpr int kWave = 64;

template <int KIND, int STACK, bool WIDE>
__global__ __launch_bounds__(kWave, 8) void k_pose_grad(const GradArgs a) {
  __shared__ int2 stk[kLdsStack][kWave];
  // plain pose-major order: contiguous or dealt ranges per XCD measured the same (2,000
  // particles in a room, whose mesh fits every XCD's L2: 1.148 ms against 1.144 and 1.141), one
  // slice of the tiles per XCD 1.265
  const uint32_t pl = fast_div(blockIdx.x, a.tl.div_tiles);
  const uint32_t tile = blockIdx.x - pl * a.tl.tiles;
  const uint32_t pose = a.pose_offset + pl;
  uint32_t vid, hid;
  const bool active = tile_ray(a.tl, a.g.grid_w, a.g.grid_h, tile, threadIdx.x, vid, hid);
  Acc<8> acc = {};
  if (active) {
    uint32_t lid;
    V3 ds, os;
    gen_ray<KIND>(a.g, vid, hid, lid, ds, os);
    const Tf Tbm = load_tf(a.Tbm[pose]);
    const Tf Tsm = uniform(tmul(Tbm, a.Tsb));
    const V3 dm = qrot(Tsm.R, ds);
    const V3 om = map_origin<KIND>(Tsm, os);
    Hit h;
    trace<STACK, kWave, WIDE, spec_mode<KIND>()>(a.map, om, dm, a.g.range_max, stk, h);
    const size_t ti = static_cast<size_t>(pose) * a.target_stride + lid;
    const float tr = a.target[ti];
    const bool tvalid = a.target_mask ? (a.target_mask[ti] != 0) : (tr >= a.g.range_min && tr <= a.g.range_max);
    if (h.slot != 0xFFFFFFFFu && static_cast<float>(h.t) >= a.g.range_min && tvalid) {
      const float4 nn = a.map.normals[h.slot];
      const double nx = nn.x, ny = nn.y, nz = nn.z;
      const double dx = dm.x, dy = dm.y, dz = dm.z;
      const double nd = nx * dx + ny * dy + nz * dz;
      if (nd != 0.0) {
        const double delta = a.delta;
        const double e = h.t - static_cast<double>(tr);
        const double ae = fabs(e);
        const double rho = ae <= delta ? 0.5 * e * e : delta * (ae - 0.5 * delta);
        const double drho = ae <= delta ? e : (e > 0 ? delta : -delta);
        const double gx = -nx / nd, gy = -ny / nd, gz = -nz / nd;
        const double lx = (double)om.x + h.t * dx - (double)Tbm.t.x;
        const double ly = (double)om.y + h.t * dy - (double)Tbm.t.y;
        const double lz = (double)om.z + h.t * dz - (double)Tbm.t.z;
        acc.v[0] = rho;
        acc.v[1] = drho * gx;
        acc.v[2] = drho * gy;
        acc.v[3] = drho * gz;
        acc.v[4] = drho * (ly * gz - lz * gy);
        acc.v[5] = drho * (lz * gx - lx * gz);
        acc.v[6] = drho * (lx * gy - ly * gx);
        acc.v[7] = 1.0;
      }
    }
  }
  // value k in lanes [8 k, 8 k + 8); with a butterfly of LDS permutes per value 2,000 particles
  // took 1,151 us instead of 1,113 (recomputing the ray set-up here, as k_simulate does, 1,147)
  const double s = wave_sum(acc);
  const uint32_t lane = threadIdx.x;
  if ((lane & 7u) == 0) a.partial[(static_cast<size_t>(pose) * a.tl.tiles + tile) * 8 + (lane >> 3)] = s;
}

// Sums the tiles' partials of every pose in a fixed order, one wave per pose: 8 lanes side by
// side over the values, 8 over the tiles (one thread per pose and value, walking all tiles,
// took 43 us for 2,000 poses of 225 tiles).  With xi, the sums of the perturbed poses become
// the loss and its gradient with respect to xi: out is then the losses, grad 6 doubles per
// pose, J_l(omega)^T applied to the rotation part (J_l = I + c1 W + c2 W^2 the SO(3) left
// Jacobian, W = [omega]x).
__global__ __launch_bounds__(256) void k_pose_grad_combine(const double* __restrict__ partial, uint32_t chunks,
                                                           uint32_t n_poses, double* __restrict__ out,
                                                           const double* __restrict__ xi, double* __restrict__ grad) {
  const uint32_t p = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x & 63u;
  if (p >= n_poses) return;
  const uint32_t k = lane & 7u;
  const double* v = partial + static_cast<size_t>(p) * chunks * 8 + k;
  double s = 0.0;
#pragma unroll 4
  for (uint32_t c = lane >> 3; c < chunks; c += 8) s += v[static_cast<size_t>(c) * 8];
  for (int off = 8; off < 64; off <<= 1) s += __shfl_xor(s, off, 64);
  if (!xi) {
    if (lane < 8) out[static_cast<size_t>(p) * 8 + k] = s;
    return;
  }
  const double gx = __shfl(s, 4, 64), gy = __shfl(s, 5, 64), gz = __shfl(s, 6, 64);
  if (lane == 0) out[p] = s;
  if (lane >= 1 && lane <= 3) grad[static_cast<size_t>(p) * 6 + lane - 1] = s;
  if (lane != 0) return;
  const double* x = xi + static_cast<size_t>(p) * 6;
  const double wx = x[3], wy = x[4], wz = x[5];
  const double a2 = wx * wx + wy * wy + wz * wz, a = sqrt(a2);
  const bool small = a < 1e-6;
  const double c1 = small ? 0.5 - a * a / 24.0 : (1.0 - cos(a)) / (a * a);
  const double c2 = small ? 1.0 / 6.0 - a * a / 120.0 : (a - sin(a)) / (a * a * a);
  // W^T g = g x w and (W^2)^T g = (g x w) x w
  const double ux = gy * wz - gz * wy, uy = gz * wx - gx * wz, uz = gx * wy - gy * wx;
  const double tx = uy * wz - uz * wy, ty = uz * wx - ux * wz, tz = ux * wy - uy * wx;
  double* g = grad + static_cast<size_t>(p) * 6 + 3;
  g[0] = gx + c1 * ux + c2 * tx;
  g[1] = gy + c1 * uy + c2 * ty;
  g[2] = gz + c1 * uz + c2 * tz;
}

// Poses (t0 + tau, Exp(omega) R0) of xi = (tau, omega), the quaternion product in FP64 and
// rounded once.
__global__ __launch_bounds__(256) void k_pose_perturb(const rmh_transform* __restrict__ T0, const double* __restrict__ xi,
                                                      uint32_t n, rmh_transform* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const double* x = xi + static_cast<size_t>(i) * 6;
  const rmh_transform T = T0[i];
  const double a = sqrt(x[3] * x[3] + x[4] * x[4] + x[5] * x[5]), half = 0.5 * a;
  const double s = a > 0.0 ? sin(half) / a : 0.5;
  const double x1 = x[3] * s, y1 = x[4] * s, z1 = x[5] * s, w1 = cos(half);
  const double x2 = T.R.x, y2 = T.R.y, z2 = T.R.z, w2 = T.R.w;
  rmh_transform r;
  r.R.x = static_cast<float>(w1 * x2 + x1 * w2 + y1 * z2 - z1 * y2);
  r.R.y = static_cast<float>(w1 * y2 - x1 * z2 + y1 * w2 + z1 * x2);
  r.R.z = static_cast<float>(w1 * z2 + x1 * y2 - y1 * x2 + z1 * w2);
  r.R.w = static_cast<float>(w1 * w2 - x1 * x2 - y1 * y2 - z1 * z2);
  r.t.x = static_cast<float>(static_cast<double>(T.t.x) + x[0]);
  r.t.y = static_cast<float>(static_cast<double>(T.t.y) + x[1]);
  r.t.z = static_cast<float>(static_cast<double>(T.t.z) + x[2]);
  r.stamp = 0;
  out[i] = r;
}

template <int KIND, int STACK, bool WIDE>
hipError_t launch_grad(const GradArgs& a, uint32_t np, hipStream_t stream) {
  k_pose_grad<KIND, STACK, WIDE><<<np * a.tl.tiles, kWave, 0, stream>>>(a);
  return hipGetLastError();
}

template <int STACK, bool WIDE>
hipError_t launch_grad_stack(int kind, const GradArgs& a, uint32_t np, hipStream_t stream) {
  switch (kind) {
    case RMH_MODEL_SPHERICAL: return launch_grad<RMH_MODEL_SPHERICAL, STACK, WIDE>(a, np, stream);
    case RMH_MODEL_PINHOLE: return launch_grad<RMH_MODEL_PINHOLE, STACK, WIDE>(a, np, stream);
    case RMH_MODEL_O1DN: return launch_grad<RMH_MODEL_O1DN, STACK, WIDE>(a, np, stream);
    default: return launch_grad<RMH_MODEL_ONDN, STACK, WIDE>(a, np, stream);
  }
}

hipError_t launch_grad_sel(const TravSel& ts, int kind, const GradArgs& a, uint32_t np, hipStream_t stream) {
  if (ts.wide) {
    if (ts.stack == 32) return launch_grad_stack<32, true>(kind, a, np, stream);
    if (ts.stack == 64) return launch_grad_stack<64, true>(kind, a, np, stream);
    return launch_grad_stack<128, true>(kind, a, np, stream);
  }
  if (ts.stack == 32) return launch_grad_stack<32, false>(kind, a, np, stream);
  if (ts.stack == 64) return launch_grad_stack<64, false>(kind, a, np, stream);
  return launch_grad_stack<128, false>(kind, a, np, stream);
}

struct Scratch {
  void* p = nullptr;
  ~Scratch() { if (p) (void)hipFree(p); }
};

size_t partial_bytes(const rmh_sensor* sensor, uint32_t n_poses) {
  return sizeof(double) * 8 * static_cast<size_t>(sensor_tiling(sensor).tiles) * n_poses;
}

// rmh_pose_grad (xi NULL) and rmh_pose_loss.  Workspace: the partials, then the perturbed poses.
int pose_grad(const char* who, const rmh_map* map, const rmh_sensor* sensor, const rmh_transform* Tsb,
              const rmh_transform* Tbm, const double* xi, uint32_t n_poses, const float* target,
              const uint8_t* target_mask, int per_pose_targets, float huber_delta, double* out, double* grad,
              void* workspace, size_t workspace_bytes, void* stream_) {
  const std::string w(who);
  if (!map) return fail(RMH_ERR_NOMAP, w + ": no map set");
  if (!sensor || !out || !target) return fail(RMH_ERR_INVALID, w + ": NULL argument");
  if (n_poses == 0) return RMH_OK;
  if (n_poses > (1u << 28)) return fail(RMH_ERR_UNSUPPORTED, w + ": too many poses");
  if (!Tbm) return fail(RMH_ERR_INVALID, w + ": poses are NULL");
  if (!(huber_delta > 0.0f)) return fail(RMH_ERR_INVALID, w + ": huber_delta must be > 0");
  const TravSel ts = trav_select(map);
  if (ts.stack < 0) return fail(RMH_ERR_UNSUPPORTED, w + ": BVH deeper than 128 levels");
  const uint64_t rc = static_cast<uint64_t>(sensor->width) * sensor->height;
  if (rc == 0 || rc > (1ull << 30)) return fail(RMH_ERR_UNSUPPORTED, w + ": bad ray count");
  GradArgs a;
  a.map = make_mapdata(map);
  a.g = make_raygen(sensor);
  rmh_transform I{};
  I.R.w = 1.0f;
  a.Tsb = load_tf(Tsb ? *Tsb : I);
  a.Tbm = Tbm;
  a.target = target;
  a.target_mask = target_mask;
  a.target_stride = per_pose_targets ? static_cast<uint32_t>(rc) : 0u;
  a.delta = huber_delta;
  a.tl = sensor_tiling(sensor);
  if (a.tl.tiles > 65535u) return fail(RMH_ERR_UNSUPPORTED, w + ": more than 65535 ray tiles per pose");
  const size_t sums = partial_bytes(sensor, n_poses);
  const size_t need = sums + (xi ? sizeof(rmh_transform) * static_cast<size_t>(n_poses) : 0);
  Scratch scratch;
  if (workspace) {
    if (workspace_bytes < need) return fail(RMH_ERR_INVALID, w + ": workspace too small");
  } else {
    RMH_HIP_TRY(hipMalloc(&scratch.p, need));
  }
  char* ws = static_cast<char*>(workspace ? workspace : scratch.p);
  a.partial = reinterpret_cast<double*>(ws);
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (xi) {
    rmh_transform* Tp = reinterpret_cast<rmh_transform*>(ws + sums);
    k_pose_perturb<<<(n_poses + 255u) / 256u, 256, 0, stream>>>(Tbm, xi, n_poses, Tp);
    RMH_HIP_TRY(hipGetLastError());
    a.Tbm = Tp;
  }
  const uint32_t poses_per_launch = static_cast<uint32_t>(kMaxTileBlocks / a.tl.tiles);  // >= 512
  for (uint32_t p0 = 0; p0 < n_poses; p0 += poses_per_launch) {
    const uint32_t np = std::min<uint32_t>(poses_per_launch, n_poses - p0);
    a.pose_offset = p0;
    const hipError_t e = launch_grad_sel(ts, sensor->kind, a, np, stream);
    if (e != hipSuccess) return hip_fail(e, (w + " launch").c_str());
  }
  k_pose_grad_combine<<<(n_poses + 3u) / 4u, 256, 0, stream>>>(a.partial, a.tl.tiles, n_poses, out, xi, grad);
  RMH_HIP_TRY(hipGetLastError());
  if (scratch.p) RMH_HIP_TRY(hipStreamSynchronize(stream));
  return RMH_OK;
}

}  // namespace

extern "C" {

int rmh_pose_grad_workspace_size(const rmh_map* map, const rmh_sensor* sensor, uint32_t n_poses, size_t* bytes) {
  if (!map || !sensor || !bytes) return fail(RMH_ERR_INVALID, "rmh_pose_grad_workspace_size: NULL argument");
  *bytes = partial_bytes(sensor, n_poses);
  return RMH_OK;
}

int rmh_pose_grad(const rmh_map* map, const rmh_sensor* sensor, const rmh_transform* Tsb, const rmh_transform* Tbm,
                  uint32_t n_poses, const float* target, const uint8_t* target_mask, int per_pose_targets,
                  float huber_delta, double* out, void* workspace, size_t workspace_bytes, void* stream_) {
  return pose_grad("rmh_pose_grad", map, sensor, Tsb, Tbm, nullptr, n_poses, target, target_mask, per_pose_targets,
                   huber_delta, out, nullptr, workspace, workspace_bytes, stream_);
}

int rmh_pose_loss_workspace_size(const rmh_map* map, const rmh_sensor* sensor, uint32_t n_poses, size_t* bytes) {
  if (!map || !sensor || !bytes) return fail(RMH_ERR_INVALID, "rmh_pose_loss_workspace_size: NULL argument");
  *bytes = partial_bytes(sensor, n_poses) + sizeof(rmh_transform) * static_cast<size_t>(n_poses);
  return RMH_OK;
}

int rmh_pose_loss(const rmh_map* map, const rmh_sensor* sensor, const rmh_transform* Tsb, const rmh_transform* T0,
                  const double* xi, uint32_t n_poses, const float* target, const uint8_t* target_mask,
                  int per_pose_targets, float huber_delta, double* loss, double* grad, void* workspace,
                  size_t workspace_bytes, void* stream_) {
  if (n_poses > 0 && (!xi || !grad)) return fail(RMH_ERR_INVALID, "rmh_pose_loss: NULL argument");
  return pose_grad("rmh_pose_loss", map, sensor, Tsb, T0, xi, n_poses, target, target_mask, per_pose_targets,
                   huber_delta, loss, grad, workspace, workspace_bytes, stream_);
}

}  // extern "C"
