// gfx950 kernels of the batch raytrace query (VDBMapping.hpp:675-721).
//
// The reference marches each ray with openvdb::tools::VolumeRayIntersector
// built by updateVolumeRayIntersectors (VDBMapping.hpp:1436-1449): a topology
// copy of the map at that moment, walked by a hierarchical DDA over node sizes
// 4096 -> 128 -> 8 (math::VolumeHDDA), then a voxel DDA that stops at the first
// active voxel of the live map. Here the topology copy is a snapshot of three
// device sets (a bit per leaf under a hash of 128^3 nodes, a hash of 4096^3
// nodes) plus the padded bounding box of the leaves holding an active voxel;
// one lane walks one ray with exactly the double-precision operations of
// math::Ray / math::DDA. The steps themselves cannot be skipped (their times
// are accumulated sums), so the lookups beside them are what there is to save:
// a leaf step reads a bit of a word it mostly holds already, a voxel step
// tests the OR of its leaf's mask words first.
//
// Build with -ffp-contract=off (every double operation rounds on its own).
#include <float.h>

#include "device_common.h"
#include "kernels.h"
#include "rt_common.h"

namespace vdbgpu {

__device__ __forceinline__ int rt_lane() { return (int)__lane_id(); }

// Start of a snapshot build: empty bbox, the leaf count at this point of the
// stream, and on a full build no nodes.
__global__ void k_snapshot_begin(RtInfo* info, const Status* stmap, uint32_t full) {
  if (threadIdx.x == 0) {
    for (int a = 0; a < 3; ++a) {
      info->bbox[a] = INT_MAX;
      info->bbox[3 + a] = INT_MIN;
    }
    info->leaves = stmap->leaf_count;
    if (full) info->nodes = 0;
  }
}

// Nodes of the snapshot: the 128^3 and 4096^3 parents of the leaves from
// `first` on (leaves are only ever appended to the pool, so the earlier ones
// are in), the root children of updates that created no leaf (value and state
// unchanged, e.g. probability 0.5), and the leaf-granular bounding box of
// active voxels (evalActiveBoundingBox with visitVoxels = false) of all
// leaves. Every atomic is preceded by a read: the parents and the box are the
// same few addresses for the whole grid (116 us of a fast-mode scan with an
// atomic per leaf).
__global__ __launch_bounds__(256) void k_snapshot_nodes(MapView mp, uint32_t first, RtView rt, RtInfo* info,
                                                        const unsigned long long* __restrict__ noop,
                                                        uint32_t noop_cap, uint32_t old_nodes) {
  __shared__ int smin[3][4], smax[3][4];
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
  const uint32_t leaf_count = info->leaves;
  const uint32_t G = gridDim.x * blockDim.x, t = blockIdx.x * blockDim.x + threadIdx.x;
  for (uint32_t i = t; i < noop_cap; i += G)
    if (noop[i] != kEmpty) set_add(rt.n4096, rt.n4096_mask, noop[i]);
  // active leaves are listed anew by the next launch
  for (uint64_t i = t; i < (uint64_t)old_nodes * 64; i += G) rt.bits[2 * i + 1] = 0;
  for (uint32_t i = t; i < leaf_count; i += G) {
    int o[3];
    key_origin(mp.leaf_keys[i], o);
    uint64_t any = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) any |= mp.active[(size_t)i * 8 + j];
    if (any) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        lo[a] = min(lo[a], o[a]);
        hi[a] = max(hi[a], o[a] + 7);
      }
    }
    if (i < first) continue;
    const uint64_t key = node_key(o[0], o[1], o[2], 7);
    uint32_t h = (uint32_t)fmix64(key) & rt.n128_mask;
    for (uint32_t p = 0; p <= rt.n128_mask; ++p) {
      unsigned long long k = __hip_atomic_load(&rt.n128[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (k == kEmpty) {
        k = atomicCAS(&rt.n128[h], kEmpty, (unsigned long long)key);
        if (k == kEmpty) {  // a new node: its index is read by the next launch
          rt.nidx[h] = atomicAdd(&info->nodes, 1u);
          set_add(rt.n4096, rt.n4096_mask, node_key(o[0], o[1], o[2], 12));
          break;
        }
      }
      if (k == key) break;
      h = (h + 1) & rt.n128_mask;
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    for (int off = 32; off > 0; off >>= 1) {
      lo[a] = min(lo[a], __shfl_xor(lo[a], off, 64));
      hi[a] = max(hi[a], __shfl_xor(hi[a], off, 64));
    }
  }
  const int w = threadIdx.x >> 6;
  if (rt_lane() == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      smin[a][w] = lo[a];
      smax[a][w] = hi[a];
    }
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int a = threadIdx.x;
    int l = INT_MAX, h = INT_MIN;
    for (int k = 0; k < (int)(blockDim.x >> 6); ++k) {
      l = min(l, smin[a][k]);
      h = max(h, smax[a][k]);
    }
    if (l < __hip_atomic_load(&info->bbox[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMin(&info->bbox[a], l);
    if (h > __hip_atomic_load(&info->bbox[3 + a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(&info->bbox[3 + a], h);
  }
}

// Leaf bits of the leaves from `first` on, active bits of all. An inactive
// tile is neither a leaf nor an active value for the HDDA; an active tile is a
// hit at the leaf level, as a leaf is.
__global__ __launch_bounds__(256) void k_snapshot_bits(MapView mp, uint32_t first, RtView rt, const RtInfo* info,
                                                       TileView tv) {
  const uint32_t leaf_count = info->leaves;
  const uint32_t G = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < leaf_count; i += G) {
    uint64_t any = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) any |= mp.active[(size_t)i * 8 + j];
    const bool leaf = i >= first && !(tile_at(tv, i) && !tile_active(tv, i));
    if (!leaf && !any) continue;
    int o[3];
    key_origin(mp.leaf_keys[i], o);
    const uint64_t key = node_key(o[0], o[1], o[2], 7);
    uint32_t h = (uint32_t)fmix64(key) & rt.n128_mask;
    for (uint32_t p = 0; p <= rt.n128_mask; ++p) {
      const unsigned long long k = rt.n128[h];
      if (k == key) {
        unsigned long long* w = &rt.bits[(size_t)rt.nidx[h] * kRtNodeWords + 2 * rt_word(o[0], o[1], o[2])];
        const unsigned long long bit = 1ull << rt_bit(o[0], o[1], o[2]);
        if (leaf) atomicOr(&w[0], bit);
        if (any) atomicOr(&w[1], bit);
        break;
      }
      if (k == kEmpty) break;
      h = (h + 1) & rt.n128_mask;
    }
  }
}

// One lane per query ray. Mirrors VDBMapping::raytrace: normalise (multiply by
// 1/length unless length <= 1e-7), scale by the max length, continuous
// worldToIndex, clip to the padded bbox (result ignored), VolumeHDDA march,
// then a voxel DDA over the first leaf run that stops at an active voxel.
__global__ __launch_bounds__(256, 4) void k_raytrace(RtView rt, MapView mp, double inv, double res,
                                                  int64_t n, const double* __restrict__ origins,
                                                  const double* __restrict__ dirs,
                                                  const double* __restrict__ lens,
                                                  uint8_t* __restrict__ success,
                                                  double* __restrict__ ends,
                                                  unsigned int* __restrict__ err, int spread) {
  const int64_t G = ((int64_t)gridDim.x * blockDim.x) >> spread;
  if (threadIdx.x & ((1 << spread) - 1)) return;
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> spread; i < n; i += G) {
    double d[3] = {dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]};
    const double len = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    if (!(fabs(0.0 - len) <= 1e-7)) {
      const double r = 1.0 / len;
      d[0] *= r;
      d[1] *= r;
      d[2] *= r;
    }
    const double L = lens[i];
    RtRay r;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      d[a] *= L;
      r.eye[a] = origins[3 * i + a] * inv;
      r.dir[a] = d[a] * inv;
      r.idir[a] = 1.0 / r.dir[a];
    }
    // A query whose DDA cannot end (non-finite numbers) or would take more
    // than kMaxQuerySteps voxel steps is rejected instead of marched.
    const double span = fabs(r.dir[0]) + fabs(r.dir[1]) + fabs(r.dir[2]);
    if (!(isfinite(r.eye[0]) && isfinite(r.eye[1]) && isfinite(r.eye[2]) && isfinite(span) &&
          span < (double)kMaxQuerySteps)) {
      atomicOr(err, 1u);
      success[i] = 0;
      ends[3 * i] = ends[3 * i + 1] = ends[3 * i + 2] = NAN;
      continue;
    }
    // every DDA level takes at most span/dim + 3 steps over t in [0, 1]
    int budget = 4 * ((int)span + 8);
    double rt0 = 0.0, rt1 = 1.0;
    rt_clip(rt, r, rt0, rt1);  // Ray::clip to the padded active bbox
    double s0 = -1, s1 = -1;   // TimeSpan of the first leaf run
    LeafBits lb;
    bool run = false;
    if ((rt1 - rt0) > (double)1e-5f) {  // Ray::valid
      SpanFinder<true, 8> f;
      f.init(r, rt0, rt1);
      run = f.next(rt, r, lb, budget, s0, s1);
    }
    double* out = ends + 3 * i;
    if (run) {
      RtDda<1> fd;
      fd.init(r, s0, s1);
      ActiveProbe probe;
      // to the first active voxel after the first one; a leaf without any is
      // left in one go
      bool can_skip = true;  // refused once: the run ends in that leaf
      for (;;) {
        int n = 1;
        bool moved = can_skip && !probe.leaf(mp, rt, lb, fd.vox);
        if (moved) moved = can_skip = fd.skip<8>(r, n);
        if (!moved && !fd.step(r)) break;
        budget -= n - 1;
        if (probe.leaf(mp, rt, lb, fd.vox) && probe.on(mp, fd.vox)) break;
        if (--budget <= 0) break;
      }
      if (budget <= 0) atomicOr(err, 2u);
#pragma unroll
      for (int a = 0; a < 3; ++a) out[a] = (double)fd.vox[a] * res;
      success[i] = 1;
    } else {
#pragma unroll
      for (int a = 0; a < 3; ++a) out[a] = (r.eye[a] + r.dir[a]) * res;
      success[i] = 0;
    }
  }
}

hipError_t launch_snapshot_nodes(hipStream_t s, MapView mp, uint32_t first, uint64_t leaf_bound, RtView rt,
                                 RtInfo* info, const unsigned long long* noop, uint32_t noop_cap,
                                 uint32_t old_nodes, const Status* stmap, bool full) {
  hipLaunchKernelGGL(k_snapshot_begin, dim3(1), dim3(64), 0, s, info, stmap, full ? 1u : 0u);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int grid = (int)std::min<uint64_t>(2048, (std::max<uint64_t>(leaf_bound, noop_cap) + 255) / 256);
  hipLaunchKernelGGL(k_snapshot_nodes, dim3(grid), dim3(256), 0, s, mp, first, rt, info, noop, noop_cap, old_nodes);
  return hipGetLastError();
}

hipError_t launch_snapshot_bits(hipStream_t s, MapView mp, uint32_t first, uint32_t leaf_count, RtView rt,
                                const RtInfo* info, TileView tv) {
  if (leaf_count == 0) return hipSuccess;
  const int grid = (int)std::min<uint32_t>(2048, (leaf_count + 255) / 256);
  hipLaunchKernelGGL(k_snapshot_bits, dim3(grid), dim3(256), 0, s, mp, first, rt, info, tv);
  return hipGetLastError();
}

hipError_t launch_raytrace(hipStream_t s, int num_cu, RtView rt, MapView mp, double inv, double res,
                           int64_t n, const double* origins, const double* dirs,
                           const double* lens, uint8_t* success, double* ends,
                           unsigned int* err) {
  const int spread = ray_spread(n, num_cu);
  const int grid = (int)std::min<int64_t>((int64_t)num_cu * 16, ((n << spread) + 255) / 256);
  hipLaunchKernelGGL(k_raytrace, dim3(grid), dim3(256), 0, s, rt, mp, inv, res, n, origins, dirs,
                     lens, success, ends, err, spread);
  return hipGetLastError();
}

}  // namespace vdbgpu
