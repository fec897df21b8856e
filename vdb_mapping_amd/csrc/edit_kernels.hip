// gfx950 kernels of the direct map edits, artificial areas and map sections.
//
//   k_mark_points     addPointsToGrid / removePointsFromGrid (VDBMapping.hpp:413-447):
//                     one lane per point, voxel floor(p * 1/res), marked in an
//                     edit set (update-set layout: leaf key -> voxel mask)
//   k_mark_walls      addArtificialWall (VDBMapping.hpp:1217-1236): one lane per
//                     (polygon edge, height layer); rounded edge ends
//                     (VDBMapping.hpp:612-631) shifted by the layer, then the
//                     castRayIntoGrid walk (VDBMapping.hpp:550-566) marks the
//                     artificial set
//   k_set_voxels      one edit op on the marked voxels of listed edit-set leaves
//                     (set occupied / set free / restore state / activate)
//   k_section_pick    getMapSection (VDBMapping.hpp:922-1014): per map leaf, the
//                     section leaf it yields (full or sparse), appended to a list
//   k_upsert_leaves   find or create the map leaf of each section leaf
//   k_section_write   applyMapSectionGrid (VDBMapping.hpp:1022-1050) voxel writes
//   k_section_tiles   the section's internal-node tiles visited by the same loop
//   k_section_clear   applyMapSectionUpdateGrid (VDBMapping.hpp:1058-1085):
//                     deactivate map voxels inside the box, then OR the section
//
// Build with -ffp-contract=off like the other kernels.
#include <float.h>

#include "dda_math.h"
#include "device_common.h"
#include "kernels.h"
#include "upd_common.h"

namespace vdbgpu {

// One lane per point. A NaN or out-of-range voxel sets kErrRange (the host
// then discards the whole edit set); the others are marked visited.
__global__ __launch_bounds__(256) void k_mark_points(const float* __restrict__ pts, int64_t stride_f,
                                                     uint32_t n, double inv, UpdView u, Status* st) {
  const uint32_t G = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += G) {
    const float* p = pts + (int64_t)i * stride_f;
    int c[3];
    bool ok = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double f = floor((double)p[a] * inv);
      ok = ok && f >= -(double)kCoordLimit && f < (double)kCoordLimit;
      c[a] = ok ? (int)f : 0;
    }
    if (!ok) {
      atomicOr(&st->error, kErrRange);
      continue;
    }
    mark_voxel(u, &st->overflow, c[0], c[1], c[2], false);
  }
}

// One lane per (wall, layer): wall w = {a, b, k0, k1} joins vertices a and b
// of `verts` (x, y, z doubles); its layers k in [k0, k1) are lanes
// prefix[w] .. prefix[w + 1] - 1 and shift both rounded ends by (0, 0, k). A
// zero-length wall marks nothing (castRayIntoGrid's e == s guard); otherwise
// the walk visits 1 + |dx| + |dy| + |dz| voxels in exact DDA order (integer
// crossing comparisons, the crossing table for equal-time ties).
__global__ __launch_bounds__(64) void k_mark_walls(const double* __restrict__ verts,
                                                   const int4* __restrict__ walls,
                                                   const uint64_t* __restrict__ prefix, uint32_t n_walls,
                                                   double res, double inv, const double* __restrict__ tbl,
                                                   uint32_t tbl_n, UpdView u, Status* st) {
  const uint64_t total = prefix[n_walls];
  const uint64_t G = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += G) {
    uint32_t lo = 0, hi = n_walls - 1;  // last wall with prefix <= t
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (prefix[mid] <= t)
        lo = mid;
      else
        hi = mid - 1;
    }
    const int4 wr = walls[lo];
    const int k = wr.z + (int)(t - prefix[lo]);
    const double* a = verts + 3 * (int64_t)wr.x;
    const double* b = verts + 3 * (int64_t)wr.y;
    int s[3], e[3];
    bool ok = true;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      s[j] = world_to_index1(a[j], res, inv);
      e[j] = world_to_index1(b[j], res, inv);
    }
    const long long sz = (long long)s[2] + k, ez = (long long)e[2] + k;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      ok = ok && s[j] >= -kCoordLimit && s[j] < kCoordLimit && e[j] >= -kCoordLimit && e[j] < kCoordLimit;
    ok = ok && s[2] != INT_MIN && e[2] != INT_MIN && sz >= -kCoordLimit && sz < kCoordLimit &&
         ez >= -kCoordLimit && ez < kCoordLimit;
    if (!ok) {
      atomicOr(&st->error, kErrRange);
      continue;
    }
    s[2] = (int)sz;
    e[2] = (int)ez;
    if (s[0] == e[0] && s[1] == e[1] && s[2] == e[2]) continue;
    const uint32_t nn[3] = {(uint32_t)abs(e[0] - s[0]), (uint32_t)abs(e[1] - s[1]),
                            (uint32_t)abs(e[2] - s[2])};
    if (nn[0] > tbl_n || nn[1] > tbl_n || nn[2] > tbl_n) {
      atomicOr(&st->error, kErrTable);
      continue;
    }
    const int stx = e[0] > s[0] ? 1 : (e[0] < s[0] ? -1 : 0);
    const int sty = e[1] > s[1] ? 1 : (e[1] < s[1] ? -1 : 0);
    const int stz = e[2] > s[2] ? 1 : (e[2] < s[2] ? -1 : 0);
    const uint32_t cc[3] = {0, 0, 0};
    IntDda d;
    d.init(nn, cc);
    int vx = s[0], vy = s[1], vz = s[2];
    const uint32_t m = 1 + nn[0] + nn[1] + nn[2];
    for (uint32_t v = 0;;) {
      mark_voxel(u, &st->overflow, vx, vy, vz, false);
      if (++v == m) break;
      const int ax = d.next_axis(tbl);
      d.advance(ax);
      vx += ax == 0 ? stx : 0;
      vy += ax == 1 ? sty : 0;
      vz += ax == 2 ? stz : 0;
    }
  }
}

// One lane per (listed leaf, mask word): the op on every marked voxel of the
// word. kEditOccupied: (val, on) (setNodeToOccupied, OccupancyVDBMapping.hpp:124-129);
// kEditFree: (val, off) (setNodeToFree, :118-123); kEditState: on = value > t_max
// (setNodeState, :130-134); kEditActivate: on (setActiveState). Optionally
// clears the edit-set slots.
__global__ __launch_bounds__(256) void k_set_voxels(UpdView u, const uint32_t* __restrict__ list,
                                                    const uint32_t* __restrict__ eidx, uint32_t count,
                                                    MapView mp, int op, float val, float t_max,
                                                    uint32_t clear) {
  const uint64_t G = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (uint64_t)count * 8; t += G) {
    const uint32_t e = (uint32_t)(t >> 3);
    const int j = (int)(t & 7);
    const uint32_t slot = list[e];
    unsigned long long* w = &u.masks[(size_t)slot * 16];
    const uint64_t vis = w[j];
    if (clear) {
      if (vis) {
        w[j] = 0;
        w[8 + j] = 0;
      }
      if (j == 0) u.keys[slot] = kEmpty;
    }
    const uint32_t idx = eidx[e];
    if (vis == 0 || idx == kNone) continue;
    float* pv = mp.values + (size_t)idx * 512 + j * 64;
    unsigned long long* pa = mp.active + (size_t)idx * 8 + j;
    uint64_t aw = *pa;
    if (op == kEditOccupied || op == kEditFree) {
      for (uint64_t b = vis; b; b &= b - 1) pv[__builtin_ctzll(b)] = val;
      aw = op == kEditOccupied ? (aw | vis) : (aw & ~vis);
    } else if (op == kEditState) {
      for (uint64_t b = vis; b; b &= b - 1) {
        const int k = __builtin_ctzll(b);
        const uint64_t bit = 1ull << k;
        aw = pv[k] > t_max ? (aw | bit) : (aw & ~bit);
      }
    } else {
      aw |= vis;
    }
    *pa = aw;
    mp.dirty[idx] = 1;
  }
}

// Voxels of the leaf at origin o inside the inclusive box b, as 8 words (one
// per x slab, bit (y & 7) * 8 + (z & 7)).
__device__ __forceinline__ uint64_t box_word(const int o[3], const int* b, int j) {
  const int x = o[0] + j;
  if (x < b[0] || x > b[3]) return 0;
  uint64_t ym = 0, zm = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (o[1] + k >= b[1] && o[1] + k <= b[4]) ym |= 1ull << (8 * k);
    if (o[2] + k >= b[2] && o[2] + k <= b[5]) zm |= 1ull << k;
  }
  return ym * zm;  // product of the y-rows and z-columns selected
}

// One wave per map leaf: the section leaf it yields, if any. Full grid: the
// section's leaf appears at the first voxel inside the box that is on or has
// a value other than 0 (a setValueOff of 0 on the background tile changes
// nothing); from there every inside voxel keeps value and state, earlier ones
// stay (0, off). Sparse: inside active voxels become (1.0, on). The leaf's
// pool index is appended to `out` (order arbitrary; the host sorts).
__global__ __launch_bounds__(256) void k_section_pick(MapView mp, uint32_t leaf_count, const int* bbox,
                                                      int full, uint32_t* __restrict__ out,
                                                      unsigned int* counter, TileView tv) {
  const uint32_t waves = gridDim.x * (blockDim.x >> 6);
  const int lane = lane_id();
  __shared__ int sb[6];
  if (threadIdx.x < 6) sb[threadIdx.x] = bbox[threadIdx.x];
  __syncthreads();
  for (uint32_t L = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); L < leaf_count; L += waves) {
    if (tile_at(tv, L)) continue;  // the leaf iteration of getMapSection (VM:937) skips tiles
    int o[3];
    key_origin(mp.leaf_keys[L], o);
    if (o[0] + 7 < sb[0] || o[0] > sb[3] || o[1] + 7 < sb[1] || o[1] > sb[4] || o[2] + 7 < sb[2] ||
        o[2] > sb[5])
      continue;
    bool any = false;
    if (lane < 8) {
      const uint64_t in = box_word(o, sb, lane);
      const uint64_t act = mp.active[(size_t)L * 8 + lane];
      any = (in & act) != 0;
      if (full && !any && in) {
        const float* v = mp.values + (size_t)L * 512 + lane * 64;
        for (uint64_t b = in; b; b &= b - 1)
          if (v[__builtin_ctzll(b)] != 0.0f) {
            any = true;
            break;
          }
      }
    }
    if (__ballot(any) != 0 && lane == 0) out[atomicAdd(counter, 1u)] = L;
  }
}

// One wave per picked leaf: its section values and masks (see k_section_pick).
__global__ __launch_bounds__(256) void k_section_gather(MapView mp, const uint32_t* __restrict__ list,
                                                        uint32_t count, const int* bbox, int full,
                                                        unsigned long long* keys_out, float* vals_out,
                                                        unsigned long long* act_out) {
  const uint32_t waves = gridDim.x * (blockDim.x >> 6);
  const int lane = lane_id();
  for (uint32_t i = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); i < count; i += waves) {
    const uint32_t L = list[i];
    const uint64_t key = mp.leaf_keys[L];
    int o[3];
    key_origin(key, o);
    // first creating voxel (full grid): lowest offset inside the box that is on or non-zero
    int first = 512;
    uint64_t in = 0, act = 0;
    if (lane < 8) {
      in = box_word(o, bbox, lane);
      act = mp.active[(size_t)L * 8 + lane];
      act_out[(size_t)i * 8 + lane] = in & act;
      if (full) {
        uint64_t cre = in & act;
        const float* v = mp.values + (size_t)L * 512 + lane * 64;
        for (uint64_t b = in & ~act; b; b &= b - 1)
          if (v[__builtin_ctzll(b)] != 0.0f) cre |= b & (~b + 1);
        if (cre) first = lane * 64 + __builtin_ctzll(cre);
      }
    }
#pragma unroll
    for (int s = 1; s < 8; s <<= 1) first = min(first, __shfl_xor(first, s, 64));
    first = __shfl(first, 0, 64);  // lanes 0-7 hold the minimum; broadcast it
    if (lane == 0) keys_out[i] = key;
    for (int n = lane; n < 512; n += 64) {
      const uint64_t w = __shfl(in, n >> 6, 64), aw = __shfl(act, n >> 6, 64);
      const bool inside = (w >> (n & 63)) & 1, on = (aw >> (n & 63)) & 1;
      float x = 0.0f;
      if (full)
        x = inside && n >= first ? mp.values[(size_t)L * 512 + n] : 0.0f;
      else
        x = inside && on ? 1.0f : 0.0f;
      vals_out[(size_t)i * 512 + n] = x;
    }
  }
}

// Section of a box of moderate size, by its cells: a hash probe per cell
// instead of a pass over every leaf of the map (116 us for 2.7 M leaves; 2,048
// cells take 14-22), and the cell order is the order of sorted origins, so the
// host sorts nothing. One wave per cell; lane l holds the leaf's row x = l >> 3,
// y = l & 7 (eight voxels along z). See k_section_pick for what a section leaf
// is.

// Voxels of row (x, y) of the leaf at origin o inside the box, bit z.
__device__ __forceinline__ uint32_t box_row(const int o[3], const int* b, int x, int y) {
  if (o[0] + x < b[0] || o[0] + x > b[3] || o[1] + y < b[1] || o[1] + y > b[4]) return 0;
  const int z0 = max(b[2] - o[2], 0), z1 = min(b[5] - o[2], 7);
  return z0 > z1 ? 0u : (0xFFu >> (7 - z1)) & (0xFFu << z0);
}

__device__ __forceinline__ void cell_origin(const SectionBox& sb, uint32_t c, int o[3]) {
  const uint32_t z = c % sb.dims[2], q = c / sb.dims[2], y = q % sb.dims[1], x = q / sb.dims[1];
  o[0] = (sb.lo[0] + (int)x) * 8;
  o[1] = (sb.lo[1] + (int)y) * 8;
  o[2] = (sb.lo[2] + (int)z) * 8;
}

// The lane's eight voxels of leaf idx: inside the box, active, and (full
// sections) the values with the ones that are not 0.
struct SectionRow {
  uint32_t in, act, cre;
  float4 a, b;
  __device__ __forceinline__ void load(const MapView& mp, const SectionBox& sb, const int o[3], uint32_t idx,
                                       int lane, bool full) {
    in = box_row(o, sb.box, lane >> 3, lane & 7);
    act = (uint32_t)(mp.active[(size_t)idx * 8 + (lane >> 3)] >> ((lane & 7) * 8)) & 0xFFu;
    cre = in & act;
    if (!full) return;
    const float4* v = reinterpret_cast<const float4*>(mp.values) + (size_t)idx * 128 + 2 * lane;
    a = v[0];
    b = v[1];
    const uint32_t nz = (a.x != 0.0f ? 1u : 0u) | (a.y != 0.0f ? 2u : 0u) | (a.z != 0.0f ? 4u : 0u) |
                        (a.w != 0.0f ? 8u : 0u) | (b.x != 0.0f ? 16u : 0u) | (b.y != 0.0f ? 32u : 0u) |
                        (b.z != 0.0f ? 64u : 0u) | (b.w != 0.0f ? 128u : 0u);
    cre |= in & nz;
  }
};

__global__ __launch_bounds__(256) void k_section_cells(MapView mp, SectionBox sb, uint32_t cells, uint32_t full,
                                                       uint32_t* __restrict__ cell, uint64_t* __restrict__ bsum,
                                                       TileView tv) {
  __shared__ uint32_t s_n[4];
  const int lane = lane_id(), w = threadIdx.x >> 6;
  uint32_t n = 0;
#pragma unroll 1
  for (uint32_t q = 0; q < kSectionCells / 4; ++q) {
    const uint32_t c = blockIdx.x * kSectionCells + w * (kSectionCells / 4) + q;
    if (c >= cells) break;  // the whole wave
    int o[3];
    cell_origin(sb, c, o);
    const uint64_t key = leaf_key(o[0], o[1], o[2]);
    uint32_t idx = kNone, h = map_hash(key) & mp.cap_mask;
    for (uint32_t p = 0; p <= mp.cap_mask; ++p) {  // every lane probes alike
      const unsigned long long k = mp.keys[h];
      if (k == key) {
        idx = mp.idx[h];
        break;
      }
      if (k == kEmpty) break;
      h = (h + 1) & mp.cap_mask;
    }
    bool any = false;
    if (idx != kNone && !tile_at(tv, idx)) {  // the leaf iteration of getMapSection (VM:937) skips tiles
      SectionRow r;
      r.load(mp, sb, o, idx, lane, full != 0);
      any = r.cre != 0;
    }
    const bool picked = __ballot(any) != 0;
    if (lane == 0) cell[c] = picked ? idx : kNone;
    n += picked ? 1u : 0u;
  }
  if (lane == 0) s_n[w] = n;
  __syncthreads();
  if (threadIdx.x == 0) bsum[blockIdx.x] = s_n[0] + s_n[1] + s_n[2] + s_n[3];
}

// The picked cells' leaves at their ranks (host-visible memory mostly: each wave
// writes its leaf's 2 KiB as one run). Full: every inside voxel from the
// leaf's first creating one on keeps its value; sparse: active ones are 1.
__global__ __launch_bounds__(256) void k_section_rows(MapView mp, SectionBox sb, uint32_t cells, uint32_t full,
                                                      uint32_t values, const uint32_t* __restrict__ cell,
                                                      const uint64_t* __restrict__ boff, SectionDest dest) {
  const int lane = lane_id(), w = threadIdx.x >> 6;
  const uint32_t c0 = blockIdx.x * kSectionCells;
  const uint32_t mine = lane < (int)kSectionCells && c0 + lane < cells ? cell[c0 + lane] : kNone;
  const uint64_t picked = __ballot(mine != kNone);
#pragma unroll 1
  for (uint32_t q = 0; q < kSectionCells / 4; ++q) {
    const int k = w * (int)(kSectionCells / 4) + (int)q;
    if (!((picked >> k) & 1)) continue;  // the whole wave
    const uint64_t at = boff[blockIdx.x] + (uint64_t)__popcll(picked & ((1ull << k) - 1));
    if (at >= dest.cap) return;
    const bool pinned = at < dest.pinned;
    char* base = dest.rest;
    uint32_t leaves = dest.cap - dest.pinned, i = (uint32_t)at - dest.pinned;
    if (pinned) {
      base = dest.chunk[at / kSectionChunk];
      leaves = kSectionChunk;
      i = (uint32_t)at % kSectionChunk;
    }
    const uint32_t idx = __shfl(mine, k, 64);
    int o[3];
    cell_origin(sb, c0 + (uint32_t)k, o);
    SectionRow r;
    r.load(mp, sb, o, idx, lane, full != 0);
    int first = r.cre ? lane * 8 + __builtin_ctz(r.cre) : 512;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) first = min(first, __shfl_xor(first, s, 64));
    uint32_t keep = r.in;  // voxels that carry a value
    if (!full) {
      r.a = make_float4(1.f, 1.f, 1.f, 1.f);
      r.b = r.a;
      keep &= r.act;
    } else if (first > lane * 8) {
      keep &= first >= lane * 8 + 8 ? 0u : 0xFFu << (first - lane * 8);
    }
    if (!(keep & 1u)) r.a.x = 0.f;
    if (!(keep & 2u)) r.a.y = 0.f;
    if (!(keep & 4u)) r.a.z = 0.f;
    if (!(keep & 8u)) r.a.w = 0.f;
    if (!(keep & 16u)) r.b.x = 0.f;
    if (!(keep & 32u)) r.b.y = 0.f;
    if (!(keep & 64u)) r.b.z = 0.f;
    if (!(keep & 128u)) r.b.w = 0.f;
    if (values) {
      float4* out = reinterpret_cast<float4*>(base) + (size_t)i * 128 + 2 * lane;
      out[0] = r.a;
      out[1] = r.b;
    }
    uint64_t m = (uint64_t)(r.in & r.act) << ((lane & 7) * 8);
#pragma unroll
    for (int s = 1; s < 8; s <<= 1) m |= __shfl_xor(m, s, 64);
    char* heads = base + (size_t)leaves * 2048;
    if ((lane & 7) == 0) reinterpret_cast<unsigned long long*>(heads)[(size_t)i * 8 + (lane >> 3)] = m;
    if (lane < 3)
      reinterpret_cast<int*>(heads + (size_t)leaves * 64)[(size_t)i * 3 + lane] =
          lane == 0 ? o[0] : (lane == 1 ? o[1] : o[2]);
  }
}

// One lane per record: find the map leaf of keys[i], or create it when
// need[i] is set (leaf count in st->leaf_count; never past the pool, else
// st->map_full). Records that create nothing leave kNone in eidx. With
// `first`, a record whose leaf already existed gets first[i] = 0 (all of its
// voxels are written).
__global__ __launch_bounds__(256) void k_upsert_leaves(const unsigned long long* __restrict__ keys,
                                                       const uint8_t* __restrict__ need, uint32_t n,
                                                       MapView mp, uint32_t* __restrict__ eidx,
                                                       uint16_t* __restrict__ first, Status* st) {
  __shared__ uint32_t s_wave[4], s_base;
  const uint32_t G = gridDim.x * blockDim.x;
  const uint32_t rounds = (n + G - 1) / G;
  for (uint32_t rd = 0; rd < rounds; ++rd) {
    const uint32_t e = rd * G + blockIdx.x * blockDim.x + threadIdx.x;
    bool created = false;
    uint32_t h = kNone, idx = kNone;
    uint64_t key = 0;
    if (e < n) {
      key = keys[e];
      const bool nd = need[e] != 0;
      uint32_t p = map_hash(key) & mp.cap_mask;
      for (uint32_t probe = 0; probe <= mp.cap_mask; ++probe) {
        const unsigned long long k = mp.keys[p];
        if (k == key) {
          idx = mp.idx[p];
          break;
        }
        if (k == kEmpty) {
          if (!nd) break;
          const unsigned long long prev = atomicCAS(&mp.keys[p], kEmpty, (unsigned long long)key);
          if (prev == kEmpty) {
            created = true;
            h = p;
            break;
          }
        }
        p = (p + 1) & mp.cap_mask;
      }
    }
    const uint32_t pos = block_append(created, &st->leaf_count, s_wave, &s_base);
    if (created) {
      if (pos < mp.lcap) {
        idx = pos;
        mp.idx[h] = idx;
        mp.leaf_keys[idx] = key;
      } else {
        mp.idx[h] = kNone;
        atomicOr(&st->map_full, 1u);
      }
    }
    if (e < n) {
      eidx[e] = idx;
      if (idx != kNone) mp.dirty[idx] = 1;
      if (first && idx != kNone && !created) first[e] = 0;
    }
  }
}

// One wave per section leaf: write its voxels into the map leaf eidx[i].
// A leaf that existed before gets all 512 voxels; a created one (first[i] >
// 0) keeps the background for the voxels before its creating voxel.
__global__ __launch_bounds__(256) void k_section_write(const float* __restrict__ vals,
                                                       const unsigned long long* __restrict__ act,
                                                       const uint32_t* __restrict__ eidx,
                                                       const uint16_t* __restrict__ first, uint32_t n,
                                                       MapView mp) {
  const uint32_t waves = gridDim.x * (blockDim.x >> 6);
  const int lane = lane_id();
  for (uint32_t i = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); i < n; i += waves) {
    const uint32_t idx = eidx[i];
    if (idx == kNone) continue;
    const int f = first[i];
    for (int k = lane; k < 512; k += 64)
      if (k >= f) mp.values[(size_t)idx * 512 + k] = vals[(size_t)i * 512 + k];
    if (lane < 8) {
      const uint64_t keep = f >= (lane + 1) * 64 ? ~0ull : (f <= lane * 64 ? 0ull : ((1ull << (f - lane * 64)) - 1));
      unsigned long long* pa = mp.active + (size_t)idx * 8 + lane;
      *pa = (*pa & keep) | (act[(size_t)i * 8 + lane] & ~keep);
    }
  }
}

// The inactive tiles of the section's internal nodes, each visited at its
// origin: 4096 8^3 slots per 128^3 node (slots holding a section leaf are
// children, skipped), 32768 128^3 slots per 4096^3 node (slots holding a
// 128^3 node skipped). A visit sets the voxel at the slot origin of an
// existing map leaf to (0, off).
__global__ __launch_bounds__(256) void k_section_tiles(const unsigned long long* __restrict__ n128,
                                                       uint32_t c128, const unsigned long long* __restrict__ n4096,
                                                       uint32_t c4096, const unsigned long long* __restrict__ sleaf,
                                                       uint32_t sleaf_mask, const unsigned long long* __restrict__ s128,
                                                       uint32_t s128_mask, MapView mp) {
  const uint64_t total = (uint64_t)c128 * 4096 + (uint64_t)c4096 * 32768;
  const uint64_t G = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += G) {
    int o[3], x, y, z;
    if (t < (uint64_t)c128 * 4096) {
      key_origin(n128[t >> 12], o);  // origin / 128 * 8
      const int j = (int)(t & 4095);
      x = o[0] * 16 + 8 * (j >> 8);
      y = o[1] * 16 + 8 * ((j >> 4) & 15);
      z = o[2] * 16 + 8 * (j & 15);
      if (set_has(sleaf, sleaf_mask, leaf_key(x, y, z))) continue;
    } else {
      const uint64_t u = t - (uint64_t)c128 * 4096;
      key_origin(n4096[u >> 15], o);  // origin / 4096 * 8
      const int j = (int)(u & 32767);
      x = o[0] * 512 + 128 * (j >> 10);
      y = o[1] * 512 + 128 * ((j >> 5) & 31);
      z = o[2] * 512 + 128 * (j & 31);
      if (set_has(s128, s128_mask, node_key(x, y, z, 7))) continue;
    }
    const uint64_t key = leaf_key(x, y, z);
    uint32_t p = map_hash(key) & mp.cap_mask;
    for (uint32_t probe = 0; probe <= mp.cap_mask; ++probe) {
      const unsigned long long k = mp.keys[p];
      if (k == key) {
        const uint32_t idx = mp.idx[p];
        if (idx != kNone) {
          mp.values[(size_t)idx * 512] = 0.0f;  // voxel offset 0: the slot origin
          atomicAnd(&mp.active[(size_t)idx * 8], ~1ull);
          mp.dirty[idx] = 1;
        }
        break;
      }
      if (k == kEmpty) break;
      p = (p + 1) & mp.cap_mask;
    }
  }
}

// applyMapSectionUpdateGrid, first loop: every active map voxel inside the box
// set inactive. One lane per (leaf, word).
__global__ __launch_bounds__(256) void k_section_clear(MapView mp, uint32_t leaf_count, const int* bbox,
                                                       TileView tv) {
  const uint64_t G = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (uint64_t)leaf_count * 8; t += G) {
    const uint32_t L = (uint32_t)(t >> 3);
    const int j = (int)(t & 7);
    int o[3];
    key_origin(mp.leaf_keys[L], o);
    const uint64_t in = box_word(o, bbox, j);
    if (tile_at(tv, L)) {
      // cbeginValueOn (VM:1072) yields an active tile once, at its origin: only that
      // voxel is switched off, which turns the tile into a leaf
      if (j == 0 && (in & 1u) && tile_active(tv, L)) {
        mp.active[(size_t)L * 8] &= ~1ull;
        mp.dirty[L] = 1;
        atomicAnd(&tv.bits[L >> 5], ~(1u << (L & 31)));
      }
      continue;
    }
    if (!in) continue;
    unsigned long long* pa = mp.active + (size_t)L * 8 + j;
    const uint64_t aw = *pa;
    if (aw & in) {
      *pa = aw & ~in;
      mp.dirty[L] = 1;
    }
  }
}

// Second loop: OR the section's active masks into the map leaves eidx[i].
__global__ __launch_bounds__(256) void k_section_or(const unsigned long long* __restrict__ act,
                                                    const uint32_t* __restrict__ eidx, uint32_t n,
                                                    MapView mp) {
  const uint64_t G = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (uint64_t)n * 8; t += G) {
    const uint32_t i = (uint32_t)(t >> 3);
    const uint32_t idx = eidx[i];
    if (idx == kNone) continue;
    mp.active[(size_t)idx * 8 + (t & 7)] |= act[t];
  }
}

// One wave per section leaf (origins as x, y, z triples): its leaf key, and
// the offset of its creating voxel, the first voxel that is on or (with
// values) non-zero (512: none, applying it creates no missing leaf). With
// topology sets: inserts the leaf key, and the 128^3 and 4096^3 node keys,
// each new node key appended to its list (counters[0], counters[1]).
__global__ __launch_bounds__(256) void k_section_prep(const int* __restrict__ origins,
                                                      const float* __restrict__ vals,
                                                      const unsigned long long* __restrict__ act,
                                                      uint32_t n, unsigned long long* __restrict__ keys,
                                                      uint8_t* __restrict__ need, uint16_t* __restrict__ first,
                                                      unsigned long long* sleaf, uint32_t sleaf_mask,
                                                      unsigned long long* s128, uint32_t s128_mask,
                                                      unsigned long long* n128, unsigned long long* s4096,
                                                      uint32_t s4096_mask, unsigned long long* n4096,
                                                      unsigned int* counters) {
  const uint32_t waves = gridDim.x * (blockDim.x >> 6);
  const int lane = lane_id();
  for (uint32_t i = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); i < n; i += waves) {
    // lane owns voxels 8 lane .. 8 lane + 7
    uint32_t cre = (uint32_t)(act[(size_t)i * 8 + (lane >> 3)] >> ((lane & 7) * 8)) & 0xFFu;
    if (vals) {
      const float4* pv = reinterpret_cast<const float4*>(vals + (size_t)i * 512 + lane * 8);
      const float4 a = pv[0], b = pv[1];
      cre |= (a.x != 0.0f ? 1u : 0u) | (a.y != 0.0f ? 2u : 0u) | (a.z != 0.0f ? 4u : 0u) |
             (a.w != 0.0f ? 8u : 0u) | (b.x != 0.0f ? 16u : 0u) | (b.y != 0.0f ? 32u : 0u) |
             (b.z != 0.0f ? 64u : 0u) | (b.w != 0.0f ? 128u : 0u);
    }
    int f = cre ? lane * 8 + __builtin_ctz(cre) : 512;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) f = min(f, __shfl_xor(f, o, 64));
    if (lane == 0) {
      const int x = origins[3 * i], y = origins[3 * i + 1], z = origins[3 * i + 2];
      const uint64_t key = leaf_key(x, y, z);
      keys[i] = key;
      need[i] = f < 512 ? 1 : 0;
      first[i] = (uint16_t)f;
      if (sleaf) {
        set_insert(sleaf, sleaf_mask, key);
        const uint64_t k7 = node_key(x, y, z, 7), k12 = node_key(x, y, z, 12);
        if (set_insert(s128, s128_mask, k7)) n128[atomicAdd(&counters[0], 1u)] = k7;
        if (set_insert(s4096, s4096_mask, k12)) n4096[atomicAdd(&counters[1], 1u)] = k12;
      }
    }
  }
}

// evalActiveVoxelBoundingBox: min / max voxel coordinate of the active
// voxels, folded into box[0..2] (atomicMin) and box[3..5] (atomicMax). One
// lane per (leaf, word); one atomic per workgroup and side, and only when it
// still moves that side.
__global__ __launch_bounds__(256) void k_active_bbox(MapView mp, uint32_t leaf_count, int* box) {
  __shared__ int s_box[4][6];
  const uint64_t G = (uint64_t)gridDim.x * blockDim.x;
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (uint64_t)leaf_count * 8; t += G) {
    const uint32_t L = (uint32_t)(t >> 3);
    const int j = (int)(t & 7);
    const uint64_t a = mp.active[(size_t)L * 8 + j];
    if (!a) continue;
    int o[3];
    key_origin(mp.leaf_keys[L], o);
    uint32_t rows = 0, cols = 0;  // y rows and z columns present in the word
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if ((a >> (8 * k)) & 0xFFu) rows |= 1u << k;
      cols |= (uint32_t)(a >> (8 * k)) & 0xFFu;
    }
    lo[0] = min(lo[0], o[0] + j);
    hi[0] = max(hi[0], o[0] + j);
    lo[1] = min(lo[1], o[1] + __builtin_ctz(rows));
    hi[1] = max(hi[1], o[1] + 31 - __builtin_clz(rows));
    lo[2] = min(lo[2], o[2] + __builtin_ctz(cols));
    hi[2] = max(hi[2], o[2] + 31 - __builtin_clz(cols));
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      lo[a] = min(lo[a], __shfl_xor(lo[a], o, 64));
      hi[a] = max(hi[a], __shfl_xor(hi[a], o, 64));
    }
  }
  if (lane_id() == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      s_box[threadIdx.x >> 6][a] = lo[a];
      s_box[threadIdx.x >> 6][3 + a] = hi[a];
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int a = threadIdx.x;
    int v = s_box[0][a];
    for (int w = 1; w < 4; ++w) v = a < 3 ? min(v, s_box[w][a]) : max(v, s_box[w][a]);
    const int cur = __hip_atomic_load(&box[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (a < 3 ? v < cur : v > cur) {
      if (a < 3)
        atomicMin(&box[a], v);
      else
        atomicMax(&box[a], v);
    }
  }
}

// Active points of the map (saveMapToPCD, VM:218-256) in OpenVDB's
// cbeginValueOn order, on the device.
//
// Position of a leaf in that order: root children by origin, then 128^3 nodes
// and leaves by offset, all x-major; 12 + 5 + 4 bits per axis of its biased
// leaf coordinates, most significant level first.
__device__ __forceinline__ uint64_t tree_order(const int o[3]) {
  uint32_t u[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) u[a] = (uint32_t)((o[a] >> 3) + (1 << 20));
  uint64_t k = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) k = k << 12 | (u[a] >> 9);
#pragma unroll
  for (int a = 0; a < 3; ++a) k = k << 5 | ((u[a] >> 4) & 31u);
#pragma unroll
  for (int a = 0; a < 3; ++a) k = k << 4 | (u[a] & 15u);
  return k;
}

// Leaves with an active value, their order keys and counts; cbeginValueOn
// yields an active tile once, at its origin (an inactive one not at all).
__global__ __launch_bounds__(256) void k_point_leaves(MapView mp, const Status* __restrict__ stmap, TileView tv,
                                                      uint64_t* __restrict__ keys, uint32_t* __restrict__ cnt,
                                                      uint32_t* __restrict__ idx, Status* st) {
  __shared__ uint32_t s_wave[4], s_base;
  __shared__ unsigned long long s_sum[4];
  const uint32_t leaf_count = stmap->leaf_count;
  const uint32_t G = gridDim.x * blockDim.x;
  unsigned long long sum = 0;
  for (uint32_t base = blockIdx.x * blockDim.x; base < leaf_count; base += G) {
    const uint32_t i = base + threadIdx.x;
    uint32_t c = 0;
    if (i < leaf_count) {
      const unsigned long long* w = mp.active + (size_t)i * 8;
      if (tile_at(tv, i)) {
        c = (uint32_t)(w[0] & 1u);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) c += (uint32_t)__popcll(w[j]);
      }
    }
    const uint32_t pos = block_append(c != 0, &st->entries, s_wave, &s_base);
    if (c) {
      int o[3];
      key_origin(mp.leaf_keys[i], o);
      keys[pos] = tree_order(o);
      cnt[pos] = c;
      idx[pos] = i;
      sum += c;
    }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
  if (lane_id() == 0) s_sum[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    sum = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
    if (sum) atomicAdd(&st->total, sum);
  }
}

// First point of each listed leaf: the counts of the leaves before it, by
// comparing it with all of them (slice blockIdx.y of the list, 256 at a time
// in LDS). n^2 compares, but the list of a room of 200,000 points takes 17 us and
// needs no sort; the host takes over above kMaxPointLeaves.
__global__ __launch_bounds__(256) void k_point_offsets(const uint64_t* __restrict__ keys,
                                                       const uint32_t* __restrict__ cnt, uint32_t n,
                                                       unsigned long long* off) {
  __shared__ uint64_t s_key[256];
  __shared__ uint32_t s_cnt[256];
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  const uint64_t mine = i < n ? keys[i] : 0;
  unsigned long long sum = 0;
  for (uint32_t base = blockIdx.y * 256u; base < n; base += gridDim.y * 256u) {
    __syncthreads();
    const uint32_t j = base + threadIdx.x;
    s_key[threadIdx.x] = j < n ? keys[j] : ~0ull;  // after every key
    s_cnt[threadIdx.x] = j < n ? cnt[j] : 0u;
    __syncthreads();
    uint32_t part = 0;  // <= 256 * 512
#pragma unroll 8
    for (int k = 0; k < 256; ++k) part += s_key[k] < mine ? s_cnt[k] : 0u;
    sum += part;
  }
  if (i < n && sum) atomicAdd(&off[i], sum);
}

// One wave per listed leaf: the centres of its active voxels, in offset order.
__global__ __launch_bounds__(256) void k_point_rows(MapView mp, TileView tv, const uint32_t* __restrict__ idx,
                                                    const unsigned long long* __restrict__ off, uint32_t n, double res,
                                                    float* __restrict__ xyz) {
  const uint32_t waves = gridDim.x * (blockDim.x >> 6);
  const int lane = lane_id();
  for (uint32_t i = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); i < n; i += waves) {
    const uint32_t L = idx[i];
    uint32_t row = (uint32_t)(mp.active[(size_t)L * 8 + (lane >> 3)] >> ((lane & 7) * 8)) & 0xFFu;
    if (tile_at(tv, L)) row = lane == 0 ? row & 1u : 0u;
    uint32_t v = (uint32_t)__popc(row);
    const uint32_t c = v;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const uint32_t t = __shfl_up(v, s, 64);
      if (lane >= s) v += t;
    }
    int o[3];
    key_origin(mp.leaf_keys[L], o);
    float* p = xyz + 3 * (off[i] + v - c);
    for (uint32_t r = row; r; r &= r - 1) {
      const int q[3] = {o[0] + (lane >> 3), o[1] + (lane & 7), o[2] + __builtin_ctz(r)};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        double w = (double)q[a] * res;  // indexToWorld (ScaleMap::applyMap)
        w += 0.5 * res;
        *p++ = (float)w;
      }
    }
  }
}

// Keys of every leaf overlapping the box (leaf-grid origin lo, extents dims,
// x-major), each with the same creation flag.
__global__ __launch_bounds__(256) void k_box_keys(int lx, int ly, int lz, uint32_t dx, uint32_t dy, uint32_t dz,
                                                  unsigned long long* __restrict__ keys, uint8_t* __restrict__ need,
                                                  uint8_t need_v) {
  const uint64_t n = (uint64_t)dx * dy * dz;
  const uint64_t G = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += G) {
    const uint32_t z = (uint32_t)(i % dz), y = (uint32_t)((i / dz) % dy), x = (uint32_t)(i / ((uint64_t)dz * dy));
    keys[i] = leaf_key((lx + (int)x) * 8, (ly + (int)y) * 8, (lz + (int)z) * 8);
    need[i] = need_v;
  }
}

// The background of createMapFromPointCloud: inside the box, every inactive
// voxel of the leaves eidx[i] gets value v (its state stays off). One wave per
// leaf, eight voxels per lane as two float4 where all of them are written (the
// usual leaf): one lane per word, storing voxel by voxel, took 84 us for 32,000
// leaves, now 23.
__global__ __launch_bounds__(256) void k_box_fill(const unsigned long long* __restrict__ keys,
                                                  const uint32_t* __restrict__ eidx, uint32_t n, const int* box,
                                                  MapView mp, float v) {
  const uint32_t waves = gridDim.x * (blockDim.x >> 6);
  const int lane = lane_id();
  for (uint32_t i = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); i < n; i += waves) {
    const uint32_t idx = eidx[i];
    if (idx == kNone) continue;
    int o[3];
    key_origin(keys[i], o);
    const uint32_t act = (uint32_t)(mp.active[(size_t)idx * 8 + (lane >> 3)] >> ((lane & 7) * 8)) & 0xFFu;
    const uint32_t m = box_row(o, box, lane >> 3, lane & 7) & ~act;
    float* pv = mp.values + (size_t)idx * 512 + lane * 8;
    if (m == 0xFFu) {
      reinterpret_cast<float4*>(pv)[0] = make_float4(v, v, v, v);
      reinterpret_cast<float4*>(pv)[1] = make_float4(v, v, v, v);
    } else {
      for (uint32_t b = m; b; b &= b - 1) pv[__builtin_ctz(b)] = v;
    }
    if (__ballot(m != 0) != 0 && lane == 0) mp.dirty[idx] = 1;
  }
}

// ------------------------------------------------------------- launchers --

hipError_t launch_mark_points(hipStream_t s, const float* pts, int64_t stride_bytes, uint32_t n, double inv,
                              UpdView u, Status* st) {
  const int grid = (int)std::min<uint32_t>(4096, (n + 255) / 256);
  hipLaunchKernelGGL(k_mark_points, dim3(grid), dim3(256), 0, s, pts, stride_bytes / 4, n, inv, u, st);
  return hipGetLastError();
}

hipError_t launch_mark_walls(hipStream_t s, const double* verts, const int4* walls, const uint64_t* prefix,
                             uint32_t n_walls, uint64_t total, double res, double inv, const double* tbl,
                             uint32_t tbl_n, UpdView u, Status* st) {
  if (total == 0 || n_walls == 0) return hipSuccess;
  const int grid = (int)std::min<uint64_t>(16384, (total + 63) / 64);
  hipLaunchKernelGGL(k_mark_walls, dim3(grid), dim3(64), 0, s, verts, walls, prefix, n_walls, res, inv, tbl,
                     tbl_n, u, st);
  return hipGetLastError();
}

hipError_t launch_set_voxels(hipStream_t s, UpdView u, const uint32_t* list, const uint32_t* eidx,
                             uint32_t count, MapView mp, int op, float val, float t_max, bool clear) {
  const int grid = (int)std::min<uint64_t>(8192, ((uint64_t)count * 8 + 255) / 256);
  hipLaunchKernelGGL(k_set_voxels, dim3(grid), dim3(256), 0, s, u, list, eidx, count, mp, op, val, t_max,
                     clear ? 1u : 0u);
  return hipGetLastError();
}

hipError_t launch_section_pick(hipStream_t s, MapView mp, uint32_t leaf_count, const int* bbox, bool full,
                               uint32_t* out, unsigned int* counter, TileView tv) {
  const int grid = (int)std::min<uint32_t>(8192, (leaf_count + 3) / 4);
  hipLaunchKernelGGL(k_section_pick, dim3(grid), dim3(256), 0, s, mp, leaf_count, bbox, full ? 1 : 0, out,
                     counter, tv);
  return hipGetLastError();
}

hipError_t launch_section_gather(hipStream_t s, MapView mp, const uint32_t* list, uint32_t count,
                                 const int* bbox, bool full, unsigned long long* keys_out, float* vals_out,
                                 unsigned long long* act_out) {
  const int grid = (int)std::min<uint32_t>(8192, (count + 3) / 4);
  hipLaunchKernelGGL(k_section_gather, dim3(grid), dim3(256), 0, s, mp, list, count, bbox, full ? 1 : 0,
                     keys_out, vals_out, act_out);
  return hipGetLastError();
}

hipError_t launch_section_cells(hipStream_t s, MapView mp, const SectionBox& sb, uint32_t cells, bool full,
                                uint32_t* cell, uint64_t* bsum, uint64_t* boff, unsigned int* total, TileView tv) {
  const uint32_t nb = (cells + kSectionCells - 1) / kSectionCells;
  hipLaunchKernelGGL(k_section_cells, dim3(nb), dim3(256), 0, s, mp, sb, cells, full ? 1u : 0u, cell, bsum, tv);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_scan_u64(s, bsum, boff, nb, total);
}

hipError_t launch_section_rows(hipStream_t s, MapView mp, const SectionBox& sb, uint32_t cells, bool full, bool values,
                               const uint32_t* cell, const uint64_t* boff, const SectionDest& dest) {
  const uint32_t nb = (cells + kSectionCells - 1) / kSectionCells;
  hipLaunchKernelGGL(k_section_rows, dim3(nb), dim3(256), 0, s, mp, sb, cells, full ? 1u : 0u, values ? 1u : 0u, cell,
                     boff, dest);
  return hipGetLastError();
}

hipError_t launch_upsert_leaves(hipStream_t s, const unsigned long long* keys, const uint8_t* need, uint32_t n,
                                MapView mp, uint32_t* eidx, uint16_t* first, Status* st) {
  const int grid = (int)std::min<uint32_t>(4096, (n + 255) / 256);
  hipLaunchKernelGGL(k_upsert_leaves, dim3(grid), dim3(256), 0, s, keys, need, n, mp, eidx, first, st);
  return hipGetLastError();
}

hipError_t launch_section_write(hipStream_t s, const float* vals, const unsigned long long* act,
                                const uint32_t* eidx, const uint16_t* first, uint32_t n, MapView mp) {
  const int grid = (int)std::min<uint32_t>(8192, (n + 3) / 4);
  hipLaunchKernelGGL(k_section_write, dim3(grid), dim3(256), 0, s, vals, act, eidx, first, n, mp);
  return hipGetLastError();
}

hipError_t launch_section_tiles(hipStream_t s, const unsigned long long* n128, uint32_t c128,
                                const unsigned long long* n4096, uint32_t c4096,
                                const unsigned long long* sleaf, uint32_t sleaf_mask,
                                const unsigned long long* s128, uint32_t s128_mask, MapView mp) {
  const uint64_t total = (uint64_t)c128 * 4096 + (uint64_t)c4096 * 32768;
  if (total == 0) return hipSuccess;
  const int grid = (int)std::min<uint64_t>(8192, (total + 255) / 256);
  hipLaunchKernelGGL(k_section_tiles, dim3(grid), dim3(256), 0, s, n128, c128, n4096, c4096, sleaf, sleaf_mask,
                     s128, s128_mask, mp);
  return hipGetLastError();
}

hipError_t launch_section_clear(hipStream_t s, MapView mp, uint32_t leaf_count, const int* bbox, TileView tv) {
  if (leaf_count == 0) return hipSuccess;
  const int grid = (int)std::min<uint64_t>(8192, ((uint64_t)leaf_count * 8 + 255) / 256);
  hipLaunchKernelGGL(k_section_clear, dim3(grid), dim3(256), 0, s, mp, leaf_count, bbox, tv);
  return hipGetLastError();
}

hipError_t launch_section_or(hipStream_t s, const unsigned long long* act, const uint32_t* eidx, uint32_t n,
                             MapView mp) {
  if (n == 0) return hipSuccess;
  const int grid = (int)std::min<uint64_t>(8192, ((uint64_t)n * 8 + 255) / 256);
  hipLaunchKernelGGL(k_section_or, dim3(grid), dim3(256), 0, s, act, eidx, n, mp);
  return hipGetLastError();
}

hipError_t launch_section_prep(hipStream_t s, const int* origins, const float* vals, const unsigned long long* act,
                               uint32_t n, unsigned long long* keys, uint8_t* need, uint16_t* first,
                               unsigned long long* sleaf, uint32_t sleaf_mask, unsigned long long* s128,
                               uint32_t s128_mask, unsigned long long* n128, unsigned long long* s4096,
                               uint32_t s4096_mask, unsigned long long* n4096, unsigned int* counters) {
  if (n == 0) return hipSuccess;
  const int grid = (int)std::min<uint32_t>(8192, (n + 3) / 4);
  hipLaunchKernelGGL(k_section_prep, dim3(grid), dim3(256), 0, s, origins, vals, act, n, keys, need, first,
                     sleaf, sleaf_mask, s128, s128_mask, n128, s4096, s4096_mask, n4096, counters);
  return hipGetLastError();
}

hipError_t launch_active_bbox(hipStream_t s, MapView mp, uint32_t leaf_count, int* box) {
  if (leaf_count == 0) return hipSuccess;
  const int grid = (int)std::min<uint64_t>(1024, ((uint64_t)leaf_count * 8 + 255) / 256);
  hipLaunchKernelGGL(k_active_bbox, dim3(grid), dim3(256), 0, s, mp, leaf_count, box);
  return hipGetLastError();
}

hipError_t launch_box_keys(hipStream_t s, const int lo[3], const uint32_t dims[3], unsigned long long* keys,
                           uint8_t* need, bool need_v) {
  const uint64_t n = (uint64_t)dims[0] * dims[1] * dims[2];
  if (n == 0) return hipSuccess;
  const int grid = (int)std::min<uint64_t>(8192, (n + 255) / 256);
  hipLaunchKernelGGL(k_box_keys, dim3(grid), dim3(256), 0, s, lo[0], lo[1], lo[2], dims[0], dims[1], dims[2], keys,
                     need, (uint8_t)(need_v ? 1 : 0));
  return hipGetLastError();
}

hipError_t launch_box_fill(hipStream_t s, const unsigned long long* keys, const uint32_t* eidx, uint32_t n,
                           const int* box, MapView mp, float v) {
  if (n == 0) return hipSuccess;
  const int grid = (int)std::min<uint32_t>(8192, (n + 3) / 4);
  hipLaunchKernelGGL(k_box_fill, dim3(grid), dim3(256), 0, s, keys, eidx, n, box, mp, v);
  return hipGetLastError();
}

hipError_t launch_point_leaves(hipStream_t s, MapView mp, uint64_t leaf_bound, const Status* stmap, TileView tv,
                               uint64_t* keys, uint32_t* cnt, uint32_t* idx, Status* st) {
  const int grid = (int)std::min<uint64_t>(2048, (leaf_bound + 255) / 256 + 1);
  hipLaunchKernelGGL(k_point_leaves, dim3(grid), dim3(256), 0, s, mp, stmap, tv, keys, cnt, idx, st);
  return hipGetLastError();
}

hipError_t launch_points(hipStream_t s, MapView mp, TileView tv, const uint64_t* keys, const uint32_t* cnt,
                         const uint32_t* idx, uint32_t n, unsigned long long* off, double res, float* xyz) {
  if (n == 0) return hipSuccess;
  const uint32_t nb = (n + 255) / 256;
  hipError_t e = launch_fill_u64(s, off, n, 0);
  if (e != hipSuccess) return e;
  // slices: about four workgroups per CU
  const uint32_t slices = std::max(1u, std::min(nb, 1024u / nb));
  hipLaunchKernelGGL(k_point_offsets, dim3(nb, slices), dim3(256), 0, s, keys, cnt, n, off);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_point_rows, dim3(std::min(8192u, (n + 3) / 4)), dim3(256), 0, s, mp, tv, idx, off, n, res, xyz);
  return hipGetLastError();
}

}  // namespace vdbgpu
