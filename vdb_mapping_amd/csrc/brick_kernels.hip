// gfx950 kernels of the brick path of one scan (the raycast of
// insertPointCloud, VDBMapping.hpp:466-566). Space is cut into bricks of
// 32^3 voxels (4^3 leaves). Each ray is cut into per-brick segments in
// closed form (dda_math.h), the segments are bucketed by brick, and one
// workgroup owns a brick's visited/hit bitmap (8 KiB of LDS) while it walks
// that brick's segments. The result is the scan's update set as a list of
// leaf records (key + 8 visited + 8 hit mask words), every update leaf
// exactly once, written with plain stores into the scan's record set (a brick
// takes its run of records with one atomic on one of 16 counters), which the
// map stream reads, possibly several scans later. (Records at 64 fixed
// positions per work item, listed and copied densely afterwards, needed no
// counters but four launches and a copy: 105 us of an outdoor scan's cast.)
// No global atomics touch voxel bits except for the few
// bricks so crowded (more segments than a work item takes, around the sensor)
// that several workgroups share them.
//
//   k_seg_count     one lane per ray: enumerate its bricks, count segments
//                   per brick (aggregated per workgroup in an LDS table,
//                   which is stored for the fill)
//   k_brick_offsets segment offset and work items of each brick
//   k_seg_fill      reserve the run of each entry of the workgroup's stored
//                   table, enumerate again, write each segment record at its
//                   brick's next position
//   k_brick_walk    one workgroup per work item: walk the item's segments
//                   into the LDS bitmap, append the brick's leaf records to
//                   the scan's record set (named in device memory), or OR
//                   into the shared bitmap of a split brick
//   k_split_emit    leaf records of split bricks
//   k_rec_total     ray, visit and record counts of the scan, overflow
//
// Segment record (uint4), self-contained so the walk loads nothing else:
//   x = n0 | n1 << 14, y = n2 | c0 << 14, z = c1 | c2 << 14  (|delta| per axis
//       and the crossing counts at the segment's first visit, <= 8192 each)
//   w = brick-local first voxel lx | ly << 5 | lz << 10 | visits m << 16 |
//       negative-step bits x, y, z << 24 | end-voxel hit flag << 31
// The walk of a segment starts at that voxel with the integer DDA state of
// those counts and visits m (<= 94) voxels, all inside the brick (checked).
#include <cstddef>

#include "dda_math.h"
#include "device_common.h"
#include "kernels.h"

namespace vdbgpu {

namespace {

constexpr int kLdsBricks = kSegTab;  // per-workgroup brick aggregation table
constexpr int kLdsBrickProbe = 32;
constexpr uint32_t kMaxBrickProbe = 512;
constexpr int kBrickWords = 1024;  // 64 leaves x (8 visited + 8 hit) words
// The walk's LDS bitmap: one 32-bit word per (x, y) row of the brick, bit z,
// rows of a plane 33 words apart so that the rows of a column do not share a
// bank. Merged into leaf-major visited words before the records are written.
constexpr int kWalkPlane = 33;
constexpr int kWalkWords = 32 * kWalkPlane;

__device__ __forceinline__ int bw_lane() { return (int)__lane_id(); }

struct RayGeom {
  int s[3], e[3];
  uint32_t cnt;
  bool hit;
};

// Geometry of ray i, false if it marks nothing (NaN, zero range, rejected).
__device__ __forceinline__ bool ray_geom(const int4* __restrict__ rayinfo,
                                         const ScanInfo* __restrict__ scans, uint32_t i,
                                         RayGeom& g) {
  const int4 r = rayinfo[i];
  const uint32_t w = (uint32_t)r.w;
  g.cnt = w & kCntMask;
  g.hit = (w & kHitBit) != 0;
  if (g.cnt == 0 && !g.hit) return false;
  const uint32_t sc = (w >> kScanShift) & kScanMask;
  g.s[0] = scans[sc].s[0];
  g.s[1] = scans[sc].s[1];
  g.s[2] = scans[sc].s[2];
  g.e[0] = r.x;
  g.e[1] = r.y;
  g.e[2] = r.z;
  return true;
}

__device__ __forceinline__ int lds_brick(unsigned long long* lkey, uint64_t key, bool insert) {
  uint32_t h = (uint32_t)(fmix64(key) >> 40) & (kLdsBricks - 1);
  for (int p = 0; p < kLdsBrickProbe; ++p) {
    const unsigned long long k =
        __hip_atomic_load(&lkey[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (k == key) return (int)h;
    if (k == kEmpty) {
      if (!insert) return -1;
      const unsigned long long prev = atomicCAS(&lkey[h], kEmpty, (unsigned long long)key);
      if (prev == kEmpty || prev == key) return (int)h;
    }
    h = (h + 1) & (kLdsBricks - 1);
  }
  return -1;
}

// Slot of a brick in the scan's brick table (inserted if `insert`), kNone if
// absent or after kMaxBrickProbe probes (then the table is flagged full).
__device__ __forceinline__ uint32_t brick_slot(const BrickView& bv, uint64_t key, bool insert,
                                               unsigned int* ovf) {
  if (bv.cells) {
    int b[3];
    brick_coords(key, b);
    const uint32_t D = 2u * (uint32_t)bv.half + 1;
    const uint32_t x = (uint32_t)(b[0] - (bv.scan->s[0] >> kBrickLog) + bv.half),
                   y = (uint32_t)(b[1] - (bv.scan->s[1] >> kBrickLog) + bv.half),
                   z = (uint32_t)(b[2] - (bv.scan->s[2] >> kBrickLog) + bv.half);
    // every ray ends within the range the cube was sized for; a brick outside
    // would be an error, and is treated like a full table
    if (x < D && y < D && z < D) return (x * D + y) * D + z;
    atomicOr(ovf, kOvfBricks);
    return kNone;
  }
  uint32_t h = (uint32_t)fmix64(key) & bv.cap_mask;
  const uint32_t limit = bv.cap_mask < kMaxBrickProbe ? bv.cap_mask + 1 : kMaxBrickProbe;
  for (uint32_t p = 0; p < limit; ++p) {
    const unsigned long long k =
        __hip_atomic_load(&bv.keys[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (k == key) return h;
    if (k == kEmpty) {
      if (!insert) return kNone;
      const unsigned long long prev = atomicCAS(&bv.keys[h], kEmpty, (unsigned long long)key);
      if (prev == kEmpty || prev == key) return h;
    }
    h = (h + 1) & bv.cap_mask;
  }
  if (insert) atomicOr(ovf, kOvfBricks);
  return kNone;
}

// Coordinates of the brick in a slot.
__device__ __forceinline__ void brick_of(const BrickView& bv, uint32_t slot, int b[3]) {
  if (bv.cells) {
    const uint32_t D = 2u * (uint32_t)bv.half + 1;
    const uint32_t z = slot % D, q = slot / D, y = q % D, x = q / D;
    b[0] = (int)x - bv.half + (bv.scan->s[0] >> kBrickLog);
    b[1] = (int)y - bv.half + (bv.scan->s[1] >> kBrickLog);
    b[2] = (int)z - bv.half + (bv.scan->s[2] >> kBrickLog);
  } else {
    brick_coords(bv.keys[slot], b);
  }
}

// Workgroup-uniform stop flag: error or any overflow already raised.
__device__ __forceinline__ bool stopped(const Status* st, unsigned int* s_stop) {
  if (threadIdx.x == 0)
    *s_stop = __hip_atomic_load(&st->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) |
              __hip_atomic_load(&st->overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  return *s_stop != 0;
}

// Regions in use for a scan of n_items work items: enough counters that the
// appends of tens of thousands of bricks do not queue on one (a single one made
// the walk 0.75 -> 1.27 ms), one for small scans, whose few bricks would fill
// many regions unevenly.
__device__ __forceinline__ uint32_t rec_regions(uint32_t n_items) {
  return n_items >= kRecRegionItems ? kRecRegions : 1u;
}

// Leaf records of the brick bitmap `bits` (brick origin o), appended to region
// `reg` of the record set: one atomic per brick on the region's counter, every
// leaf with a visited voxel a record (key, 8 visited and 8 hit words) after the
// next. A brick that does not fit is counted but not written (k_rec_total
// flags it). Called by the whole workgroup.
__device__ void emit_leaves(const unsigned long long* bits, int ox, int oy, int oz, const RecDest& d, uint32_t reg,
                            uint32_t stride, unsigned int* rcnt, uint32_t* s_pos) {
  const int tid = threadIdx.x;
  if (tid < 64) {  // lane l = leaf l of the brick
    uint64_t any = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) any |= bits[tid * 8 + j];
    const uint64_t m = __ballot(any != 0);
    const uint32_t n = (uint32_t)__popcll(m);
    uint32_t base = 0;
    if (tid == 0 && n) base = atomicAdd(&rcnt[reg * kRecCountStride], n);
    base = __shfl(base, 0, 64);
    const bool ok = any != 0 && base + n <= stride;
    const uint32_t pos = reg * stride + base + (uint32_t)__popcll(m & ((1ull << tid) - 1));
    s_pos[tid] = ok ? pos : kNone;
    if (ok) d.keys[pos] = leaf_key(ox + (tid >> 4) * 8, oy + ((tid >> 2) & 3) * 8, oz + (tid & 3) * 8);
  }
  __syncthreads();
  // 16 records x 16 words per pass: contiguous 128-byte rows
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int l = p * 16 + (tid >> 4), w = tid & 15;
    const uint32_t pos = s_pos[l];
    if (pos != kNone) d.masks[(size_t)pos * 16 + w] = bits[(w < 8 ? 0 : 512) + l * 8 + (w & 7)];
  }
}

// The ray of this lane in the cut: every 2^spread-th lane has one (cut_spread).
__device__ __forceinline__ uint32_t cut_ray(int spread) {
  return (threadIdx.x & ((1u << spread) - 1)) ? kNone : (blockIdx.x * blockDim.x + threadIdx.x) >> spread;
}

}  // namespace

__global__ __launch_bounds__(256) void k_seg_count(const int4* __restrict__ rayinfo,
                                                   const ScanInfo* __restrict__ scans,
                                                   const BatchCtl* __restrict__ ctl,
                                                   const double* __restrict__ tbl, BrickView bv,
                                                   unsigned long long* __restrict__ wkey,
                                                   unsigned long long* __restrict__ wsc, Status* st, int spread) {
  __shared__ unsigned long long lkey[kLdsBricks];
  __shared__ uint32_t lcnt[kLdsBricks];
  __shared__ unsigned int s_stop;
  if (stopped(st, &s_stop)) return;
  for (int e = threadIdx.x; e < kLdsBricks; e += blockDim.x) {
    lkey[e] = kEmpty;
    lcnt[e] = 0;
  }
  __syncthreads();
  const uint32_t i = cut_ray(spread);
  RayGeom g;
  if (i < ctl->n_rays && ray_geom(rayinfo, scans, i, g)) {
    SegEnum en;
    en.init(tbl, g.s, g.e, g.cnt);
    Segment sg;
    while (en.next(tbl, sg)) {
      const uint64_t key = brick_key(sg.bx, sg.by, sg.bz);
      const int ls = lds_brick(lkey, key, true);
      if (ls >= 0) {
        atomicAdd(&lcnt[ls], 1u);
      } else {
        const uint32_t gs = brick_slot(bv, key, true, &st->overflow);
        if (gs != kNone) atomicAdd(&bv.cnt[gs], 1u);
      }
    }
  }
  __syncthreads();
  // the table, as it stands, for the fill: a segment is counted here iff its
  // brick is in the table (a key once in the table stays; one that found its
  // probe run full never gets in), so the fill's lookups in the same table
  // split the workgroup's segments exactly as the counts did
  const size_t tb = (size_t)blockIdx.x * kLdsBricks;
  for (int e = threadIdx.x; e < kLdsBricks; e += blockDim.x) {
    const uint64_t key = lkey[e];
    wkey[tb + e] = key;
    if (key == kEmpty) continue;
    const uint32_t gs = brick_slot(bv, key, true, &st->overflow);
    if (gs != kNone) atomicAdd(&bv.cnt[gs], lcnt[e]);
    wsc[tb + e] = ((uint64_t)gs << 32) | lcnt[e];
  }
}

// Exclusive scan of nb sums (one workgroup); their total to *total.
__global__ __launch_bounds__(256) void k_scan_u64(const uint64_t* __restrict__ bsum,
                                                  uint64_t* __restrict__ boff, uint32_t nb,
                                                  unsigned int* total) {
  __shared__ uint64_t wsum[4];
  uint64_t carry = 0;
  for (uint32_t base = 0; base < nb; base += 256) {
    const uint32_t i = base + threadIdx.x;
    const uint64_t x = i < nb ? bsum[i] : 0ull;
    uint64_t v = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint64_t t = __shfl_up(v, o, 64);
      if (bw_lane() >= o) v += t;
    }
    const int wv = threadIdx.x >> 6;
    if (bw_lane() == 63) wsum[wv] = v;
    __syncthreads();
    uint64_t add = 0, tot = 0;
    for (int w = 0; w < 4; ++w) {
      if (w < wv) add += wsum[w];
      tot += wsum[w];
    }
    if (i < nb) boff[i] = carry + add + v - x;
    carry += tot;
    __syncthreads();
  }
  if (threadIdx.x == 0) *total = (unsigned int)carry;
}

// Segment offset and work items of each brick, kOffsetSlots slots a workgroup
// (four to a lane). A workgroup takes its run of segments and of items with one
// atomic on the pair of totals; which run a brick gets does not matter, so no
// scan over the workgroups is needed (it took two more launches, 9 us of a
// 2,000-point scan's 160 us of GPU time). A range of 1,000 voxels has 269
// workgroups, and only those with a segment touch the counter.
__global__ __launch_bounds__(256) void k_brick_offsets(BrickView bv, BrickItem* __restrict__ items,
                                                       uint32_t seg_cap, uint32_t item_cap,
                                                       uint32_t* __restrict__ split_slot,
                                                       uint32_t split_cap, uint32_t item_segs, Status* st) {
  static_assert(offsetof(Status, segs) % 8 == 0 && offsetof(Status, items) == offsetof(Status, segs) + 4,
                "segs and items are one 64-bit counter");
  __shared__ uint64_t s_w[4];
  __shared__ uint64_t s_base;
  const uint32_t slot0 = blockIdx.x * kOffsetSlots + threadIdx.x * 4;
  const uint4 q = *reinterpret_cast<const uint4*>(bv.cnt + slot0);
  const uint32_t c[4] = {q.x, q.y, q.z, q.w};
  uint64_t x = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) x += ((uint64_t)((c[k] + item_segs - 1) / item_segs) << 32) | c[k];
  uint64_t v = x;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t t = __shfl_up(v, o, 64);
    if (bw_lane() >= o) v += t;
  }
  const int wv = threadIdx.x >> 6;
  if (bw_lane() == 63) s_w[wv] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint64_t sum = s_w[0] + s_w[1] + s_w[2] + s_w[3];
    s_base = sum ? atomicAdd(reinterpret_cast<unsigned long long*>(&st->segs), (unsigned long long)sum) : 0ull;
  }
  __syncthreads();
  uint64_t off = s_base + v - x;
  for (int w = 0; w < wv; ++w) off += s_w[w];
  uint32_t seg0 = (uint32_t)off, item0 = (uint32_t)(off >> 32);
  const uint32_t s1 = seg0 + c[0], s2 = s1 + c[1];
  *reinterpret_cast<uint4*>(bv.cur + slot0) = make_uint4(seg0, s1, s2, s2 + c[2]);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t slot = slot0 + k, n = c[k], ni = (n + item_segs - 1) / item_segs;
    if (ni == 0) continue;
    if ((uint64_t)seg0 + n > seg_cap) {
      atomicOr(&st->overflow, kOvfSegs);
    } else if ((uint64_t)item0 + ni > item_cap) {
      atomicOr(&st->overflow, kOvfItems);
    } else {
      const uint32_t shared = ni > 1 ? atomicAdd(&st->splits, 1u) : kNone;
      if (ni > 1 && shared >= split_cap) {
        atomicOr(&st->overflow, kOvfSplit);
      } else {
        if (ni > 1) split_slot[shared] = slot;
        for (uint32_t j = 0; j < ni; ++j) {
          const uint32_t a = seg0 + j * item_segs;
          items[item0 + j] = BrickItem{slot, a, min(a + item_segs, seg0 + n), shared};
        }
      }
    }
    seg0 += n;
    item0 += ni;
  }
}

__global__ __launch_bounds__(256) void k_seg_fill(const int4* __restrict__ rayinfo,
                                                  const ScanInfo* __restrict__ scans,
                                                  const BatchCtl* __restrict__ ctl,
                                                  const double* __restrict__ tbl, BrickView bv,
                                                  const unsigned long long* __restrict__ wkey,
                                                  const unsigned long long* __restrict__ wsc,
                                                  uint4* __restrict__ segs, uint32_t seg_cap,
                                                  Status* st, int spread) {
  __shared__ unsigned long long lkey[kLdsBricks];
  __shared__ uint32_t lcnt[kLdsBricks];
  __shared__ uint32_t lbase[kLdsBricks];
  __shared__ unsigned int s_stop;
  // stops when the count stopped: a count workgroup that stored no table saw
  // the flags this one sees (nothing clears them between the two launches)
  if (stopped(st, &s_stop)) return;
  // 1: the count's table of this workgroup (the same rays), one reservation
  // per (workgroup, brick)
  const size_t tb = (size_t)blockIdx.x * kLdsBricks;
  for (int e = threadIdx.x; e < kLdsBricks; e += blockDim.x) {
    const uint64_t key = wkey[tb + e];
    lkey[e] = key;
    lcnt[e] = 0;
    if (key == kEmpty) continue;
    const uint64_t sc = wsc[tb + e];
    const uint32_t gs = (uint32_t)(sc >> 32);
    if (gs == kNone) {
      atomicOr(&st->error, kErrBrick);
      lbase[e] = seg_cap;
    } else {
      lbase[e] = atomicAdd(&bv.cur[gs], (uint32_t)sc);
    }
  }
  __syncthreads();
  const uint32_t i = cut_ray(spread);
  RayGeom g;
  const bool valid = i < ctl->n_rays && ray_geom(rayinfo, scans, i, g);
  // 2: write the records
  if (valid) {
    SegEnum en;
    en.init(tbl, g.s, g.e, g.cnt);
    Segment sg;
    while (en.next(tbl, sg)) {
      const uint64_t key = brick_key(sg.bx, sg.by, sg.bz);
      const int ls = lds_brick(lkey, key, false);
      uint32_t pos;
      if (ls >= 0) {
        pos = lbase[ls] + atomicAdd(&lcnt[ls], 1u);
      } else {
        const uint32_t gs = brick_slot(bv, key, false, &st->overflow);
        pos = gs == kNone ? seg_cap : atomicAdd(&bv.cur[gs], 1u);
      }
      if (pos >= seg_cap) {
        atomicOr(&st->overflow, kOvfSegs);
        continue;
      }
      uint32_t n[3], neg = 0, loc = 0;
      bool inside = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const int d = g.e[a] - g.s[a];
        n[a] = (uint32_t)abs(d);
        neg |= (d < 0 ? 1u : 0u) << a;
        const int b = a == 0 ? sg.bx : (a == 1 ? sg.by : sg.bz);
        const int l = g.s[a] + (d < 0 ? -(int)sg.c[a] : (int)sg.c[a]) - b * kBrickDim;
        inside = inside && (unsigned)l < (unsigned)kBrickDim;
        loc |= (uint32_t)(l & (kBrickDim - 1)) << (5 * a);
      }
      if (!inside) atomicOr(&st->error, kErrBrick);  // the cut and its brick disagree
      segs[pos] = make_uint4(n[0] | n[1] << 14, n[2] | sg.c[0] << 14, sg.c[1] | sg.c[2] << 14,
                             loc | sg.m << 16 | neg << 24 | ((sg.last && g.hit) ? 0x80000000u : 0u));
    }
  }
}

// Walk one segment record into the brick's rows `vis` (and its end voxel into
// the leaf-major hit words).
//
// The walk state is one code u = (x * 33 + y) * 32 + z of the brick-local
// voxel, stepped by one add per visit: u >> 5 is the row's word, the low five
// bits of u its bit, so a visit is an OR of 1 << z into LDS. The loop is bound
// by VALU issue, and this is the least of it found: gathering the bits of a
// 64-bit word in registers and OR-ing it when the walk left it (in three
// layouts, each segment in the one whose words it left least) saved LDS
// operations but cost the loop some fifteen more instructions (a 262,144-ray
// outdoor scan alone: 496 us, now 400).
// The word index is clamped to the bitmap. The path is monotone along every
// axis, so it stayed inside the brick exactly when the end lies where m - 1
// steps of the right signs lead (a field that left [0, 31] has carried into
// the next: its apparent step then has the wrong sign or the steps the wrong
// sum).
//
// The step order is the exact integer DDA of dda_math.h (signs of the three
// pairwise differences); the rational-tie rule runs only when a lane of the
// wave meets a tie, with the crossing counts recovered from the walk state.
__device__ __forceinline__ void walk_voxel(uint32_t u, uint32_t& x, uint32_t& y, uint32_t& z) {
  const uint32_t w = u >> 5;
  x = (w * 1986u) >> 16;  // w / 33 for w < 1056
  y = w - x * 33u;
  z = u & 31u;
}

__device__ __forceinline__ void walk_segment(const uint4 sr, const double* __restrict__ tbl, uint32_t* vis,
                                             unsigned long long* hit, Status* st) {
  const uint32_t n0 = sr.x & 0x3FFFu, n1 = (sr.x >> 14) & 0x3FFFu, n2 = sr.y & 0x3FFFu;
  const uint32_t c00 = (sr.y >> 14) & 0x3FFFu, c10 = sr.z & 0x3FFFu, c20 = (sr.z >> 14) & 0x3FFFu;
  const uint32_t lx0 = sr.w & 31u, ly0 = (sr.w >> 5) & 31u, lz0 = (sr.w >> 10) & 31u;
  const uint32_t m = (sr.w >> 16) & 0x7Fu;
  const int sgx = n0 == 0 ? 0 : (((sr.w >> 24) & 1u) ? -1 : 1);
  const int sgy = n1 == 0 ? 0 : (((sr.w >> 25) & 1u) ? -1 : 1);
  const int sgz = n2 == 0 ? 0 : (((sr.w >> 26) & 1u) ? -1 : 1);
  uint32_t u = (lx0 * kWalkPlane + ly0) * 32u + lz0;
  const int ix = sgx * kWalkPlane * 32, iy = sgy * 32, iz = sgz;
  const int tn0 = 2 * (int)n0, tn1 = 2 * (int)n1, tn2 = 2 * (int)n2;
  int dyx = (int)((2 * c10 + 1) * n0) - (int)((2 * c00 + 1) * n1);
  int dzx = (int)((2 * c20 + 1) * n0) - (int)((2 * c00 + 1) * n2);
  int dzy = (int)((2 * c20 + 1) * n1) - (int)((2 * c10 + 1) * n2);
  for (uint32_t k = 0;;) {
    atomicOr(&vis[min(u >> 5, (uint32_t)kWalkWords - 1)], 1u << (u & 31u));
    if (++k >= m) break;  // m == 0: the endpoint of a zero-length ray
    bool y = dyx < 0;
    const int dzm = y ? dzy : dzx;
    bool z = dzm < 0;
    if (__any(dyx == 0 || dzm == 0)) {
      // exact rule for every lane: crossing counts from the walk state
      uint32_t lx, ly, lz;
      walk_voxel(u, lx, ly, lz);
      IntDda t;
      t.n0 = n0, t.n1 = n1, t.n2 = n2;
      t.c0 = c00 + (uint32_t)abs((int)lx - (int)lx0);
      t.c1 = c10 + (uint32_t)abs((int)ly - (int)ly0);
      t.c2 = c20 + (uint32_t)abs((int)lz - (int)lz0);
      t.dyx = dyx, t.dzx = dzx, t.dzy = dzy;
      const int ax = t.next_axis(tbl);
      z = ax == 2;
      y = ax == 1;
    }
    y = y && !z;
    const bool x = !z && !y;
    dyx += z ? 0 : (y ? tn0 : -tn1);
    dzx += y ? 0 : (z ? tn0 : -tn2);
    dzy += x ? 0 : (z ? tn1 : -tn2);
    u += (uint32_t)(z ? iz : (y ? iy : ix));
  }
  uint32_t lx, ly, lz;
  walk_voxel(u, lx, ly, lz);
  const int ex = ((int)lx - (int)lx0) * sgx, ey = ((int)ly - (int)ly0) * sgy, ez = ((int)lz - (int)lz0) * sgz;
  if (u >> 5 >= (uint32_t)kWalkWords || ly > 31u || ex < 0 || ey < 0 || ez < 0 || ex + ey + ez != (int)max(m, 1u) - 1) {
    atomicOr(&st->error, kErrBrick);  // the scan is rejected
  } else if (sr.w & 0x80000000u) {
    // setValueOn(end, true) (VDBMapping.hpp:533-536): the last visit is the end voxel
    const uint32_t hw = ((lx >> 3) << 7) | ((ly >> 3) << 5) | ((lz >> 3) << 3) | (lx & 7u);
    atomicOr(&hit[hw], 1ull << (((ly & 7u) << 3) | (lz & 7u)));
  }
}

// The brick's rows as leaf-major visited words (word j of leaf l at l * 8 + j,
// bit (y & 7) * 8 + (z & 7)). Called by the whole workgroup: a thread reads the
// eight rows of one leaf plane and writes the words of two of the four leaves
// along z; ends with a barrier.
__device__ void merge_rows(const uint32_t* vis, unsigned long long* bits) {
  const int t = (int)(threadIdx.x & 127u), half = (int)(threadIdx.x >> 7);
  const int lx = t >> 5, j = (t >> 2) & 7, ly = t & 3;
  const uint32_t* row = vis + (lx * 8 + j) * kWalkPlane + ly * 8;
  uint64_t out0 = 0, out1 = 0;
#pragma unroll
  for (int yy = 0; yy < 8; ++yy) {
    const uint32_t w = row[yy] >> (16 * half);
    out0 |= (uint64_t)(w & 0xFFu) << (8 * yy);
    out1 |= (uint64_t)((w >> 8) & 0xFFu) << (8 * yy);
  }
  unsigned long long* dst = bits + ((lx * 4 + ly) * 4 + 2 * half) * 8 + j;
  dst[0] = out0;
  dst[8] = out1;
  __syncthreads();
}

constexpr int kWalkThreads = 256;
constexpr int kSegsPerThread = kItemSegs / kWalkThreads;  // an item's segments, per thread
static_assert(kSegsPerThread <= 4, "segment lengths are packed one byte per segment");

__global__ __launch_bounds__(kWalkThreads, 8) void k_brick_walk(const BrickItem* __restrict__ items,
                                                             const uint4* __restrict__ segs,
                                                             const int4* __restrict__ rayinfo,
                                                             const ScanInfo* __restrict__ scans,
                                                             const double* __restrict__ tbl, BrickView bv,
                                                             unsigned long long* __restrict__ shared_bits,
                                                             const RecDest* __restrict__ dest,
                                                             unsigned int* __restrict__ rcnt, Status* st) {
  __shared__ unsigned long long bits[kBrickWords];
  __shared__ uint32_t vis[kWalkWords];
  __shared__ uint32_t s_pos[64];
  __shared__ uint32_t s_hist[128];
  __shared__ uint16_t s_order[kItemSegs];
  __shared__ unsigned int s_stop;
  if (stopped(st, &s_stop)) return;
  const uint32_t n_items = st->items;
  const RecDest d = *dest;
  const uint32_t regions = rec_regions(n_items), stride = d.cap / regions;
  const uint32_t t = threadIdx.x;
  // static assignment: item it -> workgroup it % grid (no shared queue counter)
  for (uint32_t it = blockIdx.x; it < n_items; it += gridDim.x) {
    const BrickItem item = items[it];
    int b[3];
    brick_of(bv, item.slot, b);
    const int ox = b[0] * kBrickDim, oy = b[1] * kBrickDim, oz = b[2] * kBrickDim;
    for (int w = t; w < kWalkWords; w += kWalkThreads) vis[w] = 0;
    for (int w = t; w < 512; w += kWalkThreads) bits[512 + w] = 0;  // hits; the visited words are merged in
    if (t < 128) s_hist[t] = 0;
    // Counting sort of the item's segments by visit count, longest first, so
    // the lanes of a wave walk segments of about the same length. Segment k
    // belongs to thread k % 256; its length is loaded once, for both passes.
    const uint32_t nseg = item.seg1 - item.seg0;  // <= kItemSegs
    uint32_t lens = 0;  // 7-bit lengths of the thread's segments, one byte each
#pragma unroll
    for (int r = 0; r < kSegsPerThread; ++r) {
      const uint32_t k = t + r * kWalkThreads;
      if (k < nseg) lens |= ((segs[item.seg0 + k].w >> 16) & 0x7Fu) << (8 * r);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSegsPerThread; ++r)
      if (t + r * kWalkThreads < nseg) atomicAdd(&s_hist[127 - ((lens >> (8 * r)) & 0xFFu)], 1u);
    __syncthreads();
    if (t < 64) {  // exclusive scan of the 128 bins, two per lane
      const uint32_t h0 = s_hist[2 * t], h1 = s_hist[2 * t + 1];
      uint32_t v = h0 + h1;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(v, o, 64);
        if ((int)t >= o) v += u;
      }
      const uint32_t ex = v - h0 - h1;
      s_hist[2 * t] = ex;
      s_hist[2 * t + 1] = ex + h0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSegsPerThread; ++r) {
      const uint32_t k = t + r * kWalkThreads;
      if (k < nseg) s_order[atomicAdd(&s_hist[127 - ((lens >> (8 * r)) & 0xFFu)], 1u)] = (uint16_t)k;
    }
    __syncthreads();
    // Round r of the walk covers the sorted segments [256 r, 256 r + 256); wave
    // w takes the 64 of block (w + r) mod 4, so over the rounds every wave
    // walks long and short ones alike. The next round's record is loaded
    // before the current one is walked.
    const uint32_t lane = t & 63u, wave = t >> 6;
    uint32_t k = (((wave + 0) & 3u) << 6) + lane;
    uint4 sr = k < nseg ? segs[item.seg0 + s_order[k]] : make_uint4(0, 0, 0, 0);
#pragma unroll 1
    for (uint32_t r = 0; k < nseg;) {
      ++r;
      const uint32_t kn = r * kWalkThreads + (((wave + r) & 3u) << 6) + lane;
      const uint4 sn = kn < nseg ? segs[item.seg0 + s_order[kn]] : make_uint4(0, 0, 0, 0);
      walk_segment(sr, tbl, vis, bits + 512, st);
      k = kn;
      sr = sn;
    }
    __syncthreads();
    merge_rows(vis, bits);
    if (item.shared == kNone) {
      emit_leaves(bits, ox, oy, oz, d, it & (regions - 1), stride, rcnt, s_pos);
    } else {
      unsigned long long* dst = shared_bits + (size_t)item.shared * kBrickWords;
      for (int w = t; w < kBrickWords; w += kWalkThreads) {
        const uint64_t v = bits[w];
        if (v) atomicOr(&dst[w], (unsigned long long)v);
      }
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) void k_split_emit(const uint32_t* __restrict__ split_slot,
                                                    unsigned long long* __restrict__ shared_bits,
                                                    BrickView bv, const RecDest* __restrict__ dest,
                                                    unsigned int* __restrict__ rcnt, Status* st) {
  __shared__ unsigned long long bits[kBrickWords];
  __shared__ uint32_t s_pos[64];
  __shared__ unsigned int s_stop;
  if (stopped(st, &s_stop)) return;
  const uint32_t ns = st->splits;
  const RecDest d = *dest;
  const uint32_t regions = rec_regions(st->items), stride = d.cap / regions;
  for (uint32_t k = blockIdx.x; k < ns; k += gridDim.x) {
    unsigned long long* src = shared_bits + (size_t)k * kBrickWords;
    for (int w = threadIdx.x; w < kBrickWords; w += blockDim.x) {
      bits[w] = src[w];
      src[w] = 0;
    }
    __syncthreads();
    int b[3];
    brick_of(bv, split_slot[k], b);
    emit_leaves(bits, b[0] * kBrickDim, b[1] * kBrickDim, b[2] * kBrickDim, d, k & (regions - 1), stride, rcnt,
                s_pos);
    __syncthreads();
  }
}

// The scan's counts (one workgroup): its valid rays and visits from the sums of
// k_prep's workgroups, its records with their prefix over the regions, and the
// overflow flag when a region did not hold its records.
__global__ __launch_bounds__(256) void k_rec_total(const uint32_t* __restrict__ bsum, const BatchCtl* __restrict__ ctl,
                                                   const RecDest* dest, const unsigned int* rcnt, Status* st) {
  __shared__ unsigned long long s_v[4];
  __shared__ unsigned int s_r[4];
  const uint32_t l = threadIdx.x;
  unsigned long long visits = 0;
  uint32_t rays = 0;
  for (uint32_t i = l; i < ctl->nb; i += 256) {
    visits += bsum[i] & kPrepVisitMask;
    rays += bsum[i] >> kPrepValidShift;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    visits += __shfl_xor(visits, o, 64);
    rays += __shfl_xor(rays, o, 64);
  }
  if (bw_lane() == 0) {
    s_v[l >> 6] = visits;
    s_r[l >> 6] = rays;
  }
  __syncthreads();
  if (l >= 64) return;
  if (l == 0) {
    st->total = s_v[0] + s_v[1] + s_v[2] + s_v[3];
    st->rays = (unsigned long long)s_r[0] + s_r[1] + s_r[2] + s_r[3];
  }
  if (st->error | st->overflow) return;
  const uint32_t stride = dest->cap / rec_regions(st->items);
  const uint32_t c = l < kRecRegions ? rcnt[l * kRecCountStride] : 0u;
  uint32_t v = c, most = c;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(v, o, 64);
    if ((int)l >= o) v += t;
    most = max(most, __shfl_xor(most, o, 64));
  }
  if (l < kRecRegions) st->rec_pre[l] = v - c;
  if (l == 63) {
    st->records = v;
    st->rec_stride = stride;
    st->rec_most = most;
    if (most > stride) atomicOr(&st->overflow, kOvfRecords);
  }
}

// The map's leaf count into host-visible memory (one lane; no copy engine).
__global__ void k_snap_count(const Status* st, uint32_t* host_dst) {
  if (threadIdx.x == 0) __hip_atomic_store(host_dst, st->leaf_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------- launchers --

hipError_t launch_rec_total(hipStream_t s, const uint32_t* bsum, const BatchCtl* ctl, const RecDest* dest,
                            const unsigned int* rcnt, Status* st) {
  hipLaunchKernelGGL(k_rec_total, dim3(1), dim3(256), 0, s, bsum, ctl, dest, rcnt, st);
  return hipGetLastError();
}

hipError_t launch_snap_count(hipStream_t s, const Status* st, uint32_t* host_dst) {
  hipLaunchKernelGGL(k_snap_count, dim3(1), dim3(64), 0, s, st, host_dst);
  return hipGetLastError();
}

hipError_t launch_seg_count(hipStream_t s, int grid, const int4* rayinfo, const ScanInfo* scans,
                            const BatchCtl* ctl, const double* tbl, BrickView bv, unsigned long long* wkey,
                            unsigned long long* wsc, Status* st, int spread) {
  hipLaunchKernelGGL(k_seg_count, dim3(grid), dim3(256), 0, s, rayinfo, scans, ctl, tbl, bv, wkey, wsc, st, spread);
  return hipGetLastError();
}

hipError_t launch_brick_offsets(hipStream_t s, BrickView bv, BrickItem* items, uint32_t seg_cap, uint32_t item_cap,
                                uint32_t* split_slot, uint32_t split_cap, uint32_t item_segs, Status* st) {
  hipLaunchKernelGGL(k_brick_offsets, dim3(bv.slots() / kOffsetSlots), dim3(256), 0, s, bv, items, seg_cap, item_cap,
                     split_slot, split_cap, item_segs, st);
  return hipGetLastError();
}

hipError_t launch_seg_fill(hipStream_t s, int grid, const int4* rayinfo, const ScanInfo* scans,
                           const BatchCtl* ctl, const double* tbl, BrickView bv,
                           const unsigned long long* wkey, const unsigned long long* wsc, uint4* segs,
                           uint32_t seg_cap, Status* st, int spread) {
  hipLaunchKernelGGL(k_seg_fill, dim3(grid), dim3(256), 0, s, rayinfo, scans, ctl, tbl, bv, wkey, wsc, segs,
                     seg_cap, st, spread);
  return hipGetLastError();
}

hipError_t launch_brick_walk(hipStream_t s, int grid, const BrickItem* items, const uint4* segs,
                             const int4* rayinfo, const ScanInfo* scans, const double* tbl,
                             BrickView bv, unsigned long long* shared_bits, const RecDest* dest,
                             unsigned int* rcnt, Status* st) {
  hipLaunchKernelGGL(k_brick_walk, dim3(grid), dim3(kWalkThreads), 0, s, items, segs, rayinfo, scans, tbl, bv,
                     shared_bits, dest, rcnt, st);
  return hipGetLastError();
}

hipError_t launch_scan_u64(hipStream_t s, const uint64_t* in, uint64_t* out, uint32_t n, unsigned int* total) {
  hipLaunchKernelGGL(k_scan_u64, dim3(1), dim3(256), 0, s, in, out, n, total);
  return hipGetLastError();
}

hipError_t launch_split_emit(hipStream_t s, int grid, const uint32_t* split_slot,
                             unsigned long long* shared_bits, BrickView bv, const RecDest* dest,
                             unsigned int* rcnt, Status* st) {
  hipLaunchKernelGGL(k_split_emit, dim3(grid), dim3(256), 0, s, split_slot, shared_bits, bv, dest, rcnt, st);
  return hipGetLastError();
}

}  // namespace vdbgpu
