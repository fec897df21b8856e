// Shared device/host definitions of the gfx950 occupancy-integration kernels.
//
// Data layout in HBM (one map handle):
//   map leaf hash   : keys u64[mcap] (open addressing, linear probing, EMPTY = ~0),
//                     idx u32[mcap] (leaf pool index of the key)
//   leaf pool       : values f32[lcap][512] (OpenVDB LeafNode<float,3> buffer
//                     order, offset ((x&7)<<6)|((y&7)<<3)|(z&7)),
//                     active u64[lcap][8] (value mask), leaf_keys u64[lcap], dirty u8[lcap]
//   update set (per source): keys u64[ucap], masks u64[ucap][16] (visited words 0..7,
//                     hit words 8..15, same bit layout as the value mask)
//   per scan        : rayinfo int4[n] (end voxel xyz, visit count | hit flag),
//                     pre u32[n] (inclusive visit-count prefix inside each 256-ray block),
//                     bsum u32[nb], boff u64[nb] (exclusive block offsets)
//   crossing table  : tbl f64, row n (n = 1..tbl_n) at n(n-1)/2 holding the
//                     DDA crossing times of an axis with |delta| = n
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vdbgpu {

constexpr uint64_t kEmpty = ~0ull;
constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr int kCoordLimit = 1 << 23;  // voxel coords in [-2^23, 2^23): 21-bit leaf coords
constexpr uint32_t kHitBit = 0x80000000u;   // rayinfo.w: endpoint is a hit
constexpr uint32_t kValidBit = 0x40000000u; // rayinfo.w: the ray is cast (not NaN, range > 0)
constexpr uint32_t kCntMask = 0xFFFFu;      // rayinfo.w bits 0-15: visit count (<= 1 + 3 * 8192)
constexpr int kScanShift = 16;              // rayinfo.w bits 16-22: scan index in a batch
constexpr uint32_t kScanMask = 0x7Fu;
constexpr int kMaxBatchScans = 128;
constexpr int kBatchCoordLimit = 1 << 21;   // batched keys: 19-bit leaf coords + 7-bit scan
constexpr int kPrepBlock = 256;
// sums of a prep workgroup: visits in the low bits (256 * (1 + 3 * 8192) < 2^23), valid rays (<= 256) above
constexpr int kPrepValidShift = 23;
constexpr uint32_t kPrepVisitMask = (1u << kPrepValidShift) - 1;
constexpr int kMaxQuerySteps = 1 << 24;  // per-axis voxel extent bound of a raytrace query

// Status bits written by kernels.
constexpr uint32_t kErrRange = 1u;  // a voxel index out of range / non-finite
constexpr uint32_t kErrTable = 2u;  // crossing table or chunk table too short
constexpr uint32_t kErrEntry = 4u;  // mid-ray DDA entry did not converge
constexpr uint32_t kErrBrick = 8u;  // brick path inconsistency (a segment left its brick)
constexpr uint32_t kErrWalk = 16u;  // fast-mode walk exceeded its step bound
constexpr uint32_t kOvfHard = 1u;   // update-set probe found no free slot
constexpr uint32_t kMapFull = 1u;   // Status::map_full: the fold needs a larger leaf pool / hash
// Brick path overflow bits (Status::overflow): a table too small for this
// scan; the host grows it and re-runs the brick stages.
constexpr uint32_t kOvfBricks = 2u;   // brick hash
constexpr uint32_t kOvfSegs = 4u;     // segment array
constexpr uint32_t kOvfItems = 8u;    // work items
constexpr uint32_t kOvfSplit = 16u;   // shared-brick bitmaps
constexpr uint32_t kOvfRecords = 32u; // update-leaf records
constexpr uint32_t kOvfSpans = 64u;   // fast-mode span lists
// Segments per brick work item, at most and for small scans: a small scan has
// too few bricks to fill the chip, and its crowded ones (all rays start in one)
// are the walk's critical path, so they are cut finer (the walk of a room scan of
// 32,768 rays 69 -> 36 us, of 65,536 outdoor rays 255 -> 238 us). Larger scans
// keep 1,024: with 256 there are more split bricks to merge (a lone outdoor scan of
// 131,072 rays over 500 voxels 443 -> 475 us, of 262,144 542 -> 625; a room scan of
// 100,000 rays over 150 voxels 200 -> 209, of 262,144 300 -> 339; at 80,000 rays
// both are within 2%).
constexpr uint32_t kItemSegs = 1024;
constexpr uint32_t kSmallItemSegs = 256;
constexpr uint32_t kSmallScanRays = 65536;

// Direct edit ops on the marked voxels of an edit set (k_set_voxels).
constexpr int kEditOccupied = 0;  // setNodeToOccupied: (max log-odds, on)
constexpr int kEditFree = 1;      // setNodeToFree: (min log-odds, off)
constexpr int kEditState = 2;     // setNodeState: on = value > t_max
constexpr int kEditActivate = 3;  // setActiveState(on)

// A scan's update-leaf records lie in up to kRecRegions equal regions of its
// record set, each filled from its start (see emit_leaves).
constexpr uint32_t kRecRegions = 16;
// Work items from which all regions are used: where many workgroups append at once one
// counter holds them up (a lone outdoor scan of 4,000 rays over 1,000 voxels 545 us with
// 16 regions, 670 with one; of 16,384 rays 870 and 1,010; of 262,144 rays 1,700 and 1,745).
// Scans of fewer items differ by 7% at most either way, and equal regions fill unevenly, so
// that their set has to be larger.
constexpr uint32_t kRecRegionItems = 4096;
constexpr uint32_t kRecCountStride = 32;    // words between the regions' counters (a line each)

struct Status {
  unsigned long long total;     // visits of the scan (sum of counts)
  unsigned long long voxels;    // visited voxels in the update set (compact)
  unsigned long long rays;      // valid rays of the scan
  unsigned int error;
  unsigned int overflow;
  unsigned int entries;         // update-set leaves (compact)
  unsigned int leaf_count;      // map leaves (map insert)
  unsigned int groups;          // leaves of a batch (fold groups)
  unsigned int map_full;
  unsigned int segs;            // brick segments of the scan (brick path)
  unsigned int items;           // brick work items
  unsigned int splits;          // bricks shared by several work items
  unsigned int records;         // update-leaf records of the scan (brick path)
  unsigned int rec_stride;      // records per region of its record set
  unsigned int rec_most;        // records of the fullest region
  unsigned int rec_pre[kRecRegions];  // records of the regions before each
  unsigned int pad;
};

// Record e of a scan (in region order) lies at at(e) of its record set.
struct RecIndex {
  uint32_t pre[kRecRegions];
  uint32_t stride;
  __host__ __device__ __forceinline__ uint32_t at(uint32_t e) const {
    uint32_t d = 0;
#if defined(__HIPCC__)
#pragma unroll
#endif
    for (uint32_t r = 1; r < kRecRegions; ++r) d = e >= pre[r] ? r * stride - pre[r] : d;
    return e + d;
  }
};

// One scan of a batch: sensor origin, max range, its rays [ray0, ray0 + nrays)
// of the concatenated cloud; s = rounded origin voxel (written by k_prep).
struct ScanInfo {
  double o[3];
  double R;
  uint32_t ray0, nrays;
  int s[3];
  int pad;
};

// Sizes read by the kernels (device memory, so a captured graph can be replayed).
struct BatchCtl {
  uint32_t n_rays;
  uint32_t nb;       // 256-ray blocks
  uint32_t n_scans;
  uint32_t batched;  // 1: update-set keys are (leaf, scan)
};

struct UpdView {
  unsigned long long* keys;
  unsigned long long* masks;  // 16 words per slot
  uint32_t cap_mask;
};

// Where the brick path puts a scan's records (one record set of the ring):
// kept in device memory, so a replayed cast graph fills the set of the scan it
// runs for.
struct RecDest {
  unsigned long long* keys;
  unsigned long long* masks;  // 16 words per record
  uint32_t cap;
  uint32_t pad;
};

// Batch fold groups: leaf (57-bit batched key) -> 128-bit scan mask + create flag.
struct GroupView {
  unsigned long long* keys;
  unsigned long long* scans;  // 2 words per slot
  unsigned int* need;
  uint32_t cap_mask;
};

// Bricks (32^3 voxels) of one scan: slot -> segment count and fill cursor. A
// slot is a cell of the cube of 2 half + 1 bricks around the sensor's brick
// where that has at most kDenseBricks cells (ranges up to 1,597 voxels), x-major:
// no key to compare or insert, a count is one atomic without a result, and the
// bricks are listed in space order. Farther rays hash the brick's key.
constexpr uint32_t kDenseBricks = 1u << 20;
constexpr uint32_t kOffsetSlots = 1024;  // slots per workgroup of k_brick_offsets; slots() is a multiple of it
struct BrickView {
  unsigned long long* keys;  // hash: kEmpty = free
  uint32_t* cnt;             // segments in the brick
  uint32_t* cur;             // next free segment position (fill stage)
  uint32_t cap_mask;         // hash slots - 1
  uint32_t cells;            // dense slots, a multiple of kOffsetSlots (0: hash)
  int half;                  // bricks to each side
  const ScanInfo* scan;      // the scan (its origin voxel)
  __host__ __device__ __forceinline__ uint32_t slots() const { return cells ? cells : cap_mask + 1; }
};
// One work item of the brick walk: segments [seg0, seg1) of brick `slot`;
// `shared` indexes the global bitmap the items of a split brick OR into
// (kNone: the item owns the brick).
struct BrickItem {
  uint32_t slot, seg0, seg1, shared;
};
struct MapView {
  unsigned long long* keys;
  uint32_t* idx;
  uint32_t cap_mask;
  float* values;
  unsigned long long* active;
  unsigned long long* leaf_keys;
  uint8_t* dirty;
  uint32_t lcap;  // leaf pool capacity
};

// Leaf-level tiles of pruneGrid (createMapFromPointCloud): leaf i of the pool
// stands for a tile of value val[i] when bit i of `bits` is set, active when
// bit i of `on` is set. bits == nullptr: the map holds no tile.
struct TileView {
  uint32_t* bits;
  uint32_t* on;
  float* val;
  uint32_t cap;  // leaves the arrays cover; a later leaf is never a tile
};

__host__ __device__ inline bool tile_at(const TileView& t, uint32_t i) {
  return t.bits && i < t.cap && ((t.bits[i >> 5] >> (i & 31)) & 1u);
}
__host__ __device__ inline bool tile_active(const TileView& t, uint32_t i) {
  return (t.on[i >> 5] >> (i & 31)) & 1u;
}

// Topology snapshot used by raytrace and the fast-mode raycast: a hash of the
// 128^3 nodes (key -> node index), one bit per leaf of every node, a hash set
// of the 4096^3 node keys, and the padded bbox of leaves with an active voxel.
// A node's 4,096 leaf bits are 64 words of 4 x 4 x 4 leaves, so a ray reads a
// word once for the two or three leaves it crosses in it; beside each word the
// one of the leaves that held an active voxel when the snapshot was taken.
struct RtView {
  unsigned long long* n128;
  uint32_t* nidx;             // node index of each slot of n128
  unsigned long long* bits;   // per node 64 x (leaves, leaves with an active voxel)
  unsigned long long* n4096;
  uint32_t n128_mask, n4096_mask;
  uint32_t live;              // 1: the map changed since, active states are read from it alone
  int bmin[3], bmax[3];
};
// A map section by the leaf cells of its index box (edit_kernels.hip): cell
// (x, y, z) of dims is the leaf at (lo + (x, y, z)) * 8, numbered x-major, the
// order of sorted origins; box is the inclusive voxel box.
struct SectionBox {
  int lo[3];
  uint32_t dims[3];
  int box[6];
};
constexpr uint32_t kSectionCells = 16;  // cells per workgroup
// Where the leaves of a section go, in cell order: the first `pinned` of them
// into host-visible chunks of kSectionChunk leaves, the others up to `cap` into
// `rest`. A chunk of k leaves holds their values, then their masks, then their
// origins (2,048, 64 and 12 bytes each); so does rest, for cap - pinned leaves.
constexpr uint32_t kSectionChunk = 256;
constexpr uint32_t kSectionChunks = 16;
constexpr size_t kSectionLeaf = 2048 + 64 + 12;
struct SectionDest {
  char* chunk[kSectionChunks];
  char* rest;
  uint32_t pinned, cap;
};

constexpr uint32_t kRtNodeWords = 128;  // words of RtView::bits per node
// What a snapshot build hands back: bbox (min, max) of leaves with an active
// voxel, nodes in the hash, leaves covered.
struct RtInfo {
  int bbox[6];
  unsigned int nodes, leaves;
};
// A run of existing leaves along a ray of a fast-mode cast.
struct FastSpan {
  double t0, t1;
  uint32_t ray;
  uint32_t len;  // about its voxels
};
constexpr uint32_t kFastSpans = 1024;  // spans per workgroup (256 rays) to start with, and per sort of the walk
// Word and bit of the leaf at (x, y, z) in its 128^3 node.
__host__ __device__ inline int rt_word(int x, int y, int z) {
  return (((x >> 5) & 3) << 4) | (((y >> 5) & 3) << 2) | ((z >> 5) & 3);
}
__host__ __device__ inline int rt_bit(int x, int y, int z) {
  return (((x >> 3) & 3) << 4) | (((y >> 3) & 3) << 2) | ((z >> 3) & 3);
}

__host__ __device__ inline uint64_t leaf_key(int x, int y, int z) {
  const uint64_t m = (1ull << 21) - 1;
  return ((uint64_t)(uint32_t)(x >> 3) & m) << 42 | ((uint64_t)(uint32_t)(y >> 3) & m) << 21 |
         ((uint64_t)(uint32_t)(z >> 3) & m);
}

__host__ __device__ inline int sext21(uint64_t v) { return (int)((int64_t)(v << 43) >> 43); }

__host__ __device__ inline void key_origin(uint64_t k, int o[3]) {
  const uint64_t m = (1ull << 21) - 1;
  o[0] = sext21((k >> 42) & m) * 8;
  o[1] = sext21((k >> 21) & m) * 8;
  o[2] = sext21(k & m) * 8;
}

// MurmurHash3 64-bit finaliser.
__host__ __device__ inline uint64_t fmix64(uint64_t k) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  k *= 0xc4ceb9fe1a85ec53ull;
  k ^= k >> 33;
  return k;
}

// Slot of a leaf key in the map's leaf hash before probing: the key without the
// low two bits of its z coordinate is hashed to a group of four slots, so the
// four leaves of a z column of a brick (neighbouring records) share one 32-byte
// sector of keys and one 16-byte run of indices instead of eight scattered lines
// (the map insert of an outdoor scan: 86 -> 44 us). Two more bits of the hash
// turn the group, so that a flat map, whose leaves all have the same z, uses all
// four slots of its groups (2.1 probes a leaf at half load without, 1.5 with).
__host__ __device__ inline uint32_t map_hash(uint64_t key) {
  const uint64_t h = fmix64(key >> 2);
  return ((uint32_t)h << 2) | (uint32_t)((key + (h >> 62)) & 3);
}

// Slots from one probe to the next in an update set, which map_hash places too.
// Odd, so that a probe run reaches every slot; not 1, because two columns whose
// groups collide would then pile up behind one another, each leaf probing past
// four slots: a step of 5 leads the leaves of the second column to the next
// group's other lanes. Hash-traversal accumulates look a slot up for every leaf
// of every ray chunk: three clouds of 1,000 outdoor rays of 300 voxels 753 us
// with steps of 1, 660 with 5 (654 with every leaf hashed by itself, which costs
// the merged clouds of dense scans their neighbouring slots).
constexpr uint32_t kUpdStep = 5;

__device__ inline bool coord_ok(int c) { return c >= -kCoordLimit && c < kCoordLimit; }

// Update-set key of the leaf holding (x,y,z): the 63-bit leaf key, or in a
// batch the 57-bit leaf key (19-bit coords) shifted left 7 with the scan index.
__host__ __device__ inline uint64_t update_key(int x, int y, int z, uint32_t scan, bool batched) {
  if (!batched) return leaf_key(x, y, z);
  const uint64_t m = (1ull << 19) - 1;
  return (((uint64_t)(uint32_t)(x >> 3) & m) << 45) | (((uint64_t)(uint32_t)(y >> 3) & m) << 26) |
         (((uint64_t)(uint32_t)(z >> 3) & m) << 7) | scan;
}

// Canonical 63-bit leaf key of a batched update key (scan bits dropped).
__host__ __device__ inline uint64_t batched_to_leaf_key(uint64_t k) {
  const uint64_t m = (1ull << 19) - 1;
  const int lx = (int)((int64_t)(((k >> 45) & m) << 45) >> 45);
  const int ly = (int)((int64_t)(((k >> 26) & m) << 45) >> 45);
  const int lz = (int)((int64_t)(((k >> 7) & m) << 45) >> 45);
  return leaf_key(lx * 8, ly * 8, lz * 8);
}

// Key of the brick (32^3 voxels) with brick coordinates (bx,by,bz) = voxel >> 5
// (19-bit fields: voxel coords in [-2^23, 2^23)).
__host__ __device__ inline uint64_t brick_key(int bx, int by, int bz) {
  const uint64_t m = (1ull << 19) - 1;
  return ((uint64_t)(uint32_t)bx & m) << 38 | ((uint64_t)(uint32_t)by & m) << 19 |
         ((uint64_t)(uint32_t)bz & m);
}
__host__ __device__ inline void brick_coords(uint64_t k, int b[3]) {
  const uint64_t m = (1ull << 19) - 1;
  b[0] = (int)((int64_t)(((k >> 38) & m) << 45) >> 45);
  b[1] = (int)((int64_t)(((k >> 19) & m) << 45) >> 45);
  b[2] = (int)((int64_t)((k & m) << 45) >> 45);
}
// Key of the internal node (2^log2dim voxels per side) holding voxel (x,y,z).
__host__ __device__ inline uint64_t node_key(int x, int y, int z, int log2dim) {
  return leaf_key((x >> log2dim) * 8, (y >> log2dim) * 8, (z >> log2dim) * 8);
}

__device__ __forceinline__ bool set_insert(unsigned long long* keys, uint32_t mask, uint64_t key) {
  uint32_t h = (uint32_t)fmix64(key) & mask;
  for (uint32_t p = 0; p <= mask; ++p) {
    const unsigned long long prev = atomicCAS(&keys[h], kEmpty, (unsigned long long)key);
    if (prev == kEmpty) return true;
    if (prev == key) return false;
    h = (h + 1) & mask;
  }
  return false;
}

// set_insert for keys that are mostly present: a read first, since atomics on
// one address (every leaf of a node, every node of a root child) run one
// after another.
__device__ __forceinline__ void set_add(unsigned long long* keys, uint32_t mask, uint64_t key) {
  uint32_t h = (uint32_t)fmix64(key) & mask;
  for (uint32_t p = 0; p <= mask; ++p) {
    unsigned long long k = __hip_atomic_load(&keys[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (k == kEmpty) k = atomicCAS(&keys[h], kEmpty, (unsigned long long)key);
    if (k == kEmpty || k == key) return;
    h = (h + 1) & mask;
  }
}

__device__ __forceinline__ bool set_has(const unsigned long long* __restrict__ keys, uint32_t mask,
                                        uint64_t key) {
  uint32_t h = (uint32_t)fmix64(key) & mask;
  for (uint32_t p = 0; p <= mask; ++p) {
    const unsigned long long k = keys[h];
    if (k == key) return true;
    if (k == kEmpty) return false;
    h = (h + 1) & mask;
  }
  return false;
}

// 8x8 bit-matrix transpose: bit 8r + c of x goes to bit 8c + r.
__device__ __forceinline__ uint64_t transpose8(uint64_t x) {
  uint64_t t = (x ^ (x >> 7)) & 0x00AA00AA00AA00AAull;
  x ^= t ^ (t << 7);
  t = (x ^ (x >> 14)) & 0x0000CCCC0000CCCCull;
  x ^= t ^ (t << 14);
  t = (x ^ (x >> 28)) & 0x00000000F0F0F0F0ull;
  x ^= t ^ (t << 28);
  return x;
}

}  // namespace vdbgpu
