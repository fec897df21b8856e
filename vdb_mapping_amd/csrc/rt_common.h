// Device pieces shared by the raytrace query and the fast-mode raycast: the
// double-precision math::DDA of openvdb (one instance per hierarchy level),
// the live-map active-state probe and the TimeSpan validity test.
#pragma once
#include <float.h>

#include "device_common.h"

namespace vdbgpu {

// An index-space ray: eye + t dir, t in [0, 1] mostly.
struct RtRay {
  double eye[3], dir[3], idir[3];
};

// math::DDA<Ray<double>, Log2Dim>. The step per axis (+-dim) and the time per
// step (step / dir, dim |1 / dir| exactly) follow from the ray, so they are
// not kept: three of these plus the voxel walk's stay in registers. Axes with
// dir 0 have next = DBL_MAX and never win a step that returns true.
template <int kDim>
struct RtDda {
  int vox[3];
  double nxt[3];
  double t0, t1;
  __device__ __forceinline__ void init(const RtRay& r, double start, double max_t) {
    t0 = start;
    t1 = max_t;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double pos = r.eye[a] + r.dir[a] * t0;
      vox[a] = (int)floor(pos) & ~(kDim - 1);
      const double edge = (double)(r.idir[a] > 0 ? vox[a] + kDim : vox[a]);
      nxt[a] = r.dir[a] == 0.0 ? DBL_MAX : t0 + (edge - pos) * r.idir[a];
    }
  }
  // math::MinIndex: ties go to the larger axis.
  __device__ __forceinline__ bool step(const RtRay& r) {
    bool y = nxt[1] <= nxt[0];
    const double m = y ? nxt[1] : nxt[0];
    const bool z = nxt[2] <= m;
    t0 = z ? nxt[2] : m;
    y = y && !z;
    const bool on[3] = {!y && !z, y, z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int st = r.dir[a] == 0.0 ? 0 : (r.idir[a] > 0 ? kDim : -kDim);
      const double next = nxt[a] + (double)kDim * fabs(r.idir[a]);
      vox[a] += on[a] ? st : 0;
      nxt[a] = on[a] ? next : nxt[a];
    }
    return t0 <= t1;
  }
  __device__ __forceinline__ double next() const { return fmin(t1, fmin(nxt[0], fmin(nxt[1], nxt[2]))); }
  // The steps up to the first one that leaves the aligned kBig cube of the
  // current cell, *n of them, or false (nothing done) when time t1 comes first.
  // The state is the one that many step() calls leave: an axis's times are its
  // own running sum whatever the other axes do, and the events before the
  // exit are those with an earlier time, or the same one and a larger axis.
  // Some ten sums and compares per axis stand for up to 3 kBig / kDim whole
  // steps.
  template <int kBig>
  __device__ __forceinline__ bool skip(const RtRay& r, int& n) {
    double T[3];
    int d[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double dlt = (double)kDim * fabs(r.idir[a]);
      const int lo = vox[a] & (kBig - 1);
      d[a] = r.dir[a] == 0.0 ? 0 : (r.idir[a] > 0 ? (kBig - lo) / kDim : lo / kDim + 1);
      T[a] = nxt[a];
      for (int k = 1; k < d[a]; ++k) T[a] += dlt;
    }
    const bool y = T[1] <= T[0];
    const double m = y ? T[1] : T[0];
    const bool z = T[2] <= m;
    const double end = z ? T[2] : m;
    const int A = z ? 2 : (y ? 1 : 0);
    if (!(end <= t1)) return false;
    n = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double dlt = (double)kDim * fabs(r.idir[a]);
      int k = 0;
      if (a == A) {
        k = d[a];
        nxt[a] = end + dlt;
      } else {
        while (nxt[a] < end || (a > A && nxt[a] == end)) {
          nxt[a] += dlt;
          ++k;
        }
      }
      vox[a] += r.idir[a] > 0 ? k * kDim : -k * kDim;  // k = 0 where dir is 0
      n += k;
    }
    t0 = end;
    return true;
  }
};

// Leaves of the snapshot along a ray: the node and the 64-leaf word last read.
// A step of the leaf DDA that rounding puts into a neighbouring node looks
// that node up, as a lookup by leaf key would.
struct LeafBits {
  int nx = 0, ny = 0, nz = 0;
  bool have = false;
  uint32_t node = kNone;
  int wi = -1;
  uint64_t word = 0, act = 0;
  __device__ __forceinline__ bool node_at(const RtView& rt, const int v[3]) {
    const int x = v[0] >> 7, y = v[1] >> 7, z = v[2] >> 7;
    if (!have || x != nx || y != ny || z != nz) {
      nx = x, ny = y, nz = z;
      have = true;
      wi = -1;
      node = kNone;
      const uint64_t key = node_key(v[0], v[1], v[2], 7);
      uint32_t h = (uint32_t)fmix64(key) & rt.n128_mask;
      for (uint32_t p = 0; p <= rt.n128_mask; ++p) {
        const unsigned long long k = rt.n128[h];
        const uint32_t i = rt.nidx[h];  // beside the key: one latency
        if (k == key) {
          node = i;
          break;
        }
        if (k == kEmpty) break;
        h = (h + 1) & rt.n128_mask;
      }
    }
    return node != kNone;
  }
  __device__ __forceinline__ bool read(const RtView& rt, const int v[3]) {
    if (!node_at(rt, v)) return false;
    const int w = rt_word(v[0], v[1], v[2]);
    if (w != wi) {
      wi = w;
      const ulonglong2 p = reinterpret_cast<const ulonglong2*>(rt.bits)[(size_t)node * 64 + w];
      word = p.x;
      act = p.y;
    }
    return true;
  }
  __device__ __forceinline__ bool leaf_at(const RtView& rt, const int v[3]) {
    return read(rt, v) && ((word >> rt_bit(v[0], v[1], v[2])) & 1);
  }
  // Might the leaf hold an active voxel? (As of the snapshot, which is the map
  // as it is when rt.live is 0; a leaf outside the snapshot holds none then.)
  __device__ __forceinline__ bool act_at(const RtView& rt, const int v[3]) {
    return read(rt, v) && ((act >> rt_bit(v[0], v[1], v[2])) & 1);
  }
};

// Active state of a voxel in the live map. While the map is the one the
// snapshot was taken of, the snapshot's bits rule out the leaves without an
// active voxel (most leaves of most rays) without a read of the map: the two
// dependent reads per leaf, to memory beyond the L2, were what a lone ray
// spent its time on. Otherwise the leaf is looked up and keeps the OR of its
// eight mask words, so a (y, z) column without an active voxel needs no
// further read, and the word of the current x.
struct ActiveProbe {
  int px = 0, py = 0, pz = 0;
  bool have = false;
  uint32_t idx = kNone;
  uint64_t any = 0;
  int wx = -1;
  uint64_t word = 0;
  // Does the leaf of voxel v hold an active voxel (as far as known: `any`)?
  __device__ __forceinline__ bool leaf(const MapView& mp, const RtView& rt, LeafBits& lb, const int v[3]) {
    const int x = v[0], y = v[1], z = v[2];
    if (!have || (((x ^ px) | (y ^ py) | (z ^ pz)) & ~7)) {
      px = x, py = y, pz = z;
      have = true;
      wx = -1;
      idx = kNone;
      any = 0;
      // (coord_ok is the same for the whole leaf)
      if (coord_ok(x) && coord_ok(y) && coord_ok(z) && (rt.live || lb.act_at(rt, v))) {
        const uint64_t k = leaf_key(x, y, z);
        uint32_t h = map_hash(k) & mp.cap_mask;
        for (uint32_t p = 0; p <= mp.cap_mask; ++p) {
          const unsigned long long kk = mp.keys[h];
          const uint32_t i = mp.idx[h];  // beside the key: one latency
          if (kk == k) {
            idx = i;
            break;
          }
          if (kk == kEmpty) break;
          h = (h + 1) & mp.cap_mask;
        }
        if (idx != kNone) {
#pragma unroll
          for (int j = 0; j < 8; ++j) any |= mp.active[(size_t)idx * 8 + j];
        }
      }
    }
    return any != 0;
  }
  // Active state of voxel v, in the leaf of the last leaf() call.
  __device__ __forceinline__ bool on(const MapView& mp, const int v[3]) {
    const int b = ((v[1] & 7) << 3) | (v[2] & 7);
    if (!((any >> b) & 1)) return false;
    if ((v[0] & 7) != wx) {
      wx = v[0] & 7;
      word = mp.active[(size_t)idx * 8 + wx];
    }
    return (word >> b) & 1;
  }
};

__device__ __forceinline__ bool span_valid(double t0, double t1) { return (t1 - t0) > 1e-9; }


// VolumeRayIntersector::setIndexRay: Ray::clip to the padded active bbox of
// the snapshot; the times change only when the ray hits the box.
__device__ __forceinline__ void rt_clip(const RtView& rt, const RtRay& r, double& rt0, double& rt1) {
  double c0 = rt0, c1 = rt1;
  bool hit = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (!hit) break;
    double ta = ((double)rt.bmin[a] - r.eye[a]) * r.idir[a];
    double tb = ((double)rt.bmax[a] - r.eye[a]) * r.idir[a];
    if (ta > tb) {
      const double t = ta;
      ta = tb;
      tb = t;
    }
    if (ta > c0) c0 = ta;
    if (tb < c1) c1 = tb;
    if (c0 > c1) hit = false;
  }
  if (hit) {
    rt0 = c0;
    rt1 = c1;
  }
}

// VolumeHDDA over the snapshot (4096 -> 128 -> 8): the runs of existing leaves
// along a ray as time spans, one per call. All lanes of a wave look for their
// next span together and then walk them together; walking a span where it was
// found, inside the three nested loops, ran one lane's span after another's.
// kSkip: leave blocks of leaves that are all there or all missing in one go. It
// pays where most are (a map built in normal mode: a million queries 1.30 ->
// 1.06 ms); the surface leaves of a fast-mode map mix them, and its short
// walks end in the block more often than not (fast cast 1.0 -> 1.2 ms).
// kTogether: a lane through with a node waits until so many lanes are, or none
// is left among leaves, and they look for their next nodes together: that
// search, a chain of probes, ran in nearly every step for a few lanes (262,144
// fast-mode rays 518 us; 409 with the node levels in one pass at the end of the
// step, 399 for 8 lanes, 379 for 16, 390 for 32; a million queries 1.06 ms; 0.91,
// 0.90, 0.93, 0.94).
template <bool kSkip, int kTogether>
struct SpanFinder {
  RtDda<4096> d12;
  RtDda<128> d7;
  RtDda<8> d3;
  bool can_skip;
  int level;       // of the cell examined next; 0: through
  double s0, s1;   // the open span
  __device__ __forceinline__ void init(const RtRay& r, double t0, double t1) {
    d12.init(r, t0, t1);
    level = 12;
    can_skip = false;
    s0 = s1 = -1;
  }
  __device__ __forceinline__ bool close(double t, double& a, double& b) {
    s1 = t;
    const bool ok = span_valid(s0, s1);
    a = s0;
    b = s1;
    s0 = s1 = -1;
    return ok;
  }
  __device__ __forceinline__ bool next(const RtView& rt, const RtRay& r, LeafBits& lb, int& budget, double& a,
                                       double& b) {
    while (level) {
      bool found = false;
      if (level == 3) {
        if (lb.leaf_at(rt, d3.vox)) {
          if (s0 < 0) s0 = d3.t0;
        } else if (s0 >= 0) {
          found = close(d3.t0, a, b);
        }
        // 64 leaves that are all there or all missing answer alike: on to
        // the end of their block
        int n = 1;
        bool more = kSkip && can_skip && lb.node != kNone && (lb.word == 0 || lb.word == ~0ull);
        if (more) more = can_skip = d3.template skip<32>(r, n);  // refused: this walk ends in the block
        if (!more) more = d3.step(r);
        if (!(more && (budget -= n) > 0)) {
          if (s0 >= 0) s1 = d3.t1;
          level = 8;  // past this node
        }
      }
      const bool up = level != 3;
      if (__popcll(__ballot(up)) < kTogether && __ballot(!up)) {
        if (found) return true;
        continue;
      }
      if (level == 8) {
        level = 7;
        if (!(d7.step(r) && --budget > 0)) {
          if (s0 >= 0) s1 = d7.t1;
          level = 13;
        }
      }
      if (level == 13) {
        level = 12;
        if (!(d12.step(r) && --budget > 0)) {
          level = 0;
          if (s0 >= 0) {
            s1 = d12.t1;
            a = s0;
            b = s1;
            found = span_valid(s0, s1);
          }
        }
      }
      if (level == 12) {
        if (set_has(rt.n4096, rt.n4096_mask, node_key(d12.vox[0], d12.vox[1], d12.vox[2], 12))) {
          d7.init(r, d12.t0, d12.next());
          level = 7;
        } else {
          if (s0 >= 0) found = close(d12.t0, a, b);
          level = 13;
        }
      }
      if (level == 7) {
        if (lb.node_at(rt, d7.vox)) {
          d3.init(r, d7.t0, d7.next());
          can_skip = true;
          level = 3;
        } else {
          if (s0 >= 0) found = close(d7.t0, a, b);
          level = 8;
        }
      }
      if (found) return true;
    }
    return false;
  }
};

}  // namespace vdbgpu
