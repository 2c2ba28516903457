// Device pieces shared by every stamp kernel (fused.hip, batch.hip,
// batchwave.hip, serve.hip, persistent.hip) and the adjoint (grad.hip): the
// planned stamp descriptor, the window tiles and their visits, the tape record,
// the snapshot ring, the shared-pixel levels, and the bounded group barrier of
// the kernels that run many stamps a launch.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "dry.hpp"
#include "internal.hpp"
#include "visit.hpp"

namespace pnt {

// Bounding box (map cells, inclusive) of the footprint's nonzero values: a
// visit whose cell lies outside it has fh = 0 and changes nothing, so its
// loads are skipped (an ALU test, no memory round trip).
struct FpBox {
  int x0, y0, x1, y1;
};


enum : uint32_t { kStDip = 1u, kStDupX = 2u, kStDupY = 4u };

// One imprint, planned on the host (FP64 geometry as stamp_args computes it).
struct PStamp {
  double cx, cy, c, s;
  float K[3], S[3];  // paint of a dip before this stamp
  uint32_t flags;    // kStDip | kStDupX | kStDupY
  int32_t dl_lev;    // first entry of this stamp's level offsets (dup stamps)
  int32_t dl_nlev;   // number of shared-pixel levels (0 if none)
  RingBox box;
  int32_t pad0;
  int64_t now_us;  // the imprint's time point when the canvas has a drying clock
  int32_t pad[4];
};
static_assert(sizeof(PStamp) % 16 == 0, "PStamp alignment");

// ------------------------------------------------------------ barriers ---
// Barrier words of one group, one 128-byte line each: 8 arrival counters,
// the leader counter, the generation, the abort flag.
constexpr int kBarLine = 32;
constexpr int kBarGroups = 8;
constexpr int kBarTop = kBarGroups * kBarLine;
constexpr int kBarGen = kBarTop + kBarLine;
constexpr int kBarAbort = kBarGen + kBarLine;
constexpr int kBarWords = kBarAbort + kBarLine;
constexpr unsigned kSpinLimit = 1u << 22;

// Barrier over the `nblocks` co-resident blocks of a group (`rank` in
// [0, nblocks)).
//  * Each wave drains its own loads and stores (s_waitcnt 0): a workgroup
//    barrier alone does not wait for global stores.  Then one wave per block
//    writes its XCD's L2 back (agent-scope release): the L2s of different
//    XCDs are not coherent with each other.
//  * Arrival is two-level (8 sub-groups by rank, then their leaders) on
//    counters that only grow, so no counter is ever reset.
//  * Waiters spin on relaxed loads (an acquire load would invalidate the L2
//    on every poll) and acquire once the generation moves.
//  * The wait is bounded: on expiry the abort flag is raised, every block
//    leaves at its next barrier, and the pinned host word reports it.
// Returns false when the run is aborted.
__device__ __forceinline__ bool group_sync(unsigned* bar, unsigned nblocks, unsigned rank,
                                           unsigned* host_err) {
  __shared__ int s_ok;
  if (nblocks == 1) {  // one block: a workgroup barrier orders everything
    __syncthreads();
    return true;
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    int ok = 1;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const unsigned gen =
        __hip_atomic_load(&bar[kBarGen], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned grp = rank & (kBarGroups - 1);
    const unsigned ngroups = nblocks < (unsigned)kBarGroups ? nblocks : (unsigned)kBarGroups;
    const unsigned in_grp = nblocks / kBarGroups + (grp < nblocks % kBarGroups ? 1u : 0u);
    const unsigned a = __hip_atomic_fetch_add(&bar[grp * kBarLine], 1u, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
    bool last = false;
    if ((a + 1) % in_grp == 0) {
      const unsigned t = __hip_atomic_fetch_add(&bar[kBarTop], 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
      last = (t + 1) % ngroups == 0;
    }
    if (last) {
      __hip_atomic_store(&bar[kBarGen], gen + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      unsigned spins = 0;
      while (__hip_atomic_load(&bar[kBarGen], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             gen) {
        __builtin_amdgcn_s_sleep(1);
        if ((++spins & 63) == 0) {
          if (__hip_atomic_load(&bar[kBarAbort], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            ok = 0;
            break;
          }
          if (spins > kSpinLimit) {
            __hip_atomic_store(&bar[kBarAbort], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(host_err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            ok = 0;
            break;
          }
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (__hip_atomic_load(&bar[kBarAbort], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) ok = 0;
    s_ok = ok;
  }
  __syncthreads();
  return s_ok != 0;
}

// --------------------------------------------------------------- visits ---
// One visit with every value it may need loaded up front (one memory round
// trip): the canvas pixel, and the pickup source -- the snapshot pixel, the
// canvas itself when the snapshot is off, or, on the window border where
// this stamp's snapshot refresh copies canvas -> snapshot just before the
// visits (FootprintBrush.hxx:307-318), the canvas value that refresh copies.
// PickAcc supplies pick(c) / set_pick(c, v) for the visit's map cell.
template <class PickAcc>
struct CachedVisit : PickAcc {
  float sv[6], cv[6];  // K, S of the pickup source and of the canvas pixel
  double svv, cvv;     // their volumes
  bool alias;          // pickup source is the canvas itself (snapshot off)
  bool src_moved;      // the pickup changed the source volume
  __device__ float src(int c) const { return sv[c]; }
  __device__ double src_v() const { return svv; }
  __device__ void set_src_v(double v) {
    svv = v;
    if (alias) cvv = v;
    src_moved = true;
  }
  __device__ float canvas(int c) const { return cv[c]; }
  __device__ double canvas_v() const { return cvv; }
  __device__ void set_canvas(int c, float v) { cv[c] = v; }
  __device__ void set_canvas_v(double v) { cvv = v; }
  // the pickup source is the canvas pixel itself
  __device__ void src_from_canvas() {
#pragma unroll
    for (int c = 0; c < 6; ++c) sv[c] = cv[c];
    svv = cvv;
  }
};

// One pixel of a layer: K, S (FP32) and V (FP64).
__device__ __forceinline__ void ld_px(const Layer7& L, int64_t i, float ks[6], double& v) {
#pragma unroll
  for (int c = 0; c < 6; ++c) ks[c] = L.ks[c][i];
  v = L.v[i];
}
__device__ __forceinline__ void st_px(const Layer7& L, int64_t i, const float ks[6], double v) {
#pragma unroll
  for (int c = 0; c < 6; ++c) L.ks[c][i] = ks[c];
  L.v[i] = v;
}

// One stamp's tape record: the canvas and pickup-source pixels as its visits
// find them, by pixel of its window box clipped to the canvas, and the map
// cells before their first visits.  Only the visited entries are written.
// A pixel's values lie together, as a cell's do: two 16-byte accesses.
struct alignas(16) TapePx {
  float ks[6];
  double v;
};
struct TapeRec {
  TapePx *c, *x;  // canvas, pickup source: `area` pixels each
  float* P;       // `m` cells (kCell)
  int64_t area, m;
  int bx0, by0, bw;
  __host__ __device__ int64_t at(int x, int y) const { return (int64_t)(y - by0) * bw + (x - bx0); }
};
__host__ __device__ inline int64_t tape_floats(int64_t area, int64_t m) {
  return 16 * area + kCell * m;
}
__host__ __device__ inline TapeRec tape_rec(float* base, int64_t area, int64_t m, const RingBox& b,
                                            int cols) {
  TapeRec t;
  t.c = reinterpret_cast<TapePx*>(base);
  t.x = t.c + area;
  t.P = base + 16 * area;
  t.area = area;
  t.m = m;
  t.bx0 = b.tl_x > 0 ? b.tl_x : 0;
  t.by0 = b.tl_y > 0 ? b.tl_y : 0;
  t.bw = (b.br_x < cols - 1 ? b.br_x : cols - 1) - t.bx0 + 1;
  return t;
}

// Where one visit reads and writes.
struct VisitTarget {
  const Layer7* canvas;
  const Layer7* src;  // snapshot planes (unused when use_snap == 0)
  uint8_t* dirty;
  int use_snap;
  double pickup_rate, dep_rate, cap;
  const TapeRec* tape = nullptr;  // StampKind::tape
};

// Tile of block b when blocks [0, ntiles) take one tile each: blocks go
// round-robin to the 8 XCDs, so each XCD gets a contiguous run of tiles and
// works on one band of the map (and of the window) in its own L2.
__device__ __forceinline__ int tile_of_block(int b, int ntiles) {
  const int x = b & 7, q = b >> 3;
  const int base = ntiles >> 3, rem = ntiles & 7;
  return x * base + (x < rem ? x : rem) + q;
}

// ----------------------------------------------------------- ring helpers -
// Does stamp p straddle canvas column/row 0 with shared-pixel visits (which
// then run by level on a block of their own)?
__host__ __device__ inline bool dup_levels(const PStamp& p) {
  return (p.flags & (kStDupX | kStDupY)) && p.dl_nlev > 0;
}

__device__ __forceinline__ bool on_dup_line(const PStamp& st, int col, int row) {
  return ((st.flags & kStDupX) && (int)(col + st.cx) == 0) ||
         ((st.flags & kStDupY) && (int)(row + st.cy) == 0);
}

// Every window offset k in [-hr, hr] with (int)(k + c) == x, ascending: one
// for most pixels, two on a duplicated canvas column/row 0, none off the
// window.  Returns how many.
__device__ __forceinline__ int window_offsets(int x, double c, int hr, int k[2]) {
#pragma clang fp contract(off)
  const int k0 = x - (int)floor(c);
  int n = 0;
  for (int d = -1; d <= 1; ++d) {
    const int kk = k0 + d;
    if (kk >= -hr && kk <= hr && (int)(kk + c) == x && n < 2) k[n++] = kk;
  }
  return n;
}

// Is canvas pixel (x, y), on the ring of this stamp, also visited with a
// footprint height > 0 by it (and therefore refreshed by that visit)?  With
// a drying clock every visited pixel counts: its window tile refreshes it
// before checkDry changes the canvas.  A pixel of a duplicated column/row 0
// counts when any of its visits does (the first of them refreshes it).
__device__ __forceinline__ bool ring_pixel_visited(const StampGeom& g, const RingBox& b,
                                                   const float* fp, int x, int y,
                                                   bool any_visit = false) {
  if (x < b.tl_x || x > b.br_x || y < b.tl_y || y > b.br_y) return false;
  int cs[2], rs[2];
  const int nc = window_offsets(x, g.cx, g.hr, cs), nr = window_offsets(y, g.cy, g.hr, rs);
  for (int r = 0; r < nr; ++r)
    for (int c = 0; c < nc; ++c) {
      int64_t ic;
      const int m = stamp_visit(g, cs[c], rs[r], &ic);
      if (m >= 0 && (any_visit || fp[m] > 0.0f)) return true;
    }
  return false;
}

__device__ __forceinline__ bool on_window_border(const RingBox& b, int x, int y) {
  return x == b.tl_x || x == b.br_x || y == b.tl_y || y == b.br_y;
}

// Snapshot ring refresh of one stamp (updateSnapshot(canvas, center),
// FootprintBrush.hxx:307-318) by block `blk` of `nblk`, kThreads threads
// each (all of which must call it).  A set dirty byte says that the pixel's
// snapshot differs from the canvas; for the set pixels of the allowed box
// outside the window interior the block copies canvas -> snapshot and clears
// the byte.  With `pull`, window-border pixels that a visit of this stamp
// refreshes itself are left to that visit.
//
// A thread reads the 8 dirty bytes of 8 pixels at an 8-aligned linear
// index in one load and lists the 4-pixel groups that hold work in LDS; then
// the block shares the list out by pixel (which border pixels a visit
// refreshes) and by plane (the copies).  The dirty strip behind a moving
// window is contiguous: where a thread copied what it found itself, the few
// that found the strip made one memory round trip per group, and the slowest
// ring block held up its launch (16 us, beside tiles of 5.6 us on average).
// Plane and dirty buffers are padded past the last pixel to a multiple of
// 16, so a unit never leaves them.
constexpr int kRingUnit = 8;                 // pixels per dirty load
constexpr int kRingGroups = kRingUnit / 4;   // 4-pixel groups per thread and pass

template <int kThreads>
struct RingList {  // the groups of a pass: pixel base relative to the box's first, mask
  unsigned n;
  unsigned g[kRingGroups * kThreads];  // group number << 8 | border bits << 4 | copy bits
};

template <int kThreads>
__device__ __forceinline__ void ring_scan(const Layer7& canvas, const Layer7& snap, uint8_t* dirty,
                                          const float* fp, const StampGeom& g, const RingBox& b,
                                          bool pull, int blk, int nblk, RingList<kThreads>& list,
                                          bool clocked = false) {
  if (b.a_x1 < b.a_x0 || b.a_y1 < b.a_y0) return;
  const int rows = b.a_y1 - b.a_y0 + 1;
  const int span = b.a_x1 - b.a_x0 + 1;
  const int per_row = (span + kRingUnit - 1) / kRingUnit + 1;  // +1: misaligned start
  const int total = per_row * rows;
  // pixel base of group q of unit e, and its canvas row and first column
  const auto unit = [&](int e, int* row, int* x0) {
    const int r = e / per_row;
    *row = b.a_y0 + r;
    const int64_t rowi = (int64_t)*row * g.cols, lo = rowi + b.a_x0;
    const int64_t base = (lo & ~(int64_t)(kRingUnit - 1)) + kRingUnit * (int64_t)(e - r * per_row);
    *x0 = (int)(base - rowi);
    return base;
  };
  for (int p0 = blk * kThreads; p0 < total; p0 += nblk * kThreads) {
    if (threadIdx.x == 0) list.n = 0;
    __syncthreads();
    const int e = p0 + (int)threadIdx.x;
    if (e < total) {
      int row, x0;
      const int64_t base = unit(e, &row, &x0);
      const bool interior_row = row > b.tl_y && row < b.br_y;
      if (x0 <= b.a_x1 && !(interior_row && x0 > b.tl_x && x0 + kRingUnit - 1 < b.br_x)) {
        const uint2 d2 = *reinterpret_cast<const uint2*>(dirty + base);
        const unsigned d[kRingGroups] = {d2.x, d2.y};
#pragma unroll
        for (int q = 0; q < kRingGroups; ++q) {
          if (!d[q]) continue;
          unsigned m = 0u, border = 0u;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int col = x0 + 4 * q + k;
            const bool in = ((d[q] >> (8 * k)) & 0xffu) && col >= b.a_x0 && col <= b.a_x1 &&
                            !(interior_row && col > b.tl_x && col < b.br_x);
            m |= (in ? 1u : 0u) << k;
            border |= (in && pull && on_window_border(b, col, row) ? 1u : 0u) << k;
          }
          if (m)
            list.g[atomicAdd(&list.n, 1u)] =
                ((unsigned)(threadIdx.x * kRingGroups + q) << 8) | (border << 4) | m;
        }
      }
    }
    __syncthreads();
    const int n = (int)list.n;
    // window-border pixels that a visit refreshes itself
    for (int i = threadIdx.x; i < 4 * n; i += kThreads) {
      const unsigned w = list.g[i >> 2];
      if (!((w >> (4 + (i & 3))) & 1u)) continue;
      int row, x0;
      unit(p0 + (int)(w >> 8) / kRingGroups, &row, &x0);
      const int col = x0 + 4 * ((int)(w >> 8) % kRingGroups) + (i & 3);
      if (ring_pixel_visited(g, b, fp, col, row, clocked)) atomicAnd(&list.g[i >> 2], ~(1u << (i & 3)));
    }
    __syncthreads();
    // the copies: a thread takes one plane (or half of the FP64 volumes) of a
    // group, eight groups' loads in flight together
    constexpr int kPer = kThreads / 8, kFlight = 8;
    const int plane = (int)threadIdx.x & 7;
    for (int i0 = (int)threadIdx.x >> 3; i0 < n; i0 += kFlight * kPer) {
      float4 v[kFlight];
      unsigned m[kFlight];
      int64_t at[kFlight];
#pragma unroll
      for (int u = 0; u < kFlight; ++u) {
        const int i = i0 + u * kPer;
        const unsigned w = i < n ? list.g[i] : 0u;
        m[u] = w & 0xfu;
        at[u] = 0;
        if (!m[u]) continue;
        int row, x0;
        at[u] = unit(p0 + (int)(w >> 8) / kRingGroups, &row, &x0) + 4 * ((int)(w >> 8) % kRingGroups);
        v[u] = plane < 6 ? *reinterpret_cast<const float4*>(canvas.ks[0] + plane * (canvas.ks[1] - canvas.ks[0]) + at[u])
                         : *reinterpret_cast<const float4*>(canvas.v + at[u] + 2 * (plane - 6));
      }
#pragma unroll
      for (int u = 0; u < kFlight; ++u) {
        if (!m[u]) continue;
        if (plane < 6) {
          float* dst = snap.ks[0] + plane * (snap.ks[1] - snap.ks[0]) + at[u];
          if (m[u] == 0xfu) {
            *reinterpret_cast<float4*>(dst) = v[u];
          } else {
            if (m[u] & 1u) dst[0] = v[u].x;
            if (m[u] & 2u) dst[1] = v[u].y;
            if (m[u] & 4u) dst[2] = v[u].z;
            if (m[u] & 8u) dst[3] = v[u].w;
          }
        } else {
          float2* dst = reinterpret_cast<float2*>(snap.v + at[u]) + 2 * (plane - 6);
          const unsigned h = m[u] >> (2 * (plane - 6));
          if (h & 1u) dst[0] = make_float2(v[u].x, v[u].y);
          if (h & 2u) dst[1] = make_float2(v[u].z, v[u].w);
        }
        if (plane == 0) {
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if ((m[u] >> k) & 1u) dirty[at[u] + k] = 0;
        }
      }
    }
    __syncthreads();  // the list is rewritten by the next pass
  }
}

// The same refresh without dirty bytes: every pixel of the ring is copied,
// one a thread, except the border pixels left to their visits.
template <int kThreads>
__device__ __forceinline__ void ring_copy(const Layer7& canvas, const Layer7& snap,
                                          const float* fp, const StampGeom& g, const RingBox& b,
                                          int blk, int nblk, bool clocked) {
  const int w = b.a_x1 - b.a_x0 + 1, h = b.a_y1 - b.a_y0 + 1;
  if (w <= 0 || h <= 0) return;
  const int64_t total = (int64_t)w * h;
  for (int64_t e = (int64_t)blk * kThreads + threadIdx.x; e < total; e += (int64_t)nblk * kThreads) {
    const int r = (int)(e / w), row = b.a_y0 + r, col = b.a_x0 + (int)(e - (int64_t)r * w);
    if (row > b.tl_y && row < b.br_y && col > b.tl_x && col < b.br_x) continue;
    const int64_t i = (int64_t)row * g.cols + col;
    float ks[6];
    double v;
    ld_px(canvas, i, ks, v);
    if (on_window_border(b, col, row) && ring_pixel_visited(g, b, fp, col, row, clocked)) continue;
    st_px(snap, i, ks, v);
  }
}

// Pickup map cell held in registers between its load and its store.
struct RegPick {
  float v[7];
  __device__ float pick(int c) const { return v[c]; }
  __device__ void set_pick(int c, float x) { v[c] = x; }
};

// Cell m of a pickup map.
__device__ __forceinline__ void ld_cell(const float* pick, int m, float v[7]) {
  const float4* p = reinterpret_cast<const float4*>(pick) + 2 * (int64_t)m;
  const float4 a = p[0], b = p[1];
  v[0] = a.x;
  v[1] = a.y;
  v[2] = a.z;
  v[3] = a.w;
  v[4] = b.x;
  v[5] = b.y;
  v[6] = b.z;
}
__device__ __forceinline__ void st_cell(float* pick, int m, const float v[7]) {
  float4* p = reinterpret_cast<float4*>(pick) + 2 * (int64_t)m;
  p[0] = make_float4(v[0], v[1], v[2], v[3]);
  p[1] = make_float4(v[4], v[5], v[6], 0.0f);
}

// Loads everything one visit reads: canvas and pickup-source pixel.
template <class PickAcc>
__device__ __forceinline__ void load_pixel(const VisitTarget& T, bool snap, int64_t ic, bool pull,
                                           CachedVisit<PickAcc>& acc) {
  ld_px(*T.canvas, ic, acc.cv, acc.cvv);
  if (snap && !pull)
    ld_px(*T.src, ic, acc.sv, acc.svv);
  else
    acc.src_from_canvas();
  acc.src_moved = false;
}

// Stores the canvas / snapshot side of a visit.
template <class PickAcc>
__device__ __forceinline__ void store_pixel(const VisitTarget& T, bool snap, int64_t ic, bool pull,
                                            const CachedVisit<PickAcc>& acc) {
  st_px(*T.canvas, ic, acc.cv, acc.cvv);
  if (snap) {
    if (pull)
      st_px(*T.src, ic, acc.sv, acc.svv);
    else if (acc.src_moved)
      T.src->v[ic] = acc.svv;
    if (T.dirty) T.dirty[ic] = 1;
  }
}

// The pixel (x, y) as a visit finds it, into the tape.
__device__ __forceinline__ void tape_pixel(const TapeRec& t, bool snap, int x, int y,
                                           const float cv[6], double cvv, const float sv[6],
                                           double svv) {
  const int64_t k = t.at(x, y);
  TapePx p;
#pragma unroll
  for (int c = 0; c < 6; ++c) p.ks[c] = cv[c];
  p.v = cvv;
  t.c[k] = p;
  if (!snap) return;
#pragma unroll
  for (int c = 0; c < 6; ++c) p.ks[c] = sv[c];
  p.v = svv;
  t.x[k] = p;
}

// One whole visit of map cell m at canvas pixel ic: everything it reads in
// one batch, the arithmetic, the stores.
__device__ __forceinline__ void cached_visit(const VisitTarget& T, float* pick, int m,
                                             float fh, int64_t ic, bool pull, const float pk[3],
                                             const float ps[3]) {
  CachedVisit<RegPick> acc;
  acc.alias = !T.use_snap;
  ld_cell(pick, m, acc.v);
  load_pixel(T, T.use_snap, ic, pull, acc);
  paint_visit_math(acc, fh, T.pickup_rate, T.dep_rate, T.cap, pk, ps);
  store_pixel(T, T.use_snap, ic, pull, acc);
  st_cell(pick, m, acc.v);
}

// Canvas::checkDry (Canvas.hxx:123-155) of a visited pixel whose canvas
// values are held in registers (ks[6], v); R0, h and the time map are in
// memory.  The same arithmetic as check_dry (dry.hpp).
__device__ __forceinline__ void check_dry_regs(const DryClock& c, float ks[6], double& v,
                                               int64_t ic) {
  if (c.dry_ms > 0 && v > 0.001) {
    const int64_t elapsed_ms = (c.now_us - c.tmap[ic]) / 1000;  // duration_cast truncation
    if (elapsed_ms >= c.dry_ms) {
      float K[3], S[3];
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) {
        K[ch] = ks[ch];
        S[ch] = ks[3 + ch];
      }
      dry_pixel_into(c, K, S, v, ic);
#pragma unroll
      for (int ch = 0; ch < 6; ++ch) ks[ch] = 0.0f;
      v = 0.0;
    }
  }
  c.tmap[ic] = c.now_us;
}

// checkDry of a visited pixel with footprint height <= 0 (no pickup or
// deposit follows).  On the window border of a stamp that refreshes its
// border itself (`pull`), the snapshot refresh comes first, as
// updateSnapshot runs before the visits (FootprintBrush.hxx:80-84).  A
// pixel that dries no longer equals its snapshot.
__device__ __forceinline__ void check_only(const VisitTarget& T, const DryClock& c, int64_t ic,
                                           bool pv) {
  if (pv) {
    float ks[6];
    double v;
    ld_px(*T.canvas, ic, ks, v);
    st_px(*T.src, ic, ks, v);
    if (T.dirty) T.dirty[ic] = 0;
  }
  const double v0 = T.canvas->v[ic];
  check_dry(c, *T.canvas, ic);
  if (T.use_snap && T.dirty && v0 > 0.001 && T.canvas->v[ic] != v0) T.dirty[ic] = 1;
}

// The map cells a stamp's visits are run over: the footprint's nonzero box,
// or, with a drying clock, the whole map (every visited pixel is checked,
// whatever its footprint height).
__host__ __device__ inline FpBox cell_domain(const FpBox& nonzero, int size_map, bool clocked) {
  return clocked ? FpBox{0, 0, size_map - 1, size_map - 1} : nonzero;
}

// The window offsets that can fall on a box of map cells and on the canvas,
// cut into tiles.
struct TileWin {
  int col0, row0, cols, rows;  // first offset, extent (<= 0: none)
};

// Rotating a cell's centre back gives a point within (|c| + |s|) / 2 <=
// 0.70711 of its visitors along both axes, so the box's corners bound the
// offsets.  Half of a window holds no footprint (its side is sqrt(2) times
// the footprint's, so that every rotation fits): without the cut, half of
// the workgroups of a stamp would find nothing to do.
__host__ __device__ __forceinline__ TileWin tile_window(const StampGeom& g, const FpBox& dom) {
#pragma clang fp contract(off)
  const double hr = (double)g.hr;
  const double u0 = (double)dom.x0 - hr, u1 = (double)dom.x1 - hr;
  const double v0 = (double)dom.y0 - hr, v1 = (double)dom.y1 - hr;
  // col = u c + v s, row = v c - u s
  const double clo = (g.c >= 0.0 ? u0 : u1) * g.c + (g.s >= 0.0 ? v0 : v1) * g.s - 0.7072;
  const double chi = (g.c >= 0.0 ? u1 : u0) * g.c + (g.s >= 0.0 ? v1 : v0) * g.s + 0.7072;
  const double rlo = (g.c >= 0.0 ? v0 : v1) * g.c - (g.s >= 0.0 ? u1 : u0) * g.s - 0.7072;
  const double rhi = (g.c >= 0.0 ? v1 : v0) * g.c - (g.s >= 0.0 ? u0 : u1) * g.s + 0.7072;
  // offsets on the canvas: -1 < offset + centre < side
  const int col0 = (int)fmax(fmax(floor(clo), -hr), floor(-g.cx) - 1.0);
  const int col1 = (int)fmin(fmin(ceil(chi), hr), ceil((double)g.cols - g.cx));
  const int row0 = (int)fmax(fmax(floor(rlo), -hr), floor(-g.cy) - 1.0);
  const int row1 = (int)fmin(fmin(ceil(rhi), hr), ceil((double)g.rows - g.cy));
  const bool any = dom.x1 >= dom.x0 && dom.y1 >= dom.y0;
  return TileWin{col0, row0, any ? col1 - col0 + 1 : 0, any ? row1 - row0 + 1 : 0};
}
// Tiles of kT x kT offsets that cover the window (at least 1).
template <int kT>
__host__ __device__ inline int tile_count(const TileWin& w) {
  if (w.cols <= 0 || w.rows <= 0) return 1;
  return ((w.cols + kT - 1) / kT) * ((w.rows + kT - 1) / kT);
}

// tile / tiles_x by r, 1 / tiles_x within an ulp: the half keeps the product at
// least 0.5 / tiles_x from a whole number.  The largest map (a footprint of
// radius 4095, 11587 cells a side) has 725 tiles a side: 6.9e-4 there, beside a
// rounding of at most 1.3e-4.
__host__ __device__ __forceinline__ int tile_row(int tile, float r) {
  return (int)(((float)tile + 0.5f) * r);
}

__host__ __device__ inline StampGeom stamp_geom(const PStamp& p, int size_map, int rows, int cols) {
  return StampGeom{p.cx, p.cy, p.c, p.s, (size_map - 1) / 2, size_map, rows, cols};
}

// A window offset's visit and who shares its map cell.
struct VisitCell {
  int mm;    // map cell, -1: no visit (outside the window, canvas, map or box)
  int x, y;  // canvas pixel
  int shared;  // 0 alone, 1..4: with the left, upper, right, lower neighbour
};

// Is z, a map coordinate before rounding, rounded to cell m?  Round half
// away from zero: m - 0.5 <= z < m + 0.5, the lower bound open for m = 0.
__host__ __device__ __forceinline__ bool rounds_to(double z, int m) {
  const double lo = (double)m - 0.5;
  return (m == 0 ? z > lo : z >= lo) && z < (double)m + 0.5;
}

// The visit of window offset (col, row), with the index arithmetic of
// stamp_visit, and the 4-neighbour that falls on the same cell: rotation
// preserves distances and a half-open unit cell holds no two points a
// distance >= 1 apart except 4-neighbours, so a cell has at most two
// visitors.
//
// A neighbour lies (+-c, +-s) or (+-s, -+c) away on the map; FP32 places it
// in or out of the cell unless it lies within 4e-6 of the cell's edge (the
// FP32 error is below 2e-7), and only then is its own FP64 index arithmetic
// run.  A stamp kernel is a chain of latencies, this test its longest
// arithmetic one.
__host__ __device__ __forceinline__ VisitCell visit_cell(const StampGeom& g, const FpBox& dom,
                                                         int col, int row) {
#pragma clang fp contract(off)
  VisitCell V{-1, 0, 0, 0};
  const double dc = (double)col, dr = (double)row, hr = (double)g.hr;
  V.x = (int)(dc + g.cx);
  V.y = (int)(dr + g.cy);
  const double zx = (dc * g.c - dr * g.s) + hr, zy = (dc * g.s + dr * g.c) + hr;
  const int mx = map_round(zx), my = map_round(zy);
  const bool ok = (unsigned)(col + g.hr) <= (unsigned)(2 * g.hr) &&
                  (unsigned)(row + g.hr) <= (unsigned)(2 * g.hr) && V.x >= 0 && V.y >= 0 &&
                  V.x < g.cols && V.y < g.rows && mx >= dom.x0 && mx <= dom.x1 &&
                  my >= dom.y0 && my <= dom.y1;
  if (!ok) return V;
  V.mm = my * g.size_map + mx;
  const float px = (float)(zx - (double)mx), py = (float)(zy - (double)my);
  const float cf = (float)g.c, sf = (float)g.s;
  constexpr float kEdge = 0.5f + 4e-6f;
  bool near_edge = false;
  int shared = 0;
  const auto test = [&](float qx, float qy, int dir) {
    const float m = fmaxf(fabsf(qx), fabsf(qy));
    if (m < kEdge) {
      shared = dir;
      near_edge |= m > 0.5f - 4e-6f;
    }
  };
  test(px - cf, py - sf, 1);
  test(px + sf, py - cf, 2);
  test(px + cf, py + sf, 3);
  test(px - sf, py + cf, 4);
  if (near_edge) {
    shared = 0;
    for (int d = 1; d <= 4; ++d) {
      const double nc = dc + (double)(d == 3) - (double)(d == 1);
      const double nr = dr + (double)(d == 4) - (double)(d == 2);
      if (rounds_to((nc * g.c - nr * g.s) + hr, mx) && rounds_to((nc * g.s + nr * g.c) + hr, my))
        shared = d;
    }
  }
  if (shared) {  // a neighbour outside the window or the canvas is no visit
    const int dx = (shared == 3) - (shared == 1), dy = (shared == 4) - (shared == 2);
    const int x = (int)((dc + (double)dx) + g.cx), y = (int)((dr + (double)dy) + g.cy);
    if ((unsigned)(col + dx + g.hr) <= (unsigned)(2 * g.hr) &&
        (unsigned)(row + dy + g.hr) <= (unsigned)(2 * g.hr) && x >= 0 && y >= 0 && x < g.cols &&
        y < g.rows)
      V.shared = shared;
  }
  return V;
}

// The visits of one kT x kT tile of a stamp's window, by one workgroup of
// kT*kT threads (all of which must call it), one visit per thread.
//
// A cell shared by two visits passes from the first to the second in
// reference order (the left or upper one first) through LDS (`hand`: 8
// floats per thread): every thread loads and stores its own pixel, in whole
// rows, and none carries a second one in registers.  Only where the second
// lies outside the tile does the first one's thread run both.  Visits on a
// duplicated canvas column/row 0 (and the visits sharing their cells) are
// left out; level_visits runs them.
//
// Bound: the L1's line lookups and the two memory round trips of a visit
// (its cell, fetched with the pixel's values, then the stores).  Map cells
// are met along a rotated row, 64 of them on about 16 rows of the map, and
// are kept whole (kCell) for that.
//
// With a drying clock (clk.tmap != nullptr) every visited pixel -- in the canvas
// and in the map, whatever its footprint height -- gets Canvas::checkDry
// before its pickup and deposit (FootprintBrush.hxx:115).
//
// F: what the stamps of the launch may need (StampKind); code for what they
// don't is left out, which shortens every wave's first pass over cold
// instruction lines and frees registers.
template <int kT, class F>
__device__ __forceinline__ void window_tile(const VisitTarget& T, float* pick,
                                            const float* fp, const FpBox& dom, const StampGeom& g,
                                            const PStamp& st, bool dup, bool pull, int tile,
                                            const TileWin& win, float (*hand)[kT * kT],
                                            const float pk[3], const float ps[3],
                                            const DryClock& clk = DryClock{}) {
  const bool clocked = F::clock && clk.tmap != nullptr;
  const bool snap = F::snap(T.use_snap);
  const int t = threadIdx.x;
  const int lx = t % kT, ly = t / kT;
  const int tiles_x = (win.cols + kT - 1) / kT;
  const int ty = tile_row(tile, __builtin_amdgcn_rcpf((float)tiles_x));
  const int col = win.col0 + (tile - ty * tiles_x) * kT + lx;
  const int row = win.row0 + ty * kT + ly;
  const VisitCell V = visit_cell(g, dom, col, row);
  bool act = V.mm >= 0;
  const bool second = V.shared == 1 || V.shared == 2;  // runs after its neighbour
  const bool inside = V.shared == 1   ? lx > 0
                      : V.shared == 2 ? ly > 0
                      : V.shared == 3 ? lx < kT - 1
                                      : ly < kT - 1;
  const int dx = V.shared == 1 ? -1 : (V.shared == 3 ? 1 : 0);
  const int dy = V.shared == 2 ? -1 : (V.shared == 4 ? 1 : 0);
  if (F::dup && dup && act && (on_dup_line(st, col, row) ||
                     (V.shared && on_dup_line(st, col + dx, row + dy))))
    act = false;
  if (second && !inside) act = false;  // the neighbour's tile runs it
  const bool first = act && !second;
  float fh = 0.0f;
  const int64_t ic = (int64_t)V.y * g.cols + V.x;
  bool pv = false;
  CachedVisit<RegPick> acc;
  acc.alias = !snap;
  if (act) {
    pv = pull && on_window_border(st.box, V.x, V.y);
    fh = fp[V.mm];
    if (first) ld_cell(pick, V.mm, acc.v);
    load_pixel(T, snap, ic, pv, acc);
    if (clocked) {
      if (fh > 0.0f) {
        check_dry_regs(clk, acc.cv, acc.cvv, ic);
        if (!snap) acc.src_from_canvas();  // the pickup source is the canvas itself
      } else {
        check_only(T, clk, ic, pv);
      }
    }
  }
  const bool paint = act && fh > 0.0f;
  if (F::tape && paint) {
    tape_pixel(*T.tape, snap, V.x, V.y, acc.cv, acc.cvv, acc.sv, acc.svv);
    if (first) st_cell(T.tape->P, V.mm, acc.v);
  }
  if (paint && first) {
    paint_visit_math(acc, fh, T.pickup_rate, T.dep_rate, T.cap, pk, ps);
    if (V.shared && inside)
#pragma unroll
      for (int c = 0; c < 7; ++c) hand[c][t] = acc.v[c];
  }
  __syncthreads();
  if (paint && second) {
    const int from = t + dx + dy * kT;
#pragma unroll
    for (int c = 0; c < 7; ++c) acc.v[c] = hand[c][from];
    paint_visit_math(acc, fh, T.pickup_rate, T.dep_rate, T.cap, pk, ps);
  }
  if (paint) {
    store_pixel(T, snap, ic, pv, acc);
    if (second || !V.shared) st_cell(pick, V.mm, acc.v);
  }
  if (first && V.shared && !inside) {  // the second visit lies in another tile
    const int px = (int)(col + dx + g.cx), py = (int)(row + dy + g.cy);
    const int64_t pic = (int64_t)py * g.cols + px;
    const bool ppv = pull && on_window_border(st.box, px, py);
    if (paint) {
      load_pixel(T, snap, pic, ppv, acc);
      if (clocked) {
        check_dry_regs(clk, acc.cv, acc.cvv, pic);
        if (!snap) acc.src_from_canvas();
      }
      if (F::tape) tape_pixel(*T.tape, snap, px, py, acc.cv, acc.cvv, acc.sv, acc.svv);
      paint_visit_math(acc, fh, T.pickup_rate, T.dep_rate, T.cap, pk, ps);
      store_pixel(T, snap, pic, ppv, acc);
      st_cell(pick, V.mm, acc.v);
    } else if (clocked) {
      check_only(T, clk, pic, ppv);
    }
  }
  __syncthreads();  // hand is rewritten by the block's next tile
}

// Is visit (col, row), at canvas pixel ic on the window border of box b,
// the first visit of that pixel in reference order (rows, then columns)
// that acts: footprint height > 0, or any visit when `any_visit` (a drying
// clock)?  Only a pixel of a duplicated column/row 0 has more than one.
__device__ __forceinline__ bool first_acting_visit(const StampGeom& g, const RingBox& b,
                                                   const float* fp, int col, int row, int64_t ic,
                                                   bool any_visit) {
  const int x = (int)(ic % g.cols), y = (int)(ic / g.cols);
  if (!on_window_border(b, x, y)) return false;
  int cs[2], rs[2];
  const int nc = window_offsets(x, g.cx, g.hr, cs), nr = window_offsets(y, g.cy, g.hr, rs);
  for (int r = 0; r < nr; ++r)
    for (int c = 0; c < nc; ++c) {
      int64_t i2;
      const int m = stamp_visit(g, cs[c], rs[r], &i2);
      if (m >= 0 && (any_visit || fp[m] > 0.0f)) return cs[c] == col && rs[r] == row;
    }
  return false;
}

// Visits sharing a canvas pixel on column/row 0 (and their map-cell
// partners), listed in reference order and grouped by dependency level; the
// threads of one workgroup, levels separated by barriers.  With a clock,
// each listed visit first checks its pixel (the second check of a pixel in
// one imprint finds its time already at the imprint's and changes nothing).
//
// With `pull` (the stamp's window tiles and ring scan run in the same
// launch), a listed visit on the window border refreshes its own snapshot
// pixel when it is the first visit of that pixel that acts (footprint
// height > 0, or any visit with a clock) in reference order; the ring scan
// leaves such pixels alone.
//
// The block is one chain of levels (3, rarely 4) beside tiles that take one
// round trip each, so what a level needs besides the pixels and cells is
// fetched for all levels first: the list entries, their geometry and
// footprint heights.  A level is then one round trip (17 us to 14.5 us of the
// launches that hold such a stamp).  Starting the block first gave 0 to 2 %.
template <int kThreads>
__device__ __forceinline__ void level_visits(const VisitTarget& T, float* pick,
                                             const float* fp, const StampGeom& g, const PStamp& st,
                                             const int2* dl, const int* dl_off, const float pk[3],
                                             const float ps[3],
                                             const DryClock& clk = DryClock{},
                                             bool pull = false) {
  const bool clocked = clk.tmap != nullptr;
  const int nlev = st.dl_nlev;
  const int* off = dl_off + st.dl_lev;
  struct Entry {
    int m;  // map cell, -1: none
    float fh;
    int64_t ic;
    bool pv;
  };
  const auto fetch = [&](int e) {
    const int2 v = dl[e];
    Entry E;
    E.m = stamp_visit(g, v.x, v.y, &E.ic);
    E.fh = 0.0f;
    E.pv = false;
    if (E.m >= 0) {
      E.fh = fp[E.m];
      E.pv = pull && first_acting_visit(g, st.box, fp, v.x, v.y, E.ic, clocked);
    }
    return E;
  };
  const auto visit = [&](const Entry& E) {
    if (E.m < 0) return;
    if (clocked) check_only(T, clk, E.ic, E.pv);  // with pv, the refresh comes first
    if (E.fh > 0.0f) cached_visit(T, pick, E.m, E.fh, E.ic, E.pv && !clocked, pk, ps);
  };
  constexpr int kPre = 4;
  Entry pre[kPre];
#pragma unroll
  for (int L = 0; L < kPre; ++L) {
    pre[L].m = -1;
    if (L < nlev && off[L] + (int)threadIdx.x < off[L + 1]) pre[L] = fetch(off[L] + (int)threadIdx.x);
  }
#pragma unroll
  for (int L = 0; L < kPre; ++L) {
    if (L >= nlev) break;
    visit(pre[L]);
    for (int e = off[L] + kThreads + (int)threadIdx.x; e < off[L + 1]; e += kThreads) visit(fetch(e));
    __builtin_amdgcn_s_waitcnt(0);  // this level's stores before the next level's loads
    __syncthreads();
  }
  for (int L = kPre; L < nlev; ++L) {
    for (int e = off[L] + (int)threadIdx.x; e < off[L + 1]; e += kThreads) visit(fetch(e));
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
}

// What the stamps of a launch may need.
//   clock  Canvas::checkDry on every visited pixel
//   dup    stamps that straddle canvas column/row 0 (shared-pixel levels)
//   kSnap  the snapshot buffer: 0 off, 1 on, 2 per stamp
//   tape   every visit's input is kept (VisitTarget::tape)
//   whole  no dirty bytes are kept: the ring is copied whole
template <bool kClock, bool kDup, int kSnap, bool kTape = false, bool kWhole = false>
struct StampKind {
  static constexpr bool clock = kClock, dup = kDup, tape = kTape, whole = kWhole;
  static __device__ __forceinline__ bool snap(int use_snap) {
    return kSnap == 2 ? use_snap != 0 : kSnap == 1;
  }
};

// What a stamp's block keeps in LDS: cells handed from a tile's first to its
// second visits, or the groups of a ring pass.
template <int kThreads>
union StampLds {
  float hand[7][kThreads];
  RingList<kThreads> ring;
};

// Block b of one imprint whose window tiles, ring scan and shared-pixel
// levels run side by side: blocks [0, ntiles) take a 16 x 16 window tile
// each, the next rb scan the snapshot ring, and one more runs the levels of
// a stamp that has them.  Visits on the window border refresh their own
// snapshot pixels (the ring scan leaves them).
template <class F>
__device__ __forceinline__ void stamp_block(const VisitTarget& T, float* pick,
                                            const float* fp, const FpBox& dom, const StampGeom& g,
                                            const PStamp& st, const TileWin& win, int ntiles, int rb,
                                            int b, StampLds<256>& lds, const int2* dl,
                                            const int* dl_off, const float pk[3],
                                            const float ps[3], const DryClock& clk) {
  const bool dup = F::dup && (st.flags & (kStDupX | kStDupY)) != 0;
  const bool pull = F::snap(T.use_snap);
  if (b < ntiles) {
    window_tile<16, F>(T, pick, fp, dom, g, st, dup, pull, tile_of_block(b, ntiles), win, lds.hand, pk,
                       ps, clk);
  } else if (b < ntiles + rb) {
    if (F::whole)
      ring_copy<256>(*T.canvas, *T.src, fp, g, st.box, b - ntiles, rb,
                     F::clock && clk.tmap != nullptr);
    else
      ring_scan<256>(*T.canvas, *T.src, T.dirty, fp, g, st.box, pull, b - ntiles, rb, lds.ring,
                     F::clock && clk.tmap != nullptr);
  } else if (F::dup && dup) {
    if (F::tape) {  // the pixels and cells the levels start from
      const bool snap = F::snap(T.use_snap);
      for (int e = dl_off[st.dl_lev] + (int)threadIdx.x; e < dl_off[st.dl_lev + st.dl_nlev]; e += 256) {
        const int2 v = dl[e];
        int64_t ic;
        const int m = stamp_visit(g, v.x, v.y, &ic);
        if (m < 0 || !(fp[m] > 0.0f)) continue;
        const int x = (int)(ic % g.cols), y = (int)(ic / g.cols);
        CachedVisit<RegPick> acc;
        load_pixel(T, snap, ic, pull && on_window_border(st.box, x, y), acc);
        tape_pixel(*T.tape, snap, x, y, acc.cv, acc.cvv, acc.sv, acc.svv);
        ld_cell(pick, m, acc.v);
        st_cell(T.tape->P, m, acc.v);
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
    level_visits<256>(T, pick, fp, g, st, dl, dl_off, pk, ps, F::clock ? clk : DryClock{}, pull);
  }
}

// ------------------------------------------------------------- host side --
// Plans stamps [0, n) of one list for brush b on canvas cv into h_st
// (appended), with the shared-pixel visit lists of dup stamps appended to
// h_dl / h_off (offsets are global indices into h_dl).
void plan_stamps(pnt_brush b, pnt_canvas cv, const pnt_stamp* st, int64_t n,
                 std::vector<PStamp>& h_st, std::vector<int2>& h_dl, std::vector<int>& h_off);
// The same for a brush geometry given explicitly (padded footprint side and
// radius), so that a list can change geometry between strokes.
void plan_stamps_geom(int size_map, double radius, pnt_canvas cv, const pnt_stamp* st, int64_t n,
                      std::vector<PStamp>& h_st, std::vector<int2>& h_dl, std::vector<int>& h_off);

}  // namespace pnt
