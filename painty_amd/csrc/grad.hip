// Differentiable composite + stamping: gradients of a loss on the composite
// R = Renderer::compose (Renderer.hxx:26-41) of a canvas after a stamp list
// (FootprintBrush::imprint, FootprintBrush.hxx:73-143, with each dip's paint
// from PaintMixer::mixSinglePaint, PaintMixer.cxx:327-355) with respect to
// the initial wet layer K, S, V, the substrate R0 and the mixing weights.
// The reference has no gradients; this is the extension it is measured on.
//
// Forward: the stamps run as PNT_EXEC_FUSED (waves of independent strokes),
// each visit leaving what it found -- its map cell, canvas pixel and pickup
// source -- on a tape, one record per stamp (TapeRec, stampcore.hpp).
//
// Backward: the waves again, in reverse, one launch each (k_adj_wave): the
// stamps of a wave touch disjoint pixels and maps, so their adjoints run side
// by side as they did.  Per stamp
//   tiles    each cell's visits replayed from the tape (the forward
//            arithmetic of visit.hpp, so branches resolve the same way) and
//            their adjoints applied in reverse order;
//   ring     the snapshot refresh's adjoint: the snapshot's adjoint of a ring
//            pixel moves onto the canvas', found by dirty bytes; a window
//            border pixel with a visit is moved by that visit;
//   levels   visits on a duplicated canvas column/row 0, replayed on the tape
//            and reversed level by level;
// and where the pickup map was cleared its adjoint is dropped.
//
// The tapes of a whole list may take kTapeFree of the free device memory (0.8
// MB per stamp at radius 32).  A longer list keeps checkpoints instead: it is
// cut into segments of at most `seg_len` stamps that never cross a dip, the
// canvas and snapshot inside a segment's snapshot boxes and the pickup map are
// saved before it, and backward restores and reruns the segment onto its tape.
//
// Bound: the chain of launches, one per wave (108 for 500 stamps on 2048^2),
// each as long as one tile's round trips and FP64 arithmetic.  500
// stamps of radius 32 on 2048^2, forward and backward: 30.3 ms with every
// segment recomputed stamp by stamp (six launches and 48 us a stamp in the
// backward, one stroke at a time), 3.9 ms from a tape in planes, 3.3 ms with a
// tape's pixels and cells each in one piece, every load of a thread's visits
// issued before the first one's arithmetic, and the ring's pixels moved one a
// thread.
#include <algorithm>
#include <initializer_list>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>

#include "handles.hpp"
#include "internal.hpp"
#include "km.hpp"
#include "persistent.hpp"
#include "stampcore.hpp"

namespace pnt {

namespace {

constexpr int kGT = 16;  // window tile of the adjoint kernel
constexpr int kBlk = 256;
constexpr int kAdjSlots = kWaveSlots;  // stamps of one adjoint launch (a wave of the forward)
constexpr int64_t kTapeFree = 8;      // tapes take at most 1/8 of the free memory,
constexpr int64_t kTapeMost = 16ll << 30;  // and 16 GiB

// ------------------------------------------------------ visit adjoint ----
struct VState {
  float P[7];          // pickup cell (FP32, as stored)
  double C[7], X[7];   // canvas and source pixel (K, S from FP32; V is FP64)
};

// Adjoint of paint_visit_math (visit.hpp) at input state `in`.  On entry g
// holds the adjoints of the outputs (P, C and, with the snapshot, X); on
// return the adjoints of the inputs.  gB accumulates the adjoint of the
// brush paint.  The intermediates are recomputed with the forward's own
// operations (FP64 on the stored FP32 values), so every threshold branch is
// the one the forward took.
__device__ __forceinline__ void visit_adj(const VState& in, VState& g, float gB[6], float fh_f,
                                          double pr, double dr, double cap, const float pk[3],
                                          const float ps[3], bool alias) {
  const double fh = fh_f;
  const double B[6] = {pk[0], pk[1], pk[2], ps[0], ps[1], ps[2]};
  const float* Pf = in.P;
  const double* Cf = in.C;
  const double* Xf = alias ? in.C : in.X;
  double P[7], C[7], X[7];
#pragma unroll
  for (int c = 0; c < 7; ++c) {
    P[c] = Pf[c];
    C[c] = Cf[c];
    X[c] = Xf[c];
  }
  const double vP = P[6], vC = X[6];
  const double vLeave = (pr * vC) * fh;
  const bool a = vLeave > kMinVolume;
  double P1[7];
#pragma unroll
  for (int c = 0; c < 7; ++c) P1[c] = P[c];
  double X6n = vC, iv1 = 0.0;
  bool bb = false;
  if (a) {
    X6n = vC - vLeave;  // the stored source volume (FP64)
    const double vt1 = vP + vLeave;
    bb = vt1 > kMinVolume;
    if (bb) {
      iv1 = rcpd(vt1);
#pragma unroll
      for (int c = 0; c < 6; ++c)
        P1[c] = (float)__builtin_fma(vP * iv1, P[c], (vLeave * iv1) * X[c]);
    }
    P1[6] = (float)(vP + vLeave);
  }
  const double u = P1[6];
  const bool f = cap - u > 0.0;
  const double vFree = fmax(0.0, cap - u);
  const double vt2 = u + vFree;
  const bool d = vt2 > kMinVolume;
  const double iv2 = d ? rcpd(vt2) : 0.0;
  double src[6];
#pragma unroll
  for (int c = 0; c < 6; ++c)
    src[c] = d ? __builtin_fma(u * iv2, P1[c], (vFree * iv2) * B[c]) : P1[c];
  double Cd[7];  // the canvas pixel as depositPaint reads it
#pragma unroll
  for (int c = 0; c < 6; ++c) Cd[c] = C[c];
  Cd[6] = alias ? X6n : C[6];
  const double vB = cap * fh, vCc = Cd[6], vt3 = vB + vCc;
  const bool e = vt3 > kMinVolume;
  const double iv3 = e ? rcpd(vt3) : 0.0;
  // ---- depositPaint
  double gCd[7], gsrc[6];
  double gvCc = g.C[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    if (e) {
      const double C1 = __builtin_fma(vB * iv3, src[c], (vCc * iv3) * Cd[c]);
      gsrc[c] = g.C[c] * (vB * iv3);
      gCd[c] = g.C[c] * (vCc * iv3);
      gvCc += g.C[c] * (Cd[c] - C1) * iv3;
    } else {
      gsrc[c] = g.C[c];
      gCd[c] = 0.0;
    }
  }
  gCd[6] = gvCc;
  double gP1[7];
  double gu = g.P[6] * (1.0 - dr * fh);
  if (d) {
    double gvFree = 0.0;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      gP1[c] = g.P[c] + gsrc[c] * (u * iv2);
      gB[c] += (float)(gsrc[c] * (vFree * iv2));
      gu += gsrc[c] * (P1[c] - src[c]) * iv2;
      gvFree += gsrc[c] * (B[c] - src[c]) * iv2;
    }
    if (f) gu -= gvFree;
  } else {
#pragma unroll
    for (int c = 0; c < 6; ++c) gP1[c] = g.P[c] + gsrc[c];
  }
  gP1[6] = gu;
  // ---- pickupPaint
  double gXo[7];
#pragma unroll
  for (int c = 0; c < 7; ++c) gXo[c] = alias ? gCd[c] : g.X[c];
  double gPin[7], gXin[7];
#pragma unroll
  for (int c = 0; c < 7; ++c) gXin[c] = gXo[c];
  if (a) {
    double gvP = gP1[6], gvLeave = gP1[6] - gXo[6], gvC = gXo[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      if (bb) {
        gPin[c] = gP1[c] * (vP * iv1);
        gXin[c] += gP1[c] * (vLeave * iv1);
        gvP += gP1[c] * (P[c] - P1[c]) * iv1;
        gvLeave += gP1[c] * (X[c] - P1[c]) * iv1;
      } else {
        gPin[c] = gP1[c];
      }
    }
    gvC += gvLeave * pr * fh;
    gPin[6] = gvP;
    gXin[6] = gvC;
  } else {
#pragma unroll
    for (int c = 0; c < 7; ++c) gPin[c] = gP1[c];
  }
#pragma unroll
  for (int c = 0; c < 7; ++c) {
    g.P[c] = (float)gPin[c];
    g.C[c] = alias ? gXin[c] : gCd[c];
    g.X[c] = alias ? 0.0 : gXin[c];
  }
}

// The forward visit on a state held in registers (the same instructions as
// every stamp kernel).
__device__ __forceinline__ void visit_fwd(VState& s, float fh, double pr, double dr, double cap,
                                          const float pk[3], const float ps[3], bool alias) {
  CachedVisit<RegPick> acc;
#pragma unroll
  for (int c = 0; c < 7; ++c) acc.v[c] = s.P[c];
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    acc.cv[c] = (float)s.C[c];
    acc.sv[c] = (float)(alias ? s.C[c] : s.X[c]);
  }
  acc.cvv = s.C[6];
  acc.svv = alias ? s.C[6] : s.X[6];
  acc.alias = alias;
  acc.src_moved = false;
  paint_visit_math(acc, fh, pr, dr, cap, pk, ps);
#pragma unroll
  for (int c = 0; c < 7; ++c) s.P[c] = acc.v[c];
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    s.C[c] = acc.cv[c];
    s.X[c] = alias ? acc.cv[c] : acc.sv[c];
  }
  s.C[6] = acc.cvv;
  s.X[6] = alias ? acc.cvv : acc.svv;
}

// One phase of an adjoint launch: a stamp, or the clear of a map's adjoint
// (the pickup map was cleared there).
struct ASlot {
  int nblk, clear, ntiles, rb;
  float* tape;     // the stamp's tape record
  float* gP;       // its chain's pickup-map adjoint, m cells
  float* gB;       // 6 floats: the stamp's paint adjoint
  float* scratch;  // records of the shared-pixel replay
  TileWin win;
  float pk[3], ps[3];
  PStamp st;
};

struct AShared {
  const float* fp;
  FpBox dom;
  int size_map, rows, cols, use_snap;
  int64_t area, m;
  Plane7 gC, gX;        // adjoints: canvas (caller's planes), snapshot
  uint8_t* dirty;       // 0: the pixel's snapshot adjoint is zero
  const int2* dl;       // shared-pixel visits (plan lists)
  const int* dl_off;
  double pr, dr, cap;
};

struct AArgs {
  AShared sh;
  ASlot slot[kAdjSlots];
};
static_assert(sizeof(AArgs) <= 4000, "kernel arguments must fit the argument segment");

__device__ __forceinline__ void load_px(const TapeRec& t, bool snap, int64_t k, VState& s) {
  const TapePx c = t.c[k], x = snap ? t.x[k] : TapePx{};
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    s.C[i] = c.ks[i];
    s.X[i] = x.ks[i];
  }
  s.C[6] = c.v;
  s.X[6] = x.v;
}

__device__ __forceinline__ void load_in(const TapeRec& t, bool snap, int64_t k, int mm, VState& s) {
  ld_cell(t.P, mm, s.P);
  load_px(t, snap, k, s);
}

__device__ __forceinline__ void store_in(const TapeRec& t, bool snap, int64_t k, int mm,
                                         const VState& s) {
  st_cell(t.P, mm, s.P);
  TapePx p;
#pragma unroll
  for (int i = 0; i < 6; ++i) p.ks[i] = (float)s.C[i];
  p.v = s.C[6];
  t.c[k] = p;
  if (!snap) return;
#pragma unroll
  for (int i = 0; i < 6; ++i) p.ks[i] = (float)s.X[i];
  p.v = s.X[6];
  t.x[k] = p;
}

__device__ __forceinline__ void load_g_pixel(const AShared& A, int64_t ic, VState& g) {
#pragma unroll
  for (int c = 0; c < 7; ++c) {
    g.C[c] = A.gC.p[c][ic];
    g.X[c] = A.use_snap ? A.gX.p[c][ic] : 0.0f;
  }
}

// `moved`: the stamp's ring refresh copied this pixel before its visits, so
// the snapshot's adjoint goes on to the canvas.
__device__ __forceinline__ void store_g_pixel(const AShared& A, int64_t ic, const VState& g,
                                              bool moved) {
#pragma unroll
  for (int c = 0; c < 7; ++c) {
    const float gc = (float)g.C[c], gx = (float)g.X[c];
    A.gC.p[c][ic] = moved ? gc + gx : gc;
    if (A.use_snap) A.gX.p[c][ic] = moved ? 0.0f : gx;
  }
  if (A.use_snap) A.dirty[ic] = moved ? 0 : 1;
}

// Adds the block's paint adjoints to out[6]: summed over each wave by
// shuffles, over its waves in LDS, one atomic per value and block.
__device__ __forceinline__ void flush_gB(float* out, const float gB[6]) {
  __shared__ float s_gB[kBlk / 64][6];
  float v[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    v[c] = gB[c];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v[c] += __shfl_xor(v[c], d);
  }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int c = 0; c < 6; ++c) s_gB[threadIdx.x >> 6][c] = v[c];
  __syncthreads();
  if (threadIdx.x < 6) {
    float t = 0.0f;
    for (int w = 0; w < kBlk / 64; ++w) t += s_gB[w][threadIdx.x];
    if (t != 0.0f) atomicAdd(&out[threadIdx.x], t);
  }
}

// Adjoint of the visits of one kGT x kGT window tile that do not share a
// canvas pixel; a cell's first visitor runs both its visits' adjoints.
__device__ __forceinline__ void adj_tile(const AShared& A, const ASlot& S, const StampGeom& g,
                                         const TapeRec& tape, bool dup, int tile) {
  const int t = threadIdx.x, lx = t % kGT, ly = t / kGT;
  const int tiles_x = (S.win.cols + kGT - 1) / kGT;
  const int col = S.win.col0 + (tile % tiles_x) * kGT + lx;
  const int row = S.win.row0 + (tile / tiles_x) * kGT + ly;
  float gB[6] = {0, 0, 0, 0, 0, 0};
  const VisitCell V = visit_cell(g, A.dom, col, row);
  const int dx = V.shared == 3 ? 1 : 0, dy = V.shared == 4 ? 1 : 0;
  const bool two = V.shared >= 3;
  bool act = V.mm >= 0 && V.shared != 1 && V.shared != 2;
  if (dup && act && (on_dup_line(S.st, col, row) || (two && on_dup_line(S.st, col + dx, row + dy))))
    act = false;
  const float fh = act ? A.fp[V.mm] : 0.0f;
  if (fh > 0.0f) {
    const bool snap = A.use_snap != 0, alias = !snap;
    const int64_t ic1 = (int64_t)V.y * A.cols + V.x;
    // everything the visits read, in one round trip
    VState in1, gs;
    load_in(tape, snap, tape.at(V.x, V.y), V.mm, in1);
    ld_cell(S.gP, V.mm, gs.P);
    load_g_pixel(A, ic1, gs);
    if (two) {
      const int x2 = (int)(col + dx + g.cx), y2 = (int)(row + dy + g.cy);
      const int64_t ic2 = (int64_t)y2 * A.cols + x2;
      VState at2, g2;
      load_px(tape, snap, tape.at(x2, y2), at2);
      load_g_pixel(A, ic2, g2);
      VState in2 = in1;
      visit_fwd(in2, fh, A.pr, A.dr, A.cap, S.pk, S.ps, alias);  // pickup cell after visit 1
#pragma unroll
      for (int c = 0; c < 7; ++c) {
        at2.P[c] = in2.P[c];
        g2.P[c] = gs.P[c];
      }
      visit_adj(at2, g2, gB, fh, A.pr, A.dr, A.cap, S.pk, S.ps, alias);
      store_g_pixel(A, ic2, g2, snap && on_window_border(S.st.box, x2, y2));
#pragma unroll
      for (int c = 0; c < 7; ++c) gs.P[c] = g2.P[c];
    }
    visit_adj(in1, gs, gB, fh, A.pr, A.dr, A.cap, S.pk, S.ps, alias);
    store_g_pixel(A, ic1, gs, snap && on_window_border(S.st.box, V.x, V.y));
    st_cell(S.gP, V.mm, gs.P);
  }
  flush_gB(S.gB, gB);
}

// Adjoint of the ring copy canvas -> snapshot (FootprintBrush.hxx:307-318) by
// block `blk` of S.rb: the pixels of the allowed box, outside the window
// interior, whose snapshot adjoint may be nonzero (dirty bytes, read eight at
// a time) and that no visit of the stamp moves itself.  The pixels found are
// listed in LDS and moved one a thread: a thread that moved its own eight one
// after another took eight round trips, longer than any tile.
__device__ __forceinline__ void adj_ring(const AShared& A, const ASlot& S, const StampGeom& g,
                                         int blk) {
  const RingBox& b = S.st.box;
  const int span = b.a_x1 - b.a_x0 + 1;
  const int per_row = (span + kRingUnit - 1) / kRingUnit + 1;
  const int total = per_row * (b.a_y1 - b.a_y0 + 1);
  __shared__ int s_n, s_list[kRingUnit * kBlk];  // e * kRingUnit + q
  for (int e0 = blk * kBlk; e0 < total; e0 += S.rb * kBlk) {
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    const int e = e0 + (int)threadIdx.x, r = e / per_row, row = b.a_y0 + r;
    const int64_t rowi = (int64_t)row * A.cols, lo = rowi + b.a_x0;
    const int64_t base = (lo & ~(int64_t)(kRingUnit - 1)) + kRingUnit * (int64_t)(e - r * per_row);
    const int x0 = (int)(base - rowi);
    const bool interior_row = row > b.tl_y && row < b.br_y;
    if (e < total && x0 <= b.a_x1 &&
        !(interior_row && x0 > b.tl_x && x0 + kRingUnit - 1 < b.br_x)) {
      const uint2 d = *reinterpret_cast<const uint2*>(A.dirty + base);
      if (d.x | d.y)
        for (int q = 0; q < kRingUnit; ++q) {
          if (!((((q < 4 ? d.x : d.y) >> (8 * (q & 3)))) & 0xffu)) continue;
          const int col = x0 + q;
          if (col < b.a_x0 || col > b.a_x1) continue;
          if (interior_row && col > b.tl_x && col < b.br_x) continue;
          s_list[atomicAdd(&s_n, 1)] = e * kRingUnit + q;
        }
    }
    __syncthreads();
    for (int j = (int)threadIdx.x; j < s_n; j += kBlk) {
      const int id = s_list[j], e2 = id / kRingUnit, r2 = e2 / per_row, y = b.a_y0 + r2;
      const int64_t rowj = (int64_t)y * A.cols, lo2 = rowj + b.a_x0;
      const int64_t i = (lo2 & ~(int64_t)(kRingUnit - 1)) +
                        kRingUnit * (int64_t)(e2 - r2 * per_row) + id % kRingUnit;
      const int x2 = (int)(i - rowj);
      if (on_window_border(b, x2, y) && ring_pixel_visited(g, b, A.fp, x2, y)) continue;
      float c[7], x[7];
#pragma unroll
      for (int k = 0; k < 7; ++k) {
        c[k] = A.gC.p[k][i];
        x[k] = A.gX.p[k][i];
      }
#pragma unroll
      for (int k = 0; k < 7; ++k) {
        A.gC.p[k][i] = c[k] + x[k];
        A.gX.p[k][i] = 0.0f;
      }
      A.dirty[i] = 0;
    }
    __syncthreads();  // the list is rewritten by the next pass
  }
}

// Adjoint of a stamp's visits on a duplicated canvas column/row 0 and their
// partners.  Only these visits touch those pixels and cells, so the tape
// holds their true starting state, and the replay runs on it in place: visits
// level by level (a level's visits share no map cell and no canvas pixel, so
// each level runs in parallel), each visit's input recorded; then the adjoints
// level by level in reverse, each putting its input back on the tape.
// The first visit of a border pixel that acts moves its snapshot adjoint.
__device__ __forceinline__ void adj_levels(const AShared& A, const ASlot& S, const StampGeom& g,
                                           const TapeRec& t) {
  const PStamp& st = S.st;
  const int base = A.dl_off[st.dl_lev];
  VState* rec = reinterpret_cast<VState*>(S.scratch);
  const bool snap = A.use_snap != 0, alias = !snap;
  for (int L = 0; L < st.dl_nlev; ++L) {  // replay in plan order, a level at a time
    const int e0 = A.dl_off[st.dl_lev + L], e1 = A.dl_off[st.dl_lev + L + 1];
    for (int e = e0 + (int)threadIdx.x; e < e1; e += kBlk) {
      const int2 v = A.dl[e];
      int64_t ic;
      const int mm = stamp_visit(g, v.x, v.y, &ic);
      if (mm < 0 || !(A.fp[mm] > 0.0f)) continue;
      const int64_t k = t.at((int)(ic % A.cols), (int)(ic / A.cols));
      VState sv;
      load_in(t, snap, k, mm, sv);
      rec[e - base] = sv;
      visit_fwd(sv, A.fp[mm], A.pr, A.dr, A.cap, S.pk, S.ps, alias);
      store_in(t, snap, k, mm, sv);
    }
    __builtin_amdgcn_s_waitcnt(0);  // this level's stores before the next level's loads
    __syncthreads();
  }
  float gB[6] = {0, 0, 0, 0, 0, 0};
  for (int L = st.dl_nlev - 1; L >= 0; --L) {  // adjoints, levels in reverse
    const int e0 = A.dl_off[st.dl_lev + L], e1 = A.dl_off[st.dl_lev + L + 1];
    for (int e = e0 + (int)threadIdx.x; e < e1; e += kBlk) {
      const int2 v = A.dl[e];
      int64_t ic;
      const int mm = stamp_visit(g, v.x, v.y, &ic);
      if (mm < 0 || !(A.fp[mm] > 0.0f)) continue;
      VState gs;
      ld_cell(S.gP, mm, gs.P);
      load_g_pixel(A, ic, gs);
      const VState in = rec[e - base];
      store_in(t, snap, t.at((int)(ic % A.cols), (int)(ic / A.cols)), mm, in);
      visit_adj(in, gs, gB, A.fp[mm], A.pr, A.dr, A.cap, S.pk, S.ps, alias);
      store_g_pixel(A, ic, gs, snap && first_acting_visit(g, st.box, A.fp, v.x, v.y, ic, false));
      st_cell(S.gP, mm, gs.P);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  flush_gB(S.gB, gB);
}

// One wave of the forward, reversed: slot y of the grid's rows.
template <bool kDup>
__global__ __launch_bounds__(kBlk) void k_adj_wave(AArgs A) {
  const ASlot& S = A.slot[blockIdx.y];
  const int b = (int)blockIdx.x;
  if (b >= S.nblk) return;
  if (S.clear) {
    for (int64_t i = (int64_t)b * kBlk + threadIdx.x; i < kCell * A.sh.m; i += (int64_t)S.nblk * kBlk)
      S.gP[i] = 0.0f;
    return;
  }
  const StampGeom g = stamp_geom(S.st, A.sh.size_map, A.sh.rows, A.sh.cols);
  const TapeRec tape = tape_rec(S.tape, A.sh.area, A.sh.m, S.st.box, A.sh.cols);
  const bool dup = kDup && (S.st.flags & (kStDupX | kStDupY)) != 0;
  if (b < S.ntiles)
    adj_tile(A.sh, S, g, tape, dup, b);
  else if (b < S.ntiles + S.rb)
    adj_ring(A.sh, S, g, b - S.ntiles);
  else if (dup)
    adj_levels(A.sh, S, g, tape);
}

// Adjoint of the first imprint's full canvas -> snapshot copy, where the
// snapshot's adjoint may be nonzero; it ends all zero, and so do the dirty
// bytes (the next backward starts from that).  A thread takes eight pixels.
__global__ __launch_bounds__(kBlk) void k_adj_full_copy(int64_t n, Plane7 gC, Plane7 gX,
                                                        uint8_t* dirty) {
  const int64_t units = (n + 7) / 8;
  for (int64_t u = (int64_t)blockIdx.x * kBlk + threadIdx.x; u < units; u += (int64_t)gridDim.x * kBlk) {
    const uint2 d = reinterpret_cast<const uint2*>(dirty)[u];
    if (!(d.x | d.y)) continue;
    for (int64_t i = 8 * u; i < 8 * u + 8 && i < n; ++i)
      if (dirty[i])
#pragma unroll
        for (int c = 0; c < 7; ++c) {
          gC.p[c][i] += gX.p[c][i];
          gX.p[c][i] = 0.0f;
        }
    reinterpret_cast<uint2*>(dirty)[u] = make_uint2(0u, 0u);
  }
}

// Adjoint of ComputeReflectance (KubelkaMunk.hxx:25-83) in the stable form
// of km.hpp, with Q = S*b*coth(x) = B (1 + 2/E), N = S - R0 (A - Q),
// D = A - R0 S + Q, R = N/D, x = B d.  The numerators are expanded so that
// the terms in Q (~ 1/d for thin layers) cancel symbolically, not in FP32:
//   dR/dR0 = (N S - (A-Q) D)/D^2 = B^2 csch^2 x / D^2
//   dR/dA  = -(R0 D + N)/D^2     = -(S (1 - R0^2) + 2 R0 Q)/D^2
//   dR/dQ  = (R0 D - N)/D^2      = (2 R0 A - R0^2 S - S)/D^2
//   dR/dS|direct = (D + R0 N)/D^2 = (A (1 - R0^2) + Q (1 + R0^2))/D^2
//   dQ/dB = coth x - x csch^2 x = d/dx (x coth x), by its Taylor series
//           2x/3 - 4x^3/45 + 12x^5/945 - 8x^7/4725 + 20x^9/93555 below x = 0.5
//   dQ/dd = -B^2 csch^2 x,  coth x = 1 + 2/E,  csch^2 x = 4(E+1)/E^2,
//   dB/dK = A/B,  dB/dS = K/B.
// Where x > 20 the reference's coth is the constant 1 (csch^2 -> 0).
__device__ __forceinline__ void km_adj_channel(float K, float Sin, float R0, float d, float gR,
                                               float* gK, float* gS, float* gd, float* gR0) {
  const bool clamp = !(__builtin_fabsf(Sin) > kKmThr);
  const float S = clamp ? kSClamp : Sin;
  const float A = S + K;
  const float q = K * (K + 2.0f * S);
  const float B = __builtin_amdgcn_sqrtf(q > 0.0f ? q : 0.0f);
  const float x = B * d;
  float y = 2.0f * x;
  const bool flat = y >= 40.0f;
  y = flat ? 40.0f : y;
  const float E = km_expm1(y);
  const float iE = rcpf(E);
  const float ct = 1.0f + 2.0f * iE;
  const float csch2 = flat ? 0.0f : 4.0f * (E + 1.0f) * iE * iE;
  const float Q = B * ct;
  const float D = A - R0 * S + Q;
  const float iD2 = rcpf(D * D);
  const float R02 = R0 * R0;
  const float dR0 = (B * B * csch2) * iD2;
  const float dA = -(S * (1.0f - R02) + 2.0f * R0 * Q) * iD2;
  const float dQ = (2.0f * R0 * A - R02 * S - S) * iD2;
  const float dSd = (A * (1.0f - R02) + Q * (1.0f + R02)) * iD2;
  const float x2 = x * x;
  const float series =
      x * (2.0f / 3.0f +
           x2 * (-4.0f / 45.0f + x2 * (12.0f / 945.0f + x2 * (-8.0f / 4725.0f + x2 * (20.0f / 93555.0f)))));
  const float dQdB = x < 0.5f ? series : ct - x * csch2;
  const float dQdd = -B * B * csch2;
  const float iB = B > 0.0f ? rcpf(B) : 0.0f;
  *gK = gR * (dA + dQ * dQdB * A * iB);
  *gS = clamp ? 0.0f : gR * (dSd + dA + dQ * dQdB * K * iB);
  *gd += gR * dQ * dQdd;
  *gR0 = gR * dR0;
}

__global__ __launch_bounds__(kBlk) void k_km_adj(int64_t n, Layer7 L, Rgb3 R0, Rgb3 gR, Plane7 gL,
                                                 Rgb3 gR0) {
  for (int64_t i = (int64_t)blockIdx.x * kBlk + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlk) {
    const float d = (float)L.v[i];
    float gd = 0.0f;
    if (__builtin_fabsf(d) < kKmThr) {  // R = R0
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        gL.p[c][i] = 0.0f;
        gL.p[3 + c][i] = 0.0f;
        gR0.p[c][i] = gR.p[c][i];
      }
    } else {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        float gk, gs, gr0;
        km_adj_channel(L.ks[c][i], L.ks[3 + c][i], R0.p[c][i], d, gR.p[c][i], &gk, &gs, &gd, &gr0);
        gL.p[c][i] = gk;
        gL.p[3 + c][i] = gs;
        gR0.p[c][i] = gr0;
      }
    }
    gL.p[6][i] = gd;
  }
}

// A w x h box at (x0, y0) of a layer's planes (row stride `cols`) <-> a
// dense buffer of 7 planes (plane stride `stride`): FP64 planes for a
// canvas or snapshot layer (K, S widened exactly, V as stored), FP32 planes
// for the pickup map's cells.  Up to three boxes per launch.
struct BoxRegion {
  Layer7 L;   // when layer
  float* P;   // otherwise: cells
  int layer;
  int cols, x0, y0, w, h;
  void* buf;  // double* (layer) or float*
  int64_t stride;
};

inline BoxRegion layer_box(const Layer7& L, int cols, int x0, int y0, int w, int h, double* buf,
                           int64_t stride) {
  BoxRegion r{};
  r.L = L;
  r.layer = 1;
  r.cols = cols;
  r.x0 = x0;
  r.y0 = y0;
  r.w = w;
  r.h = h;
  r.buf = buf;
  r.stride = stride;
  return r;
}

inline BoxRegion cell_box(float* P, int cols, int x0, int y0, int w, int h, float* buf,
                           int64_t stride) {
  BoxRegion r{};
  r.P = P;
  r.layer = 0;
  r.cols = cols;
  r.x0 = x0;
  r.y0 = y0;
  r.w = w;
  r.h = h;
  r.buf = buf;
  r.stride = stride;
  return r;
}

__global__ __launch_bounds__(kBlk) void k_box_copy(BoxRegion r0, BoxRegion r1, BoxRegion r2,
                                                   int64_t n0, int64_t n1, int64_t n2,
                                                   int to_buf) {
  const int64_t total = n0 + n1 + n2;
  for (int64_t t = (int64_t)blockIdx.x * kBlk + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * kBlk) {
    const BoxRegion& r = t < n0 ? r0 : (t < n0 + n1 ? r1 : r2);
    const int64_t e = t < n0 ? t : (t < n0 + n1 ? t - n0 : t - n0 - n1);
    const int64_t i = (int64_t)(r.y0 + e / r.w) * r.cols + (r.x0 + e % r.w);
    if (r.layer) {
      double* b = static_cast<double*>(r.buf);
      if (to_buf) {
#pragma unroll
        for (int c = 0; c < 6; ++c) b[c * r.stride + e] = r.L.ks[c][i];
        b[6 * r.stride + e] = r.L.v[i];
      } else {
#pragma unroll
        for (int c = 0; c < 6; ++c) r.L.ks[c][i] = (float)b[c * r.stride + e];
        r.L.v[i] = b[6 * r.stride + e];
      }
    } else {
      float* b = static_cast<float*>(r.buf);
#pragma unroll
      for (int c = 0; c < 7; ++c) {
        if (to_buf)
          b[c * r.stride + e] = r.P[kCell * i + c];
        else
          r.P[kCell * i + c] = b[c * r.stride + e];
      }
    }
  }
}

inline unsigned grid_for(int64_t n) {
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + kBlk - 1) / kBlk, 4096));
}

// Copies up to three boxes in one launch (boxes with w or h <= 0 are skipped).
void box_copy(std::initializer_list<BoxRegion> regions, bool to_buf, hipStream_t s) {
  BoxRegion r[3] = {};
  int64_t n[3] = {0, 0, 0};
  int k = 0;
  for (const BoxRegion& b : regions) {
    if (b.w <= 0 || b.h <= 0) continue;
    r[k] = b;
    n[k] = (int64_t)b.w * b.h;
    ++k;
  }
  const int64_t total = n[0] + n[1] + n[2];
  if (total == 0) return;
  for (int i = k; i < 3; ++i) r[i] = r[0];
  k_box_copy<<<grid_for(total), kBlk, 0, s>>>(r[0], r[1], r[2], n[0], n[1], n[2], to_buf ? 1 : 0);
  PNT_HIP_CHECK(hipGetLastError());
}

}  // namespace
}  // namespace pnt

// ===================================================================== host
using namespace pnt;

struct pnt_grad_s {
  pnt_ctx ctx = nullptr;
  pnt_brush b = nullptr;
  pnt_canvas cv = nullptr;  // owned working canvas
  int rows = 0, cols = 0;
  std::vector<pnt_stamp> st;
  std::vector<int> paint_of;
  int n_pig = 0, n_paint = 0;
  std::vector<double> palK, palS, W;
  int seg_len = 32;
  struct Seg {
    int s0, s1;
    int x0, y0, w, h;  // checkpoint box
    int64_t off;       // checkpoint offset (floats)
  };
  std::vector<Seg> segs;
  float* ckpt = nullptr;
  int64_t ckpt_cap = 0;
  float* tape = nullptr;
  int64_t tape_cap = 0;
  bool full_tape = false;  // the last forward taped the whole list
  bool canvas_final = false;  // cv is as the forward left it (segments rerun change it)
  TapeRun run;
  int2* dl = nullptr;      // the taped list's shared-pixel visits (the brush may plan again)
  int* dl_off = nullptr;
  int64_t dl_cap = 0, dl_off_cap = 0;
  // the brush as the forward found it: a backward is of that forward, whatever
  // rates or footprint the brush has been given since
  int fwd_size_map = 0;
  bool fwd_snap = false;
  uint64_t fwd_gen = 0;         // its geo_gen, for which fwd_fp was copied
  std::vector<float> fwd_fp;    // padded footprint
  double fwd_radius = 0.0, fwd_pr = 0.0, fwd_dr = 0.0, fwd_cap = 0.0;
  int fwd_fbox[4] = {0, 0, -1, -1};
  float* fp = nullptr;          // that footprint on the device, once the brush has another
  int64_t fp_cap = 0;
  float* gX = nullptr;  // 7 planes of round_up(n, 64) (snapshot adjoint)
  uint8_t* gdirty = nullptr;  // its dirty bytes
  bool adj_zero = false;  // both are zero: a backward that runs to its end leaves them so
  float* gP = nullptr;  // per chain of the waves: m cells (pickup adjoint)
  float* gB = nullptr;  // n_stamps x 6
  int64_t gX_cap = 0, gdirty_cap = 0, gP_cap = 0, gB_cap = 0;
  float* scratch = nullptr;
  int64_t scratch_cap = 0;
  bool have_forward = false;
  int64_t n_stride = 0, m = 0;
};

namespace pnt {
int guard_call(const std::function<void()>& f);  // api.hip: status + pnt_last_error
}

namespace {

// At least `need` elements at p; a failed allocation leaves none (cap 0).
template <class T>
void ensure(T*& p, int64_t& cap, int64_t need, hipStream_t s) {
  if (need <= cap) return;
  PNT_HIP_CHECK(hipStreamSynchronize(s));
  dev_free(p);
  p = nullptr;
  cap = 0;
  p = reinterpret_cast<T*>(dev_alloc((need * (int64_t)sizeof(T) + 3) / 4));
  cap = need;
}

Plane7 dense7(float* base, int64_t stride) {
  Plane7 L;
  for (int c = 0; c < 7; ++c) L.p[c] = base + c * stride;
  return L;
}

}  // namespace

static void check_status(int st) {
  if (st != PNT_OK) throw Error(st, pnt_last_error());
}

// The taped run's shared-pixel lists, copied on the brush's stream, behind the
// run and before the brush plans again; nothing else may be reading the lists
// kept before.
static void keep_lists(pnt_grad_s* g) {
  TapeRun& R = g->run;
  hipStream_t s = g->b->ctx->stream;
  if (R.n_dl == 0) return;
  ensure(g->dl, g->dl_cap, R.n_dl, s);
  ensure(g->dl_off, g->dl_off_cap, R.n_off, s);
  PNT_HIP_CHECK(hipMemcpyAsync(g->dl, R.dl, (size_t)R.n_dl * sizeof(int2), hipMemcpyDeviceToDevice, s));
  PNT_HIP_CHECK(hipMemcpyAsync(g->dl_off, R.dl_off, (size_t)R.n_off * sizeof(int),
                               hipMemcpyDeviceToDevice, s));
}

// The runner's brush with the values of the forward, for as long as this lives
// (its map side and snapshot switch are the same).
namespace {
struct BrushAsForward {
  pnt_grad_s* g;
  float* fp;
  double radius, pr, dr, cap;
  int fbox[4];
  explicit BrushAsForward(pnt_grad_s* g_) : g(g_) {
    pnt_brush b = g->b;
    hipStream_t s = b->ctx->stream;
    fp = b->fp;
    float* mine = b->fp;
    if (b->geo_gen != g->fwd_gen && b->fp_host != g->fwd_fp) {
      ensure(g->fp, g->fp_cap, b->m, s);
      PNT_HIP_CHECK(hipMemcpyAsync(g->fp, g->fwd_fp.data(), (size_t)b->m * sizeof(float),
                                   hipMemcpyHostToDevice, s));
      PNT_HIP_CHECK(hipStreamSynchronize(s));
      mine = g->fp;
    }
    radius = b->radius;
    pr = b->pickup_rate;
    dr = b->dep_rate;
    cap = b->cap;
    std::copy(b->fbox, b->fbox + 4, fbox);
    b->fp = mine;
    b->radius = g->fwd_radius;
    b->pickup_rate = g->fwd_pr;
    b->dep_rate = g->fwd_dr;
    b->cap = g->fwd_cap;
    std::copy(g->fwd_fbox, g->fwd_fbox + 4, b->fbox);
  }
  BrushAsForward(const BrushAsForward&) = delete;
  ~BrushAsForward() {
    pnt_brush b = g->b;
    b->fp = fp;
    b->radius = radius;
    b->pickup_rate = pr;
    b->dep_rate = dr;
    b->cap = cap;
    std::copy(fbox, fbox + 4, b->fbox);
  }
};
}  // namespace

// Segment sg again, from its checkpoint: canvas and snapshot in its box and the
// pickup map as before it, the brush paint of its last dip (stamp 0 dips), and
// its stamps, onto `tape` if given.  In list order over all segments this ends
// in the forward's final state.
static void rerun_segment(pnt_grad_s* g, const pnt_grad_s::Seg& sg, TapeRun* tape) {
  pnt_brush b = g->b;
  pnt_canvas cv = g->cv;
  hipStream_t s = g->ctx->stream;
  const int64_t area = (int64_t)sg.w * sg.h, m = b->m;
  const int sm = b->size_map;
  float* c0 = g->ckpt + sg.off;
  box_copy({layer_box(cv->layer(), cv->cols, sg.x0, sg.y0, sg.w, sg.h, reinterpret_cast<double*>(c0), area),
            layer_box(b->snap_planes(), cv->cols, sg.x0, sg.y0, b->use_snap ? sg.w : 0, sg.h,
                      reinterpret_cast<double*>(c0 + 14 * area), area),
            cell_box(b->pick, sm, 0, 0, sm, sm, c0 + (b->use_snap ? 28 : 14) * area, m)},
           false, s);
  cv->epoch++;
  b->dirty_canvas = nullptr;  // the snapshot's dirty bytes no longer hold
  int i = sg.s0;
  while (!(g->st[(size_t)i].flags & PNT_STAMP_DIP)) --i;
  for (int c = 0; c < 3; ++c) {
    b->paintK[c] = g->st[(size_t)i].K[c];
    b->paintS[c] = g->st[(size_t)i].S[c];
  }
  const bool other = b->ctx->stream != s;
  if (other) PNT_HIP_CHECK(hipStreamSynchronize(s));
  run_fused(b, cv, g->st.data() + sg.s0, sg.s1 - sg.s0, 0, tape);
  if (tape) keep_lists(g);
  if (other) PNT_HIP_CHECK(hipStreamSynchronize(b->ctx->stream));
}

// The adjoint of the taped run (stamps s0 .. of the list), its waves in
// reverse.  Every chain's map adjoint goes on from where it stands.
static void adjoint_waves(pnt_grad_s* g, int s0, const Plane7& gC, const Plane7& gX, hipStream_t s) {
  const TapeRun& R = g->run;
  pnt_brush b = g->b;
  AArgs A{};
  A.sh.fp = b->fp;
  A.sh.dom = FpBox{b->fbox[0], b->fbox[1], b->fbox[2], b->fbox[3]};
  A.sh.size_map = b->size_map;
  A.sh.rows = g->rows;
  A.sh.cols = g->cols;
  A.sh.use_snap = b->use_snap ? 1 : 0;
  A.sh.area = R.area;
  A.sh.m = R.m;
  A.sh.gC = gC;
  A.sh.gX = gX;
  A.sh.dirty = g->gdirty;
  A.sh.dl = g->dl;
  A.sh.dl_off = g->dl_off;
  A.sh.pr = b->pickup_rate;
  A.sh.dr = b->dep_rate;
  A.sh.cap = b->cap;
  const int64_t rec = R.n_dl * (int64_t)(sizeof(VState) / sizeof(float));  // one per listed visit
  if (rec) ensure(g->scratch, g->scratch_cap, rec, s);
  std::vector<int> dl0;  // first listed visit of each stamp
  if (R.n_dl) {
    dl0.assign(R.st.size(), 0);
    int at = 0;
    for (size_t k = 0; k < R.st.size(); ++k) {
      dl0[k] = at;
      if (R.st[k].dl_nlev > 0) at += R.n_visits[k];
    }
  }
  // the last dip up to every stamp (its paint is the brush's; stamp 0 dips)
  int dip = s0;
  while (!(g->st[(size_t)dip].flags & PNT_STAMP_DIP)) --dip;
  std::vector<int> dip_of(R.st.size());
  for (size_t k = 0; k < R.st.size(); ++k) {
    if (g->st[(size_t)s0 + k].flags & PNT_STAMP_DIP) dip = s0 + (int)k;
    dip_of[k] = dip;
  }
  for (size_t w = R.waves.size(); w-- > 0;) {
    int ns = 0, widest = 1;
    bool dup = false;
    for (const TapeRun::Phase& f : R.waves[w]) {
      ASlot& S = A.slot[ns++];
      S = ASlot{};
      S.clear = f.clear;
      S.gP = g->gP + (int64_t)f.chain * kCell * R.m;
      if (f.clear) {
        S.nblk = (int)std::min<int64_t>(64, (kCell * R.m + 4 * kBlk - 1) / (4 * kBlk));
      } else {
        const PStamp& st = R.st[(size_t)f.k];
        S.st = st;
        S.tape = R.base + R.slot * f.k;
        S.gB = g->gB + 6 * (int64_t)(s0 + f.k);
        S.scratch = R.n_dl ? g->scratch + dl0[(size_t)f.k] * (int64_t)(sizeof(VState) / sizeof(float))
                           : nullptr;
        S.win = tile_window(stamp_geom(st, b->size_map, g->rows, g->cols), A.sh.dom);
        S.ntiles = tile_count<kGT>(S.win);
        S.rb = b->use_snap ? ring_blocks_for(st.box, kBlk) : 0;
        S.nblk = S.ntiles + S.rb + (dup_levels(st) ? 1 : 0);
        for (int c = 0; c < 3; ++c) {
          S.pk[c] = g->st[(size_t)dip_of[(size_t)f.k]].K[c];
          S.ps[c] = g->st[(size_t)dip_of[(size_t)f.k]].S[c];
        }
        dup |= (st.flags & (kStDupX | kStDupY)) != 0;
      }
      widest = std::max(widest, S.nblk);
    }
    if (!ns) continue;
    const dim3 grid((unsigned)widest, (unsigned)ns);
    if (dup)
      k_adj_wave<true><<<grid, kBlk, 0, s>>>(A);
    else
      k_adj_wave<false><<<grid, kBlk, 0, s>>>(A);
    PNT_HIP_CHECK(hipGetLastError());
  }
}

extern "C" {

int pnt_grad_create(pnt_ctx ctx, int rows, int cols, pnt_brush brush, const pnt_stamp* stamps,
                    int64_t n, const int32_t* paint_of, int n_pig, const double* palK,
                    const double* palS, int n_paint, int seg_len, pnt_grad* out) {
  return guard_call([&] {
    PNT_REQUIRE(ctx && brush && out, "NULL argument");
    PNT_REQUIRE(brush->ctx->device == ctx->device, "brush on another device");
    PNT_REQUIRE(rows > 0 && cols > 0 && (int64_t)rows * cols < ((int64_t)1 << 31),
                "rows/cols out of range");
    PNT_REQUIRE(n > 0 && stamps && paint_of, "empty stamp list");
    PNT_REQUIRE(n_pig > 0 && n_paint > 0 && palK && palS, "empty palette");
    PNT_REQUIRE(seg_len > 0, "segment length must be positive");
    PNT_REQUIRE(stamps[0].flags & PNT_STAMP_DIP, "the first stamp must dip (its paint is mixed)");
    for (int64_t i = 0; i < n; ++i) {
      PNT_REQUIRE(!(stamps[i].flags & PNT_STAMP_DRY_AFTER),
                  "dryCanvas inside a differentiable stamp list is not supported");
      PNT_REQUIRE(std::isfinite(stamps[i].cx) && std::isfinite(stamps[i].cy) &&
                      std::isfinite(stamps[i].theta),
                  "non-finite stamp");
      if (stamps[i].flags & PNT_STAMP_DIP)
        PNT_REQUIRE(paint_of[i] >= 0 && paint_of[i] < n_paint, "paint index out of range");
    }
    auto* g = new pnt_grad_s;
    g->ctx = ctx;
    g->b = brush;
    g->rows = rows;
    g->cols = cols;
    g->st.assign(stamps, stamps + n);
    g->paint_of.assign(paint_of, paint_of + n);
    g->n_pig = n_pig;
    g->n_paint = n_paint;
    g->palK.assign(palK, palK + 3 * n_pig);
    g->palS.assign(palS, palS + 3 * n_pig);
    g->seg_len = seg_len;
    const int st_create = pnt_canvas_create(ctx, rows, cols, &g->cv);
    if (st_create != PNT_OK) {
      const std::string msg = pnt_last_error();
      delete g;
      throw Error(st_create, msg);
    }
    ctx_retain(ctx);
    *out = g;
  });
}

int pnt_grad_destroy(pnt_grad g) {
  return guard_call([&] {
    if (!g) return;
    (void)hipStreamSynchronize(g->ctx->stream);
    if (g->cv) pnt_canvas_destroy(g->cv);
    (void)hipFree(g->ckpt);
    (void)hipFree(g->tape);
    (void)hipFree(g->gX);
    (void)hipFree(g->gdirty);
    (void)hipFree(g->dl);
    (void)hipFree(g->dl_off);
    (void)hipFree(g->gP);
    (void)hipFree(g->gB);
    (void)hipFree(g->scratch);
    (void)hipFree(g->fp);
    pnt_ctx ctx = g->ctx;
    delete g;
    ctx_release(ctx);
  });
}

int pnt_grad_forward(pnt_grad g, pnt_dev_layer wet0, pnt_dev_rgb R0, const double* W,
                     pnt_dev_rgb R) {
  return guard_call([&] {
    PNT_REQUIRE(g && W, "NULL argument");
    for (int c = 0; c < 7; ++c) PNT_REQUIRE(wet0.p[c], "NULL wet-layer plane");
    for (int c = 0; c < 3; ++c) PNT_REQUIRE(R0.p[c] && R.p[c], "NULL plane");
    g->ctx->use();
    pnt_brush b = g->b;
    pnt_canvas cv = g->cv;
    hipStream_t s = g->ctx->stream;
    const int64_t n = cv->n;
    PNT_HIP_CHECK(hipStreamSynchronize(b->ctx->stream));
    const Layer7 L = cv->layer();
    const Rgb3 R0c = cv->R0();
    Plane7 W0;
    for (int c = 0; c < 7; ++c) W0.p[c] = wet0.p[c];
    launch_layer_from_planes(n, W0, L, s);  // V widened to FP64
    for (int c = 0; c < 3; ++c)
      PNT_HIP_CHECK(hipMemcpyAsync(R0c.p[c], R0.p[c], n * sizeof(float), hipMemcpyDeviceToDevice, s));
    cv->epoch++;
    g->W.assign(W, W + (int64_t)g->n_paint * g->n_pig);
    // each dip's paint: mixSinglePaint(W[paint_of[i]]) in FP64, stored as FP32
    for (size_t i = 0; i < g->st.size(); ++i) {
      if (!(g->st[i].flags & PNT_STAMP_DIP)) continue;
      double K[3], S[3];
      check_status(pnt_mix_single(g->n_pig, g->palK.data(), g->palS.data(), g->n_pig,
                                  g->W.data() + (int64_t)g->paint_of[i] * g->n_pig, K, S));
      for (int c = 0; c < 3; ++c) {
        g->st[i].K[c] = (float)K[c];
        g->st[i].S[c] = (float)S[c];
      }
    }
    // the brush's calls run on its own context's stream
    const bool other = b->ctx->stream != s;
    if (other) PNT_HIP_CHECK(hipStreamSynchronize(s));
    // the first imprint on a canvas copies it whole into the snapshot
    if (b->use_snap) brush_full_snapshot(b, cv);
    g->segs.clear();
    const int ns = (int)g->st.size();
    const int64_t m = b->m, side = 2 * (int64_t)((b->size_map - 1) / 2) + 2;
    g->run.area = side * side;
    g->run.m = m;
    g->run.slot = tape_floats(g->run.area, m);
    g->fwd_size_map = b->size_map;
    g->fwd_snap = b->use_snap;
    if (g->fwd_gen != b->geo_gen || g->fwd_fp.empty()) g->fwd_fp = b->fp_host;
    g->fwd_gen = b->geo_gen;
    g->fwd_radius = b->radius;
    g->fwd_pr = b->pickup_rate;
    g->fwd_dr = b->dep_rate;
    g->fwd_cap = b->cap;
    std::copy(b->fbox, b->fbox + 4, g->fwd_fbox);
    g->have_forward = false;
    const int64_t whole = g->run.slot * ns;
    g->full_tape = whole <= g->tape_cap;
    // PAINTY_GRAD_TAPE_MB bounds the tapes instead (0: always checkpoints)
    const char* bound = std::getenv("PAINTY_GRAD_TAPE_MB");
    if (bound) {
      g->full_tape = whole * (int64_t)sizeof(float) <= ((int64_t)std::atoll(bound) << 20);
    } else if (!g->full_tape) {
      size_t mem_free = 0, mem_total = 0;
      PNT_HIP_CHECK(hipMemGetInfo(&mem_free, &mem_total));
      g->full_tape = whole * (int64_t)sizeof(float) <=
                     std::min((int64_t)mem_free / kTapeFree, kTapeMost);
    }
    if (g->full_tape) {
      try {
        ensure(g->tape, g->tape_cap, whole, s);
      } catch (const Error& e) {  // less memory in one piece than free: checkpoints
        if (e.code != PNT_ENOMEM) throw;
        g->full_tape = false;
      }
    }
    if (g->full_tape) {
      g->run.base = g->tape;
      run_fused(b, cv, g->st.data(), ns, 0, &g->run);
      keep_lists(g);
      if (other) PNT_HIP_CHECK(hipStreamSynchronize(b->ctx->stream));
    } else {
      if (other) PNT_HIP_CHECK(hipStreamSynchronize(b->ctx->stream));
      // segments (at most seg_len stamps, a dip starts a new one) and their
      // checkpoint boxes: the union of their snapshot boxes (window boxes
      // without the snapshot)
      int64_t total = 0;
      for (int s0 = 0; s0 < ns;) {
        int s1 = s0 + 1;
        while (s1 < ns && s1 - s0 < g->seg_len && !(g->st[s1].flags & PNT_STAMP_DIP)) ++s1;
        int x0 = cv->cols, y0 = cv->rows, x1 = -1, y1 = -1;
        for (int i = s0; i < s1; ++i) {
          const StampArgs a = stamp_args(b, cv, g->st[i].cx, g->st[i].cy, g->st[i].theta);
          const RingBox rb = ring_box(a.g, b->radius);
          int bx0 = rb.a_x0, by0 = rb.a_y0, bx1 = rb.a_x1, by1 = rb.a_y1;
          if (!b->use_snap) {
            bx0 = std::max(rb.tl_x, 0);
            by0 = std::max(rb.tl_y, 0);
            bx1 = std::min(rb.br_x, cv->cols - 1);
            by1 = std::min(rb.br_y, cv->rows - 1);
          }
          if (bx1 < bx0 || by1 < by0) continue;
          x0 = std::min(x0, bx0);
          y0 = std::min(y0, by0);
          x1 = std::max(x1, bx1);
          y1 = std::max(y1, by1);
        }
        pnt_grad_s::Seg sg{s0, s1, x0, y0, std::max(x1 - x0 + 1, 0), std::max(y1 - y0 + 1, 0), total};
        // canvas and snapshot boxes as 7 FP64 planes (14 floats per pixel
        // each), the pickup map as 7 FP32 planes; offsets kept 8-byte aligned
        total += round_up((int64_t)sg.w * sg.h * (b->use_snap ? 28 : 14) + 7 * m, 2);
        g->segs.push_back(sg);
        s0 = s1;
      }
      ensure(g->ckpt, g->ckpt_cap, std::max<int64_t>(total, 1), s);
      for (const auto& sg : g->segs) {
        const int64_t area = (int64_t)sg.w * sg.h;
        float* c0 = g->ckpt + sg.off;
        box_copy({layer_box(L, cv->cols, sg.x0, sg.y0, sg.w, sg.h, reinterpret_cast<double*>(c0), area),
                  layer_box(b->snap_planes(), cv->cols, sg.x0, sg.y0, b->use_snap ? sg.w : 0, sg.h,
                            reinterpret_cast<double*>(c0 + 14 * area), area),
                  cell_box(b->pick, b->size_map, 0, 0, b->size_map, b->size_map,
                            c0 + (b->use_snap ? 28 : 14) * area, m)},
                 true, s);
        if (other) PNT_HIP_CHECK(hipStreamSynchronize(s));
        run_fused(b, cv, g->st.data() + sg.s0, sg.s1 - sg.s0);
        if (other) PNT_HIP_CHECK(hipStreamSynchronize(b->ctx->stream));
      }
    }
    launch_compose(n, L, R0c, Rgb3{{R.p[0], R.p[1], R.p[2]}}, s);
    g->have_forward = g->canvas_final = true;
  });
}

int pnt_grad_backward(pnt_grad g, pnt_dev_rgb gR, pnt_dev_layer gwet, pnt_dev_rgb gR0,
                      double* gW) {
  return guard_call([&] {
    PNT_REQUIRE(g && gW, "NULL argument");
    PNT_REQUIRE(g->have_forward, "backward before forward");
    for (int c = 0; c < 7; ++c) PNT_REQUIRE(gwet.p[c], "NULL gradient plane");
    for (int c = 0; c < 3; ++c) PNT_REQUIRE(gR.p[c] && gR0.p[c], "NULL plane");
    g->ctx->use();
    pnt_brush b = g->b;
    pnt_canvas cv = g->cv;
    hipStream_t s = g->ctx->stream;
    PNT_REQUIRE(b->size_map == g->fwd_size_map && b->use_snap == g->fwd_snap,
                "the brush's geometry or snapshot switch changed since the forward");
    // the brush's calls run on its own context's stream; segments use its buffers
    const bool other = b->ctx->stream != s;
    if (other) PNT_HIP_CHECK(hipStreamSynchronize(b->ctx->stream));
    const BrushAsForward as_forward(g);
    const int64_t n = cv->n, m = b->m;
    const int sm = b->size_map;
    const int ns = (int)g->st.size();
    const Layer7 L = cv->layer();
    const Plane7 gC{{gwet.p[0], gwet.p[1], gwet.p[2], gwet.p[3], gwet.p[4], gwet.p[5], gwet.p[6]}};
    // ---- composite adjoint at the final state
    if (!g->full_tape) {
      // the snapshot has this canvas' size again, should the brush have
      // stamped another since; the segments restore what they read of it
      if (b->use_snap && (b->snap_rows != cv->rows || b->snap_cols != cv->cols)) {
        brush_full_snapshot(b, cv);
        if (other) PNT_HIP_CHECK(hipStreamSynchronize(b->ctx->stream));
      }
      if (!g->canvas_final)  // a backward was here before: every segment again, in order
        for (const auto& sg : g->segs) rerun_segment(g, sg, nullptr);
      g->canvas_final = true;
    }
    k_km_adj<<<grid_for(n), kBlk, 0, s>>>(n, L, cv->R0(), Rgb3{{gR.p[0], gR.p[1], gR.p[2]}}, gC,
                                          Rgb3{{gR0.p[0], gR0.p[1], gR0.p[2]}});
    PNT_HIP_CHECK(hipGetLastError());
    const int64_t nst = round_up(n, 64);
    if (b->use_snap) {
      if (!g->adj_zero) {  // the first call, or the last one did not reach its end
        ensure(g->gX, g->gX_cap, 7 * nst, s);
        ensure(g->gdirty, g->gdirty_cap, nst + 16, s);
        launch_fill(g->gX, 7 * nst, 0.0f, s);
        launch_fill_u8(g->gdirty, nst + 16, 0, s);
      }
      g->adj_zero = false;
    }
    // a map adjoint per chain; a segment is one stroke's stamps, one chain
    const int64_t gp_floats = (g->full_tape ? g->run.chains : 1) * kCell * m;
    ensure(g->gP, g->gP_cap, gp_floats, s);
    ensure(g->gB, g->gB_cap, 6 * (int64_t)ns, s);
    launch_fill(g->gP, gp_floats, 0.0f, s);
    launch_fill(g->gB, 6 * (int64_t)ns, 0.0f, s);
    const Plane7 gXL = b->use_snap ? dense7(g->gX, nst) : gC;
    if (g->full_tape) {
      adjoint_waves(g, 0, gC, gXL, s);
    } else {
      ensure(g->tape, g->tape_cap, g->run.slot * g->seg_len, s);
      g->run.base = g->tape;
      g->canvas_final = false;
      for (int k = (int)g->segs.size() - 1; k >= 0; --k) {  // rerun onto the tape, then reversed
        rerun_segment(g, g->segs[(size_t)k], &g->run);
        PNT_REQUIRE(g->run.chains == 1, "a segment on more than one chain");
        adjoint_waves(g, g->segs[(size_t)k].s0, gC, gXL, s);
      }
      cv->epoch++;
      b->dirty_canvas = nullptr;
    }
    if (b->use_snap) {
      k_adj_full_copy<<<grid_for((n + 7) / 8), kBlk, 0, s>>>(n, gC, gXL, g->gdirty);
      PNT_HIP_CHECK(hipGetLastError());
      g->adj_zero = true;
    }
    // ---- mixing weights: dB/dW of mixSinglePaint (PaintMixer.cxx:327-355)
    std::vector<float> hB(6 * (size_t)ns);
    PNT_HIP_CHECK(hipMemcpyAsync(hB.data(), g->gB, hB.size() * sizeof(float), hipMemcpyDeviceToHost, s));
    PNT_HIP_CHECK(hipStreamSynchronize(s));
    std::fill(gW, gW + (int64_t)g->n_paint * g->n_pig, 0.0);
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (int i = ns - 1; i >= 0; --i) {
      for (int c = 0; c < 6; ++c) acc[c] += hB[6 * (size_t)i + c];
      if (!(g->st[i].flags & PNT_STAMP_DIP)) continue;
      const double* w = g->W.data() + (int64_t)g->paint_of[i] * g->n_pig;
      double wsum = 0.0;
      for (int l = 0; l < g->n_pig; ++l) wsum += w[l];
      const bool unit = std::fabs(wsum - 1.0) < 10e-6;
      const double norm = unit ? 1.0 : 1.0 / wsum;
      double Bm[6] = {0, 0, 0, 0, 0, 0};
      for (int l = 0; l < g->n_pig; ++l)
        for (int c = 0; c < 3; ++c) {
          Bm[c] += norm * w[l] * g->palK[3 * l + c];
          Bm[3 + c] += norm * w[l] * g->palS[3 * l + c];
        }
      for (int l = 0; l < g->n_pig; ++l) {
        double v = 0.0;
        for (int c = 0; c < 3; ++c) {
          const double dK = unit ? g->palK[3 * l + c] : norm * (g->palK[3 * l + c] - Bm[c]);
          const double dS = unit ? g->palS[3 * l + c] : norm * (g->palS[3 * l + c] - Bm[3 + c]);
          v += acc[c] * dK + acc[3 + c] * dS;
        }
        gW[(int64_t)g->paint_of[i] * g->n_pig + l] += v;
      }
      for (double& a : acc) a = 0.0;
    }
  });
}

}  // extern "C"
