// What a gradient runner (pnt_grad) keeps between calls, on the host stand-in
// for the HIP runtime (host_hip.hpp): no device is used, kernels are recorded
// and not run.  grad_state <check>:
//   failures  after a call that failed for memory, at whichever of its
//             allocations, the next one succeeds, its backward starts from
//             cleared adjoint planes and no kernel or copy gets a buffer that is
//             not there
//   streams   a runner and a brush on two contexts: the runner's copies of the
//             brush's plan are done when the forward returns, and a backward
//             that touches the brush's buffers waits for the brush's stream
//   brush     rates and footprint changed after the forward: the backward (and
//             its rerun of segments) has the forward's, the brush keeps the new
//   again     a second backward of one forward begins with the final state: from
//             checkpoints it reruns every segment before the composite's adjoint
//   no-tape   a forward whose tape cannot be allocated keeps checkpoints
//   maps      a map adjoint is held and cleared for each chain that the waves use
#include "host_hip.hpp"

#include <algorithm>
#include <cmath>

#include "painty_hip.h"

using host_hip::state;

static int g_fail = 0;
#define CHECK(cond, ...)                  \
  do {                                    \
    if (!(cond) && g_fail++ < 20) {       \
      std::fprintf(stderr, __VA_ARGS__);  \
      std::fprintf(stderr, " [%s]\n", #cond); \
    }                                     \
  } while (0)

constexpr int kRows = 60, kCols = 64;
constexpr int64_t kN = kRows * kCols, kStride = kN;  // a multiple of 64
constexpr size_t kAdjHead = 216;  // bytes of k_adj_wave's shared arguments

constexpr size_t kStampHead = 128;  // of k_stamp_wave's
constexpr double kOldRate = 0.625, kNewRate = 0.375;  // pickup rates
constexpr float kOldMid = 0.5f, kNewMid = 0.75f;      // the footprint's middle
constexpr int kSide = 13;                             // map side at radius 4

// What the launches since `reset` did.
struct Seen {
  int gX_filled, dirty_filled;  // clears of the whole adjoint planes / their dirty bytes
  int adj, adj_dirty_unset, adj_uncleared, stamps;
  int rate_old, rate_new, fp_old, fp_new;  // launches with either's value
  int64_t map_floats;  // the largest clear of whole map adjoints
  int box_early;  // checkpoint copies beside copies queued on another stream
  std::string order;  // 'k' composite adjoint, 's' stamps, 'a' adjoint wave
} seen;

static void on_launch(const std::string& name, void** args) {
  const auto is = [&](const char* k) { return name.find(k) != std::string::npos; };
  if (is("6k_fillE") && *(int64_t*)args[1] % (8 * kSide * kSide) == 0)
    seen.map_floats = std::max(seen.map_floats, *(int64_t*)args[1]);
  if (is("9k_fill_u8") && *(int64_t*)args[1] == kStride + 16) ++seen.dirty_filled;
  if (is("6k_fillE") && *(int64_t*)args[1] == 7 * kStride) ++seen.gX_filled;
  if (is("k_stamp_wave")) ++seen.stamps, seen.order += 's';
  if (is("k_stamp_wave") || is("k_adj_wave")) {
    const size_t head = is("k_adj_wave") ? kAdjHead : kStampHead;
    seen.rate_old += host_hip::holds(args[0], head, kOldRate);
    seen.rate_new += host_hip::holds(args[0], head, kNewRate);
    // the padded footprint on the device, by its content
    for (const auto& a : state().dev)
      if (host_hip::holds(args[0], kAdjHead, a.first) && a.second == kSide * kSide * sizeof(float)) {
        const float mid = ((const float*)a.first)[kSide * (kSide / 2) + kSide / 2];
        seen.fp_old += mid == kOldMid && is("k_adj_wave");
        seen.fp_new += mid == kNewMid;
      }
  }
  if (is("k_km_adj")) seen.order += 'k';
  if (is("k_box_copy"))
    for (const auto& o : state().queued) seen.box_early += o.stream != state().call.stream;
  if (is("k_adj_wave")) {
    seen.order += 'a';
    ++seen.adj;
    if (!host_hip::holds_alloc(args[0], kAdjHead, kStride + 16)) ++seen.adj_dirty_unset;
    if (!seen.gX_filled || !seen.dirty_filled) ++seen.adj_uncleared;
  }
}

// A runner of 24 stamps in three strokes, some across canvas column/row 0.
struct Runner {
  pnt_ctx ctx = nullptr, bctx = nullptr;
  pnt_brush b = nullptr;
  pnt_grad g = nullptr;
  std::vector<pnt_stamp> st;
  std::vector<float> fp;
  char* dev = nullptr;
  double W[2] = {0.4, 0.6}, gW[2] = {0, 0};

  static std::vector<float> footprint(double r) {
    const int w = (int)(2.0 * std::ceil(r) + 1.0);
    std::vector<float> f((size_t)w * w);
    for (int i = 0; i < w * w; ++i) f[(size_t)i] = 0.2f + 0.01f * (float)(i % 7);
    f[f.size() / 2] = kOldMid;
    return f;
  }
  static int ok(int st) {
    if (st) std::fprintf(stderr, "status %d: %s\n", st, pnt_last_error()), std::abort();
    return st;
  }
  explicit Runner(bool other_ctx = false, int strokes = 3) {
    ok(pnt_ctx_create(0, &ctx));
    bctx = ctx;
    if (other_ctx) ok(pnt_ctx_create(0, &bctx));
    fp = footprint(4.0);
    ok(pnt_brush_create(bctx, 4.0, fp.data(), 9, &b));
    ok(pnt_brush_set_pickup_rate(b, kOldRate));
    std::vector<int32_t> paint_of;
    for (int i = 0; i < 24; ++i) {
      pnt_stamp s{};
      s.cx = i < 16 ? 20.3 + i : 1.4 + 0.7 * (i - 16);
      s.cy = i < 8 ? 30.2 : 2.6 + 0.3 * (i - 8);
      s.theta = 0.2 * i;
      s.flags = i % (24 / strokes) == 0 ? PNT_STAMP_DIP : 0;
      st.push_back(s);
      paint_of.push_back(s.flags ? 0 : -1);
    }
    const double palK[6] = {.1, .2, .3, .4, .5, .6}, palS[6] = {.6, .5, .4, .3, .2, .1};
    ok(pnt_grad_create(ctx, kRows, kCols, b, st.data(), (int64_t)st.size(), paint_of.data(), 2, palK,
                       palS, 1, 8, &g));
    void* p = nullptr;
    ok(hipMalloc(&p, 27 * kN * sizeof(float)));
    dev = (char*)p;
  }
  ~Runner() {
    pnt_grad_destroy(g);
    pnt_brush_destroy(b);
    hipFree(dev);
    if (bctx != ctx) pnt_ctx_destroy(bctx);
    pnt_ctx_destroy(ctx);
  }
  float* plane(int i) const { return (float*)dev + i * kN; }
  int forward() {
    seen = Seen{};
    pnt_dev_layer L;
    for (int i = 0; i < 7; ++i) L.p[i] = plane(i);
    return pnt_grad_forward(g, L, pnt_dev_rgb{{plane(7), plane(8), plane(9)}}, W,
                            pnt_dev_rgb{{plane(10), plane(11), plane(12)}});
  }
  int backward() {
    seen = Seen{};
    pnt_dev_layer L;
    for (int i = 0; i < 7; ++i) L.p[i] = plane(13 + i);
    return pnt_grad_backward(g, pnt_dev_rgb{{plane(20), plane(21), plane(22)}}, L,
                             pnt_dev_rgb{{plane(23), plane(24), plane(25)}}, gW);
  }
};

static void check_failures() {
  for (const char* mode : {"0", "64"}) {  // segments, the whole list on tape
    setenv("PAINTY_GRAD_TAPE_MB", mode, 1);
    int reached = 0;
    for (int at = 1;; ++at) {  // the at-th allocation of a backward
      Runner r;
      Runner::ok(r.forward());
      state().fail_in = at;
      const int first = r.backward();
      const bool hit = state().fail_in == 0;
      state().fail_in = 0;
      CHECK(hit == (first != 0), "tape %s: allocation %d of a backward", mode, at);
      if (!hit) break;
      ++reached;
      CHECK(r.backward() == 0, "tape %s: backward after allocation %d failed", mode, at);
      CHECK(seen.adj > 0 && seen.adj_dirty_unset == 0,
            "tape %s: adjoint waves without dirty bytes after allocation %d failed", mode, at);
      CHECK(seen.adj_uncleared == 0,
            "tape %s: adjoint planes not cleared after allocation %d failed", mode, at);
    }
    CHECK(reached >= 4, "tape %s: allocations seen", mode);
    for (int at = 1;; ++at) {  // the at-th allocation of a forward
      Runner r;
      state().fail_in = at;
      const int first = r.forward();
      const bool hit = state().fail_in == 0;
      state().fail_in = 0;
      if (!hit) break;
      CHECK(first == 0 || r.backward() != 0, "tape %s: backward of a forward that failed", mode);
      CHECK(r.forward() == 0 && r.backward() == 0,
            "tape %s: forward and backward after allocation %d failed", mode, at);
      CHECK(seen.adj > 0 && seen.adj_dirty_unset == 0 && seen.adj_uncleared == 0,
            "tape %s: adjoint after allocation %d of a forward failed", mode, at);
    }
  }
}

static void check_streams() {
  for (const char* mode : {"0", "64"}) {
    setenv("PAINTY_GRAD_TAPE_MB", mode, 1);
    Runner r(true);
    pnt_canvas cv = nullptr;
    Runner::ok(pnt_canvas_create(r.bctx, kRows, kCols, &cv));
    for (int k = 0; k < 2; ++k) {
      Runner::ok(r.forward());
      // the brush plans the same stamps for another canvas, on its own stream
      Runner::ok(pnt_imprint_stamps(r.b, cv, r.st.data(), (int64_t)r.st.size(), PNT_EXEC_FUSED));
      Runner::ok(r.backward());
      CHECK(seen.box_early == 0, "tape %s: checkpoints restored beside the brush's stream", mode);
    }
    CHECK(state().hazards.empty(), "tape %s: copies on two streams", mode);
    pnt_canvas_destroy(cv);
  }
}

static void check_brush() {
  for (const char* mode : {"0", "64"}) {
    setenv("PAINTY_GRAD_TAPE_MB", mode, 1);
    Runner r;
    Runner::ok(r.forward());
    Runner::ok(pnt_brush_set_pickup_rate(r.b, kNewRate));
    std::vector<float> other = r.fp;
    other[other.size() / 2] = kNewMid;
    Runner::ok(pnt_brush_set_radius(r.b, 8.0, Runner::footprint(8.0).data(), 17));
    Runner::ok(pnt_brush_set_radius(r.b, 4.0, other.data(), 9));
    Runner::ok(r.backward());
    CHECK(seen.adj > 0 && seen.rate_new == 0 && seen.rate_old == seen.adj + seen.stamps,
          "tape %s: the forward's rate in %d + %d launches: %d, the new one in %d", mode, seen.adj,
          seen.stamps, seen.rate_old, seen.rate_new);
    CHECK(seen.fp_new == 0 && seen.fp_old == seen.adj, "tape %s: the forward's footprint", mode);
    pnt_canvas cv = nullptr;
    Runner::ok(pnt_canvas_create(r.ctx, kRows, kCols, &cv));
    seen = Seen{};
    Runner::ok(pnt_imprint(r.b, cv, 30.0, 30.0, 0.1));
    CHECK(seen.rate_new == 1 && seen.rate_old == 0, "tape %s: the brush's own rate", mode);
    pnt_canvas_destroy(cv);
  }
}

static void check_again() {
  for (const char* mode : {"0", "64"}) {
    setenv("PAINTY_GRAD_TAPE_MB", mode, 1);
    Runner r;
    Runner::ok(r.forward());
    const int stamps = seen.stamps;
    Runner::ok(r.backward());
    CHECK(seen.order.find('k') == 0, "tape %s: first backward %s", mode, seen.order.c_str());
    for (int k = 0; k < 2; ++k) {
      Runner::ok(r.backward());
      const int before = (int)seen.order.find('k');
      CHECK(before == (mode[0] == '0' ? stamps : 0), "tape %s: another backward: %s", mode,
            seen.order.c_str());
    }
  }
}

static void check_maps() {
  for (const char* mode : {"0", "64"}) {
    setenv("PAINTY_GRAD_TAPE_MB", mode, 1);
    Runner one(false, 1);
    Runner::ok(one.forward());
    Runner::ok(one.backward());
    CHECK(seen.map_floats == 8 * kSide * kSide, "tape %s: %lld floats of map adjoint for one stroke",
          mode, (long long)seen.map_floats);
  }
  Runner far(false, 24);  // strokes of one stamp: several run at once
  Runner::ok(far.forward());
  Runner::ok(far.backward());
  CHECK(seen.map_floats >= 16 * kSide * kSide && seen.map_floats <= 64 * kSide * kSide,
        "%lld floats of map adjoint for many strokes", (long long)seen.map_floats);
}

static void check_no_tape() {
  unsetenv("PAINTY_GRAD_TAPE_MB");
  int refused = 0;
  for (int at = 1;; ++at) {
    Runner r;
    state().fail_in = at;
    const int first = r.forward();
    const bool hit = state().fail_in == 0;
    state().fail_in = 0;
    if (!hit) break;
    if (first) continue;  // another allocation than the tape's
    ++refused;
    Runner::ok(r.backward());
    CHECK(seen.stamps > 0, "a backward without a tape reruns segments: %s", seen.order.c_str());
  }
  CHECK(refused == 1, "%d allocations a forward does without", refused);
}

int main(int argc, char** argv) {
  state().on_launch = on_launch;
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "failures")
    check_failures();
  else if (what == "streams")
    check_streams();
  else if (what == "brush")
    check_brush();
  else if (what == "again")
    check_again();
  else if (what == "no-tape")
    check_no_tape();
  else if (what == "maps")
    check_maps();
  else
    return 2;
  CHECK(state().hazards.empty(), "%s", state().hazards.empty() ? "" : state().hazards[0].c_str());
  std::printf("%s: %d failures\n", what.c_str(), g_fail);
  return g_fail ? 1 : 0;
}
