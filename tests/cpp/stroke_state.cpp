// pnt_paint_stroke on the host stand-in for the HIP runtime (host_hip.hpp): the
// memory a brush holds for its plans does not grow with the stroke's length, and
// a stroke without an imprint leaves the snapshot's dirty bytes as they are.
#include "host_hip.hpp"

#include "painty_hip.h"

static void ok(int st) {
  if (st) std::fprintf(stderr, "status %d: %s\n", st, pnt_last_error()), std::exit(1);
}

static int g_refills;  // dirty bytes set all over: the snapshot's state is not known
static void on_launch(const std::string& name, void** args) {
  g_refills += name.find("9k_fill_u8") != std::string::npos && *(int64_t*)args[1] == 32 * 32;
}

int main() {
  host_hip::state().on_launch = on_launch;
  pnt_ctx ctx;
  pnt_brush b;
  pnt_canvas cv;
  ok(pnt_ctx_create(0, &ctx));
  const std::vector<float> fp(25, 0.5f);
  ok(pnt_brush_create(ctx, 2.0, fp.data(), 5, &b));
  ok(pnt_canvas_create(ctx, 32, 32, &cv));
  size_t held[2];
  for (int k = 0; k < 2; ++k) {  // 9,000 imprints, then 200,000, half along column 0
    const double far = k == 0 ? 4500.0 : 100000.0;
    const double path[6] = {0.3, 4.2, 0.4, 4.2 + far, 0.4 + far, 4.2 + far};
    ok(pnt_paint_stroke(b, cv, path, 3));
    held[k] = host_hip::state().dev_bytes + host_hip::state().pinned_bytes;
  }
  std::printf("bytes held: %zu, then %zu\n", held[0], held[1]);
  pnt_stamp st{};
  st.cx = st.cy = 15.0;
  ok(pnt_imprint_stamps(b, cv, &st, 1, PNT_EXEC_FUSED));
  g_refills = 0;
  const double none[4] = {5.0, 5.0, 5.2, 5.1};
  ok(pnt_paint_stroke(b, cv, none, 2));
  ok(pnt_imprint_stamps(b, cv, &st, 1, PNT_EXEC_FUSED));
  const int kept = g_refills;
  const double one[4] = {15.0, 15.0, 16.2, 15.1};
  ok(pnt_paint_stroke(b, cv, one, 2));
  ok(pnt_imprint_stamps(b, cv, &st, 1, PNT_EXEC_FUSED));
  std::printf("refills after no imprint: %d, after one: %d\n", kept, g_refills - kept);
  if (kept != 0 || g_refills != 1) return 1;
  pnt_canvas_destroy(cv);
  pnt_brush_destroy(b);
  pnt_ctx_destroy(ctx);
  return held[1] > 2 * held[0] ? 1 : 0;  // (buffers grow by doubling)
}
