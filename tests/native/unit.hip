// Entry points for the tests of code that the C ABI does not reach by itself.
// Built into tests/_build/libtrc_unit.so; loaded with ctypes.
#include <hip/hip_runtime.h>

#include "../../tensorray_amd/csrc/common/tr_layout.h"
#include "../../tensorray_amd/csrc/host/window.h"

using namespace trc;

// fit_window for windows that need per_item bytes an item and per_window bytes
// each, `total` items in all, of an allocator that has free_bytes to give.
// out: window, 0 none / 1 kept / 2 allocated, bytes asked for last.
extern "C" void unit_fit_window(uint64_t first, uint64_t total, uint64_t per_item, uint64_t per_window,
                                uint64_t kept_bytes, int may_alloc, uint64_t free_bytes, uint64_t out[3]) {
  char kept, given;
  uint64_t asked = 0;
  const Window w = fit_window(
      first, [&](uint64_t n) { return n * per_item + (total + n - 1) / n * per_window; }, kept_bytes ? &kept : nullptr,
      kept_bytes, may_alloc != 0,
      [&](uint64_t bytes) -> void* {
        asked = bytes;
        return bytes <= free_bytes ? &given : nullptr;
      });
  out[0] = w.size;
  out[1] = !w.ptr ? 0u : w.kept ? 1u : 2u;
  out[2] = asked;
}

// Reciprocal of the scale of a tree with bounds box[0 .. 3) .. box[3 .. 6).
extern "C" float unit_quant_inv_scale(const float box[6]) { return 1.0f / quant_scale(box, box + 3); }

// n nodes quantized on the host.
extern "C" void unit_quantize(const Bvh4Node* nodes, int n, float inv_scale, QNode* out) {
  for (int i = 0; i < n; ++i) out[i] = quantize_node(nodes[i], inv_scale);
}
