// Entry points for the tests of code that the C ABI does not reach by itself.
// Built into tests/_build/libtrc_unit.so; loaded with ctypes.
#include <hip/hip_runtime.h>

#include "../../tensorray_amd/csrc/common/tr_layout.h"
#include "../../tensorray_amd/csrc/common/tr_math.h"
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

namespace {
constexpr int kThreads = 256;

// What a thread's arithmetic unit gives for x / b, 1 / sqrt and lengths (see below).
__global__ void k_math(int what, const float* a, const float* b, float* out, uint32_t n) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  if (what == 0) {
    const F3 q = F3{a[i], -a[i], 0.5f * a[i]} / b[i];
    out[3 * i] = q.x;
    out[3 * i + 1] = q.y;
    out[3 * i + 2] = q.z;
  } else if (what == 1) {
    out[i] = sqrt_rn(a[i]);
  } else if (what == 2) {
    out[i] = rsqrt_rn(a[i]);
  } else if (what == 3) {
    const F3 v{a[3 * i], a[3 * i + 1], a[3 * i + 2]};
    float l;
    const F3 d = over_sqrt(v, len2(v), &l);
    out[4 * i] = d.x;
    out[4 * i + 1] = d.y;
    out[4 * i + 2] = d.z;
    out[4 * i + 3] = l;
  } else {
    out[i] = ratio_self(a[i]);
  }
}

__global__ void k_quantize_nodes(const Bvh4Node* nodes, uint32_t n, float inv_scale, QNode* out) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) out[i] = quantize_node(nodes[i], inv_scale);
}
}  // namespace

// Device arithmetic on device arrays of n items; what: 0 (a, -a, a / 2) / b to
// out [n][3], 1 sqrt_rn(a), 2 rsqrt_rn(a), 3 a [n][3] normalized, and its
// length, to out [n][4], 4 ratio_self(a).
extern "C" int unit_math(int what, const float* a, const float* b, float* out, uint32_t n) {
  k_math<<<(n + kThreads - 1) / kThreads, kThreads>>>(what, a, b, out, n);
  return (int)hipGetLastError();
}

// n nodes quantized on the device (device arrays).
extern "C" int unit_quantize_device(const Bvh4Node* nodes, uint32_t n, float inv_scale, QNode* out) {
  k_quantize_nodes<<<(n + kThreads - 1) / kThreads, kThreads>>>(nodes, n, inv_scale, out);
  return (int)hipGetLastError();
}
