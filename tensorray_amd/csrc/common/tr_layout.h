// Device data layout shared by the host builder and the HIP kernels.
//
// Everything a kernel reads for one scene lives in a handful of flat HBM
// arrays owned by the library (scene residency, needed by the serving loop):
//
//   pos      float[V][3]      vertex positions (world space), AoS
//   idx      uint32[T][3]     triangle vertex indices into pos
//   vnrm     float[V][3]      vertex normals (smooth-shaded meshes only)
//   shade    TriShade[T]      per-triangle face normal, area, material, emitter
//   tris     TriRecord[T]     triangle vertices in BVH leaf order (48 B)
//   verts    TriVerts[T]      vertices and their indices by triangle id (48 B)
//   nodes    Bvh4Node[N]      4-wide BVH with float child boxes (refit, SAH cost)
//   qnodes   QNode[N]         the same tree as the traversal reads it, 64 B per node
//   mats     Material[M]
//   light_*  emitter triangles, their CDF and sampling weights
//
// The reference keeps the same information in SoA tensors
// (LibTensorRay/Renderer/Scene.cpp:46-124) and an opaque OptiX GAS
// (Scene.cpp:171-366); here the acceleration structure is explicit.
#pragma once
#include <stdint.h>
#include "tr_math.h"

namespace trc {

// Longest path the integrators record for replay (bounces after the primary hit).
constexpr int kMaxBounces = 8;

// 4-wide BVH node.  Child boxes are stored SoA; `child` encodes inner nodes
// (index), leaves (kLeafBit | triangle record) and empty slots (kEmpty).  The
// builder fills the slots with the inner children first, then the leaves,
// numbers the inner children of a node consecutively, and puts one triangle
// into each leaf, consecutive ones into the leaves of a node: QNode names all
// children by two base indices.
struct alignas(128) Bvh4Node {
  float lox[4], loy[4], loz[4];
  float hix[4], hiy[4], hiz[4];
  uint32_t child[4];
  uint32_t pad[4];
};
static_assert(sizeof(Bvh4Node) == 128, "node must be one 128-byte line");

constexpr uint32_t kEmpty = 0xFFFFFFFFu;
constexpr uint32_t kLeafBit = 0x80000000u;
constexpr uint32_t kLeafTriMask = (1u << 27) - 1u;

TR_HD bool child_is_leaf(uint32_t c) { return (c & kLeafBit) != 0u && c != kEmpty; }
TR_HD uint32_t leaf_tri(uint32_t c) { return c & kLeafTriMask; }
TR_HD uint32_t make_leaf(uint32_t tri) { return kLeafBit | tri; }

// A 4-wide node as the traversal reads it: 64 bytes, four 16-byte loads.
// Child box planes are half-precision offsets from the node's origin in units
// of the tree's scale (SceneDev::qinv_scale is its reciprocal, a power of
// two), rounded outwards; v_fma_mix_f32 reads them without a conversion.
//   w[0..1]  origin / scale, 21 bits per axis: sign, exponent and 12 mantissa
//            bits of a float rounded down (x in w0[31:11], y in w0[10:0] and
//            w1[31:22], z in w1[21:1])
//   w[2]     index of the first inner child | inner children << kQCountShift
//   w[3]     first leaf's triangle record  | leaves << kQCountShift
//   w[4k+4 .. 4k+7]  axis k: lower planes of slots 0 1, 2 3, upper planes of
//            slots 0 1, 2 3
// The forward is bound by VALU issue (92 % of the SIMDs' cycles with the 112
// bytes and 232 instructions of a Bvh4Node visit).  8-bit planes in 48 bytes
// need a conversion per plane and round the large boxes near the root so far
// out that a query tests 21 % more triangles and visits 6 % more nodes of the
// 20k-triangle sphere scene; 11 bits of mantissa do not.
struct alignas(16) QNode {
  uint32_t w[16];
};
static_assert(sizeof(QNode) == 64, "four 16-byte loads");
constexpr int kQCountShift = 27;
constexpr uint32_t kQIndexMask = (1u << kQCountShift) - 1u;
// Relative widening of the plane offsets: covers the rounding of the
// traversal's t = h i + b in its h i part (3 x 2^-24 of it).
constexpr float kQWiden = 1.0f / 1048576.0f;

// Bits of a half-precision number at or below (up = false) or at or above
// (up = true) x >= 0; beyond the largest one 65504 or infinity.  The device
// converts with v_cvt_pkrtz_f16_f32 (towards zero).
#if defined(__HIP_DEVICE_COMPILE__)
TR_HD uint32_t half_bits(float x, bool up) {
  x = x > 0.0f ? x : 0.0f;
  uint32_t h = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x, 0.0f)) & 0xFFFFu;
  if (up && (float)__builtin_bit_cast(_Float16, (uint16_t)h) < x) ++h;
  return h;
}
#else
TR_HD uint32_t half_bits(float xf, bool up) {
  const double x = (double)xf;
  if (!(x < 65504.0)) return up ? 0x7C00u : (x >= 65504.0 ? 0x7BFFu : 0u);
  if (!(x > 0.0)) return 0u;
  int e = 0;
  frexp(x, &e);  // x = m 2^e, m in [0.5, 1)
  if (e < -13) e = -13;
  const double m = ldexp(x, 11 - e);  // [1024, 2048), below for denormals
  const uint32_t k = (uint32_t)(up ? ceil(m) : floor(m));
  return ((uint32_t)(e + 13) << 10) + k;  // a normal number's leading 1024 carries into the exponent
}
#endif

// The scale of a tree with bounds lo .. hi: plane offsets up to 2^14 steps,
// which leaves room for a refit to grow the boxes fourfold (beyond that the
// upper planes become infinite: the boxes only stop culling).  A plane's offset
// is at most the tree's extent and the rounding of its node's origin (2^-12 of
// the coordinate), which is the larger part beyond 4,096 extents from zero.
TR_HD float quant_scale(const float lo[3], const float hi[3]) {
  float off = 0.0f;
  for (int k = 0; k < 3; ++k) {
    const float a = lo[k] < 0.0f ? -lo[k] : lo[k], b = hi[k] < 0.0f ? -hi[k] : hi[k];
    const float mag = (a > b ? a : b) * (1.0f / 4096.0f), ext = hi[k] - lo[k];
    off = ext > off ? ext : off;
    off = mag > off ? mag : off;
  }
  int e = 0;
  if (off > 0.0f && off < 1e30f) frexp((double)off, &e);
  e = e < -80 ? -80 : e;
  return (float)ldexp(1.0, e - 14);
}

// The QNode of `n`, whose slots are laid out as described at Bvh4Node.  The
// scaling is exact; the difference to the origin and the widening round by
// 2^-24 each, well inside the widening, so the planes never lie inside the
// padded boxes.
TR_HD QNode quantize_node(const Bvh4Node& n, float inv_scale) {
  QNode q;
  uint32_t ni = 0u, nl = 0u, leaf = 0u;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    if (n.child[s] == kEmpty) continue;
    if (n.child[s] & kLeafBit) {
      if (nl == 0u) leaf = leaf_tri(n.child[s]);
      ++nl;
    } else {
      ++ni;
    }
  }
  const uint32_t nc = ni + nl;
  const float* lo[3] = {n.lox, n.loy, n.loz};
  const float* hi[3] = {n.hix, n.hiy, n.hiz};
  uint32_t org[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float o = lo[k][0];
#pragma unroll
    for (uint32_t s = 1; s < 4; ++s) o = s < nc && lo[k][s] < o ? lo[k][s] : o;
    union { float f; uint32_t u; } c;
    c.f = o * inv_scale;
    if (c.u & 0x80000000u) c.u += 0x7FFu;  // towards minus infinity
    c.u &= ~0x7FFu;
    org[k] = c.u >> 11;
    uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (uint32_t s = 0; s < 4; ++s) {
      if (s >= nc) continue;
      const float a = lo[k][s] * inv_scale - c.f, b = hi[k][s] * inv_scale - c.f;
      w[s >> 1] |= half_bits(a * (1.0f - kQWiden), false) << (16u * (s & 1u));
      w[2 + (s >> 1)] |= half_bits(b * (1.0f + kQWiden), true) << (16u * (s & 1u));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) q.w[4 + 4 * k + j] = w[j];
  }
  q.w[0] = org[0] << 11 | org[1] >> 10;
  q.w[1] = org[1] << 22 | org[2] << 1;
  q.w[2] = (ni ? n.child[0] : 0u) | ni << kQCountShift;
  q.w[3] = leaf | nl << kQCountShift;
  return q;
}

// SAH costs of a 4-wide node visit and of a triangle test in the cost that
// decides when a refit tree is rebuilt.  The builder has no use for them: at a
// visit cost of 0.25 to 0.35, which rendered the 20k-triangle metric scene
// fastest when it built leaves of up to 4 triangles, every leaf held one (0.1
// and 0.5 +0.5-1 %; 1 +4 %; 1.5 +6 %; 2 +11 %).
constexpr double kSahTraverse = 0.25;
constexpr double kSahIntersect = 1.0;

// Triangle in leaf order for the watertight test: three world-space vertices,
// the original triangle id carried in v0.w.
struct alignas(16) TriRecord {
  float v0[4];
  float v1[4];
  float v2[4];
};

// A triangle's vertices by triangle id, the index of vertex j in vj.w: shading
// and the adjoint read one 48-byte record where idx and then pos would be two
// dependent gathers of twelve words (the checkpointed adjoint waits on memory
// for three quarters of its wave cycles).
struct alignas(16) TriVerts {
  float v0[4];
  float v1[4];
  float v2[4];
};

// Per-triangle shading data (Scene::PostIntersect inputs, Scene.cpp:668-730).
struct alignas(16) TriShade {
  float n[3];        // geometric (face) normal, normalize(cross(p1-p0, p2-p0))
  float area;        // 0.5 * |cross|
  int32_t material;  // BSDF index (mSbtIndexBuffer)
  int32_t emitter;   // -1 or emitter shape index k (mEmitterIDBuffer)
  int32_t emit_tri;  // index into the light arrays or -1 (mTriIdToEmitTriIdBuffer)
  uint32_t flags;    // bit0 smooth shading, bit1 vertices differentiable
};
constexpr uint32_t kTriSmooth = 1u;
constexpr uint32_t kTriDiff = 2u;

enum MaterialType : int32_t {
  kMatDiffuse = 0,
  kMatMicrofacet = 1,
  kMatRoughConductor = 2,
};

// Material record.  Diffuse: albedo = reflectance (Diffuse.cpp:37-85).
// Microfacet: albedo = diffuse reflectance kd, spec = F0, roughness
// (Microfacet.cpp:37-165).  Rough conductor: spec = specular reflectance,
// eta / k complex IOR (Roughconductor.cpp:38-127).
struct alignas(16) Material {
  int32_t type;
  int32_t tex;        // texture index for the albedo / kd slot, -1 = constant
  float roughness;
  float pad0;
  float albedo[3];
  float pad1;
  float spec[3];
  float pad2;
  float eta[3];
  float pad3;
  float k[3];
  float pad4;
};

// Mesh edge for the boundary terms (ObjMesh::processEdges semantics): end
// vertices v0 < v1, the opposite vertex v2 of face f0, the second face f1
// (-1 on a boundary edge).  Geometry is gathered from `pos` / face normals.
struct alignas(16) EdgeDev {
  uint32_t v0, v1, v2;
  int32_t f0, f1;
  uint32_t pad[3];
};

// Size and length integral of an edge list built on the device.
struct EdgeCount {
  int32_t n;
  float integral;
};

// A sampled edge list with its length distribution (Distribution1D over
// |p1 - p0|, Edge.cpp:90-106 / 350-367).  When `dyn` is set, the list was
// selected on the device and its size and integral are read from there
// (n and integral are then unused).
struct EdgeSet {
  const EdgeDev* e;
  const float* len;
  const float* cdf;
  int32_t n;
  float integral;
  const EdgeCount* dyn;
};

// Texture descriptor: FP32 RGB texels, row-major [h][w][3], nearest lookup
// (ImageTexture::Eval, BSDF.cpp:72-98).
struct TexDesc {
  const float* texels;
  int32_t w, h;
  int64_t grad_off;  // float offset of this texture in the texture-gradient buffer
};

// Parameters of a pinhole camera (Camera::Init/Resize, Camera.cpp:89-137 and
// EDXUtil/Graphics/BaseCamera.cpp:45-88) reduced to what the kernels need:
//   raster (rx, ry) -> camera-space point (ax*rx + bx, ay*ry + by, 1)
//   camera -> world rotation columns right/up/dir, origin = eye.
struct CameraDev {
  float eye[3];
  float right[3];
  float up[3];
  float dir[3];
  float ax, bx, ay, by;  // raster -> camera plane z = 1
  float tan_half;        // tan(fov/2)
  float ratio;           // width / height
  float inv_area;        // 1 / area of the image plane at z = 1
  int32_t width, height;
};

// Paths of a launch in its order of slots: path indices first .. first +
// count, or (blocked, whole samples only) the 8 x 8 pixel blocks of the image
// sample by sample, 64 slots each, some of them empty at the ragged edges.
struct PathRange {
  uint64_t first, count;  // paths
  uint64_t slots;
  uint32_t blocked;
  uint32_t pad;
};
// Blocks keep the rays and bounces of a wave closer together than a row of 64
// pixels does; not where the edges would leave more than an eighth of the
// slots empty.
inline PathRange path_range(const CameraDev& C, uint64_t first, uint64_t count) {
  PathRange r{first, count, count, 0u, 0u};
  const uint64_t W = (uint64_t)C.width, H = (uint64_t)C.height, wh = W * H;
  const uint64_t slots = count / wh * (((W + 7) / 8) * ((H + 7) / 8) * 64);
  if (first % wh == 0 && count % wh == 0 && slots * 8 <= count * 9) {
    r.slots = slots;
    r.blocked = 1u;
  }
  return r;
}

struct SceneDev {
  const float* pos;
  const uint32_t* idx;
  const float* vnrm;
  const float* uv;          // float[nuv][2] or null
  const uint32_t* uv_idx;   // uint32[T][3] or null
  const TriShade* shade;
  const TriRecord* tris;
  const TriVerts* verts;
  const Bvh4Node* nodes;
  const QNode* qnodes;
  const Material* mats;
  const TexDesc* texs;
  const int32_t* light_tri;   // emitter triangle -> global triangle id
  const float* light_cdf;     // normalized CDF over emitter triangles
  const float* light_f;       // luminance * area per emitter triangle
  const float* light_pdf;     // area density of its samples (light_area_pdf)
  const float* emit_rad;      // [n_emitters][3]
  EdgeSet sec;                // secondary edges (ConstructSecEdgeList, Edge.cpp:42-88)
  int32_t n_light;
  float light_integral;       // sum(f) / n_light (Distribution1D::mIntegralVal)
  int32_t n_tris;
  int32_t n_mats;
  int32_t stack_need;         // worst-case traversal stack depth of this BVH
  float qinv_scale;           // 1 / scale of the quantized nodes' offsets, a power of two
  int32_t n_verts;
  // smooth-shaded faces incident to each vertex, in triangle order (CSR:
  // faces of vertex v are vf_list[vf_off[v] .. vf_off[v+1])), for the
  // adjoint of the vertex normals; null when no differentiable mesh is smooth
  const uint32_t* vf_off;
  const uint32_t* vf_list;
};

}  // namespace trc
