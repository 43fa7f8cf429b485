// Boundary (edge) terms of the differentiable integrator, one sample per
// thread iteration.  Each term has zero value and the gradient
//
//   d/dtheta [ detach(K) * xDotN ],   xDotN = n . u2,
//   u2 = (1-u-v) P0d + u P1d + v P2d, (u, v) = RayIntersectAD(dir, org, P0, P1-P0, P2-P0)
//
// where K carries the detached radiance / importance / baseVal / pdf of the
// sample and (dir, org, P) may all depend on vertex positions.  The weight
// w = <dL/dI[pixel], K> / spp is folded in before the VJP, so each sample
// scatters a handful of vertex-gradient atomics.
//
// Reference: BoundaryPrimary.cpp:36-181, BoundaryPixel.cpp:36-159,
// BoundaryDirect.cpp:38-143, BoundaryIndirect.cpp:38-192, Edge.cpp:90-409,
// Camera.cpp:345-467, EvalImportance (Integrator.cpp:75-176).
#include <hip/hip_runtime.h>

#include "../trc_internal.h"
#include "adjoint.h"

namespace trc {

constexpr uint32_t kSensorBlock0 = 64u;

__device__ inline TraceCtx make_trace_ctx_b(uint32_t* lds, const LaunchCfg& L) {
  TraceCtx t;
  t.lds = lds + threadIdx.x;
  t.leafq = lds + kStackLds * kBlock + threadIdx.x;
  t.spill = L.spill;
  t.spill_stride = L.grid * kBlock;
  t.cap = L.cap;
  t.n_nodes = t.n_tris = t.n_queries = 0u;
  t.slot_key = nullptr;
  t.slot_uv = nullptr;
  return t;
}

__device__ inline F3 cam_eye(const CameraDev& c) { return F3{c.eye[0], c.eye[1], c.eye[2]}; }

// Context with the slots of the wave-wide leaf tests (trace_run<true>).
__device__ inline TraceCtx make_trace_ctx_bw(uint32_t* lds, const LaunchCfg& L) {
  TraceCtx t = make_trace_ctx_b(lds, L);
  uint32_t* slots = lds + kTraceLdsWords * kBlock;
  t.slot_key = reinterpret_cast<unsigned long long*>(slots) + threadIdx.x;
  t.slot_uv = reinterpret_cast<float2*>(slots + 2 * kBlock) + threadIdx.x;
  return t;
}

// One ray per lane with `has`, the whole wave together.
__device__ inline Hit trace_wave(const SceneDev& S, TraceCtx& tc, bool has, F3 o, F3 d, float tmax, bool any) {
  TraceState ts;
  if (has) trace_begin(ts, tmax);
  else trace_none(ts);
  trace_run<true>(S, tc, o, d, d, tmax, kShadowEpsilon, any, ts, 0);
  return trace_hit(ts);
}

// Calls f(i, has) for the items i of [first, end), 64 consecutive ones per
// wave at a time, taken from the launch's tile counters as waves need them
// (without counters dealt round-robin), with all lanes of the wave: has is
// false for those behind the last item.
template <class F>
__device__ inline void for_each_group(uint64_t first, uint64_t end, const LaunchCfg& L, F&& f) {
  const uint64_t nwaves = (uint64_t)L.grid * (kBlock / 64);
  const uint64_t wave = (blockIdx.x * kBlock + threadIdx.x) >> 6;
  const uint32_t lane = threadIdx.x & 63u;
  TileSupply sup = TileSupply::make(wave, nwaves, 0, end - first, 64, L.tiles);
  while (sup.next < sup.end) {
    f(first + sup.next + lane, sup.next + lane < sup.end);
    sup.more();
  }
}

// The same for the items alone: f returns to skip the rest of an item.
template <class F>
__device__ inline void for_each_item(uint64_t first, uint64_t end, const LaunchCfg& L, F&& f) {
  for_each_group(first, end, L, [&](uint64_t i, bool has) {
    if (has) f(i);
  });
}

// Edge sampling with the length distribution; returns the edge index and
// the pdf per unit length.
__device__ inline int32_t sample_edge(const EdgeSet& E, float u, float* pdf) {
  const int32_t n = E.dyn ? E.dyn->n : E.n;
  const float integral = E.dyn ? E.dyn->integral : E.integral;
  int32_t i = cdf_search(E.cdf, n, u);
  float pmf = E.len[i] / (integral * (float)n);
  *pdf = pmf / E.len[i];
  return i;
}

struct EdgeGeo {
  F3 p0, e1, n0, n1, p2;
  bool boundary;
};
__device__ inline EdgeGeo edge_geo(const SceneDev& S, const EdgeDev& e) {
  EdgeGeo g;
  g.p0 = load3(S.pos, e.v0);
  g.e1 = load3(S.pos, e.v1) - g.p0;
  g.p2 = load3(S.pos, e.v2);
  const TriShade& s0 = S.shade[e.f0];
  g.n0 = F3{s0.n[0], s0.n[1], s0.n[2]};
  g.boundary = e.f1 < 0;
  if (g.boundary) {
    g.n1 = F3{0.0f, 0.0f, 0.0f};
  } else {
    const TriShade& s1 = S.shade[e.f1];
    g.n1 = F3{s1.n[0], s1.n[1], s1.n[2]};
  }
  return g;
}

__device__ inline F3 nan0(F3 v) { return finite3(v) ? v : F3{0.0f, 0.0f, 0.0f}; }

// BSDF::Eval with the shading-normal correction (BSDF.cpp:172-195).
__device__ inline F3 bsdf_eval_corrected(const SceneDev& S, const Its& s, F3 wo, F3 wi) {
  F3 f = bsdf_eval(S, s, wo, wi);
  F3 lo = to_local(s, wo), li = to_local(s, wi);
  float corr = fabsf(lo.z * dot(s.ng, wi) / (li.z * dot(s.ng, wo)));
  return f * corr;
}

// One vertex of EvalImportance (Integrator.cpp:75-176): the contribution to
// the pixel seen through the camera and the next (BSDF-sampled) vertex.
struct ImpStep {
  bool contrib;
  int32_t pixel;
  F3 value;
  bool next;
};
__device__ ImpStep importance_step(const SceneDev& S, const CameraDev& C, TraceCtx& tc, Its& its, F3& rdir, F3& thr,
                                   Rnd4 rnd) {
  ImpStep r;
  r.contrib = false;
  r.next = false;
  r.pixel = 0;
  r.value = F3{0.0f, 0.0f, 0.0f};
  const F3 eye = cam_eye(C);
  F3 wo = -rdir;
  SensorSample sd = sensor_sample(C, its.p);
  if (sd.valid) {
    F3 cd = camera_dir(C, sd.qx * (float)C.width, sd.qy * (float)C.height);
    float tmax = length(its.p - eye) - kShadowEpsilon;
    bool vis = trace_ray<true>(S, tc, eye, cd, kShadowEpsilon, tmax).tri < 0;
    if (vis) {
      F3 t = sd.value * thr;
      F3 bv{0.0f, 0.0f, 0.0f};
      if (bsdf_dir_valid(S, its, wo)) {
        F3 wi = normalize(eye - its.p);
        float wiok = bsdf_dir_valid(S, its, wi) ? 1.0f : 0.0f;
        bv = bsdf_eval_corrected(S, its, wo, wi) * fabsf(dot(its.ns, wi)) * wiok;
      }
      F3 v = t * bv;
      if (finite3(v)) {
        r.contrib = true;
        r.pixel = sd.pixel;
        r.value = v;
      }
    }
  }
  if (bsdf_dir_valid(S, its, wo)) {
    float pdf;
    F3 wi = bsdf_sample(S, its, wo, rnd.a, rnd.b, &pdf);
    F3 bv = bsdf_eval_corrected(S, its, wo, wi) * fabsf(dot(its.ns, wi));
    Hit h = trace_ray<false>(S, tc, its.p, wi, kShadowEpsilon, 1e32f);
    if (h.tri >= 0 && pdf > 0.0f && bsdf_dir_valid(S, its, wi)) {
      r.next = true;
      thr = thr * bv / pdf;
      its = post_intersect(S, h.tri, h.u, h.v);
      rdir = wi;
    }
  }
  return r;
}

// baseVal of the camera-side terms (BoundaryPrimary.cpp:117-129,
// BoundaryPixel.cpp:95-107; the pixel term reverts the sign).
__device__ inline float base_val_camera(F3 itp, F3 ng, F3 raydir, F3 p_edge, F3 eye, F3 edge, F3 edge2, F3* n_out,
                                        bool revert) {
  float dist = length(itp - eye);
  float dist1 = length(p_edge - eye);
  float cos2 = fabsf(dot(ng, -raydir));
  F3 e = cross(edge, raydir);
  float sinphi = length(e);
  F3 proj = normalize(cross(e, ng));
  float sinphi2 = length(cross(raydir, proj));
  F3 n = normalize(cross(ng, proj));
  bool sign0 = dot(e, edge2) > 0.0f, sign1 = dot(e, n) > 0.0f;
  float bv = (dist / dist1) * (sinphi / sinphi2) * cos2;
  bv = bv * (sinphi > kEpsilon ? 1.0f : 0.0f) * (sinphi2 > kEpsilon ? 1.0f : 0.0f);
  float sg = (sign0 == sign1) ? 1.0f : -1.0f;
  *n_out = n;
  return bv * (revert ? -sg : sg);
}

// baseVal of the secondary terms (Edge.cpp:245-257, BoundaryIndirect.cpp:100-112).
__device__ inline float base_val_secondary(F3 its_p, F3 far_p, F3 far_n, F3 dir_to_near, F3 p_edge, F3 edge, F3 edge2,
                                           F3* n_out) {
  float dist = length(far_p - its_p);
  float cos2 = fabsf(dot(far_n, dir_to_near));
  F3 e = cross(edge, -dir_to_near);
  float sinphi = length(e);
  F3 proj = normalize(cross(e, far_n));
  float sinphi2 = length(cross(-dir_to_near, proj));
  float itsT = length(its_p - p_edge);
  F3 n = normalize(cross(far_n, proj));
  bool sign0 = dot(e, edge2) > 0.0f, sign1 = dot(e, n) > 0.0f;
  float bv = (itsT / dist) * (sinphi / sinphi2) * cos2;
  bv = bv * (sinphi > kEpsilon ? 1.0f : 0.0f) * (sinphi2 > kEpsilon ? 1.0f : 0.0f);
  *n_out = n;
  return bv * ((sign0 == sign1) ? 1.0f : -1.0f);
}

// VJP of w * xDotN with respect to the triangle vertices P0..P2 (of the
// RayIntersectAD), the ray origin and the point the ray passes through.
// xDotN = n . ((1-u-v) P0d + u P1d + v P2d).
struct XdnAdj {
  F3 P0, P1, P2, org, through;
};
__device__ inline XdnAdj x_dot_n_vjp(F3 P0, F3 P1, F3 P2, F3 org, F3 through, F3 n, float w) {
  XdnAdj a;
  F3 dr = through - org;
  float dl;
  F3 dir = over_sqrt(dr, len2(dr), &dl);
  F3 e1 = P1 - P0, e2 = P2 - P0;
  F3 h = cross(dir, e2);
  float aa = dot(e1, h);
  float f = 1.0f / aa;
  F3 s0 = org - P0;
  float su = dot(s0, h);
  F3 q = cross(s0, e1);
  float sv = dot(dir, q);
  float adj_u = w * dot(n, P1 - P0);
  float adj_v = w * dot(n, P2 - P0);
  float adj_f = adj_u * su + adj_v * sv;
  float adj_su = adj_u * f, adj_sv = adj_v * f;
  float adj_a = -adj_f * f * f;
  F3 adj_s0 = adj_su * h;
  F3 adj_h = adj_su * s0 + adj_a * e1;
  F3 adj_dir = adj_sv * q;
  F3 adj_q = adj_sv * dir;
  adj_s0 += cross(e1, adj_q);
  F3 adj_e1 = cross(adj_q, s0) + adj_a * h;
  adj_dir += cross(e2, adj_h);
  F3 adj_e2 = cross(adj_h, dir);
  a.org = adj_s0;
  a.P0 = -(adj_s0 + adj_e1 + adj_e2);
  a.P1 = adj_e1;
  a.P2 = adj_e2;
  F3 adj_dr = normalize_vjp(dir, dl, adj_dir);
  a.through = adj_dr;
  a.org -= adj_dr;
  return a;
}

template <class Sink>
__device__ inline void vtx_add(const SceneDev& S, uint32_t v, int32_t tri, F3 g, Sink& sk) {
  if (!(S.shade[tri].flags & kTriDiff)) return;
  if (!finite3(g)) return;
  sk.pos(v, g);
}

__device__ inline F3 dLdI_at(const float* dLdI, uint32_t WH, int32_t pix) {
  return F3{dLdI[pix], dLdI[WH + pix], dLdI[2 * WH + pix]};
}

// Scatter of one sample: triangle of the RayIntersectAD (tri), edge point
// (through = q0 + t (q1 - q0) when the edge is given) and material-form
// origin (otri, ou, ov) when given.  GradSink: gradients of w * xDotN;
// TangentSink with w = 1: the derivative of xDotN along the tangents.
template <class Sink>
__device__ void scatter_xdn(const SceneDev& S, int32_t tri, F3 org, F3 through, F3 n, float w, const EdgeDev* edge,
                            float et, int32_t ef0, int32_t otri, float ou, float ov, Sink& sk) {
  const TriCorners q = tri_corners(S, tri);
  XdnAdj a = x_dot_n_vjp(q.p0, q.p1, q.p2, org, through, n, w);
  vtx_add(S, q.i0, tri, a.P0, sk);
  vtx_add(S, q.i1, tri, a.P1, sk);
  vtx_add(S, q.i2, tri, a.P2, sk);
  if (edge) {
    vtx_add(S, edge->v0, ef0, (1.0f - et) * a.through, sk);
    vtx_add(S, edge->v1, ef0, et * a.through, sk);
  }
  if (otri >= 0) {
    float ow = 1.0f - ou - ov;
    const TriCorners oq = tri_corners(S, otri);
    vtx_add(S, oq.i0, otri, ow * a.org, sk);
    vtx_add(S, oq.i1, otri, ou * a.org, sk);
    vtx_add(S, oq.i2, otri, ov * a.org, sk);
  }
}

// Derivative-image contribution v at a pixel (non-finite values dropped).
__device__ inline void add_deriv(float* dimg, uint32_t WH, int32_t pix, F3 v) {
  if (!finite3(v)) return;
  if (v.x != 0.0f) atomicAdd(&dimg[pix], v.x);
  if (v.y != 0.0f) atomicAdd(&dimg[WH + pix], v.y);
  if (v.z != 0.0f) atomicAdd(&dimg[2 * WH + pix], v.z);
}

struct BoundaryParams {
  uint32_t seed;
  int32_t max_bounces;
  int32_t spp;
  uint32_t pad;
};

// ---------------------------------------------------------------------------
// Survivor queues.  All terms start, per chunk of samples, with a select kernel
// that draws the samples, traces their first rays and keeps the few that can
// contribute.  Of those only, an eval kernel (direct, indirect) or a bounce and
// a scatter kernel (primary, pixel) trace the long radiance / importance paths,
// so their waves start full instead of carrying the lanes whose samples died at
// the first test.  The queue is structure-of-arrays (word k of slot s at
// w[k * cap + s]) and filled by wave-level ballot compaction: one atomic
// per wave and consecutive slots for the surviving lanes.  Chunks are large
// (4M samples, one chunk for a 512^2 x 16 request): every chunk ends in two
// kernel tails, and at 1M samples per chunk those cost more than the
// compaction saved (kBndChunk; less where that much scratch is not to be had).
// Survivors of the 512^2 metric scene: 10 % of the
// primary, 0.8 % of the direct and 13 % of the indirect samples.
// ---------------------------------------------------------------------------
// One counter word serves an append every 11.5 ns (16,384 groups of 64 samples:
// 0.19 ms), so the queue has kTileCtrs segments, each with a counter in a cache
// line of its own: samples of group g go to segment g % kTileCtrs, which has
// room for all of its groups.  Readers take the survivors of a segment 64 at a
// time, as one list of groups over the segments.  (512 x 512 x 4 pixel select
// 197 us with one counter, 146 us with eight.)
struct BndQueue {
  uint32_t* count;  // survivors of this chunk: kTileSet words
  uint32_t* w;      // kBndWords x cap words
  uint32_t cap;     // kTileCtrs segments of cap / kTileCtrs slots
  __device__ uint32_t groups() const {
    uint32_t n = 0u;
#pragma unroll
    for (int k = 0; k < kTileCtrs; ++k) n += (count[k * kTileCtrStride] + 63u) >> 6;
    return n;
  }
  // first slot of group g, which is less than groups(), and its survivors
  __device__ uint32_t group(uint32_t g, uint32_t* n) const {
    uint32_t base = 0u;
    *n = 0u;
#pragma unroll
    for (int k = 0; k < kTileCtrs; ++k) {
      const uint32_t c = count[k * kTileCtrStride], m = (c + 63u) >> 6;
      if (g < m) {
        base = (uint32_t)k * (cap / (uint32_t)kTileCtrs) + g * 64u;
        *n = c - g * 64u < 64u ? c - g * 64u : 64u;
        break;
      }
      g -= m;
    }
    return base;
  }
};
constexpr int kBndWords = 20;

// Slot of the calling lane in the queue when `keep`, else -1; group: the
// wave's, of 64 samples of the chunk.  Every active lane of the wave calls it
// at the same point.
__device__ inline int64_t wave_append(bool keep, const BndQueue& Q, uint64_t group) {
  const uint64_t act = __ballot(1);
  const uint64_t m = __ballot(keep);
  if (m == 0ull) return -1;
  const int lane = (int)(threadIdx.x & 63u);
  const int leader = __ffsll((unsigned long long)act) - 1;
  uint32_t base = 0u;
  const uint32_t seg = (uint32_t)(group % (uint64_t)kTileCtrs);
  if (lane == leader) base = atomicAdd(Q.count + seg * (uint32_t)kTileCtrStride, (uint32_t)__popcll(m));
  base = (uint32_t)__shfl((int)base, leader);
  if (!keep) return -1;
  return (int64_t)(seg * (Q.cap / (uint32_t)kTileCtrs) + base) + (int64_t)__popcll(m & ((1ull << lane) - 1ull));
}

// Calls f(s) for the survivors' slots s, a group per wave at a time from the
// launch's second set of tile counters.
template <class F>
__device__ inline void for_each_survivor(const BndQueue& Q, LaunchCfg L, F&& f) {
  if (L.tiles) L.tiles += kTileSet;
  const uint32_t lane = threadIdx.x & 63u;
  for_each_group(0, (uint64_t)Q.groups() * 64u, L, [&](uint64_t i, bool) {
    uint32_t n;
    const uint32_t s = Q.group((uint32_t)(i >> 6), &n) + lane;
    if (lane < n) f(s);
  });
}

struct QWriter {
  const BndQueue& q;
  uint32_t s;
  int k = 0;
  __device__ void f(float x) { q.w[(size_t)(k++) * q.cap + s] = __float_as_uint(x); }
  __device__ void u(uint32_t x) { q.w[(size_t)(k++) * q.cap + s] = x; }
  __device__ void i(int32_t x) { u((uint32_t)x); }
  __device__ void f3(F3 v) { f(v.x); f(v.y); f(v.z); }
  __device__ void u64(uint64_t x) { u((uint32_t)x); u((uint32_t)(x >> 32)); }
};
struct QReader {
  const BndQueue& q;
  uint32_t s;
  int k = 0;
  __device__ float f() { return __uint_as_float(q.w[(size_t)(k++) * q.cap + s]); }
  __device__ uint32_t u() { return q.w[(size_t)(k++) * q.cap + s]; }
  __device__ int32_t i() { return (int32_t)u(); }
  __device__ F3 f3() { F3 v; v.x = f(); v.y = f(); v.z = f(); return v; }
  __device__ uint64_t u64() { uint64_t lo = u(); uint64_t hi = u(); return lo | (hi << 32); }
};

// ---------------------------------------------------------------------------
// The camera-side terms: primary edges and the pixel boundary.
//
// A select kernel per term finds the samples that count and their first hits;
// one bounce kernel runs the radiance paths of both (render_bounces: a lane
// whose path has ended takes the next survivor); one scatter kernel weighs and
// scatters.  A path per lane in one loop over the samples, as before, waits for
// the longest of 64 paths and carries the samples that hit nothing.
// ---------------------------------------------------------------------------
// Words of a survivor: random index 0-1, hit 2-4, camera ray 5-7 (replaced by
// the radiance along it), sensor value 8, pixel 9, baseVal 10, pdf 11, edge
// normal 12-14, point 15-17, and for an edge its index 18 and the position on
// it 19.
constexpr int kQHit = 2, kQRad = 5, kQValue = 8, kQPixel = 9;

// Survivors as a source of the bounce pass; paths are queue slots.
template <uint32_t kRng>
struct QueuePaths {
  BndQueue q;
  uint32_t base;
  static constexpr uint32_t kDomain = kRng;
  __device__ float word(int k, uint64_t s) const { return __uint_as_float(q.w[(size_t)k * q.cap + s]); }
  __device__ bool open(uint64_t i, uint32_t lane) {
    uint32_t n;
    base = q.group((uint32_t)(i >> 6), &n);
    return lane < n;
  }
  __device__ uint64_t path(uint32_t off) const { return base + off; }
  __device__ uint64_t rng_index(uint64_t s) const {
    return (uint64_t)q.w[s] | ((uint64_t)q.w[(size_t)q.cap + s] << 32);
  }
  __device__ void first_hit(PathLane& L) const {
    L.tri = (int32_t)q.w[(size_t)kQHit * q.cap + L.path];
    L.u = word(kQHit + 1, L.path);
    L.v = word(kQHit + 2, L.path);
  }
  // throughput = sensor importance (GenerateBoundaryRays)
  __device__ void first_vertex(const SceneDev&, const Its&, PathLane& L) const {
    L.raydir = F3{word(kQRad, L.path), word(kQRad + 1, L.path), word(kQRad + 2, L.path)};
    const float value = word(kQValue, L.path);
    L.beta = F3{value, value, value};
  }
};

// bounces: the radiance along each survivor's camera ray, all detached.
template <uint32_t kRng>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kBounceWaves)))
k_bnd_bounces(SceneDev S, BoundaryParams P, LaunchCfg L, BndQueue Q) {
  __shared__ __align__(8) uint32_t lds_stack[(kTraceLdsWords + kTraceSlotWords) * kBlock];
  TraceCtx tc = make_trace_ctx_bw(lds_stack, L);
  const uint64_t nwaves = (uint64_t)L.grid * (kBlock / 64);
  const uint64_t wave = (blockIdx.x * kBlock + threadIdx.x) >> 6;
  TileSupply sup = TileSupply::make(wave, nwaves, 0, (uint64_t)Q.groups() * 64u, 64, L.tiles ? L.tiles + kTileSet : nullptr);
  render_bounces<false>(S, QueuePaths<kRng>{Q, 0}, P.seed, P.max_bounces, tc, sup, CkptDev{},
                        [&](uint64_t s, F3 c) {
                          uint32_t* w = Q.w + (size_t)kQRad * Q.cap + s;
                          w[0] = __float_as_uint(c.x);
                          w[(size_t)Q.cap] = __float_as_uint(c.y);
                          w[2 * (size_t)Q.cap] = __float_as_uint(c.z);
                        });
}

// Vertex gradients of a wave on their way to memory: every lane puts up to kN
// of them down in LDS, and the wave then adds them with four lanes to a vertex
// (three components and one idle), so that the components of a vertex go out
// as one request to one line instead of one each.
template <int kN>
struct WaveGrads {
  float4* e;  // [kN][64]: the gradient, and the vertex's bits (~0: none)
  int k;
  __device__ bool has_vn() const { return false; }
  __device__ void open() {
    const uint32_t lane = threadIdx.x & 63u;
    k = 0;
#pragma unroll
    for (int j = 0; j < kN; ++j) e[j * 64 + lane].w = __uint_as_float(~0u);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  __device__ void pos(uint32_t v, F3 g) {
    e[(k++) * 64 + (threadIdx.x & 63u)] = make_float4(g.x, g.y, g.z, __uint_as_float(v));
  }
  // Sums the entries of the lanes whose hit is the same triangle into those of
  // the first of them; all lanes of the wave.
  __device__ void merge(int32_t tri, bool live) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t first = lane;
    for (uint64_t todo = __builtin_amdgcn_ballot_w64(live); todo != 0ull;) {
      const int l = __ffsll((unsigned long long)todo) - 1;
      const uint64_t m = __builtin_amdgcn_ballot_w64(live && tri == __builtin_amdgcn_readlane(tri, l));
      if ((m >> lane) & 1ull) first = (uint32_t)l;
      todo &= ~m;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (live && first != lane) {
      for (int j = 0; j < k; ++j) {
        const float4 g = e[j * 64 + lane];
        float* d = reinterpret_cast<float*>(e + j * 64 + first);
        if (__float_as_uint(d[3]) != __float_as_uint(g.w)) continue;
        atomicAdd(&d[0], g.x);
        atomicAdd(&d[1], g.y);
        atomicAdd(&d[2], g.z);
        e[j * 64 + lane].w = __uint_as_float(~0u);
      }
    }
  }
  // all lanes of the wave
  __device__ void flush(float* dpos) {
    const uint32_t lane = threadIdx.x & 63u, c = lane & 3u;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
    for (int j = 0; j < kN * 64; j += 16) {
      const float* p = reinterpret_cast<const float*>(e + j + (lane >> 2));
      const uint32_t v = __float_as_uint(p[3]);
      const float g = p[c];
      if (v != ~0u && c < 3u && g != 0.0f) atomicAdd(&dpos[3 * (size_t)v + c], g);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
};

// scatter: weight and vertex gradients of each survivor; kTangent: the
// derivative image along tpos goes to dimg instead.  kEdge: a primary edge,
// whose end points move too.
template <bool kEdge, bool kTangent>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kBndWaves)))
k_bnd_scatter(SceneDev S, CameraDev C, BoundaryParams P, LaunchCfg L, EdgeSet E, BndQueue Q, const float* dLdI,
              float* dpos, const float* tpos, float* dimg) {
  const uint32_t WH = (uint32_t)C.width * (uint32_t)C.height;
  const F3 eye = cam_eye(C);
  const uint32_t n_g = Q.groups(), nwaves = (uint32_t)L.grid * (kBlock / 64), lane = threadIdx.x & 63u;
  constexpr int kN = kEdge ? 5 : 3;
  __shared__ float4 lds[kTangent ? 1 : kN * kBlock];
  WaveGrads<kN> sk{lds + (kTangent ? 0 : kN * 64 * (threadIdx.x >> 6)), 0};
  for (uint32_t g = (blockIdx.x * kBlock + threadIdx.x) >> 6; g < n_g; g += nwaves) {
    uint32_t n_live;
    const uint32_t s = Q.group(g, &n_live) + lane;
    bool live = lane < n_live;
    int32_t pixel = 0;
    F3 K{0.0f, 0.0f, 0.0f}, n = K, p = K;
    float w = 1.0f;
    QReader r{Q, s, kQRad};
    if (live) {
      const F3 rad = r.f3();
      r.k = kQPixel;
      pixel = r.i();
      const float bv = r.f(), pdf = r.f();
      K = rad * bv / pdf;
      live = finite3(K) && (!kEdge || length(K) > 0.0f);
      if (!kTangent && live) {
        w = dot(dLdI_at(dLdI, WH, pixel), K) / (float)P.spp;
        live = w != 0.0f;
      }
    }
    if (!kTangent) sk.open();
    int32_t tri = -1;
    if (live) {
      n = r.f3();
      p = r.f3();
      tri = (int32_t)Q.w[(size_t)kQHit * Q.cap + s];
      EdgeDev ed{};
      float rb = 0.0f;
      int32_t f0 = -1;
      if (kEdge) {
        ed = E.e[r.i()];
        rb = r.f();
        f0 = ed.f0;
      }
      if constexpr (kTangent) {
        TangentSink tk{tpos, nullptr, nullptr, 0.0f};
        scatter_xdn(S, tri, eye, p, n, 1.0f, kEdge ? &ed : nullptr, rb, f0, -1, 0.0f, 0.0f, tk);
        add_deriv(dimg, WH, pixel, K * (tk.acc / (float)P.spp));
      } else {
        scatter_xdn(S, tri, eye, p, n, w, kEdge ? &ed : nullptr, rb, f0, -1, 0.0f, 0.0f, sk);
      }
    }
    if (!kTangent) {
      if (!kEdge) sk.merge(tri, live);
      sk.flush(dpos);
    }
  }
}

// Primary edges (BoundaryPrimary.cpp:36-181): edge point, the ray away from
// the camera, its projection onto the sensor, the edge point's visibility from
// the camera and baseVal.
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kBndWaves)))
k_bnd_primary_select(SceneDev S, CameraDev C, BoundaryParams P, LaunchCfg L, EdgeSet E, uint64_t first, uint64_t end,
                     BndQueue Q) {
  __shared__ __align__(8) uint32_t lds_stack[(kTraceLdsWords + kTraceSlotWords) * kBlock];
  TraceCtx tc = make_trace_ctx_bw(lds_stack, L);
  const F3 eye = cam_eye(C);
  // no silhouette or boundary edge seen from this camera: no samples
  if ((E.dyn ? E.dyn->n : E.n) <= 0) return;
  for_each_group(first, end, L, [&](uint64_t i, bool has) {
    const Rnd4 rnd = rng4(P.seed, kRngPrimaryEdge, i, 0u);
    float pdf;
    const int32_t ei = sample_edge(E, rnd.a, &pdf);
    const EdgeGeo g = edge_geo(S, E.e[ei]);
    const F3 p = g.p0 + rnd.b * g.e1;
    const F3 dir = normalize(p - eye);
    const Hit h = trace_wave(S, tc, has, p, dir, 1e32f, false);
    const SensorSample sd = sensor_sample(C, p + h.t * dir);
    const bool seen = h.tri >= 0 && sd.valid;
    const F3 rd = camera_dir(C, sd.qx * (float)C.width, sd.qy * (float)C.height);
    const float tmax = length(p - eye) - kShadowEpsilon;
    const bool hidden = trace_wave(S, tc, seen, eye, rd, tmax, true).tri >= 0;
    bool keep = false;
    float bv = 0.0f;
    F3 n{0.0f, 0.0f, 0.0f};
    if (seen && !hidden) {
      const Its its = post_intersect(S, h.tri, h.u, h.v);
      bv = base_val_camera(its.p, its.ng, rd, p, eye, normalize(g.e1), normalize(g.p2 - g.p0), &n, false);
      // K = rad * bv / pdf vanishes or is not finite for every radiance
      keep = bv != 0.0f && isfinite(bv);
    }
    const int64_t s = wave_append(keep, Q, (i - first) >> 6);
    if (s >= 0) {
      QWriter w{Q, (uint32_t)s};
      w.u64(i); w.i(h.tri); w.f(h.u); w.f(h.v); w.f3(rd); w.f(sd.value); w.i(sd.pixel);
      w.f(bv); w.f(pdf); w.f3(n); w.f3(p); w.i(ei); w.f(rnd.b);
    }
  });
}

// Pixel boundary of the box filter (BoundaryPixel.cpp:36-159, Edge.cpp:377-409,
// Camera.cpp:433-467).  4 antithetic positions per random number.
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kBndWaves)))
k_bnd_pixel_select(SceneDev S, CameraDev C, BoundaryParams P, LaunchCfg L, uint64_t N, PathRange range, BndQueue Q) {
  __shared__ __align__(8) uint32_t lds_stack[(kTraceLdsWords + kTraceSlotWords) * kBlock];
  TraceCtx tc = make_trace_ctx_bw(lds_stack, L);
  const uint32_t WH = (uint32_t)C.width * (uint32_t)C.height;
  const F3 eye = cam_eye(C);
  const F3 R{C.right[0], C.right[1], C.right[2]}, U{C.up[0], C.up[1], C.up[2]}, D{C.dir[0], C.dir[1], C.dir[2]};
  const float plx = 2.0f * C.ratio * C.tan_half, ply = 2.0f * C.tan_half;
  const F3 vdir = normalize(C.ay * U), hdir = normalize(C.ax * R);
  const uint64_t per_anti = N / 4;
  const uint32_t lane = threadIdx.x & 63u;
  for_each_group(0, range.slots, L, [&](uint64_t slot, bool) {
    const PathGroup g = PathGroup::at(C, range, slot - lane);
    const bool has = g.has(lane);
    const uint64_t i = has ? g.path(lane) : g.base;
    const uint64_t j = i % per_anti, anti = i / per_anti;
    float rr = rng4(P.seed, kRngPixelEdge, j, 0u).a;
    float rv;
    if (anti == 0) rv = rr;
    else if (anti == 1) rv = rr < 0.5f ? rr + 0.5f : rr - 0.5f;
    else if (anti == 2) rv = rr < 0.75f ? 0.75f - rr : 1.75f - rr;
    else rv = rr < 0.25f ? 0.25f - rr : 1.25f - rr;
    float r4 = rv * 4.0f;
    int side = (int)floorf(r4);
    float ox, oy;
    if (side == 0) { ox = 0.0f; oy = r4; }
    else if (side == 1) { ox = r4 - 1.0f; oy = 1.0f; }
    else if (side == 2) { ox = 1.0f; oy = 3.0f - r4; }
    else { ox = 4.0f - r4; oy = 0.0f; }
    const uint32_t pix = (uint32_t)(i % WH);
    float rx = (float)(pix % (uint32_t)C.width) + ox, ry = (float)(pix / (uint32_t)C.width) + oy;
    F3 p0 = ((eye + (C.ax * rx + C.bx) * R) + (C.ay * ry + C.by) * U) + D;
    F3 dir = normalize(p0 - eye);
    const Hit h = trace_wave(S, tc, has, p0, dir, 1e32f, false);
    bool keep = false;
    float bv = 0.0f, pdf = 0.0f, value = 0.0f;
    F3 n{0.0f, 0.0f, 0.0f}, rd = n;
    if (h.tri >= 0) {
      F3 edge = (side == 0 || side == 2) ? vdir : hdir;
      F3 edge2 = side == 0 ? hdir : (side == 1 ? -vdir : (side == 2 ? -hdir : vdir));
      pdf = (side == 0 || side == 2) ? 0.25f / (ply * (float)C.width) : 0.25f / (plx * (float)C.height);
      const SensorSample sd = sensor_sample(C, p0 + h.t * dir);
      value = sd.value;
      rd = camera_dir(C, sd.qx * (float)C.width, sd.qy * (float)C.height);
      const Its its = post_intersect(S, h.tri, h.u, h.v);
      bv = base_val_camera(its.p, its.ng, rd, p0, eye, edge, edge2, &n, true);
      // K = rad * bv / pdf vanishes or is not finite for every radiance
      keep = bv != 0.0f && isfinite(bv);
    }
    const int64_t s = wave_append(keep, Q, slot >> 6);
    if (s >= 0) {
      QWriter w{Q, (uint32_t)s};
      w.u64(j); w.i(h.tri); w.f(h.u); w.f(h.v); w.f3(rd); w.f(value); w.i((int32_t)pix);
      w.f(bv); w.f(pdf); w.f3(n); w.f3(p0);
    }
  });
}

// ---------------------------------------------------------------------------
// Secondary edges, direct illumination (BoundaryDirect.cpp:38-143,
// Edge.cpp:108-144 and 201-309)
// ---------------------------------------------------------------------------
// Guide evaluation (AdaptiveQuadratureDistribution::setup and
// GuideDirectBoundary_Helper, AQ_distrb.h:63-76 and 100-175): sample k of
// leaf i draws x uniformly in the leaf's CDF interval and (y, z) in [0,1]^2
// and records |baseVal| / spp of the guiding-mode evaluation, where only
// the two hit tests and the same-point test of Edge.cpp:201-262 apply.
// Waves take samples 64 at a time from the launch's counter (2M-triangle
// sphere, 16 samples per leaf: 26.7 ms dealt grid-stride, 21.6 ms so).
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kBndWaves))) k_guide_eval(SceneDev S, LaunchCfg L, uint32_t seed, GuideDev G) {
  __shared__ uint32_t lds_stack[kTraceLdsWords * kBlock];
  TraceCtx tc = make_trace_ctx_b(lds_stack, L);
  const EdgeSet& E = S.sec;
  const uint64_t N = (uint64_t)G.n * (uint64_t)G.spp;
  for_each_item(0, N, L, [&](uint64_t j) {
    const int32_t leaf = (int32_t)(j / (uint64_t)G.spp);
    Rnd4 r = rng4(seed, kRngGuide, j, 0u);
    const float x0 = leaf > 0 ? E.cdf[leaf - 1] : 0.0f, x1 = E.cdf[leaf];
    const float x = x0 + r.a * (x1 - x0);
    float pdf_e;
    int32_t ei = sample_edge(E, x, &pdf_e);
    const EdgeDev ed = E.e[ei];
    EdgeGeo g = edge_geo(S, ed);
    float t = cdf_reuse(E.cdf, ei, x);
    F3 p = g.p0 + t * g.e1;
    F3 edge = normalize(g.e1);
    F3 edge2 = normalize(g.p2 - g.p0);
    LightSample ls = light_sample(S, r.b, r.c);
    F3 rdir = normalize(p - ls.p);
    float v = 0.0f;
    Hit h0 = trace_ray<false>(S, tc, p, -rdir, kShadowEpsilon, 1e32f);
    if (h0.tri >= 0) {
      Hit h = trace_ray<false>(S, tc, p, rdir, kShadowEpsilon, 1e32f);
      F3 hitP = p + h0.t * (-rdir);
      if (h.tri >= 0 && length(hitP - ls.p) < kShadowEpsilon) {
        Its its = post_intersect(S, h.tri, h.u, h.v);
        F3 n;
        v = fabsf(base_val_secondary(its.p, ls.p, ls.n, rdir, p, edge, edge2, &n));
        if (!isfinite(v)) v = 0.0f;
      }
    }
    G.vals[j] = v / (float)G.spp;
  });
}

// Guide normalization (AQ_distrb.h:166-180): poly_i = sum_k vals in sample
// order, w = poly / sum(poly), poly = eps + (1 - eps) w, f = poly * volume,
// then the Distribution1D CDF of f (Distribution.cpp:45-60).  The sums over
// leaves use the blocked order of kSumChunk, so the result does not depend on
// the launch shape and every pass is parallel.
__global__ void k_guide_poly(GuideDev G) {
  const int stride = gridDim.x * blockDim.x;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < G.n; i += stride) {
    float acc = 0.0f;
    const float* v = G.vals + (size_t)i * (size_t)G.spp;
    for (int k = 0; k < G.spp; ++k) acc = acc + v[k];
    G.poly[i] = acc;
  }
}

// One wave per chunk of kSumChunk values: the lanes stage the chunk in LDS and
// one lane runs the dependent additions from there (reading the chunk from
// memory, one lane each, k_chunk_sums took 70 us and k_chunk_prefix 129 us for
// 12,000 leaves).  Returns (lane 0) the sequential sum;
// with `prefix` the inclusive prefix of every value is left in v.
__device__ inline float chunk_sum(float* v, const float* src, int m, bool prefix) {
  for (int i = (int)threadIdx.x; i < kSumChunk; i += 64) v[i] = i < m ? src[i] : 0.0f;
  __syncthreads();
  float acc = 0.0f;
  if (threadIdx.x == 0u) {
    int i = 0;
    for (; i + 16 <= m; i += 16) {
      float4 q[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) q[k] = reinterpret_cast<const float4*>(v + i)[k];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        q[k].x = acc = acc + q[k].x;
        q[k].y = acc = acc + q[k].y;
        q[k].z = acc = acc + q[k].z;
        q[k].w = acc = acc + q[k].w;
      }
      if (prefix) {
#pragma unroll
        for (int k = 0; k < 4; ++k) reinterpret_cast<float4*>(v + i)[k] = q[k];
      }
    }
    for (; i < m; ++i) {
      acc = acc + v[i];
      if (prefix) v[i] = acc;
    }
  }
  __syncthreads();
  return acc;
}

// part[c] = sequential sum of chunk c of v[0, n).
__global__ void __launch_bounds__(64) k_chunk_sums(const float* v, int n, float* part) {
  __shared__ __align__(16) float s[kSumChunk];
  const int lo = (int)blockIdx.x * kSumChunk;
  const float acc = chunk_sum(s, v + lo, min(n - lo, kSumChunk), false);
  if (threadIdx.x == 0u) part[blockIdx.x] = acc;
}

// One thread: part[c] becomes the exclusive prefix of the chunk sums,
// part[nc] their total.
__global__ void k_chunk_scan(float* part, int nc) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  float run = 0.0f;
  for (int c = 0; c < nc; ++c) {
    const float s = part[c];
    part[c] = run;
    run = run + s;
  }
  part[nc] = run;
}

// f_i = (eps + (1 - eps) poly_i / total) * (leaf's x extent), stored in cdf.
__global__ void k_guide_weights(const float* sec_cdf, GuideDev G, const float* total) {
  const float sum = *total;
  const int stride = gridDim.x * blockDim.x;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < G.n; i += stride) {
    const float w = sum > 0.0f ? G.poly[i] / sum : 0.0f;
    const float poly = G.eps + (1.0f - G.eps) * w;
    const float x0 = i > 0 ? sec_cdf[i - 1] : 0.0f;
    G.poly[i] = poly;
    G.cdf[i] = poly * ((sec_cdf[i] - x0) * 1.0f * 1.0f);
  }
}

// cdf_i = (blocked inclusive prefix of f) / n, from the chunk offsets.
__global__ void __launch_bounds__(64) k_chunk_prefix(float* v, int n, const float* part, float inv) {
  __shared__ __align__(16) float s[kSumChunk];
  const int lo = (int)blockIdx.x * kSumChunk, m = min(n - lo, kSumChunk);
  const float off = part[blockIdx.x];
  chunk_sum(s, v + lo, m, true);
  for (int i = (int)threadIdx.x; i < m; i += 64) v[lo + i] = (off + s[i]) * inv;
}

// fsum = total of f; cdf_i /= cdf_{n-1} (the integral) when it is positive.
__global__ void k_guide_normalize(GuideDev G, const float* total) {
  const float integral = G.cdf[G.n - 1];
  if (blockIdx.x == 0 && threadIdx.x == 0) G.fsum[0] = *total;
  if (!(integral > 0.0f)) return;
  const int stride = gridDim.x * blockDim.x;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < G.n - 1; i += stride) G.cdf[i] = G.cdf[i] / integral;
}

// The last element is divided after every other thread has read it.
__global__ void k_guide_normalize_last(GuideDev G) {
  const float integral = G.cdf[G.n - 1];
  if (integral > 0.0f) G.cdf[G.n - 1] = integral / integral;
}

// select: edge point and light point, the two rays from the edge point,
// the emitted radiance and baseVal.
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kBndWaves))) k_bnd_direct_select(SceneDev S, CameraDev C, BoundaryParams P, LaunchCfg L,
                                                              GuideDev G, uint64_t first, uint64_t end, BndQueue Q) {
  __shared__ uint32_t lds_stack[kTraceLdsWords * kBlock];
  TraceCtx tc = make_trace_ctx_b(lds_stack, L);
  const EdgeSet& E = S.sec;
  for_each_item(first, end, L, [&](uint64_t i) {
    bool keep = false;
    Hit h0, h;
    F3 K0, rdir, p, n;
    float t;
    int32_t ei;
    do {
      Rnd4 rnd = rng4(P.seed, kRngDirectEdge, i, 0u);
      float pdf_b = 1.0f;
      if (G.enabled) {
        // AdaptiveQuadratureDistribution::sample (AQ_distrb.h:182-197)
        const int32_t leaf = cdf_search(G.cdf, G.n, rnd.d);
        const float x0 = leaf > 0 ? E.cdf[leaf - 1] : 0.0f, x1 = E.cdf[leaf];
        rnd.a = x0 + rnd.a * (x1 - x0);
        pdf_b = G.poly[leaf] / G.fsum[0];
      }
      float pdf_e;
      ei = sample_edge(E, rnd.a, &pdf_e);
      const EdgeDev ed = E.e[ei];
      EdgeGeo g = edge_geo(S, ed);
      t = cdf_reuse(E.cdf, ei, rnd.a);
      p = g.p0 + t * g.e1;
      F3 edge = normalize(g.e1);
      F3 edge2 = normalize(g.p2 - g.p0);
      LightSample ls = light_sample(S, rnd.b, rnd.c);
      F3 ev = ls.p - p;
      float d2 = len2(ev), dist;
      F3 en = over_sqrt(ev, d2, &dist);
      float cosT = dot(ls.n, -en);
      float c0 = dot(en, g.n0), c1 = dot(en, g.n1);
      bool valid0 = fabsf(c0) > kEdgeEpsilon;
      bool valid1 = (c0 > kEdgeEpsilon && c1 < -kEdgeEpsilon) || (c0 < -kEdgeEpsilon && c1 > kEdgeEpsilon);
      bool right = (g.boundary && valid0) || (!g.boundary && valid1);
      if (!(right && cosT > kEpsilon && dist > kShadowEpsilon)) break;
      float pdf = pdf_e * ls.pdf * d2 / cosT * pdf_b;
      rdir = normalize(p - ls.p);
      h0 = trace_ray<false>(S, tc, p, -rdir, kShadowEpsilon, 1e32f);
      if (h0.tri < 0) break;
      h = trace_ray<false>(S, tc, p, rdir, kShadowEpsilon, 1e32f);
      if (h.tri < 0) break;
      F3 hitP = p + h0.t * (-rdir);
      if (!(length(hitP - ls.p) < kShadowEpsilon)) break;
      F3 Le{0.0f, 0.0f, 0.0f};
      const TriShade& sh0 = S.shade[h0.tri];
      if (sh0.emitter >= 0) Le = emitted(S, sh0.emitter, F3{sh0.n[0], sh0.n[1], sh0.n[2]}, rdir);
      Its its = post_intersect(S, h.tri, h.u, h.v);
      float bv = base_val_secondary(its.p, ls.p, ls.n, rdir, p, edge, edge2, &n);
      K0 = Le * bv / pdf;
      // every contribution K0 * importance then vanishes or is not finite
      keep = finite3(K0) && (K0.x != 0.0f || K0.y != 0.0f || K0.z != 0.0f);
    } while (false);
    const int64_t s = wave_append(keep, Q, (i - first) >> 6);
    if (s >= 0) {
      QWriter w{Q, (uint32_t)s};
      w.u64(i); w.f3(K0); w.i(h.tri); w.f(h.u); w.f(h.v); w.f3(rdir); w.i(h0.tri); w.f3(p); w.f3(n); w.i(ei);
      w.f(t);
    }
  });
}

// eval: EvalImportance from the sensor-side hit for B bounces and the scatter.
// kTangent: the derivative image along tpos goes to dimg instead.
template <bool kTangent>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kBndWaves))) k_bnd_direct_eval(SceneDev S, CameraDev C, BoundaryParams P, LaunchCfg L,
                                                            BndQueue Q, const float* dLdI, float* dpos,
                                                            const float* tpos, float* dimg) {
  __shared__ uint32_t lds_stack[kTraceLdsWords * kBlock];
  TraceCtx tc = make_trace_ctx_b(lds_stack, L);
  const uint32_t WH = (uint32_t)C.width * (uint32_t)C.height;
  const EdgeSet& E = S.sec;
  for_each_survivor(Q, L, [&](uint32_t s) {
    QReader r{Q, s};
    const uint64_t i = r.u64();
    const F3 K0 = r.f3();
    const int32_t tri = r.i();
    const float hu = r.f(), hv = r.f();
    const F3 rdir = r.f3();
    const int32_t tri0 = r.i();
    const F3 p = r.f3();
    const F3 n = r.f3();
    const int32_t ei = r.i();
    const float t = r.f();
    Its its = post_intersect(S, tri, hu, hv);
    const EdgeDev ed = E.e[ei];
    float ds = 0.0f;  // tangent mode: derivative of xDotN
    if constexpr (kTangent) {
      TangentSink sk{tpos, nullptr, nullptr, 0.0f};
      scatter_xdn(S, tri0, its.p, p, n, 1.0f, &ed, t, ed.f0, tri, hu, hv, sk);
      ds = sk.acc / (float)P.spp;
      if (ds == 0.0f || !isfinite(ds)) return;
    }
    // sensor side: EvalImportance for B bounces, throughput 1
    float w = 0.0f;
    Its cur = its;
    F3 cdir = rdir, thr{1.0f, 1.0f, 1.0f};
    for (int b = 0; b < P.max_bounces; ++b) {
      ImpStep st = importance_step(S, C, tc, cur, cdir, thr, rng4(P.seed, kRngDirectEdge, i, kSensorBlock0 + (uint32_t)b));
      if (st.contrib) {
        F3 v = K0 * st.value;
        if (length(v) > 0.0f) {
          if constexpr (kTangent) add_deriv(dimg, WH, st.pixel, v * ds);
          else w += dot(dLdI_at(dLdI, WH, st.pixel), v);
        }
      }
      if (!st.next) break;
    }
    if constexpr (!kTangent) {
      w = w / (float)P.spp;
      if (w == 0.0f || !isfinite(w)) return;
      GradSink sk{dpos, nullptr, nullptr, nullptr, nullptr};
      scatter_xdn(S, tri0, its.p, p, n, w, &ed, t, ed.f0, tri, hu, hv, sk);
    }
  });
}

// ---------------------------------------------------------------------------
// Secondary edges, indirect illumination (BoundaryIndirect.cpp:38-192,
// Edge.cpp:146-199)
// ---------------------------------------------------------------------------
// select: edge point and direction, the two rays from the edge point and
// baseVal / pdf.
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kBndWaves))) k_bnd_indirect_select(SceneDev S, CameraDev C, BoundaryParams P, LaunchCfg L,
                                                                uint64_t first, uint64_t end, BndQueue Q) {
  __shared__ uint32_t lds_stack[kTraceLdsWords * kBlock];
  TraceCtx tc = make_trace_ctx_b(lds_stack, L);
  const EdgeSet& E = S.sec;
  for_each_item(first, end, L, [&](uint64_t i) {
    bool keep = false;
    Hit he, hs;
    F3 dir, p, n;
    float v0, t;
    int32_t ei;
    do {
      Rnd4 rnd = rng4(P.seed, kRngIndirectEdge, i, 0u);
      float pdf_e;
      ei = sample_edge(E, rnd.a, &pdf_e);
      const EdgeDev ed = E.e[ei];
      EdgeGeo g = edge_geo(S, ed);
      t = cdf_reuse(E.cdf, ei, rnd.a);
      p = g.p0 + t * g.e1;
      F3 edge = normalize(g.e1);
      F3 edge2 = normalize(g.p2 - g.p0);
      float pdf_d;
      if (g.boundary) {
        F3 nrm = cross(g.n0, edge);
        F3 ft, fb;
        coordinate_system(nrm, &ft, &fb);
        float z = minf(1.0f - 2.0f * rnd.b, 1.0f - kEdgeEpsilon);
        float rr = sqrt_rn(maxf(0.0f, 1.0f - z * z));
        float sp, cp;
        tr_sincos(2.0f * kPi * rnd.c, &sp, &cp);
        dir = ((rr * cp) * ft + (rr * sp) * fb) + z * nrm;
        pdf_d = 0.25f / kPi;
      } else {
        float phi0 = tr_acos(dot(g.n0, g.n1));
        pdf_d = 0.25f / phi0;
        F3 z = normalize(g.n0 + g.n1);
        F3 y = normalize(cross(g.n0, z));
        F3 x = cross(y, z);
        float phi = (rnd.b - 0.5f) * phi0;
        phi = minf(maxf(phi, -0.5f * phi0 + kEdgeEpsilon), 0.5f * phi0 - kEdgeEpsilon);
        float sp, cp;
        tr_sincos(phi, &sp, &cp);
        F3 x1 = x * cp + z * sp;
        bool m0 = rnd.c > 0.5f;
        float bb = 4.0f * rnd.c - (m0 ? 3.0f : 1.0f);
        float aa = sqrt_rn(1.0f - bb * bb) * (m0 ? -1.0f : 1.0f);
        dir = x1 * aa + y * bb;
      }
      float pdf = pdf_e * pdf_d;
      he = trace_ray<false>(S, tc, p, -dir, kShadowEpsilon, 1e32f);
      if (he.tri < 0) break;
      hs = trace_ray<false>(S, tc, p, dir, kShadowEpsilon, 1e32f);
      if (hs.tri < 0) break;
      Its ite = post_intersect(S, he.tri, he.u, he.v);
      Its its = post_intersect(S, hs.tri, hs.u, hs.v);
      float bv = base_val_secondary(its.p, ite.p, ite.ng, dir, p, edge, edge2, &n);
      v0 = bv / pdf;
      // with max_bounces <= 1 no path length fits; a zero or non-finite v0
      // makes every contribution vanish or not finite
      keep = P.max_bounces > 1 && v0 != 0.0f && isfinite(v0);
    } while (false);
    const int64_t s = wave_append(keep, Q, (i - first) >> 6);
    if (s >= 0) {
      QWriter w{Q, (uint32_t)s};
      w.u64(i); w.i(he.tri); w.f(he.u); w.f(he.v); w.i(hs.tri); w.f(hs.u); w.f(hs.v); w.f3(dir); w.f(v0);
      w.f3(p); w.f3(n); w.i(ei); w.f(t);
    }
  });
}

// eval: the emitter-side radiance after 1..B-1 bounces, the sensor-side
// importance, their combination by total length and the scatter.
// kTangent: the derivative image along tpos goes to dimg instead.
template <bool kTangent>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kBndWaves))) k_bnd_indirect_eval(SceneDev S, CameraDev C, BoundaryParams P, LaunchCfg L,
                                                              BndQueue Q, const float* dLdI, float* dpos,
                                                              const float* tpos, float* dimg) {
  __shared__ uint32_t lds_stack[kTraceLdsWords * kBlock];
  TraceCtx tc = make_trace_ctx_b(lds_stack, L);
  const uint32_t WH = (uint32_t)C.width * (uint32_t)C.height;
  const EdgeSet& E = S.sec;
  const int B = P.max_bounces;
  for_each_survivor(Q, L, [&](uint32_t s) {
    QReader r{Q, s};
    const uint64_t i = r.u64();
    const int32_t tri_e = r.i();
    const float ue = r.f(), ve = r.f();
    const int32_t tri_s = r.i();
    const float us = r.f(), vs = r.f();
    const F3 dir = r.f3();
    const float v0 = r.f();
    const F3 p = r.f3();
    const F3 n = r.f3();
    const int32_t ei = r.i();
    const float t = r.f();
    Its ite = post_intersect(S, tri_e, ue, ve);
    Its its = post_intersect(S, tri_s, us, vs);
    const EdgeDev ed = E.e[ei];
    float ds = 0.0f;  // tangent mode: derivative of xDotN
    if constexpr (kTangent) {
      TangentSink sk{tpos, nullptr, nullptr, 0.0f};
      scatter_xdn(S, tri_e, its.p, p, n, 1.0f, &ed, t, ed.f0, tri_s, us, vs, sk);
      ds = sk.acc / (float)P.spp;
      if (ds == 0.0f || !isfinite(ds)) return;
    }
    // emitter side: cumulative radiance after 1..B-1 bounces
    F3 cum[kMaxBounces];
    F3 per[kMaxBounces];
    for (int k = 0; k < kMaxBounces; ++k) per[k] = F3{0.0f, 0.0f, 0.0f};
    F3 acc{0.0f, 0.0f, 0.0f};
    if (B > 1)
      path_bounces<false, true>(S, tc, ite, F3{1.0f, 1.0f, 1.0f}, -dir, P.seed, kRngIndirectEdge, i, 1u, B - 1, acc,
                                nullptr, per);
    F3 run{0.0f, 0.0f, 0.0f};
    for (int k = 0; k < B - 1; ++k) {
      run = run + per[k];
      cum[k] = run;
    }
    // sensor side
    float w = 0.0f;
    Its cur = its;
    F3 cdir = dir, thr{1.0f, 1.0f, 1.0f};
    for (int b = 0; b < B - 1; ++b) {
      ImpStep st = importance_step(S, C, tc, cur, cdir, thr, rng4(P.seed, kRngIndirectEdge, i, kSensorBlock0 + (uint32_t)b));
      int ri = B - b - 2;
      if (st.contrib && ri >= 0) {
        F3 v = (v0 * cum[ri]) * st.value;
        if (length(v) > 0.0f) {
          if constexpr (kTangent) add_deriv(dimg, WH, st.pixel, v * ds);
          else w += dot(dLdI_at(dLdI, WH, st.pixel), v);
        }
      }
      if (!st.next) break;
    }
    if constexpr (!kTangent) {
      w = w / (float)P.spp;
      if (w == 0.0f || !isfinite(w)) return;
      GradSink sk{dpos, nullptr, nullptr, nullptr, nullptr};
      scatter_xdn(S, tri_e, its.p, p, n, w, &ed, t, ed.f0, tri_s, us, vs, sk);
    }
  });
}

hipError_t launch_guide_build(const SceneDev& S, const LaunchCfg& L, uint32_t seed, const GuideDev& g,
                              hipStream_t st) {
  const LaunchCfg Lg = fit_grid(k_guide_eval, L);
  if (Lg.tiles) {
    const hipError_t z = launch_fill_zero(reinterpret_cast<float*>(Lg.tiles), kTileSet, st);
    if (z != hipSuccess) return z;
  }
  hipLaunchKernelGGL(k_guide_eval, dim3(Lg.grid), dim3(kBlock), 0, st, S, Lg, seed, g);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int n = g.n, nc = (n + kSumChunk - 1) / kSumChunk;
  const int gl = (n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096;  // grid over leaves
  float* total = g.part + nc;
  hipLaunchKernelGGL(k_guide_poly, dim3(gl), dim3(256), 0, st, g);
  hipLaunchKernelGGL(k_chunk_sums, dim3(nc), dim3(64), 0, st, g.poly, n, g.part);
  hipLaunchKernelGGL(k_chunk_scan, dim3(1), dim3(64), 0, st, g.part, nc);
  hipLaunchKernelGGL(k_guide_weights, dim3(gl), dim3(256), 0, st, S.sec.cdf, g, total);
  hipLaunchKernelGGL(k_chunk_sums, dim3(nc), dim3(64), 0, st, g.cdf, n, g.part);
  hipLaunchKernelGGL(k_chunk_scan, dim3(1), dim3(64), 0, st, g.part, nc);
  hipLaunchKernelGGL(k_chunk_prefix, dim3(nc), dim3(64), 0, st, g.cdf, n, g.part, 1.0f / (float)n);
  hipLaunchKernelGGL(k_guide_normalize, dim3(gl), dim3(256), 0, st, g, total);
  hipLaunchKernelGGL(k_guide_normalize_last, dim3(1), dim3(64), 0, st, g);
  return hipGetLastError();
}

// Slots for the survivors of `count` samples: whole groups of 64 in each
// segment; the pixel boundary's blocks of pixels may leave an eighth empty.
static uint64_t queue_slots(int kind, uint64_t count) {
  const uint64_t slots = kind == 1 ? count + count / 8 : count;
  const uint64_t groups = (slots + 63) / 64;
  return (groups + kTileCtrs - 1) / kTileCtrs * kTileCtrs * 64;
}

uint64_t boundary_queue_bytes(int kind, uint64_t n_samples, uint64_t chunk) {
  if (n_samples == 0) return 0;
  const uint64_t nchunk = (n_samples + chunk - 1) / chunk;
  const uint64_t cap = queue_slots(kind, n_samples < chunk ? n_samples : chunk);
  return ((uint64_t)kBndWords * cap + nchunk * kTileSet) * sizeof(uint32_t);
}

template <bool kTangent>
static hipError_t launch_boundary_t(int kind, const SceneDev& S, const CameraDev& C, const BoundaryParams& P,
                                    uint64_t N, const LaunchCfg& L, const EdgeSet& prim, const GuideDev& guide,
                                    const float* dLdI, float* dpos, const float* tpos, float* dimg, void* queue,
                                    uint64_t chunk, hipStream_t st) {
  // select / eval per chunk of samples over one survivor queue;
  // the chunks' counters are cleared by a kernel (no memset node when captured)
  if (!queue) return hipErrorInvalidValue;
  const uint64_t nchunk = (N + chunk - 1) / chunk;
  const uint32_t cap = (uint32_t)queue_slots(kind, N < chunk ? N : chunk);
  uint32_t* buf = (uint32_t*)queue;
  uint32_t* counts = buf + (size_t)kBndWords * cap;
  hipError_t e = launch_fill_zero((float*)counts, nchunk * kTileSet, st);
  for (uint64_t c = 0; c < nchunk && e == hipSuccess; ++c) {
    const uint64_t first = c * chunk, end = first + chunk < N ? first + chunk : N;
    const BndQueue Q{counts + c * kTileSet, buf, cap};
    if (L.tiles && (e = launch_fill_zero(reinterpret_cast<float*>(L.tiles), 2 * kTileSet, st)) != hipSuccess) break;
    if (kind == 0) {
      const LaunchCfg Ls = fit_grid(k_bnd_primary_select, L), Lb = fit_grid(k_bnd_bounces<kRngPrimaryEdge>, L);
      hipLaunchKernelGGL(k_bnd_primary_select, dim3(Ls.grid), dim3(kBlock), 0, st, S, C, P, Ls, prim, first, end, Q);
      hipLaunchKernelGGL(k_bnd_bounces<kRngPrimaryEdge>, dim3(Lb.grid), dim3(kBlock), 0, st, S, P, Lb, Q);
      hipLaunchKernelGGL((k_bnd_scatter<true, kTangent>), dim3(L.grid), dim3(kBlock), 0, st, S, C, P, L, prim, Q, dLdI,
                         dpos, tpos, dimg);
    } else if (kind == 1) {
      const LaunchCfg Ls = fit_grid(k_bnd_pixel_select, L), Lb = fit_grid(k_bnd_bounces<kRngPixelEdge>, L);
      hipLaunchKernelGGL(k_bnd_pixel_select, dim3(Ls.grid), dim3(kBlock), 0, st, S, C, P, Ls, N,
                         path_range(C, first, end - first), Q);
      hipLaunchKernelGGL(k_bnd_bounces<kRngPixelEdge>, dim3(Lb.grid), dim3(kBlock), 0, st, S, P, Lb, Q);
      hipLaunchKernelGGL((k_bnd_scatter<false, kTangent>), dim3(L.grid), dim3(kBlock), 0, st, S, C, P, L, prim, Q, dLdI,
                         dpos, tpos, dimg);
    } else if (kind == 2) {
      const LaunchCfg Ls = fit_grid(k_bnd_direct_select, L), Le = fit_grid(k_bnd_direct_eval<kTangent>, L);
      hipLaunchKernelGGL(k_bnd_direct_select, dim3(Ls.grid), dim3(kBlock), 0, st, S, C, P, Ls, guide, first, end, Q);
      hipLaunchKernelGGL(k_bnd_direct_eval<kTangent>, dim3(Le.grid), dim3(kBlock), 0, st, S, C, P, Le, Q, dLdI, dpos,
                         tpos, dimg);
    } else {
      const LaunchCfg Ls = fit_grid(k_bnd_indirect_select, L), Le = fit_grid(k_bnd_indirect_eval<kTangent>, L);
      hipLaunchKernelGGL(k_bnd_indirect_select, dim3(Ls.grid), dim3(kBlock), 0, st, S, C, P, Ls, first, end, Q);
      hipLaunchKernelGGL(k_bnd_indirect_eval<kTangent>, dim3(Le.grid), dim3(kBlock), 0, st, S, C, P, Le, Q, dLdI,
                         dpos, tpos, dimg);
    }
    e = hipGetLastError();
  }
  return e;
}

hipError_t launch_boundary(int kind, const SceneDev& S, const CameraDev& C, uint32_t seed, int max_bounces, int spp,
                           const LaunchCfg& L, const EdgeSet& prim, const GuideDev& guide, const float* dLdI,
                           float* dpos, const float* tpos, float* dimg, void* queue,
                           uint64_t chunk, hipStream_t st) {
  const BoundaryParams P{seed, max_bounces, spp, 0u};
  const uint64_t N = (uint64_t)spp * (uint64_t)C.width * (uint64_t)C.height;
  if (N == 0) return hipSuccess;
  if (dimg)
    return launch_boundary_t<true>(kind, S, C, P, N, L, prim, guide, nullptr, nullptr, tpos, dimg, queue, chunk, st);
  return launch_boundary_t<false>(kind, S, C, P, N, L, prim, guide, dLdI, dpos, nullptr, nullptr, queue, chunk, st);
}

}  // namespace trc
