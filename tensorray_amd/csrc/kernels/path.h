// Paths of the interior integrator with next-event estimation and MIS.
//
// path_forward evaluates one camera path per thread: the adjoint kernels
// re-evaluate a path from its checkpoint with it (kRecord = true, which stores
// the discrete decisions and throughputs of the path in a small per-thread
// record instead of an expression tape), and k_render_stats counts the work of
// the paths it traces (kRecord = false).  path_bounces is its bounce loop, and
// the indirect boundary term's.  The forward itself runs in two passes over
// waves, trace_primary and render_bounces below.
//
// Reference: PathTracer::Radiance (LibTensorRay/Renderer/PathTracer.cpp:37-76),
// EvalRadianceEmitted (Integrator.cpp:55-73), EvalRadianceDirect
// (Integrator.cpp:178-303), Camera::GenerateAntitheticRays (Camera.cpp:224-277)
// and Camera::EvalFilter (Camera.cpp:279-303).
#pragma once
#include "../common/tr_bsdf.h"
#include "trace.h"

namespace trc {

struct PathParams {
  uint32_t seed;
  int32_t max_bounces;   // B: NEE + BSDF steps after the primary hit
  int32_t spp;
  uint32_t path_offset;  // index of the first path of this launch (spp passes)
};

// Per-path record for replay: hit vertices x_0..x_K, throughputs, light
// samples and the constant (detached) factors of every contribution.
struct PathRec {
  int32_t K;                     // index of the last hit vertex, -1 = camera ray missed
  int32_t tri[kMaxBounces + 1];
  float bu[kMaxBounces + 1], bv[kMaxBounces + 1];
  F3 beta[kMaxBounces + 1];
  F3 e0c;                        // emission at x_0 (constant factor)
  int32_t ltri[kMaxBounces];     // light sample of bounce i
  float lbu[kMaxBounces], lbv[kMaxBounces];
  F3 neec[kMaxBounces];          // valid * Le * mis / pdf_L, zero when unused
  float ppdf[kMaxBounces];       // pdf_bsdf * detach(G) of segment i -> i+1
  F3 emc[kMaxBounces];           // Le * mis at x_{i+1}, zero when not an emitter
  uint32_t tflag;                // bit i: throughput of segment i is nonzero (G > 0)
};

TR_HD F3 nan_to_zero(F3 v) { return finite3(v) ? v : F3{0.0f, 0.0f, 0.0f}; }

// Path checkpoint: the outcome of every ray query of a path, written by the
// forward pass so that the adjoint re-evaluates the path without tracing.
// Per path: meta = (K + 1) | (NEE visibility of bounce b) << (8 + b), where
// K is the last hit vertex (-1: the camera ray missed), and for each vertex
// i <= K the hit triangle and barycentrics.  Fields are [vertex][path]
// planes, so lanes with consecutive paths touch consecutive words.
struct CkptDev {
  uint32_t* meta;   // [npaths]
  int32_t* tri;     // [nv][npaths]
  float* u;         // [nv][npaths]
  float* v;         // [nv][npaths]
  uint64_t npaths;
  int32_t nv;       // max_bounces + 1
};
// 4 bytes of meta + 12 bytes per vertex.
TR_HD uint64_t ckpt_bytes(uint64_t npaths, int max_bounces) {
  return npaths * (4ull + 12ull * (uint64_t)(max_bounces + 1));
}
TR_HD CkptDev ckpt_view(void* base, uint64_t npaths, int max_bounces) {
  CkptDev c;
  const uint64_t nv = (uint64_t)(max_bounces + 1);
  c.meta = (uint32_t*)base;
  c.tri = (int32_t*)(c.meta + npaths);
  c.u = (float*)(c.tri + nv * npaths);
  c.v = c.u + nv * npaths;
  c.npaths = npaths;
  c.nv = (int32_t)nv;
  return c;
}
// The checkpoint of paths first .. first + count alone, in as many bytes as
// ckpt_bytes(count): its planes are addressed by path index like a whole one's.
TR_HD CkptDev ckpt_window(void* base, uint64_t first, uint64_t count, int max_bounces) {
  CkptDev c = ckpt_view(base, count, max_bounces);
  c.meta -= first;
  c.tri -= first;
  c.u -= first;
  c.v -= first;
  return c;
}
__device__ inline void ckpt_put_vertex(const CkptDev& c, uint64_t path, int i, int32_t tri, float u, float v) {
  const uint64_t k = (uint64_t)i * c.npaths + path;
  c.tri[k] = tri;
  c.u[k] = u;
  c.v[k] = v;
}

// Where a path's ray queries come from: the BVH (TraceCtx) or a checkpoint.
__device__ inline Hit src_camera(const SceneDev& S, TraceCtx& tc, F3 o, F3 d) {
  return trace_ray<false>(S, tc, o, d, kShadowEpsilon, 1e32f);
}
__device__ inline bool src_visible(const SceneDev& S, TraceCtx& tc, int b, F3 o, F3 wi, float dist) {
  return trace_ray<true>(S, tc, o, wi, kShadowEpsilon, dist - kShadowEpsilon).tri < 0;
}
__device__ inline Hit src_bsdf(const SceneDev& S, TraceCtx& tc, int b, F3 o, F3 d) {
  return trace_ray<false>(S, tc, o, d, kShadowEpsilon, 1e32f);
}

struct CkptSrc {
  const CkptDev* c;
  uint64_t path;
  uint32_t meta;
  __device__ Hit vertex(int i) const {
    Hit h;
    const int K = (int)(meta & 0xFFu) - 1;
    if (i > K) {
      h.tri = -1; h.u = 0.0f; h.v = 0.0f; h.t = -1.0f;
      return h;
    }
    const uint64_t k = (uint64_t)i * c->npaths + path;
    h.tri = c->tri[k];
    h.u = c->u[k];
    h.v = c->v[k];
    h.t = 0.0f;
    return h;
  }
};
__device__ inline Hit src_camera(const SceneDev&, CkptSrc& s, F3, F3) { return s.vertex(0); }
__device__ inline bool src_visible(const SceneDev&, CkptSrc& s, int b, F3, F3, float) {
  return ((s.meta >> (8 + b)) & 1u) != 0u;
}
__device__ inline Hit src_bsdf(const SceneDev&, CkptSrc& s, int b, F3, F3) { return s.vertex(b + 1); }

// Bounce loop (PathTracer.cpp:55-73, EvalRadianceDirect Integrator.cpp:178-303)
// from surface point `its` reached along `raydir` with throughput `beta`.
// Bounce b draws blocks block0 + 2b (light) and block0 + 2b + 1 (BSDF) of
// (seed, domain, index).  kRecord fills the replay record (interior
// adjoint); kPerBounce stores each executed bounce's contribution.
template <bool kRecord, bool kPerBounce, class Src>
__device__ void path_bounces(const SceneDev& S, Src& tc, Its its, F3 beta, F3 raydir, uint32_t seed,
                             uint32_t domain, uint64_t index, uint32_t block0, int B, F3& contrib, PathRec* R,
                             F3* per_bounce) {
  const F3 zero{0.0f, 0.0f, 0.0f};
  for (int b = 0; b < B; ++b) {
    Rnd4 rl = rng4(seed, domain, index, block0 + 2u * (uint32_t)b);
    Rnd4 rb = rng4(seed, domain, index, block0 + 2u * (uint32_t)b + 1u);
    F3 ret = zero;
    F3 wo = -raydir;
    // ---- next-event estimation ----
    LightSample ls = light_sample(S, rl.a, rl.b);
    F3 neec = zero;
    {
      F3 wi = ls.p - its.p;
      float d2 = len2(wi);
      float dist;
      wi = over_sqrt(wi, d2, &dist);
      float dsh = dot(its.ns, wi), dgeo = dot(its.ng, wi);
      bool stable = dist > kShadowEpsilon && fabsf(dsh) > kEdgeEpsilon;
      bool noleak = (dsh * dgeo) > 0.0f;
      bool visible = false;
      if (stable && noleak) visible = src_visible(S, tc, b, its.p, wi, dist);
      float valid = (stable && noleak && visible) ? 1.0f : 0.0f;
      float Gl = fabsf(dot(ls.n, -wi)) / d2;
      float pbs;
      F3 f = bsdf_eval_pdf(S, its, wo, wi, &pbs) * fabsf(dsh);
      F3 Le = emitted(S, ls.emitter, ls.n, -wi);
      float JL = ratio_self(S.shade[ls.tri].area);
      F3 val = valid * beta * f * JL * Gl * Le / ls.pdf;
      float pb = pbs * Gl;
      float mis = (ls.pdf * ls.pdf) / (ls.pdf * ls.pdf + pb * pb);
      val = val * mis;
      ret = ret + val;
      if (kRecord) neec = valid * Le / ls.pdf * mis;
    }
    if (kRecord) {
      R->ltri[b] = ls.tri; R->lbu[b] = ls.bu; R->lbv[b] = ls.bv;
      R->neec[b] = neec;
      R->emc[b] = zero;
    }
    // ---- BSDF sampling ----
    float pdfb;
    F3 wib = bsdf_sample(S, its, wo, rb.a, rb.b, &pdfb);
    Hit h2 = src_bsdf(S, tc, b, its.p, wib);
    bool ok = h2.tri >= 0 && pdfb > 0.0f && bsdf_dir_valid(S, its, wib);
    if (!ok) {
      if (finite3(ret)) {
        contrib = contrib + ret;
        if (kPerBounce) per_bounce[b] = ret;
      } else if (kRecord) {
        R->neec[b] = zero;
      }
      break;
    }
    Its its2 = post_intersect(S, h2.tri, h2.u, h2.v);
    F3 dd = its2.p - its.p;
    float dd2 = len2(dd);
    float dl;
    F3 nd = over_sqrt(dd, dd2, &dl);
    float G2 = fabsf(dot(its2.ng, -nd)) / dd2;
    F3 f2 = bsdf_eval(S, its, wo, nd) * fabsf(dot(its.ns, nd));
    float ppdf = pdfb * G2;
    float J2 = ratio_self(S.shade[its2.tri].area);
    F3 beta2 = beta * f2 * G2 * J2 / ppdf;
    bool gpos = G2 > 0.0f;
    if (!gpos) beta2 = zero;
    F3 emc = zero;
    if (its2.emitter >= 0) {
      F3 Le2 = emitted(S, its2.emitter, its2.ng, -nd);
      F3 val2 = beta2 * Le2;
      float pn = light_pdf_tri(S, its2.tri);
      float mis2 = (ppdf * ppdf) / (ppdf * ppdf + pn * pn);
      val2 = val2 * mis2;
      ret = ret + val2;
      emc = Le2 * mis2;
    }
    bool fin = finite3(ret);
    if (fin) {
      contrib = contrib + ret;
      if (kPerBounce) per_bounce[b] = ret;
    }
    if (kRecord) {
      if (!fin) { R->neec[b] = zero; emc = zero; }
      R->emc[b] = emc;
      R->ppdf[b] = ppdf;
      if (gpos) R->tflag |= 1u << b;
      R->K = b + 1;
      R->tri[b + 1] = its2.tri; R->bu[b + 1] = h2.u; R->bv[b + 1] = h2.v;
      R->beta[b + 1] = beta2;
    }
    its = its2;
    beta = beta2;
    raydir = nd;
  }
}

template <bool kRecord, class Src>
__device__ F3 path_forward(const SceneDev& S, const CameraDev& C, const PathParams& P, uint64_t path,
                           Src& tc, PathRec* R) {
  const F3 zero{0.0f, 0.0f, 0.0f};
  const uint32_t WH = (uint32_t)C.width * (uint32_t)C.height;
  const uint32_t pix = (uint32_t)(path % WH);
  const uint32_t px = pix % (uint32_t)C.width, py = pix / (uint32_t)C.width;
  if (kRecord) { R->K = -1; R->tflag = 0u; }
  // --- primary ray (box filter: the sample stays inside its pixel) ---
  Rnd4 rc = rng4(P.seed, kRngInterior, path, 0u);
  const F3 eye{C.eye[0], C.eye[1], C.eye[2]};
  const F3 cdir{C.dir[0], C.dir[1], C.dir[2]};
  F3 d0 = camera_dir(C, (float)px + rc.a, (float)py + rc.b);
  Hit h = src_camera(S, tc, eye, d0);
  if (h.tri < 0) return zero;
  Its its = post_intersect(S, h.tri, h.u, h.v);
  // EvalFilter: G / detach(G) with G = |cos_x| / (cos_y^3 d^2); times J
  float beta0;
  F3 raydir;
  {
    F3 cd = its.p - eye;
    float dist;
    cd = over_sqrt(cd, len2(cd), &dist);
    raydir = cd;
    float cosy = dot(cd, cdir);
    float cosx = dot(-cd, its.ng);
    float G = fabsf(cosx) / (cosy * cosy * cosy * (dist * dist));
    beta0 = ratio_self(G) * ratio_self(S.shade[its.tri].area);
  }
  F3 beta{beta0, beta0, beta0};
  F3 contrib = zero;
  F3 e0c = zero;
  if (its.emitter >= 0) {
    F3 Le = emitted(S, its.emitter, its.ng, -raydir);
    F3 e0 = beta * Le;
    if (finite3(e0)) { contrib = contrib + e0; e0c = Le; }
  }
  if (kRecord) {
    R->K = 0;
    R->tri[0] = its.tri; R->bu[0] = h.u; R->bv[0] = h.v;
    R->beta[0] = beta;
    R->e0c = e0c;
  }
  path_bounces<kRecord, false>(S, tc, its, beta, raydir, P.seed, kRngInterior, path, 1u, P.max_bounces, contrib,
                               R, nullptr);
  return contrib;
}

// ---------------------------------------------------------------------------
// Forward paths in two passes.
//
// The primary pass (trace_primary) traces the camera rays of 64 neighbouring
// paths per wave and leaves each path's first hit where its radiance will go.
// The bounce pass (render_bounces) runs the surviving paths as a per-lane
// state machine with path regeneration: each loop iteration traces the two
// rays of a bounce per lane (the NEE shadow ray, then the BSDF-sampled ray, as
// one chained query from the vertex) and shades the lanes whose query has
// finished; a lane whose path ends takes the next surviving path of its
// wave's tiles and joins the others at the next bounce's set-up.  A query
// that is still running when most of the wave's have finished keeps its
// traversal state and continues in the next iteration.  Each path evaluates
// the same expressions in the same order as path_forward<false>, so the
// per-path radiance is identical.
//
// One pass whose lanes trace either a camera ray or a bounce shades both
// kinds in every iteration, each at the lanes of its kind (about half), and
// carries the camera rays that miss.
// ---------------------------------------------------------------------------
enum PathStage : uint32_t { kStageIdle = 0, kStageBounce = 1 };

// Fraction (of 64) of a wave's queries still unfinished at which the wave
// stops traversing and shades the finished ones.
// (closed room / 512 x 512 step / large-mesh step / eight views at 16: 1.25 /
// 3.38 / 5.27 / 1.73 ms, at 20: 1.24 / 3.35 / 5.18 / 1.74, at 24 and 5 waves
// per SIMD: 1.42 / 3.42 / 5.11 / 1.82 against 1.40 / 3.44 / 5.25 / 1.79 at 16)
constexpr int kTraceKeep64 = 20;

struct PathLane {
  uint64_t path;
  // stage (bits 0-1), the bounce's BSDF direction has a nonzero pdf (bit 2),
  // its shadow ray is traced (bit 3), bounce index b (bits 4-31): one register
  uint32_t sb;
  __device__ uint32_t stage() const { return sb & 3u; }
  __device__ uint32_t b() const { return sb >> 4; }
  __device__ void set_stage(uint32_t s) { sb = (sb & ~3u) | s; }
  int32_t tri;           // current vertex x_b
  float u, v;
  F3 beta, raydir, contrib;
  // light sample of bounce b: emitter triangle and squared distance (its
  // direction is d); shading needs nothing else of it, so the sample is not
  // drawn and its geometry not evaluated a second time
  int32_t li;
  float ld2;
  float pdfb;            // pdf of the BSDF direction d2 of bounce b
  // query of this iteration from o (tmin = kShadowEpsilon): the bounce's
  // shadow ray along d (any hit) chained with its BSDF-sampled ray along d2;
  // the traversal state holds the far bound
  F3 o, d, d2;
  TraceState ts;
};

// NEE geometry of bounce b at `its` (Integrator.cpp:196-213).
struct NeeGeo {
  LightSample ls;
  F3 wi;
  float d2, dist, dsh;
  bool ray;  // stable && noleak: a shadow ray is traced
};
__device__ inline NeeGeo nee_geo(const SceneDev& S, const Its& its, float la, float lb) {
  NeeGeo g;
  g.ls = light_sample(S, la, lb);
  F3 wi = g.ls.p - its.p;
  g.d2 = len2(wi);
  g.wi = over_sqrt(wi, g.d2, &g.dist);
  g.dsh = dot(its.ns, g.wi);
  float dgeo = dot(its.ng, g.wi);
  bool stable = g.dist > kShadowEpsilon && fabsf(g.dsh) > kEdgeEpsilon;
  bool noleak = (g.dsh * dgeo) > 0.0f;
  g.ray = stable && noleak;
  return g;
}

// The slots a wave works on: its tiles of `tile` slots of a range of `slots`
// that starts at tile t0 of the launch.  The wave moves to its next tile as
// soon as the current one is handed out, without waiting for its lanes to
// drain.  All fields are wave-uniform.
//
// Tile counters: when set, the wave's tiles after its first (tile t, one per
// wave: tiles 0 .. step-1 of the launch are dealt so) are taken as the wave
// needs one; otherwise t, t + step, ...  One word serves an atomic every
// 11.5 ns (65,536 tiles of 64 paths: 0.755 ms, whatever the paths cost), so
// there are kTileCtrs of them, each in its own cache line, which share the
// tiles evenly; a wave uses that of its block (blocks b and b + 8 run on one
// XCD).  Tile numbers count over the whole launch.
struct TileSupply {
  uint64_t next, end;  // slots not yet handed out of the current tile
  uint64_t t, tend, step;
  uint64_t t0, slots;
  uint32_t tile;
  uint32_t q, nq;      // the wave's counter and how many there are
  uint32_t* ctr;
  __device__ void load() {
    next = (t - t0) * tile;
    end = next + tile < slots ? next + tile : slots;
  }
  // Starts at tile t; ctr: the launch's counters or null.
  __device__ static TileSupply make(uint64_t t, uint64_t step, uint64_t t0, uint64_t slots, uint32_t tile,
                                    uint32_t* ctr) {
    TileSupply s;
    s.t = t;
    s.step = step;
    s.t0 = t0;
    s.slots = slots;
    s.tile = tile;
    s.tend = t0 + (slots + tile - 1) / tile;
    s.nq = gridDim.x < (uint32_t)kTileCtrs ? 1u : (uint32_t)kTileCtrs;
    s.q = blockIdx.x % s.nq;
    s.ctr = ctr ? ctr + s.q * (uint32_t)kTileCtrStride : nullptr;
    if (t < s.tend) s.load();
    else s.next = s.end = 0;
    return s;
  }
  // Moves to the wave's next tile; false (and an empty range) when none is
  // left, in which case t stays at the first tile past tend.
  __device__ bool more() {
    if (t >= tend) {
      next = end;
      return false;
    }
    t = next_tile();
    if (t >= tend) {
      next = end;
      return false;
    }
    load();
    return true;
  }
  // The number of the wave's next tile.
  __device__ uint64_t next_tile() const {
    if (!ctr) return t + step;
    uint32_t v = 0u;
    if ((threadIdx.x & 63u) == 0u) v = atomicAdd(ctr, 1u);
    return step + (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)v) * nq + q;
  }
};

// The first hit of a path between the passes, in the three words of its
// radiance: (triangle + 1, u, v); zero for a camera ray that missed, whose
// radiance that is.
__device__ inline void put_first_hit(float* w, const Hit& h) {
  w[0] = __uint_as_float((uint32_t)(h.tri + 1));
  w[1] = h.u;
  w[2] = h.v;
}

// 64 slots of a range.  All fields are wave-uniform.
struct PathGroup {
  uint64_t base;     // path of offset 0
  uint32_t cols, rows;  // blocked: pixels of the block inside the image; else cols = paths, rows = 0
  uint32_t width;
  __device__ static PathGroup linear(uint64_t first, uint64_t end) {
    PathGroup g;
    g.base = first;
    g.cols = end - first < 64u ? (uint32_t)(end - first) : 64u;
    g.rows = 0u;
    g.width = 0u;
    return g;
  }
  // block `k` of the blocks of all samples from path `first` on (a multiple of W * H)
  __device__ static PathGroup block(const CameraDev& C, uint64_t first, uint64_t k) {
    const uint32_t W = (uint32_t)C.width, H = (uint32_t)C.height;
    const uint32_t bx = (W + 7u) / 8u, nb = bx * ((H + 7u) / 8u);
    const uint64_t s = k / nb;
    const uint32_t r = (uint32_t)(k - s * nb), by = r / bx, x = (r - by * bx) * 8u, y = by * 8u;
    PathGroup g;
    g.base = first + s * ((uint64_t)W * H) + (uint64_t)y * W + x;
    g.cols = W - x < 8u ? W - x : 8u;
    g.rows = H - y < 8u ? H - y : 8u;
    g.width = W;
    return g;
  }
  // the group of slots i .. i + 63 (i a multiple of 64)
  __device__ static PathGroup at(const CameraDev& C, const PathRange& R, uint64_t i) {
    return R.blocked ? block(C, R.first, i >> 6) : linear(R.first + i, R.first + R.count);
  }
  __device__ bool has(uint32_t j) const { return rows ? (j & 7u) < cols && (j >> 3) < rows : j < cols; }
  __device__ uint64_t path(uint32_t j) const { return base + (rows ? (j >> 3) * width + (j & 7u) : j); }
};

// The primary pass over one group: camera rays of the box filter (the sample
// stays inside its pixel) and first hits, from the group's 64 lanes at once.
// `paths` points at the words of path `paths_first`.  mask: dL/dI or null; the
// paths of pixels where it is zero are not traced and count as missed.
template <bool kCkpt>
__device__ inline void trace_primary(const SceneDev& S, const CameraDev& C, const PathParams& P, TraceCtx& tc, const PathGroup& g,
                                     const CkptDev& ck, float* paths, uint64_t paths_first, const float* mask = nullptr) {
  const uint32_t lane = threadIdx.x & 63u;
  const bool has = g.has(lane);
  const uint64_t path = has ? g.path(lane) : g.base;
  const uint32_t pix = (uint32_t)(path % ((uint32_t)C.width * (uint32_t)C.height));
  const uint32_t px = pix % (uint32_t)C.width, py = pix / (uint32_t)C.width;
  const Rnd4 rc = rng4(P.seed, kRngInterior, path, 0u);
  const F3 eye{C.eye[0], C.eye[1], C.eye[2]};
  const F3 d = camera_dir(C, (float)px + rc.a, (float)py + rc.b);
  const uint32_t wh = (uint32_t)C.width * (uint32_t)C.height;
  const bool traced = has && (!mask || mask[pix] != 0.0f || mask[wh + pix] != 0.0f || mask[2 * wh + pix] != 0.0f);
  TraceState ts;
  if (traced) trace_begin(ts, 1e32f);
  else trace_none(ts);
  trace_run<true>(S, tc, eye, d, d, 1e32f, kShadowEpsilon, false, ts, 0);
  const Hit h = trace_hit(ts);
  if (!has) return;
  put_first_hit(paths + 3 * (path - paths_first), h);
  if (kCkpt) {
    ck.meta[path] = h.tri < 0 ? 0u : 1u;
    if (h.tri >= 0) ckpt_put_vertex(ck, path, 0, h.tri, h.u, h.v);
  }
}

// The BSDF-sampled ray of bounce b from `its` came back with hit `h`:
// MIS-weighted emission, throughput update and the move to the next vertex,
// or the end of the path (Integrator.cpp:232-293).  ret: the bounce's NEE
// contribution.  Returns true when the path continues from the new vertex
// x_{b+1} (L.tri, L.u, L.v).
template <bool kCkpt, class Finish>
__device__ inline bool bsdf_hit(const SceneDev& S, int max_bounces, const CkptDev& ck, const Its& its, F3 wo,
                                const Hit& h, F3 ret, PathLane& L, uint32_t& meta, Finish& finish) {
  const F3 zero{0.0f, 0.0f, 0.0f};
  bool ok = h.tri >= 0 && L.pdfb > 0.0f && bsdf_dir_valid(S, its, L.d2);
  if (!ok) {
    if (finite3(ret)) L.contrib = L.contrib + ret;
    if (kCkpt) ck.meta[L.path] = meta;
    finish(L.path, L.contrib);
    L.set_stage(kStageIdle);
    return false;
  }
  Its its2 = post_intersect(S, h.tri, h.u, h.v);
  F3 dd = its2.p - its.p;
  float dd2 = len2(dd);
  float dl;
  F3 nd = over_sqrt(dd, dd2, &dl);
  float G2 = fabsf(dot(its2.ng, -nd)) / dd2;
  F3 f2 = bsdf_eval(S, its, wo, nd) * fabsf(dot(its.ns, nd));
  float ppdf = L.pdfb * G2;
  float J2 = ratio_self(S.shade[its2.tri].area);
  F3 beta2 = L.beta * f2 * G2 * J2 / ppdf;
  if (!(G2 > 0.0f)) beta2 = zero;
  if (its2.emitter >= 0) {
    F3 Le2 = emitted(S, its2.emitter, its2.ng, -nd);
    F3 val2 = beta2 * Le2;
    float pn = light_pdf_tri(S, its2.tri);
    float mis2 = (ppdf * ppdf) / (ppdf * ppdf + pn * pn);
    val2 = val2 * mis2;
    ret = ret + val2;
  }
  if (finite3(ret)) L.contrib = L.contrib + ret;
  L.tri = h.tri; L.u = h.u; L.v = h.v;
  L.beta = beta2;
  L.raydir = nd;
  L.sb += 16u;  // b + 1
  if (kCkpt) {
    ckpt_put_vertex(ck, L.path, (int)L.b(), h.tri, h.u, h.v);
    meta += 1u;
  }
  if ((int)L.b() >= max_bounces) {
    if (kCkpt) ck.meta[L.path] = meta;
    finish(L.path, L.contrib);
    L.set_stage(kStageIdle);
    return false;
  }
  return true;
}

// The camera paths of the interior integrator as a source of the bounce pass:
// slots count the launch's order of paths R, first hits lie in `paths`.
struct CameraPaths {
  const CameraDev& C;
  const PathRange& R;
  const float* paths;
  uint64_t paths_first;
  PathGroup group;
  static constexpr uint32_t kDomain = kRngInterior;
  // takes the group of slots i .. i + 63: whether the calling lane's survives
  __device__ bool open(uint64_t i, uint32_t lane) {
    group = PathGroup::at(C, R, i);
    return group.has(lane) && __float_as_uint(paths[3 * (group.path(lane) - paths_first)]) != 0u;
  }
  // path of the group's offset
  __device__ uint64_t path(uint32_t off) const { return group.path(off); }
  __device__ uint64_t rng_index(uint64_t path) const { return path; }
  __device__ void first_hit(PathLane& L) const {
    const float* w = paths + 3 * (L.path - paths_first);
    L.tri = (int32_t)(__float_as_uint(w[0]) - 1u);
    L.u = w[1];
    L.v = w[2];
  }
  // direction to and throughput at the first vertex (Integrator.cpp:55-73)
  __device__ void first_vertex(const SceneDev& S, const Its& its, PathLane& L) const {
    const F3 eye{C.eye[0], C.eye[1], C.eye[2]};
    const F3 cdir{C.dir[0], C.dir[1], C.dir[2]};
    F3 cd = its.p - eye;
    float dist;
    cd = over_sqrt(cd, len2(cd), &dist);
    L.raydir = cd;
    float cosy = dot(cd, cdir);
    float cosx = dot(-cd, its.ng);
    float G = fabsf(cosx) / (cosy * cosy * cosy * (dist * dist));
    const float beta0 = ratio_self(G) * ratio_self(S.shade[its.tri].area);
    L.beta = F3{beta0, beta0, beta0};
  }
};

// The bounce pass: the wave renders the surviving paths of its tile supply,
// which counts slots of the source (camera paths, or the survivors of a
// boundary term's selection).  A bounce is two ray queries, the shadow ray of
// next-event estimation and the BSDF-sampled ray, traced as one chained query
// and shaded together.
template <bool kCkpt, class Source, class Finish>
__device__ void render_bounces(const SceneDev& S, Source src, uint32_t seed, int max_bounces, TraceCtx& tc,
                               TileSupply& sup, const CkptDev& ck, Finish finish) {
  const F3 zero{0.0f, 0.0f, 0.0f};
  const uint32_t lane = threadIdx.x & 63u;
  PathLane L;
  L.sb = kStageIdle;
  trace_none(L.ts);
  uint32_t meta = 0u;  // checkpoint meta word of the current path
  // the current group's surviving paths, not yet handed out from `pool_next`
  // on: lane r holds the offset of the r-th
  uint32_t pool = 0u, pool_next = 0u, pool_n = 0u;
  for (;;) {
    // ---- one chained query per lane ----
    // The wave leaves the traversal loop once at most kTraceKeep64 / 64 of
    // its queries are unfinished; those lanes skip shading and resume their
    // query in the next iteration, beside the new rays of the others.
    // (a BSDF direction of pdf 0 ends the path whatever it hits: its query
    // is given an empty interval)
    trace_run<true>(S, tc, L.o, L.d, L.d2, (L.sb & 4u) ? 1e32f : -1.0f, kShadowEpsilon, true, L.ts, kTraceKeep64);
    bool setup = false;  // the lane stands at a vertex whose bounce is to be set up
    if (L.stage() == kStageBounce && trace_finished(L.ts)) {
      // ---- shade: next-event estimation of bounce b (Integrator.cpp:196-230)
      // with the traced shadow ray's outcome, then the BSDF-sampled ray's hit
      const Hit h = trace_hit(L.ts);
      const Its its = post_intersect(S, L.tri, L.u, L.v);
      const F3 wo = -L.raydir;
      const TriShade& lsh = S.shade[S.light_tri[L.li]];
      const F3 ln{lsh.n[0], lsh.n[1], lsh.n[2]};
      const float lpdf = S.light_pdf[L.li];
      const F3 wi = L.d;
      bool visible = (L.sb & 8u) != 0u && !trace_first_hit(L.ts);
      if (kCkpt && visible) meta |= 1u << (8u + L.b());
      float valid = visible ? 1.0f : 0.0f;
      float Gl = fabsf(dot(ln, -wi)) / L.ld2;
      float pbs;
      F3 f = bsdf_eval_pdf(S, its, wo, wi, &pbs) * fabsf(dot(its.ns, wi));
      F3 Le = emitted(S, lsh.emitter, ln, -wi);
      float JL = ratio_self(lsh.area);
      F3 val = valid * L.beta * f * JL * Gl * Le / lpdf;
      float pb = pbs * Gl;
      float mis = (lpdf * lpdf) / (lpdf * lpdf + pb * pb);
      val = val * mis;
      F3 ret = zero;
      ret = ret + val;
      setup = bsdf_hit<kCkpt>(S, max_bounces, ck, its, wo, h, ret, L, meta, finish);
    }
    // ---- regenerate: idle lanes take the next surviving paths ----
    const uint64_t idle_mask = __builtin_amdgcn_ballot_w64(L.stage() == kStageIdle);
    if (idle_mask != 0ull) {
      while (pool_next == pool_n) {
        if (sup.next >= sup.end && !sup.more()) break;
        const bool live = src.open(sup.next, lane);
        sup.next += 64u;
        const uint64_t m = __builtin_amdgcn_ballot_w64(live);
        // lane r of the list: the r-th live lane (dead lanes write behind it)
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        pool_n = (uint32_t)__popcll(m);
        pool_next = 0u;
        pool = (uint32_t)__builtin_amdgcn_ds_permute((int)((live ? below : pool_n + lane - below) << 2), (int)lane);
      }
      const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(idle_mask >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)idle_mask, 0u));
      const uint32_t off = (uint32_t)__shfl((int)pool, (int)((pool_next + rank) & 63u));
      const bool take = L.stage() == kStageIdle && pool_next + rank < pool_n;
      const uint32_t n_idle = (uint32_t)__popcll(idle_mask);
      pool_next = pool_next + n_idle < pool_n ? pool_next + n_idle : pool_n;
      if (take) {
        L.path = src.path(off);
        src.first_hit(L);
        L.sb = kStageBounce;  // b = 0
        meta = 1u;
        setup = true;
      }
      if (__builtin_amdgcn_ballot_w64(L.stage() != kStageIdle) == 0ull) break;  // the supply is used up
    }
    if (setup) {
      // The vertex is evaluated here, once for the lanes that continue and
      // those that start, rather than kept from the shading above: its
      // frame would be live through the hand-out.
      const Its its = post_intersect(S, L.tri, L.u, L.v);
      if (L.b() == 0u) {
        src.first_vertex(S, its, L);
        L.contrib = zero;
        if (its.emitter >= 0) {
          F3 Le = emitted(S, its.emitter, its.ng, -L.raydir);
          F3 e0 = L.beta * Le;
          if (finite3(e0)) L.contrib = L.contrib + e0;
        }
      }
      if (max_bounces <= 0) {
        // no bounce: the path ends at its first vertex, and the lane takes
        // another one in the next iteration
        if (kCkpt) ck.meta[L.path] = meta;
        finish(L.path, L.contrib);
        L.set_stage(kStageIdle);
        trace_none(L.ts);
        continue;
      }
      // ---- bounce b at `its`: light sample, shadow ray and BSDF direction ----
      // (Integrator.cpp:196-213 and 232-245; the draws of the reference's
      // loop in its order: light sample 1 + 2b, BSDF sample 2 + 2b)
      const uint64_t index = src.rng_index(L.path);
      const Rnd4 rl = rng4(seed, Source::kDomain, index, 1u + 2u * L.b());
      const NeeGeo g2 = nee_geo(S, its, rl.a, rl.b);
      L.li = g2.ls.index;
      L.ld2 = g2.d2;
      const Rnd4 rb = rng4(seed, Source::kDomain, index, 1u + 2u * L.b() + 1u);
      L.d2 = bsdf_sample(S, its, -L.raydir, rb.a, rb.b, &L.pdfb);
      L.sb = (L.sb & ~15u) | kStageBounce | (L.pdfb > 0.0f ? 4u : 0u) | (g2.ray ? 8u : 0u);
      L.o = its.p;
      L.d = g2.wi;
      trace_begin_chain(L.ts, g2.ray ? g2.dist - kShadowEpsilon : -1.0f);
    }
    // a lane without a path or query must not look live to the traversal
    if (L.stage() == kStageIdle) trace_none(L.ts);
  }
}

}  // namespace trc
