// Ray queries against the 4-wide BVH: watertight FP32 ray/triangle test and
// closest-hit / any-hit traversal with a short stack in LDS that spills to a
// per-thread HBM slice only when a path is deeper than the LDS part.
//
// Replaces RayIntersectOptix (LibTensorRay/Renderer/Optix.cpp:252-305) and
// the OptiX programs __raygen__/__miss__/__closesthit__ (ptx.cu:61-113).
// Hit record semantics follow ptx.cu:92-113: a miss has tri = -1, u = v = 0,
// t = -1; barycentrics (u, v) weight vertices 1 and 2.
#pragma once
#include "../common/tr_layout.h"

namespace trc {

// Ray precomputation of the watertight test (Woop, Benthin, Wald, "Watertight
// Ray/Triangle Intersection", JCGT 2(1), 2013): kz is the dominant axis of
// the direction, kx / ky the two after it, S the shear constants.  The paper
// swaps kx and ky when d[kz] < 0 to keep the winding; that only flips the
// signs of U, V, W, of det and of T, so (t, u, v) are the same bits without
// it (but for the sign of a zero u or v, where the ray meets an edge), and the
// test below accepts either winding.
struct RayPre {
  F3 o;
  int kz;
  float Sx, Sy, Sz;
};

TR_HD int ray_major(F3 d) {
  float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
  return (ax >= ay && ax >= az) ? 0 : (ay >= az ? 1 : 2);
}
// v rotated so that axis kz comes last.
TR_HD F3 rotate_to(F3 v, int kz) {
  return F3{kz == 2 ? v.x : (kz == 0 ? v.y : v.z), kz == 2 ? v.y : (kz == 0 ? v.z : v.x),
            kz == 2 ? v.z : (kz == 0 ? v.x : v.y)};
}

TR_HD RayPre ray_pre(F3 o, F3 d) {
  RayPre r;
  r.o = o;
  r.kz = ray_major(d);
  const F3 k = rotate_to(d, r.kz);
  r.Sx = k.x / k.z;
  r.Sy = k.y / k.z;
  r.Sz = 1.0f / k.z;
  return r;
}

// Watertight test.  Returns true and (t, u, v) when the ray's line crosses
// the triangle (edges included, degenerate triangles excluded); the caller
// applies the (tmin, tmax) interval.
TR_HD bool tri_intersect(const RayPre& r, F3 p0, F3 p1, F3 p2, float* t_out, float* u_out,
                         float* v_out) {
  const F3 A = rotate_to(p0 - r.o, r.kz), B = rotate_to(p1 - r.o, r.kz), C = rotate_to(p2 - r.o, r.kz);
  float Ax = A.x - r.Sx * A.z;
  float Ay = A.y - r.Sy * A.z;
  float Bx = B.x - r.Sx * B.z;
  float By = B.y - r.Sy * B.z;
  float Cx = C.x - r.Sx * C.z;
  float Cy = C.y - r.Sy * C.z;
  float U = Cx * By - Cy * Bx;
  float V = Ax * Cy - Ay * Cx;
  float W = Bx * Ay - By * Ax;
  if (U == 0.0f || V == 0.0f || W == 0.0f) {
    // edge case: redo the 2-D edge functions in double precision
    U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
    V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
    W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
  }
  if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
  float det = U + V + W;
  if (det == 0.0f) return false;
  float Az = r.Sz * A.z, Bz = r.Sz * B.z, Cz = r.Sz * C.z;
  float T = U * Az + V * Bz + W * Cz;
  float inv = 1.0f / det;
  *t_out = T * inv;
  *u_out = V * inv;
  *v_out = W * inv;
  return true;
}

struct Hit {
  int32_t tri;
  float u, v, t;
};

// Slab test against the quantized planes, in units of the tree's scale (all
// scalings are by powers of two).  With i = rcp(d) along an axis, the plane at
// offset h from the node's origin g is met at t = (g + h - o) i, evaluated as
// fma(h, i, b) over b = (g - o) i.  In units of e = 2^-24: i is off by at
// most 2 e (v_rcp_f32), b by 2 e more relative to (g - o) / d, and the fma
// rounds once, so t is off by at most 3 e |h i| + 5 e |b| (+ second order).
// The stored offsets are widened by 16 e of themselves; kSlabWiden (8 e)
// moves b towards the ray's start for near planes and away for far ones, its
// own rounding included: rounding never culls a box the exact ray enters.
constexpr float kSlabWiden = 4.76837158203125e-7f;

// 1 / d to within an ulp; a direction component of (nearly) zero counts as 1e-30.
__device__ inline float slab_rcp(float d) {
  return fabsf(d) > 1e-30f ? __builtin_amdgcn_rcpf(d) : (d >= 0.0f ? 1e30f : -1e30f);
}

// The half-precision number in the low (i = 0) or high (i = 1) half of w; an
// fma on it becomes one v_fma_mix_f32.
__device__ inline float half_of(uint32_t w, uint32_t i) {
  typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
  return (float)__builtin_bit_cast(half2_t, w)[i];
}

// Per-thread traversal context: the LDS part of the stack (kStackLds entries,
// stride kBlock: lane-interleaved so consecutive lanes use consecutive banks)
// and an HBM spill slice for deeper entries.
struct TraceCtx {
  uint32_t* lds;        // &lds_stack[threadIdx.x]
  uint32_t* leafq;      // postponed-leaf queue of this lane (kLeafQueue entries)
  uint32_t* spill;      // the grid's spill buffer [depth][grid threads] (wave-uniform)
  int spill_stride;     // total threads of the grid
  int cap;              // total stack capacity (kStackLds + spill depth)
  // this lane's result slots in LDS for the wave-wide leaf tests of
  // trace_run<true> (best hit key, its barycentrics); null where unused
  unsigned long long* slot_key;
  float2* slot_uv;
  // work counters (node visits, triangle tests, queries); read only by the
  // statistics kernel, otherwise dead code
  uint32_t n_nodes, n_tris, n_queries;
};

// This thread's column of the spill buffer, computed where it is used so
// that no per-lane pointer stays live through the traversal.
__device__ inline uint32_t spill_lane() { return blockIdx.x * (uint32_t)kBlock + threadIdx.x; }

// The stack's LDS part through an LDS pointer: a load that is either from
// LDS or from the spill buffer would otherwise become one flat load, which
// waits on both memories for every entry popped.
typedef __attribute__((address_space(3))) uint32_t lds_u32;
__device__ inline lds_u32* lds_ptr(uint32_t* p) { return (lds_u32*)p; }

__device__ inline void stack_push(TraceCtx& c, int& sp, uint32_t v) {
  if (sp < kStackLds) lds_ptr(c.lds)[sp * kBlock] = v;
  else c.spill[(size_t)(sp - kStackLds) * c.spill_stride + spill_lane()] = v;
  ++sp;
}
__device__ inline uint32_t stack_pop(TraceCtx& c, int& sp) {
  --sp;
  if (sp < kStackLds) return lds_ptr(c.lds)[sp * kBlock];
  return c.spill[(size_t)(sp - kStackLds) * c.spill_stride + spill_lane()];
}

__device__ inline F3 tri_vertex(const float* v) { return F3{v[0], v[1], v[2]}; }

// State of one ray query between calls of trace_run.  The stack and the
// postponed-leaf queue stay in LDS (and the spill slice) meanwhile, so a
// wave can leave the traversal loop with some lanes unfinished, give its
// finished lanes new rays, and continue all of them together.
struct TraceState {
  float best_t, u, v;  // closest accepted hit so far (t, barycentrics)
  uint32_t best_id;    // its triangle, kNoHit if none
  uint32_t node;       // next inner node to visit
  uint32_t bits;       // stack depth (bits 0-7), queued leaves (8-11), inner_done (12), found (13),
                       // chain (14), second (15), first query hit (16)
};
constexpr uint32_t kNoHit = 0xFFFFFFFFu;
constexpr uint32_t kNoChild = 0xFFFFFFFFu;  // sort key of a child slot without a hit inner child
constexpr uint32_t kTsInnerDone = 1u << 12;
constexpr uint32_t kTsFound = 1u << 13;
// A chained pair of queries from one origin: an any-hit query (a shadow
// ray) and then a closest-hit query in a second direction.  kTsChain: the
// second query is still to start; kTsSecond: the current query is the
// second; kTsFirstHit: the first query found a hit.
constexpr uint32_t kTsChain = 1u << 14;
constexpr uint32_t kTsSecond = 1u << 15;
constexpr uint32_t kTsFirstHit = 1u << 16;
constexpr uint32_t kTsKeep = kTsChain | kTsSecond | kTsFirstHit;  // bits carried across trace_run calls

// A new query with far bound tmax.
__device__ inline void trace_begin(TraceState& s, float tmax) {
  s.best_t = tmax;
  s.u = 0.0f;
  s.v = 0.0f;
  s.best_id = kNoHit;
  s.node = 0u;
  s.bits = 0u;
}
// A chained pair: the any-hit query with far bound tmax, then the
// closest-hit query (trace_run's d and d2, tmax2).
__device__ inline void trace_begin_chain(TraceState& s, float tmax) {
  trace_begin(s, tmax);
  s.bits = kTsChain;
}
// No query (a lane without a ray): finished and missed.
__device__ inline void trace_none(TraceState& s) {
  s.best_id = kNoHit;
  s.bits = kTsInnerDone;
}
// The query (or both of a chained pair) has finished: no inner node left,
// no leaf queued, no chained query to start.
__device__ inline bool trace_finished(const TraceState& s) {
  return (s.bits & (kTsInnerDone | 0xF00u | kTsChain)) == kTsInnerDone;
}
// Of a finished chained pair: whether the first (any-hit) query hit.
__device__ inline bool trace_first_hit(const TraceState& s) { return (s.bits & kTsFirstHit) != 0u; }
// Hit record of a finished query (ptx.cu:92-113 semantics).
__device__ inline Hit trace_hit(const TraceState& s) {
  Hit h;
  if (s.best_id != kNoHit) {
    h.tri = (int32_t)s.best_id;
    h.u = s.u;
    h.v = s.v;
    h.t = s.best_t;
  } else {
    h.tri = -1;
    h.u = 0.0f;
    h.v = 0.0f;
    h.t = -1.0f;
  }
  return h;
}

// Stalled lanes (queue full, or no inner node left with leaves queued), in
// 64ths of the live lanes, at which trace_run<true> tests the queued leaves.
constexpr int kWaveStall64 = 16;
// Lanes with leaves queued, in 64ths of the live lanes, at which it does.
constexpr int kWavePend64 = 48;

// Leaf tests of the whole wave at once.  The queued leaves of all 64 lanes
// form one list (lane by lane, in queue order), dealt round-robin over the
// lanes: lane j tests items j, j + 64, ... against the ray of the item's
// owner, read from the owner's registers, and offers its best hit to the
// owner's slot in LDS with an atomic minimum on the key (t bits, triangle
// id), which orders positive t first and ties by the smaller id, as the
// lane-serial loop does.  The winner of each round also leaves its
// barycentrics in the owner's slot.  So a flush takes ceil(total / 64)
// rounds instead of the longest queue's length, and the hit of every query
// is the one the lane-serial loop finds (closest hit) or a hit inside the
// query's interval (any hit).  All 64 lanes of the wave must be active.
__device__ inline void flush_wave(const SceneDev& S, TraceCtx& ctx, const RayPre& rp, float tmin, bool any,
                                  int nq, float& best_t, float& hu, float& hv, uint32_t& best_id, bool& found) {
  const int lane = (int)(threadIdx.x & 63u);
  // exclusive prefix sum of the queue lengths over the wave (nq < 16: one
  // ballot per bit)
  const uint64_t below = (1ull << lane) - 1ull;
  int pre = 0, total = 0;
#pragma unroll
  for (int bit = 0; bit < 4; ++bit) {
    const uint64_t m = __builtin_amdgcn_ballot_w64(((nq >> bit) & 1) != 0);
    pre += __popcll(m & below) << bit;
    total += __popcll(m) << bit;
  }
  const int incl = pre + nq;
  unsigned long long* keys = ctx.slot_key - lane;
  float2* uvs = ctx.slot_uv - lane;
  const unsigned long long key0 = ((unsigned long long)__float_as_uint(best_t) << 32) | best_id;
  keys[lane] = key0;
  // LDS accesses of the lanes of one wave execute in program order; the
  // wavefront fences keep the compiler from moving the slot accesses across
  // the rounds
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  const int kz_any = rp.kz | (any ? 4 : 0);
  const uint32_t* leafq_w = ctx.leafq - lane;
  constexpr int qs = kBlock;
  for (int base = 0; base < total; base += 64) {
    const int k = base + lane;
    // owner: the number of lanes whose items all lie below k
    int owner = 0;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1) {
      if (__shfl(incl, owner + step - 1) <= k) owner += step;
    }
    const int qi = k - __shfl(pre, owner);
    RayPre r;
    r.o = F3{__shfl(rp.o.x, owner), __shfl(rp.o.y, owner), __shfl(rp.o.z, owner)};
    r.Sx = __shfl(rp.Sx, owner);
    r.Sy = __shfl(rp.Sy, owner);
    r.Sz = __shfl(rp.Sz, owner);
    const int kk = __shfl(kz_any, owner);
    r.kz = kk & 3;
    const bool any_o = (kk & 4) != 0;
    const float bt_o = __shfl(best_t, owner);
    const uint32_t bid_o = (uint32_t)__shfl((int)best_id, owner);
    unsigned long long bkey = ~0ull;
    float bu = 0.0f, bv = 0.0f;
    if (k < total) {
      ctx.n_tris++;
      const TriRecord& tr = S.tris[leafq_w[owner + qi * qs]];
      const float4 a = *reinterpret_cast<const float4*>(tr.v0);
      const float4 b = *reinterpret_cast<const float4*>(tr.v1);
      const float4 e = *reinterpret_cast<const float4*>(tr.v2);
      float tt;
      if (tri_intersect(r, F3{a.x, a.y, a.z}, F3{b.x, b.y, b.z}, F3{e.x, e.y, e.z}, &tt, &bu, &bv)) {
        const uint32_t id = __float_as_uint(a.w);
        // inside (tmin, tmax) and better than the owner's hit so far
        const bool ok = any_o ? tt < bt_o : (tt < bt_o || (tt == bt_o && bid_o != kNoHit && id < bid_o));
        if (tt > tmin && ok) bkey = ((unsigned long long)__float_as_uint(tt) << 32) | id;
      }
    }
    if (bkey != ~0ull) {
      atomicMin(&keys[owner], bkey);
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (keys[owner] == bkey) uvs[owner] = make_float2(bu, bv);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  const unsigned long long kf = keys[lane];
  if (kf != key0) {
    best_t = __uint_as_float((uint32_t)(kf >> 32));
    best_id = (uint32_t)kf;
    const float2 uv = uvs[lane];
    hu = uv.x;
    hv = uv.y;
    if (any) found = true;
  }
}

// Closest hit (any = false) or first found hit (any = true) in (tmin, tmax),
// tmax being the far bound the query's state was begun with.
// Ties in t resolve to the smallest triangle id, so the result does not
// depend on traversal order.  A ray with tmax < tmin visits the root only
// and misses (used for lanes without a query).
//
// Per node visit: slab tests of the four children; hit inner children are
// sorted near to far and pushed, hit leaves are appended to a per-lane queue
// in LDS.  Leaves (one triangle each) are tested later, when the wave decides
// to: at least three quarters of its live lanes
// have queued leaves, or some lane has no inner node left or a nearly full
// queue (the threshold was picked by timing 1/4, 1/2 and 3/4).
// Testing a leaf late only loosens culling (best_t shrinks later); it never
// changes the result, since the closest hit does not depend on test order.
// Lanes run this loop in step with ballots, so the triangle test executes
// with most lanes active instead of once per child slot that any lane hit.
//
// Runs the wave's queries until all have finished or until at most
// keep64/64 of the queries live on entry are still unfinished (keep64 = 0:
// to the end).  The state of unfinished queries is in `st`; calling again
// with the same ray continues them exactly where they stopped, so the
// result is the same however the traversal is split.
//
// kWave: the queued leaves are tested by the whole wave (flush_wave), which
// needs all 64 lanes active and the LDS slots of the context; otherwise
// each lane tests its own queue.
//
// A chained pair (trace_begin_chain) runs its any-hit query along d, then,
// within the same loop, its closest-hit query along d2 from the same origin
// with far bound tmax2.
template <bool kWave>
__device__ inline void trace_run(const SceneDev& S, TraceCtx& ctx, F3 o, F3 d, F3 d2, float tmax2, float tmin,
                                 bool any, TraceState& st, int keep64) {
  uint32_t keep = st.bits & kTsKeep;
  const F3 dq = (keep & kTsSecond) ? d2 : d;
  bool anyq = any && !(keep & kTsSecond);
  RayPre rp = ray_pre(o, dq);
  float ix = slab_rcp(dq.x), iy = slab_rcp(dq.y), iz = slab_rcp(dq.z);
  float best_t = st.best_t, hu = st.u, hv = st.v;
  uint32_t best_id = st.best_id;
  uint32_t node = st.node;
  int sp = (int)(st.bits & 0xFFu);
  int nq = (int)((st.bits >> 8) & 0xFu);
  bool inner_done = (st.bits & kTsInnerDone) != 0u;
  bool found = (st.bits & kTsFound) != 0u;
  bool chain = (keep & kTsChain) != 0u;
  int n_keep = 0;
  if (keep64 > 0) n_keep = (__popcll(__builtin_amdgcn_ballot_w64(!inner_done || nq > 0 || chain)) * keep64) >> 6;
  constexpr int qs = kBlock;
  lds_u32* const stack = lds_ptr(ctx.lds);
  lds_u32* const leafq = lds_ptr(ctx.leafq);
  for (;;) {
    // ---- the first query of a chained pair has ended: start the second ----
    if (chain && inner_done && nq == 0) {
      chain = false;
      keep = kTsSecond | (best_id != kNoHit ? kTsFirstHit : 0u);
      anyq = false;
      rp = ray_pre(o, d2);
      ix = slab_rcp(d2.x);
      iy = slab_rcp(d2.y);
      iz = slab_rcp(d2.z);
      best_t = tmax2;
      hu = 0.0f;
      hv = 0.0f;
      best_id = kNoHit;
      node = 0u;
      sp = 0;
      inner_done = false;
      found = false;
    }
    // ---- visit one inner node (lanes with room in their leaf queue) ----
    if (!inner_done && nq <= kLeafQueue - 4) {
      ctx.n_nodes++;
      const uint4* np = reinterpret_cast<const uint4*>(S.qnodes + node);
      const uint4 n0 = np[0], qx = np[1], qy = np[2], qz = np[3];
      // offsets of the node's origin, widened for near and far planes
      const float bx = fmaf(-o.x, S.qinv_scale, __uint_as_float(n0.x & 0xFFFFF800u)) * ix;
      const float by =
          fmaf(-o.y, S.qinv_scale, __uint_as_float(__builtin_amdgcn_alignbit(n0.x, n0.y, 11) & 0xFFFFF800u)) * iy;
      const float bz = fmaf(-o.z, S.qinv_scale, __uint_as_float((n0.y << 10) & 0xFFFFF800u)) * iz;
      const float bnx = fmaf(-kSlabWiden, fabsf(bx), bx), bfx = fmaf(kSlabWiden, fabsf(bx), bx);
      const float bny = fmaf(-kSlabWiden, fabsf(by), by), bfy = fmaf(kSlabWiden, fabsf(by), by);
      const float bnz = fmaf(-kSlabWiden, fabsf(bz), bz), bfz = fmaf(kSlabWiden, fabsf(bz), bz);
      // near and far planes by the direction's signs
      const bool px = ix >= 0.0f, py = iy >= 0.0f, pz = iz >= 0.0f;
      const uint32_t nx[2] = {px ? qx.x : qx.z, px ? qx.y : qx.w}, fx[2] = {px ? qx.z : qx.x, px ? qx.w : qx.y};
      const uint32_t ny[2] = {py ? qy.x : qy.z, py ? qy.y : qy.w}, fy[2] = {py ? qy.z : qy.x, py ? qy.w : qy.y};
      const uint32_t nz[2] = {pz ? qz.x : qz.z, pz ? qz.y : qz.w}, fz[2] = {pz ? qz.z : qz.x, pz ? qz.w : qz.y};
      const float tmin_q = tmin * S.qinv_scale, tmax_q = best_t * S.qinv_scale;
      const uint32_t ni = n0.z >> kQCountShift, nc = ni + (n0.w >> kQCountShift);
      const uint32_t child0 = n0.z & kQIndexMask;
      const uint32_t leaf0 = (n0.w & kQIndexMask) - ni;  // slot s >= ni: triangle record leaf0 + s
      // hit inner children as sort keys: the entry distance's bits (t > 0
      // sorts as an integer) with the slot in the two lowest
      uint32_t key[4];
#pragma unroll
      for (uint32_t s = 0; s < 4; ++s) {
        const float tx = fmaf(half_of(nx[s >> 1], s & 1u), ix, bnx), ux = fmaf(half_of(fx[s >> 1], s & 1u), ix, bfx);
        const float ty = fmaf(half_of(ny[s >> 1], s & 1u), iy, bny), uy = fmaf(half_of(fy[s >> 1], s & 1u), iy, bfy);
        const float tz = fmaf(half_of(nz[s >> 1], s & 1u), iz, bnz), uz = fmaf(half_of(fz[s >> 1], s & 1u), iz, bfz);
        const float tn = fmaxf(fmaxf(tx, ty), fmaxf(tz, tmin_q));
        const float tf = fminf(fminf(ux, uy), fminf(uz, tmax_q));
        const bool hit = tn <= tf;
        const bool inner = s < ni;
        key[s] = hit && inner ? (__float_as_uint(tn) & ~3u) | s : kNoChild;
        // the entry behind the last is written anyway and counts only for a
        // hit leaf (kLeafQueue - 4 entries at most are queued here)
        leafq[nq * qs] = leaf0 + s;
        nq += hit && !inner && s < nc ? 1 : 0;
      }
      // 4-element sorting network, near to far
#define TR_CSWAP(i, j)                                                   \
      {                                                                  \
        const uint32_t _a = key[i], _b = key[j];                         \
        key[i] = _a < _b ? _a : _b;                                      \
        key[j] = _a < _b ? _b : _a;                                      \
      }
      TR_CSWAP(0, 1) TR_CSWAP(2, 3) TR_CSWAP(0, 2) TR_CSWAP(1, 3) TR_CSWAP(1, 2)
#undef TR_CSWAP
      if (__builtin_amdgcn_ballot_w64(sp > kStackLds - 3) == 0ull) {
        // room in LDS for three more entries on every lane: the far children
        // are written unconditionally and the top moves past the hit ones
#pragma unroll
        for (int j = 3; j > 0; --j) {
          stack[sp * qs] = child0 + (key[j] & 3u);
          sp += key[j] != kNoChild ? 1 : 0;
        }
      } else {
        // sp < cap always holds: the host refuses a launch whose BVH needs
        // more than `cap` entries (stack_need, computed at build time); the
        // test only keeps the stack in bounds
#pragma unroll
        for (int j = 3; j > 0; --j)
          if (key[j] != kNoChild && sp < ctx.cap) stack_push(ctx, sp, child0 + (key[j] & 3u));
      }
      if (key[0] != kNoChild) {
        node = child0 + (key[0] & 3u);
      } else if (sp > 0) {
        node = stack_pop(ctx, sp);
      } else {
        inner_done = true;
      }
    }
    // ---- decide, wave-wide, whether queued leaves are tested now ----
    const bool pend = nq > 0;
    const bool live = !inner_done || pend || chain;
    const uint64_t m_live = __builtin_amdgcn_ballot_w64(live);
    if (m_live == 0ull) break;
    if (__popcll(m_live) <= n_keep) break;
    const uint64_t m_pend = __builtin_amdgcn_ballot_w64(pend);
    const uint64_t m_urgent = __builtin_amdgcn_ballot_w64(pend && (inner_done || nq > kLeafQueue - 4));
    bool flush;
    if constexpr (kWave) {
      // a wave-wide flush costs one round for up to 64 leaves: wait until
      // kWaveStall64/64 of the live lanes are stalled on their queue,
      // kWavePend64/64 have leaves queued, or no lane can visit a node
      const uint64_t m_visit = __builtin_amdgcn_ballot_w64(!inner_done && nq <= kLeafQueue - 4);
      flush = m_visit == 0ull || __popcll(m_urgent) * 64 >= kWaveStall64 * __popcll(m_live) ||
              __popcll(m_pend) * 64 >= kWavePend64 * __popcll(m_live);
    } else {
      flush = m_urgent != 0ull || 4 * __popcll(m_pend) >= 3 * __popcll(m_live);
    }
    if constexpr (kWave) {
      if (flush) {
        flush_wave(S, ctx, rp, tmin, anyq, nq, best_t, hu, hv, best_id, found);
        nq = 0;
        if (found) inner_done = true;
      }
    } else if (flush && pend) {
      for (int qi = 0; qi < nq; ++qi) {
        ctx.n_tris++;
        const TriRecord& tr = S.tris[leafq[qi * qs]];
        float4 a = *reinterpret_cast<const float4*>(tr.v0);
        float4 b = *reinterpret_cast<const float4*>(tr.v1);
        float4 e = *reinterpret_cast<const float4*>(tr.v2);
        float tt, uu, vv;
        if (!tri_intersect(rp, F3{a.x, a.y, a.z}, F3{b.x, b.y, b.z}, F3{e.x, e.y, e.z}, &tt, &uu, &vv)) continue;
        uint32_t id = __float_as_uint(a.w);
        // best_t is the far bound tmax until a hit is accepted, and below
        // it afterwards, so these tests keep every hit inside (tmin, tmax)
        if (!(tt > tmin)) continue;
        if (anyq) {
          if (!(tt < best_t)) continue;
          best_id = id; best_t = tt; hu = uu; hv = vv;
          found = true;
          break;
        }
        if (tt < best_t || (tt == best_t && best_id != kNoHit && id < best_id)) {
          best_t = tt; best_id = id; hu = uu; hv = vv;
        }
      }
      nq = 0;
      if (found) inner_done = true;
    }
  }
  st.best_t = best_t;
  st.u = hu;
  st.v = hv;
  st.best_id = best_id;
  st.node = node;
  st.bits = (uint32_t)sp | ((uint32_t)nq << 8) | (inner_done ? kTsInnerDone : 0u) | (found ? kTsFound : 0u) | keep;
}

// One query to the end.
__device__ inline Hit trace_ray_rt(const SceneDev& S, TraceCtx& ctx, F3 o, F3 d, float tmin, float tmax, bool any) {
  ctx.n_queries++;
  TraceState st;
  trace_begin(st, tmax);
  trace_run<false>(S, ctx, o, d, d, tmax, tmin, any, st, 0);
  return trace_hit(st);
}

template <bool kAnyHit>
__device__ inline Hit trace_ray(const SceneDev& S, TraceCtx& ctx, F3 o, F3 d, float tmin, float tmax) {
  return trace_ray_rt(S, ctx, o, d, tmin, tmax, kAnyHit);
}

}  // namespace trc
