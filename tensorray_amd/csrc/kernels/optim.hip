// Optimizer step on device parameters: Adam (Kingma & Ba 2015) with the
// update order of the reference's C++ examples (Optimizer.h:66-123):
//   m = b1*m + (1-b1)*g;  v = b2*v + (1-b2)*g*g;
//   x -= lr * (m / bc1) / (sqrt(v / bc2) + eps),  bc_i = 1 - b_i^t.
// Non-finite gradient entries count as zero (the reference scrubs NaN
// gradients before its optimizer, renderer_single_view.py:82).
#include <hip/hip_runtime.h>

#include "../trc_internal.h"

namespace trc {

__global__ void k_adam(float* x, const float* g, float* m, float* v, uint64_t n, float lr, float b1, float b2,
                       float eps, float bc1, float bc2) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const float c1 = 1.0f - b1, c2 = 1.0f - b2;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    float gi = g[i];
    if (!(gi - gi == 0.0f)) gi = 0.0f;  // NaN or infinity
    const float mi = b1 * m[i] + c1 * gi;
    const float vi = b2 * v[i] + c2 * (gi * gi);
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / bc1;
    const float vh = vi / bc2;
    x[i] = x[i] - (lr * mh) / (sqrtf(vh) + eps);
  }
}

hipError_t launch_adam(float* x, const float* g, float* m, float* v, uint64_t n, float lr, float b1, float b2,
                       float eps, float bc1, float bc2, hipStream_t st) {
  if (n == 0) return hipSuccess;
  const uint64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(k_adam, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(256), 0, st, x, g, m, v, n, lr,
                     b1, b2, eps, bc1, bc2);
  return hipGetLastError();
}

}  // namespace trc

namespace trc {

// ---------------------------------------------------------------------------
// Uniform Adam (the step of the reference's LargeSteps optimizer,
// pyTensorRay/optimizer.py:40-63, AdamUniform of Nicolet et al. 2021): Adam
// moments as above, but every coordinate is scaled by the one largest
// second moment, x -= lr / (bc1 * sqrt(max(v) / bc2)) * m.
// ---------------------------------------------------------------------------
__global__ void k_adam_uniform_moments(const float* g, float* m, float* v, uint64_t n, float b1, float b2,
                                       unsigned int* vmax_bits) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const float c1 = 1.0f - b1, c2 = 1.0f - b2;
  float local = 0.0f;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    float gi = g[i];
    if (!(gi - gi == 0.0f)) gi = 0.0f;
    m[i] = b1 * m[i] + c1 * gi;
    const float vi = b2 * v[i] + c2 * (gi * gi);
    v[i] = vi;
    local = fmaxf(local, vi);
  }
  // v >= 0, so the order of the float bit patterns is the order of the
  // values; one atomic per block (atomics on one word from every wave of a
  // large grid serialise)
  __shared__ float wmax[4];
  for (int o = 32; o > 0; o >>= 1) local = fmaxf(local, __shfl_xor(local, o));
  if ((threadIdx.x & 63u) == 0u) wmax[threadIdx.x >> 6] = local;
  __syncthreads();
  if (threadIdx.x == 0u) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) local = fmaxf(local, wmax[w]);
    atomicMax(vmax_bits, __float_as_uint(local));
  }
}

__global__ void k_adam_uniform_apply(float* x, const float* m, uint64_t n, float lr, float bc1, float bc2,
                                     const unsigned int* vmax_bits) {
  const float vmax = __uint_as_float(*vmax_bits);
  if (!(vmax > 0.0f)) return;
  const float scale = lr / (bc1 * sqrtf(vmax / bc2));
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) x[i] = x[i] - scale * m[i];
}

__global__ void k_zero_u32(unsigned int* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

hipError_t launch_adam_uniform(float* x, const float* g, float* m, float* v, uint64_t n, float lr, float b1, float b2,
                               float bc1, float bc2, unsigned int* vmax_bits, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, st, vmax_bits, 1);
  if (n == 0) return hipGetLastError();
  const uint64_t blocks = (n + 255) / 256;
  const dim3 grid((unsigned)(blocks < 8192 ? blocks : 8192));
  const dim3 grid_m((unsigned)(blocks < 1024 ? blocks : 1024));  // 256 threads = 4 waves per block
  hipLaunchKernelGGL(k_adam_uniform_moments, grid_m, dim3(256), 0, st, g, m, v, n, b1, b2, vmax_bits);
  hipLaunchKernelGGL(k_adam_uniform_apply, grid, dim3(256), 0, st, x, m, n, lr, bc1, bc2, vmax_bits);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Conjugate gradients for M x = b with M = I + lambda L symmetric positive
// definite, three right-hand sides at once in the [V][3] layout of the
// vertex buffers.  Scalars live on the device (CgScalars); every kernel
// returns at once when all three columns have converged, so the host can
// queue iterations without waiting for anything.  A dot product is a partial
// per block (no atomics: the partials are summed in block order by every
// kernel that needs the total, so all of them see the same bits).
//
// An iteration is two kernels.  k_cg_matvec forms the search direction p = r
// + beta p_old of a row's neighbours where it gathers them (the direction of
// one iteration is the other buffer of the last) and the new direction's
// product; k_cg_update moves x and r.  With a kernel each for the product,
// the update, the direction and the scalars, a mesh of 100,002 vertices (4-5 us
// of work per iteration) was bound by queueing launches: 1,600 per call of 400
// iterations, 8-12 ms for a LargeSteps step of two calls.  The word `done` in
// host memory tells the host, which is still queueing, to stop; it never
// waits for it.
// ---------------------------------------------------------------------------
constexpr int kCgThreads = 256;

// The block's sum of (a, b, c) into part[blockIdx.x], in a fixed order.
__device__ inline void block_partial3(float a, float b, float c, float4* part) {
  __shared__ float w[kCgThreads / 64][3];
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o);
    b += __shfl_xor(b, o);
    c += __shfl_xor(c, o);
  }
  if ((threadIdx.x & 63u) == 0u) {
    w[threadIdx.x >> 6][0] = a;
    w[threadIdx.x >> 6][1] = b;
    w[threadIdx.x >> 6][2] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
    for (int k = 0; k < kCgThreads / 64; ++k) {
      s0 += w[k][0];
      s1 += w[k][1];
      s2 += w[k][2];
    }
    part[blockIdx.x] = make_float4(s0, s1, s2, 0.0f);
  }
}

// Sum of part[0 .. nb) per column, the same bits in every block: the first
// wave sums a fixed subset per lane, then reduces across lanes.  The loads go
// out together (their latency is most of a small solve's kernels).
__device__ inline void sum_partials3(const float4* part, int nb, float out[3]) {
  __shared__ float tot[3];
  if (threadIdx.x < 64u) {
    float4 v[kCgBlocks / 64];
#pragma unroll
    for (int j = 0; j < kCgBlocks / 64; ++j) {
      const int k = (int)threadIdx.x + 64 * j;
      v[j] = k < nb ? part[k] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    float a = 0.0f, b = 0.0f, c = 0.0f;
#pragma unroll
    for (int j = 0; j < kCgBlocks / 64; ++j) {
      a += v[j].x;
      b += v[j].y;
      c += v[j].z;
    }
    for (int o = 32; o > 0; o >>= 1) {
      a += __shfl_xor(a, o);
      b += __shfl_xor(b, o);
      c += __shfl_xor(c, o);
    }
    if (threadIdx.x == 0u) {
      tot[0] = a;
      tot[1] = b;
      tot[2] = c;
    }
  }
  __syncthreads();
  out[0] = tot[0];
  out[1] = tot[1];
  out[2] = tot[2];
}

// y_i = sum over row i's columns j, in ascending order, of M_ij x_j; x(j)
// gives a vector's row.
template <class X>
__device__ inline F3 row_product(const LaplaceDev& M, int i, X&& x) {
  const int len = M.len[i];
  const float diag = 1.0f + M.lambda * (float)(len - 1);
  const int* col = M.col + (size_t)M.off[i >> 6] * 64u + (i & 63);
  F3 a{0.0f, 0.0f, 0.0f};
  for (int k = 0; k < len; ++k) {
    const int j = col[(size_t)k * 64u];
    a = a + (j == i ? diag : -M.lambda) * x(j);
  }
  return a;
}
__device__ inline F3 row3(const float* v, int i) { return F3{v[3 * (size_t)i], v[3 * (size_t)i + 1], v[3 * (size_t)i + 2]}; }
__device__ inline void put_row3(float* v, int i, F3 a) {
  v[3 * (size_t)i] = a.x;
  v[3 * (size_t)i + 1] = a.y;
  v[3 * (size_t)i + 2] = a.z;
}

// y = M x
__global__ void __launch_bounds__(kCgThreads) k_laplace_apply(LaplaceDev M, const float* x, float* y) {
  const int stride = gridDim.x * blockDim.x;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < M.n; i += stride)
    put_row3(y, i, row_product(M, i, [&](int j) { return row3(x, j); }));
}

// r = b - M x; partials of r.r and b.b
__global__ void __launch_bounds__(kCgThreads) k_cg_init(LaplaceDev M, const float* b, const float* x, float* r,
                                                        CgScalars* s) {
  F3 d{0.0f, 0.0f, 0.0f}, e{0.0f, 0.0f, 0.0f};
  const int stride = gridDim.x * blockDim.x;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < M.n; i += stride) {
    const F3 bi = row3(b, i);
    const F3 ri = bi - row_product(M, i, [&](int j) { return row3(x, j); });
    put_row3(r, i, ri);
    d = d + ri * ri;
    e = e + bi * bi;
  }
  block_partial3(d.x, d.y, d.z, s->part_rr);
  __syncthreads();  // block_partial3's LDS is reused
  block_partial3(e.x, e.y, e.z, s->part_b);
}

// Scalars of iteration `it` from the partials the last kernels left: rr = r.r
// and the columns still active.  Every block computes them; block 0 stores
// them at parity (it + 1) & 1 (others still read parity it & 1).
__device__ inline uint32_t cg_scalars(CgScalars* s, int it, float tol2, float rr[3], float beta[3], uint32_t* done,
                                      uint32_t seq) {
  const int nb = (int)gridDim.x;
  sum_partials3(s->part_rr, nb, rr);
  uint32_t active = 0u;
  if (it == 0) {
    float b2[3];
    __syncthreads();  // sum_partials3's LDS is reused
    sum_partials3(s->part_b, nb, b2);
    for (int c = 0; c < 3; ++c) {
      beta[c] = 0.0f;
      if (rr[c] > tol2 * b2[c] && rr[c] > 0.0f) active |= 1u << c;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
      for (int c = 0; c < 3; ++c) s->rr0[c] = b2[c];
  } else {
    active = s->active[it & 1];
    for (int c = 0; c < 3; ++c) {
      const float old = s->rr[it & 1][c];
      beta[c] = old > 0.0f ? rr[c] / old : 0.0f;
      if (!(rr[c] > tol2 * s->rr0[c])) active &= ~(1u << c);
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int c = 0; c < 3; ++c) s->rr[(it + 1) & 1][c] = rr[c];
    s->active[(it + 1) & 1] = active;
    s->iters = (uint32_t)it;
    s->last = (uint32_t)((it + 1) & 1);
    if (active == 0u && done) __hip_atomic_store(done, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  return active;
}
// A converged solve: the state is handed on to the other parity unchanged.
__device__ inline bool cg_done(CgScalars* s, int it) {
  if (it == 0 || s->active[it & 1] != 0u) return false;
  if (blockIdx.x == 0 && threadIdx.x == 0) s->active[(it + 1) & 1] = 0u;
  return true;
}

// p = r + beta p_old (it = 0: r), ap = M p; partials of p.ap.  r.r of the last
// update decides whether any column still iterates.
__global__ void __launch_bounds__(kCgThreads) k_cg_matvec(LaplaceDev M, const float* r, const float* p_old, float* p,
                                                          float* ap, CgScalars* s, int it, float tol2, uint32_t* done,
                                                          uint32_t seq) {
  if (cg_done(s, it)) return;
  float rr[3], beta[3];
  if (cg_scalars(s, it, tol2, rr, beta, done, seq) == 0u) return;
  F3 dot3{0.0f, 0.0f, 0.0f};
  const F3 bt{beta[0], beta[1], beta[2]};
  const int stride = gridDim.x * blockDim.x;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < M.n; i += stride) {
    F3 pi, y;
    if (it == 0) {
      pi = row3(r, i);
      y = row_product(M, i, [&](int j) { return row3(r, j); });
    } else {
      pi = row3(r, i) + bt * row3(p_old, i);
      y = row_product(M, i, [&](int j) { return row3(r, j) + bt * row3(p_old, j); });
    }
    put_row3(p, i, pi);
    put_row3(ap, i, y);
    dot3 = dot3 + pi * y;
  }
  block_partial3(dot3.x, dot3.y, dot3.z, s->part_pap);
}

// x += alpha p, r -= alpha Ap (alpha = rr / pAp); partials of the new r.r
__global__ void __launch_bounds__(kCgThreads) k_cg_update(float* x, float* r, const float* p, const float* ap, int n,
                                                          CgScalars* s, int it) {
  const uint32_t active = s->active[(it + 1) & 1];
  if (active == 0u) return;
  float pap[3];
  sum_partials3(s->part_pap, (int)gridDim.x, pap);
  float al[3];
  for (int c = 0; c < 3; ++c)
    al[c] = ((active >> c) & 1u) && pap[c] > 0.0f ? s->rr[(it + 1) & 1][c] / pap[c] : 0.0f;
  const F3 alpha{al[0], al[1], al[2]};
  F3 d{0.0f, 0.0f, 0.0f};
  const int stride = gridDim.x * blockDim.x;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    put_row3(x, i, row3(x, i) + alpha * row3(p, i));
    const F3 ri = row3(r, i) - alpha * row3(ap, i);
    put_row3(r, i, ri);
    d = d + ri * ri;
  }
  block_partial3(d.x, d.y, d.z, s->part_rr);
}

// The scalars after the last update (one block standing for the grid of nb).
__global__ void __launch_bounds__(kCgThreads) k_cg_finish(CgScalars* s, int it, float tol2, int nb) {
  if (it > 0 && s->active[it & 1] == 0u) return;  // the last k_cg_matvec stored them
  float rr[3], b2[3];
  sum_partials3(s->part_rr, nb, rr);
  if (it == 0) {
    __syncthreads();  // sum_partials3's LDS is reused
    sum_partials3(s->part_b, nb, b2);
  }
  if (threadIdx.x != 0u) return;
  for (int c = 0; c < 3; ++c) {
    s->rr[0][c] = rr[c];
    if (it == 0) s->rr0[c] = b2[c];
  }
  s->iters = (uint32_t)it;
  s->last = 0u;
}

static int cg_grid(int n) {
  const int g = (n + kCgThreads - 1) / kCgThreads;
  return g < 1 ? 1 : (g > kCgBlocks ? kCgBlocks : g);
}

hipError_t launch_laplace_apply(const LaplaceDev& M, const float* x, float* y, hipStream_t st) {
  hipLaunchKernelGGL(k_laplace_apply, dim3(cg_grid(M.n)), dim3(kCgThreads), 0, st, M, x, y);
  return hipGetLastError();
}

hipError_t launch_cg(const LaplaceDev& M, const float* b, float* x, float* r, float* p0, float* p1, float* ap,
                     CgScalars* s, int max_iter, float tol, uint32_t* done, uint32_t seq, hipStream_t st) {
  const int n = M.n;
  const int nb = cg_grid(n);
  const dim3 g(nb), blk(kCgThreads);
  const float tol2 = tol * tol;
  float* p[2] = {p0, p1};
  hipLaunchKernelGGL(k_cg_init, g, blk, 0, st, M, b, (const float*)x, r, s);
  int it = 0;
  for (; it < max_iter; ++it) {
    if (done && __atomic_load_n(done, __ATOMIC_RELAXED) == seq) break;
    hipLaunchKernelGGL(k_cg_matvec, g, blk, 0, st, M, (const float*)r, (const float*)p[(it + 1) & 1], p[it & 1], ap, s,
                       it, tol2, done, seq);
    hipLaunchKernelGGL(k_cg_update, g, blk, 0, st, x, r, (const float*)p[it & 1], (const float*)ap, n, s, it);
  }
  hipLaunchKernelGGL(k_cg_finish, dim3(1), blk, 0, st, s, it, tol2, nb);
  return hipGetLastError();
}

}  // namespace trc
