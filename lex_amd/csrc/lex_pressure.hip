// P3/P4: pseudo-incompressible pressure equation (pressure_equations.py) and the
// unpreconditioned BiCGSTAB of jax.scipy.sparse.linalg.bicgstab that the reference
// calls (one_step_integration.py:468-487).  Vectors are FP32 (nx, ny, nz); every
// reduction (dot product) and the scalar recurrence run in FP64.
//
// One iteration = 3 kernels, each a grid-stride pass whose dot products leave FP64
// per-block partials that the following kernels sum in a fixed order (deterministic).
// All kernels check a device-side `done` flag, so the host can enqueue iterations ahead
// and poll the flag only every few iterations.
#pragma once
#include "lex_common.hpp"

namespace lex {

// --------------------------- rtt, RHS, matvec ------------------------------------
// calculate_rtt (pressure_equations.py:175-195)
__global__ void k_rtt(Dims d, const float* __restrict__ rtc, const float* __restrict__ th,
                      const float* __restrict__ qv, const float* __restrict__ buoy, float* __restrict__ rtt) {
  int K = blockIdx.x * blockDim.x + threadIdx.x;  // 0..nz+1
  int J = blockIdx.y * blockDim.y + threadIdx.y;  // padded
  int I = blockIdx.z;
  if (K >= d.nz + 2 || J >= d.ny + 6) return;
  long c = ic(d, I, J, K);
  float val;
  if (K >= 1 && K <= d.nz) {
    val = rtc[K] * th[c] * (1.0f + (float)kReps * qv[c]) / (1.0f + qv[c]);
  } else {
    int i = (I - 3 + d.nx) % d.nx, j = (J - 3 + d.ny) % d.ny;
    const float* bcol = buoy + ((long)i * d.ny + j) * d.nz;
    auto rb = [&](int k) { return rtc[k + 1] * bcol[k] / (float)kCp; };
    int nz = d.nz;
    val = (K == 0) ? (1.875f * rb(0) + (-1.25f) * rb(1) + 0.375f * rb(2))
                   : (1.875f * rb(nz - 1) + (-1.25f) * rb(nz - 2) + 0.375f * rb(nz - 3));
  }
  rtt[c] = val;
}

// rhs_of_pressure_equation (pressure_equations.py:51-77) on interior (nx,ny,nz) arrays
__global__ void k_p_rhs(Dims d, const float* __restrict__ rtc, const float* __restrict__ au,
                        const float* __restrict__ av, const float* __restrict__ aw, const float* __restrict__ fu,
                        const float* __restrict__ fv, const float* __restrict__ buoy, float* __restrict__ rhs) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  int j = blockIdx.y * blockDim.y + threadIdx.y;
  int i = blockIdx.z;
  if (k >= d.nz || j >= d.ny) return;
  const int nx = d.nx, ny = d.ny, nz = d.nz;
  float rt = rtc[k + 1];
  auto U = [&](const float* a, int f) { return a[((long)f * ny + j) * nz + k]; };
  auto V = [&](const float* a, int f) { return a[((long)i * (ny + 1) + f) * nz + k]; };
  auto r8w = [&](int l) -> float { return (l <= 0 || l >= nz) ? 0.0f : 0.5f * (rtc[l] + rtc[l + 1]); };
  auto W = [&](int l) { return aw[((long)i * ny + j) * (nz + 1) + l]; };
  float adv = (rt * U(au, i + 1) - rt * U(au, i)) * d.idx + (rt * V(av, j + 1) - rt * V(av, j)) * d.idy +
              (r8w(k + 1) * W(k + 1) - r8w(k) * W(k)) * d.idz;
  float cor = 0.0f;
  if (fu && fv) cor = (rt * U(fv, i + 1) - rt * U(fv, i)) * d.idx + (rt * (-V(fu, j + 1)) - rt * (-V(fu, j))) * d.idy;
  const float* bcol = buoy + ((long)i * ny + j) * nz;
  auto rb = [&](int kk) { return rtc[kk + 1] * bcol[kk]; };
  auto rbw = [&](int l) -> float {
    if (l == 0) return 1.875f * rb(0) + (-1.25f) * rb(1) + 0.375f * rb(2);
    if (l == nz) return 1.875f * rb(nz - 1) + (-1.25f) * rb(nz - 2) + 0.375f * rb(nz - 3);
    return 0.5f * (rb(l - 1) + rb(l));
  };
  float bz = (rbw(k + 1) - rbw(k)) * d.idz;
  rhs[((long)i * ny + j) * nz + k] = adv + cor + bz;
  (void)nx;
}

// affine matvec laplace_of_pressure (pressure_equations.py:8-48) at interior (i,j,k)
__device__ __forceinline__ float matvec_point(const Dims& d, const float* __restrict__ rtt,
                                              const float* __restrict__ x, int i, int j, int k) {
  const int nx = d.nx, ny = d.ny, nz = d.nz;
  auto X = [&](int a, int b, int c) {
    a = (a + nx) % nx;
    b = (b + ny) % ny;
    c = c < 0 ? 0 : (c >= nz ? nz - 1 : c);
    return x[((long)a * ny + b) * nz + c];
  };
  long cc = ic(d, i + 3, j + 3, k + 1);
  const long sx = d.sxc(), sy = d.syc();
  float xc = X(i, j, k);
  float px0 = 0.5f * (rtt[cc] + rtt[cc - sx]) * ((xc - X(i - 1, j, k)) * d.idx);
  float px1 = 0.5f * (rtt[cc + sx] + rtt[cc]) * ((X(i + 1, j, k) - xc) * d.idx);
  float py0 = 0.5f * (rtt[cc] + rtt[cc - sy]) * ((xc - X(i, j - 1, k)) * d.idy);
  float py1 = 0.5f * (rtt[cc + sy] + rtt[cc]) * ((X(i, j + 1, k) - xc) * d.idy);
  float pz0 = (k == 0) ? rtt[cc - 1] : 0.5f * (rtt[cc] + rtt[cc - 1]) * ((xc - X(i, j, k - 1)) * d.idz);
  float pz1 = (k == nz - 1) ? rtt[cc + 1] : 0.5f * (rtt[cc + 1] + rtt[cc]) * ((X(i, j, k + 1) - xc) * d.idz);
  return (float)kCp * ((px1 - px0) * d.idx + (py1 - py0) * d.idy + (pz1 - pz0) * d.idz);
}

__global__ void k_p_matvec(Dims d, const float* __restrict__ rtt, const float* __restrict__ x, float* __restrict__ out) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  int j = blockIdx.y * blockDim.y + threadIdx.y;
  int i = blockIdx.z;
  if (k >= d.nz || j >= d.ny) return;
  out[((long)i * d.ny + j) * d.nz + k] = matvec_point(d, rtt, x, i, j, k);
}

// ------------------------------- BiCGSTAB ----------------------------------------
// Every dot product is reduced in two phases across a kernel boundary: a kernel writes
// one FP64 partial sum per block, and each block of the next kernel sums all partials
// itself, in the same fixed order, so every block derives bit-identical scalars.  No
// kernel needs a grid-wide fence or a last-block ticket (on a multi-XCD part a
// device-scope release writes back the XCD's L2, which made those tails dominate).
//
// Scalars entering iteration `it` (rho, alpha, omega, k) are double-buffered by parity:
// iteration it reads s[it & 1] and its last kernel's block 0 writes s[(it + 1) & 1].
// The loop test (JAX: |r|^2 > atol^2 and 0 <= k < maxiter) runs at the top of each
// iteration; the first kernel that finds it false sets the sticky `done` and `k_final`.
struct BicgScalars {
  double rho, alpha, omega;
  int k, pad;
};
struct BicgState {
  BicgScalars s[2];
  int done;      // sticky: the loop has ended
  int k_final;   // exit code (iterations, or -10 / -11 on breakdown)
  int maxiter;
  int pad;
  // what block 0 of one kernel hands to the next, so that each sum is reduced once: K1
  // writes atol2 (iteration 0) and rho_new, K2 alpha
  double atol2, rho_new, alpha;
};
static_assert(sizeof(BicgState) <= 256, "BiCGSTAB loop state fits its 256-byte slot");

constexpr int kBicgThreads = 256;
constexpr int kBicgBlocks = 1024;   // upper bound on blocks (partials per sum)
constexpr int kBicgCellsPerThread = 2;   // grid size (1-16 measured within 15 % on 64x64x40)
// partial-sum slots (each kBicgBlocks doubles): b.b; (r.r, rhat.r) x 2 parities;
// rhat.q; (t.s, t.t, s.s)
constexpr int kBicgSlots = 1 + 4 + 1 + 3;
constexpr size_t kBicgPartialBytes = (size_t)kBicgSlots * kBicgBlocks * sizeof(double);
struct BicgPartials {
  double* base;
  // Addresses by arithmetic: an array of pointers indexed at run time would go through LDS,
  // and the kernel would read its dispatch packet from host memory for the workgroup size
  // (10 us of each launch's 20).
  __host__ __device__ double* bb() const { return base; }                                    // [nb]
  __host__ __device__ double* rr(int par) const { return base + (1 + 2 * par) * kBicgBlocks; }  // [2][nb]: r.r, rhat.r
  __host__ __device__ double* rq() const { return base + 5 * kBicgBlocks; }                  // [nb]
  __host__ __device__ double* ts() const { return base + 6 * kBicgBlocks; }                  // [3][nb]: t.s, t.t, s.s
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// Block-level sum of NV per-thread values; the result is returned to every thread.
template <int NV>
__device__ __forceinline__ void block_sum_all(const double (&v)[NV], double (&out)[NV]) {
  __shared__ double sh[NV][kBicgThreads / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const double s = wave_sum(v[q]);
    if (lane == 0) sh[q][wv] = s;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kBicgThreads / 64; ++w) t += sh[q][w];
    out[q] = t;
  }
}

// This thread's share of NV partial arrays (nb entries each, strided over the block), in a
// fixed order.  Every entry of every array is requested before the first is needed, so the
// prologue of a kernel waits once for what other XCDs wrote, not once per array.
template <int NV>
struct PartialShare {
  static constexpr int kEach = kBicgBlocks / kBicgThreads;
  double v[NV][kEach];
  __device__ __forceinline__ void request(const double* const (&P)[NV], int nb) {
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const int b = threadIdx.x + e * kBicgThreads;
      const uint32_t c = (uint32_t)min(b, nb - 1);   // loads without a branch per thread
#pragma unroll
      for (int q = 0; q < NV; ++q) {
        v[q][e] = 0.0;
        if (e * kBicgThreads < nb) {
          const double x = P[q][c];
          v[q][e] = b < nb ? x : 0.0;
        }
      }
    }
  }
  __device__ __forceinline__ void sum(double (&tot)[NV]) const {
    double s[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      s[q] = 0.0;
#pragma unroll
      for (int e = 0; e < kEach; ++e) s[q] += v[q][e];
    }
    block_sum_all<NV>(s, tot);
  }
};

// Write this block's sums of NV per-thread values to P[q * kBicgBlocks + blockIdx.x].
template <int NV>
__device__ __forceinline__ void put_partials(const double (&acc)[NV], double* __restrict__ P) {
  double tot[NV];
  __syncthreads();   // the prologue's sums have been read
  block_sum_all<NV>(acc, tot);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q) P[q * kBicgBlocks + blockIdx.x] = tot[q];
  }
}

// The pressure operator's stencil at the unpadded linear index t (x slowest, z fastest): the
// offsets of the seven points in an unpadded vector (periodic in x and y, z clamped to the
// end levels) and the cell's offset in the padded rtt.
struct Stencil {
  uint32_t c, xm, xp, ym, yp, zm, zp, rc;
  bool first, last;   // lowest / highest level
};
__device__ __forceinline__ Stencil stencil_at(const Dims& d, uint32_t t) {
  const uint32_t nz = d.nz, ny = d.ny, nx = d.nx;
  const uint32_t jt = t / nz, k = t - jt * nz, i = jt / ny, j = jt - i * ny, syz = ny * nz;
  Stencil s;
  s.c = t;
  s.xm = (i == 0) ? t + (nx - 1) * syz : t - syz;
  s.xp = (i == nx - 1) ? t - (nx - 1) * syz : t + syz;
  s.ym = (j == 0) ? t + (ny - 1) * nz : t - nz;
  s.yp = (j == ny - 1) ? t - (ny - 1) * nz : t + nz;
  s.first = k == 0;
  s.last = k == nz - 1;
  s.zm = s.first ? t : t - 1;
  s.zp = s.last ? t : t + 1;
  s.rc = ((i + 3) * (ny + 6) + j + 3) * (nz + 2) + k + 1;
  return s;
}
// A value per stencil point.
struct Seven {
  float c, xm, xp, ym, yp, zm, zp;
};
__device__ __forceinline__ Seven load7(const float* __restrict__ a, const Stencil& s) {
  return Seven{ld32(a, s.c), ld32(a, s.xm), ld32(a, s.xp), ld32(a, s.ym), ld32(a, s.yp), ld32(a, s.zm), ld32(a, s.zp)};
}
__device__ __forceinline__ Seven load_rtt(const Dims& d, const float* __restrict__ rtt, const Stencil& s) {
  const uint32_t sy = d.nz + 2, sx = (d.ny + 6) * sy;
  return Seven{ld32(rtt, s.rc), ld32(rtt, s.rc - sx), ld32(rtt, s.rc + sx), ld32(rtt, s.rc - sy), ld32(rtt, s.rc + sy),
               ld32(rtt, s.rc - 1), ld32(rtt, s.rc + 1)};
}
// laplace_of_pressure (pressure_equations.py:8-48) from the stencil values of rtt and x;
// arithmetic in the order of matvec_point.
__device__ __forceinline__ float matvec7(const Dims& d, const Stencil& s, const Seven& r, const Seven& x) {
  float px0 = 0.5f * (r.c + r.xm) * ((x.c - x.xm) * d.idx);
  float px1 = 0.5f * (r.xp + r.c) * ((x.xp - x.c) * d.idx);
  float py0 = 0.5f * (r.c + r.ym) * ((x.c - x.ym) * d.idy);
  float py1 = 0.5f * (r.yp + r.c) * ((x.yp - x.c) * d.idy);
  float pz0 = s.first ? r.zm : 0.5f * (r.c + r.zm) * ((x.c - x.zm) * d.idz);
  float pz1 = s.last ? r.zp : 0.5f * (r.zp + r.c) * ((x.zp - x.c) * d.idz);
  return (float)kCp * ((px1 - px0) * d.idx + (py1 - py0) * d.idy + (pz1 - pz0) * d.idz);
}

// clear the loop state (a kernel, not a memset, so the solve can be graph-captured)
__global__ void k_bicg_reset(BicgState* st, int maxiter) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    for (int q = 0; q < 2; ++q) {
      st->s[q].rho = st->s[q].alpha = st->s[q].omega = 1.0;
      st->s[q].k = 0;
    }
    st->maxiter = maxiter;
    st->done = 0;
    st->k_final = 0;
  }
}

// init: r = b - A(x0), rhat = p = q = r, x = x0; partials b.b and (r.r, rhat.r = r.r)
// in the parity slot iteration 0 reads
__global__ void __launch_bounds__(kBicgThreads) k_bicg_init(Dims d, const float* __restrict__ rtt,
                                                           const float* __restrict__ b, const float* __restrict__ x0,
                                                           float* __restrict__ x, float* __restrict__ r,
                                                           float* __restrict__ rhat, float* __restrict__ p,
                                                           float* __restrict__ q, double* __restrict__ partials) {
  const BicgPartials P{partials};
  const uint32_t n = (uint32_t)d.nx * d.ny * d.nz, stride = gridDim.x * blockDim.x;
  double acc[2] = {0.0, 0.0};
  for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride) {
    const Stencil s = stencil_at(d, t);
    const Seven xv = load7(x0, s);
    const float bt = b[t];
    const float ri = bt - matvec7(d, s, load_rtt(d, rtt, s), xv);
    x[t] = xv.c;
    r[t] = ri;
    rhat[t] = ri;
    p[t] = ri;
    q[t] = ri;
    acc[0] += (double)bt * bt;
    acc[1] += (double)ri * ri;
  }
  double v[3] = {acc[0], acc[1], acc[1]};
  double tot[3];
  block_sum_all<3>(v, tot);
  if (threadIdx.x == 0) {
    P.bb()[blockIdx.x] = tot[0];
    P.rr(1)[blockIdx.x] = tot[1];
    P.rr(1)[kBicgBlocks + blockIdx.x] = tot[2];
  }
}

// What the three kernels of an iteration share.  They are latency-bound: the fields of the
// sizes solved here stay in the caches and a kernel is one chain of launch, loads, block
// reduction, arithmetic, block reduction.  So everything a thread reads - its first two
// cells' operands, the partial sums, the loop state - is requested before the first wait,
// and each sum is reduced by one kernel only.  64x64x40, us per launch of K1, K2, K3: 6.5, 5.5, 5.7
// (20.5, 21.1, 21.0 with a wait per array and per cell, 64-bit indices and a pointer table
// in LDS; an empty kernel of this grid takes 2.7).
constexpr int kBicgAhead = 2;   // cells of a thread whose operands are requested up front

// K1 of iteration it: the loop test; beta; p' = r + beta (p - omega q) (recomputed on
// the stencil's points); q' = A(p'); partials rhat.q'
__global__ void __launch_bounds__(kBicgThreads) k_bicg_pq(Dims d, const float* __restrict__ rtt,
                                                         const float* __restrict__ r, const float* __restrict__ rhat,
                                                         const float* __restrict__ p, const float* __restrict__ q,
                                                         float* __restrict__ pn, float* __restrict__ qn,
                                                         double* __restrict__ partials, BicgState* st, int it, int nb,
                                                         double tol, double atol) {
  const uint32_t n = (uint32_t)d.nx * d.ny * d.nz, stride = gridDim.x * blockDim.x;
  const uint32_t t0 = blockIdx.x * blockDim.x + threadIdx.x;
  const BicgPartials P{partials};
  const int done = st->done, maxiter = st->maxiter;
  const BicgScalars sc = st->s[it & 1];
  const double* const rr = P.rr((it + 1) & 1);
  const double atol2_prev = st->atol2;
  PartialShare<2> sh;
  PartialShare<1> shb;
  sh.request({rr, rr + kBicgBlocks}, nb);
  if (it == 0) shb.request({P.bb()}, nb);
  Stencil s[kBicgAhead];
  Seven rt[kBicgAhead], rv[kBicgAhead], pv[kBicgAhead], qv[kBicgAhead];
  float rh[kBicgAhead];
  auto fetch = [&](int e, uint32_t t) {
    s[e] = stencil_at(d, t);
    rt[e] = load_rtt(d, rtt, s[e]);
    rv[e] = load7(r, s[e]);
    pv[e] = load7(p, s[e]);
    qv[e] = load7(q, s[e]);
    rh[e] = ld32(rhat, t);
  };
#pragma unroll
  for (int e = 0; e < kBicgAhead; ++e) fetch(e, min(t0 + e * stride, n - 1));
  if (done) return;
  double a[2];
  sh.sum(a);
  const double rho_new = a[1];
  double atol2 = atol2_prev;
  if (it == 0) {
    double bb[1];
    shb.sum(bb);
    atol2 = fmax(tol * tol * bb[0], atol * atol);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (it == 0) st->atol2 = atol2;
    st->rho_new = rho_new;
  }
  if (!(a[0] > atol2 && sc.k < maxiter && sc.k >= 0)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      st->done = 1;
      st->k_final = sc.k;
    }
    return;
  }
  const double beta_d = rho_new / sc.rho * sc.alpha / sc.omega;
  const float beta = (float)beta_d, om = (float)sc.omega;
  double acc[1] = {0.0};
  auto cell = [&](int e, uint32_t t) {
    auto Pv = [&](float ro, float po, float qo) { return ro + beta * (po - om * qo); };
    const Seven& R = rv[e];
    const Seven& Q = pv[e];
    const Seven& W = qv[e];
    const Seven x{Pv(R.c, Q.c, W.c),    Pv(R.xm, Q.xm, W.xm), Pv(R.xp, Q.xp, W.xp), Pv(R.ym, Q.ym, W.ym),
                  Pv(R.yp, Q.yp, W.yp), Pv(R.zm, Q.zm, W.zm), Pv(R.zp, Q.zp, W.zp)};
    const float y = matvec7(d, s[e], rt[e], x);
    pn[t] = x.c;
    qn[t] = y;
    acc[0] += (double)rh[e] * y;
  };
#pragma unroll
  for (int e = 0; e < kBicgAhead; ++e)
    if (t0 + e * stride < n) cell(e, t0 + e * stride);
  for (uint32_t t = t0 + kBicgAhead * stride; t < n; t += stride) {
    fetch(0, t);
    cell(0, t);
  }
  put_partials<1>(acc, P.rq());
}

// K2: alpha = rho_new / rhat.q; s = r - alpha q (recomputed on the stencil), t = A(s);
// partials t.s, t.t, s.s
__global__ void __launch_bounds__(kBicgThreads) k_bicg_st(Dims d, const float* __restrict__ rtt,
                                                         const float* __restrict__ r, const float* __restrict__ q,
                                                         float* __restrict__ sv, float* __restrict__ tv,
                                                         double* __restrict__ partials, BicgState* st, int nb) {
  const uint32_t n = (uint32_t)d.nx * d.ny * d.nz, stride = gridDim.x * blockDim.x;
  const uint32_t t0 = blockIdx.x * blockDim.x + threadIdx.x;
  const BicgPartials P{partials};
  const int done = st->done;
  const double rho_new = st->rho_new;
  PartialShare<1> sh;
  sh.request({P.rq()}, nb);
  Stencil s[kBicgAhead];
  Seven rt[kBicgAhead], rv[kBicgAhead], qv[kBicgAhead];
  auto fetch = [&](int e, uint32_t t) {
    s[e] = stencil_at(d, t);
    rt[e] = load_rtt(d, rtt, s[e]);
    rv[e] = load7(r, s[e]);
    qv[e] = load7(q, s[e]);
  };
#pragma unroll
  for (int e = 0; e < kBicgAhead; ++e) fetch(e, min(t0 + e * stride, n - 1));
  if (done) return;
  double rq[1];
  sh.sum(rq);
  const double alpha = rho_new / rq[0];
  if (blockIdx.x == 0 && threadIdx.x == 0) st->alpha = alpha;
  const float al = (float)alpha;
  double acc[3] = {0.0, 0.0, 0.0};
  auto cell = [&](int e, uint32_t t) {
    auto Sv = [&](float ro, float qo) { return ro - al * qo; };
    const Seven& R = rv[e];
    const Seven& Q = qv[e];
    const Seven x{Sv(R.c, Q.c),   Sv(R.xm, Q.xm), Sv(R.xp, Q.xp), Sv(R.ym, Q.ym),
                  Sv(R.yp, Q.yp), Sv(R.zm, Q.zm), Sv(R.zp, Q.zp)};
    const float y = matvec7(d, s[e], rt[e], x);
    sv[t] = x.c;
    tv[t] = y;
    acc[0] += (double)y * x.c;
    acc[1] += (double)y * y;
    acc[2] += (double)x.c * x.c;
  };
#pragma unroll
  for (int e = 0; e < kBicgAhead; ++e)
    if (t0 + e * stride < n) cell(e, t0 + e * stride);
  for (uint32_t t = t0 + kBicgAhead * stride; t < n; t += stride) {
    fetch(0, t);
    cell(0, t);
  }
  put_partials<3>(acc, P.ts());
}

// K3: omega = t.s / t.t; x, r updates (early exit when |s|^2 < atol^2); partials r.r,
// rhat.r for the next iteration; block 0 advances the recurrence scalars
__global__ void __launch_bounds__(kBicgThreads) k_bicg_xr(long nl, const float* __restrict__ p,
                                                         const float* __restrict__ sv, const float* __restrict__ tv,
                                                         const float* __restrict__ rhat, float* __restrict__ x,
                                                         float* __restrict__ r, double* __restrict__ partials,
                                                         BicgState* st, int it, int nb) {
  const uint32_t n = (uint32_t)nl, stride = gridDim.x * blockDim.x;
  const uint32_t t0 = blockIdx.x * blockDim.x + threadIdx.x;
  const BicgPartials P{partials};
  const int done = st->done;
  const int k0 = st->s[it & 1].k;
  const double rho_new = st->rho_new, alpha_new = st->alpha, atol2 = st->atol2;
  PartialShare<3> sh;
  sh.request({P.ts(), P.ts() + kBicgBlocks, P.ts() + 2 * kBicgBlocks}, nb);
  float xv[kBicgAhead], pv[kBicgAhead], ss[kBicgAhead], tt[kBicgAhead], rh[kBicgAhead];
  auto fetch = [&](int e, uint32_t t) {
    xv[e] = ld32(x, t);
    pv[e] = ld32(p, t);
    ss[e] = ld32(sv, t);
    tt[e] = ld32(tv, t);
    rh[e] = ld32(rhat, t);
  };
#pragma unroll
  for (int e = 0; e < kBicgAhead; ++e) fetch(e, min(t0 + e * stride, n - 1));
  if (done) return;
  double a[3];   // t.s, t.t, s.s
  sh.sum(a);
  const double omega_new = a[0] / a[1];
  const bool early = a[2] < atol2;
  const float al = (float)alpha_new, om = (float)omega_new;
  double acc[2] = {0.0, 0.0};
  auto cell = [&](int e, uint32_t t) {
    float rn;
    if (early) {
      x[t] = xv[e] + al * pv[e];
      rn = ss[e];
    } else {
      x[t] = xv[e] + (al * pv[e] + om * ss[e]);
      rn = ss[e] - om * tt[e];
    }
    r[t] = rn;
    acc[0] += (double)rn * rn;
    acc[1] += (double)rh[e] * rn;
  };
#pragma unroll
  for (int e = 0; e < kBicgAhead; ++e)
    if (t0 + e * stride < n) cell(e, t0 + e * stride);
  for (uint32_t t = t0 + kBicgAhead * stride; t < n; t += stride) {
    fetch(0, t);
    cell(0, t);
  }
  put_partials<2>(acc, P.rr(it & 1));
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    int kn = (omega_new == 0.0 || alpha_new == 0.0) ? -11 : k0 + 1;
    if (rho_new == 0.0) kn = -10;
    BicgScalars nx;
    nx.rho = rho_new;
    nx.alpha = alpha_new;
    nx.omega = omega_new;
    nx.k = kn;
    nx.pad = 0;
    st->s[(it + 1) & 1] = nx;
  }
}

// after the host's loop: the exit code when no kernel ended the loop (maxiter reached)
__global__ void k_bicg_finish(BicgState* st, int iters) {
  if (threadIdx.x == 0 && blockIdx.x == 0 && !st->done) {
    st->done = 1;
    st->k_final = st->s[iters & 1].k;
  }
}

// ------------------------------ I1: base state -----------------------------------
// Hydrostatic base state in FP64 on one column (setup_lex.py:103-137): pi0 by the
// cumulative sum from pi=1 at the surface, qv0 = RH * rslf iterated to 1e-9.
__device__ double rslf_d(double p, double t) {
  double esl = 611.2 * exp(17.67 * (t - 273.15) / (t - 29.65));
  if (esl > p * 0.5) esl = p * 0.5;
  return (kRd / kRv) * esl / (p - esl);
}

__global__ void k_base_state(int nz, double dz, double theta0v, const double* __restrict__ rh, double* __restrict__ out,
                             int max_iter, double tol, double* iters) {
  // single thread: out holds 5 columns of nz+2 (pi0, rho0_theta0, rho0, theta0, qv0)
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double* pi0 = out;
  double* rt0 = out + (nz + 2);
  double* rho0 = out + 2 * (nz + 2);
  double* th0 = out + 3 * (nz + 2);
  double* qv0 = out + 4 * (nz + 2);
  for (int k = 0; k < nz + 2; ++k) {
    th0[k] = theta0v;
    qv0[k] = 0.0;
  }
  auto integrate = [&]() {
    double acc = 0.0, prev = 1.0;
    for (int k = 1; k <= nz; ++k) {
      double trho = th0[k] * (1.0 + kReps * qv0[k]) / (1.0 + qv0[k]);
      acc += -kG / kCp / trho;
      double cur = acc * dz + 1.0;
      pi0[k] = 0.5 * (prev + cur);
      prev = cur;
    }
    pi0[0] = pi0[1];
    pi0[nz + 1] = pi0[nz];
  };
  auto update_qv = [&](double* dst) {
    for (int k = 0; k < nz + 2; ++k)
      dst[k] = rslf_d(pow(pi0[k], kCp / kRd) * kP00, th0[k] * pi0[k]) * rh[k];
  };
  integrate();
  update_qv(qv0);
  // prev = 1.5 qv0; iterate while max|qv0 - prev| > tol
  double diff = 0.0;
  for (int k = 0; k < nz + 2; ++k) diff = fmax(diff, fabs(qv0[k] - 1.5 * qv0[k]));
  int it = 0;
  while (diff > tol && it < max_iter) {
    // keep the previous profile in rt0 as scratch
    for (int k = 0; k < nz + 2; ++k) rt0[k] = qv0[k];
    integrate();
    update_qv(qv0);
    diff = 0.0;
    for (int k = 0; k < nz + 2; ++k) diff = fmax(diff, fabs(qv0[k] - rt0[k]));
    ++it;
  }
  for (int k = 0; k < nz + 2; ++k) {
    double rt = pow(pi0[k], kCv / kRd) * kP00 / kRd;
    rho0[k] = rt / th0[k] / ((1.0 + kReps * qv0[k]) / (1.0 + qv0[k]));
    rt0[k] = rho0[k] * th0[k];  // setup_lex.py:64
  }
  *iters = (double)it;
}

}  // namespace lex
