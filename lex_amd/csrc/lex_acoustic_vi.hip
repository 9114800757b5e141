// solver_opt 3: vertically implicit acoustic substep (sound_implicit_rk_step0/1/2,
// one_step_integration.py:559-635, :678-754, :797-873).
//
// u and v are stepped forward as in the explicit substep; w and pi' are coupled
// implicitly in the vertical with off-centring alpha (namelist_n_constants.py:14), which
// leaves one tridiagonal system per column for the new w at levels 1..nz-1.  Columns are
// independent within a substep (the horizontal terms are explicit).  In k_acoustic_vi a workgroup
// owns one column: lane k holds cell k (its lower w level k), the column's pressure tendency
// and the system live in LDS, and the system is solved by parallel cyclic reduction
// (ceil(log2 nz) rounds of neighbour elimination at doubling distance, every lane one
// equation; the reference calls jax.lax.linalg.tridiagonal_solve).  Everything else -
// PGF, divergence, advection_pi, the 1.1 divergence damping, halos - is the explicit
// substep's arithmetic (k_acoustic).
#pragma once
#include "lex_common.hpp"
#include "lex_ops.hip"
#include "lex_acoustic_rows.hip"

namespace lex {

constexpr float kAlphaImplicit = 0.6f;  // off-centring of the implicit step (namelist_n_constants.py:14)

// column workgroup: nzl = 64 * ceil(nz / 64) lanes; LDS 6 * nzl + 1 floats
inline int acoustic_vi_lanes(const Dims& d) { return 64 * ((d.nz + 63) / 64); }
inline size_t acoustic_vi_lds(const Dims& d) { return (6 * (size_t)acoustic_vi_lanes(d) + 1) * sizeof(float); }

__device__ __forceinline__ float advpi_cell(float un0, float un1, float vn0, float vn1, float wn0, float wn1, float sc,
                                            float sxm, float sxp, float sym, float syp, float szm, float szp, float pim,
                                            float pic, float pip, float rcm, float rcc, float rcp, bool bottom, bool top,
                                            const Dims& d) {
  // advection_pi (advection.py:152-197) as in k_acoustic; the w term is zero at the lids
  float udx0 = un0 * ((sc - sxm) * d.idx);
  float udx1 = un1 * ((sxp - sc) * d.idx);
  float vdy0 = vn0 * ((sc - sym) * d.idy);
  float vdy1 = vn1 * ((syp - sc) * d.idy);
  float dz0 = (pic - pim) * d.idz + (sc - szm) * d.idz;
  float dz1 = (pip - pic) * d.idz + (szp - sc) * d.idz;
  float wdz0 = bottom ? 0.0f : wn0 * dz0;
  float wdz1 = top ? 0.0f : wn1 * dz1;
  float r8w0 = 0.5f * (rcm + rcc);
  float r8w1 = 0.5f * (rcc + rcp);
  return -(0.5f * (udx1 + udx0) + 0.5f * (vdy1 + vdy0) + (0.5f * wdz0 * r8w0 + 0.5f * wdz1 * r8w1) / rcc);
}

__global__ void __launch_bounds__(256) k_acoustic_vi(Dims d, const float* __restrict__ rc,
                                                     const float* __restrict__ pi0c, const float* __restrict__ u,
                                                     const float* __restrict__ v, const float* __restrict__ w,
                                                     const float* __restrict__ p, const float* __restrict__ ps,
                                                     const float* __restrict__ ru, const float* __restrict__ rv,
                                                     const float* __restrict__ rw, const float* __restrict__ tr,
                                                     float* __restrict__ uo, float* __restrict__ vo,
                                                     float* __restrict__ wo, float* __restrict__ po, float dts,
                                                     float alpha) {
  extern __shared__ float lds[];
  const int nzl = blockDim.x, nz = d.nz;
  float* A = lds;
  float* B = A + nzl;
  float* C = B + nzl;
  float* D = C + nzl;
  float* PT = D + nzl;   // pressure tendency with beta * w_now, per cell
  float* WN = PT + nzl;  // new w at levels 0..nz
  const TileId tb = xcd_tile();
  const int j = tb.x, i = tb.y;
  const int k = threadIdx.x;
  const bool act = k < nz;
  const int kc = act ? k : nz - 1;
  const int I = i + 3, J = j + 3, K = kc + 1;
  const long c = ic(d, I, J, K);
  const long sx = d.sxc(), sy = d.syc();
  const float beta = 1.0f - alpha;
  const float h = (float)(-kCp * 0.5);
  const float cr = (float)(-kRd / kCv);
  // ---- loads (all in bounds: levels K-2 .. K+1 clamped at 0)
  const float rcm = rc[K - 1], rcc = rc[K], rcp = rc[K + 1];
  const float pim2 = pi0c[max(K - 2, 0)], pim = pi0c[K - 1], pic = pi0c[K], pip = pi0c[K + 1];
  const long cu = iu(d, I, J, K), cv = iv(d, I, J, K), cw = iw(d, I, J, K);
  const long ou = ((long)i * d.ny + j) * nz + kc, ov = ((long)i * (d.ny + 1) + j) * nz + kc;
  const long ow = ((long)i * d.ny + j) * (nz + 1) + kc;
  const float u0 = u[cu], u1 = u[cu + d.sxu()], v0 = v[cv], v1 = v[cv + d.syc()], w0 = w[cw], w1 = w[cw + 1];
  const float ru0 = ru[ou], ru1 = ru[ou + (long)d.ny * nz], rv0 = rv[ov], rv1 = rv[ov + nz], rw0 = rw[ow];
  const float pc = p[c], pxm = p[c - sx], pxp = p[c + sx], pym = p[c - sy], pyp = p[c + sy], pzm = p[c - 1];
  const float tc = tr[c], txm = tr[c - sx], txp = tr[c + sx], tym = tr[c - sy], typ = tr[c + sy], tzm = tr[c - 1];
  const float sc = ps[c], sxm = ps[c - sx], sxp = ps[c + sx], sym = ps[c - sy], syp = ps[c + sy], szm = ps[c - 1],
              szp = ps[c + 1], szm2 = ps[c - (K >= 2 ? 2 : 1)];
  // ---- explicit u, v (pressure_gradient_force_horizontal with pi' now)
  const float un0 = u0 + (h * (tc + txm) * ((pc - pxm) * d.idx) + ru0) * dts;
  const float un1 = u1 + (h * (txp + tc) * ((pxp - pc) * d.idx) + ru1) * dts;
  const float vn0 = v0 + (h * (tc + tym) * ((pc - pym) * d.idy) + rv0) * dts;
  const float vn1 = v1 + (h * (typ + tc) * ((pyp - pc) * d.idy) + rv1) * dts;
  const bool bottom = kc == 0, top = kc == nz - 1;
  const float piadv = pic + sc;
  // ---- pressure tendency with beta * w_now (conv_mix + adv4pi_mix)
  {
    const float wb0 = beta * w0, wb1 = beta * w1;
    const float div = (un1 - un0) * d.idx + (vn1 - vn0) * d.idy + (wb1 - wb0) * d.idz;
    const float adv = advpi_cell(un0, un1, vn0, vn1, wb0, wb1, sc, sxm, sxp, sym, syp, szm, szp, pim, pic, pip, rcm,
                                 rcc, rcp, bottom, top, d);
    PT[k] = act ? cr * (piadv * div) + adv : 0.0f;
  }
  __syncthreads();
  // ---- the system at level l = k (1..nz-1): cells below (padded K-1) and above (K)
  float a = 0.f, bb = 1.f, cc = 0.f, dd = 0.f;
  if (act && k >= 1) {
    const float thr8w = 0.5f * (tc + tzm);
    const float lhs = (alpha * dts) * (alpha * dts) * (float)kCp * thr8w * d.idz;
    const float pa_m2 = pim2 + szm2, pa_m = pim + szm, pa_c = pic + sc, pa_p = pip + szp;
    const float rdcv = (float)(kRd / kCv);
    a = (k == 1) ? 0.0f : -lhs * (rdcv * pa_m * d.idz - (pa_m - pa_m2) * d.idz * 0.5f);
    cc = (k == nz - 1) ? 0.0f : -lhs * (rdcv * pa_c * d.idz + (pa_p - pa_c) * d.idz * 0.5f);
    bb = 1.0f + lhs * rdcv * (pa_c * d.idz + pa_m * d.idz);
    const float rhs3 = alpha * dts * dts * (float)kCp * thr8w;
    const float pw = h * (tc + tzm) * ((pc - pzm) * d.idz);
    dd = w0 + dts * (rw0 + pw) - rhs3 * ((PT[k] - PT[k - 1]) * d.idz);
  }
  // ---- parallel cyclic reduction over the column (rows 0 and >= nz are identity rows)
  for (int s = 1; s < nz; s <<= 1) {
    const bool hm = k - s >= 0, hp = k + s < nzl;
    __syncthreads();
    A[k] = a;
    B[k] = bb;
    C[k] = cc;
    D[k] = dd;
    __syncthreads();
    const float am = hm ? A[k - s] : 0.f, bm = hm ? B[k - s] : 1.f, cm = hm ? C[k - s] : 0.f, dm = hm ? D[k - s] : 0.f;
    const float ap = hp ? A[k + s] : 0.f, bp = hp ? B[k + s] : 1.f, cp = hp ? C[k + s] : 0.f, dp = hp ? D[k + s] : 0.f;
    const float k1 = a / bm, k2 = cc / bp;
    a = -am * k1;
    cc = -cp * k2;
    bb = bb - cm * k1 - ap * k2;
    dd = dd - dm * k1 - dp * k2;
  }
  WN[k] = (act && k >= 1) ? dd / bb : 0.0f;
  if (k == 0) WN[nz] = 0.0f;
  __syncthreads();
  if (!act) return;
  // ---- pi' with w_mix = alpha w_new + beta w_now
  const float wn0 = WN[k], wn1 = WN[k + 1];
  const float wm0 = alpha * wn0 + beta * w0, wm1 = alpha * wn1 + beta * w1;
  const float div = (un1 - un0) * d.idx + (vn1 - vn0) * d.idy + (wm1 - wm0) * d.idz;
  const float adv = advpi_cell(un0, un1, vn0, vn1, wm0, wm1, sc, sxm, sxp, sym, syp, szm, szp, pim, pic, pip, rcm,
                               rcc, rcp, bottom, top, d);
  const float pn = pc + 1.1f * (cr * (piadv * div) + adv) * dts;
  store_c_fast(d, po, i, j, k, pn);
  store_u_fast(d, uo, i, j, k, un0);
  if (i == d.nx - 1) store_u(d, uo, d.nx, j, k, un1);
  store_v_fast(d, vo, i, j, k, vn0);
  if (j == d.ny - 1) store_v(d, vo, i, d.ny, k, vn1);
  store_w_fast(d, wo, i, j, k, wn0);
  if (k == nz - 1) store_w(d, wo, i, j, nz, 0.0f);
}

// The same substep for columns of one wave (nz <= 64 V): a wave owns a row of y with V levels
// per lane and marches along x as in k_acoustic, every face evaluated once and nothing in LDS.
// The tridiagonal system has its rows scaled to a unit diagonal, so a round of reduction
// exchanges three coefficients and needs one reciprocal; with two levels per lane the odd rows
// are first eliminated within the lanes, and the 64 even rows left take the parallel reduction.
// The workgroup-per-column form waited on two barriers and eight LDS reads in each of its
// seven rounds, with three IEEE divisions.

// 1 / b to within a rounding: the hardware's estimate and one Newton step.
__device__ __forceinline__ float recip(float b) {
  const float r = __builtin_amdgcn_rcpf(b);
  return fmaf(fmaf(-b, r, 1.0f), r, r);
}

// x_l + a x_(l-1) + c x_(l+1) = d over the first n lanes; a of lane 0 and c of lane n - 1 are 0.
__device__ __forceinline__ float solve_lanes(float a, float c, float d, int n) {
  for (int s = 1; s < n; s <<= 1) {
    float am, cm, dm, ap, cp, dp;
    if (s == 1) {
      am = lane_below(a);
      cm = lane_below(c);
      dm = lane_below(d);
      ap = lane_above(a);
      cp = lane_above(c);
      dp = lane_above(d);
    } else {
      am = __shfl_up(a, s, 64);
      cm = __shfl_up(c, s, 64);
      dm = __shfl_up(d, s, 64);
      ap = __shfl_down(a, s, 64);
      cp = __shfl_down(c, s, 64);
      dp = __shfl_down(d, s, 64);
    }
    const float ib = recip(fmaf(-c, ap, fmaf(-a, cm, 1.0f)));
    d = fmaf(-c, dp, fmaf(-a, dm, d)) * ib;
    a = -a * am * ib;
    c = -c * cp * ib;
  }
  return d;
}

template <int V>
__global__ void __launch_bounds__(256) k_acoustic_vi_rows(Dims d, AcousticArgs g, float alpha, int ax) {
  const int lane = threadIdx.x;
  const TileId tb = xcd_tile();
  const int j = __builtin_amdgcn_readfirstlane(tb.x * (int)blockDim.y + (int)threadIdx.y);
  const int nx = d.nx, ny = d.ny, nz = d.nz;
  if (j >= ny) return;
  const int x0 = tb.y * ax, x1 = min(x0 + ax, nx);
  const int kl = lane * V;
  const int kc = min(kl, nz - 1);
  LevelSlots ls;
  ls.n = min(max(nz - kl, 0), V);
  ls.first = kl == 0;
  ls.last = ls.n > 0 && kl + ls.n == nz;
  const uint32_t eK = (uint32_t)(kc + 1);
  const uint32_t ek = (uint32_t)min(kc, nz - V);
  const bool past = (V == 2) && kc == nz - 1;
  const float dts = g.dts, beta = 1.0f - alpha;
  const float h = (float)(-kCp * 0.5), cr = (float)(-kRd / kCv), rdcv = (float)(kRd / kCv);
  const float lh = (alpha * dts) * (alpha * dts) * (float)kCp, rh = alpha * dts * dts * (float)kCp;
  float rr[V], ir[V], r8[V], pic[V], dpi[V];
#pragma unroll
  for (int q = 0; q < V; ++q) {
    const int K = min(kc + q + 1, nz + 1);
    rr[q] = g.rc[K];
    ir[q] = 1.0f / rr[q];
    r8[q] = 0.5f * (g.rc[K - 1] + rr[q]);
    pic[q] = g.pi0[K];
    dpi[q] = (pic[q] - g.pi0[K - 1]) * d.idz;
  }
  const int syc = nz + 2, syw = nz + 3;
  const int sxc = (ny + 6) * syc, sxv = (ny + 7) * syc, sxw = (ny + 6) * syw;
  const int sxiu = ny * nz, sxiv = (ny + 1) * nz, sxiw = ny * (nz + 1);
  const uint32_t oc = (uint32_t)((j + 3) * syc) + eK, ocm = oc - (uint32_t)syc, ocp = oc + (uint32_t)syc;
  const uint32_t ow = (uint32_t)((j + 3) * syw) + eK;
  const uint32_t oi = (uint32_t)(j * nz) + ek, oin = oi + (uint32_t)nz;
  const uint32_t og = (uint32_t)(j * (nz + 1) + kc);
  // w as it is read: lanes above the column hold the lid level
  const uint32_t owr = (uint32_t)((j + 3) * syw + min(kl, nz) + 1);
  const bool top63 = ls.last && lane == 63;
  const float *pX = g.p + (long)(x0 + 3) * sxc, *tX = g.tr + (long)(x0 + 3) * sxc, *sX = g.ps + (long)(x0 + 3) * sxc;
  const float *uX = g.u + (long)(x0 + 3) * sxc, *guX = g.ru + (long)x0 * sxiu;
  const float *vX = g.v + (long)(x0 + 3) * sxv, *gvX = g.rv + (long)x0 * sxiv;
  const float *wX = g.w + (long)(x0 + 3) * sxw, *gwX = g.rw + (long)x0 * sxiw;
  float P0[V], T0[V], S0[V], ul[V], dl[V];
  {
    float pm[V], tm[V], sm[V], u0[V], g0[V];
    ld_levels<V>(pX, oc, P0);
    ld_levels<V>(tX, oc, T0);
    ld_levels<V>(sX, oc, S0);
    ld_levels<V>(pX - sxc, oc, pm);
    ld_levels<V>(tX - sxc, oc, tm);
    ld_levels<V>(sX - sxc, oc, sm);
    ld_levels<V>(uX, oc, u0);
    ld_levels_in<V>(guX, oi, past, g0);
#pragma unroll
    for (int q = 0; q < V; ++q) {
      ul[q] = u0[q] + (h * (T0[q] + tm[q]) * ((P0[q] - pm[q]) * d.idx) + g0[q]) * dts;
      dl[q] = ul[q] * ((S0[q] - sm[q]) * d.idx);
    }
  }
#pragma unroll 1
  for (int x = x0; x < x1; ++x) {
    float p1[V], t1[V], s1[V], py[2][V], ty[2][V], sy[2][V], uf[V], gu[V], vf[2][V], gv[2][V], wf[V], gw[V];
    float wlid = 0.0f;
    ld_levels<V>(pX, ocm, py[0]);
    ld_levels<V>(tX, ocm, ty[0]);
    ld_levels<V>(sX, ocm, sy[0]);
    ld_levels<V>(pX, ocp, py[1]);
    ld_levels<V>(tX, ocp, ty[1]);
    ld_levels<V>(sX, ocp, sy[1]);
    ld_levels<V>(vX, oc, vf[0]);
    ld_levels<V>(vX, ocp, vf[1]);
    ld_levels_in<V>(gvX, oi, past, gv[0]);
    ld_levels_in<V>(gvX, oin, past, gv[1]);
    ld_levels<V>(wX, owr, wf);
    ld_levels<V>(gwX, og, gw);
    if (top63) wlid = ld32(wX, owr + (uint32_t)ls.n);
    pX += sxc;
    tX += sxc;
    sX += sxc;
    uX += sxc;
    guX += sxiu;
    vX += sxv;
    gvX += sxiv;
    wX += sxw;
    gwX += sxiw;
    ld_levels<V>(pX, oc, p1);
    ld_levels<V>(tX, oc, t1);
    ld_levels<V>(sX, oc, s1);
    ld_levels<V>(uX, oc, uf);
    ld_levels_in<V>(guX, oi, past, gu);
    // explicit u, v; the horizontal part of the divergence and of the advection of pi
    float un[V], vn[2][V], hdiv[V], hadv[V], us[V];
#pragma unroll
    for (int q = 0; q < V; ++q) {
      un[q] = uf[q] + (h * (t1[q] + T0[q]) * ((p1[q] - P0[q]) * d.idx) + gu[q]) * dts;
      vn[0][q] = vf[0][q] + (h * (T0[q] + ty[0][q]) * ((P0[q] - py[0][q]) * d.idy) + gv[0][q]) * dts;
      vn[1][q] = vf[1][q] + (h * (ty[1][q] + T0[q]) * ((py[1][q] - P0[q]) * d.idy) + gv[1][q]) * dts;
      const float du = un[q] * ((s1[q] - S0[q]) * d.idx);
      const float dv0 = vn[0][q] * ((S0[q] - sy[0][q]) * d.idy), dv1 = vn[1][q] * ((sy[1][q] - S0[q]) * d.idy);
      hdiv[q] = (un[q] - ul[q]) * d.idx + (vn[1][q] - vn[0][q]) * d.idy;
      hadv[q] = 0.5f * (du + dl[q]) + 0.5f * (dv1 + dv0);
      us[q] = ul[q];
      ul[q] = un[q];
      dl[q] = du;
    }
    // z neighbours: the level below (and two below), the level above
    float pa[V], pz[V], tz[V], sz[V], pab[V], pabb[V], pat[V], dz[V];
#pragma unroll
    for (int q = 0; q < V; ++q) pa[q] = pic[q] + S0[q];
    pz[0] = lane_below(P0[V - 1]);
    tz[0] = lane_below(T0[V - 1]);
    sz[0] = lane_below(S0[V - 1]);
    pab[0] = lane_below(pa[V - 1]);
    pat[V - 1] = lane_above(pa[0]);
    if (V == 2) {
      pz[V - 1] = P0[0];
      tz[V - 1] = T0[0];
      sz[V - 1] = S0[0];
      pabb[0] = lane_below(pa[0]);
      pabb[V - 1] = pab[0];
      pab[V - 1] = pa[0];
      pat[0] = pa[V - 1];
    } else {
      pabb[0] = lane_below(pab[0]);
    }
    // pressure tendency of a vertical velocity wl at the lower and wu at the upper level of
    // every cell; the advection's vertical part vanishes at the surface and the lid
    auto tendency = [&](const float(&wl)[V], const float(&wu)[V], float(&out)[V]) {
      float fz[V];
#pragma unroll
      for (int q = 0; q < V; ++q) fz[q] = (kl + q == 0) ? 0.0f : 0.5f * (wl[q] * dz[q]) * r8[q];
      const float ft = lane_above(fz[0]);
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const float f1 = (kl + q >= nz - 1) ? 0.0f : (q < V - 1 ? fz[V - 1] : ft);
        const float div = hdiv[q] + (wu[q] - wl[q]) * d.idz;
        out[q] = cr * (pa[q] * div) - (hadv[q] + quotient(fz[q] + f1, rr[q], ir[q]));
      }
    };
    float wu[V], wb0[V], wb1[V], pt[V];
    {
      const float wa = lane_above(wf[0]);
#pragma unroll
      for (int q = 0; q < V; ++q) {
        dz[q] = dpi[q] + (S0[q] - sz[q]) * d.idz;
        wu[q] = q < V - 1 ? wf[V - 1] : (top63 ? wlid : wa);
        wb0[q] = beta * wf[q];
        wb1[q] = beta * wu[q];
      }
    }
    tendency(wb0, wb1, pt);
    // the system at levels 1 .. nz - 1, scaled to a unit diagonal; elsewhere the value is 0
    float A[V], C[V], D[V];
    const float ptb = lane_below(pt[V - 1]);
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const int l = kl + q;
      const bool row = l >= 1 && l < nz;
      const float thr8w = 0.5f * (T0[q] + tz[q]);
      const float lhs = lh * thr8w * d.idz;
      const float a = -lhs * (rdcv * pab[q] * d.idz - (pab[q] - pabb[q]) * d.idz * 0.5f);
      const float c = -lhs * (rdcv * pa[q] * d.idz + (pat[q] - pa[q]) * d.idz * 0.5f);
      const float ib = recip(1.0f + lhs * rdcv * (pa[q] * d.idz + pab[q] * d.idz));
      const float pw = h * (T0[q] + tz[q]) * ((P0[q] - pz[q]) * d.idz);
      const float dd = wf[q] + dts * (gw[q] + pw) - rh * thr8w * ((pt[q] - (q ? pt[0] : ptb)) * d.idz);
      A[q] = (row && l > 1) ? a * ib : 0.0f;
      C[q] = (row && l < nz - 1) ? c * ib : 0.0f;
      D[q] = row ? dd * ib : 0.0f;
    }
    float wn[V];
    if (V == 1) {
      wn[0] = solve_lanes(A[0], C[0], D[0], nz);
    } else {
      const float ao = lane_below(A[V - 1]), co = lane_below(C[V - 1]), od = lane_below(D[V - 1]);
      const float ib = recip(fmaf(-A[0], co, fmaf(-C[0], A[V - 1], 1.0f)));
      wn[0] = solve_lanes(-A[0] * ao * ib, -C[0] * C[V - 1] * ib, fmaf(-A[0], od, fmaf(-C[0], D[V - 1], D[0])) * ib,
                          (nz + 1) / 2);
      wn[V - 1] = fmaf(-C[V - 1], lane_above(wn[0]), fmaf(-A[V - 1], wn[0], D[V - 1]));
    }
    // pi' with w_mix = alpha w_new + beta w_now
    float pn[V], wm0[V], wm1[V];
    const float wa = lane_above(wn[0]);
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const float w1 = (kl + q >= nz - 1) ? 0.0f : (q < V - 1 ? wn[V - 1] : wa);
      wm0[q] = alpha * wn[q] + wb0[q];
      wm1[q] = alpha * w1 + wb1[q];
    }
    tendency(wm0, wm1, pt);
#pragma unroll
    for (int q = 0; q < V; ++q) {
      pn[q] = P0[q] + 1.1f * pt[q] * dts;
      P0[q] = p1[q];
      T0[q] = t1[q];
      S0[q] = s1[q];
    }
    if (x >= 4 && x < nx - 3 && j >= 4 && j < ny - 3) {   // no periodic images
      float *poX = g.po + (long)(x + 3) * sxc, *uoX = g.uo + (long)(x + 3) * sxc;
      float *voX = g.vo + (long)(x + 3) * sxv, *woX = g.wo + (long)(x + 3) * sxw;
      st_levels<V>(poX, oc, ls, pn);
      st_levels<V>(uoX, oc, ls, us);
      st_levels<V>(voX, oc, ls, vn[0]);
      st_levels<V>(woX, ow, ls, wn);
      if (ls.first || ls.last) {
        st_ghosts<V>(poX, oc, ls, pn);
        st_ghosts<V>(uoX, oc, ls, us);
        st_ghosts<V>(voX, oc, ls, vn[0]);
        st_ghosts_w<V>(woX, ow, ls, wn);
      }
    } else {
      st_images<V, false>(g.po, sxc, syc, x, nx, false, j, ny, false, eK, ls, pn);
      st_images<V, false>(g.uo, sxc, syc, x, nx, true, j, ny, false, eK, ls, us);
      if (x == nx - 1) st_images<V, false>(g.uo, sxc, syc, nx, nx, true, j, ny, false, eK, ls, un);
      st_images<V, false>(g.vo, sxv, syc, x, nx, false, j, ny, true, eK, ls, vn[0]);
      if (j == ny - 1) st_images<V, false>(g.vo, sxv, syc, x, nx, false, ny, ny, true, eK, ls, vn[1]);
      st_images<V, true>(g.wo, sxw, syw, x, nx, false, j, ny, false, eK, ls, wn);
    }
  }
}

// us per substep, a workgroup per column (left, kept for nz > 128) and rows: 40x40x40 10.4 and
// 10.2, 96x96x48 17.9 and 13.8, 128x128x64 25.7 and 19.6, 181x147x71 63 and 42, 192x160x96 71
// and 44, 256x256x128 158 and 112.
inline void launch_acoustic_vi(const Dims& d, const AcousticArgs& a, float alpha, hipStream_t st) {
  if (d.nz > 128) {
    LEX_LAUNCH(KID_ACOUSTIC_VI, k_acoustic_vi, dim3(d.ny, d.nx, 1), dim3(acoustic_vi_lanes(d)), acoustic_vi_lds(d), st,
               d, a.rc, a.pi0, a.u, a.v, a.w, a.p, a.ps, a.ru, a.rv, a.rw, a.tr, a.uo, a.vo, a.wo, a.po, a.dts, alpha);
    return;
  }
  const int ax = (int)std::min(4L, std::max(1L, ((long)d.nx * d.ny + 8192) / 16384));   // as k_acoustic
  const dim3 g((d.ny + 3) / 4, (d.nx + ax - 1) / ax), b(64, 4);
  if (d.nz > 64)
    LEX_LAUNCH(KID_ACOUSTIC_VI, k_acoustic_vi_rows<2>, g, b, 0, st, d, a, alpha, ax);
  else
    LEX_LAUNCH(KID_ACOUSTIC_VI, k_acoustic_vi_rows<1>, g, b, 0, st, d, a, alpha, ax);
}

}  // namespace lex
