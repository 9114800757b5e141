// S1: one forward-backward acoustic substep (one_step_integration.py:528-553), V levels per
// lane, marched along x.
//
// A wave owns one row of y and 64 V levels, lane l the levels V l .. V l + V - 1, and marches
// `ax` cells along x with no barrier and no LDS: the x neighbours and the x face below are
// carried in registers, the z neighbours are the lane's other level or the adjacent lane's
// (a wave shift in the vector pipe), and the x and z faces are evaluated once.  Two levels
// per lane halve the vector-memory instructions, which kept the address unit of the
// cell-per-thread form 77 % busy (29 loads per cell; here 10 for one level, 20 of 8 bytes
// for two).
//
// Contraction is spelled out (fmaf) and otherwise off, in k_acoustic, in k_acoustic_cells and
// in both substeps of k_acoustic2, so the results do not depend on which of them computed a cell.
#pragma once
#include <algorithm>
#include "lex_ops.hip"
#include "lex_prof.hpp"

namespace lex {

// Two floats at a 4-byte aligned address in one access.
struct __attribute__((packed, aligned(4))) Pair32 {
  float x, y;
};

template <int V>
__device__ __forceinline__ void ld_levels(const float* __restrict__ row, uint32_t e, float (&o)[V]) {
  if constexpr (V == 1) {
    o[0] = ld32(row, e);
  } else {
    const Pair32 t = *reinterpret_cast<const Pair32*>(reinterpret_cast<const char*>(row) + (size_t)(e * 4u));
    o[0] = t.x;
    o[1] = t.y;
  }
}
// The same from an unpadded row: the lane whose second level would lie past the row (odd nz)
// reads one level lower (e already is) and takes the upper value as its first.
template <int V>
__device__ __forceinline__ void ld_levels_in(const float* __restrict__ row, uint32_t e, bool past, float (&o)[V]) {
  ld_levels<V>(row, e, o);
  if constexpr (V == 2) o[0] = past ? o[1] : o[0];
}

// The value of the lane below / above (DPP wave shift by one); lane 0 / 63 get 0.
__device__ __forceinline__ float lane_below(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_above(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, false));
}

// Where a lane's levels go in a padded column: n of its V levels exist, the first / last of
// the column also fill the z ghosts.
struct LevelSlots {
  int n;
  bool first, last;
};

// Store the lane's levels at element e (its first level) of a padded field.
template <int V>
__device__ __forceinline__ void st_levels(float* __restrict__ f, uint32_t e, const LevelSlots& s, const float (&val)[V]) {
  if (V == 2 && s.n == 2) {
    Pair32 t;
    t.x = val[0];
    t.y = val[V - 1];
    *reinterpret_cast<Pair32*>(reinterpret_cast<char*>(f) + (size_t)(e * 4u)) = t;
  } else if (s.n >= 1) {
    st32(f, e, val[0]);
  }
}
// The z ghosts of a column: copies of its first and last level.
template <int V>
__device__ __forceinline__ void st_ghosts(float* __restrict__ f, uint32_t e, const LevelSlots& s, const float (&val)[V]) {
  if (s.first) st32(f, e - 1u, val[0]);
  if (s.last) st32(f, e + (uint32_t)s.n, (V == 2 && s.n == 2) ? val[V - 1] : val[0]);
}
// w: the lid level and its ghost above the last cell are zero.
template <int V>
__device__ __forceinline__ void st_ghosts_w(float* __restrict__ f, uint32_t e, const LevelSlots& s, const float (&val)[V]) {
  if (s.first) st32(f, e - 1u, val[0]);
  if (s.last) {
    st32(f, e + (uint32_t)s.n, 0.0f);
    st32(f, e + (uint32_t)s.n + 1u, 0.0f);
  }
}

// Periodic images of index i on an axis of n cells (face: of n + 1 faces, whose ghosts skip
// the duplicate), as a mask: bit 0 the point itself, 1 its image one period up, 2 down.
__device__ __forceinline__ int image_mask(int i, int n, bool face) {
  if (face) return 1 | ((i >= 1 && i <= 3) ? 2 : 0) | ((i >= n - 3 && i <= n - 1) ? 4 : 0);
  return 1 | (i < 3 ? 2 : 0) | (i >= n - 3 ? 4 : 0);
}

// Store a column of point (i, j) and its periodic images; i, j uniform over the wave, sx and
// sy the field's strides, e the lane's first level within a column.
template <int V, bool ONW>
__device__ __forceinline__ void st_images(float* __restrict__ f, int sx, int sy, int i, int nx, bool fx, int j, int ny,
                                          bool fy, uint32_t e, const LevelSlots& s, const float (&val)[V]) {
  const int mx = image_mask(i, nx, fx), my = image_mask(j, ny, fy);
#pragma unroll 1
  for (int a = 0; a < 3; ++a) {
    if (!((mx >> a) & 1)) continue;
    const int X = i + 3 + (a == 1 ? nx : (a == 2 ? -nx : 0));
#pragma unroll 1
    for (int b = 0; b < 3; ++b) {
      if (!((my >> b) & 1)) continue;
      const int Y = j + 3 + (b == 1 ? ny : (b == 2 ? -ny : 0));
      const uint32_t o = (uint32_t)(X * sx + Y * sy) + e;
      st_levels<V>(f, o, s, val);
      if (ONW)
        st_ghosts_w<V>(f, o, s, val);
      else
        st_ghosts<V>(f, o, s, val);
    }
  }
}

// MZ: the column spans several waves (nz > 64 V), whose edge lanes load their outer z
// neighbours.
template <int V, bool MZ>
__global__ void __launch_bounds__(256) k_acoustic(Dims d, const float* __restrict__ rc, const float* __restrict__ pi0c,
                                                  const float* __restrict__ u, const float* __restrict__ v,
                                                  const float* __restrict__ w, const float* __restrict__ p,
                                                  const float* __restrict__ ps, const float* __restrict__ ru,
                                                  const float* __restrict__ rv, const float* __restrict__ rw,
                                                  const float* __restrict__ tr, float* __restrict__ uo,
                                                  float* __restrict__ vo, float* __restrict__ wo,
                                                  float* __restrict__ po, float dts, int ax) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x;
  const TileId tb = xcd_tile();
  const int j = __builtin_amdgcn_readfirstlane(tb.x * (int)blockDim.y + (int)threadIdx.y);
  const int nx = d.nx, ny = d.ny, nz = d.nz;
  if (j >= ny) return;
  const int x0 = tb.y * ax, x1 = min(x0 + ax, nx);
  const int kl = (tb.z * 64 + lane) * V;         // the lane's first level
  const int kc = min(kl, nz - 1);                // idle lanes repeat the last level
  LevelSlots ls;
  ls.n = min(max(nz - kl, 0), V);
  ls.first = kl == 0;
  ls.last = ls.n > 0 && kl + ls.n == nz;
  const uint32_t eK = (uint32_t)(kc + 1);        // padded level of the lane's first level
  const uint32_t ek = (uint32_t)min(kc, nz - V); // its level in an unpadded row
  const bool past = (V == 2) && kc == nz - 1;
  // column constants: reciprocal density, density at the lower w level, pi0 and its lower gradient
  const float h = (float)(-kCp * 0.5);
  float rr[V], ir[V], r8[V], pic[V], dpi[V];
#pragma unroll
  for (int q = 0; q < V; ++q) {
    const int K = min(kc + q + 1, nz + 1);
    rr[q] = rc[K];
    ir[q] = 1.0f / rr[q];
    r8[q] = 0.5f * (rc[K - 1] + rr[q]);
    pic[q] = pi0c[K];
    dpi[q] = (pic[q] - pi0c[K - 1]) * d.idz;
  }
  float r8e = 0.f, dpie = 0.f;   // of the level above the lane's last
  if (MZ) {
    const int K = min(kc + V + 1, nz + 1);
    r8e = 0.5f * (rc[K - 1] + rc[K]);
    dpie = (pi0c[K] - pi0c[K - 1]) * d.idz;
  }
  const bool edge = MZ && (lane == 0 || lane == 63);
  const uint32_t eE = (uint32_t)(lane == 0 ? kc : min(kc + V + 1, nz + 1));
  const uint32_t eW = (uint32_t)min(kc + V, nz);

  const int syc = nz + 2, syw = nz + 3;
  const int sxc = (ny + 6) * syc, sxv = (ny + 7) * syc, sxw = (ny + 6) * syw;
  const int sxiu = ny * nz, sxiv = (ny + 1) * nz, sxiw = ny * (nz + 1);
  // lane offsets within an x-plane: oc the cell rows j-1, j, j+1 (oc[1], oc[2] also the v
  // faces j, j+1 and oc[1] the u row), ow the w row, oi the unpadded row and og rw's
  const uint32_t oc[3] = {(uint32_t)((j + 2) * syc) + eK, (uint32_t)((j + 3) * syc) + eK, (uint32_t)((j + 4) * syc) + eK};
  const uint32_t ow = (uint32_t)((j + 3) * syw) + eK;
  const uint32_t oi = (uint32_t)(j * nz) + ek, oin = oi + (uint32_t)nz;
  const uint32_t og = (uint32_t)(j * (nz + 1) + kc);
  // the planes of x (cells, v, w) and of x + 1 (cells and u), advanced with the march
  const float *pX = p + (long)(x0 + 3) * sxc, *tX = tr + (long)(x0 + 3) * sxc, *sX = ps + (long)(x0 + 3) * sxc;
  const float *uX = u + (long)(x0 + 3) * sxc, *guX = ru + (long)x0 * sxiu;
  const float *vX = v + (long)(x0 + 3) * sxv, *gvX = rv + (long)x0 * sxiv;
  const float *wX = w + (long)(x0 + 3) * sxw, *gwX = rw + (long)x0 * sxiw;
  float *poX = po + (long)(x0 + 3) * sxc, *uoX = uo + (long)(x0 + 3) * sxc, *voX = vo + (long)(x0 + 3) * sxv,
        *woX = wo + (long)(x0 + 3) * sxw;

  float P0[3][V], T0[3][V], S0[3][V];   // plane x, rows j-1, j, j+1
  float ul[V], dl[V];                   // new u at face x and u dpi*/dx there
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    ld_levels<V>(pX, oc[r], P0[r]);
    ld_levels<V>(tX, oc[r], T0[r]);
    ld_levels<V>(sX, oc[r], S0[r]);
  }
  {
    float pm[V], tm[V], sm[V], u0[V], g0[V];
    ld_levels<V>(pX - sxc, oc[1], pm);
    ld_levels<V>(tX - sxc, oc[1], tm);
    ld_levels<V>(sX - sxc, oc[1], sm);
    ld_levels<V>(uX, oc[1], u0);
    ld_levels_in<V>(guX, oi, past, g0);
#pragma unroll
    for (int q = 0; q < V; ++q) {
      ul[q] = fmaf(fmaf(h * (T0[1][q] + tm[q]), (P0[1][q] - pm[q]) * d.idx, g0[q]), dts, u0[q]);
      dl[q] = ul[q] * ((S0[1][q] - sm[q]) * d.idx);
    }
  }
#pragma unroll 1
  for (int x = x0; x < x1; ++x) {
    float P1[3][V], T1[3][V], S1[3][V], uf[V], gu[V];
    float vf[2][V], gv[2][V], wf[V], gw[V];
    float pe, te, se, we, ge;
    ld_levels<V>(vX, oc[1], vf[0]);
    ld_levels<V>(vX, oc[2], vf[1]);
    ld_levels_in<V>(gvX, oi, past, gv[0]);
    ld_levels_in<V>(gvX, oin, past, gv[1]);
    ld_levels<V>(wX, ow, wf);
    ld_levels<V>(gwX, og, gw);
    if (edge) {
      pe = ld32(pX, oc[1] - eK + eE);
      te = ld32(tX, oc[1] - eK + eE);
      se = ld32(sX, oc[1] - eK + eE);
      we = ld32(wX, ow - eK + eW + 1u);
      ge = ld32(gwX, og - (uint32_t)kc + eW);
    }
    pX += sxc;
    tX += sxc;
    sX += sxc;
    uX += sxc;
    guX += sxiu;
    vX += sxv;
    gvX += sxiv;
    wX += sxw;
    gwX += sxiw;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      ld_levels<V>(pX, oc[r], P1[r]);
      ld_levels<V>(tX, oc[r], T1[r]);
      ld_levels<V>(sX, oc[r], S1[r]);
    }
    ld_levels<V>(uX, oc[1], uf);
    ld_levels_in<V>(guX, oi, past, gu);
    // y faces j, j+1
    float vn[2][V], dv[2][V];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int q = 0; q < V; ++q) {
        vn[r][q] = fmaf(fmaf(h * (T0[r + 1][q] + T0[r][q]), (P0[r + 1][q] - P0[r][q]) * d.idy, gv[r][q]), dts, vf[r][q]);
        dv[r][q] = vn[r][q] * ((S0[r + 1][q] - S0[r][q]) * d.idy);
      }
    const float(&pc)[V] = P0[1];
    const float(&tc)[V] = T0[1];
    const float(&sc)[V] = S0[1];
    // lower z faces: new w, and its pi* term (half, then times the density)
    float wn[V], a0[V], b0[V];
    float pb = lane_below(pc[V - 1]), tb_ = lane_below(tc[V - 1]), sb = lane_below(sc[V - 1]);
    if (MZ && lane == 0) {
      pb = pe;
      tb_ = te;
      sb = se;
    }
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const float pl = q ? pc[0] : pb, tl = q ? tc[0] : tb_, sl = q ? sc[0] : sb;
      const float pz = h * (tc[q] + tl) * ((pc[q] - pl) * d.idz);
      const float wv = fmaf(pz + gw[q], dts, wf[q]);
      const float dz = fmaf(sc[q] - sl, d.idz, dpi[q]);
      const bool floor_ = q == 0 && kl == 0;
      wn[q] = floor_ ? 0.0f : wv;
      a0[q] = 0.5f * (floor_ ? 0.0f : wv * dz);
      b0[q] = a0[q] * r8[q];
    }
    float wt = lane_above(wn[0]), bt = lane_above(b0[0]);
    if (MZ && lane == 63) {
      const float pz = h * (te + tc[V - 1]) * ((pe - pc[V - 1]) * d.idz);
      wt = fmaf(pz + ge, dts, we);
      bt = (0.5f * (wt * fmaf(se - sc[V - 1], d.idz, dpie))) * r8e;
    }
    float un[V], pn[V], us[V];
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const bool lid = kl + q >= nz - 1;
      const float w1 = lid ? 0.0f : (q < V - 1 ? wn[V - 1] : wt);
      const float b1 = lid ? 0.0f : (q < V - 1 ? b0[V - 1] : bt);
      un[q] = fmaf(fmaf(h * (T1[1][q] + tc[q]), (P1[1][q] - pc[q]) * d.idx, gu[q]), dts, uf[q]);
      const float du = un[q] * ((S1[1][q] - sc[q]) * d.idx);
      const float div = fmaf(w1 - wn[q], d.idz, fmaf(vn[1][q] - vn[0][q], d.idy, (un[q] - ul[q]) * d.idx));
      const float z = quotient(fmaf(a0[q], r8[q], b1), rr[q], ir[q]);
      const float advp = -(fmaf(0.5f, du + dl[q], 0.5f * (dv[1][q] + dv[0][q])) + z);
      const float dpdt = fmaf((float)(-kRd / kCv), (pic[q] + sc[q]) * div, advp);
      pn[q] = fmaf(1.1f * dpdt, dts, pc[q]);
      us[q] = ul[q];
      ul[q] = un[q];
      dl[q] = du;
    }
    if (x >= 4 && x < nx - 3 && j >= 4 && j < ny - 3) {   // no periodic images
      st_levels<V>(poX, oc[1], ls, pn);
      st_levels<V>(uoX, oc[1], ls, us);
      st_levels<V>(voX, oc[1], ls, vn[0]);
      st_levels<V>(woX, ow, ls, wn);
      if (ls.first || ls.last) {
        st_ghosts<V>(poX, oc[1], ls, pn);
        st_ghosts<V>(uoX, oc[1], ls, us);
        st_ghosts<V>(voX, oc[1], ls, vn[0]);
        st_ghosts_w<V>(woX, ow, ls, wn);
      }
    } else {
      st_images<V, false>(po, sxc, syc, x, nx, false, j, ny, false, eK, ls, pn);
      st_images<V, false>(uo, sxc, syc, x, nx, true, j, ny, false, eK, ls, us);
      if (x == nx - 1) st_images<V, false>(uo, sxc, syc, nx, nx, true, j, ny, false, eK, ls, un);
      st_images<V, false>(vo, sxv, syc, x, nx, false, j, ny, true, eK, ls, vn[0]);
      if (j == ny - 1) st_images<V, false>(vo, sxv, syc, x, nx, false, ny, ny, true, eK, ls, vn[1]);
      st_images<V, true>(wo, sxw, syw, x, nx, false, j, ny, false, eK, ls, wn);
    }
    poX += sxc;
    uoX += sxc;
    voX += sxv;
    woX += sxw;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int q = 0; q < V; ++q) {
        P0[r][q] = P1[r][q];
        T0[r][q] = T1[r][q];
        S0[r][q] = S1[r][q];
      }
  }
}

// The same substep with a thread per cell, which evaluates every face twice and loads 29 values
// at once: for columns of more than two waves.
__global__ void __launch_bounds__(256) k_acoustic_cells(Dims d, const float* __restrict__ rc,
                                                        const float* __restrict__ pi0c, const float* __restrict__ u,
                                                        const float* __restrict__ v, const float* __restrict__ w,
                                                        const float* __restrict__ p, const float* __restrict__ ps,
                                                        const float* __restrict__ ru, const float* __restrict__ rv,
                                                        const float* __restrict__ rw, const float* __restrict__ tr,
                                                        float* __restrict__ uo, float* __restrict__ vo,
                                                        float* __restrict__ wo, float* __restrict__ po, float dts) {
#pragma clang fp contract(off)
  const TileId tb = xcd_tile();
  const int k = tb.x * (int)blockDim.x + (int)threadIdx.x, j = tb.y * (int)blockDim.y + (int)threadIdx.y, i = tb.z;
  if (k >= d.nz || j >= d.ny) return;
  const int I = i + 3, J = j + 3, K = k + 1;
  const long c = ic(d, I, J, K), sx = d.sxc(), sy = d.syc();
  const long cu = iu(d, I, J, K), cv = iv(d, I, J, K), cw = iw(d, I, J, K);
  const long ou = ((long)i * d.ny + j) * d.nz + k, ov = ((long)i * (d.ny + 1) + j) * d.nz + k;
  const long ow = ((long)i * d.ny + j) * (d.nz + 1) + k;
  // every operand is loaded unconditionally (all indices are inside the arrays) so that the
  // loads issue back to back; the surface and lid cases are selected afterwards
  const float rcm = rc[K - 1], rcc = rc[K], rcp = rc[K + 1];
  const float pim = pi0c[K - 1], pic = pi0c[K], pip = pi0c[K + 1];
  const float u0 = u[cu], u1 = u[cu + d.sxu()], v0 = v[cv], v1 = v[cv + sy], w0 = w[cw], w1 = w[cw + 1];
  const float ru0 = ru[ou], ru1 = ru[ou + (long)d.ny * d.nz], rv0 = rv[ov], rv1 = rv[ov + d.nz];
  const float rw0 = rw[ow], rw1 = rw[ow + 1];
  const float pc = p[c], pxm = p[c - sx], pxp = p[c + sx], pym = p[c - sy], pyp = p[c + sy], pzm = p[c - 1],
              pzp = p[c + 1];
  const float tc = tr[c], txm = tr[c - sx], txp = tr[c + sx], tym = tr[c - sy], typ = tr[c + sy], tzm = tr[c - 1],
              tzp = tr[c + 1];
  const float sc = ps[c], sxm = ps[c - sx], sxp = ps[c + sx], sym = ps[c - sy], syp = ps[c + sy], szm = ps[c - 1],
              szp = ps[c + 1];
  const bool floor_ = k == 0, lid = k == d.nz - 1;
  const float h = (float)(-kCp * 0.5);
  const float un0 = fmaf(fmaf(h * (tc + txm), (pc - pxm) * d.idx, ru0), dts, u0);
  const float un1 = fmaf(fmaf(h * (txp + tc), (pxp - pc) * d.idx, ru1), dts, u1);
  const float vn0 = fmaf(fmaf(h * (tc + tym), (pc - pym) * d.idy, rv0), dts, v0);
  const float vn1 = fmaf(fmaf(h * (typ + tc), (pyp - pc) * d.idy, rv1), dts, v1);
  const float wn0 = floor_ ? 0.0f : fmaf(h * (tc + tzm) * ((pc - pzm) * d.idz) + rw0, dts, w0);
  const float wn1 = lid ? 0.0f : fmaf(h * (tzp + tc) * ((pzp - pc) * d.idz) + rw1, dts, w1);
  const float div = fmaf(wn1 - wn0, d.idz, fmaf(vn1 - vn0, d.idy, (un1 - un0) * d.idx));
  const float du = un1 * ((sxp - sc) * d.idx) + un0 * ((sc - sxm) * d.idx);
  const float dv = vn1 * ((syp - sc) * d.idy) + vn0 * ((sc - sym) * d.idy);
  const float wd0 = floor_ ? 0.0f : wn0 * fmaf(sc - szm, d.idz, (pic - pim) * d.idz);
  const float wd1 = lid ? 0.0f : wn1 * fmaf(szp - sc, d.idz, (pip - pic) * d.idz);
  const float z = fmaf(0.5f * wd0, 0.5f * (rcm + rcc), 0.5f * wd1 * (0.5f * (rcc + rcp))) / rcc;
  const float advp = -(fmaf(0.5f, du, 0.5f * dv) + z);
  const float dpdt = fmaf((float)(-kRd / kCv), (pic + sc) * div, advp);
  store_c_fast(d, po, i, j, k, fmaf(1.1f * dpdt, dts, pc));
  store_u_fast(d, uo, i, j, k, un0);
  if (i == d.nx - 1) store_u(d, uo, d.nx, j, k, un1);
  store_v_fast(d, vo, i, j, k, vn0);
  if (j == d.ny - 1) store_v(d, vo, i, d.ny, k, vn1);
  store_w_fast(d, wo, i, j, k, wn0);
  if (lid) store_w(d, wo, i, j, d.nz, 0.0f);
}

struct AcousticArgs {
  const float *rc, *pi0, *u, *v, *w, *p, *ps, *ru, *rv, *rw, *tr;
  float *uo, *vo, *wo, *po;
  float dts;
};

template <int V, bool MZ>
inline void launch_acoustic_v(const Dims& d, const AcousticArgs& a, hipStream_t st) {
  const int chunks = (d.nz + 64 * V - 1) / (64 * V);
  // Cells per wave along x: the prologue of a longer march is shared, as long as the launch
  // has some 16 waves per SIMD, two rounds or more.  us per substep at ax = 1, 2, 3, 4, one
  // level per lane: 128x128x64 15.6, 16.8, -, 19.4; 200x200x64 27.1, 27.1, 26.6, 27.1; 300x200x64
  // 37.6, 35.8, 39.0, 41.2; 1000x60x64 38.7, 36.7, 40.0, 44.6; 512x300x64 139, 133, 131, 133; two:
  // 128x96x96 20.2, 20.9, 19.9, -; 150x130x80 27.0, 25.3, 27.3, -; 192x160x96 43.6, 38.8, -, 40.9;
  // 200x200x80 49.6, 43.2, 40.3, 43.5; 240x240x120 111, 99, -, 97; 256x256x128 129, 115, -, 113.
  const long waves = (long)d.nx * d.ny * chunks;
  const int fill = V == 1 ? (int)std::min(2L, std::max(1L, (waves + 8192) / 16384))
                          : (int)std::min(4L, std::max(1L, (waves + 14000) / 16384));
  const int ax = std::max(fill, (d.nx + 65535) / 65536);   // the grid's second dimension holds 2^16
  LEX_LAUNCH(KID_ACOUSTIC, (k_acoustic<V, MZ>), dim3((d.ny + 3) / 4, (d.nx + ax - 1) / ax, chunks), dim3(64, 4, 1), 0, st,
             d, a.rc, a.pi0, a.u, a.v, a.w, a.p, a.ps, a.ru, a.rv, a.rw, a.tr, a.uo, a.vo, a.wo, a.po, a.dts, ax);
}
inline void launch_acoustic_cells(const Dims& d, const AcousticArgs& a, hipStream_t st) {
  LEX_LAUNCH(KID_ACOUSTIC, k_acoustic_cells, dim3((d.nz + 63) / 64, (d.ny + 3) / 4, d.nx), dim3(64, 4, 1), 0, st, d, a.rc,
             a.pi0, a.u, a.v, a.w, a.p, a.ps, a.ru, a.rv, a.rw, a.tr, a.uo, a.vo, a.wo, a.po, a.dts);
}

// One substep.  Two levels per lane where a column has more than one wave of them; us with
// one and with two: 96x96x48 11.2 and 17.9, 128x128x64 15.6 and 26.6 (half the lanes idle);
// 181x147x70 33.1 and 31.6, 240x240x120 120 and 97, 256x256x128 139 and 110.  A thread per
// cell took 13.9, 17.9, 35.8, 113 and 131; a copy of the thirteen fields of 240x240x120 at
// 5 TB/s takes 72.
// Above 128 levels a row of lanes leaves its last wave part empty, which costs as much as a
// full one, and rows take longer chains of loads than cells: us with rows and cells,
// 128x128x129 39 and 31, 192x160x160 91 and 66, 256x256x160 207 and 161, 192x160x300 160 and
// 141, 256x256x384 422 and 365.  With both waves of two levels nearly full the rows win while
// the chip is not, and again where memory bounds both: 64x64x224 16.4 and 17.5, 128x96x224 36
// and 33, 128x128x256 48 and 44, 192x160x224 108 and 116, 256x256x256 230 and 254.
inline void launch_acoustic(const Dims& d, const AcousticArgs& a, hipStream_t st) {
  const long cells = (long)d.nx * d.ny * d.nz;
  if (d.nz <= 64)
    launch_acoustic_v<1, false>(d, a, st);
  else if (d.nz <= 128)
    launch_acoustic_v<2, false>(d, a, st);
  else if ((d.nz > 192 && d.nz <= 256 && (cells < 1500000 || cells >= 5000000)) || d.nx >= 65536)
    launch_acoustic_v<2, true>(d, a, st);   // also where a launch has no place for the cells' x
  else
    launch_acoustic_cells(d, a, st);
}

// k_acoustic2: two consecutive substeps in one launch, bit for bit what two k_acoustic
// launches give.  A workgroup of R rows (the outer two are halo rows) marches along x; a wave
// owns the 64 V levels of one row, as in k_acoustic.  In step s it
//   finishes the y and z faces of the second substep at cell s - 1 (the neighbour rows' new
//   pi' of that position is in LDS, everything else in its registers),
//   advances cell s by the first substep and puts the new pi' into LDS,
//   asks for the operands of cell s + 1,
//   finishes the second substep at cell s - 1, whose x face needed the new pi' of cell s,
// with one barrier per step and two slabs of pi'.  Halo rows and the positions x0 - 1 and x1
// are taken at their periodic images, so the second substep reads what it would read from
// the ghosts.
//
// Bound by memory (the thirteen fields once for two substeps: 72 us at 240x240x120 and
// 5 TB/s) and by the barrier that holds a CU's waves together.  us per pair against two
// k_acoustic launches: 40x40x40 9.8 and 19, 96x96x48 19 and 23, 128x128x64 23 and 31,
// 181x147x70 53 and 61, 192x160x96 64 and 73, 240x240x120 141 and 195, 256x256x128 150 and 225,
// 256x256x200 309 and 441, 512x512x64 300 and 437 (acoustic_pairs has the shapes where two
// launches win).  With a cell per thread, faces evaluated twice and the levels exchanged
// through the LDS pipe it took 194 and 194 at 240x240x120 and 256x256x128.  Eight rows of two
// levels per lane: 166 and 188, sixteen (spills) 172 and 194.
template <int V>
struct Pair2Operands {
  float p1[V], t1[V], s1[V];               // row j of plane x + 1
  float py[2][V], ty[2][V], sy[2][V];      // rows j - 1, j + 1 of plane x
  float uf[V], gu[V], vf[2][V], gv[2][V], wf[V], gw[V];
  float pe, te, se, we, ge;                // beyond the wave's levels (edge lanes)
};

template <int V, bool MZ, int MAXT>
__global__ void __launch_bounds__(MAXT) k_acoustic2(Dims d, AcousticArgs a, int ax) {
#pragma clang fp contract(off)
  extern __shared__ float ring[];  // [2 slabs][R rows][64 V levels of every wave of a row]
  const int lane = threadIdx.x & 63;
  const int chunk = MZ ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
  const int r = __builtin_amdgcn_readfirstlane((int)threadIdx.y), R = blockDim.y, LR = blockDim.x * V;
  const TileId tb = xcd_tile();
  const int nx = d.nx, ny = d.ny, nz = d.nz;
  const int j = tb.x * (R - 2) - 1 + r;          // -1 .. ny (rows past ny repeat it, never stored)
  const int jw = wrap_cell(min(j, ny), ny);
  const bool rowb = r >= 1 && r <= R - 2 && j < ny;
  const int x0 = tb.y * ax, x1 = min(x0 + ax, nx);
  const int kl = (chunk * 64 + lane) * V;
  const int kc = min(kl, nz - 1);
  LevelSlots ls;
  ls.n = min(max(nz - kl, 0), V);
  ls.first = kl == 0;
  ls.last = ls.n > 0 && kl + ls.n == nz;
  const uint32_t eK = (uint32_t)(kc + 1);
  const uint32_t ek = (uint32_t)min(kc, nz - V);
  const bool past = (V == 2) && kc == nz - 1;
  const float h = (float)(-kCp * 0.5);
  const float dts = a.dts;
  float rr[V], ir[V], r8[V], pic[V], dpi[V];
#pragma unroll
  for (int q = 0; q < V; ++q) {
    const int K = min(kc + q + 1, nz + 1);
    rr[q] = a.rc[K];
    ir[q] = 1.0f / rr[q];
    r8[q] = 0.5f * (a.rc[K - 1] + rr[q]);
    pic[q] = a.pi0[K];
    dpi[q] = (pic[q] - a.pi0[K - 1]) * d.idz;
  }
  float r8e = 0.f, dpie = 0.f;
  if (MZ) {
    const int K = min(kc + V + 1, nz + 1);
    r8e = 0.5f * (a.rc[K - 1] + a.rc[K]);
    dpie = (a.pi0[K] - a.pi0[K - 1]) * d.idz;
  }
  const bool edge = MZ && (lane == 0 || lane == 63);
  const uint32_t eE = (uint32_t)(lane == 0 ? kc : min(kc + V + 1, nz + 1));
  const uint32_t eW = (uint32_t)min(kc + V, nz);

  const int syc = nz + 2, syw = nz + 3;
  const int sxc = (ny + 6) * syc, sxv = (ny + 7) * syc, sxw = (ny + 6) * syw;
  const int sxiu = ny * nz, sxiv = (ny + 1) * nz, sxiw = ny * (nz + 1);
  const uint32_t oc = (uint32_t)((jw + 3) * syc) + eK, ow = (uint32_t)((jw + 3) * syw) + eK;
  const uint32_t ocm = oc - (uint32_t)syc, ocp = oc + (uint32_t)syc;
  const uint32_t oi = (uint32_t)(jw * nz) + ek, oin = oi + (uint32_t)nz;
  const uint32_t og = (uint32_t)(jw * (nz + 1) + kc);
  float* const own = ring + r * LR + (chunk * 64 + lane) * V;
  const int slab = R * LR;

  // input planes of the cell in hand
  const float *pX, *tX, *sX, *uX, *vX, *wX, *guX, *gvX, *gwX;
  auto place = [&](int xw) {
    pX = a.p + (long)(xw + 3) * sxc;
    tX = a.tr + (long)(xw + 3) * sxc;
    sX = a.ps + (long)(xw + 3) * sxc;
    uX = a.u + (long)(xw + 3) * sxc;
    vX = a.v + (long)(xw + 3) * sxv;
    wX = a.w + (long)(xw + 3) * sxw;
    guX = a.ru + (long)xw * sxiu;
    gvX = a.rv + (long)xw * sxiv;
    gwX = a.rw + (long)xw * sxiw;
  };
  auto fetch = [&](Pair2Operands<V>& o) {
    ld_levels<V>(pX, ocm, o.py[0]);
    ld_levels<V>(tX, ocm, o.ty[0]);
    ld_levels<V>(sX, ocm, o.sy[0]);
    ld_levels<V>(pX, ocp, o.py[1]);
    ld_levels<V>(tX, ocp, o.ty[1]);
    ld_levels<V>(sX, ocp, o.sy[1]);
    ld_levels<V>(vX, oc, o.vf[0]);
    ld_levels<V>(vX, ocp, o.vf[1]);
    ld_levels_in<V>(gvX, oi, past, o.gv[0]);
    ld_levels_in<V>(gvX, oin, past, o.gv[1]);
    ld_levels<V>(wX, ow, o.wf);
    ld_levels<V>(gwX, og, o.gw);
    if (edge) {
      o.pe = ld32(pX, oc - eK + eE);
      o.te = ld32(tX, oc - eK + eE);
      o.se = ld32(sX, oc - eK + eE);
      o.we = ld32(wX, ow - eK + eW + 1u);
      o.ge = ld32(gwX, og - (uint32_t)kc + eW);
    }
    ld_levels<V>(pX + sxc, oc, o.p1);
    ld_levels<V>(tX + sxc, oc, o.t1);
    ld_levels<V>(sX + sxc, oc, o.s1);
    ld_levels<V>(uX + sxc, oc, o.uf);
    ld_levels_in<V>(guX + sxiu, oi, past, o.gu);
  };

  // first substep, row j of the cell in hand, and its lower x face: new u, u dpi*/dx
  float P0[V], T0[V], S0[V], ul[V], dl[V];
  // second substep: operands of cell s - 1 and of the x face in hand, new pi' there, new u
  // and u dpi*/dx of its lower x face
  float hty[2][V], dsy[2][V], gvb[2][V], vb[2][V], htz[V], dzb[V], gwb[V], wb[V], pab[V], pb[V];
  float ub[V], gub[V], htx[V], dsx[V], ulb[V], dlb[V];
  float hte = 0.f, dze = 0.f, geb = 0.f, web = 0.f;
#pragma unroll
  for (int q = 0; q < V; ++q) {
    pb[q] = ulb[q] = dlb[q] = pab[q] = 0.f;
    ub[q] = gub[q] = htx[q] = dsx[q] = 0.f;
  }
  Pair2Operands<V> o;
  place(wrap_cell(x0 - 1, nx));
  fetch(o);
#pragma unroll 1
  for (int s = x0 - 1; s <= x1; ++s) {
    const bool second = s > x0 && rowb;
    // y and z faces of the second substep at cell s - 1
    float dvn[V], hdv[V], dwn[V], zz[V];
    if (second) {
      const int x = s - 1;
      const float* L = own + ((s - x0) & 1) * slab;
      float vn[2][V], pm[V], pp[V];
#pragma unroll
      for (int q = 0; q < V; ++q) {
        pm[q] = L[q - LR];
        pp[q] = L[q + LR];
      }
#pragma unroll
      for (int q = 0; q < V; ++q) {
        vn[0][q] = fmaf(fmaf(hty[0][q], (pb[q] - pm[q]) * d.idy, gvb[0][q]), dts, vb[0][q]);
        vn[1][q] = fmaf(fmaf(hty[1][q], (pp[q] - pb[q]) * d.idy, gvb[1][q]), dts, vb[1][q]);
        dvn[q] = vn[1][q] - vn[0][q];
        hdv[q] = 0.5f * (vn[1][q] * dsy[1][q] + vn[0][q] * dsy[0][q]);
      }
      float wn[V], a0[V], b0[V];
      float pl0 = lane_below(pb[V - 1]);
      float pu = 0.f;
      if (MZ && lane == 0 && kl > 0) pl0 = L[-1];
      if (MZ && lane == 63) pu = kl + V < LR ? L[V] : 0.f;
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const float pl = q ? pb[0] : pl0;
        const float wv = fmaf(htz[q] * ((pb[q] - pl) * d.idz) + gwb[q], dts, wb[q]);
        const bool floor_ = q == 0 && kl == 0;
        wn[q] = floor_ ? 0.0f : wv;
        a0[q] = 0.5f * (floor_ ? 0.0f : wv * dzb[q]);
        b0[q] = a0[q] * r8[q];
      }
      float wt = lane_above(wn[0]), bt = lane_above(b0[0]);
      if (MZ && lane == 63) {
        wt = fmaf(hte * ((pu - pb[V - 1]) * d.idz) + geb, dts, web);
        bt = (0.5f * (wt * dze)) * r8e;
      }
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const bool lid = kl + q >= nz - 1;
        const float w1 = lid ? 0.0f : (q < V - 1 ? wn[V - 1] : wt);
        const float b1 = lid ? 0.0f : (q < V - 1 ? b0[V - 1] : bt);
        dwn[q] = w1 - wn[q];
        zz[q] = quotient(fmaf(a0[q], r8[q], b1), rr[q], ir[q]);
      }
      if (x >= 4 && x < nx - 3 && j >= 4 && j < ny - 3) {   // no periodic images
        float* voX = a.vo + (long)(x + 3) * sxv;
        float* woX = a.wo + (long)(x + 3) * sxw;
        st_levels<V>(voX, oc, ls, vn[0]);
        st_levels<V>(woX, ow, ls, wn);
        if (ls.first || ls.last) {
          st_ghosts<V>(voX, oc, ls, vn[0]);
          st_ghosts_w<V>(woX, ow, ls, wn);
        }
      } else {
        st_images<V, false>(a.vo, sxv, syc, x, nx, false, j, ny, true, eK, ls, vn[0]);
        if (j == ny - 1) st_images<V, false>(a.vo, sxv, syc, x, nx, false, ny, ny, true, eK, ls, vn[1]);
        st_images<V, true>(a.wo, sxw, syw, x, nx, false, j, ny, false, eK, ls, wn);
      }
    }
    // a march starts, or continues at the other end of the period
    if (s == x0 - 1 || s == 0 || s == nx) {
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
        const float ht = h * (T0[q] + tm[q]), ds = (S0[q] - sm[q]) * d.idx;
        ul[q] = fmaf(fmaf(ht, (P0[q] - pm[q]) * d.idx, g0[q]), dts, u0[q]);
        dl[q] = ul[q] * ds;
        if (s <= x0) {   // the face where the second substep's march starts
          ub[q] = ul[q];
          gub[q] = g0[q];
          htx[q] = ht;
          dsx[q] = ds;
        }
      }
    }
    // first substep at cell s
    float pn[V], pa1[V], ub1[V], gu1[V], htx1[V], dsx1[V];
    {
      float dv[2][V], div0[V];
#pragma unroll
      for (int q = 0; q < V; ++q) {
        hty[0][q] = h * (T0[q] + o.ty[0][q]);
        hty[1][q] = h * (o.ty[1][q] + T0[q]);
        dsy[0][q] = (S0[q] - o.sy[0][q]) * d.idy;
        dsy[1][q] = (o.sy[1][q] - S0[q]) * d.idy;
        vb[0][q] = fmaf(fmaf(hty[0][q], (P0[q] - o.py[0][q]) * d.idy, o.gv[0][q]), dts, o.vf[0][q]);
        vb[1][q] = fmaf(fmaf(hty[1][q], (o.py[1][q] - P0[q]) * d.idy, o.gv[1][q]), dts, o.vf[1][q]);
        gvb[0][q] = o.gv[0][q];
        gvb[1][q] = o.gv[1][q];
        dv[0][q] = vb[0][q] * dsy[0][q];
        dv[1][q] = vb[1][q] * dsy[1][q];
      }
      float a0[V], b0[V];
      float pl0 = lane_below(P0[V - 1]), tl0 = lane_below(T0[V - 1]), sl0 = lane_below(S0[V - 1]);
      if (MZ && lane == 0) {
        pl0 = o.pe;
        tl0 = o.te;
        sl0 = o.se;
      }
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const float pl = q ? P0[0] : pl0, tl = q ? T0[0] : tl0, sl = q ? S0[0] : sl0;
        htz[q] = h * (T0[q] + tl);
        dzb[q] = fmaf(S0[q] - sl, d.idz, dpi[q]);
        gwb[q] = o.gw[q];
        const float wv = fmaf(htz[q] * ((P0[q] - pl) * d.idz) + o.gw[q], dts, o.wf[q]);
        const bool floor_ = q == 0 && kl == 0;
        wb[q] = floor_ ? 0.0f : wv;
        a0[q] = 0.5f * (floor_ ? 0.0f : wv * dzb[q]);
        b0[q] = a0[q] * r8[q];
      }
      float wt = lane_above(wb[0]), bt = lane_above(b0[0]);
      if (MZ && lane == 63) {
        hte = h * (o.te + T0[V - 1]);
        dze = fmaf(o.se - S0[V - 1], d.idz, dpie);
        geb = o.ge;
        web = fmaf(hte * ((o.pe - P0[V - 1]) * d.idz) + o.ge, dts, o.we);
        wt = web;
        bt = (0.5f * (wt * dze)) * r8e;
      }
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const bool lid = kl + q >= nz - 1;
        const float w1 = lid ? 0.0f : (q < V - 1 ? wb[V - 1] : wt);
        const float b1 = lid ? 0.0f : (q < V - 1 ? b0[V - 1] : bt);
        htx1[q] = h * (o.t1[q] + T0[q]);
        dsx1[q] = (o.s1[q] - S0[q]) * d.idx;
        gu1[q] = o.gu[q];
        ub1[q] = fmaf(fmaf(htx1[q], (o.p1[q] - P0[q]) * d.idx, o.gu[q]), dts, o.uf[q]);
        const float du = ub1[q] * dsx1[q];
        div0[q] = fmaf(w1 - wb[q], d.idz, fmaf(vb[1][q] - vb[0][q], d.idy, (ub1[q] - ul[q]) * d.idx));
        const float z = quotient(fmaf(a0[q], r8[q], b1), rr[q], ir[q]);
        const float advp = -(fmaf(0.5f, du + dl[q], 0.5f * (dv[1][q] + dv[0][q])) + z);
        pa1[q] = pic[q] + S0[q];
        const float dpdt = fmaf((float)(-kRd / kCv), pa1[q] * div0[q], advp);
        pn[q] = fmaf(1.1f * dpdt, dts, P0[q]);
        ul[q] = ub1[q];
        dl[q] = du;
        P0[q] = o.p1[q];
        T0[q] = o.t1[q];
        S0[q] = o.s1[q];
      }
    }
    {
      float* L = own + ((s + 1 - x0) & 1) * slab;
#pragma unroll
      for (int q = 0; q < V; ++q) L[q] = pn[q];
    }
    if (s < x1) {
      if (s + 1 == 0 || s + 1 == nx) {
        place(0);
      } else {
        pX += sxc;
        tX += sxc;
        sX += sxc;
        uX += sxc;
        vX += sxv;
        wX += sxw;
        guX += sxiu;
        gvX += sxiv;
        gwX += sxiw;
      }
      fetch(o);
    }
    // second substep: x face s, then pi' of cell s - 1
    if (s >= x0) {
      float pn2[V], us[V], un[V];
#pragma unroll
      for (int q = 0; q < V; ++q) {
        un[q] = fmaf(fmaf(htx[q], (pn[q] - pb[q]) * d.idx, gub[q]), dts, ub[q]);
        const float du = un[q] * dsx[q];
        const float div = fmaf(dwn[q], d.idz, fmaf(dvn[q], d.idy, (un[q] - ulb[q]) * d.idx));
        const float advp = -(fmaf(0.5f, du + dlb[q], hdv[q]) + zz[q]);
        const float dpdt = fmaf((float)(-kRd / kCv), pab[q] * div, advp);
        pn2[q] = fmaf(1.1f * dpdt, dts, pb[q]);
        us[q] = ulb[q];
        ulb[q] = un[q];
        dlb[q] = du;
      }
      if (second) {
        const int x = s - 1;
        if (x >= 4 && x < nx - 3 && j >= 4 && j < ny - 3) {
          float* poX = a.po + (long)(x + 3) * sxc;
          float* uoX = a.uo + (long)(x + 3) * sxc;
          st_levels<V>(poX, oc, ls, pn2);
          st_levels<V>(uoX, oc, ls, us);
          if (ls.first || ls.last) {
            st_ghosts<V>(poX, oc, ls, pn2);
            st_ghosts<V>(uoX, oc, ls, us);
          }
        } else {
          st_images<V, false>(a.po, sxc, syc, x, nx, false, j, ny, false, eK, ls, pn2);
          st_images<V, false>(a.uo, sxc, syc, x, nx, true, j, ny, false, eK, ls, us);
          if (x == nx - 1) st_images<V, false>(a.uo, sxc, syc, nx, nx, true, j, ny, false, eK, ls, un);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < V; ++q) {
      pb[q] = pn[q];
      pab[q] = pa1[q];
      ub[q] = ub1[q];
      gub[q] = gu1[q];
      htx[q] = htx1[q];
      dsx[q] = dsx1[q];
    }
    __syncthreads();
  }
}

// Columns of at most three waves; a taller one would leave a workgroup too few rows.
inline bool acoustic2_ok(const Dims& d) { return d.nz <= 256; }

// Whether a step takes its substeps in pairs.  A pair costs by rows, whatever their levels; two
// substeps in the caches cost little more than their launches.  us of two substeps and of a pair:
// shallow and wide 256x256x20 63 and 78, 512x512x16 184 and 280, 512x300x20 109 and 156,
// 256x256x48 73 and 79, against 128x128x20 26 and 22, 200x200x20 46 and 47, 1024x512x20 445 and
// 449, 300x200x64 72 and 66, 512x300x48 215 and 178; in part empty waves 96x96x160 43 and 53,
// 128x128x192 68 and 78, 192x160x144 119 and 145, against 200x200x160 204 and 189.
inline bool acoustic_pairs(const Dims& d) {
  const long columns = (long)d.nx * d.ny, cells = columns * d.nz;
  if (!acoustic2_ok(d)) return false;
  if (d.nz <= 64) return columns < 40000 || (d.nz > 24 && cells >= 3600000);
  if (d.nz > 128 && d.nz <= 192) return cells >= 5200000;
  return true;
}

// ROWS: two levels per lane need 142 to 160 VGPRs, three waves per SIMD, so one workgroup of
// twelve waves fills a CU; with one level (87 VGPRs) two workgroups of eight.  The march is the
// one of 1 to 8 full rounds of workgroups that takes the fewest steps, a workgroup of ax cells
// taking ax + 3.  One round is best while its strips divide the CUs; us with one round and with
// this plan, 500x520x130 (131 strips) 2130 and 1082, 1024x1024x32 (171 of 512) 1587 and 869,
// 300x1600x40 939 and 456, 512x512x100 620 and 540, 240x240x120 (24) 141 and 141.
// 129 to 192 levels on wide grids: three waves of one level per row instead of two of two levels,
// the second of which would be part empty; us with two and with three, 150x130x160 97 and 122,
// 200x200x192 194 and 221, 300x200x129 270 and 247, 256x256x160 296 and 260, 512x300x192 691 and 625.
template <int V, bool MZ, int ROWS>
inline void launch_acoustic2_v(const Dims& d, const AcousticArgs& a, hipStream_t st) {
  constexpr int kLanes = MZ ? (V == 1 ? 192 : 128) : 64;
  const int strips = (d.ny + ROWS - 3) / (ROWS - 2);
  const long slots = (long)device_cus() * (V == 1 && !MZ ? 2 : 1);
  int ax = d.nx;
  long least = 0;
  for (int rounds = 1; rounds <= 8; ++rounds) {
    const int parts = (int)std::max(1L, std::min((long)d.nx, rounds * slots / strips)), len = (d.nx + parts - 1) / parts;
    const long n = (long)strips * ((d.nx + len - 1) / len), cost = (n + slots - 1) / slots * (len + 3);
    if (rounds == 1 || cost < least) {
      ax = len;
      least = cost;
    }
  }
  if (V == 1 && MZ) ax = std::min(ax, 24);   // of five rows two are halo: neighbours close enough to share them in L2
  const dim3 g(strips, (d.nx + ax - 1) / ax), b(kLanes, ROWS);
  const size_t lds = (size_t)2 * ROWS * kLanes * V * sizeof(float);
  LEX_LAUNCH(KID_ACOUSTIC2, (k_acoustic2<V, MZ, kLanes * ROWS>), g, b, lds, st, d, a, ax);
}
inline void launch_acoustic2(const Dims& d, const AcousticArgs& a, hipStream_t st) {
  if (d.nz <= 64)
    launch_acoustic2_v<1, false, 8>(d, a, st);
  else if (d.nz <= 128)
    launch_acoustic2_v<2, false, 12>(d, a, st);
  else if (d.nz <= 192 && (long)d.nx * d.ny >= 50000)
    launch_acoustic2_v<1, true, 5>(d, a, st);
  else
    launch_acoustic2_v<2, true, 6>(d, a, st);
}

}  // namespace lex
