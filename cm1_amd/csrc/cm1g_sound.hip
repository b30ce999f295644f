// Split-explicit acoustic substeps with the vertically implicit w-pi solve
// (psolver=3, no terrain, Cartesian): src/sound.F:10-859, called from
// src/solve2.F:1122-1136 with thv=t11, ppterm=t22, piadv=sadv, mm=dum5,
// ppd=dum7, fpk=dum8, qk=t12, pk1=t13, pk2=t23.
// Also getdiv/getdivx (src/misclibs.F:108-370) and calccflquick
// (src/misclibs.F:2726-2814).
#include "cm1g_internal.h"


static void sound_nloop(int nrk, int nsound, float dt, int *nloop_out, float *dts_out) {
  int nloop;
  float dts;
  if (nrk == 1) {
    nloop = (int)lroundf((float)nsound / 3.0f);
    dts = dt / ((float)nloop * 3.0f);
    if (dts > (dt / (float)nsound)) {
      nloop = nloop + 1;
      dts = dt / ((float)nloop * 3.0f);
    }
  } else if (nrk == 2) {
    nloop = (int)(0.5f * (float)nsound);
    dts = dt / (float)nsound;
  } else {
    nloop = nsound;
    dts = dt / (float)nsound;
  }
  *nloop_out = nloop;
  *dts_out = dts;
}

// Arguments of one fused acoustic substep.
struct SubArgs {
  float dts, alph, beta, asq, kdiv, tavg;
  float tem1, tem2, temx, temy;   // cp*rdx/2, cp*rdy/2, dts*rdx/2, dts*rdy/2
  int last, opw, ope, ops, opn;
  const float *uX, *vX;           // u, v at the start of the substep
  float *uY, *vY, *wY;            // u, v after the substep (wY: explicit substeps)
  const float *ppdX;              // pi' + divergence damping from the previous substep
  float *ppdY;                    // ... written by this substep
  const float *uten, *vten, *wten, *thv, *piadv, *ppterm, *ppten, *dtu0, *dtv0;
  const float *radbcw, *radbce, *radbcs, *radbcn;
  float *w3d, *pp3d, *fpk, *dum1, *dum2, *rru, *rrv, *rrw;
  // first substep: w and pi' are read from wR/ppR (wa/ppi after the first
  // RK stage) and the averages start from 0 (u, v) and beta*wa (w), which
  // is what the reference's copies before the substep loop set
  // (src/sound.F:191-250)
  const float *wR, *ppR, *wa;
  // per level k: tem, r1, r2, temm, c1(k), c1(k+1), c2(k), c2(k+1) of the
  // solver coefficients (src/sound.F:117-180), 8 floats at coef + 8k
  const float *coef;
  int first;
  int nring;                      // trailing workgroups that do the averaging ring
  // The averages take in u, v, w of two substeps at a time: substep n - 1's
  // values are substep n's input, so every other substep leaves rru, rrv,
  // rrw alone (no read, no write) and the next one adds both values, in the
  // order of the substeps.  fold: this substep updates the averages; pair:
  // with the previous substep's values too; init: they start here.
  int fold, pair, init;
  const float *wring, *wringp;    // w on the averaging ring, this substep's and the previous one's
  int expl;                       // explicit substeps: w enters its average like u and v
  float *ppx;                     // last substep of the last stage: the damping term
};

// new u at (i,j,k): radiative open-boundary update (ssopenbcw/e,
// src/bc.F:2392-2530) then the pressure-gradient step (src/sound.F:307-325)
__device__ __forceinline__ float sub_u(const KP &P, const SubArgs &a, int i, int j, int k) {
  const int c = IXD(P, i, j, k);
  float u = a.uX[c];
  if (j >= 1 && j <= P.nj) {
    if (a.opw && i == 1)
      u = u + a.dts * (-a.radbcw[(j + 2) + k * P.py] * (a.uX[IXD(P, 2, j, k)] - u) * P.rdx +
                       a.uten[c]);
    if (a.ope && i == P.ni + 1)
      u = u + a.dts * (-a.radbce[(j + 2) + k * P.py] * (u - a.uX[IXD(P, P.ni, j, k)]) * P.rdx +
                       a.uten[c]);
  }
  const float dtu = a.dts * a.dtu0[IX2D(P, i, j)];
  return u + dtu * (a.uten[c] - a.tem1 * (a.ppdX[c] - a.ppdX[c - 1]) * (a.thv[c] + a.thv[c - 1]));
}

// new v at (i,j,k) (ssopenbcs/n, src/bc.F:2538-2684; src/sound.F:327-345)
__device__ __forceinline__ float sub_v(const KP &P, const SubArgs &a, int i, int j, int k) {
  const int c = IXD(P, i, j, k);
  float v = a.vX[c];
  if (i >= 1 && i <= P.ni) {
    if (a.ops && j == 1)
      v = v + a.dts * (-a.radbcs[(i + 2) + k * P.px] * (a.vX[IXD(P, i, 2, k)] - v) * P.rdy +
                       a.vten[c]);
    if (a.opn && j == P.nj + 1)
      v = v + a.dts * (-a.radbcn[(i + 2) + k * P.px] * (v - a.vX[IXD(P, i, P.nj, k)]) * P.rdy +
                       a.vten[c]);
  }
  const float dtv = a.dts * a.dtv0[IX2D(P, i, j)];
  const int cs = c - P.px;
  return v + dtv * (a.vten[c] - a.tem2 * (a.ppdX[c] - a.ppdX[cs]) * (a.thv[c] + a.thv[cs]));
}

// the running average r (rru, rrv) with the previous substep's value x0 and
// this one's x (src/sound.F:806-835)
__device__ __forceinline__ float avg_uv(const SubArgs &a, float r, float x0, float x) {
  if (a.pair) r = r + x0;
  return a.last ? (r + x) * a.tavg : r + x;
}
// store a new u (v) and fold it into the substep average
__device__ __forceinline__ void put_u(const SubArgs &a, int c, float u) {
  if (a.fold) a.rru[c] = avg_uv(a, a.init ? 0.0f : a.rru[c], a.uX[c], u);
  a.uY[c] = u;
}
__device__ __forceinline__ void put_v(const SubArgs &a, int c, float v) {
  if (a.fold) a.rrv[c] = avg_uv(a, a.init ? 0.0f : a.rrv[c], a.vX[c], v);
  a.vY[c] = v;
}
// w on the ring, where the step does not change it
__device__ __forceinline__ void put_w_ring(const SubArgs &a, int c) {
  if (!a.fold) return;
  const float w = a.wring[c];
  if (a.expl) {
    a.rrw[c] = avg_uv(a, a.init ? 0.0f : a.rrw[c], w, w);
    return;
  }
  float r = a.init ? a.wa[c] * a.beta : a.rrw[c];
  if (a.pair) r = r + a.wringp[c];
  a.rrw[c] = a.last ? (r + w * a.alph) * a.tavg : r + w;
}

// The averaging ring of one substep: u and v on the faces i = ni+1 and
// j = nj+1 (unchanged by the step where the open-boundary masks are zero,
// advanced otherwise) and the w average there (w is not advanced at those
// points).  Point t walks the ring (i = 1..ni+1 at j = nj+1, then
// j = 1..nj at i = ni+1) at level k.  It reads uX/vX/ppdX and writes only
// ring points, which the column tiles neither read nor write, so the ring
// runs alongside them.
__device__ __forceinline__ void sound_ring_point(const KP &P, const SubArgs &a, int t, int k) {
  const int ni = P.ni, nj = P.nj;
  int i, j;
  if (t <= ni) {
    i = 1 + t;
    j = nj + 1;
  } else if (t <= ni + nj) {
    i = ni + 1;
    j = t - ni;
  } else {
    return;
  }
  const int c = IXD(P, i, j, k);
  put_u(a, c, sub_u(P, a, i, j, k));
  put_v(a, c, sub_v(P, a, i, j, k));
  put_w_ring(a, c);
}

// Operands of one level of the upward sweep of sound_sub (raw loads).
struct SubLoads {
  float uXc, uXe, utc, ute, vXc, vXn, vtc, vtn;
  float pdc, pdw, pde, pds, pdn;
  float thc, thw, the, ths, thn;
  float rruc, rrvc;
  float paw, pae, pas, pan, pa_p;
  float ppterm, ppten, wten, pp_c, w_p;
  float rw, re, rs, rn;
};

__device__ __forceinline__ void sub_load(const KP &P, const SubArgs &a, int c, int k, int i, int j, bool bw,
                                         bool be, bool bs, bool bn, SubLoads &L) {
  const int px = P.px, pxy = P.pxy;
  L.uXc = a.uX[c]; L.uXe = a.uX[c + 1]; L.utc = a.uten[c]; L.ute = a.uten[c + 1];
  L.vXc = a.vX[c]; L.vXn = a.vX[c + px]; L.vtc = a.vten[c]; L.vtn = a.vten[c + px];
  L.pdc = a.ppdX[c]; L.pdw = a.ppdX[c - 1]; L.pde = a.ppdX[c + 1]; L.pds = a.ppdX[c - px];
  L.pdn = a.ppdX[c + px];
  L.thc = a.thv[c]; L.thw = a.thv[c - 1]; L.the = a.thv[c + 1]; L.ths = a.thv[c - px]; L.thn = a.thv[c + px];
  L.rruc = (!a.fold || a.init) ? 0.0f : a.rru[c];
  L.rrvc = (!a.fold || a.init) ? 0.0f : a.rrv[c];
  L.paw = a.piadv[c - 1]; L.pae = a.piadv[c + 1]; L.pas = a.piadv[c - px]; L.pan = a.piadv[c + px];
  L.pa_p = a.piadv[c + pxy];
  L.ppterm = a.ppterm[c]; L.ppten = a.ppten[c]; L.wten = a.wten[c]; L.pp_c = a.ppR[c];
  L.w_p = (k == P.nk) ? a.w3d[c + pxy] : a.wR[c + pxy];
  L.rw = bw ? a.radbcw[(j + 2) + k * P.py] : 0.0f;
  L.re = be ? a.radbce[(j + 2) + k * P.py] : 0.0f;
  L.rs = bs ? a.radbcs[(i + 2) + k * px] : 0.0f;
  L.rn = bn ? a.radbcn[(i + 2) + k * px] : 0.0f;
}

// One acoustic substep for a column (i,j): u/v forward step (also the
// faces i+1 / j+1 the divergence needs, recomputed from the same inputs),
// explicit pi forcing fpk (src/sound.F:484-505), Thomas forward sweep of the
// implicit w-pi system (src/sound.F:659-717), back substitution (:720-733),
// pi update with divergence damping (:739-765) and the w average.  The
// solver coefficients qk, pk1, pk2, mm (src/sound.F:117-180) are evaluated
// on the fly with the same expressions.  u and v are read from uX/vX and
// written to uY/vY (pi'+damping likewise ppdX/ppdY) so that neighbouring
// columns see the old values.
//
// Both sweeps load the next level's operands before the current level is
// evaluated and stored, so two levels' loads are in flight per column.
//
// The a.nring workgroups after the column tiles do the averaging ring (one
// thread per ring point and level); they fill the CUs the last tiles leave
// idle.
__device__ __forceinline__ void sound_sub(const KP &P, const SubArgs &a, const ColGrid &cg, int bx) {
  const int nmain = cg.per * NXCD;
  if (bx >= nmain) {
    const int npts = P.ni + P.nj + 1;
    const int t = (bx - nmain) * (int)blockDim.x + (int)threadIdx.x;
    if (t < npts * P.nk) sound_ring_point(P, a, t % npts, 1 + t / npts);
    return;
  }
  int i, j;
  if (!col_tile_b(cg, bx, i, j)) return;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  if (i > ni || j > nj) return;
  const float dts = a.dts, rdz = P.rdz, cp = P.K.cp, smeps = P.K.smeps;
  const float rdx = P.rdx, rdy = P.rdy;
  const int px = P.px, pxy = P.pxy;
  const bool bw = a.opw && i == 1, be = a.ope && i == ni, bs = a.ops && j == 1, bn = a.opn && j == nj;
  // k-invariant factors
  const float dtu_c = dts * a.dtu0[IX2D(P, i, j)], dtu_e = dts * a.dtu0[IX2D(P, i + 1, j)];
  const float dtv_c = dts * a.dtv0[IX2D(P, i, j)], dtv_n = dts * a.dtv0[IX2D(P, i, j + 1)];
  const float uf_c = P.uf[i + 2], uf_e = P.uf[i + 3], vf_c = P.vf[j + 2], vf_n = P.vf[j + 3];
  const float uh_c = P.uh[i + 2], vh_c = P.vh[j + 2];
  const float tem1 = a.tem1, tem2 = a.tem2, temx = a.temx, temy = a.temy;
  const float alph = a.alph, beta = a.beta, asq = a.asq;

  // level k-1 quantities carried up the column
  float A_m = 0.0f, B_m = 0.0f, fpk_m = 0.0f, pp_m = 0.0f;
  float d1p = 0.0f, d2p = 0.0f, w_top = 0.0f, w_bot = 0.0f, w_nk1 = 0.0f;
  int c = IXD(P, i, j, 1);
  float pa_m = a.piadv[c - pxy], pa_c = a.piadv[c];
  float th_m = a.thv[c - pxy];
  float w_c = a.wR[c];
  SubLoads nx;
  sub_load(P, a, c, 1, i, j, bw, be, bs, bn, nx);
  for (int k = 1; k <= nk; k++, c += pxy) {
    // ---- this level's operands; the next level's are loaded before this
    // level is evaluated and stored
    const SubLoads L = nx;
    if (k < nk) sub_load(P, a, c + pxy, k + 1, i, j, bw, be, bs, bn, nx);
    const float uXc = L.uXc, uXe = L.uXe, utc = L.utc, ute = L.ute;
    const float vXc = L.vXc, vXn = L.vXn, vtc = L.vtc, vtn = L.vtn;
    const float pdc = L.pdc, pdw = L.pdw, pde = L.pde, pds = L.pds, pdn = L.pdn;
    const float thc = L.thc, thw = L.thw, the = L.the, ths = L.ths, thn = L.thn;
    const float rruc = L.rruc, rrvc = L.rrvc;
    const float paw = L.paw, pae = L.pae, pas = L.pas, pan = L.pan;
    const float pa_p = L.pa_p;
    const float ppterm = L.ppterm, ppten = L.ppten, wten = L.wten, pp_c = L.pp_c;
    const float w_p = L.w_p;
    const float rw = L.rw, re = L.re, rs = L.rs, rn = L.rn;
    // ---- u, v (ssopenbc* then src/sound.F:307-345)
    float uo0 = uXc, uo1 = uXe, vo0 = vXc, vo1 = vXn;
    if (bw) uo0 = uo0 + dts * (-rw * (uXe - uo0) * rdx + utc);
    if (be) uo1 = uo1 + dts * (-re * (uo1 - uXc) * rdx + ute);
    if (bs) vo0 = vo0 + dts * (-rs * (vXn - vo0) * rdy + vtc);
    if (bn) vo1 = vo1 + dts * (-rn * (vo1 - vXc) * rdy + vtn);
    const float un0 = uo0 + dtu_c * (utc - tem1 * (pdc - pdw) * uf_c * (thc + thw));
    const float un1 = uo1 + dtu_e * (ute - tem1 * (pde - pdc) * uf_e * (the + thc));
    const float vn0 = vo0 + dtv_c * (vtc - tem2 * (pdc - pds) * vf_c * (thc + ths));
    const float vn1 = vo1 + dtv_n * (vtn - tem2 * (pdn - pdc) * vf_n * (thn + thc));
    // ---- coefficients (src/sound.F:117-180)
    const float *cf = a.coef + 8 * k;
    const float tem = cf[0], r1 = cf[1], r2 = cf[2], temm = cf[3];
    const float c1a = cf[4], c1b = cf[5], c2a = cf[6], c2b = cf[7];
    const float qk = tem * ppterm;
    const float pk2 = (k == nk) ? 0.0f : r2 * (-c2b * pa_p + (1.0f - c1b) * pa_c);
    const float pk1 = (k == 1) ? 0.0f : r1 * (+c1a * pa_m + (c2a - 1.0f) * pa_c);
    const float mm = temm * (c2a * thc + c1a * th_m);
    const float A = pk1 + qk, B = pk2 - qk;
    // ---- explicit pi forcing
    float div = (un1 - un0) * rdx * uh_c + (vn1 - vn0) * rdy * vh_c;
    if (fabsf(div) < smeps) div = 0.0f;
    const float fpk = dts * (ppten - ppterm * div) +
                      (-(un0 * (pa_c - paw) + un1 * (pae - pa_c)) * temx * uh_c -
                       (vn0 * (pa_c - pas) + vn1 * (pan - pa_c)) * temy * vh_c) +
                      beta * (w_c * (pk1 + qk) + w_p * (pk2 - qk));
    // ---- Thomas forward sweep
    if (k == 1) {
      w_bot = w_c;
    } else {
      const float aa = -asq * (+mm * A_m);
      const float cc = -asq * (-mm * B);
      const float bb = 1.0f - asq * (+mm * (-A + B_m));
      const float fwk = dts * wten + beta * (-mm * (pp_c - pp_m));
      const float dd = w_c + fwk + alph * (-mm * ((pp_c + fpk) - (pp_m + fpk_m)));
      if (k == 2) {
        const float rr = 1.0f / bb;
        d1p = -cc * rr;
        d2p = dd * rr;
      } else {
        const float rr = 1.0f / (aa * d1p + bb);
        d1p = -cc * rr;
        d2p = (dd - aa * d2p) * rr;
      }
      if (k == nk) w_top = d2p;
    }
    // ---- stores
    a.uY[c] = un0;
    a.vY[c] = vn0;
    if (a.fold) {
      a.rru[c] = avg_uv(a, rruc, uXc, un0);
      a.rrv[c] = avg_uv(a, rrvc, vXc, vn0);
    }
    a.fpk[c] = fpk;
    // d1 depends only on the stage's fixed coefficients (thv, piadv,
    // ppterm, dts): stored on the first substep, read on the others
    if (k >= 2 && k < nk) {
      if (a.first) a.dum1[c] = d1p;
      a.dum2[c] = d2p;
    }
    if (k == nk) w_nk1 = w_p;
    A_m = A;
    B_m = B;
    fpk_m = fpk;
    pp_m = pp_c;
    pa_m = pa_c;
    pa_c = pa_p;
    th_m = thc;
    w_c = w_p;
  }

  // back substitution, pi update, w average (top down)
  c = IXD(P, i, j, nk);
  float w_above = w_nk1;
  float pa_p = a.piadv[c + pxy];
  float pa_c2 = a.piadv[c];
  // operands of the current level
  float q_d1 = 0.0f, q_d2 = 0.0f;
  float q_pp = a.ppR[c], q_fpk = a.fpk[c], q_pm = a.piadv[c - pxy], q_term = a.ppterm[c];
  auto rrw_of = [&](int cc) -> float {  // the w average before this substep's w
    if (!a.fold) return 0.0f;
    const float r = a.init ? a.wa[cc] * a.beta : a.rrw[cc];
    return a.pair ? r + a.wR[cc] : r;
  };
  float q_rrw = rrw_of(c);
  for (int k = nk; k >= 1; k--, c -= pxy) {
    const float p_old = q_pp, fk = q_fpk, pa_m2 = q_pm, pterm = q_term, rrwc = q_rrw;
    float wk;
    if (k == nk) {
      wk = w_top;
    } else if (k >= 2) {
      wk = q_d1 * w_above + q_d2;
    } else {
      wk = w_bot;
    }
    // prefetch the level below
    if (k > 1) {
      const int cb = c - pxy;
      if (k - 1 >= 2) {
        q_d1 = a.dum1[cb];
        q_d2 = a.dum2[cb];
      }
      q_pp = a.ppR[cb];
      q_fpk = a.fpk[cb];
      q_pm = a.piadv[cb - pxy];
      q_term = a.ppterm[cb];
      q_rrw = rrw_of(cb);
    }
    const float *cf = a.coef + 8 * k;
    const float tem = cf[0], r1 = cf[1], r2 = cf[2];
    const float c1a = cf[4], c1b = cf[5], c2a = cf[6], c2b = cf[7];
    const float qk = tem * pterm;
    const float pk2 = (k == nk) ? 0.0f : r2 * (-c2b * pa_p + (1.0f - c1b) * pa_c2);
    const float pk1 = (k == 1) ? 0.0f : r1 * (+c1a * pa_m2 + (c2a - 1.0f) * pa_c2);
    float pn = p_old + fk + alph * (wk * (pk1 + qk) + w_above * (pk2 - qk));
    if (fabsf(pn) < smeps) pn = 0.0f;
    const float d = a.kdiv * (pn - p_old);
    if (k >= 2 || a.wR != a.w3d) a.w3d[c] = wk;
    a.pp3d[c] = pn;
    if (a.ppx) a.ppx[c] = d;
    a.ppdY[c] = pn + d;
    if (!a.last) put_p_halo(P, a.ppdY, i, j, k, pn + d);
    if (a.fold) a.rrw[c] = a.last ? (rrwc + wk * alph) * a.tavg : rrwc + wk;
    w_above = wk;
    pa_p = pa_c2;
    pa_c2 = pa_m2;
  }
}

// ------------------------------------------------- acoustic substep, slabs
// The same substep with a workgroup per 64 columns of one row and NW
// wavefronts that each own L consecutive levels of those columns, so that
// what the vertical solve carries from its upward to its downward sweep
// stays on the chip (the solver's terms in registers, the pi coefficients
// and the old pi' in LDS) instead of going through fpk, dum2 and a second
// read of pi', ppterm and piadv.  Per column and substep that leaves 13
// arrays read (12 on a stage's first substep) and 5 written, plus the
// averages on every other substep.
//   1. every wavefront advances u, v and forms fpk and the solver's terms of
//      its levels;
//   2. the tridiagonal recurrences run up, then down the column, wavefront
//      after wavefront, in the reference's order (the values are exactly
//      those of one thread marching the column);
//   3. every wavefront updates pi' and the w average of its levels.
//
// Bound by memory: at 1024 x 1024 x 96, 2.03 ms a substep against 2.93 ms
// for sound_sub; 7.5 + 2.8 GB to and from memory (10.7 + 4.2 before), 5.0
// TB/s, what a plain copy reaches.  On small grids a column's levels are in
// flight together instead of one after the other: 256 x 256 x 64 104 us
// against 201, 64 x 64 x 40 20 us against 85.  12 levels per wavefront is
// the most that 128 registers hold (two workgroups of 8 wavefronts per CU):
// 6 and 8 levels (one workgroup of 16 or 12) 2.50 and 2.48 ms, 16 levels
// 3.04 ms; loading the next level's centre values ahead, paid for with a
// second read of dum1, 2.11 ms.
//
// The horizontal metrics uh, uf, vh, vf of sound_sub are all 1 (cm1g_create
// sets no other), and a product with 1 changes no value: left out here.
// Points are addressed by 32-bit byte offsets (ldo, sto): fields are below
// 4 GiB (slab_variant checks it).
struct SlabGrid {
  int nt, gx, per, nj, nw;  // tiles (64 columns x 1 row), tiles along i, tiles per XCD, rows, wavefronts
};
// Tiles are walked row by row in strips of this many tiles along i, a strip
// after the other, so that a tile's neighbours along i and j run on its XCD
// at about the same time and find each other's lines in its L2.  Measured at
// 1024 x 1024 x 96: strips of 1, 2, 4, 8 and 16 tiles 2.26, 2.09, 2.05, 2.02
// and 2.04 ms per substep (4.62e6 KB fetched with 16, 3.65e6 with 4).
constexpr int SLAB_STRIP = 8;

template <int L, int CAP, bool FIRST>
__device__ __forceinline__ void sound_slab(const KP &P, const SubArgs &a, const SlabGrid &sg, int bx) {
  __shared__ float sA[CAP][64], sB[CAP][64], sP[CAP][64];  // pk1 + qk, pk2 - qk, old pi'
  __shared__ float h0[CAP / L][64], h1[CAP / L][64];       // hand-over between wavefronts
  const int nmain = sg.per * NXCD;
  if (bx >= nmain) {
    const int npts = P.ni + P.nj + 1;
    const int t = (bx - nmain) * (int)blockDim.x + (int)threadIdx.x;
    if (t < npts * P.nk) sound_ring_point(P, a, t % npts, 1 + t / npts);
    return;
  }
  const int t = (bx % NXCD) * sg.per + bx / NXCD;
  if (t >= sg.nt) return;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  const int lane = (int)threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int strip = t / (SLAB_STRIP * sg.nj), t2 = t - strip * SLAB_STRIP * sg.nj;
  const int wid = min(SLAB_STRIP, sg.gx - strip * SLAB_STRIP);
  const int j = 1 + t2 / wid;
  const int iraw = 1 + (strip * SLAB_STRIP + t2 % wid) * 64 + lane;
  const bool on = iraw <= ni;
  const int i = on ? iraw : ni;  // lanes past the row's end follow its last column and store nothing
  const float dts = a.dts, rdx = P.rdx, rdy = P.rdy;
  const float alph = a.alph, beta = a.beta, asq = a.asq, smeps = P.K.smeps;
  // sides whose radiative update falls on this column; bw, be vary along the
  // wavefront, bs, bn do not (one row)
  const bool bw = a.opw && i == 1, be = a.ope && i == ni, bs = a.ops && j == 1, bn = a.opn && j == nj;
  const bool edge = bs || bn || __builtin_amdgcn_ballot_w64(bw || be) != 0ULL;
  const unsigned pxB = 4u * (unsigned)P.px, pxyB = 4u * (unsigned)P.pxy;
  const int k0 = 1 + wv * L;
  const unsigned c0 = 4u * (unsigned)IXD(P, i, j, k0);
  float sv[L], aa[L], rr[L], d1[L], dd[L];
  // the first level's terms that need the level below, kept for after the
  // wavefronts have met
  float mm0 = 0.0f, A0 = 0.0f, B0 = 0.0f, p0 = 0.0f, w0 = 0.0f, wt0 = 0.0f, d1m = 0.0f;
  float w_bot = 0.0f, w_top1 = 0.0f;
  if (k0 <= nk) {
    // dts times the masks dtu0, dtv0 at (i,j), (i+1,j), (i,j), (i,j+1): zero
    // on the faces of a non-periodic side (src/param.F:9182-9218)
    const float dtu_c = (P.ibw && i == 1) ? 0.0f : dts, dtu_e = (P.ibe && i == ni) ? 0.0f : dts;
    const float dtv_c = (P.ibs && j == 1) ? 0.0f : dts, dtv_n = (P.ibn && j == nj) ? 0.0f : dts;
    const float tem1 = a.tem1, tem2 = a.tem2, temx = a.temx, temy = a.temy;
    unsigned c = c0;
    float pa_m = ldo(a.piadv, c - pxyB), pa_c = ldo(a.piadv, c), th_m = ldo(a.thv, c - pxyB);
    float w_c = ldo(a.wR, c);
    if (!FIRST && k0 >= 3) d1m = ldo(a.dum1, c - pxyB);
    float A_m = 0.0f, B_m = 0.0f, s_m = 0.0f, pp_m = 0.0f;
#pragma unroll
    for (int l = 0; l < L; l++, c += pxyB) {
      const int k = k0 + l;
      if (k > nk) break;
      const unsigned cN = c + pxB, cS = c - pxB, cU = c + pxyB;
      const float uXc = ldo(a.uX, c), utc = ldo(a.uten, c), vXc = ldo(a.vX, c), vtc = ldo(a.vten, c), pdc = ldo(a.ppdX, c), thc = ldo(a.thv, c);
      const float ppterm = ldo(a.ppterm, c), ppten = ldo(a.ppten, c), wten = ldo(a.wten, c), pp_c = ldo(a.ppR, c);
      const float uXe = ldo(a.uX, c + 4u), ute = ldo(a.uten, c + 4u);
      const float vXn = ldo(a.vX, cN), vtn = ldo(a.vten, cN);
      const float pdw = ldo(a.ppdX, c - 4u), pde = ldo(a.ppdX, c + 4u);
      const float pds = ldo(a.ppdX, cS), pdn = ldo(a.ppdX, cN);
      const float thw = ldo(a.thv, c - 4u), the = ldo(a.thv, c + 4u);
      const float ths = ldo(a.thv, cS), thn = ldo(a.thv, cN);
      const float paw = ldo(a.piadv, c - 4u), pae = ldo(a.piadv, c + 4u);
      const float pas = ldo(a.piadv, cS), pan = ldo(a.piadv, cN), pa_p = ldo(a.piadv, cU);
      const float w_p = (k == nk) ? ldo(a.w3d, cU) : ldo(a.wR, cU);
      float rruc = 0.0f, rrvc = 0.0f;
      if (a.fold && !a.init) {
        rruc = ldo(a.rru, c);
        rrvc = ldo(a.rrv, c);
      }
      float d1c = 0.0f;
      if (!FIRST && k >= 2 && k < nk) d1c = ldo(a.dum1, c);
      // ---- u, v (ssopenbc* then src/sound.F:307-345)
      float uo0 = uXc, uo1 = uXe, vo0 = vXc, vo1 = vXn;
      if (edge) {
        if (bw) uo0 = uo0 + dts * (-a.radbcw[(j + 2) + k * P.py] * (uXe - uo0) * rdx + utc);
        if (be) uo1 = uo1 + dts * (-a.radbce[(j + 2) + k * P.py] * (uo1 - uXc) * rdx + ute);
        if (bs) vo0 = vo0 + dts * (-a.radbcs[(i + 2) + k * P.px] * (vXn - vo0) * rdy + vtc);
        if (bn) vo1 = vo1 + dts * (-a.radbcn[(i + 2) + k * P.px] * (vo1 - vXc) * rdy + vtn);
      }
      const float un0 = uo0 + dtu_c * (utc - tem1 * (pdc - pdw) * (thc + thw));
      const float un1 = uo1 + dtu_e * (ute - tem1 * (pde - pdc) * (the + thc));
      const float vn0 = vo0 + dtv_c * (vtc - tem2 * (pdc - pds) * (thc + ths));
      const float vn1 = vo1 + dtv_n * (vtn - tem2 * (pdn - pdc) * (thn + thc));
      // ---- coefficients (src/sound.F:117-180)
      const float *cf = a.coef + 8 * k;
      const float tem = cf[0], r1 = cf[1], r2 = cf[2], temm = cf[3];
      const float c1a = cf[4], c1b = cf[5], c2a = cf[6], c2b = cf[7];
      const float qk = tem * ppterm;
      const float pk2 = (k == nk) ? 0.0f : r2 * (-c2b * pa_p + (1.0f - c1b) * pa_c);
      const float pk1 = (k == 1) ? 0.0f : r1 * (+c1a * pa_m + (c2a - 1.0f) * pa_c);
      const float mm = temm * (c2a * thc + c1a * th_m);
      const float A = pk1 + qk, B = pk2 - qk;
      // ---- explicit pi forcing
      float div = (un1 - un0) * rdx + (vn1 - vn0) * rdy;
      if (fabsf(div) < smeps) div = 0.0f;
      const float fpk = dts * (ppten - ppterm * div) +
                        (-(un0 * (pa_c - paw) + un1 * (pae - pa_c)) * temx -
                         (vn0 * (pa_c - pas) + vn1 * (pan - pa_c)) * temy) +
                        beta * (w_c * (pk1 + qk) + w_p * (pk2 - qk));
      const float s = pp_c + fpk;
      sA[k - 1][lane] = A;
      sB[k - 1][lane] = B;
      sP[k - 1][lane] = pp_c;
      // ---- terms of the Thomas forward sweep
      if (l == 0) {
        mm0 = mm;
        A0 = A;
        B0 = B;
        p0 = pp_c;
        w0 = w_c;
        wt0 = wten;
      } else {
        aa[l] = -asq * (+mm * A_m);
        const float cc = -asq * (-mm * B);
        const float bb = 1.0f - asq * (+mm * (-A + B_m));
        const float fwk = dts * wten + beta * (-mm * (pp_c - pp_m));
        dd[l] = w_c + fwk + alph * (-mm * (s - s_m));
        if (FIRST) {
          rr[l] = bb;
          d1[l] = cc;
        } else {
          // d1 is fixed over a stage: its first substep stored it
          rr[l] = 1.0f / ((k == 2) ? bb : aa[l] * d1[l - 1 < 0 ? 0 : l - 1] + bb);
          d1[l] = d1c;
        }
      }
      if (!FIRST && l == 0) d1[0] = d1c;
      sv[l] = s;
      if (k == 1) w_bot = w_c;
      if (k == nk) w_top1 = w_p;
      // ---- u, v and their averages
      if (on) {
        sto(a.uY, c, un0);
        sto(a.vY, c, vn0);
        if (a.fold) {
          sto(a.rru, c, avg_uv(a, rruc, uXc, un0));
          sto(a.rrv, c, avg_uv(a, rrvc, vXc, vn0));
        }
      }
      A_m = A;
      B_m = B;
      s_m = s;
      pp_m = pp_c;
      pa_m = pa_c;
      pa_c = pa_p;
      th_m = thc;
      w_c = w_p;
    }
    h0[wv][lane] = s_m;
  }
  __syncthreads();
  if (k0 <= nk && k0 > 1) {
    const float A_m = sA[k0 - 2][lane], B_m = sB[k0 - 2][lane], pp_m = sP[k0 - 2][lane], s_m = h0[wv - 1][lane];
    aa[0] = -asq * (+mm0 * A_m);
    const float cc = -asq * (-mm0 * B0);
    const float bb = 1.0f - asq * (+mm0 * (-A0 + B_m));
    const float fwk = dts * wt0 + beta * (-mm0 * (p0 - pp_m));
    dd[0] = w0 + fwk + alph * (-mm0 * (sv[0] - s_m));
    if (FIRST) {
      rr[0] = bb;
      d1[0] = cc;
    } else {
      rr[0] = 1.0f / ((k0 == 2) ? bb : aa[0] * d1m + bb);
    }
  }
  __syncthreads();
  // forward sweep, wavefront after wavefront; h0 hands over d2, h1 d1
  for (int q = 0; q < sg.nw; q++) {
    if (wv == q && k0 <= nk) {
      float d1p = (FIRST && q > 0) ? h1[q - 1][lane] : 0.0f, d2p = (q > 0) ? h0[q - 1][lane] : 0.0f;
#pragma unroll
      for (int l = 0; l < L; l++) {
        const int k = k0 + l;
        if (k > nk) break;
        if (k == 1) continue;
        if (FIRST) {
          const float bb = rr[l], cc = d1[l];
          const float r = 1.0f / ((k == 2) ? bb : aa[l] * d1p + bb);
          d1p = -cc * r;
          d2p = (k == 2) ? dd[l] * r : (dd[l] - aa[l] * d2p) * r;
          d1[l] = d1p;
        } else {
          d2p = (k == 2) ? dd[l] * rr[l] : (dd[l] - aa[l] * d2p) * rr[l];
        }
        dd[l] = d2p;
      }
      h0[q][lane] = d2p;
      if (FIRST) h1[q][lane] = d1p;
    }
    __syncthreads();
  }
  // The old w and its running average for step 3, in the registers of the
  // forward sweep's terms (the last-level cache still holds the w that step
  // 1 read); d1 of a later substep likewise
  if (k0 <= nk) {
    if (a.fold) {
      const float *src = a.init ? a.wa : a.rrw;
#pragma unroll
      for (int l = 0; l < L; l++)
        if (k0 + l <= nk) {
          aa[l] = ldo(src, c0 + l * pxyB);
          rr[l] = a.pair ? ldo(a.wR, c0 + l * pxyB) : 0.0f;
        }
    }
  }
  // backward sweep; dd becomes w, h1 hands over the lowest w of a wavefront
  for (int q = sg.nw - 1; q >= 0; q--) {
    if (wv == q && k0 <= nk) {
      float w_above = (k0 + L <= nk) ? h1[q + 1][lane] : w_top1;
#pragma unroll
      for (int l = L - 1; l >= 0; l--) {
        const int k = k0 + l;
        if (k > nk) continue;
        float w;
        if (k == nk) w = dd[l];
        else if (k >= 2) w = d1[l] * w_above + dd[l];
        else w = w_bot;
        dd[l] = w;
        w_above = w;
      }
      h1[q][lane] = w_above;
    }
    __syncthreads();
  }
  // pi' update with divergence damping (src/sound.F:739-765), w average
  if (k0 > nk || !on) return;
  unsigned c = c0;
  const float w_next = (k0 + L <= nk) ? h1[wv + 1][lane] : w_top1;
#pragma unroll
  for (int l = 0; l < L; l++, c += pxyB) {
    const int k = k0 + l;
    if (k > nk) break;
    const float wk = dd[l];
    const float w_above = (k == nk) ? w_top1 : (l + 1 < L) ? dd[l + 1 < L ? l + 1 : l] : w_next;
    const float p_old = sP[k - 1][lane];
    float pn = sv[l] + alph * (wk * sA[k - 1][lane] + w_above * sB[k - 1][lane]);
    if (fabsf(pn) < smeps) pn = 0.0f;
    const float d = a.kdiv * (pn - p_old);
    if (a.fold) {
      float r = a.init ? aa[l] * beta : aa[l];
      if (a.pair) r = r + rr[l];
      sto(a.rrw, c, a.last ? (r + wk * alph) * a.tavg : r + wk);
    }
    if (k >= 2 || a.wR != a.w3d) sto(a.w3d, c, wk);
    sto(a.pp3d, c, pn);
    if (a.ppx) sto(a.ppx, c, d);
    sto(a.ppdY, c, pn + d);
    if (!a.last) put_p_halo(P, a.ppdY, i, j, k, pn + d);
    if (FIRST && k >= 2 && k < nk) sto(a.dum1, c, d1[l]);
  }
}

// The slab variants: levels per wavefront and levels a workgroup holds.
constexpr int SLAB_L[] = {0, 4, 8, 12, 12}, SLAB_CAP[] = {0, 64, 64, 96, 192};

template <int V, bool FIRST>
static void slab_go(cm1g_model *m, dim3 grd, dim3 blk, const KP &P, const SubArgs &a, const SlabGrid &sg) {
  constexpr int L = SLAB_L[V], CAP = SLAB_CAP[V], NT = 64 * (CAP / L);
  launch<NT, 4>(m, grd, blk, [=] __device__(int bx, int, int) { sound_slab<L, CAP, FIRST>(P, a, sg, bx); });
}
static void slab_launch(cm1g_model *m, int v, dim3 grd, dim3 blk, const KP &P, const SubArgs &a,
                        const SlabGrid &sg) {
  if (v == 1) a.first ? slab_go<1, true>(m, grd, blk, P, a, sg) : slab_go<1, false>(m, grd, blk, P, a, sg);
  else if (v == 2) a.first ? slab_go<2, true>(m, grd, blk, P, a, sg) : slab_go<2, false>(m, grd, blk, P, a, sg);
  else if (v == 3) a.first ? slab_go<3, true>(m, grd, blk, P, a, sg) : slab_go<3, false>(m, grd, blk, P, a, sg);
  else a.first ? slab_go<4, true>(m, grd, blk, P, a, sg) : slab_go<4, false>(m, grd, blk, P, a, sg);
}

// Which kernel runs the substep (0: sound_sub, one thread per column).
// sound_sub takes columns too deep for a workgroup's LDS, fields of 4 GiB and
// more, and shallow columns of a wide grid: a slab workgroup is then one to
// three wavefronts, and its LDS lets a CU hold three of them, while a thread
// per column fills the chip.  Six substeps, sound_sub / slabs of 8 levels:
// 1024 x 1024 x 7 1127 / 1778 us, x 16 2490 / 2805, x 20 3150 / 3188, x 24
// 3823 / 3535; 512 x 512 x 9 359 / 529, x 20 841 / 923; 100 x 2000 x 18 761 / 901;
// 512 x 256 x 8 225 / 280, x 12 291 / 316, x 16 369 / 349; 512 x 384 x 16 547 /
// 526; 384 x 256 x 8 192 / 218, x 12 257 / 246.
// Up to 64 levels 8 per wavefront, and under 1024 tiles (four workgroups per
// CU) 4, which put more wavefronts on a column.  Six substeps, 4 / 8 levels:
// 64 x 64 x 40 122 / 161 us, x 64 160 / 191; 256 x 128 x 20 148 / 170, but x 40
// 261 / 218; 256 x 256 x 24 247 / 288, x 64 817 / 658.  Above 64 levels there are
// 12 per wavefront for any grid: a workgroup's 16 wavefronts of 4 levels end
// there, and fewer than 12 lost on the large grid (above); on a small one only
// sound_sub was compared (64 x 64 x 96 1266 us, with 12 levels 247).
static int slab_variant(const cm1g_model *m) {
  const int nk = m->plan_nk > m->P.nk ? m->plan_nk : m->P.nk;
  const long tiles = m->plan_tiles > 0 ? m->plan_tiles : (long)((m->P.ni + 63) / 64) * m->P.nj;
  if (nk > 192 || m->ntot >= ((size_t)1 << 30)) return 0;
  if (tiles >= (nk <= 12 ? 2048 : 3840) && nk <= 20) return 0;
  if (nk <= 64) return tiles < 1024 ? 1 : 2;
  return nk <= 96 ? 3 : 4;
}

const char *sound_kernel(const cm1g_model *m) { return slab_variant(m) ? "sound_slab" : "sound_sub"; }

// the arguments that do not change over a stage, and its substep count
static void sub_args(cm1g_model *m, int nrk, SubArgs &a, int *nloop) {
  const KP &P = m->P;
  memset(&a, 0, sizeof(a));
  sound_nloop(nrk, m->c.nsound, m->c.dt, nloop, &a.dts);
  a.alph = m->c.alph;
  a.beta = 1.0f - a.alph;
  a.asq = a.alph * a.alph;
  a.kdiv = m->c.kdiv;
  a.tavg = 1.0f / (float)*nloop;
  a.tem1 = P.rdx * P.K.cp * 0.5f;
  a.tem2 = P.rdy * P.K.cp * 0.5f;
  a.temx = a.dts * 0.5f * P.rdx;
  a.temy = a.dts * 0.5f * P.rdy;
  a.opw = (P.wbc == 2 && P.ibw == 1);
  a.ope = (P.ebc == 2 && P.ibe == 1);
  a.ops = (P.sbc == 2 && P.ibs == 1);
  a.opn = (P.nbc == 2 && P.ibn == 1);
  a.uten = m->f[CM1G_UTEN];
  a.vten = m->f[CM1G_VTEN];
  a.wten = m->f[CM1G_WTEN];
  a.thv = m->f[CM1G_T11];
  a.piadv = m->f[CM1G_SADV];
  a.ppterm = m->f[CM1G_T22];
  a.ppten = m->f[CM1G_PPTEN];
  a.dtu0 = m->dtu0;
  a.dtv0 = m->dtv0;
  a.radbcw = m->d2[CM1G_D_RADBCW];
  a.radbce = m->d2[CM1G_D_RADBCE];
  a.radbcs = m->d2[CM1G_D_RADBCS];
  a.radbcn = m->d2[CM1G_D_RADBCN];
  a.w3d = m->f[CM1G_W3D];
  a.pp3d = m->f[CM1G_PP3D];
  a.fpk = m->f[CM1G_DUM8];
  a.dum1 = m->f[CM1G_DUM1];
  a.dum2 = m->f[CM1G_DUM2];
  a.rru = m->f[CM1G_RRU];
  a.rrv = m->f[CM1G_RRV];
  a.rrw = m->f[CM1G_RRW];
  a.wa = m->f[CM1G_WA];
}

// a last stage of one substep: its damping term waited in scratch, since
// other columns read ppx in the same launch
static void ppx_single(cm1g_model *m, int nrk, int nloop) {
  if (nrk != 3 || nloop != 1) return;
  const KP P = m->P;
  const float *d = m->tz;
  float *ppx = m->f[CM1G_PPX];
  for3(m, 1, P.ni, 1, P.nj, 1, P.nk, [=] __device__(int i, int j, int k) {
    const int c = IXD(P, i, j, k);
    ppx[c] = d[c];
  });
}

void sound_run(cm1g_model *m, int nrk, bool fold1) {
  const KP P = m->P;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  int nloop;
  SubArgs a;
  sub_args(m, nrk, a, &nloop);
  const float dts = a.dts;
  float *ppd = m->f[CM1G_DUM7];
  float *u3d = m->f[CM1G_U3D], *v3d = m->f[CM1G_V3D], *w3d = m->f[CM1G_W3D];
  const float *ua = m->f[CM1G_UA], *va = m->f[CM1G_VA], *wa = m->f[CM1G_WA];
  const float *ppi = m->f[CM1G_PPI];
  float *pp3d = m->f[CM1G_PP3D], *ppx = m->f[CM1G_PPX];

  // The copies the reference makes before the substeps (u3d=ua, ..., ppd=ppx,
  // src/sound.F:191-250) are folded into the first substep, which reads ua,
  // va, wa, ppi, ppx directly (after the first RK stage) and starts the
  // averages itself.  u, v and ppd alternate between the state arrays and
  // scratch arrays so that neighbouring columns read the old values; the
  // last substep writes u3d/v3d.
  // (at the first stage u3d..pp3d equal ua..ppi where the substep reads
  // them when the caller says so, fold1: the folded form then needs no
  // copy of the scratch pair back into u3d/v3d)
  const bool fold = (nrk >= 2) || fold1;
  const int slab = slab_variant(m);
  const ColGrid cg = col_grid(ni, nj, m->tile_rows);
  SlabGrid sg;
  sg.nj = nj;
  sg.gx = (ni + 63) / 64;
  sg.nt = sg.gx * nj;
  sg.per = (sg.nt + NXCD - 1) / NXCD;
  const int plan_nk = m->plan_nk > nk ? m->plan_nk : nk;
  const int lev = slab == 0 ? 1 : SLAB_L[slab];
  sg.nw = (plan_nk + lev - 1) / lev;
  const dim3 blk = slab ? dim3(64 * sg.nw) : col_threads(cg);
  dim3 grd = slab ? dim3(sg.per * NXCD) : col_blocks(cg);
  {
    const int nthr = (int)blk.x, npts = (ni + nj + 1) * nk;
    a.nring = (npts + nthr - 1) / nthr;
  }
  grd.x += a.nring;
  // the per-level solver coefficients of this stage's dts, with the
  // reference's expressions (src/sound.F:117-180)
  {
    float *cf = m->scoef;
    const float rdz = P.rdz, cp = P.K.cp;
    launch<64>(m, dim3((nk + 63) / 64), dim3(64), [=] __device__(int bx, int, int) {
      const int k = 1 + bx * 64 + (int)threadIdx.x;
      if (k > nk) return;
      float *o = cf + 8 * k;
      o[0] = dts * rdz * P.mh[k];
      o[1] = dts * rdz * P.mh[k] * P.rr0[k] * P.rf0[k];
      o[2] = dts * rdz * P.mh[k] * P.rr0[k] * P.rf0[k + 1];
      o[3] = dts * rdz * cp * P.mf[k];
      o[4] = P.c1[k];
      o[5] = P.c1[k + 1];
      o[6] = P.c2[k];
      o[7] = P.c2[k + 1];
    });
    a.coef = cf;
  }
  float *ppdb[2] = {ppd, m->tx};
  float *uprev = nullptr, *vprev = nullptr;
  for (int n = 1; n <= nloop; n++) {
    // destination of this substep: u3d on the last one, alternating before
    float *udst, *vdst;
    if (fold) {
      const bool scratch = ((nloop - n) & 1) != 0;
      udst = scratch ? m->scr1 : u3d;
      vdst = scratch ? m->scr2 : v3d;
    } else {
      const bool scratch = (n & 1) != 0;
      udst = scratch ? m->scr1 : u3d;
      vdst = scratch ? m->scr2 : v3d;
    }
    a.uX = (n == 1) ? (fold ? ua : u3d) : uprev;
    a.vX = (n == 1) ? (fold ? va : v3d) : vprev;
    a.uY = udst;
    a.vY = vdst;
    a.ppdX = (n == 1) ? ppx : ppdb[(n - 2) & 1];
    a.ppdY = ppdb[(n - 1) & 1];
    a.wR = (n == 1 && fold) ? wa : w3d;
    a.ppR = (n == 1 && fold) ? ppi : pp3d;
    a.wring = a.wR;
    a.wringp = (n == 2 && fold) ? wa : w3d;
    a.first = (n == 1);
    a.last = (n == nloop);
    a.fold = ((nloop - n) & 1) == 0;
    a.pair = (n > 1);
    a.init = (n <= 2);
    // the stage's damping term goes straight to ppx, unless this substep
    // also reads ppx at neighbouring columns (a single-substep stage)
    a.ppx = (nrk == 3 && a.last) ? (a.first ? m->tz : ppx) : nullptr;
    ktimer_mark(m, CM1G_KT_SOUND_SUBSTEP);
    if (slab == 0)
      launch<256>(m, grd, blk, [=] __device__(int bx, int, int) { sound_sub(P, a, cg, bx); });
    else
      slab_launch(m, slab, grd, blk, P, a, sg);
    ktimer_mark(m, CM1G_KT_SOUND_SUBSTEP);
    uprev = udst;
    vprev = vdst;
  }
  if (!fold && (nloop & 1)) {
    // the last substep wrote the scratch pair: copy the updated range back
    const float *us = m->scr1, *vs = m->scr2;
    for3(m, 1, ni + 1, 1, nj + 1, 1, nk, [=] __device__(int i, int j, int k) {
      int c = IXD(P, i, j, k);
      u3d[c] = us[c];
      v3d[c] = vs[c];
    });
  }
  ppx_single(m, nrk, nloop);
}

// ------------------------------------------------- explicit substeps
// Operands of one level of a sounde_col column (raw loads; w and wten at
// k + 1, which is where the level above starts).
struct EXLoads {
  float uXc, uXe, utc, ute, vXc, vXn, vtc, vtn;
  float pdw, pde, pds, pdn, pdp;
  float thw, the, ths, thn, thp;
  float paw, pae, pas, pan, pap;
  float ppterm, ppten, pp, w_p, wt_p;
  float rru, rrv, rrw;
};

// c: the point's byte offset (O: 32 bits, or 64 for fields of 4 GiB and more)
template <class O>
__device__ __forceinline__ void ex_load(const KP &P, const SubArgs &a, O c, int k, EXLoads &L) {
  const O pxB = (O)4 * P.px, pxyB = (O)4 * P.pxy, cN = c + pxB, cS = c - pxB, cU = c + pxyB;
  L.uXc = ldo(a.uX, c); L.uXe = ldo(a.uX + 1, c);
  L.utc = ldo(a.uten, c); L.ute = ldo(a.uten + 1, c);
  L.vXc = ldo(a.vX, c); L.vXn = ldo(a.vX, cN);
  L.vtc = ldo(a.vten, c); L.vtn = ldo(a.vten, cN);
  L.pdw = ldo(a.ppdX - 1, c); L.pde = ldo(a.ppdX + 1, c); L.pds = ldo(a.ppdX, cS); L.pdn = ldo(a.ppdX, cN);
  L.thw = ldo(a.thv - 1, c); L.the = ldo(a.thv + 1, c); L.ths = ldo(a.thv, cS); L.thn = ldo(a.thv, cN);
  L.paw = ldo(a.piadv - 1, c); L.pae = ldo(a.piadv + 1, c); L.pas = ldo(a.piadv, cS); L.pan = ldo(a.piadv, cN);
  L.ppterm = ldo(a.ppterm, c); L.ppten = ldo(a.ppten, c); L.pp = ldo(a.ppR, c);
  if (k < P.nk) {
    L.pdp = ldo(a.ppdX, cU); L.thp = ldo(a.thv, cU); L.pap = ldo(a.piadv, cU);
    L.w_p = ldo(a.wR, cU); L.wt_p = ldo(a.wten, cU);
  } else {
    L.pdp = L.thp = L.pap = L.wt_p = 0.0f;
    L.w_p = ldo(a.w3d, cU);  // the lid
  }
  L.rru = L.rrv = L.rrw = 0.0f;
  if (a.fold && !a.init) {
    L.rru = ldo(a.rru, c); L.rrv = ldo(a.rrv, c); L.rrw = ldo(a.rrw, c);
  }
}

// One explicit acoustic substep of a column (src/sounde.F:333-352, 548-563,
// 770-795): u, v, w from the previous substep's ppd, and the pressure from the
// new velocities, whose values at i+1, j+1 and k+1 are formed here too (the
// one at k+1 is then the level above's own).  u, v, w and ppd alternate
// between two arrays, so neighbours read the old values; the averages take in
// two substeps at a time, as in sound.  Per level row k of coef: p3, p4, p1,
// p2 of the pi0 advection (src/sounde.F:117-136, 160-170), temw, c1, c2, mh.
//
// Memory bound: 12 arrays read and 5 written a substep, and the averages
// every other one, against 18 and 8 for a velocity pass and a pressure pass.
// Measured on 512 x 512 x 128: 0.70 ms a substep at 4.7 TB/s, what a large copy
// reaches here, against 0.74 ms in two passes, and 0.9 ms a stage of copies that
// set the substep's fields up no longer run.
template <class O>
__device__ __forceinline__ void sounde_col(const KP &P, const SubArgs &a, const ColGrid &cg, int bx) {
  const int nmain = cg.per * NXCD;
  if (bx >= nmain) {
    const int npts = P.ni + P.nj + 1;
    const int t = (bx - nmain) * (int)blockDim.x + (int)threadIdx.x;
    if (t < npts * P.nk) sound_ring_point(P, a, t % npts, 1 + t / npts);
    return;
  }
  int i, j, ks, ke;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  if (!col_tile_seg(cg, bx, nk, i, j, ks, ke)) return;
  if (i > ni || j > nj) return;
  const bool bw = a.opw && i == 1, be = a.ope && i == ni, bs = a.ops && j == 1, bn = a.opn && j == nj;
  const bool edge = __builtin_amdgcn_ballot_w64(bw || be || bs || bn) != 0ULL;
  const float dts = a.dts, rdx = P.rdx, rdy = P.rdy, rdz = P.rdz, smeps = P.K.smeps;
  const float tem1 = a.tem1, tem2 = a.tem2, temx = a.temx, temy = a.temy;
  // dts times the masks dtu0, dtv0 (zero on the faces of a non-periodic side)
  const float dtu_c = (P.ibw && i == 1) ? 0.0f : dts, dtu_e = (P.ibe && i == ni) ? 0.0f : dts;
  const float dtv_c = (P.ibs && j == 1) ? 0.0f : dts, dtv_n = (P.ibn && j == nj) ? 0.0f : dts;
  const O pxyB = (O)4 * P.pxy;
  O c = (O)4 * IX2D(P, i, j) + (O)ks * pxyB;
  // values of this level carried from the one below
  float pd_c = ldo(a.ppdX, c), th_c = ldo(a.thv, c), pa_c = ldo(a.piadv, c), pa_m = 0.0f;
  float wo_c = ldo(a.wR, c), wn_c = wo_c;  // old and new w(k); w(1) does not change
  EXLoads nx;
  ex_load<O>(P, a, c, ks, nx);
  if (ks > 1) {
    const float *cf = a.coef + 8 * ks;
    pa_m = ldo(a.piadv, c - pxyB);
    wn_c = wo_c + dts * (ldo(a.wten, c) - cf[4] * (pd_c - ldo(a.ppdX, c - pxyB)) *
                                                 (cf[6] * th_c + cf[5] * ldo(a.thv, c - pxyB)));
  }
  for (int k = ks; k <= ke; k++, c += pxyB) {
    const EXLoads L = nx;
    if (k < ke) ex_load<O>(P, a, c + pxyB, k + 1, nx);
    float uo0 = L.uXc, uo1 = L.uXe, vo0 = L.vXc, vo1 = L.vXn;
    if (edge) {
      if (bw) uo0 = uo0 + dts * (-a.radbcw[(j + 2) + k * P.py] * (L.uXe - uo0) * rdx + L.utc);
      if (be) uo1 = uo1 + dts * (-a.radbce[(j + 2) + k * P.py] * (uo1 - L.uXc) * rdx + L.ute);
      if (bs) vo0 = vo0 + dts * (-a.radbcs[(i + 2) + k * P.px] * (L.vXn - vo0) * rdy + L.vtc);
      if (bn) vo1 = vo1 + dts * (-a.radbcn[(i + 2) + k * P.px] * (vo1 - L.vXc) * rdy + L.vtn);
    }
    const float u0 = uo0 + dtu_c * (L.utc - tem1 * (pd_c - L.pdw) * (th_c + L.thw));
    const float u1 = uo1 + dtu_e * (L.ute - tem1 * (L.pde - pd_c) * (L.the + th_c));
    const float v0 = vo0 + dtv_c * (L.vtc - tem2 * (pd_c - L.pds) * (th_c + L.ths));
    const float v1 = vo1 + dtv_n * (L.vtn - tem2 * (L.pdn - pd_c) * (L.thn + th_c));
    const float *cf = a.coef + 8 * k;
    float w1 = L.w_p, pk1 = 0.0f, pk2 = 0.0f;
    if (k < nk) {
      w1 = w1 + dts * (L.wt_p - cf[8 + 4] * (L.pdp - pd_c) * (cf[8 + 6] * L.thp + cf[8 + 5] * th_c));
      pk2 = cf[3] * L.pap + cf[2] * pa_c;
    }
    if (k > 1) pk1 = cf[0] * pa_m + cf[1] * pa_c;
    const float w0 = wn_c;
    float div = ((u1 - u0) * rdx + (v1 - v0) * rdy) + (w1 - w0) * rdz * cf[7];
    if (fabsf(div) < smeps) div = 0.0f;
    const float delp = dts * (L.ppten - L.ppterm * div) +
                       (-(u0 * (pa_c - L.paw) + u1 * (L.pae - pa_c)) * temx -
                        (v0 * (pa_c - L.pas) + v1 * (L.pan - pa_c)) * temy) +
                       (w0 * pk1 + w1 * pk2);
    float p = L.pp + delp;
    if (fabsf(p) < smeps) p = 0.0f;
    const float d = a.kdiv * delp;
    sto(a.uY, c, u0);
    sto(a.vY, c, v0);
    sto(a.wY, c, w0);
    sto(a.pp3d, c, p);
    sto(a.ppdY, c, p + d);
    if (!a.last) put_p_halo(P, a.ppdY, i, j, k, p + d);
    if (a.ppx) sto(a.ppx, c, d);
    if (a.fold) {
      sto(a.rru, c, avg_uv(a, L.rru, L.uXc, u0));
      sto(a.rrv, c, avg_uv(a, L.rrv, L.vXc, v0));
      sto(a.rrw, c, avg_uv(a, L.rrw, wo_c, w0));
    }
    pd_c = L.pdp;
    th_c = L.thp;
    pa_m = pa_c;
    pa_c = L.pap;
    wo_c = L.w_p;
    wn_c = w1;
  }
}

// The part of those copies that lies outside the points the substeps write:
// point r of the border i = 0, ni+1 or j = 0, nj+1 at level k.  rru, rrv, rrw
// are 0, and u3d, v3d the state's, at i = 0 and j = 0; w3d and pp3d are the
// state's on the whole border (copy: where the reference copies).
struct SoundeBorder {
  float *u, *v, *w, *p, *rru, *rrv, *rrw;
  const float *ua, *va, *wa, *ppi;
  int npts, copy;
};
__device__ __forceinline__ void sounde_border(const KP &P, const SoundeBorder &b, int q) {
  const int k = 1 + q / b.npts, ni = P.ni, nj = P.nj;
  if (k > P.nk) return;
  int r = q % b.npts, i, j;
  if (r < 2 * (ni + 2)) {
    j = (r < ni + 2) ? 0 : nj + 1;
    i = (r < ni + 2) ? r : r - (ni + 2);
  } else {
    r -= 2 * (ni + 2);
    i = (r < nj) ? 0 : ni + 1;
    j = 1 + ((r < nj) ? r : r - nj);
  }
  const int c = IXD(P, i, j, k);
  if (i == 0 || j == 0) {
    b.rru[c] = 0.0f;
    b.rrv[c] = 0.0f;
    b.rrw[c] = 0.0f;
    if (b.copy) {
      b.u[c] = b.ua[c];
      b.v[c] = b.va[c];
    }
  }
  if (b.copy) {
    b.w[c] = b.wa[c];
    b.p[c] = b.ppi[c];
  }
}

// Explicit acoustic substeps, psolver=2 (sounde, src/sounde.F:10-1026;
// Cartesian, no terrain).  The copies the reference makes before the substeps
// (u3d=ua, ..., ppd=ppx, src/sounde.F:181-233) are folded into the first one
// (fold: from the second stage on, or where the caller says that u3d..pp3d
// equal ua..ppi); the border around its points is set with the coefficients.
void sounde_run(cm1g_model *m, int nrk, bool fold1) {
  const KP P = m->P;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  int nloop;
  SubArgs a;
  sub_args(m, nrk, a, &nloop);
  a.expl = 1;
  const bool fold = (nrk >= 2) || fold1;
  float *u3d = m->f[CM1G_U3D], *v3d = m->f[CM1G_V3D], *w3d = m->f[CM1G_W3D], *pp3d = m->f[CM1G_PP3D];
  const float *ua = m->f[CM1G_UA], *va = m->f[CM1G_VA], *wa = m->f[CM1G_WA], *ppi = m->f[CM1G_PPI];
  {
    float *cf = m->scoef;
    const float dts = a.dts, rdz = P.rdz, cp = P.K.cp;
    SoundeBorder bd = {u3d, v3d, w3d, pp3d, a.rru, a.rrv, a.rrw, ua, va, wa, ppi};
    bd.npts = 2 * (ni + 2) + 2 * nj;
    // (the first stage steps from u3d.. as they are, unless an exchanging
    // solve3 has left the previous step in them)
    bd.copy = nrk >= 2 || m->swapped;
    const int nkb = (nk + 63) / 64;
    launch<64>(m, dim3(nkb + (bd.npts * nk + 63) / 64), dim3(64), [=] __device__(int bx, int, int) {
      if (bx >= nkb) {
        sounde_border(P, bd, (bx - nkb) * 64 + (int)threadIdx.x);
        return;
      }
      const int k = 1 + bx * 64 + (int)threadIdx.x;
      if (k > nk) return;
      float *o = cf + 8 * k;
      const float mh = P.mh[k], rr0 = P.rr0[k];
      o[0] = dts * rdz * mh * rr0 * P.rf0[k] * P.c1[k];
      o[1] = dts * rdz * mh * rr0 * P.rf0[k] * (P.c2[k] - 1.0f);
      o[2] = dts * rdz * mh * rr0 * P.rf0[k + 1] * (1.0f - P.c1[k + 1]);
      o[3] = -(dts * rdz * mh * rr0 * P.rf0[k + 1] * P.c2[k + 1]);
      o[4] = rdz * cp * P.mf[k];
      o[5] = P.c1[k];
      o[6] = P.c2[k];
      o[7] = mh;
    });
    a.coef = cf;
  }
  ColGrid cg = col_grid(ni, nj, m->tile_rows);
  col_split(m, cg, nk);
  const dim3 blk = col_threads(cg);
  dim3 grd = col_blocks(cg);
  a.nring = ((ni + nj + 1) * nk + (int)blk.x - 1) / (int)blk.x;
  grd.x += a.nring;
  float *ppx = m->f[CM1G_PPX], *ppdb[2] = {m->f[CM1G_DUM7], m->tx};
  float *us = m->scr1, *vs = m->scr2, *ws = m->ty;
  const float *up = nullptr, *vp = nullptr, *wp = nullptr;
  a.wring = fold ? wa : w3d;
  for (int n = 1; n <= nloop; n++) {
    // the last substep writes u3d; from the state arrays themselves the first
    // one writes the scratch set
    const bool scratch = fold ? ((nloop - n) & 1) != 0 : (n & 1) != 0;
    a.uX = (n == 1) ? (fold ? ua : u3d) : up;
    a.vX = (n == 1) ? (fold ? va : v3d) : vp;
    a.wR = (n == 1) ? (fold ? wa : w3d) : wp;
    a.uY = scratch ? us : u3d;
    a.vY = scratch ? vs : v3d;
    a.wY = scratch ? ws : w3d;
    a.ppdX = (n == 1) ? ppx : ppdb[n & 1];
    a.ppdY = ppdb[(n - 1) & 1];
    a.ppR = (n == 1 && fold) ? ppi : pp3d;
    a.first = (n == 1);
    a.last = (n == nloop);
    a.fold = ((nloop - n) & 1) == 0;
    a.pair = (n > 1);
    a.init = (n <= 2);
    a.ppx = (nrk == 3 && a.last) ? (a.first ? m->tz : ppx) : nullptr;
    if (m->ntot < ((size_t)1 << 30))
      launch<256>(m, grd, blk, [=] __device__(int bx, int, int) { sounde_col<unsigned>(P, a, cg, bx); });
    else
      launch<256>(m, grd, blk, [=] __device__(int bx, int, int) { sounde_col<size_t>(P, a, cg, bx); });
    up = a.uY;
    vp = a.vY;
    wp = a.wY;
  }
  if (!fold && (nloop & 1)) {
    // the last substep wrote the scratch set: copy the updated range back
    for3(m, 1, ni + 1, 1, nj + 1, 1, nk, [=] __device__(int i, int j, int k) {
      const int c = IXD(P, i, j, k);
      u3d[c] = us[c];
      v3d[c] = vs[c];
      if (i <= ni && j <= nj) w3d[c] = ws[c];
    });
  }
  ppx_single(m, nrk, nloop);
}

// getdiv (t11 from the time-averaged velocities) and getdivx (divx from the
// mass fluxes scaled by rho0/rf0; inside the time step the advection
// kernels apply the same scaling on the fly instead of storing scaled
// copies).  want_divx = 0 computes only the divergence into `div`.
void getdiv_both(cm1g_model *m, int want_t11, int want_divx, float *div) {
  const KP P = m->P;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  const float *rru = m->f[CM1G_RRU], *rrv = m->f[CM1G_RRV], *rrw = m->f[CM1G_RRW];
  float *t11 = div ? div : m->f[CM1G_T11], *divx = m->f[CM1G_DIVX];
  const float smeps = P.K.smeps;
  for3(m, 1, ni, 1, nj, 1, nk, [=] __device__(int i, int j, int k) {
    int c = IXD(P, i, j, k);
    if (want_t11) {
      float d = ((rru[IXD(P, i + 1, j, k)] - rru[c]) * P.rdx +
                 (rrv[IXD(P, i, j + 1, k)] - rrv[c]) * P.rdy) +
                (rrw[IXD(P, i, j, k + 1)] - rrw[c]) * P.rdz * P.mh[k];
      if (fabsf(d) < smeps) d = 0.0f;
      t11[c] = d;
    }
    if (!want_divx) return;
    float ru1 = rru[IXD(P, i + 1, j, k)] * P.rho0[k], ru0 = rru[c] * P.rho0[k];
    float rv1 = rrv[IXD(P, i, j + 1, k)] * P.rho0[k], rv0 = rrv[c] * P.rho0[k];
    float rw1 = (k == nk) ? 0.0f : rrw[IXD(P, i, j, k + 1)] * P.rf0[k + 1];
    float rw0 = (k == 1) ? 0.0f : rrw[c] * P.rf0[k];
    float d = ((ru1 - ru0) * P.rdx + (rv1 - rv0) * P.rdy) +
              (rw1 - rw0) * P.rdz * P.mh[k];
    if (fabsf(d) < smeps) d = 0.0f;
    divx[c] = d;
  });
}

// The in-place scaling of getdivx (src/misclibs.F:246-273): rru, rrv by
// rho0, rrw by rf0 with rrw = 0 at k = 1 and nk+1, over the reference's
// ranges.  Only the routine-level entry stores the scaled fluxes.
void scale_mass_fluxes(cm1g_model *m) {
  const KP P = m->P;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  float *rru = m->f[CM1G_RRU], *rrv = m->f[CM1G_RRV], *rrw = m->f[CM1G_RRW];
  for3(m, 1, ni + 1, 1, nj + 1, 1, nk, [=] __device__(int i, int j, int k) {
    const int c = IXD(P, i, j, k);
    if (j <= nj) rru[c] = rru[c] * P.rho0[k];
    if (i <= ni) rrv[c] = rrv[c] * P.rho0[k];
    if (i <= ni && j <= nj) {
      if (k == 1) {
        rrw[c] = 0.0f;
        rrw[IXD(P, i, j, nk + 1)] = 0.0f;
      } else {
        rrw[c] = rrw[c] * P.rf0[k];
      }
    }
  });
}

// calccflquick: per-level maximum of the Courant magnitude, then the max.
#define CFL_NB 32
__device__ __forceinline__ void cfl_levels(const KP &P, float dt, const float *ua, const float *va,
                                           const float *wa, float *out, int bx, int by) {
  __shared__ float red[256];
  const int k = 1 + bx, b = by;
  const float dtdx = 0.5f * dt * P.rdx, dtdy = 0.5f * dt * P.rdy, dtdz = 0.5f * dt * P.rdz;
  float cfl = 0.0f;
  for (int j = 1 + b; j <= P.nj; j += CFL_NB)
    for (int i = 1 + (int)threadIdx.x; i <= P.ni; i += blockDim.x) {
      float a = (ua[IXD(P, i, j, k)] + ua[IXD(P, i + 1, j, k)]) * dtdx;
      float bb = (va[IXD(P, i, j, k)] + va[IXD(P, i, j + 1, k)]) * dtdy;
      float c = (wa[IXD(P, i, j, k)] + wa[IXD(P, i, j, k + 1)]) * dtdz * P.mh[k];
      float wsp = sqrtf((a * a + bb * bb) + c * c);
      cfl = fmaxf(cfl, wsp);
    }
  cfl = block_reduce256(cfl, red, OpMaxF());
  if (threadIdx.x == 0) out[1 + (k - 1) * CFL_NB + b] = cfl;
}

// maximum over the per-level partial maxima (exact in any order); one thread
// walking them took 54 us at 40 levels and 134 us at 96
__device__ __forceinline__ void cfl_final(int n, float *out) {
  __shared__ float red[256];
  float cfl = -99999999.0f;
  for (int t = 1 + (int)threadIdx.x; t <= n; t += 256) cfl = fmaxf(cfl, out[t]);
  cfl = block_reduce256(cfl, red, OpMaxF());
  if (threadIdx.x == 0) out[0] = cfl;
}

void cfl_run(cm1g_model *m, float dt, const float *u, const float *v, const float *w) {
  const KP P = m->P;
  float *out = m->fred;
  launch<256>(m, dim3(P.nk, CFL_NB), dim3(256),
              [=] __device__(int bx, int by, int) { cfl_levels(P, dt, u, v, w, out, bx, by); });
  const int n = P.nk * CFL_NB;
  launch<256>(m, dim3(1), dim3(256), [=] __device__(int, int, int) { cfl_final(n, out); });
}
