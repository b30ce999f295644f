// Flux-form advection on the device.
// flx3/flx5: src/adv_routines.F:5971-5984, :6006-6019.  hadv_flx5
// :1335-1476, vadv_flx5 :3269-3388 (+ vadv_lwr_flx_23 :4817-4995,
// vadv_lwr_flx_35 :5001-5169).  advs: src/adv.F:14-903, advu :911-1839,
// advv :1847-2770, advw :2778-3610; pdef: src/pdef.F:15-581.
//
// Every flux is evaluated with the reference's operation order in FP32
// without contraction, so results are bitwise those of the reference.
#include "cm1g_adv_common.h"
#include "cm1g_pdef_visit.h"

// ------------------------------------------------------------------ pdef
// The positive-definite correction (pdscheme=1, src/pdef.F:15-581), per
// direction: dum = rho0*s0 + dt*(adv + s*div) (pdefx1/pdefy1/pdefz), its
// halo fill (bcs, or zero below and above the column), and the mass each
// cell takes from or gives to its two neighbours (pdefx2/pdefy2/pdefz).
// The reference scatters inside a sequential loop; here each cell gathers
// the same terms in the same order (left neighbour, itself, right
// neighbour), which reproduces the sequential sums bit for bit.
//
// Only a cell with a negative dum, and the cells next to it, are corrected.
// So the advection kernel itself forms every cell's dum (it holds all the
// operands), writes the uncorrected update and a bit per cell that says
// whether a dum was negative; pdef_fix then reads the bits, and where one is
// set nearby it evaluates dum at the points a cell needs, mapping halo points
// to the interior point the fill copies, and writes the corrected update.

// mass flux of direction dir at the lower face of (c, level k) and at the
// upper one (c + stride): with scale, the getdivx scaling rho0(k) for u,v
// and rf0 for w (zero at k=1 and nk+1)
__device__ __forceinline__ void pdef_faces(const KP &P, int dir, const float *vel, int scale, int c,
                                           int k, float &lo, float &hi) {
  if (dir == 0) {
    lo = vel[c];
    hi = vel[c + 1];
    if (scale) { lo = lo * P.rho0[k]; hi = hi * P.rho0[k]; }
  } else if (dir == 1) {
    lo = vel[c];
    hi = vel[c + P.px];
    if (scale) { lo = lo * P.rho0[k]; hi = hi * P.rho0[k]; }
  } else {
    lo = vel[c];
    hi = vel[c + P.pxy];
    if (scale) {
      lo = (k == 1) ? 0.0f : lo * P.rf0[k];
      hi = (k + 1 == P.nk + 1) ? 0.0f : hi * P.rf0[k + 1];
    }
  }
}

// dum at (i,j,k) for direction dir (0 x, 1 y, 2 z), interior point
__device__ __forceinline__ float pdef_dum(const KP &P, int dir, const float *vel, int scale,
                                          const float *adv, const float *s0, const float *s, float dt,
                                          int i, int j, int k) {
  const int c = IXD(P, i, j, k);
  float lo, hi;
  pdef_faces(P, dir, vel, scale, c, k, lo, hi);
  // s*(flux difference)*metric, associated left to right as the reference
  // writes it (src/pdef.F:44-45, :256-257, :482-483)
  const float sc = s[c];
  float sdiv;
  if (dir == 0) sdiv = sc * (hi - lo) * P.rdx;
  else if (dir == 1) sdiv = sc * (hi - lo) * P.rdy;
  else sdiv = sc * (hi - lo) * P.rdz * P.mh[k];
  float d = P.rho0[k] * s0[c] + dt * (adv[c] + sdiv);
  if (dir == 0) {
    if (P.wbc == 2 && P.ibw == 1 && i == 1 && lo >= 0.0f) d = P.rho0[k] * s0[c];
    if (P.ebc == 2 && P.ibe == 1 && i == P.ni && hi <= 0.0f) d = P.rho0[k] * s0[c];
  } else if (dir == 1) {
    if (P.sbc == 2 && P.ibs == 1 && j == 1 && lo >= 0.0f) d = P.rho0[k] * s0[c];
    if (P.nbc == 2 && P.ibn == 1 && j == P.nj && hi <= 0.0f) d = P.rho0[k] * s0[c];
  }
  return d;
}

// the corrected tendency of one cell from dum at offsets -2..2 along the
// direction; vm/vp: the neighbours -1/+1 are cells the reference visits
__device__ __forceinline__ float pdef_gather(float dm2, float dm1, float d0, float dp1, float dp2,
                                             bool vm, bool vp, float smeps, bool &flag) {
  float mass = 0.0f;
  flag = false;
  if (vm && dm1 < 0.0f) {
    const float foo1 = fmaxf(0.0f, dm2), foo2 = fmaxf(0.0f, d0);
    if (foo1 + foo2 > smeps) {
      const float foo3 = fmaxf(dm1, -(foo1 + foo2)) / (foo1 + foo2);
      mass = mass + foo2 * foo3;
      if (d0 > smeps) flag = true;
    }
  }
  if (d0 < 0.0f) {
    const float foo1 = fmaxf(0.0f, dm1), foo2 = fmaxf(0.0f, dp1);
    if (foo1 + foo2 > smeps) {
      const float foo3 = fmaxf(d0, -(foo1 + foo2)) / (foo1 + foo2);
      mass = mass - (foo1 + foo2) * foo3;
      flag = true;
    }
  }
  if (vp && dp1 < 0.0f) {
    const float foo1 = fmaxf(0.0f, d0), foo2 = fmaxf(0.0f, dp2);
    if (foo1 + foo2 > smeps) {
      const float foo3 = fmaxf(dp1, -(foo1 + foo2)) / (foo1 + foo2);
      mass = mass + foo1 * foo3;
      if (d0 > smeps) flag = true;
    }
  }
  return mass;
}

struct PdefArgs {
  const float *rru, *rrv, *rrw, *advx, *advy, *advz, *s0, *s, *sten0, *divx;
  const unsigned long long *marks;  // per level, row and 64 columns: advs_col
  float *out_sten, *out_new;
  float dt;
  int smeps_flush, scale, gx, lev;
};

constexpr int PDEF_L = 8;  // most levels a pdef_fix workgroup looks after

// One workgroup per tile of 64 x 4 columns and a.lev levels: its threads
// read the marks of the tile and of its neighbours, and the workgroup visits
// the levels on which a cell of the tile can be corrected.  There each cell's
// dum in x and in y is evaluated once and shared through LDS (the tile's own
// points and two-point halos); dum in z stays in registers, as a window that
// moves up while consecutive levels are visited.  A cell no correction
// reaches keeps what the advection kernel wrote.
//
// Memory bound, in all 25 arrays a field before (advx, advy, advz written,
// a pass over x and y, a pass over z), 11 and the visited tiles' now.
// Measured, advection and correction of a field: 1024 x 1024 x 96 (qv, qc, qr)
// 2.53 -> 1.48 ms, of which pdef_fix 0.25; 512 x 512 x 128 (WENO, tracers) 0.95
// -> 0.55, pdef_fix 0.03; 64 x 64 x 40, where every tile is visited, 25 -> 19 us.
__device__ __forceinline__ void pdef_fix(const KP &P, const PdefArgs &a, int bx, int by, int bz) {
  __shared__ float dxs[4][68];
  __shared__ float dys[8][64];
  __shared__ unsigned need;
  const int tx = (int)threadIdx.x, ty = (int)threadIdx.y, t = ty * 64 + tx;
  const int i0 = 1 + bx * 64, j0 = 1 + by * 4;
  const int i = i0 + tx, j = j0 + ty;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  const int lev = a.lev, k0 = 1 + bz * lev, k1 = min(k0 + lev - 1, nk);
  const bool perx = (P.wbc == 1), pery = (P.sbc == 1);
  if (t == 0) need = 0u;
  __syncthreads();
  {
    static_assert(6 * (PDEF_L + 2) + 8 * PDEF_L <= 256, "one word a thread");
    const int own = 6 * (lev + 2);  // rows j0-1..j0+4, levels k0-1..k0+lev
    const unsigned all = (1u << lev) - 1u;
    unsigned m = 0u;
    if (t < own) {
      const int b = t / 6 - 1, r = t - 6 * (b + 1), k = k0 + b;
      const int jj = pdef_wrap(j0 - 1 + r, nj, pery);
      if (k >= 1 && k <= nk && a.marks[((size_t)(k - 1) * nj + (jj - 1)) * a.gx + bx])
        m = (r == 0 || r == 5) ? (b >= 0 ? 1u << b : 0u) : (7u << (b + 1)) >> 2;
    } else if (t < own + 8 * lev) {
      // the columns on either side, rows j0..j0+3
      const int u = t - own, b = u >> 3, k = k0 + b;
      const int ii = pdef_side_col(i0, ni, u & 1, perx);
      const int jj = pdef_wrap(j0 + ((u >> 1) & 3), nj, pery);
      if (k <= nk &&
          ((a.marks[((size_t)(k - 1) * nj + (jj - 1)) * a.gx + ((ii - 1) >> 6)] >> ((ii - 1) & 63)) & 1ULL))
        m = 1u << b;
    }
    m &= all;
    if (m) atomicOr(&need, m);
  }
  __syncthreads();
  const unsigned nd = __builtin_amdgcn_readfirstlane(need);
  if (nd == 0u) return;
  const bool in = (i <= ni && j <= nj);
  const int ii = pdef_wrap(i, ni, perx), jj = pdef_wrap(j, nj, pery);
  const int ic = min(i, ni), jc = min(j, nj);
  const int o = (tx < 2) ? tx - 2 : 62 + tx, hr = (ty < 2) ? ty : ty + 4;
  const int ih = pdef_wrap(i0 + o, ni, perx), jh = pdef_wrap(j0 - 2 + hr, nj, pery);
  const float smeps = P.K.smeps, rdt = 1.0f / a.dt;
  auto dz = [&](int kk) -> float {  // dum of pdefz; zero outside 1..nk
    if (kk < 1 || kk > nk) return 0.0f;
    return pdef_dum(P, 2, a.rrw, a.scale, a.advz, a.s0, a.s, a.dt, ic, jc, kk);
  };
  float dm2 = 0.0f, dm1 = 0.0f, d0 = 0.0f, dp1 = 0.0f, dp2 = 0.0f;
  for (int k = k0, last = -1; k <= k1; k++) {
    if (!((nd >> (k - k0)) & 1u)) continue;
    // (the previous level's cells have been read)
    if (last >= 0) __syncthreads();
    dxs[ty][tx + 2] = pdef_dum(P, 0, a.rru, a.scale, a.advx, a.s0, a.s, a.dt, ii, jc, k);
    if (tx < 4)
      dxs[ty][(tx < 2) ? tx : 64 + tx] = pdef_dum(P, 0, a.rru, a.scale, a.advx, a.s0, a.s, a.dt, ih, jc, k);
    dys[ty + 2][tx] = pdef_dum(P, 1, a.rrv, a.scale, a.advy, a.s0, a.s, a.dt, ic, jj, k);
    dys[hr][tx] = pdef_dum(P, 1, a.rrv, a.scale, a.advy, a.s0, a.s, a.dt, ic, jh, k);
    if (last == k - 1) {
      dm2 = dm1;
      dm1 = d0;
      d0 = dp1;
      dp1 = dp2;
    } else {
      dm2 = dz(k - 2);
      dm1 = dz(k - 1);
      d0 = dz(k);
      dp1 = dz(k + 1);
    }
    dp2 = dz(k + 2);
    last = k;
    __syncthreads();
    bool fx, fy, fz;
    const float *dx = &dxs[ty][tx];
    const float mx = pdef_gather(dx[0], dx[1], dx[2], dx[3], dx[4], true, true, smeps, fx);
    const float my = pdef_gather(dys[ty][tx], dys[ty + 1][tx], dys[ty + 2][tx], dys[ty + 3][tx], dys[ty + 4][tx],
                                 true, true, smeps, fy);
    const float mz = pdef_gather(dm2, dm1, d0, dp1, dp2, k - 1 >= 1, k + 1 <= nk, smeps, fz);
    if (in && (fx || fy || fz)) {
      const int c = IXD(P, i, j, k);
      const float sc = a.s[c], s0 = a.s0[c], r0s0 = P.rho0[k] * s0;
      float ax = a.advx[c], ay = a.advy[c], az = a.advz[c], lo, hi;
      if (fx) {
        pdef_faces(P, 0, a.rru, a.scale, c, k, lo, hi);
        ax = (dx[2] + mx - r0s0) * rdt - sc * (hi - lo) * P.rdx;
      }
      if (fy) {
        pdef_faces(P, 1, a.rrv, a.scale, c, k, lo, hi);
        ay = (dys[ty + 2][tx] + my - r0s0) * rdt - sc * (hi - lo) * P.rdy;
      }
      if (fz) {
        pdef_faces(P, 2, a.rrw, a.scale, c, k, lo, hi);
        az = (d0 + mz - r0s0) * rdt - sc * (hi - lo) * P.rdz * P.mh[k];
      }
      const float st = a.sten0[c] + ((ax + ay) + az + sc * a.divx[c]) * P.rr0[k];
      if (a.out_sten) a.out_sten[c] = st;
      if (a.out_new) {
        float v = s0 + a.dt * st;
        if (a.smeps_flush && fabsf(v) < smeps) v = 0.0f;
        a.out_new[c] = v;
      }
    }
  }
}

// ------------------------------------------------------ fused advs column
struct AdvsArgs {
  const float *s;                 // advected scalar
  float sadd;                     // nonzero: advect (th0(k)-th0r) + s
  const float *s0, *sten0, *t11, *thterm, *rru, *rrv, *rrw, *divx;
  float *out_sten, *out_new;      // tendency and/or s0 + dt*tendency
  float *advx, *advy, *advz;      // positive-definite pass: the three advective tendencies,
  unsigned long long *marks;      // and a bit per cell, set where a dum is negative
  float dt;
  int smeps_flush, gx;            // gx: words of marks per row
  int pdef, pdefweno;             // WENO5 magnitude tests (horizontal / vertical)
  double weps;
  int scale;                      // rru/rrv/rrw are the averaged velocities: scale by
                                  // rho0 / rf0 on the fly (getdivx, src/misclibs.F:222-370)
};

// Operands of one level of a advs_col column (raw loads; the theta
// offset th0-th0r is applied when they are used).
struct AdvLevel {
  float xm3, xm2, xm1, xp1, xp2, xp3;  // s(i-3..i+3), centre excluded
  float ym3, ym2, ym1, yp1, yp2, yp3;  // s(j-3..j+3)
  float ru0, ru1, rv0, rv1, rw1;       // face mass fluxes (rw1: face k+1)
  float dv, st0, sv0, t11v, thtv;      // divx, initial tendency, s0, t11, thterm
  float wnew;                          // s(k+4), entering the vertical window
};

// o: the column's byte offset in a level.  The start of level k of an array,
// and of its neighbouring rows, is formed in scalar registers, so a level's
// loads need no address arithmetic in vector registers.
template <bool PD, bool TH>
__device__ __forceinline__ void advs_load(const KP &P, const AdvsArgs &a, unsigned o, int k,
                                          AdvLevel &L) {
  const int nk = P.nk;
  const int px = P.px;
  const size_t kb = (size_t)k * P.pxy;
  const float *s = a.s + kb;
  L.xm3 = ldo(s - 3, o); L.xm2 = ldo(s - 2, o); L.xm1 = ldo(s - 1, o);
  L.xp1 = ldo(s + 1, o); L.xp2 = ldo(s + 2, o); L.xp3 = ldo(s + 3, o);
  L.ym3 = ldo(s - 3 * px, o); L.ym2 = ldo(s - 2 * px, o); L.ym1 = ldo(s - px, o);
  L.yp1 = ldo(s + px, o); L.yp2 = ldo(s + 2 * px, o); L.yp3 = ldo(s + 3 * px, o);
  L.ru0 = ldo(a.rru + kb, o); L.ru1 = ldo(a.rru + kb + 1, o);
  L.rv0 = ldo(a.rrv + kb, o); L.rv1 = ldo(a.rrv + kb + px, o);
  // (unscaled, pdefz takes the top face as it is given)
  L.rw1 = (k < nk || (PD && !a.scale)) ? ldo(a.rrw + kb + P.pxy, o) : 0.0f;
  if (a.scale) {
    const float r0 = P.rho0[k];
    L.ru0 = L.ru0 * r0; L.ru1 = L.ru1 * r0;
    L.rv0 = L.rv0 * r0; L.rv1 = L.rv1 * r0;
    if (k < nk) L.rw1 = L.rw1 * P.rf0[k + 1];
  }
  L.wnew = (k + 4 <= nk) ? ldo(s + 4 * (size_t)P.pxy, o) : 0.0f;
  L.dv = ldo(a.divx + kb, o);
  L.st0 = ldo(a.sten0 + kb, o);
  L.sv0 = ldo(a.s0 + kb, o);
  L.t11v = TH ? ldo(a.t11 + kb, o) : 0.0f;
  L.thtv = TH ? ldo(a.thterm + kb, o) : 0.0f;
}

// One column (i,j) of advs (src/adv.F:14-658 with hadv_flx5/vadv_flx5, or
// hadv_weno5/vadv_weno5 when WENO): face fluxes at i, i+1, j, j+1 with the
// open-boundary inflow fixes (src/adv.F:211-340), the vertical fluxes
// marched up the column with a six-level register window, and the tendency
// assembly.  Each flux is the same FP32 expression as the reference's, so
// results are bitwise equal to separate flux / divergence passes.  The
// operands of level k+1 are loaded before level k is evaluated and stored.
// The uniform switches are compile-time: SADD (theta's offset form), TH
// (theta's t11*thterm term), PD (positive definite: advx/advy/advz and the
// marks are written as well, for pdef_fix).
template <bool WENO, bool SADD, bool TH, bool PD>
__device__ __forceinline__ void advs_col(const KP &P, const AdvsArgs &a, const ColGrid &cg, int bx) {
  int i, j, ks, ke;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  if (!col_tile_seg(cg, bx, nk, i, j, ks, ke)) return;
  if (i > ni || j > nj) return;
  const bool doitw = (P.wbc == 2 && P.ibw == 1), doite = (P.ebc == 2 && P.ibe == 1);
  const bool doits = (P.sbc == 2 && P.ibs == 1), doitn = (P.nbc == 2 && P.ibn == 1);
  constexpr bool sadd = SADD;
  const float th0r = P.K.th0r;
  const unsigned o = 4u * (unsigned)IX2D(P, i, j);
  auto val = [&](int kk) -> float {  // column value at level kk (1..nk)
    if (kk < 1 || kk > nk) return 0.0f;
    const float v = ldo(a.s + (size_t)kk * P.pxy, o);
    return sadd ? (P.th0[kk] - th0r) + v : v;
  };
  // window: wv[0..5] = S(k-2 .. k+3)
  float wv0 = val(ks - 2), wv1 = val(ks - 1), wv2 = val(ks), wv3 = val(ks + 1), wv4 = val(ks + 2), wv5 = val(ks + 3);
  AdvLevel nx;
  advs_load<PD, TH>(P, a, o, ks, nx);
  float fz_lo = 0.0f, rw0 = 0.0f;
  if (PD && ks == 1 && !a.scale) rw0 = ldo(a.rrw + P.pxy, o);
  if (ks > 1) {
    // the flux through a segment's lowest face
    float rw = ldo(a.rrw + (size_t)ks * P.pxy, o);
    if (a.scale) rw = rw * P.rf0[ks];
    if (PD) rw0 = rw;
    const float wm = val(ks - 3);
    auto S = [=](int kk) -> float {
      const int q = kk - ks;  // -3..2
      return q == -3 ? wm : q == -2 ? wv0 : q == -1 ? wv1 : q == 0 ? wv2 : q == 1 ? wv3 : wv4;
    };
    fz_lo = WENO ? vfluxw_of(P, 1, rw, S, ks, a.pdefweno, a.weps) : vflux5_of(P, 1, rw, S, ks);
  }
  for (int k = ks; k <= ke; k++) {
    const AdvLevel L = nx;
    if (k < ke) advs_load<PD, TH>(P, a, o, k + 1, nx);
    const size_t kb = (size_t)k * P.pxy;
    const float tem = sadd ? (P.th0[k] - th0r) : 0.0f;
    auto H = [=](float v) -> float { return sadd ? tem + v : v; };
    const float sc = wv2;
    // x faces i and i+1
    const float xm3 = H(L.xm3), xm2 = H(L.xm2), xm1 = H(L.xm1), xp1 = H(L.xp1), xp2 = H(L.xp2),
                xp3 = H(L.xp3);
    const float ru0 = L.ru0, ru1 = L.ru1;
    float fx0 = hface5<WENO>(ru0, xm3, xm2, xm1, sc, xp1, xp2, a.pdef, a.weps);
    float fx1 = hface5<WENO>(ru1, xm2, xm1, sc, xp1, xp2, xp3, a.pdef, a.weps);
    const float fx0_raw = fx0;
    if (doitw && i == 1 && ru0 >= 0.0f) fx0 = fx1;
    if (doite && i == ni && ru1 <= 0.0f) fx1 = fx0_raw;
    // y faces j and j+1
    const float ym3 = H(L.ym3), ym2 = H(L.ym2), ym1 = H(L.ym1), yp1 = H(L.yp1), yp2 = H(L.yp2),
                yp3 = H(L.yp3);
    const float rv0 = L.rv0, rv1 = L.rv1;
    float fy0 = hface5<WENO>(rv0, ym3, ym2, ym1, sc, yp1, yp2, a.pdef, a.weps);
    float fy1 = hface5<WENO>(rv1, ym2, ym1, sc, yp1, yp2, yp3, a.pdef, a.weps);
    const float fy0_raw = fy0;
    if (doits && j == 1 && rv0 >= 0.0f) fy0 = fy1;
    if (doitn && j == nj && rv1 <= 0.0f) fy1 = fy0_raw;
    // (uh, vh are 1)
    float ax = -(fx1 - fx0) * P.rdx;
    float ay = -(fy1 - fy0) * P.rdy;
    if (doitw && i == 1 && ru0 >= 0.0f) ax = ax - sc * (ru1 - ru0) * P.rdx;
    if (doite && i == ni && ru1 <= 0.0f) ax = ax - sc * (ru1 - ru0) * P.rdx;
    if (doits && j == 1 && rv0 >= 0.0f) ay = ay - sc * (rv1 - rv0) * P.rdy;
    if (doitn && j == nj && rv1 <= 0.0f) ay = ay - sc * (rv1 - rv0) * P.rdy;
    // vertical face k+1 from S(k-2..k+3)
    float fz_hi = 0.0f;
    if (k + 1 <= nk) {
      const int kf = k + 1;
      auto S = [=](int kk) -> float {
        const int o = kk - kf;  // -3..2
        return o == -3 ? wv0 : o == -2 ? wv1 : o == -1 ? wv2 : o == 0 ? wv3 : o == 1 ? wv4 : wv5;
      };
      fz_hi = WENO ? vfluxw_of(P, 1, L.rw1, S, kf, a.pdefweno, a.weps)
                   : vflux5_of(P, 1, L.rw1, S, kf);
    }
    float az;
    if (k == 1) az = -fz_hi * P.rdz * P.mh[1];
    else if (k == nk) az = +fz_lo * P.rdz * P.mh[nk];
    else az = -(fz_hi - fz_lo) * P.rdz * P.mh[k];
    if (PD) {
      sto(a.advx + kb, o, ax);
      sto(a.advy + kb, o, ay);
      sto(a.advz + kb, o, az);
      // pdef_dum of the three directions from what the column holds
      const float r0s0 = P.rho0[k] * L.sv0;
      float dx = r0s0 + a.dt * (ax + sc * (ru1 - ru0) * P.rdx);
      float dy = r0s0 + a.dt * (ay + sc * (rv1 - rv0) * P.rdy);
      const float dz = r0s0 + a.dt * (az + sc * (L.rw1 - rw0) * P.rdz * P.mh[k]);
      if ((doitw && i == 1 && ru0 >= 0.0f) || (doite && i == ni && ru1 <= 0.0f)) dx = r0s0;
      if ((doits && j == 1 && rv0 >= 0.0f) || (doitn && j == nj && rv1 <= 0.0f)) dy = r0s0;
      const unsigned long long neg = __ballot(dx < 0.0f || dy < 0.0f || dz < 0.0f);
      if ((threadIdx.x & 63) == 0) a.marks[((size_t)(k - 1) * nj + (j - 1)) * a.gx + ((i - 1) >> 6)] = neg;
      rw0 = L.rw1;
    }
    float st = L.st0;
    if (TH) st = st - L.t11v * L.thtv;
    st = st + ((ax + ay) + az + sc * L.dv) * P.rr0[k];
    if (a.out_sten) sto(a.out_sten + kb, o, st);
    if (a.out_new) {
      float v = L.sv0 + a.dt * st;
      if (a.smeps_flush && fabsf(v) < P.K.smeps) v = 0.0f;
      sto(a.out_new + kb, o, v);
    }
    fz_lo = fz_hi;
    wv0 = wv1;
    wv1 = wv2;
    wv2 = wv3;
    wv3 = wv4;
    wv4 = wv5;
    wv5 = (k + 4 <= nk) ? (sadd ? (P.th0[k + 4] - th0r) + L.wnew : L.wnew) : 0.0f;
  }
}

// ------------------------------------------------------------------ advs
// sadd: when nonzero, s(i,j,k) = (th0(k) - th0r) + s_in(i,j,k) is formed on
// the fly (the theta equation's sadv, src/solve2.F:1354-1374).
// sten0/thterm_div: initial tendency; with thterm_div != nullptr the
// initial tendency is thten1 - t11*thterm (src/solve2.F:1320-1330), where
// sten0 = thten1, thterm_div[0] = t11 and thterm_div[1] = thterm.
// out_new, if given, receives s0 + dt*tendency with the smeps flush
// (src/solve2.F:1416-1426, :1518-1528).
template <bool WENO, bool SADD, bool TH, bool PD>
static void advs_launch(cm1g_model *m, const KP &P, const AdvsArgs &a, const ColGrid &cg) {
  // (the WENO form with marks takes 97 registers uncapped, four wavefronts a
  // SIMD; five: 578 -> 522 us at 512 x 512 x 128.  Six for the other: no gain)
  launch<256, PD && WENO ? 5 : 0>(m, col_blocks(cg), col_threads(cg),
                                  [=] __device__(int bx, int, int) { advs_col<WENO, SADD, TH, PD>(P, a, cg, bx); });
}

void advs_run(cm1g_model *m, int nrk, const float *s_in, float sadd, const float *s0,
              const float *sten0, const float *thterm_div, float *out_sten, float *out_new,
              int pdef, int pdefweno, float dt, double weps, int smeps_flush) {
  const KP P = m->P;
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  // WENO5 on every stage (advwenos=1) or the last one (2), src/adv.F:75-78
  const bool weno = (m->c.advwenos == 1) || (m->c.advwenos == 2 && nrk == 3);
  AdvsArgs g;
  g.s = s_in;
  g.sadd = sadd;
  g.s0 = s0;
  g.sten0 = sten0;
  g.t11 = thterm_div;
  g.thterm = thterm_div ? m->f[CM1G_THTERM] : nullptr;
  g.rru = m->f[CM1G_RRU];
  g.rrv = m->f[CM1G_RRV];
  g.rrw = m->f[CM1G_RRW];
  g.scale = m->advs_unscaled ? 0 : 1;
  g.divx = m->f[CM1G_DIVX];
  g.out_sten = out_sten;
  g.out_new = out_new;
  g.advx = m->tx;
  g.advy = m->ty;
  g.advz = m->tz;
  g.dt = dt;
  g.smeps_flush = smeps_flush;
  g.pdef = pdef;
  g.pdefweno = pdefweno;
  g.weps = weps;
  // compile-time variants: theta (offset form, with or without the t11
  // term), any other scalar in the plain or the positive-definite pass
  const bool sadd_on = (sadd != 0.0f), th_on = (thterm_div != nullptr);
  using Launcher = void (*)(cm1g_model *, const KP &, const AdvsArgs &, const ColGrid &);
  auto pick = [&](bool pd) -> Launcher {
    if (sadd_on && th_on && !pd) return weno ? advs_launch<true, true, true, false> : advs_launch<false, true, true, false>;
    if (sadd_on && !th_on && !pd) return weno ? advs_launch<true, true, false, false> : advs_launch<false, true, false, false>;
    if (!sadd_on && !th_on && !pd) return weno ? advs_launch<true, false, false, false> : advs_launch<false, false, false, false>;
    if (!sadd_on && th_on && !pd) return weno ? advs_launch<true, false, true, false> : advs_launch<false, false, true, false>;
    return weno ? advs_launch<true, false, false, true> : advs_launch<false, false, false, true>;
  };
  ColGrid cg = col_grid(ni, nj, m->tile_rows);
  col_split(m, cg, nk);
  // an in-place update (out_new aliasing the advected field) writes a
  // partner array, since neighbouring columns still read the old values;
  // the field and its partner then exchange buffers
  const bool inplace = (out_new != nullptr && out_new == s_in);
  if (inplace) g.out_new = m->thb;
  if (pdef != 1) {
    pick(false)(m, P, g, cg);
  } else {
    // the positive-definite pass reads the advected values themselves
    // (never the theta offset form: pdef is for moisture and tracers)
    if (sadd != 0.0f || th_on) {
      cm1g_set_error("advs: pdef with an offset field is not supported");
      return;
    }
    // a tendency asked for may be the array its initial value stands in, which
    // pdef_fix reads again: it is formed in a work array
    float *const ten = g.out_sten;
    if (ten) g.out_sten = m->sy;
    g.marks = (unsigned long long *)m->sx;
    g.gx = cg.gx;
    pick(true)(m, P, g, cg);
    PdefArgs pa;
    pa.rru = g.rru;
    pa.rrv = g.rrv;
    pa.rrw = g.rrw;
    pa.scale = g.scale;
    pa.advx = m->tx;
    pa.advy = m->ty;
    pa.advz = m->tz;
    pa.s0 = s0;
    pa.s = s_in;
    pa.sten0 = sten0;
    pa.divx = g.divx;
    pa.marks = g.marks;
    pa.gx = g.gx;
    pa.out_sten = g.out_sten;
    pa.out_new = g.out_new;
    pa.dt = dt;
    pa.smeps_flush = smeps_flush;
    // levels a workgroup: visited levels follow one another (two barriers and
    // their loads' latency each), so a small grid takes fewer of them, down
    // to one, until there are 4096 workgroups (eight levels against these: 64 x
    // 64 x 40 25.6 -> 8.5 us; 301 x 227 x 63 37 -> 29 us, at 2048 37).
    const long rows = m->plan_tiles > 0 ? m->plan_tiles : (long)cg.gx * cg.gy * cg.ty;
    const long lev = rows / 4 * nk / 4096;
    pa.lev = (int)(lev < 1 ? 1 : lev > PDEF_L ? PDEF_L : lev);
    launch<256>(m, dim3((ni + 63) / 64, (nj + 3) / 4, (nk + pa.lev - 1) / pa.lev), dim3(64, 4, 1),
                [=] __device__(int bx, int by, int bz) { pdef_fix(P, pa, bx, by, bz); });
    if (ten) {
      const float *w = m->sy;
      for3(m, 1, ni, 1, nj, 1, nk, [=] __device__(int i, int j, int k) {
        const int c = IXD(P, i, j, k);
        ten[c] = w[c];
      });
    }
  }
  if (inplace) {
    // the partner now holds the new field: exchange the two buffers
    for (int id = 0; id < CM1G_NFIELDS; id++)
      if (m->f[id] == out_new) {
        m->f[id] = m->thb;
        m->thb = out_new;
        break;
      }
  }
}

// ----------------------------------------------------------- advu/v/w
// The momentum tendencies use the pre-acoustic mass fluxes rru/rrv/rrw
// (model fields) and divx; uten/vten/wten are updated in place, or, with
// from_ten1, set to uten1/vten1/wten1 plus advection (column kernels in
// cm1g_advm.hip).
void adv_uvw(cm1g_model *m, int nrk, int mask, int buoy, int from_ten1, int own, const float *const *src3) {
  advm_run(m, nrk, mask, buoy, from_ten1, own, src3);
}
