// Boundary / halo fills on the device (single GPU: periodic and open
// boundaries become on-device copies instead of comm.F MPI exchanges).
// Semantics follow src/bc.F (non-MPI build): bcs :180-364, bcp :372-520,
// bcu :528-714, bcv :722-934, bcw :942-1143.  The reference fills two sides
// of an array, then the other two over the columns the first pass filled, so
// a halo point ends up with the value of one interior point, corners
// included: its i and j each wrapped (periodic) or clamped (open).  Every
// halo point is written from that interior point directly, in one pass.  (An
// open second side covers the first's fill one point deep only: the outer
// corner points then keep, as in the reference, what the first pass copied
// from the halo before the second wrote it; the thread that writes the source
// point makes that copy first.)  One launch fills any list of arrays of any
// kind: the two passes per kind
// and array were 40 of the 117 launches of a supercell step, 4.7 us each
// whatever the grid (190 of 960 us at 64 x 64 x 40).
#include "cm1g_internal.h"

struct BcArrs {
  float *a[BC_MAX];
  signed char kind[BC_MAX];
  signed char top[BC_MAX];  // arrays with BC_W1's zero levels k = 1 and nk+1
  int n;
};

// Halo point number q of one level of one array: the three columns on either
// side of every row (8 slots a row, so a wavefront covers 8 rows), then the
// three rows on either side of the interior columns.
__device__ __forceinline__ void bc_point(const KP &P, int kind, float *a, int q, int k) {
  const int ni = P.ni, nj = P.nj;
  const int nx = (kind == BC_U) ? ni + 1 : ni, ny = (kind == BC_V) ? nj + 1 : nj;
  const int d = (kind == BC_P) ? 1 : 3;
  int i, j;
  if (q < 8 * (nj + 7)) {
    const int c = q & 7;
    j = (q >> 3) - 2;
    if (c >= 6) return;
    i = (c < 3) ? c - 2 : nx + c - 2;
  } else {
    q -= 8 * (nj + 7);
    const int r = q / (ni + 1);
    i = 1 + q - r * (ni + 1);
    if (i > nx || r >= 6) return;
    j = (r < 3) ? r - 2 : ny + r - 2;
  }
  if (i < 1 - d || i > nx + d || j < 1 - d || j > ny + d) return;
  const bool ih = i < 1 || i > nx, jh = j < 1 || j > ny;
  const bool second_open = (kind == BC_V) ? P.wbc != 1 : P.sbc != 1;
  if (kind != BC_P && second_open && jh && (kind != BC_V || ih)) {
    if (kind == BC_V) {
      if (j < 0 || j > ny + 1) return;
    } else if (ih) {
      if (i < 0 || i > nx + 1) return;
    } else {
      // what the first pass copied from here before this pass writes it
      const float old = a[IXD(P, i, j, k)];
      if (P.wbc == 1) {
        if (i - ni == -2 || i - ni == -1) a[IXD(P, i - ni, j, k)] = old;
        if (i + ni == nx + 2 || i + ni == nx + 3) a[IXD(P, i + ni, j, k)] = old;
      } else if (j == 0 || j == ny + 1) {
        if (i == 1) a[IXD(P, -2, j, k)] = a[IXD(P, -1, j, k)] = old;
        if (i == nx) a[IXD(P, nx + 2, j, k)] = a[IXD(P, nx + 3, j, k)] = old;
      }
    }
  } else if (kind == BC_V && second_open && ih) {
    const float old = a[IXD(P, i, j, k)];
    if (P.sbc == 1) {
      if (j - nj == -2 || j - nj == -1) a[IXD(P, i, j - nj, k)] = old;
      if (j + nj == ny + 2 || j + nj == ny + 3) a[IXD(P, i, j + nj, k)] = old;
    } else if (i == 0 || i == nx + 1) {
      if (j == 1) a[IXD(P, i, -2, k)] = a[IXD(P, i, -1, k)] = old;
      if (j == ny) a[IXD(P, i, ny + 2, k)] = a[IXD(P, i, ny + 3, k)] = old;
    }
  }
  const int si = (i < 1) ? (P.wbc == 1 ? i + ni : 1) : (i > nx) ? (P.ebc == 1 ? i - ni : nx) : i;
  const int sj = (j < 1) ? (P.sbc == 1 ? j + nj : 1) : (j > ny) ? (P.nbc == 1 ? j - nj : ny) : j;
  if (si == i && sj == j) return;
  a[IXD(P, i, j, k)] = a[IXD(P, si, sj, k)];
}

__device__ __forceinline__ void bc_run(const KP &P, const BcArrs &A, int nbx, int bx, int by, int bz) {
  if (bz < A.n) {
    const int kind = A.kind[bz], k = 1 + by;
    if ((kind == BC_W1 || kind == BC_W0) && k < 2) return;
    bc_point(P, kind, A.a[bz], bx * 256 + (int)threadIdx.x, k);
    return;
  }
  // bcw, flag=1: zero at the top and bottom
  float *a = A.a[A.top[bz - A.n]];
  const int w = P.ni + 2, np = w * (P.nj + 2);
  for (int t = (by * nbx + bx) * 256 + (int)threadIdx.x; t < np; t += P.nk * nbx * 256) {
    const int j = t / w, i = t - j * w;
    a[IXD(P, i, j, 1)] = 0.0f;
    a[IXD(P, i, j, P.nk + 1)] = 0.0f;
  }
}

void bc_fill_list(cm1g_model *m, const BcItem *it, int n) {
  const KP P = m->P;
  BcArrs A;
  memset(&A, 0, sizeof(A));
  int ntop = 0;
  for (int q = 0; q < n; q++) {
    A.a[q] = it[q].a;
    A.kind[q] = (signed char)it[q].kind;
    if (it[q].kind == BC_W1) A.top[ntop++] = (signed char)q;
  }
  A.n = n;
  const int nbx = (8 * (P.nj + 7) + 6 * (P.ni + 1) + 255) / 256;
  launch<256>(m, dim3(nbx, P.nk, n + ntop), dim3(256),
              [=] __device__(int bx, int by, int bz) { bc_run(P, A, nbx, bx, by, bz); });
}

void bc_fill_n(cm1g_model *m, int kind, float *const *arrs, int n) {
  BcItem it[BC_MAX];
  for (int q = 0; q < n; q++) it[q] = BcItem{arrs[q], kind};
  bc_fill_list(m, it, n);
}

void bc_fill(cm1g_model *m, int kind, float *a) { bc_fill_n(m, kind, &a, 1); }

// radbcew4 / radbcns4 (src/bc.F:2054-2172): per boundary column, the
// vertical mean of the clipped phase speed, stored at every level.  A
// workgroup takes 64 columns of one side: its 8 wavefronts evaluate the
// levels' speeds (a division each) side by side, 64 levels at a time, and the
// first adds them in the reference's order.  One thread per column added them
// as it went, a level's loads after the other: 19 us a stage at 64 x 64 x 40
// and 73 us at 1024 x 1024 x 96, now 9 and 42.
constexpr int RAD_LEV = 64;

__device__ __forceinline__ void radbc_cols(const KP &P, const float *u1, const float *u2, const float *v1,
                                           const float *v2, float dt, float csmax, float *radbcw,
                                           float *radbce, float *radbcs, float *radbcn, int bx, int by) {
  __shared__ float term[RAD_LEV][64];
  __shared__ float mean[64];
  const int ni = P.ni, nj = P.nj, nk = P.nk;
  const int side = by, lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6;
  const bool we = side < 2;
  const int n = we ? nj : ni;
  // the side's condition and first column are the same for the workgroup
  const bool mine = (side == 0) ? (P.ibw == 1 && P.wbc == 2) : (side == 1) ? (P.ibe == 1 && P.ebc == 2)
                  : (side == 2) ? (P.ibs == 1 && P.sbc == 2) : (P.ibn == 1 && P.nbc == 2);
  if (!mine || bx * 64 >= n) return;
  const int t = 1 + bx * 64 + lane;
  const bool on = t <= n;
  const int tc = on ? t : n;
  // the face whose change gives the speed, and the one inside (outside) of it
  const int c0 = (side == 0) ? IXD(P, 2, tc, 0) : (side == 1) ? IXD(P, ni, tc, 0)
               : (side == 2) ? IXD(P, tc, 2, 0) : IXD(P, tc, nj, 0);
  const int step = we ? 1 : P.px;
  const bool low = (side == 0 || side == 2);
  const float *a1 = we ? u1 : v1, *a2 = we ? u2 : v2;
  const float dxy = we ? P.dx * (1.0f / P.uf[(side == 0 ? 2 : ni) + 2]) : P.dy * (1.0f / P.vf[(side == 2 ? 2 : nj) + 2]);
  float avg = 0.0f;
  for (int kb = 1; kb <= nk; kb += RAD_LEV) {
    const int ke = min(nk, kb + RAD_LEV - 1);
    for (int k = kb + wv; k <= ke; k += 8) {
      const int c = c0 + k * P.pxy;
      const float foo = low ? a1[c + step] - a1[c] : a1[c] - a1[c - step];
      const float s = dxy * (a1[c] - a2[c]) / (dt * (copysignf(1.e-10f, foo) + foo));
      term[k - kb][lane] = low ? fmaxf(fminf(s, 0.0f), -csmax) : fminf(fmaxf(s, 0.0f), csmax);
    }
    __syncthreads();
    if (wv == 0)
      for (int q = 0; q <= ke - kb; q++) avg = avg + term[q][lane];
    __syncthreads();
  }
  if (wv == 0) mean[lane] = avg / (float)nk;
  __syncthreads();
  if (!on) return;
  const float r = mean[lane];
  float *out = (side == 0) ? radbcw : (side == 1) ? radbce : (side == 2) ? radbcs : radbcn;
  const int pitch = we ? P.py : P.px;
  for (int k = 1 + wv; k <= nk; k += 8) out[(t + 2) + k * pitch] = r;
}

void radbc4(cm1g_model *m, const float *ua, const float *u3d, const float *va, const float *v3d,
            float dt) {
  const KP P = m->P;
  const int n = (P.ni > P.nj ? P.ni : P.nj);
  const float csmax = m->c.csmax;
  float *rw = m->d2[CM1G_D_RADBCW], *re = m->d2[CM1G_D_RADBCE], *rs = m->d2[CM1G_D_RADBCS],
        *rn = m->d2[CM1G_D_RADBCN];
  launch<512>(m, dim3((n + 63) / 64, 4), dim3(512), [=] __device__(int bx, int by, int) {
    radbc_cols(P, ua, u3d, va, v3d, dt, csmax, rw, re, rs, rn, bx, by);
  });
}
