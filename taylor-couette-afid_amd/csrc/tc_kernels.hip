// MI355X (gfx950) kernels for the stencil, Helmholtz and reduction parts of
// the Taylor-Couette RK3 step.  FP64 throughout, wave64.
//
// Device layout: every 3-D field is [r][z][theta] with theta contiguous,
// r-plane k (1-based, k = 1..nr) at offset (k-1)*P, P = nzm*nthm.  The
// reference's periodic halos (InitVariables.F90:26-35, halo_common.f90:67-108)
// become index wrap-around, so no halo update is ever launched.
#include <algorithm>
#include <map>
#include <mutex>

#include "tc_internal.h"

namespace tc {

#define DEVI __device__ __forceinline__

DEVI long long IX(const GridDev &g, int k, int j, int i) {
  return (long long)(k - 1) * g.P + (long long)j * g.nthm + i;
}
DEVI int wrap_p(int i, int n) { return (i + 1 == n) ? 0 : i + 1; }
DEVI int wrap_m(int i, int n) { return (i == 0) ? n - 1 : i - 1; }

// Non-temporal access for arrays streamed once per kernel (no other block
// re-reads them soon): a streaming copy runs 5.8% faster with both.
DEVI double ld_nt(const double *p) { return __builtin_nontemporal_load(p); }
DEVI void st_nt(double *p, double v) { __builtin_nontemporal_store(v, p); }
typedef double d2v __attribute__((ext_vector_type(2)));
DEVI double2 ld2_nt(const double *p) {
  const d2v v = __builtin_nontemporal_load(reinterpret_cast<const d2v *>(p));
  return make_double2(v.x, v.y);
}
DEVI void st2_nt(double *p, double u, double v) {
  const d2v w = {u, v};
  __builtin_nontemporal_store(w, reinterpret_cast<d2v *>(p));
}

// ---------------------------------------------------------------------------
// Explicit terms.  Written once, generic over an accessor A with
// A(dk, dj, di) = field value at (k+dk, j+dj, i+di) of the point being
// computed, so the routine-level kernels (global loads) and the fused
// Helmholtz kernel (LDS tiles) evaluate identical arithmetic.
// ---------------------------------------------------------------------------

// Global-memory accessor with periodic wrap in z and theta.
struct GAcc {
  const double *__restrict__ a;
  long long base;  // IX(k, j, i)
  long long P;
  int i, j, nthm, nzm;
  DEVI double operator()(int dk, int dj, int di) const {
    int jj = j + dj, ii = i + di;
    jj = (jj < 0) ? jj + nzm : (jj >= nzm ? jj - nzm : jj);
    ii = (ii < 0) ? ii + nthm : (ii >= nthm ? ii - nthm : ii);
    return a[base + dk * P + (long long)(jj - j) * nthm + (ii - i)];
  }
};
DEVI GAcc gacc(const GridDev &g, const double *a, int k, int j, int i) {
  GAcc r;
  r.a = a;
  r.base = IX(g, k, j, i);
  r.P = g.P;
  r.i = i;
  r.j = j;
  r.nthm = g.nthm;
  r.nzm = g.nzm;
  return r;
}

// ExplicitTermsQT.F90:44-125 at (kc, j, i)
template <class A>
DEVI double explicit_qt_g(const GridDev &g, const HelmPlane &c, const A &T, const A &R,
                          const A &Z, int kc) {
  const int dkm = kc > 1 ? -1 : 0, dkp = kc < g.nrm ? 1 : 0;  // kmv, kpv clamps
  const double udxt = c.udxt_m;
  const double udxtq = c.udxtq_m;
  const double udxzq = c.udxzq;
  const double udxz = g.dxz * 0.25;
  const double t_c = T(0, 0, 0), t_ip = T(0, 0, 1), t_im = T(0, 0, -1);
  const double t_jp = T(0, 1, 0), t_jm = T(0, -1, 0);
  const double t_kp = T(dkp, 0, 0), t_km = T(dkm, 0, 0);
  const double r_c = R(0, 0, 0), r_im = R(0, 0, -1);
  const double r_kp = R(1, 0, 0), r_kpim = R(1, 0, -1);
  const double z_c = Z(0, 0, 0), z_im = Z(0, 0, -1);
  const double z_jp = Z(0, 1, 0), z_jpim = Z(0, 1, -1);
  const double usrc_kp = c.usrc_p, usrc_k = c.usrc;

  const double h11 = ((t_ip + t_c) * (t_ip + t_c) - (t_c + t_im) * (t_c + t_im)) * udxt;
  const double h12d = ((r_kp + r_kpim) * (t_kp + t_c) - (r_c + r_im) * (t_c + t_km)) * 0.25 * c.udx2rm;
  const double h12n = t_c * c.usrm * ((r_kp + r_kpim) * usrc_kp + (r_c + r_im) * usrc_k) * 0.25;
  const double h12 = h12d + h12n;
  const double h13 = ((z_jp + z_jpim) * (t_jp + t_c) - (z_c + z_im) * (t_c + t_jm)) * udxz;
  const double d11qt = (t_ip - 2.0 * t_c + t_im) * udxtq;
  const double d22qt = (t_jp - 2.0 * t_c + t_jm) * udxzq;
  const double qre = r_kp * usrc_kp + r_c * usrc_k;
  const double qrw = r_kpim * usrc_kp + r_im * usrc_k;
  const double d11qre = (qre - qrw) * c.udx1vis1 * 0.5;
  const double coriol = -((r_c + r_im) * usrc_k + (r_kp + r_kpim) * usrc_kp) * 0.25 * g.romeg;
  return -(h11 + h12 + h13) + d11qre + d22qt + d11qt + coriol;
}

// ExplicitTermsQR.F90:46-146 at (kc, j, i), kc = 2..nrm
template <class A>
DEVI double explicit_qr_g(const GridDev &g, const HelmPlane &c, const A &T, const A &R,
                          const A &Z, int kc) {
  const double udxt = c.udxt_c;
  const double udxtq = c.udxtq_c;
  const double udxzq = c.udxzq;
  const double udxz = g.dxz * 0.25;
  const double t_c = T(0, 0, 0), t_ip = T(0, 0, 1);
  const double t_m = T(-1, 0, 0), t_mip = T(-1, 0, 1);
  const double r_c = R(0, 0, 0), r_ip = R(0, 0, 1), r_im = R(0, 0, -1);
  const double r_jp = R(0, 1, 0), r_jm = R(0, -1, 0);
  const double r_kp = R(1, 0, 0), r_km = R(-1, 0, 0);
  const double z_c = Z(0, 0, 0), z_jp = Z(0, 1, 0);
  const double z_m = Z(-1, 0, 0), z_mjp = Z(-1, 1, 0);

  const double tavg = (t_ip + t_mip + t_c + t_m) * 0.25;
  const double h11n = tavg * tavg;
  const double h21 = ((t_ip + t_mip) * (r_ip + r_c) - (t_c + t_m) * (r_c + r_im)) * udxt;
  const double h22 = ((r_kp * c.usrc_p + r_c * c.usrc) * (r_kp + r_c) -
                      (r_c * c.usrc + r_km * c.usrc_m) * (r_c + r_km)) *
                     c.udx2c * 0.25;
  const double h23 = ((z_jp + z_mjp) * (r_jp + r_c) - (z_c + z_m) * (r_c + r_jm)) * udxz;
  const double qte = (t_ip + t_mip);
  const double qtw = (t_c + t_m);
  const double d11qre = -(qte - qtw) * c.udx1vis2;
  const double d11qr = (r_ip - 2.0 * r_c + r_im) * udxtq;
  const double d22qr = (r_jp - 2.0 * r_c + r_jm) * udxzq;
  const double coriol = (t_c + t_ip + t_m + t_mip) * 0.25 * c.rc * g.romeg;
  return -(h21 + h22 + h23) + h11n + d11qr + d22qr + d11qre + coriol;
}

// ExplicitTermsQZ.F90:40-102 at (kc, j, i)
template <class A>
DEVI double explicit_qz_g(const GridDev &g, const HelmPlane &c, const A &T, const A &R,
                          const A &Z, int kc) {
  const int dkm = kc > 1 ? -1 : 0, dkp = kc < g.nrm ? 1 : 0;
  const double udxt = c.udxt_m;
  const double udxtq = c.udxtq_m;
  const double udxzq = c.udxzq;
  const double udxz = g.dxz * 0.25;
  const double t_c = T(0, 0, 0), t_ip = T(0, 0, 1);
  const double t_jm = T(0, -1, 0), t_jmip = T(0, -1, 1);
  const double r_c = R(0, 0, 0), r_jm = R(0, -1, 0);
  const double r_kp = R(1, 0, 0), r_kpjm = R(1, -1, 0);
  const double z_c = Z(0, 0, 0), z_ip = Z(0, 0, 1), z_im = Z(0, 0, -1);
  const double z_jp = Z(0, 1, 0), z_jm = Z(0, -1, 0);
  const double z_kp = Z(dkp, 0, 0), z_km = Z(dkm, 0, 0);

  const double h31 = ((t_ip + t_jmip) * (z_ip + z_c) - (t_c + t_jm) * (z_c + z_im)) * udxt;
  const double h32 = (((r_kp + r_kpjm) * (z_kp + z_c)) - ((r_c + r_jm) * (z_c + z_km))) * c.udx2rm * 0.25;
  const double h33 = ((z_jp + z_c) * (z_jp + z_c) - (z_c + z_jm) * (z_c + z_jm)) * udxz;
  const double dqz1 = (z_im - 2.0 * z_c + z_ip) * udxtq;
  const double dqz2 = (z_jm - 2.0 * z_c + z_jp) * udxzq;
  return -(h31 + h32 + h33) + dqz1 + dqz2;
}

template <int WHICH, class A>
DEVI double explicit_g(const GridDev &g, const HelmPlane &c, const A &T, const A &R, const A &Z, int kc) {
  if constexpr (WHICH == 0) return explicit_qt_g(g, c, T, R, Z, kc);
  else if constexpr (WHICH == 1) return explicit_qr_g(g, c, T, R, Z, kc);
  else return explicit_qz_g(g, c, T, R, Z, kc);
}

template <int WHICH>
__global__ __launch_bounds__(256) void k_explicit(GridDev g, const double *__restrict__ qt,
                                                  const double *__restrict__ qr,
                                                  const double *__restrict__ qz,
                                                  double *__restrict__ out) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.nthm || j >= g.nzm) return;
  const int kc = blockIdx.z + (WHICH == 1 ? 2 : 1);
  const GAcc T = gacc(g, qt, kc, j, i), R = gacc(g, qr, kc, j, i), Z = gacc(g, qz, kc, j, i);
  const HelmPlane c = g.hp[kc];
  out[IX(g, kc, j, i)] = explicit_g<WHICH>(g, c, T, R, Z, kc);
}

// Point U (0, 1) of a theta pair (i, i+1), i even: the pair itself is one
// 16-byte load, which the two points share, as they do the outer neighbours.
template <int U>
struct PairAcc {
  const double *__restrict__ a;
  long long base, P;  // IX(k, j, i)
  int jm, jp, im, ip;  // offsets of rows j-1, j+1, of points i-1, i+2
  DEVI double operator()(int dk, int dj, int di) const {
    const double *p = a + (base + dk * P + (dj < 0 ? jm : (dj > 0 ? jp : 0)));
    const int e = U + di;
    if (e < 0) return p[im];
    if (e > 1) return p[ip];
    const double2 v = *reinterpret_cast<const double2 *>(p);
    return e ? v.y : v.x;
  }
};

// Even nthm: a theta pair per thread, pairs of a plane in one row so that no
// lane idles at the end of a theta line.  The 17 loads of 8 bytes a point,
// 16 cycles of the address unit each, bounded the one-point form:
// 256x256x193, q_theta / q_r / q_z 132 / 130 / 131 us, in pairs 92 / 109 / 98
// (4.4 / 3.7 / 4.1 TB/s).  Contiguous planes per XCD gave nothing (92 / 112 /
// 101 us).  Odd nthm, whose rows are not 16-byte aligned, keeps one point.
template <int WHICH>
__global__ __launch_bounds__(256) void k_explicit2(GridDev g, const double *__restrict__ qt,
                                                   const double *__restrict__ qr,
                                                   const double *__restrict__ qz,
                                                   double *__restrict__ out) {
  const int n = g.nthm, h = n / 2, l = blockIdx.x * 256 + threadIdx.x;
  const int j = l / h, i = 2 * (l - j * h);
  if (j >= g.nzm) return;
  const int kc = blockIdx.y + (WHICH == 1 ? 2 : 1);
  const long long base = IX(g, kc, j, i);
  const int jm = (wrap_m(j, g.nzm) - j) * n, jp = (wrap_p(j, g.nzm) - j) * n;
  const int im = wrap_m(i, n) - i, ip = wrap_p(i + 1, n) - i;
  const HelmPlane c = g.hp[kc];
  auto at = [&](auto u, const double *f) {
    return PairAcc<decltype(u)::value>{f, base, g.P, jm, jp, im, ip};
  };
  using U0 = std::integral_constant<int, 0>;
  using U1 = std::integral_constant<int, 1>;
  const double v0 = explicit_g<WHICH>(g, c, at(U0{}, qt), at(U0{}, qr), at(U0{}, qz), kc);
  const double v1 = explicit_g<WHICH>(g, c, at(U1{}, qt), at(U1{}, qr), at(U1{}, qz), kc);
  *reinterpret_cast<double2 *>(out + base) = make_double2(v0, v1);
}

static dim3 point_grid(const tc_ctx *c, int planes) {
  return dim3((unsigned)((c->nthm + 63) / 64), (unsigned)((c->nzm + 3) / 4), (unsigned)planes);
}

template <int WHICH>
static void launch_explicit(tc_ctx *c, const char *name, int out) {
  const int planes = WHICH == 1 ? c->nrm - 1 : c->nrm;
  timer_begin(c, name);
  if (c->nthm % 2 == 0)
    hipLaunchKernelGGL(k_explicit2<WHICH>, dim3((unsigned)((c->P / 2 + 255) / 256), (unsigned)planes),
                       dim3(256), 0, c->stream, c->gd, c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], c->f[out]);
  else
    hipLaunchKernelGGL(k_explicit<WHICH>, point_grid(c, planes), dim3(64, 4), 0, c->stream, c->gd,
                       c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], c->f[out]);
  timer_end(c);
}
void launch_explicit_qt(tc_ctx *c) { launch_explicit<0>(c, "explicit_qt", TC_DQ); }
void launch_explicit_qr(tc_ctx *c) { launch_explicit<1>(c, "explicit_qr", TC_DPH); }
void launch_explicit_qz(tc_ctx *c) { launch_explicit<2>(c, "explicit_qz", TC_QCAP); }

// ---------------------------------------------------------------------------
// Helmholtz solves.  The LU factors (of the row-normalised matrices of
// SolveImpEqnUpdate_*; by dgttrf where it exchanges rows) do not depend on the line
// (j, i) except through the wall masks, so they come from a per-substep
// table with one entry per mask combination.  Lanes run along theta so every
// plane access is coalesced.  The right-hand sides are formed point by point
// in one kernel and written to a scratch field; a second kernel reads them
// back and solves, each line's rows in registers.
// ---------------------------------------------------------------------------

struct LUView {
  const double *b;  // rows of LU_ROW doubles
  DEVI double dl(int r) const { return b[LU_ROW * r]; }
  DEVI double du(int r) const { return b[LU_ROW * r + 1]; }
  DEVI double du2(int r) const { return b[LU_ROW * r + 2]; }
  DEVI double rd(int r) const { return b[LU_ROW * r + 3]; }
  DEVI double pv(int r) const { return b[LU_ROW * r + 4]; }
  DEVI double m(int r) const { return dl(r); }
  DEVI double u(int r) const { return du(r); }
};
DEVI LUView lu_view(const double *base) {
  LUView v;
  v.b = base;
  return v;
}

// streamed L-solve step for row r (0-based): f is the right-hand side of row r+1
DEVI void lsolve_step(const LUView &T, int r, double f, double &carry, double &out) {
  if (T.pv(r) == 0.0) {
    out = carry;
    carry = f - T.dl(r) * carry;
  } else {
    out = f;
    carry = carry - T.dl(r) * f;
  }
}

// Right-hand side row k of the q_theta solve (ImplicitAndUpdateQT.F90:45-115);
// qm, q0, qp = qt(k-1), qt(k), qt(k+1) on the line.
// NOSLIP: every wall mask is 1, so the blends with the free-slip
// coefficients reduce to the no-slip ones (x*1 + y*0 == x for the nonzero
// wall coefficients).
template <bool NOSLIP = false>
DEVI double rhs_qt(const GridDev &g, const HelmPlane &c, const ImpArgs &a, int k, double qm,
                   double q0, double qp, double pr_c, double pr_im, double dqv, double ruold,
                   double fic, double foc) {
  double d33;
  if (k == 1) {
    const double app = c.ap1j;
    const double acc = NOSLIP ? c.ac1j : (c.ac1j * fic + g.ac1j_fs1 * (1 - fic));
    const double amm = NOSLIP ? c.am1j : (c.am1j * fic + g.am1j_fs1 * (1 - fic));
    d33 = qp * app + q0 * acc + a.vwall_in * amm;
  } else if (k < g.nrm) {
    d33 = qp * c.ap1j + q0 * c.ac1j + qm * c.am1j;
  } else {
    const double app = NOSLIP ? c.ap1j : (c.ap1j * foc + g.ap1j_fs2 * (1 - foc));
    const double acc = NOSLIP ? c.ac1j : (c.ac1j * foc + g.ac1j_fs2 * (1 - foc));
    d33 = a.virotext * app + q0 * acc + qm * c.am1j;
  }
  const double dpx = (pr_c - pr_im) * g.dxt * a.al * c.usrm;
  return (a.ga * dqv + a.ro * ruold + a.alre * d33 - dpx) * a.dt;
}

// Right-hand side row k = 2..nrm of the q_r solve (ImplicitAndUpdateQR.F90:41-63).
DEVI double rhs_qr(const HelmPlane &c, const ImpArgs &a, double qm, double q0, double qp,
                   double pr_c, double pr_km, double dphv, double ruold) {
  const double d33 = qp * c.ap2je + q0 * c.ac2je + qm * c.am2je;
  const double udx2 = c.rc * a.al * c.udx2c;
  const double dpx = (pr_c - pr_km) * udx2;
  return (a.ga * dphv + a.ro * ruold + a.alre * d33 - dpx) * a.dt;
}

// Right-hand side row k of the q_z solve (ImplicitAndUpdateQZ.F90:42-113).
// Row nrm is the one the reference leaves behind: assembled a second time
// after the loop overwrote ru3(nrm) with qcap(nrm), so its history term is
// ro*qcap(nrm), with the loop's amm = am3j(nrm).
template <bool NOSLIP = false>
DEVI double rhs_qz(const GridDev &g, const HelmPlane &c, const ImpArgs &a, int k, double qm,
                   double q0, double qp, double pr_c, double pr_jm, double qcv, double ruold,
                   double fic, double foc) {
  double d33, hist = ruold;
  if (k == 1) {
    const double app = c.ap3j;
    const double acc = NOSLIP ? c.ac3j : (c.ac3j * fic + g.ac3j_fs1 * (1 - fic));
    const double amm = NOSLIP ? c.am3j : (c.am3j * fic + g.am3j_fs1 * (1 - fic));
    d33 = qp * app + q0 * acc + q0 * amm;
  } else if (k < g.nrm) {
    d33 = qp * c.ap3j + q0 * c.ac3j + qm * c.am3j;
  } else {
    const double app = NOSLIP ? c.ap3j : (c.ap3j * foc + g.ap3j_fs2 * (1 - foc));
    const double acc = NOSLIP ? c.ac3j : (c.ac3j * foc + g.ac3j_fs2 * (1 - foc));
    d33 = q0 * app + q0 * acc + qm * c.am3j;
    hist = qcv;
  }
  const double dpx = (pr_c - pr_jm) * a.udxz;
  return (a.ga * qcv + a.ro * hist + a.alre * d33 - dpx) * a.dt;
}

// Routine-level right-hand sides, one point per thread: component WHICH of
// ImplicitAndUpdateQT/QR/QZ (F90:40-117, :39-63, :36-115) with the history
// update, scaled as SolveImpEqnUpdate_* scales its rows.
template <int WHICH>
__global__ __launch_bounds__(256) void k_implicit(GridDev g, ImpArgs a, const double *__restrict__ q,
                                                  const double *__restrict__ pr,
                                                  const double *__restrict__ expl,
                                                  double *__restrict__ ru, double *__restrict__ y,
                                                  const unsigned char *__restrict__ icyl,
                                                  const unsigned char *__restrict__ ocyl,
                                                  const RhsRow *__restrict__ rows) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.nthm || j >= g.nzm) return;
  const int k = blockIdx.z + (WHICH == 1 ? 2 : 1), n = g.nrm;
  const long long l = (long long)j * g.nthm + i, o = (long long)(k - 1) * g.P + l;
  const HelmPlane &hc = g.hp[k];
  const RhsRow &t = rows[k];
  const bool wr = WHICH == 1;  // q_r has both walls as planes
  const double q0 = q[o], qm = (wr || k > 1) ? q[o - g.P] : 0.0, qp = (wr || k < n) ? q[o + g.P] : 0.0;
  const double e = expl[o];
  double r;
  if (WHICH == 1) {
    r = rhs_qr(hc, a, qm, q0, qp, pr[o], pr[o - g.P], e, ru[o]) * t.sc_r;
  } else {
    const double fic = (double)icyl[l], foc = (double)ocyl[l];
    if (WHICH == 0) {
      const double pim = pr[o - i + wrap_m(i, g.nthm)];
      r = rhs_qt(g, hc, a, k, qm, q0, qp, pr[o], pim, e, ru[o], fic, foc);
      if (k == 1) r = r + a.bc1;
      r = r * t.sc_t;
    } else {
      const double pjm = pr[o + (long long)(wrap_m(j, g.nzm) - j) * g.nthm];
      r = rhs_qz(g, hc, a, k, qm, q0, qp, pr[o], pjm, e, ru[o], fic, foc) * t.sc_z;
    }
  }
  ru[o] = e;
  y[o] = r;
}

// ---------------------------------------------------------------------------
// Tridiagonal solves of the radial Helmholtz systems.  FOLD: the right-hand
// sides are sc*rhs + A q, so the solution of A x' = sc*rhs + A q is
// x' = q + x, the updated velocity itself, and q is not read; otherwise
// q += x, as the reference adds it.  What the fold rounds passes through
// A^-1, whose norm grows with beta*max|ac|, and so does a difference between
// the A that is folded and the one that the rounded factors solve.  Hence the
// factors of write_partitioned and row_fold's differences.  Relative error of
// one solve of a smooth q, a model against extended precision, at beta*ac =
// 2 / 4e4: 8e-17 / 1.4e-16 (a fold of U q behind the forward sweep 1.2e-16 /
// 2.7e-16, of A q as it stands 1.3e-16 / 3.6e-15, q += x 4.5e-17); the
// explicit radial term of the right-hand side alone rounds to 7e-15 at 4e4.
// 30 steps of 256x256x193 against plain FP64: q_theta 5.6e-16, inner torque
// 1.2e-14 (U q 1.6e-15 and 9e-14, A q 1.7e-15 and 1.4e-13).
//
// Partitioned over the block: a block owns 64 lines (lanes along theta) and
// each of its waves a segment of at most R rows of them, held in registers,
// so a line's rows are loaded as one batch and its dependent chain is as
// long as a segment instead of the line.  Without row exchanges the sweeps
// are y_q = g_q + m_q y_(q-1) and x_q = y_q r_q + u_q x_(q+1).  Each wave sweeps its segment with a zero incoming value and leaves
// the outgoing value and the product of its factors in LDS; the waves then
// chain those (at most 15 terms) to their true incoming value, whose
// contribution down the segment is the same recurrence on one number.  Twice:
// downwards for L, upwards for U.  The factor products of a diagonally
// dominant matrix stay below one, so this is as stable as the sweeps.  All
// multiply-adds are written out: a line has the same bits whether its block
// shares one table or reads one a lane.
//
// The factors of a segment's rows are the same for all lanes (UNIFORM): the
// lanes hold those of one row each and broadcast them by readlane.
// ---------------------------------------------------------------------------
DEVI double rlane(double v, int i) {
  union {
    double d;
    int w[2];
  } u, r;
  u.d = v;
  r.w[0] = __builtin_amdgcn_readlane(u.w[0], i);
  r.w[1] = __builtin_amdgcn_readlane(u.w[1], i);
  return r.d;
}

// comp: 0 q_theta, 1 q_r (rows 2..nrm; both walls are set to zero), 2 q_z.
// lu: the line's table, the same for all lines of the block with UNIFORM.
// CHUNKS: lines of more rows than the block's registers hold (R a wave) go
// in chunks, the first of what the full ones leave over.  L needs only the
// value that enters a chunk, so the chunks are read downwards once for those
// (kept in LDS), the last one is solved while it is held, and the others are
// read a second time on the way up: 1025 rows move 6.7 passes instead of 6.
// The serial form, 12 passes and one dependent chain a line, took 1337 us at
// 256x256x1025 and 5450 us at 512x512x1025; this one takes 820 and 3533.
template <int R, bool UNIFORM, bool FOLD, bool CHUNKS>
DEVI void helm_solve_lines(const long long lgrp, const int comp, const GridDev &g,
                           double *__restrict__ q, const double *__restrict__ y,
                           const double *__restrict__ lu, double *ex) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x, NS = blockDim.y;
  const int p = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const long long P = g.P, l = lgrp * 64 + lane;
  const bool ok = l < P;
  const long long lc = ok ? l : P - 1;
  const int first = comp == 1 ? 1 : 0, n = g.nrm - first;
  const LUView T = lu_view(lu);
  double *exc = ex, *exw = ex + NS * 64;  // outgoing values and factors, L
  double *uxc = ex + 2 * NS * 64, *uxw = ex + 3 * NS * 64;  // and U
  double *enter = ex + 4 * NS * 64;       // CHUNKS: value entering each chunk
  const int cap = R * NS, nc = CHUNKS ? (n + cap - 1) / cap : 1, n0 = n - (nc - 1) * cap;
  if (CHUNKS && p == 0) enter[lane] = 0.0;
  double below = 0.0;  // solution of the row below the chunk
  for (int pass = 0; pass < 2 * nc - 1; pass++) {
    const int ch = pass < nc ? pass : 2 * (nc - 1) - pass;
    const int r0 = first + (ch > 0 ? n0 + (ch - 1) * cap : 0), rn = ch > 0 ? cap : n0;
    const int lo = r0 + p * rn / NS, S = r0 + (p + 1) * rn / NS - lo, Sm = max(S - 1, 0);
    // m, r and u of row lo + i (UNIFORM: of rows lo + lane and, past 64 rows,
    // lo + 64 + lane, loaded before the rows so that their latency is not
    // behind them).  Past the segment's S rows they are those
    // of rows that pass a value on unchanged in both sweeps (right-hand side
    // zero), so the sweeps carry no conditions.
    constexpr int NK = (R + 63) / 64;
    double km[NK], ku[NK], kr[NK];
    if constexpr (UNIFORM) {
#pragma unroll
      for (int u = 0; u < NK; u++) {
        const int r = lo + min(lane + 64 * u, Sm);
        km[u] = T.m(r);
        ku[u] = T.u(r);
        kr[u] = T.rd(r);
      }
    }
    double v[R];
    {
      const double *yp = y + (long long)lo * P + lc;
      if constexpr (CHUNKS) {
        constexpr int B = 20;  // the first chunk's segments may be short
        static_assert(R % B == 0, "row batches");
#pragma unroll
        for (int b = 0; b < R; b += B) {
          if (b < S) {
#pragma unroll
            for (int i = b; i < b + B; i++) v[i] = yp[(long long)min(i, Sm) * P];
          } else {
#pragma unroll
            for (int i = b; i < b + B; i++) v[i] = 0.0;
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < R; i++) v[i] = ld_nt(yp + (long long)min(i, Sm) * P);
      }
    }
    if constexpr (UNIFORM) {
#pragma unroll
      for (int u = 0; u < NK; u++) {
        const int i = lane + 64 * u;
        km[u] = i < S ? km[u] : 1.0;
        ku[u] = i < S ? ku[u] : 1.0;
        kr[u] = i < S ? kr[u] : 0.0;
      }
    }
    auto m = [&](int i) {
      if constexpr (UNIFORM) return rlane(km[i >> 6], i & 63);
      else return T.m(lo + i);
    };
    auto rd = [&](int i) {
      if constexpr (UNIFORM) return rlane(kr[i >> 6], i & 63);
      else return T.rd(lo + i);
    };
    auto up = [&](int i) {
      if constexpr (UNIFORM) return rlane(ku[i >> 6], i & 63);
      else return T.u(lo + i);
    };
    double c = 0.0, w = 1.0;
#pragma unroll
    for (int i = 0; i < R; i++) {
      if (!UNIFORM && i >= S) continue;
      const double d = m(i);
      c = fma(d, c, i < S ? v[i] : 0.0);
      v[i] = c;
      w = w * d;
    }
    exc[p * 64 + lane] = c;
    exw[p * 64 + lane] = w;
    __syncthreads();
    w = CHUNKS ? enter[ch * 64 + lane] : 0.0;
    if (CHUNKS && pass < nc - 1) {
      // downwards: only the value that enters the next chunk
      for (int s = 0; s < NS; s++) w = fma(exw[s * 64 + lane], w, exc[s * 64 + lane]);
      if (p == 0) enter[(ch + 1) * 64 + lane] = w;
      __syncthreads();
      continue;
    }
    for (int s = 0; s < p; s++) w = fma(exw[s * 64 + lane], w, exc[s * 64 + lane]);
#pragma unroll
    for (int i = 0; i < R; i++) {
      if (!UNIFORM && i >= S) continue;
      const double d = m(i);
      v[i] = fma(w, d, v[i]);
      w = w * d;
    }
    c = 0.0;
    w = 1.0;
#pragma unroll
    for (int i = R - 1; i >= 0; i--) {
      if (!UNIFORM && i >= S) continue;
      const double u = up(i);
      c = fma(u, c, v[i] * rd(i));
      v[i] = c;
      w = w * u;
    }
    uxc[p * 64 + lane] = c;
    uxw[p * 64 + lane] = w;
    __syncthreads();
    w = below;
    for (int s = NS - 1; s > p; s--) w = fma(uxw[s * 64 + lane], w, uxc[s * 64 + lane]);
    if constexpr (CHUNKS) {
      for (int s = NS - 1; s >= 0; s--) below = fma(uxw[s * 64 + lane], below, uxc[s * 64 + lane]);
    }
    double *qp = q + (long long)lo * P + l;
#pragma unroll
    for (int i = R - 1; i >= 0; i--) {
      if (!UNIFORM && i >= S) continue;
      const double u = up(i), x = fma(w, u, v[i]);
      w = w * u;
      if (i < S && ok) {
        double *o = qp + (long long)i * P;
        st_nt(o, FOLD ? x : *o + x);
      }
    }
    if constexpr (CHUNKS) __syncthreads();  // exc and uxc are written again
  }
  if (comp == 1 && ok) {  // ImplicitAndUpdateQR.F90:70-71
    if (p == 0) q[l] = 0.0;
    if (p == NS - 1) q[(long long)(g.nr - 1) * P + l] = 0.0;
  }
}

// The table of a block's lines: one for all of them where their wall masks
// agree (always with no-slip walls, and for the lines of a wave along a
// groove), else one for each lane.
template <int R, bool UNIFORM, bool FOLD, bool CHUNKS>
DEVI void helm_solve_body(const long long lgrp, const int comp, const GridDev &g,
                          double *__restrict__ q, const double *__restrict__ y,
                          const unsigned char *__restrict__ icyl,
                          const unsigned char *__restrict__ ocyl, const double *__restrict__ lu,
                          int nt, double *ex) {
  if (UNIFORM || comp == 1) {
    helm_solve_lines<R, true, FOLD, CHUNKS>(lgrp, comp, g, q, y, lu + (size_t)(comp == 1 ? 0 : 3) * nt,
                                            ex);
  } else {
    const long long l = lgrp * 64 + threadIdx.x, lc = l < g.P ? l : g.P - 1;
    const int var = icyl[lc] + 2 * ocyl[lc], v0 = __builtin_amdgcn_readfirstlane(var);
    if (__all(var == v0))  // the same lines in every wave of the block
      helm_solve_lines<R, true, FOLD, CHUNKS>(lgrp, comp, g, q, y, lu + (size_t)v0 * nt, ex);
    else
      helm_solve_lines<R, false, FOLD, CHUNKS>(lgrp, comp, g, q, y, lu + (size_t)var * nt, ex);
  }
}

struct SolveIO {
  double *q[3];
  const double *y[3];
  const double *lu[3];
};

// The components of a line group are consecutive, and the groups contiguous
// per XCD: the six arrays then move together (1024x1024x769: 7.82 ms against
// 8.43-8.56 with one component after the other, the step alike; no difference
// at 512x512x385 and below).
template <int R, bool UNIFORM, bool FOLD, bool CHUNKS>
__global__ __launch_bounds__(R > 32 ? 512 : 1024) void k_helm_solve(
    GridDev g, SolveIO io, const unsigned char *__restrict__ icyl,
    const unsigned char *__restrict__ ocyl, int nt, int comp0) {
  extern __shared__ double ex[];
  const int lin = xcd_tile(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
  const int comp = lin % (int)gridDim.y + comp0;
  helm_solve_body<R, UNIFORM, FOLD, CHUNKS>(
      lin / (int)gridDim.y, comp, g, comp == 0 ? io.q[0] : (comp == 1 ? io.q[1] : io.q[2]),
      comp == 0 ? io.y[0] : (comp == 1 ? io.y[1] : io.y[2]), icyl, ocyl,
      comp == 0 ? io.lu[0] : (comp == 1 ? io.lu[1] : io.lu[2]), nt, ex);
}

// Grouped: blockIdx.z = instance; right-hand sides in rhs, dq, qcap.
template <int R, bool UNIFORM, bool CHUNKS>
__global__ __launch_bounds__(R > 32 ? 512 : 1024) void k_helm_solve_g(
    const StepDesc *__restrict__ tab, int comp0) {
  extern __shared__ double ex[];
  const StepDesc &d = tab[blockIdx.z];
  if (inst_stopped(d)) return;
  const int lin = xcd_tile(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
  const int comp = lin % (int)gridDim.y + comp0;
  helm_solve_body<R, UNIFORM, true, CHUNKS>(
      lin / (int)gridDim.y, comp, glob(d.g),
      glob(d.f[comp == 0 ? TC_QT : (comp == 1 ? TC_QR : TC_QZ)]),
      glob(d.f[comp == 0 ? TC_RHS : (comp == 1 ? TC_DQ : TC_QCAP)]), glob(d.icyl), glob(d.ocyl),
      glob(comp == 0 ? d.lut : (comp == 1 ? d.lur : d.luz)), d.lu_nt, ex);
}

// Serial form, one line per lane: dgttrs as it is, for factors with row
// exchanges.  y is overwritten by the forward sweep.  Loads are issued a chunk
// of rows ahead of the dependent recurrence.
DEVI void helm_solve_serial_body(const long long l, const int comp, const GridDev &g,
                                 double *__restrict__ q, double *__restrict__ y,
                                 const unsigned char *__restrict__ icyl,
                                 const unsigned char *__restrict__ ocyl,
                                 const double *__restrict__ lu, int nt, bool fold) {
  constexpr int CH = 16;
  if (l >= g.P) return;
  const long long P = g.P;
  const int var = comp == 1 ? 0 : icyl[l] + 2 * ocyl[l];
  const LUView T = lu_view(lu + (size_t)var * nt);
  const int first = comp == 1 ? 1 : 0, last = g.nrm - 1;
  double carry = y[(long long)first * P + l], out;
  for (int r0 = first + 1; r0 <= last; r0 += CH) {
    double f[CH];
#pragma unroll
    for (int u = 0; u < CH; u++)
      if (r0 + u <= last) f[u] = y[(long long)(r0 + u) * P + l];
#pragma unroll
    for (int u = 0; u < CH; u++) {
      const int r = r0 + u;
      if (r <= last) {
        lsolve_step(T, r - 1, f[u], carry, out);
        y[(long long)(r - 1) * P + l] = out;
      }
    }
  }
  // q_r: x' is zero at both walls, so row nrm couples to nothing above it
  double x1 = 0.0, x0 = carry * T.rd(last);
  auto put = [&](int r, double x) {
    double *o = q + (long long)r * P + l;
    *o = fold ? x : *o + x;
  };
  put(last, x0);
  for (int r0 = last - 1; r0 >= first; r0 -= CH) {
    double f[CH];
#pragma unroll
    for (int u = 0; u < CH; u++)
      if (r0 - u >= first) f[u] = y[(long long)(r0 - u) * P + l];
#pragma unroll
    for (int u = 0; u < CH; u++) {
      const int r = r0 - u;
      if (r >= first) {
        const double x = (f[u] - T.du(r) * x0 - T.du2(r) * x1) * T.rd(r);
        put(r, x);
        x1 = x0;
        x0 = x;
      }
    }
  }
  if (comp == 1) q[l] = q[(long long)(g.nr - 1) * P + l] = 0.0;
}

__global__ __launch_bounds__(256) void k_helm_solve_serial(GridDev g, SolveIO io,
                                                           const unsigned char *__restrict__ icyl,
                                                           const unsigned char *__restrict__ ocyl,
                                                           int nt, int comp, bool fold) {
  helm_solve_serial_body((long long)blockIdx.x * 256 + threadIdx.x, comp, g,
                         comp == 0 ? io.q[0] : (comp == 1 ? io.q[1] : io.q[2]),
                         const_cast<double *>(comp == 0 ? io.y[0] : (comp == 1 ? io.y[1] : io.y[2])),
                         icyl, ocyl, comp == 0 ? io.lu[0] : (comp == 1 ? io.lu[1] : io.lu[2]), nt, fold);
}

// Grouped: blockIdx.y = instance.
__global__ __launch_bounds__(256) void k_helm_solve_serial_g(const StepDesc *__restrict__ tab,
                                                             int comp) {
  const StepDesc &d = tab[blockIdx.y];
  if (inst_stopped(d)) return;
  helm_solve_serial_body((long long)blockIdx.x * 256 + threadIdx.x, comp, glob(d.g),
                         glob(d.f[comp == 0 ? TC_QT : (comp == 1 ? TC_QR : TC_QZ)]),
                         glob(d.f[comp == 0 ? TC_RHS : (comp == 1 ? TC_DQ : TC_QCAP)]),
                         glob(d.icyl), glob(d.ocyl),
                         glob(comp == 0 ? d.lut : (comp == 1 ? d.lur : d.luz)), d.lu_nt, true);
}

// ---------------------------------------------------------------------------
// Fused substep front: explicit terms and right-hand sides of all three
// components.  A block owns a 64 (theta) x 4*LPT (z) tile of radial lines
// over a segment of r planes; the planes k-1, k, k+1 of qt, qr, qz (with a
// one-point periodic halo) rotate through an LDS ring and plane k+2 is
// fetched into registers while plane k is computed.  The explicit terms
// never reach HBM.  Every value is local to its point, so the segments and
// tiles of a launch do not change the results.
// ---------------------------------------------------------------------------
// One point of CorrectVelocity.F90:32-40 and CorrectPressure.F90:37-46
// (amm = apph), without FMA contraction: the pair kernel and the Helmholtz
// kernel that applies a deferred correction round the same way.
// dm: the dph neighbour at i-1 (qt), k-1 (qr), j-1 (qz).
DEVI double corr_qt(const GridDev &g, int kc, double t, double d, double dm, double dt, double al) {
#pragma clang fp contract(off)
  return t - (d - dm) * dt * al * g.dxt * ldk(g.usrm + kc);
}
DEVI double corr_qr(const GridDev &g, int kc, double r, double d, double dm, double dt, double al) {
#pragma clang fp contract(off)
  return r - (d - dm) * dt * al * ldk(g.rudx2c + kc);
}
DEVI double corr_qz(const GridDev &g, double z, double d, double dm, double dt, double al) {
#pragma clang fp contract(off)
  return z - (d - dm) * al * dt * g.dxz;
}
DEVI double corr_pr(const GridDev &g, int kc, double p, double d, double dim, double dip, double djm,
                    double djp, double dkm, double dkp, double be) {
#pragma clang fp contract(off)
  const double amm = ldk(g.apph + kc), acc = ldk(g.acph + kc), app = amm;
  return p + d -
         be * ((dip - 2.0 * d + dim) * ldk(g.udx1qm + kc) + (djp - 2.0 * d + djm) * g.dxzq +
               (dkp * app + d * acc + dkm * amm));
}

// Row k of D (sc rhs + A q) from the records' scaled entries, with A q in
// differences: (s + e) q + am (q(k-1) - q) + ap (q(k+1) - q) with the row sum
// s + e, which is small where beta*ac is large, as the differences are there.
// The term of q's size is added last, so that it is rounded once.
DEVI double row_fold(double s, double e, double am, double ap, double scr, double qm, double q0,
                     double qp) {
  return fma(s, q0, fma(e, q0, fma(am, qm - q0, fma(ap, qp - q0, scr))));
}
// The same for a point beside a free-slip wall: one off-diagonal, x, towards
// the interior value qi, and the row sum xs, read here so that the planes
// without walls hold neither.
DEVI double wall_fold(const double *x, const double *xs, double scr, double q0, double qi) {
  return fma(ldk(xs), q0, fma(ldk(x), qi - q0, scr));
}

constexpr int FT_N = 256, FT_I = 64, FT_J = FT_N / FT_I, FT_W = FT_I + 2;

// A pressure correction still to be applied: the Helmholtz kernel of the
// next substep applies it to every plane it stages (velocity and pressure)
// and writes the corrected pressure of its tile to pr_out.  The two arrays
// travel as separate __restrict__ arguments: through a struct member the
// compiler could not tell that the pr_out stores leave the grid tables
// alone, and it then loads those with vector loads whose waits also drain
// the plane prefetch.
struct CorrIn {
  double dt, al, be;  // al of the substep that produced dph
};

// CARRY: plane k-1 is not read from the ring but from values the thread
// kept from the previous plane.  The explicit terms and right-hand sides
// read plane k-1 only at (dj, di) = (0, 0), (0, +1) and (+1, 0): m00, m01
// and m10 hold those (the centre, theta+1 and z+1 values of the previous
// iteration's plane k).
template <bool CARRY, int W = FT_W>
struct LAcc {
  const double *m, *c, *p;  // planes k-1, k, k+1 of one field
  int base;                 // of the point in a tile of rows W apart
  double m00, m01, m10;
  DEVI double operator()(int dk, int dj, int di) const {
    if constexpr (CARRY) {
      if (dk < 0) return dj != 0 ? m10 : (di != 0 ? m01 : m00);
    }
    const double *s = dk < 0 ? m : (dk > 0 ? p : c);
    return s[base + dj * W + di];
  }
};

// A block of 256 threads owns a 64 (theta) x 4*LPT (z) tile of radial lines
// from plane k0 to plane k1, LPT lines per thread (rows ty and ty+4).
// UNIFORM: every wall mask is 1 (no-slip everywhere, the SlipBCs default).
template <bool UNIFORM, int LPT>
DEVI void helm_rhs_body(
    const int tile, const int k0, const int k1, const GridDev &g, const ImpArgs &a,
    const double *__restrict__ qt, const double *__restrict__ qr, const double *__restrict__ qz,
    const double *__restrict__ pr, double *__restrict__ ru1, double *__restrict__ ru2,
    double *__restrict__ ru3, double *__restrict__ yt, double *__restrict__ yr,
    double *__restrict__ yz, const unsigned char *__restrict__ icyl,
    const unsigned char *__restrict__ ocyl, const RhsRow *__restrict__ rows, int ntx) {
  constexpr int TJ = FT_J * LPT, H = TJ + 2, S = FT_W * H, NE = (S + FT_N - 1) / FT_N;
  __shared__ double sq[3][3][S];  // field, ring slot, tile
  __shared__ double sp[2][S];     // pressure planes k and k+1
  const int i0 = (tile % ntx) * FT_I, j0 = (tile / ntx) * TJ;
  const int tx = threadIdx.x % FT_I, ty = threadIdx.x / FT_I;
  const long long P = g.P;
  // the tile elements this thread stages per plane: chunks 0..NE-2 are
  // full; in the last one threads past S load a valid element and do not
  // store it, so every global load is unconditional
  int off[NE];
  const bool has_last = threadIdx.x + (NE - 1) * FT_N < S;
#pragma unroll
  for (int q = 0; q < NE; q++) {
    const int e = threadIdx.x + q * FT_N;
    const int ee = e < S ? e : 0;
    int jj = j0 + ee / FT_W - 1, ii = i0 + ee % FT_W - 1;
    jj = ((jj % g.nzm) + g.nzm) % g.nzm;
    ii = ((ii % g.nthm) + g.nthm) % g.nthm;
    off[q] = jj * g.nthm + ii;
  }
  // stage plane p of the velocity (before the first iteration)
  auto stage_q = [&](int p) {
    const long long oq = (long long)(p - 1) * P;
    double t[3][NE];
#pragma unroll
    for (int q = 0; q < NE; q++) {
      t[0][q] = qt[oq + off[q]];
      t[1][q] = qr[oq + off[q]];
      t[2][q] = qz[oq + off[q]];
    }
#pragma unroll
    for (int q = 0; q < NE; q++)
      if (q < NE - 1 || has_last) {
        const int e = threadIdx.x + q * FT_N;
        sq[0][p % 3][e] = t[0][q];
        sq[1][p % 3][e] = t[1][q];
        sq[2][p % 3][e] = t[2][q];
      }
  };
  // the RK history ru enters as ro*ru only: with ro = 0 (the first RK3
  // substep) it is not read at all
  const bool hist = a.ro != 0.0;
  const int nrm = g.nrm;
  // per-line state
  bool valid[LPT];
  long long l[LPT];
  int base[LPT];
  double fic[LPT], foc[LPT], h1[LPT], h2[LPT], h3[LPT], pr_km[LPT];
  // plane k-1 values carried from the previous iteration (qt centre,
  // qt theta+1, qr centre, qz centre, qz z+1), so that no thread reads the
  // ring slot of plane k-1 and the staging of plane k+2 into it needs no
  // barrier of its own
  double cm[LPT][5];
#pragma unroll
  for (int u = 0; u < LPT; u++) {
    const int row = ty + FT_J * u;
    const int i = i0 + tx, j = j0 + row;
    valid[u] = (i < g.nthm) && (j < g.nzm);
    l[u] = valid[u] ? (long long)j * g.nthm + i : 0;
    base[u] = (row + 1) * FT_W + tx + 1;
    fic[u] = (UNIFORM || !valid[u]) ? 1.0 : (double)icyl[l[u]];
    foc[u] = (UNIFORM || !valid[u]) ? 1.0 : (double)ocyl[l[u]];
    const long long o = (long long)(k0 - 1) * P + l[u];
    h1[u] = hist ? ld_nt(ru1 + o) : 0.0;
    h2[u] = hist ? ld_nt(ru2 + o) : 0.0;
    h3[u] = hist ? ld_nt(ru3 + o) : 0.0;
    pr_km[u] = k0 > 1 ? pr[o - P] : 0.0;
#pragma unroll
    for (int q = 0; q < 5; q++) cm[u][q] = 0.0;
  }
  // planes k0-1 (if any), k0 and k0+1 of the velocity, k0 of the pressure
  if (k0 > 1) stage_q(k0 - 1);
  stage_q(k0);
  stage_q(k0 + 1);
  {
    const long long op = (long long)(k0 - 1) * P;
#pragma unroll
    for (int q = 0; q < NE; q++) {
      const double v = pr[op + off[q]];
      if (q < NE - 1 || has_last) sp[k0 & 1][threadIdx.x + q * FT_N] = v;
    }
  }
  __syncthreads();
  if (k0 > 1) {
    const int sm = (k0 - 1) % 3;
#pragma unroll
    for (int u = 0; u < LPT; u++) {
      cm[u][0] = sq[0][sm][base[u]];
      cm[u][1] = sq[0][sm][base[u] + 1];
      cm[u][2] = sq[1][sm][base[u]];
      cm[u][3] = sq[2][sm][base[u]];
      cm[u][4] = sq[2][sm][base[u] + FT_W];
    }
    __syncthreads();  // the first iteration overwrites that slot
  }

  for (int k = k0; k <= k1; k++) {
    // prefetch plane k+2 of the velocity, plane k+1 of the pressure and of
    // the RK histories.  In the last iteration these re-read planes just
    // read (their values are not used), so the loads carry no condition.
    double nq[3][NE], np[NE], n1[LPT], n2[LPT], n3[LPT];
    const long long oq = (long long)min(k + 1, k1) * P;
    const long long op = (long long)min(k, k1 - 1) * P;
#pragma unroll
    for (int q = 0; q < NE; q++) {
      nq[0][q] = qt[oq + off[q]];
      nq[1][q] = qr[oq + off[q]];
      nq[2][q] = qz[oq + off[q]];
      np[q] = pr[op + off[q]];
    }
    if (hist) {
#pragma unroll
      for (int u = 0; u < LPT; u++) {
        n1[u] = ld_nt(ru1 + op + l[u]);
        n2[u] = ld_nt(ru2 + op + l[u]);
        n3[u] = ld_nt(ru3 + op + l[u]);
      }
    } else {
#pragma unroll
      for (int u = 0; u < LPT; u++) n1[u] = n2[u] = n3[u] = 0.0;
    }
    const int sm = (k + 2) % 3, sc = k % 3, sn = (k + 1) % 3;  // planes k-1, k, k+1
    const double *spk = sp[k & 1];
    const HelmPlane hc = ldk_record(g.hp + k);
    const RhsRow rw = ldk_record(rows + k);
#pragma unroll
    for (int u = 0; u < LPT; u++) {
      if (!valid[u]) continue;
      LAcc<true> T, R, Z;
      T.m = sq[0][sm]; T.c = sq[0][sc]; T.p = sq[0][sn]; T.base = base[u];
      R.m = sq[1][sm]; R.c = sq[1][sc]; R.p = sq[1][sn]; R.base = base[u];
      Z.m = sq[2][sm]; Z.c = sq[2][sc]; Z.p = sq[2][sn]; Z.base = base[u];
      T.m00 = cm[u][0]; T.m01 = cm[u][1]; T.m10 = 0.0;
      R.m00 = cm[u][2]; R.m01 = R.m10 = 0.0;
      Z.m00 = cm[u][3]; Z.m01 = 0.0; Z.m10 = cm[u][4];
      const double pr_c = spk[base[u]], pr_im = spk[base[u] - 1], pr_jm = spk[base[u] - FT_W];
      const long long o = (long long)(k - 1) * P + l[u];
      // whether the matrix rows of q_theta and q_z are those beside a free-slip wall
      const bool slip1 = !UNIFORM && k == 1 && fic[u] == 0.0, slipn = !UNIFORM && k == nrm && foc[u] == 0.0;
      // q_theta
      {
        const double dqv = explicit_qt_g(g, hc, T, R, Z, k);
        const double qm = (k > 1) ? T(-1, 0, 0) : 0.0, qp = (k < nrm) ? T(1, 0, 0) : 0.0;
        double r = rhs_qt<UNIFORM>(g, hc, a, k, qm, T(0, 0, 0), qp, pr_c, pr_im, dqv, h1[u], fic[u], foc[u]);
        st_nt(ru1 + o, dqv);
        if (k == 1) r = r + a.bc1;
        double y = row_fold(rw.s_t, rw.e_t, rw.am_t, rw.ap_t, r * rw.sc_t, qm, T(0, 0, 0), qp);
        if (slip1 || slipn)
          y = wall_fold(&rows[k].x_t, &rows[k].xs_t, r * rw.sc_t, T(0, 0, 0), slip1 ? qp : qm);
        st_nt(yt + o, y);
      }
      // q_r (planes 2..nrm; the walls have no row)
      if (k >= 2) {
        const double dphv = explicit_qr_g(g, hc, T, R, Z, k);
        const double r = rhs_qr(hc, a, R(-1, 0, 0), R(0, 0, 0), R(1, 0, 0), pr_c, pr_km[u], dphv, h2[u]);
        st_nt(ru2 + o, dphv);
        st_nt(yr + o, row_fold(rw.s_r, rw.e_r, rw.am_r, rw.ap_r, r * rw.sc_r, R(-1, 0, 0), R(0, 0, 0),
                                R(1, 0, 0)));
      }
      // q_z
      {
        const double qcv = explicit_qz_g(g, hc, T, R, Z, k);
        const double qm = (k > 1) ? Z(-1, 0, 0) : 0.0, qp = (k < nrm) ? Z(1, 0, 0) : 0.0;
        const double r = rhs_qz<UNIFORM>(g, hc, a, k, qm, Z(0, 0, 0), qp, pr_c, pr_jm, qcv, h3[u], fic[u], foc[u]);
        st_nt(ru3 + o, qcv);
        double y = row_fold(rw.s_z, rw.e_z, rw.am_z, rw.ap_z, r * rw.sc_z, qm, Z(0, 0, 0), qp);
        if (slip1 || slipn)
          y = wall_fold(&rows[k].x_z, &rows[k].xs_z, r * rw.sc_z, Z(0, 0, 0), slip1 ? qp : qm);
        st_nt(yz + o, y);
      }
      pr_km[u] = pr_c;
      cm[u][0] = T(0, 0, 0);
      cm[u][1] = T(0, 0, 1);
      cm[u][2] = R(0, 0, 0);
      cm[u][3] = Z(0, 0, 0);
      cm[u][4] = Z(0, 1, 0);
    }
    if (k == k1) break;
#pragma unroll
    for (int u = 0; u < LPT; u++) {
      h1[u] = n1[u];
      h2[u] = n2[u];
      h3[u] = n3[u];
    }
    const int s2 = (k + 2) % 3;
#pragma unroll
    for (int q = 0; q < NE; q++) {
      const int e = threadIdx.x + q * FT_N;
      if (q < NE - 1 || has_last) {
        sq[0][s2][e] = nq[0][q];
        sq[1][s2][e] = nq[1][q];
        sq[2][s2][e] = nq[2][q];
        sp[(k + 1) & 1][e] = np[q];
      }
    }
    __syncthreads();
  }
}

// Even theta sizes: a thread owns two theta-adjacent lines, so that planes,
// histories and results move as 16-byte pairs (the address unit takes a
// 64-lane load or store 16 cycles whatever its width) and the two points
// share the LDS reads and the sums that their stencils have in common.  A
// block of 32*TJ threads owns a 64 (theta) x TJ (z) tile from plane k0 to k1.
// CORR: qt, qr, qz hold the previous substep's velocity before its pressure
// correction and pr its pressure before the correction; the correction (dph
// of that substep) is applied to each plane as it is staged, from a ring of
// dph planes with one more row of halo on either side, so the corrected
// fields are the ones the per-substep path would have stored, bit for bit.
// Against one line or two z-rows of lines per thread, with the correction:
// 256x256x193 343 -> 313 us, 512x512x385 2576 -> 2491 us, 1024x1024x769 20.5
// -> 18.4 ms (HBM bound at the larger sizes: 4.9 of the 5.7 TB/s that fifteen
// streamed arrays reach; with the fold in differences 303, 2490 us, 18.8 ms).
// The kernels ask for two waves per SIMD: the masked form, corrected, once
// left that when it was not asked to (192x128x129 125 us at one wave, 88 at
// two).  It holds what only the two wall planes need nowhere else (wall_fold)
// and takes 222 registers with none spilled; with the wall rows' entries in
// every plane 24 to 53 were.
// (The outermost column of the tile on either side is staged only to keep
// pairs aligned; nothing reads it.)
constexpr int PT_W = FT_I + 4, PT_P = PT_W / 2;  // tile row: i0-2 .. i0+65
template <bool UNIFORM, int TJ, bool CORR>
DEVI void helm_rhs_pair_body(
    const int tile, const int k0, const int k1, const GridDev &g, const ImpArgs &a,
    const double *__restrict__ qt, const double *__restrict__ qr, const double *__restrict__ qz,
    const double *__restrict__ pr, double *__restrict__ ru1, double *__restrict__ ru2,
    double *__restrict__ ru3, double *__restrict__ yt, double *__restrict__ yr,
    double *__restrict__ yz, const unsigned char *__restrict__ icyl,
    const unsigned char *__restrict__ ocyl, const RhsRow *__restrict__ rows, int ntx,
    const CorrIn &ci, const double *__restrict__ dph, double *__restrict__ pr_out) {
  constexpr int NT = 32 * TJ, S = PT_P * (TJ + 2), NE = (S + NT - 1) / NT;      // pairs
  constexpr int S2 = PT_P * (TJ + 4), NE2 = (S2 + NT - 1) / NT;
  __shared__ __align__(16) double sq[3][3][2 * S];  // field, ring slot, tile
  __shared__ __align__(16) double sp[2][2 * S];     // pressure planes k and k+1
  __shared__ __align__(16) double sd[CORR ? 3 : 1][CORR ? 2 * S2 : 2];  // dph planes (slot = plane % 3)
  const int i0 = (tile % ntx) * FT_I, j0 = (tile / ntx) * TJ;
  const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;
  const long long P = g.P;
  auto ld2 = [](const double *p) { return *reinterpret_cast<const double2 *>(p); };
  auto put2 = [](double *p, double2 v) { *reinterpret_cast<double2 *>(p) = v; };
  // the pairs of the tile that this thread stages per plane: in the last
  // chunk threads past S load a valid pair and do not store it, so every
  // global load is unconditional
  auto wrapped = [&](int row, int pair) {
    int jj = j0 + row, ii = i0 - 2 + 2 * pair;
    jj = ((jj % g.nzm) + g.nzm) % g.nzm;
    ii = ((ii % g.nthm) + g.nthm) % g.nthm;
    return jj * g.nthm + ii;
  };
  int off[NE], off2[CORR ? NE2 : 1];
  bool wpr[NE];
  const bool has_last = threadIdx.x + (NE - 1) * NT < S;
  const bool has_last2 = threadIdx.x + (NE2 - 1) * NT < S2;
#pragma unroll
  for (int q = 0; q < NE; q++) {
    const int e = threadIdx.x + q * NT, ee = e < S ? e : 0;
    const int row = ee / PT_P, pair = ee % PT_P;
    off[q] = wrapped(row - 1, pair);
    // an interior pair, whose corrected pressure this thread writes
    wpr[q] = CORR && e < S && row >= 1 && row <= TJ && pair >= 1 && pair <= 32 &&
             j0 + row - 1 < g.nzm && i0 - 2 + 2 * pair < g.nthm;
  }
  if constexpr (CORR) {
#pragma unroll
    for (int q = 0; q < NE2; q++) {
      const int e = threadIdx.x + q * NT, ee = e < S2 ? e : 0;
      off2[q] = wrapped(ee / PT_P - 2, ee % PT_P);
    }
  }
  // the corrected velocity of plane p at the tile pair e (correct_pair's
  // arithmetic; q_r is zero on both walls)
  auto corr_q = [&](int p, int e, double2 &vt, double2 &vr, double2 &vz) {
    const int e2 = 2 * (e + PT_P);  // the same point in a dph plane
    const double *dc = sd[CORR ? p % 3 : 0];
    const double2 d = ld2(dc + e2);
    if (p <= g.nrm) {
      const double2 djm = ld2(dc + e2 - PT_W);
      vt.x = corr_qt(g, p, vt.x, d.x, dc[e2 - 1], ci.dt, ci.al);
      vt.y = corr_qt(g, p, vt.y, d.y, d.x, ci.dt, ci.al);
      vz.x = corr_qz(g, vz.x, d.x, djm.x, ci.dt, ci.al);
      vz.y = corr_qz(g, vz.y, d.y, djm.y, ci.dt, ci.al);
    }
    if (p == 1 || p >= g.nr) {
      vr = make_double2(0.0, 0.0);
    } else {
      const double2 dkm = ld2(sd[CORR ? (p - 1) % 3 : 0] + e2);
      vr.x = corr_qr(g, p, vr.x, d.x, dkm.x, ci.dt, ci.al);
      vr.y = corr_qr(g, p, vr.y, d.y, dkm.y, ci.dt, ci.al);
    }
  };
  // the corrected pressure of plane p <= nrm at the tile pair e
  auto corr_p = [&](int p, int e, double2 v) {
    const int e2 = 2 * (e + PT_P);
    const double *dc = sd[CORR ? p % 3 : 0];
    const double2 dkp = ld2(sd[CORR ? (p < g.nrm ? p + 1 : p) % 3 : 0] + e2);
    const double2 dkm = ld2(sd[CORR ? (p > 1 ? p - 1 : p) % 3 : 0] + e2);
    const double2 d = ld2(dc + e2), djm = ld2(dc + e2 - PT_W), djp = ld2(dc + e2 + PT_W);
    return make_double2(
        corr_pr(g, p, v.x, d.x, dc[e2 - 1], d.y, djm.x, djp.x, dkm.x, dkp.x, ci.be),
        corr_pr(g, p, v.y, d.y, d.x, dc[e2 + 2], djm.y, djp.y, dkm.y, dkp.y, ci.be));
  };
  // stage dph plane p (clamped to 1..nrm: beyond it no correction reads dph)
  auto stage_dph = [&](int p) {
    const long long od = (long long)(min(max(p, 1), g.nrm) - 1) * P;
    double2 t[CORR ? NE2 : 1];
#pragma unroll
    for (int q = 0; q < NE2; q++) t[q] = ld2(dph + od + off2[q]);
#pragma unroll
    for (int q = 0; q < NE2; q++)
      if (q < NE2 - 1 || has_last2) put2(sd[(p + 3) % 3] + 2 * (threadIdx.x + q * NT), t[q]);
  };
  // stage plane p of the velocity (before the first iteration)
  auto stage_q = [&](int p) {
    const long long oq = (long long)(p - 1) * P;
    double2 t[3][NE];
#pragma unroll
    for (int q = 0; q < NE; q++) {
      t[0][q] = ld2(qt + oq + off[q]);
      t[1][q] = ld2(qr + oq + off[q]);
      t[2][q] = ld2(qz + oq + off[q]);
    }
#pragma unroll
    for (int q = 0; q < NE; q++)
      if (q < NE - 1 || has_last) {
        const int e = threadIdx.x + q * NT;
        if constexpr (CORR) corr_q(p, e, t[0][q], t[1][q], t[2][q]);
#pragma unroll
        for (int f = 0; f < 3; f++) put2(sq[f][p % 3] + 2 * e, t[f][q]);
      }
  };
  // the RK history ru enters as ro*ru only: with ro = 0 (the first RK3
  // substep) it is not read at all
  const bool hist = CORR || a.ro != 0.0;
  const int nrm = g.nrm;
  const int i = i0 + 2 * tx, j = j0 + ty;
  const bool valid = i < g.nthm && j < g.nzm;
  const long long l = valid ? (long long)j * g.nthm + i : 0;
  const int base = (ty + 1) * PT_W + 2 * tx + 2;
  // wall masks: bits 0, 1 the inner wall's at the two points, 2, 3 the outer's
  int wall = 15;
  if (!UNIFORM && valid) wall = icyl[l] + 2 * icyl[l + 1] + 4 * ocyl[l] + 8 * ocyl[l + 1];
  const double2 zero = make_double2(0.0, 0.0);
  double2 h1, h2, h3, pkm;
  {
    const long long o = (long long)(k0 - 1) * P + l;
    h1 = hist ? ld2_nt(ru1 + o) : zero;
    h2 = hist ? ld2_nt(ru2 + o) : zero;
    h3 = hist ? ld2_nt(ru3 + o) : zero;
    pkm = k0 > 1 ? ld2(pr + o - P) : zero;
  }
  // !CORR: plane k-1 values carried from the previous iteration (qt at
  // theta, +1, +2; qr and qz at theta, +1; qz of row z+1), so that no thread
  // reads the ring slot of plane k-1 and the staging of plane k+2 into it
  // needs no barrier of its own
  double cm[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  auto carry = [&](const double *t, const double *r, const double *z) {
    cm[0] = t[base], cm[1] = t[base + 1], cm[2] = t[base + 2];
    cm[3] = r[base], cm[4] = r[base + 1];
    cm[5] = z[base], cm[6] = z[base + 1];
    cm[7] = z[base + PT_W], cm[8] = z[base + PT_W + 1];
  };
  // planes k0-1 (if any), k0 and k0+1 of the velocity, k0 of the pressure
  // and the pressure of k0-1 on the lines themselves.  CORR: with the dph
  // planes that each of these corrections reads staged before it.
  if constexpr (CORR) {
    if (k0 > 1) {
      stage_dph(k0 - 2);
      stage_dph(k0 - 1);
      stage_dph(k0);
      __syncthreads();
      stage_q(k0 - 1);
      pkm = corr_p(k0 - 1, base / 2, pkm);
      __syncthreads();
      stage_dph(k0 + 1);
    } else {
      stage_dph(1);
      stage_dph(2);
    }
    __syncthreads();
  } else if (k0 > 1) {
    stage_q(k0 - 1);
  }
  stage_q(k0);
  stage_q(k0 + 1);
  {
    const long long op = (long long)(k0 - 1) * P;
#pragma unroll
    for (int q = 0; q < NE; q++) {
      double2 v = ld2(pr + op + off[q]);
      const int e = threadIdx.x + q * NT;
      if (q < NE - 1 || has_last) {
        if constexpr (CORR) {
          v = corr_p(k0, e, v);
          if (wpr[q]) st2_nt(pr_out + op + off[q], v.x, v.y);
        }
        put2(sp[k0 & 1] + 2 * e, v);
      }
    }
  }
  __syncthreads();
  if constexpr (!CORR) {
    if (k0 > 1) {
      const int sm = (k0 - 1) % 3;
      carry(sq[0][sm], sq[1][sm], sq[2][sm]);
      __syncthreads();  // the first iteration overwrites that slot
    }
  }

  for (int k = k0; k <= k1; k++) {
    // prefetch plane k+2 of the velocity, plane k+1 of the pressure and of
    // the RK histories.  In the last iteration these re-read planes just
    // read (their values are not used), so the loads carry no condition.
    double2 nq[3][NE], np[NE], n1 = zero, n2 = zero, n3 = zero, nd[CORR ? NE2 : 1];
    const long long oq = (long long)min(k + 1, k1) * P;
    const long long op = (long long)min(k, k1 - 1) * P;
#pragma unroll
    for (int q = 0; q < NE; q++) {
      nq[0][q] = ld2(qt + oq + off[q]);
      nq[1][q] = ld2(qr + oq + off[q]);
      nq[2][q] = ld2(qz + oq + off[q]);
      np[q] = ld2(pr + op + off[q]);
    }
    if constexpr (CORR) {
      const long long od = (long long)(min(min(k + 2, k1 + 1), nrm) - 1) * P;
#pragma unroll
      for (int q = 0; q < NE2; q++) nd[q] = ld2(dph + od + off2[q]);
    }
    if (hist) {
      n1 = ld2_nt(ru1 + op + l);
      n2 = ld2_nt(ru2 + op + l);
      n3 = ld2_nt(ru3 + op + l);
    }
    const int sm = (k + 2) % 3, sc = k % 3, sn = (k + 1) % 3;  // planes k-1, k, k+1
    const HelmPlane hc = ldk_record(g.hp + k);
    const RhsRow rw = ldk_record(rows + k);
    if (valid) {
      const double *spk = sp[k & 1];
      const long long o = (long long)(k - 1) * P + l;
      double e1[2], e2[2], e3[2], g1[2], g2[2], g3[2];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int b = base + u;
        LAcc<!CORR, PT_W> T, R, Z;
        T.m = sq[0][sm]; T.c = sq[0][sc]; T.p = sq[0][sn]; T.base = b;
        R.m = sq[1][sm]; R.c = sq[1][sc]; R.p = sq[1][sn]; R.base = b;
        Z.m = sq[2][sm]; Z.c = sq[2][sc]; Z.p = sq[2][sn]; Z.base = b;
        T.m00 = cm[u]; T.m01 = cm[u + 1]; T.m10 = 0.0;
        R.m00 = cm[3 + u]; R.m01 = R.m10 = 0.0;
        Z.m00 = cm[5 + u]; Z.m01 = 0.0; Z.m10 = cm[7 + u];
        const double fic = (double)(wall >> u & 1), foc = (double)(wall >> u >> 2 & 1);
        const double pr_c = spk[b], pr_im = spk[b - 1], pr_jm = spk[b - PT_W];
        // whether the matrix rows of q_theta and q_z are those beside a free-slip wall
        const bool slip1 = !UNIFORM && k == 1 && !(wall >> u & 1);
        const bool slipn = !UNIFORM && k == nrm && !(wall >> u & 4);
        // q_theta
        e1[u] = explicit_qt_g(g, hc, T, R, Z, k);
        const double tm = (k > 1) ? T(-1, 0, 0) : 0.0, tp = (k < nrm) ? T(1, 0, 0) : 0.0;
        double r = rhs_qt<UNIFORM>(g, hc, a, k, tm, T(0, 0, 0), tp, pr_c, pr_im, e1[u],
                                   u ? h1.y : h1.x, fic, foc);
        if (k == 1) r = r + a.bc1;
        g1[u] = row_fold(rw.s_t, rw.e_t, rw.am_t, rw.ap_t, r * rw.sc_t, tm, T(0, 0, 0), tp);
        if (slip1 || slipn)
          g1[u] = wall_fold(&rows[k].x_t, &rows[k].xs_t, r * rw.sc_t, T(0, 0, 0), slip1 ? tp : tm);
        // q_r (planes 2..nrm; the walls have no row)
        if (k >= 2) {
          e2[u] = explicit_qr_g(g, hc, T, R, Z, k);
          r = rhs_qr(hc, a, R(-1, 0, 0), R(0, 0, 0), R(1, 0, 0), pr_c, u ? pkm.y : pkm.x, e2[u],
                     u ? h2.y : h2.x);
          g2[u] = row_fold(rw.s_r, rw.e_r, rw.am_r, rw.ap_r, r * rw.sc_r, R(-1, 0, 0), R(0, 0, 0),
                           R(1, 0, 0));
        }
        // q_z
        e3[u] = explicit_qz_g(g, hc, T, R, Z, k);
        const double zm = (k > 1) ? Z(-1, 0, 0) : 0.0, zp = (k < nrm) ? Z(1, 0, 0) : 0.0;
        r = rhs_qz<UNIFORM>(g, hc, a, k, zm, Z(0, 0, 0), zp, pr_c, pr_jm, e3[u], u ? h3.y : h3.x,
                            fic, foc);
        g3[u] = row_fold(rw.s_z, rw.e_z, rw.am_z, rw.ap_z, r * rw.sc_z, zm, Z(0, 0, 0), zp);
        if (slip1 || slipn)
          g3[u] = wall_fold(&rows[k].x_z, &rows[k].xs_z, r * rw.sc_z, Z(0, 0, 0), slip1 ? zp : zm);
        if (u)
          pkm.y = pr_c;
        else
          pkm.x = pr_c;
      }
      st2_nt(ru1 + o, e1[0], e1[1]);
      st2_nt(yt + o, g1[0], g1[1]);
      if (k >= 2) {
        st2_nt(ru2 + o, e2[0], e2[1]);
        st2_nt(yr + o, g2[0], g2[1]);
      }
      st2_nt(ru3 + o, e3[0], e3[1]);
      st2_nt(yz + o, g3[0], g3[1]);
      if constexpr (!CORR) carry(sq[0][sc], sq[1][sc], sq[2][sc]);
    }
    if (k == k1) break;
    h1 = n1;
    h2 = n2;
    h3 = n3;
    if constexpr (CORR) {
      // dph slot (k+2)%3 held plane k-1, last read before the previous barrier
#pragma unroll
      for (int q = 0; q < NE2; q++)
        if (q < NE2 - 1 || has_last2) put2(sd[(k + 2) % 3] + 2 * (threadIdx.x + q * NT), nd[q]);
      // the ring slot of plane k-1 is read above, and the dph plane k+2 just
      // written is read by the staging below
      __syncthreads();
    }
    const int s2 = (k + 2) % 3;
#pragma unroll
    for (int q = 0; q < NE; q++) {
      const int e = threadIdx.x + q * NT;
      if (q < NE - 1 || has_last) {
        if constexpr (CORR) {
          corr_q(k + 2, e, nq[0][q], nq[1][q], nq[2][q]);
          np[q] = corr_p(k + 1, e, np[q]);
          if (wpr[q]) st2_nt(pr_out + (long long)k * P + off[q], np[q].x, np[q].y);
        }
#pragma unroll
        for (int f = 0; f < 3; f++) put2(sq[f][s2] + 2 * e, nq[f][q]);
        put2(sp[(k + 1) & 1] + 2 * e, np[q]);
      }
    }
    __syncthreads();
  }
}

// Planes k0..k1 of segment s of ns.
DEVI int seg_first(int s, int ns, int nrm) { return 1 + (int)(((long long)s * nrm) / ns); }

// PAIR: the pair form (even nthm), tiles of 4*LPT rows; otherwise LPT lines
// per thread.
template <bool UNIFORM, int LPT, bool CORR, bool PAIR>
__global__ __launch_bounds__(PAIR ? 128 * LPT : FT_N, 2) void k_helm_rhs(
    GridDev g, ImpArgs a, const double *__restrict__ qt, const double *__restrict__ qr,
    const double *__restrict__ qz, const double *__restrict__ pr, double *__restrict__ ru1,
    double *__restrict__ ru2, double *__restrict__ ru3, double *__restrict__ yt,
    double *__restrict__ yr, double *__restrict__ yz, const unsigned char *__restrict__ icyl,
    const unsigned char *__restrict__ ocyl, const RhsRow *__restrict__ rows, int ntx, int ntz,
    int nseg, CorrIn ci, const double *__restrict__ dph, double *__restrict__ pr_out) {
  const int lin = xcd_tile(blockIdx.x, gridDim.x), seg = lin / (ntx * ntz);
  const int tile = lin - seg * (ntx * ntz);
  const int k0 = seg_first(seg, nseg, g.nrm), k1 = seg_first(seg + 1, nseg, g.nrm) - 1;
  if constexpr (PAIR)
    helm_rhs_pair_body<UNIFORM, 4 * LPT, CORR>(tile, k0, k1, g, a, qt, qr, qz, pr, ru1, ru2, ru3,
                                               yt, yr, yz, icyl, ocyl, rows, ntx, ci, dph, pr_out);
  else
    helm_rhs_body<UNIFORM, LPT>(tile, k0, k1, g, a, qt, qr, qz, pr, ru1, ru2, ru3, yt, yr, yz, icyl,
                                ocyl, rows, ntx);
}

// Grouped: blockIdx.x = tile and segment, blockIdx.y = instance of the shape
// group; the XCD remap runs over the flattened index.
template <bool UNIFORM, int LPT, bool CORR, bool PAIR>
__global__ __launch_bounds__(PAIR ? 128 * LPT : FT_N, 2) void k_helm_rhs_g(
    const StepDesc *__restrict__ tab, const BatchDyn *__restrict__ dyn, int ns, int ntx, int ntz,
    int nseg) {
  const int lin = xcd_tile(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
  const int inst = lin / (int)gridDim.x, rest = lin - inst * (int)gridDim.x;
  const int seg = rest / (ntx * ntz), tile = rest - seg * (ntx * ntz);
  const StepDesc &d = tab[inst];
  if (inst_stopped(d)) return;
  ImpArgs a = d.a;
  a.vwall_in = glob(dyn)[inst].vwall[ns - 1];
  a.bc1 = glob(dyn)[inst].bc1[ns - 1];
  const int k0 = seg_first(seg, nseg, d.g.nrm), k1 = seg_first(seg + 1, nseg, d.g.nrm) - 1;
  if constexpr (PAIR)
    helm_rhs_pair_body<UNIFORM, 4 * LPT, CORR>(
        tile, k0, k1, glob(d.g), a, glob(d.f[TC_QT]), glob(d.f[TC_QR]), glob(d.f[TC_QZ]),
        glob(d.pr_in), glob(d.f[TC_RU1]), glob(d.f[TC_RU2]), glob(d.f[TC_RU3]), glob(d.f[TC_RHS]),
        glob(d.f[TC_DQ]), glob(d.f[TC_QCAP]), glob(d.icyl), glob(d.ocyl), glob(d.rows), ntx,
        CorrIn{d.dt, d.corr_al, d.beta}, glob(d.f[TC_DPH]), glob(d.pr_out));
  else
    helm_rhs_body<UNIFORM, LPT>(
        tile, k0, k1, glob(d.g), a, glob(d.f[TC_QT]), glob(d.f[TC_QR]), glob(d.f[TC_QZ]),
        glob(d.pr_in), glob(d.f[TC_RU1]), glob(d.f[TC_RU2]), glob(d.f[TC_RU3]), glob(d.f[TC_RHS]),
        glob(d.f[TC_DQ]), glob(d.f[TC_QCAP]), glob(d.icyl), glob(d.ocyl), glob(d.rows), ntx);
}

static ImpArgs imp_args(const tc_ctx *c) {
  ImpArgs a;
  a.al = c->al;
  a.ga = c->ga;
  a.ro = c->ro;
  a.dt = c->dt;
  a.alre = c->al / c->p.ren;
  a.vwall_in = c->p.virotint + c->vinner_t;
  a.virotext = c->p.virotext;
  a.bc1 = 0.5 * c->al * c->dt * c->dvinner_t * c->g.am1j[1] / c->p.ren;
  a.udxz = c->g.dxz * c->al;
  return a;
}

// Layout of c->lu: [slot = ns-1] of tables [comp][variant 0..3][lu_nt], then
// the records of the right-hand sides for k = 0..nrm (record 0 unused).
size_t lu_slot_doubles(const tc_ctx *c) {
  return (size_t)3 * 4 * c->lu_nt + (size_t)(c->nrm + 1) * (sizeof(RhsRow) / sizeof(double));
}
const double *lu_table(const tc_ctx *c, int ns, int comp) {
  return c->lu + (size_t)(ns - 1) * lu_slot_doubles(c) + (size_t)comp * 4 * c->lu_nt;
}
const RhsRow *rhs_rows(const tc_ctx *c, int ns) {
  return reinterpret_cast<const RhsRow *>(c->lu + (size_t)(ns - 1) * lu_slot_doubles(c) +
                                          (size_t)3 * 4 * c->lu_nt);
}

static unsigned line_blocks(const tc_ctx *c) { return (unsigned)((c->P + 255) / 256); }

// Shape of the partitioned solve: waves per block and the row capacity R of
// its kernel, by the grid's shape alone (an instance's bits must not depend on
// what it shares a launch with).  Past eight waves of 100 rows a line goes in
// chunks.  Few rows a wave shorten the chain where there are few lines, many
// keep more loads in flight where there are many: measured us with R = 25 / 50
// / 100, 128x128x97 19 / 19 / 24, 256x256x193 120 / 124 / 128, 512x512x193 481
// / 490 / 485, 1024x512x193 938 / 971 / 956, 256x256x385 260 / 248 / 244,
// 512x512x385 1016 / 955 / 970 (941 / 869 / 828 in processes where every
// kernel of the step ran faster).  Nine waves of 25 and more no longer pair up
// on a compute unit: 96x96x250 27 / 23, 128x128x225 39.5 / 37.8, 192x128x240
// 66 / 61, 256x256x205 161 / 140, 256x256x250 178 / 164, 512x512x225 633 /
// 571, 480x512x250 640 / 592 (64x64x225 17.7 / 19.4).
struct SolveShape {
  int ns, rows;
  bool chunks;  // lines of more than ns*rows rows
};
static SolveShape solve_shape(const tc_ctx *c) {
  const int n = c->nrm;
  const int R =
      n <= 72 ? 8 : (n <= 200 ? 25 : (n <= 256 || (n <= 400 && c->P < (1 << 17)) ? 50 : 100));
  const int ns = (n + R - 1) / R, most = R > 32 ? 8 : 16;
  return {std::min(ns, most), R, ns > most};
}
// LDS of a block: what its waves pass on in L and in U, and for a line in
// chunks what enters each of them
static size_t solve_lds(const SolveShape s, int n) {
  const size_t chunks = s.chunks ? (size_t)((n + s.ns * s.rows - 1) / (s.ns * s.rows)) : 0;
  return sizeof(double) * 64 * (4 * (size_t)s.ns + chunks);
}

template <bool U, bool FOLD>
static void launch_solve_u(const SolveShape s, dim3 grid, hipStream_t st, const tc_ctx *c,
                           const SolveIO &io, int comp0) {
  const dim3 block(64, (unsigned)s.ns);
  const size_t lds = solve_lds(s, c->nrm);
#define TC_SOLVE(R, CHUNKS)                                                              \
  hipLaunchKernelGGL((k_helm_solve<R, U, FOLD, CHUNKS>), grid, block, lds, st, c->gd, io, \
                     c->mask, c->mask + c->P, c->lu_nt, comp0)
  switch (s.rows) {
    case 8: TC_SOLVE(8, false); break;
    case 25: TC_SOLVE(25, false); break;
    case 50: TC_SOLVE(50, false); break;
    default:
      if (s.chunks) TC_SOLVE(100, true);
      else TC_SOLVE(100, false);
  }
#undef TC_SOLVE
}

// FOLD: all three components (one by one where some take the serial form);
// otherwise the one component comp0
template <bool FOLD>
static void launch_solve(tc_ctx *c, const SolveIO &io, int comp0, int ncomp) {
  const unsigned serial = c->lu_serial;
  if (ncomp > 1 && serial) {
    for (int q = 0; q < ncomp; q++) launch_solve<FOLD>(c, io, comp0 + q, 1);
    return;
  }
  if (serial >> comp0 & 1) {
    hipLaunchKernelGGL(k_helm_solve_serial, dim3(line_blocks(c)), dim3(256), 0, c->stream, c->gd, io,
                       c->mask, c->mask + c->P, c->lu_nt, comp0, FOLD);
    return;
  }
  const SolveShape s = solve_shape(c);
  const dim3 grid((unsigned)((c->P + 63) / 64), (unsigned)ncomp);
  if (c->masks_uniform_one)
    launch_solve_u<true, FOLD>(s, grid, c->stream, c, io, comp0);
  else
    launch_solve_u<false, FOLD>(s, grid, c->stream, c, io, comp0);
}

static SolveIO solve_io(const tc_ctx *c) {
  SolveIO io;
  io.q[0] = c->f[TC_QT];
  io.q[1] = c->f[TC_QR];
  io.q[2] = c->f[TC_QZ];
  io.y[0] = c->f[TC_RHS];
  io.y[1] = c->f[TC_DQ];
  io.y[2] = c->f[TC_QCAP];
  for (int q = 0; q < 3; q++) io.lu[q] = lu_table(c, c->ns, q);
  return io;
}

// Routine-level entries: right-hand side into the rhs field, then the solve.
template <int WHICH>
static void launch_implicit(tc_ctx *c, const char *name, int q, int expl, int ru) {
  timer_begin(c, name);
  hipLaunchKernelGGL(k_implicit<WHICH>, point_grid(c, WHICH == 1 ? c->nrm - 1 : c->nrm),
                     dim3(64, 4), 0, c->stream, c->gd, imp_args(c), c->f[q], c->f[TC_PR],
                     c->f[expl], c->f[ru], c->f[TC_RHS], c->mask, c->mask + c->P,
                     rhs_rows(c, c->ns));
  timer_end(c);
  SolveIO io = solve_io(c);
  io.y[WHICH] = c->f[TC_RHS];
  launch_solve<false>(c, io, WHICH, 1);
}
void launch_implicit_qt(tc_ctx *c) { launch_implicit<0>(c, "implicit_qt", TC_QT, TC_DQ, TC_RU1); }
void launch_implicit_qr(tc_ctx *c) { launch_implicit<1>(c, "implicit_qr", TC_QR, TC_DPH, TC_RU2); }
void launch_implicit_qz(tc_ctx *c) { launch_implicit<2>(c, "implicit_qz", TC_QZ, TC_QCAP, TC_RU3); }

static unsigned helm_threads(const tc_ctx *c, int lpt) { return c->nthm % 2 == 0 ? 128 * lpt : FT_N; }
static long long helm_tiles(const tc_ctx *c, int lpt) {
  return (long long)((c->nthm + FT_I - 1) / FT_I) * ((c->nzm + FT_J * lpt - 1) / (FT_J * lpt));
}

// r segments of the fused front over n instances of this shape.  A launch
// takes (rounds of resident blocks) x (planes per segment and about four for
// what a segment stages before its first and for its start), and its blocks,
// which run apart, end within about a sixth of a segment of each other.  Of
// the counts within 2% of the least of that, the largest, of at least two
// planes each; up to 128 planes one segment where no count saves 2.5% (longer
// ones drift apart, and tiles no longer find their neighbours' halo rows in
// cache).  Measured us, one segment / the count taken (with the correction
// from the second pair on): 64x64x65 133 / 16, 256x256x193 553 / 207 and 810 /
// 303, 512x512x385 1912 / 1632 and 2728 / 2465, 1024x1024x769 14082 / 12488
// and 20394 / 18653; one is the best where the tiles fill the device and there
// are few planes (two: 512x512x97 412 / 428 and 614 / 631, 512x512x65 281 /
// 330 and 414 / 502).  Over 30 sizes it is at most 3.4% over the best count.
static int helm_segments(const tc_ctx *c, int lpt, bool corr, int n) {
  const long long tiles = n * helm_tiles(c, lpt), slots = c->helm_slots[c->masks_uniform_one][corr];
  auto cost = [&](int s) {
    const long long len = (c->nrm + s - 1) / s, rounds = (tiles * s + slots - 1) / slots;
    return 32 * rounds * (len + 4) + 5 * len;
  };
  const int most = std::max(c->nrm / 2, 1);
  long long least = cost(1);
  for (int s = 2; s <= most; s++) least = std::min(least, cost(s));
  if (c->nrm <= 128 && 40 * least > 39 * cost(1)) return 1;
  int s = most;
  while (50 * cost(s) > 51 * least) s--;
  return s;
}

// Fused path: right-hand sides of q_theta -> rhs, q_r -> dq, q_z -> qcap (the
// explicit terms stay in registers, so those fields serve as scratch).
template <bool U, int LPT, bool CORR>
static void launch_rhs(tc_ctx *c, const double *pr, const CorrIn &ci, double *pr_out) {
  const int ntx = (c->nthm + FT_I - 1) / FT_I, ntz = (c->nzm + FT_J * LPT - 1) / (FT_J * LPT);
  const int nseg = helm_segments(c, LPT, CORR, 1);
  auto *kernel = c->nthm % 2 == 0 ? k_helm_rhs<U, LPT, CORR, true> : k_helm_rhs<U, LPT, false, false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(ntx * ntz * nseg)), dim3(helm_threads(c, LPT)), 0,
                     c->stream, c->gd, imp_args(c), c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], pr,
                     c->f[TC_RU1], c->f[TC_RU2], c->f[TC_RU3], c->f[TC_RHS], c->f[TC_DQ],
                     c->f[TC_QCAP], c->mask, c->mask + c->P, rhs_rows(c, c->ns), ntx, ntz, nseg,
                     ci, c->f[TC_DPH], pr_out);
}

// blocks of the fused front that one compute unit holds (asked once: every
// device this library is built for is alike)
template <bool UNIFORM, int LPT, bool CORR, bool PAIR>
static int resident_blocks(int cus) {
  static const int per_cu = [] {
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &n, k_helm_rhs<UNIFORM, LPT, CORR, PAIR>, PAIR ? 128 * LPT : FT_N, 0);
    return e == hipSuccess && n > 0 ? n : 2;
  }();
  return per_cu * cus;
}

// Schedule of the fused front (lpt 0: chosen here) and its blocks resident
// at once.  Even nthm, the pair form: tiles of 4*lpt rows; eight rows stage
// 1.29 elements per point instead of 1.55 and are the faster at every size
// (us, four / eight, with the correction from the second on: 64x64x65 17.1 /
// 16.9, 128x128x97 52.9 / 49.7, 192x128x129 90 / 82, 256x256x193 358 / 313,
// 512x512x385 2688 / 2558).  Odd nthm: lpt lines per thread, two where their
// tiles fill the device in segments of 32 planes (375x240x151 362 / 336).
void choose_helm_schedule(tc_ctx *c, int lpt) {
  int dev = 0, cus = 0;
  hipGetDevice(&dev);
  hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (cus <= 0) cus = 256;
  const bool pair = c->nthm % 2 == 0;
  if (lpt == 0)
    lpt = pair || helm_tiles(c, 2) * (c->nrm / 32) >= resident_blocks<true, 2, false, false>(cus) ? 2 : 1;
  c->helm_lpt = lpt;
  auto ask = [&](auto uniform, int *slots) {
    constexpr bool U = decltype(uniform)::value;
    if (pair) {
      slots[0] = lpt == 2 ? resident_blocks<U, 2, false, true>(cus) : resident_blocks<U, 1, false, true>(cus);
      slots[1] = lpt == 2 ? resident_blocks<U, 2, true, true>(cus) : resident_blocks<U, 1, true, true>(cus);
    } else {
      slots[0] = slots[1] =
          lpt == 2 ? resident_blocks<U, 2, false, false>(cus) : resident_blocks<U, 1, false, false>(cus);
    }
  };
  ask(std::false_type{}, c->helm_slots[0]);
  ask(std::true_type{}, c->helm_slots[1]);
}

void launch_helmholtz_fused(tc_ctx *c) {
  timer_begin(c, "helm_fwd");
  const CorrIn ci{};
  if (c->masks_uniform_one) {
    if (c->helm_lpt == 2) launch_rhs<true, 2, false>(c, c->f[TC_PR], ci, nullptr);
    else launch_rhs<true, 1, false>(c, c->f[TC_PR], ci, nullptr);
  } else {
    if (c->helm_lpt == 2) launch_rhs<false, 2, false>(c, c->f[TC_PR], ci, nullptr);
    else launch_rhs<false, 1, false>(c, c->f[TC_PR], ci, nullptr);
  }
  timer_end(c);
  timer_begin(c, "helm_bwd");
  launch_solve<true>(c, solve_io(c), 0, 3);
  timer_end(c);
}

// The same with the previous substep's pressure correction (dph, al_prev)
// applied while staging: the velocity fields hold that substep's uncorrected
// velocity, pr_in its uncorrected pressure; the corrected pressure goes to
// pr_out (a different array: neighbouring tiles still read pr_in).
void launch_helmholtz_fused_corr(tc_ctx *c, const double *pr_in, double *pr_out, double al_prev) {
  timer_begin(c, "helm_fwd_corr");
  const CorrIn ci{c->dt, al_prev, c->beta};
  if (c->masks_uniform_one) {
    if (c->helm_lpt == 2) launch_rhs<true, 2, true>(c, pr_in, ci, pr_out);
    else launch_rhs<true, 1, true>(c, pr_in, ci, pr_out);
  } else {
    if (c->helm_lpt == 2) launch_rhs<false, 2, true>(c, pr_in, ci, pr_out);
    else launch_rhs<false, 1, true>(c, pr_in, ci, pr_out);
  }
  timer_end(c);
  timer_begin(c, "helm_bwd");
  launch_solve<true>(c, solve_io(c), 0, 3);
  timer_end(c);
}

// ---------------------------------------------------------------------------
// Divergence and projection updates, one point per thread
// ---------------------------------------------------------------------------

DEVI double divergence_at(const GridDev &g, const double *__restrict__ qt,
                          const double *__restrict__ qr, const double *__restrict__ qz, int kc,
                          int j, int i) {
  // CalcLocalDivergence.F90:33-35 (also CheckDivergence.F90:34-36)
  const int ip = wrap_p(i, g.nthm), jp = wrap_p(j, g.nzm);
  const long long o = IX(g, kc, j, i);
  return ((qt[IX(g, kc, j, ip)] - qt[o]) * g.dxt + (qr[o + g.P] - qr[o]) * g.udx2m[kc]) * g.usrm[kc] +
         (qz[IX(g, kc, jp, i)] - qz[o]) * g.dxz;
}

__global__ __launch_bounds__(256) void k_divergence(GridDev g, const double *__restrict__ qt,
                                                    const double *__restrict__ qr,
                                                    const double *__restrict__ qz,
                                                    double *__restrict__ dph, double usdt) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.nthm || j >= g.nzm) return;
  const int kc = blockIdx.z + 1;
  dph[IX(g, kc, j, i)] = divergence_at(g, qt, qr, qz, kc, j, i) * usdt;
}

void launch_divergence(tc_ctx *c, double usdt) {
  timer_begin(c, "divergence");
  hipLaunchKernelGGL(k_divergence, point_grid(c, c->nrm), dim3(64, 4), 0, c->stream, c->gd,
                     c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], c->f[TC_DPH], usdt);
  timer_end(c);
}

// CorrectVelocity.F90:32-40 (qr walls zeroed by k_zero_wall_qr)
DEVI void correct_velocity_at(const GridDev &g, double *__restrict__ qt, double *__restrict__ qr,
                              double *__restrict__ qz, const double *__restrict__ dph, int kc,
                              int j, int i, double dt, double al) {
  const int im = wrap_m(i, g.nthm), jm = wrap_m(j, g.nzm);
  const int km = kc > 1 ? kc - 1 : 1;
  const long long o = IX(g, kc, j, i);
  const double locdph = dph[o];
  qt[o] = qt[o] - (locdph - dph[IX(g, kc, j, im)]) * dt * al * g.dxt * g.usrm[kc];
  qr[o] = qr[o] - (locdph - dph[IX(g, km, j, i)]) * dt * al * g.rudx2c[kc];
  qz[o] = qz[o] - (locdph - dph[IX(g, kc, jm, i)]) * al * dt * g.dxz;
}

// CorrectPressure.F90:37-46 (amm = apph, be = beta)
DEVI void correct_pressure_at(const GridDev &g, double *__restrict__ pr,
                              const double *__restrict__ dph, int kc, int j, int i, double be) {
  const int ip = wrap_p(i, g.nthm), im = wrap_m(i, g.nthm);
  const int jp = wrap_p(j, g.nzm), jm = wrap_m(j, g.nzm);
  const int kp = kc < g.nrm ? kc + 1 : g.nrm, km = kc > 1 ? kc - 1 : 1;
  const double amm = g.apph[kc], acc = g.acph[kc], app = g.apph[kc];
  const long long o = IX(g, kc, j, i);
  const double d0 = dph[o];
  pr[o] = pr[o] + d0 -
          be * ((dph[IX(g, kc, j, ip)] - 2.0 * d0 + dph[IX(g, kc, j, im)]) * g.udx1qm[kc] +
                (dph[IX(g, kc, jp, i)] - 2.0 * d0 + dph[IX(g, kc, jm, i)]) * g.dxzq +
                (dph[IX(g, kp, j, i)] * app + d0 * acc + dph[IX(g, km, j, i)] * amm));
}

__global__ __launch_bounds__(256) void k_correct_velocity(GridDev g, double *__restrict__ qt,
                                                          double *__restrict__ qr,
                                                          double *__restrict__ qz,
                                                          const double *__restrict__ dph,
                                                          double dt, double al) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.nthm || j >= g.nzm) return;
  correct_velocity_at(g, qt, qr, qz, dph, blockIdx.z + 1, j, i, dt, al);
}

__global__ __launch_bounds__(256) void k_correct_pressure(GridDev g, double *__restrict__ pr,
                                                          const double *__restrict__ dph,
                                                          double be) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.nthm || j >= g.nzm) return;
  correct_pressure_at(g, pr, dph, blockIdx.z + 1, j, i, be);
}

__global__ __launch_bounds__(256) void k_correct_both(GridDev g, double *__restrict__ qt,
                                                      double *__restrict__ qr,
                                                      double *__restrict__ qz,
                                                      double *__restrict__ pr,
                                                      const double *__restrict__ dph, double dt,
                                                      double al, double be) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.nthm || j >= g.nzm) return;
  const int kc = blockIdx.z + 1;
  correct_velocity_at(g, qt, qr, qz, dph, kc, j, i, dt, al);
  correct_pressure_at(g, pr, dph, kc, j, i, be);
  if (kc == 1) qr[IX(g, 1, j, i)] = 0.0;
  if (kc == g.nrm) qr[IX(g, g.nr, j, i)] = 0.0;
}

// CorrectVelocity + CorrectPressure + the qr wall reset on a theta pair
// (nthm even): one lane owns points i, i+1 (i even) and moves them as 16-byte
// loads and stores; the arithmetic per point is that of correct_velocity_at
// and correct_pressure_at.
DEVI void correct_pair(const GridDev &g, double *__restrict__ qt, double *__restrict__ qr,
                       double *__restrict__ qz, double *__restrict__ pr,
                       const double *__restrict__ dph, int kc, int j, int i, double dt, double al,
                       double be) {
  // no FMA contraction: every caller (plain and grouped) rounds the same way
#pragma clang fp contract(off)
  const int im = wrap_m(i, g.nthm), ip = wrap_p(i + 1, g.nthm);
  const int jp = wrap_p(j, g.nzm), jm = wrap_m(j, g.nzm);
  const int kp = kc < g.nrm ? kc + 1 : g.nrm, km = kc > 1 ? kc - 1 : 1;
  const long long o = IX(g, kc, j, i);
  auto ld2 = [](const double *a, long long x) { return *reinterpret_cast<const double2 *>(a + x); };
  auto st2 = [](double *a, long long x, double u, double v) {
    *reinterpret_cast<double2 *>(a + x) = make_double2(u, v);
  };
  const double2 d = ld2(dph, o), djm = ld2(dph, IX(g, kc, jm, i)), djp = ld2(dph, IX(g, kc, jp, i));
  const double2 dkm = ld2(dph, IX(g, km, j, i)), dkp = ld2(dph, IX(g, kp, j, i));
  const double dim_ = dph[IX(g, kc, j, im)], dip = dph[IX(g, kc, j, ip)];
  const double2 t = ld2_nt(qt + o), r = ld2_nt(qr + o), z = ld2_nt(qz + o), p = ld2_nt(pr + o);
  // CorrectVelocity.F90:32-40
  st2_nt(qt + o, corr_qt(g, kc, t.x, d.x, dim_, dt, al), corr_qt(g, kc, t.y, d.y, d.x, dt, al));
  st2_nt(qr + o, corr_qr(g, kc, r.x, d.x, dkm.x, dt, al), corr_qr(g, kc, r.y, d.y, dkm.y, dt, al));
  st2_nt(qz + o, corr_qz(g, z.x, d.x, djm.x, dt, al), corr_qz(g, z.y, d.y, djm.y, dt, al));
  // CorrectPressure.F90:37-46 (be = beta)
  st2_nt(pr + o, corr_pr(g, kc, p.x, d.x, dim_, d.y, djm.x, djp.x, dkm.x, dkp.x, be),
      corr_pr(g, kc, p.y, d.y, d.x, dip, djm.y, djp.y, dkm.y, dkp.y, be));
  // CorrectVelocity.F90:46-47
  if (kc == 1) st2(qr, IX(g, 1, j, i), 0.0, 0.0);
  if (kc == g.nrm) st2(qr, IX(g, g.nr, j, i), 0.0, 0.0);
}

__global__ __launch_bounds__(256) void k_correct_both2(GridDev g, double *__restrict__ qt,
                                                       double *__restrict__ qr,
                                                       double *__restrict__ qz,
                                                       double *__restrict__ pr,
                                                       const double *__restrict__ dph, double dt,
                                                       double al, double be) {
  const int i = 2 * (blockIdx.x * 64 + threadIdx.x);
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.nthm || j >= g.nzm) return;
  correct_pair(g, qt, qr, qz, pr, dph, blockIdx.z + 1, j, i, dt, al, be);
}

// Grouped, theta pairs: blockIdx.z = instance * nrm + plane.
__global__ __launch_bounds__(256) void k_correct_both2_g(const StepDesc *__restrict__ tab, int nrm) {
  const int inst = blockIdx.z / nrm, kc = blockIdx.z - inst * nrm + 1;
  const StepDesc &d = tab[inst];
  if (inst_stopped(d)) return;
  const int i = 2 * (blockIdx.x * 64 + threadIdx.x);
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= d.g.nthm || j >= d.g.nzm) return;
  correct_pair(glob(d.g), glob(d.f[TC_QT]), glob(d.f[TC_QR]), glob(d.f[TC_QZ]), glob(d.f[TC_PR]),
               glob(d.f[TC_DPH]), kc, j, i, d.dt, d.al, d.beta);
}

// Grouped: blockIdx.z = instance * nrm + plane.
__global__ __launch_bounds__(256) void k_correct_both_g(const StepDesc *__restrict__ tab, int nrm) {
  const int inst = blockIdx.z / nrm, kc = blockIdx.z - inst * nrm + 1;
  const StepDesc &d = tab[inst];
  if (inst_stopped(d)) return;
  const GridDev g = glob(d.g);
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.nthm || j >= g.nzm) return;
  double *qr = glob(d.f[TC_QR]);
  correct_velocity_at(g, glob(d.f[TC_QT]), qr, glob(d.f[TC_QZ]), glob(d.f[TC_DPH]), kc, j, i, d.dt,
                      d.al);
  correct_pressure_at(g, glob(d.f[TC_PR]), glob(d.f[TC_DPH]), kc, j, i, d.beta);
  if (kc == 1) qr[IX(g, 1, j, i)] = 0.0;
  if (kc == g.nrm) qr[IX(g, g.nr, j, i)] = 0.0;
}

// qr(1,:,:) = qr(nr,:,:) = 0 (CorrectVelocity.F90:46-47)
__global__ void k_zero_wall_qr(GridDev g, double *__restrict__ qr) {
  const long long l = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= g.P) return;
  qr[l] = 0.0;
  qr[(long long)(g.nr - 1) * g.P + l] = 0.0;
}

void launch_correct_velocity(tc_ctx *c, double aldt_al) {
  timer_begin(c, "correct_velocity");
  hipLaunchKernelGGL(k_correct_velocity, point_grid(c, c->nrm), dim3(64, 4), 0, c->stream, c->gd,
                     c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], c->f[TC_DPH], c->dt, aldt_al);
  timer_end(c);
  launch_zero_wall_qr(c);
}
void launch_correct_pressure(tc_ctx *c) {
  timer_begin(c, "correct_pressure");
  hipLaunchKernelGGL(k_correct_pressure, point_grid(c, c->nrm), dim3(64, 4), 0, c->stream, c->gd,
                     c->f[TC_PR], c->f[TC_DPH], c->beta);
  timer_end(c);
}
void launch_correct_both(tc_ctx *c) {
  timer_begin(c, "correct_both");
  if (c->nthm % 2 == 0)
    hipLaunchKernelGGL(k_correct_both2,
                       dim3((unsigned)((c->nthm / 2 + 63) / 64), (unsigned)((c->nzm + 3) / 4),
                            (unsigned)c->nrm),
                       dim3(64, 4), 0, c->stream, c->gd, c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ],
                       c->f[TC_PR], c->f[TC_DPH], c->dt, c->al, c->beta);
  else
    hipLaunchKernelGGL(k_correct_both, point_grid(c, c->nrm), dim3(64, 4), 0, c->stream, c->gd,
                       c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], c->f[TC_PR], c->f[TC_DPH], c->dt,
                       c->al, c->beta);
  timer_end(c);
}
void launch_zero_wall_qr(tc_ctx *c) {
  hipLaunchKernelGGL(k_zero_wall_qr, dim3(line_blocks(c)), dim3(256), 0, c->stream, c->gd,
                     c->f[TC_QR]);
}

// ---------------------------------------------------------------------------
// Reductions: per-block partials, then one block per value combines them in
// a fixed order, so sums are deterministic run to run.
// ---------------------------------------------------------------------------

constexpr int RED_THREADS = 256;
constexpr int RED_TARGET = 1024;    // blocks of a column reduction that fill the device
constexpr int CDIAG_TARGET = 1536;  // blocks of the fused last correction

template <int NV>
DEVI void block_reduce(double (&v)[NV], const int *ops /*0 sum, 1 max*/, double *out) {
  __shared__ double sh[NV][RED_THREADS / 64];
  // linear thread index: the blocks are 256 x 1 or 64 x 4
  const int t = (int)(threadIdx.y * blockDim.x + threadIdx.x);
  const int lane = t & 63, wid = t >> 6;
#pragma unroll
  for (int q = 0; q < NV; q++) {
    double x = v[q];
    for (int off = 32; off > 0; off >>= 1) {
      const double y = __shfl_xor(x, off, 64);
      x = ops[q] ? fmax(x, y) : x + y;
    }
    if (lane == 0) sh[q][wid] = x;
  }
  __syncthreads();
  if (t == 0) {
#pragma unroll
    for (int q = 0; q < NV; q++) {
      double x = sh[q][0];
      for (int w = 1; w < RED_THREADS / 64; w++) x = ops[q] ? fmax(x, sh[q][w]) : x + sh[q][w];
      out[q] = x;
    }
  }
}

// Point reductions march along r: thread = (j, i) column, k = 1..nrm, so the
// qr(k+1) plane of one step is the qr(k) plane of the next.
// Block blk of nb * nseg owns 256 columns over segment blk / nb of r.
struct Col {
  long long l;
  long long lip, ljp;  // in-plane offsets of (j, i+1) and (j+1, i)
  int k0, k1;          // planes of the segment
  bool ok;
};
DEVI Col column(const GridDev &g, int blk, int nseg) {
  Col c;
  const int nb = (int)((g.P + RED_THREADS - 1) / RED_THREADS), seg = blk / nb;
  c.k0 = seg_first(seg, nseg, g.nrm);
  c.k1 = seg_first(seg + 1, nseg, g.nrm) - 1;
  c.l = (long long)(blk - seg * nb) * RED_THREADS + threadIdx.x;
  c.ok = c.l < g.P;
  const long long l = c.ok ? c.l : 0;
  const int j = (int)(l / g.nthm), i = (int)(l - (long long)j * g.nthm);
  c.lip = (long long)j * g.nthm + wrap_p(i, g.nthm);
  c.ljp = (long long)wrap_p(j, g.nzm) * g.nthm + i;
  return c;
}

// CalcMaxCFL.F90:30-43 (WHICH 0) and CheckDivergence.F90:28-40 (WHICH 1)
template <int WHICH>
DEVI void pointmax_body(const int blk, const int nseg, const GridDev &g, const double *__restrict__ qt,
                        const double *__restrict__ qr, const double *__restrict__ qz,
                        double *__restrict__ part) {
#pragma clang fp contract(off)
  double m[1] = {0.0};
  const Col c = column(g, blk, nseg);
  if (c.ok) {
    double r_c = qr[(long long)(c.k0 - 1) * g.P + c.l];
#pragma unroll 2
    for (int kc = c.k0; kc <= c.k1; kc++) {
      const long long b = (long long)(kc - 1) * g.P;
      const double t_c = qt[b + c.l], t_ip = qt[b + c.lip];
      const double r_kp = qr[b + g.P + c.l];
      const double z_c = qz[b + c.l], z_jp = qz[b + c.ljp];
      double val;
      if (WHICH == 0)
        val = (fabs((t_ip + t_c) * 0.5 * g.dxt * ldk(g.usrm + kc)) +
               fabs((r_kp + r_c) * 0.5 * ldk(g.udx2rm + kc)) + fabs((z_jp + z_c) * 0.5 * g.dxz));
      else
        val = fabs(((t_ip - t_c) * g.dxt + (r_kp - r_c) * ldk(g.udx2m + kc)) * ldk(g.usrm + kc) +
                   (z_jp - z_c) * g.dxz);
      m[0] = fmax(m[0], val);
      r_c = r_kp;
    }
  }
  const int ops[1] = {1};
  block_reduce<1>(m, ops, part + blk);
}

template <int WHICH>
__global__ __launch_bounds__(RED_THREADS) void k_pointmax(GridDev g, const double *__restrict__ qt,
                                                         const double *__restrict__ qr,
                                                         const double *__restrict__ qz,
                                                         double *__restrict__ part, int nseg) {
  pointmax_body<WHICH>(blockIdx.x, nseg, g, qt, qr, qz, part);
}

// Grouped CalcMaxCFL partials: blockIdx.y = instance.
__global__ __launch_bounds__(RED_THREADS) void k_pointmax_cfl_g(const StepDesc *__restrict__ tab,
                                                               int nseg) {
  const StepDesc &d = tab[blockIdx.y];
  if (inst_stopped(d)) return;
  pointmax_body<0>(blockIdx.x, nseg, glob(d.g), glob(d.f[TC_QT]), glob(d.f[TC_QR]), glob(d.f[TC_QZ]),
                   glob(d.red));
}

// CalcTorque.F90:36-45 masked wall sums
__global__ __launch_bounds__(RED_THREADS) void k_torque(GridDev g, const double *__restrict__ qt,
                                                       const unsigned char *__restrict__ icyl,
                                                       const unsigned char *__restrict__ ocyl,
                                                       double virotint, double virotext,
                                                       double del, double deln,
                                                       double *__restrict__ part) {
  double s[2] = {0.0, 0.0};
  const int nrm = g.nrm, nr = g.nr;
  const long long l = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (l < g.P) {
    const double grtlow = ((qt[l + g.P] * g.usrm[2] + qt[l] * g.usrm[1]) * 0.5 - virotint * g.usrc[1]) * del;
    s[0] = grtlow * (double)icyl[l];
    const double grtup = (virotext * g.usrc[nr] - (qt[(long long)(nrm - 2) * g.P + l] * g.usrm[nrm - 1] +
                                                   qt[(long long)(nrm - 1) * g.P + l] * g.usrm[nrm]) * 0.5) * deln;
    s[1] = grtup * (double)ocyl[l];
  }
  const int ops[2] = {0, 0};
  block_reduce<2>(s, ops, part + 2 * blockIdx.x);
}

// CalcVelocityStats.F90:29-48
__global__ __launch_bounds__(RED_THREADS) void k_velstats(GridDev g, const double *__restrict__ qt,
                                                         const double *__restrict__ qr,
                                                         const double *__restrict__ qz,
                                                         double pi, double *__restrict__ part,
                                                         int nseg) {
  double v[6] = {-100.0, -100.0, -100.0, 0.0, 0.0, 0.0};
  const Col c = column(g, blockIdx.x, nseg);
  if (c.ok) {
    double r_c = qr[(long long)(c.k0 - 1) * g.P + c.l];
#pragma unroll 2
    for (int kc = c.k0; kc <= c.k1; kc++) {
      const long long b = (long long)(kc - 1) * g.P;
      const double a = qt[b + c.l], cz = qz[b + c.l];
      const double r_kp = qr[b + g.P + c.l];
      v[0] = fmax(v[0], fabs(a));
      v[1] = fmax(v[1], fabs(r_c));
      v[2] = fmax(v[2], fabs(cz));
      const double t = a + qt[b + c.lip];
      v[3] += t * t * ldk(g.pvol + kc) * pi * 0.25;
      const double u = r_c * ldk(g.usrc + kc) + r_kp * ldk(g.usrc + kc + 1);
      v[4] += u * u * ldk(g.pvol + kc) * pi * 0.25;
      const double w = cz + qz[b + c.ljp];
      v[5] += w * w * ldk(g.pvol + kc) * pi * 0.25;
      r_c = r_kp;
    }
  }
  const int ops[6] = {1, 1, 1, 0, 0, 0};
  block_reduce<6>(v, ops, part + 6 * blockIdx.x);
}

// combine: block q reduces value q over the nb partials (fixed order: strided
// per-thread sums, then a fixed tree)
DEVI void combine_body(const int q, const double *__restrict__ part, int nb, int nv,
                       unsigned opmask, double *__restrict__ out) {
  __shared__ double sh[256];
  const bool mx = (opmask >> q) & 1u;
  double x = mx ? -1.0e308 : 0.0;
  for (int b = threadIdx.x; b < nb; b += 256) {
    const double y = part[(size_t)b * nv + q];
    x = mx ? fmax(x, y) : x + y;
  }
  sh[threadIdx.x] = x;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      const double y = sh[threadIdx.x + w];
      sh[threadIdx.x] = mx ? fmax(sh[threadIdx.x], y) : sh[threadIdx.x] + y;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[q] = sh[0];
}

__global__ __launch_bounds__(256) void k_combine(const double *__restrict__ part, int nb, int nv,
                                                 unsigned opmask, double *__restrict__ out) {
  combine_body(blockIdx.x, part, nb, nv, opmask, out);
}

// Grouped combine: blockIdx.x = value, blockIdx.y = instance; with dyn, only
// instances logging this step.
__global__ __launch_bounds__(256) void k_combine_g(const StepDesc *__restrict__ tab,
                                                   const BatchDyn *__restrict__ dyn, int nb,
                                                   int nv, unsigned opmask) {
  if (dyn && !dyn[blockIdx.y].log) return;
  const StepDesc &d = tab[blockIdx.y];
  if (inst_stopped(d)) return;
  combine_body(blockIdx.x, glob(d.red), nb, nv, opmask, glob(d.red_out));
}

// CalcMaxCFL floor and the fixed-dt guard of main.F90:156,172-173, one
// thread per instance: remember the first step with cfl*dt > CFLMAX.
__global__ void k_cfl_check_g(const StepDesc *__restrict__ tab, const BatchDyn *__restrict__ dyn,
                              BatchRes *__restrict__ res, int n) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const StepDesc &d = tab[q];
  if (inst_stopped(d)) return;
  const double cfl = fmax(1.0e-8, d.red_out[0]);
  res[q].cfl = cfl;
  if (res[q].fail165 == 0 && cfl * d.dt > d.limitcfl) {
    res[q].fail165 = dyn[q].ntime + 1;
    res[q].fail_time = dyn[q].tnew;
  }
}

// Keep the logging pass's values of the instances that logged this step.
__global__ void k_diag_store_g(const StepDesc *__restrict__ tab, const BatchDyn *__restrict__ dyn,
                               BatchRes *__restrict__ res, int n) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n || !dyn[q].log || inst_stopped(tab[q])) return;
  const double *o = tab[q].red_out;
  for (int v = 0; v < 10; v++) res[q].diag[v] = o[v];
  res[q].log_ntime = dyn[q].ntime;
  // main.F90:182,203: 266 when both vmax(1) and vmax(2) exceed VMAX, then
  // 169 (assigned later, so it wins) when max|div| > RESID
  int code = 0;
  if (o[2] > tab[q].limitvel && o[3] > tab[q].limitvel) code = 266;
  if (fabs(o[1]) > tab[q].resid) code = 169;
  if (code && res[q].faillog == 0) {
    res[q].faillog = dyn[q].ntime + 1;
    res[q].faillog_code = code;
    if (res[q].fail165 == 0) res[q].fail_time = dyn[q].tnew;
  }
}

static unsigned red_blocks(const tc_ctx *c) { return (unsigned)((c->P + RED_THREADS - 1) / RED_THREADS); }

// r segments of a column reduction: about four blocks per CU in all, at
// least four planes each.  (One segment: 64x64x65 runs 16 blocks that march
// 65 planes each, 14-18 us a pass over 6 MB.)
static int red_segments(const tc_ctx *c) {
  const int nb = (int)red_blocks(c);
  return std::max(1, std::min(RED_TARGET / nb, c->nrm / 4));
}

size_t reduction_doubles(const tc_ctx *c) {
  const size_t cols = (size_t)((c->nthm / 2 + 63) / 64) * ((c->nzm + 3) / 4);
  return 10 * std::max({(size_t)red_blocks(c), cols, (size_t)RED_TARGET, (size_t)CDIAG_TARGET + cols});
}

// The results go to pinned host memory (coherent), which the host reads
// after the stream has drained: no copy is queued behind the kernel.
void combine_partials(tc_ctx *c, unsigned nb, int nv, unsigned opmask) {
  hipLaunchKernelGGL(k_combine, dim3((unsigned)nv), dim3(256), 0, c->stream, c->red, (int)nb, nv,
                     opmask, c->red_host);
}

void launch_max_cfl(tc_ctx *c) {
  timer_begin(c, "max_cfl");
  const int ns = red_segments(c);
  hipLaunchKernelGGL(k_pointmax<0>, dim3(red_blocks(c) * ns), dim3(RED_THREADS), 0, c->stream, c->gd,
                     c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], c->red, ns);
  combine_partials(c, red_blocks(c) * ns, 1, 1u);
  timer_end(c);
}
void launch_max_div(tc_ctx *c) {
  timer_begin(c, "max_div");
  const int ns = red_segments(c);
  hipLaunchKernelGGL(k_pointmax<1>, dim3(red_blocks(c) * ns), dim3(RED_THREADS), 0, c->stream, c->gd,
                     c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], c->red, ns);
  combine_partials(c, red_blocks(c) * ns, 1, 1u);
  timer_end(c);
}
// ---------------------------------------------------------------------------
// Scratch of the no-allocation entry point tc_check_divergence_noalloc: the
// per-block partials of its divergence reduction live in this fixed device
// array instead of the context's reduction buffer.  Each GPU the library
// runs on holds its own copy, at its own address, until the process ends;
// in host code `scratch` names no device memory, so host code uses only the
// address looked up per device below.  Every block writes its own partial
// before the combine reads it, so nothing in it needs clearing; calls that
// overlap on one GPU race on it.
// ---------------------------------------------------------------------------
constexpr size_t NOALLOC_SCRATCH_DOUBLES = 65536;  // 512 KiB: planes up to 16 Mi points
static __device__ __align__(256) double scratch[NOALLOC_SCRATCH_DOUBLES];

static std::mutex scratch_mu;
static std::map<int, double *> scratch_dev;  // device -> address of scratch there

// The device address of scratch on device dev, looked up once per device
// with that device current.
static int scratch_on(int dev, double **out) {
  std::lock_guard<std::mutex> lock(scratch_mu);
  const auto it = scratch_dev.find(dev);
  if (it != scratch_dev.end()) {
    *out = it->second;
    return 0;
  }
  int cur = -1;
  if (hipGetDevice(&cur) != hipSuccess) return set_error("hipGetDevice failed");
  if (cur != dev && hipSetDevice(dev) != hipSuccess) return set_error("hipSetDevice failed");
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (cur != dev) (void)hipSetDevice(cur);
  if (e != hipSuccess || !ptr) {
    (void)hipGetLastError();
    return set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  }
  scratch_dev[dev] = static_cast<double *>(ptr);
  *out = static_cast<double *>(ptr);
  return 0;
}

int check_divergence_noalloc(tc_ctx *c, double *qmax_dev) {
  const unsigned nb = red_blocks(c);
  if ((size_t)nb > NOALLOC_SCRATCH_DOUBLES)
    return set_error("tc_check_divergence_noalloc: a plane of " + std::to_string(c->P) +
                     " points needs " + std::to_string(nb) + " partials; the fixed scratch holds " +
                     std::to_string(NOALLOC_SCRATCH_DOUBLES) + " (nzm*nthm <= " +
                     std::to_string(NOALLOC_SCRATCH_DOUBLES * RED_THREADS) + ")");
  double *part = nullptr;
  int rc = scratch_on(c->device, &part);
  if (rc) return rc;
  const int ns = red_segments(c);  // nb * ns stays within the larger of nb and RED_TARGET
  hipLaunchKernelGGL(k_pointmax<1>, dim3(nb * ns), dim3(RED_THREADS), 0, c->stream, c->gd,
                     c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], part, ns);
  hipLaunchKernelGGL(k_combine, dim3(1u), dim3(256), 0, c->stream, part, (int)(nb * ns), 1, 1u,
                     qmax_dev);
  return check_launch();
}

void launch_torque(tc_ctx *c) {
  const double del = -1.0 / (c->g.rc[2] - c->g.rc[1]);
  const double deln = -1.0 / (c->g.rc[c->nr] - c->g.rc[c->nrm]);
  hipLaunchKernelGGL(k_torque, dim3(red_blocks(c)), dim3(RED_THREADS), 0, c->stream, c->gd,
                     c->f[TC_QT], c->mask, c->mask + c->P, c->p.virotint, c->p.virotext, del,
                     deln, c->red);
  combine_partials(c, red_blocks(c), 2, 0u);
}
void launch_velocity_stats(tc_ctx *c) {
  const int ns = red_segments(c);
  hipLaunchKernelGGL(k_velstats, dim3(red_blocks(c) * ns), dim3(RED_THREADS), 0, c->stream, c->gd,
                     c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], c->g.pi, c->red, ns);
  combine_partials(c, red_blocks(c) * ns, 6, 7u);
}

// One pass over the velocity for the logging step of main.F90:180-186:
// CalcMaxCFL (CalcMaxCFL.F90:36-39), CheckDivergence (CheckDivergence.F90:34-37),
// CalcVelocityStats (CalcVelocityStats.F90:35-44) and CalcTorque
// (CalcTorque.F90:38-43).  v = cfl, |div|, vmax1..3, rms sums 1..3,
// torque sums inner/outer.
DEVI void diagnostics_body(const int blk, const int nseg, const GridDev &g, const double *__restrict__ qt,
                           const double *__restrict__ qr, const double *__restrict__ qz,
                           const unsigned char *__restrict__ icyl,
                           const unsigned char *__restrict__ ocyl, double virotint,
                           double virotext, double del, double deln, double pi,
                           double *__restrict__ part) {
  // no FMA contraction: the per-point values equal those of the fused
  // correction pass (correct_diag_body) and of the CFL pass bit for bit
#pragma clang fp contract(off)
  double v[10] = {0.0, 0.0, -100.0, -100.0, -100.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  const Col c = column(g, blk, nseg);
  if (c.ok) {
    const long long b0 = (long long)(c.k0 - 1) * g.P;
    double r_c = qr[b0 + c.l], t_prev = c.k0 > 1 ? qt[b0 - g.P + c.l] : 0.0;
    for (int kc = c.k0; kc <= c.k1; kc++) {
      const long long b = (long long)(kc - 1) * g.P;
      const double t_c = qt[b + c.l], t_ip = qt[b + c.lip];
      const double r_kp = qr[b + g.P + c.l];
      const double z_c = qz[b + c.l], z_jp = qz[b + c.ljp];
      const double cfl = (fabs((t_ip + t_c) * 0.5 * g.dxt * ldk(g.usrm + kc)) +
                          fabs((r_kp + r_c) * 0.5 * ldk(g.udx2rm + kc)) + fabs((z_jp + z_c) * 0.5 * g.dxz));
      const double dv = ((t_ip - t_c) * g.dxt + (r_kp - r_c) * ldk(g.udx2m + kc)) * ldk(g.usrm + kc) + (z_jp - z_c) * g.dxz;
      v[0] = fmax(v[0], cfl);
      v[1] = fmax(v[1], fabs(dv));
      v[2] = fmax(v[2], fabs(t_c));
      v[3] = fmax(v[3], fabs(r_c));
      v[4] = fmax(v[4], fabs(z_c));
      const double t = t_c + t_ip;
      v[5] += t * t * ldk(g.pvol + kc) * pi * 0.25;
      const double u = r_c * ldk(g.usrc + kc) + r_kp * ldk(g.usrc + kc + 1);
      v[6] += u * u * ldk(g.pvol + kc) * pi * 0.25;
      const double w = z_c + z_jp;
      v[7] += w * w * ldk(g.pvol + kc) * pi * 0.25;
      if (kc == 2) {
        const double grtlow = ((t_c * g.usrm[2] + t_prev * g.usrm[1]) * 0.5 - virotint * g.usrc[1]) * del;
        v[8] += grtlow * (double)icyl[c.l];
      }
      if (kc == g.nrm) {
        const double grtup = (virotext * g.usrc[g.nr] - (t_prev * g.usrm[g.nrm - 1] + t_c * g.usrm[g.nrm]) * 0.5) * deln;
        v[9] += grtup * (double)ocyl[c.l];
      }
      t_prev = t_c;
      r_c = r_kp;
    }
  }
  const int ops[10] = {1, 1, 1, 1, 1, 0, 0, 0, 0, 0};
  block_reduce<10>(v, ops, part + 10 * blk);
}

__global__ __launch_bounds__(RED_THREADS) void k_diagnostics(
    GridDev g, const double *__restrict__ qt, const double *__restrict__ qr,
    const double *__restrict__ qz, const unsigned char *__restrict__ icyl,
    const unsigned char *__restrict__ ocyl, double virotint, double virotext, double del,
    double deln, double pi, double *__restrict__ part, int nseg) {
  diagnostics_body(blockIdx.x, nseg, g, qt, qr, qz, icyl, ocyl, virotint, virotext, del, deln, pi, part);
}

// Grouped logging pass: blockIdx.y = instance; instances not logging this
// step leave at once.
__global__ __launch_bounds__(RED_THREADS) void k_diagnostics_g(const StepDesc *__restrict__ tab,
                                                              const BatchDyn *__restrict__ dyn,
                                                              int nseg) {
  if (!dyn[blockIdx.y].log) return;
  const StepDesc &d = tab[blockIdx.y];
  if (inst_stopped(d)) return;
  diagnostics_body(blockIdx.x, nseg, glob(d.g), glob(d.f[TC_QT]), glob(d.f[TC_QR]), glob(d.f[TC_QZ]),
                   glob(d.icyl), glob(d.ocyl), d.virotint, d.virotext, d.del, d.deln, d.pi,
                   glob(d.red));
}

void launch_diagnostics(tc_ctx *c) {
  const double del = -1.0 / (c->g.rc[2] - c->g.rc[1]);
  const double deln = -1.0 / (c->g.rc[c->nr] - c->g.rc[c->nrm]);
  timer_begin(c, "diagnostics");
  const int ns = red_segments(c);
  hipLaunchKernelGGL(k_diagnostics, dim3(red_blocks(c) * ns), dim3(RED_THREADS), 0, c->stream, c->gd,
                     c->f[TC_QT], c->f[TC_QR], c->f[TC_QZ], c->mask, c->mask + c->P,
                     c->p.virotint, c->p.virotext, del, deln, c->g.pi, c->red, ns);
  combine_partials(c, red_blocks(c) * ns, 10, 0x1Fu);
  timer_end(c);
}

// ---------------------------------------------------------------------------
// End of a logging step in one pass: the last substep's CorrectVelocity +
// CorrectPressure + qr wall reset (the arithmetic of correct_pair) and the
// logging diagnostics of main.F90:180-186 (those of diagnostics_body) on the
// corrected fields, so the diagnostics read nothing from HBM themselves.
// A thread owns a theta pair (i, i+1) of one z row and marches a segment of
// r-planes: dph(k-1), dph(k) come from the previous plane and qr(k+1) is
// loaded once for the two planes that use it.  The corrected neighbours
// qt(i+2) and qz(j+1) are corrected again where they are needed: qt(i+2)
// comes from the next lane where it holds it, else from the raw field.  So
// that every raw read (neighbours, and qr(k+1) across r segments) sees the
// raw value, the corrected velocity goes to the three spare arrays tout,
// rout, zout (the caller then swaps the field pointers); pr is corrected in
// place (no pressure neighbour is read).  Blocks: 64 pairs x 4 rows, one
// segment of r each; per-block partials of the ten diagnostics in part
// (diagnostics_body order).
// ---------------------------------------------------------------------------
DEVI void correct_diag_body(const int bx, const int by, const int seg, const int nseg,
                            const GridDev &g, const double *__restrict__ qt,
                            const double *__restrict__ qr, const double *__restrict__ qz,
                            double *__restrict__ pr, double *__restrict__ tout,
                            double *__restrict__ rout, double *__restrict__ zout,
                            const double *__restrict__ dph, double dt, double al, double be,
                            const unsigned char *__restrict__ icyl,
                            const unsigned char *__restrict__ ocyl, double virotint,
                            double virotext, double del, double deln, double pi,
                            double *__restrict__ part, int blk) {
#pragma clang fp contract(off)
  double v[10] = {0.0, 0.0, -100.0, -100.0, -100.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  const int lane = threadIdx.x;
  const int i = 2 * (bx * 64 + lane);
  const int j = by * 4 + threadIdx.y;
  const bool ok = i < g.nthm && j < g.nzm;
  // the lane whose pair is the next one along theta holds qt(i+2)
  const bool next_in_wave = lane < 63 && i + 2 < g.nthm;
  const int k0 = 1 + (int)(((long long)seg * g.nrm) / nseg);
  const int k1 = (int)(((long long)(seg + 1) * g.nrm) / nseg);
  const int ic = ok ? i : 0, jc = ok ? j : 0;
  const int im = wrap_m(ic, g.nthm), ip = wrap_p(ic + 1, g.nthm);
  const int jp = wrap_p(jc, g.nzm), jm = wrap_m(jc, g.nzm);
  const long long l = (long long)jc * g.nthm + ic;
  const long long lim = (long long)jc * g.nthm + im, lip = (long long)jc * g.nthm + ip;
  const long long ljm = (long long)jm * g.nthm + ic, ljp = (long long)jp * g.nthm + ic;
  auto ld2 = [](const double *a, long long x) { return *reinterpret_cast<const double2 *>(a + x); };
  auto st2 = [](double *a, long long x, double u, double w) {
    *reinterpret_cast<double2 *>(a + x) = make_double2(u, w);
  };
  const long long P = g.P;
  // planes k0-1 and k0 of dph, the raw qr(k0), the corrected qt(k0-1)
  double2 dkm = ld2(dph, (long long)((k0 > 1 ? k0 - 1 : 1) - 1) * P + l);
  double2 d = ld2(dph, (long long)(k0 - 1) * P + l);
  double2 rraw = ld2(qr, (long long)(k0 - 1) * P + l);
  double2 tprev = make_double2(0.0, 0.0);
  if (k0 > 1) {
    const double2 tr = ld2(qt, (long long)(k0 - 2) * P + l);
    const double dimm = dph[(long long)(k0 - 2) * P + lim];
    tprev = make_double2(corr_qt(g, k0 - 1, tr.x, dkm.x, dimm, dt, al),
                         corr_qt(g, k0 - 1, tr.y, dkm.y, dkm.x, dt, al));
  }
  for (int kc = k0; kc <= k1; kc++) {
    const long long b = (long long)(kc - 1) * P;
    const int kp = kc < g.nrm ? kc + 1 : g.nrm;
    const double2 dkp = ld2(dph, (long long)(kp - 1) * P + l);
    const double2 djm = ld2(dph, b + ljm), djp = ld2(dph, b + ljp);
    const double dim_ = dph[b + lim], dip = dph[b + lip];
    const double2 t = ld2(qt, b + l), z = ld2(qz, b + l), p = ld2_nt(pr + b + l);
    // qr(k+1): the wall plane nr is not corrected and ends at zero
    const double2 rnext = ld2(qr, b + P + l);
    const double2 tc = make_double2(corr_qt(g, kc, t.x, d.x, dim_, dt, al),
                                    corr_qt(g, kc, t.y, d.y, d.x, dt, al));
    double2 rc = make_double2(corr_qr(g, kc, rraw.x, d.x, dkm.x, dt, al),
                              corr_qr(g, kc, rraw.y, d.y, dkm.y, dt, al));
    const double2 zc = make_double2(corr_qz(g, z.x, d.x, djm.x, dt, al),
                                    corr_qz(g, z.y, d.y, djm.y, dt, al));
    const double2 pc =
        make_double2(corr_pr(g, kc, p.x, d.x, dim_, d.y, djm.x, djp.x, dkm.x, dkp.x, be),
                     corr_pr(g, kc, p.y, d.y, d.x, dip, djm.y, djp.y, dkm.y, dkp.y, be));
    if (ok) {
      st2_nt(tout + b + l, tc.x, tc.y);
      // CorrectVelocity.F90:46-47: qr(1) = qr(nr) = 0
      if (kc == 1)
        st2_nt(rout + b + l, 0.0, 0.0);
      else
        st2_nt(rout + b + l, rc.x, rc.y);
      st2_nt(zout + b + l, zc.x, zc.y);
      st2_nt(pr + b + l, pc.x, pc.y);
      if (kc == g.nrm) {
        // the plane k = nr: qr's wall, and the unused plane of qt and qz
        // carried over as it was
        const long long bn = (long long)g.nrm * P + l;
        st2_nt(rout + bn, 0.0, 0.0);
        const double2 tw = ld2(qt, bn), zw = ld2(qz, bn);
        st2_nt(tout + bn, tw.x, tw.y);
        st2_nt(zout + bn, zw.x, zw.y);
      }
    }
    {
      if (kc == 1) rc = make_double2(0.0, 0.0);
      // corrected neighbours: qr(k+1) (zero at the wall nr), qt(i+2), qz(j+1)
      double2 rkp = make_double2(0.0, 0.0);
      if (kc < g.nrm)
        rkp = make_double2(corr_qr(g, kc + 1, rnext.x, dkp.x, d.x, dt, al),
                           corr_qr(g, kc + 1, rnext.y, dkp.y, d.y, dt, al));
      double tn = __shfl_down(tc.x, 1, 64);
      if (!next_in_wave) tn = corr_qt(g, kc, qt[b + lip], dip, d.y, dt, al);
      const double2 zr = ld2(qz, b + ljp);
      const double2 zn = make_double2(corr_qz(g, zr.x, djp.x, d.x, dt, al),
                                      corr_qz(g, zr.y, djp.y, d.y, dt, al));
      if (ok) {
        const double tt[2] = {tc.x, tc.y}, tip[2] = {tc.y, tn};
        const double rr[2] = {rc.x, rc.y}, rp[2] = {rkp.x, rkp.y};
        const double zz[2] = {zc.x, zc.y}, zp[2] = {zn.x, zn.y};
        const double tpv[2] = {tprev.x, tprev.y};
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const double t_c = tt[e], t_ip = tip[e], r_c = rr[e], r_kp = rp[e], z_c = zz[e],
                       z_jp = zp[e];
          const double cfl = (fabs((t_ip + t_c) * 0.5 * g.dxt * ldk(g.usrm + kc)) +
                              fabs((r_kp + r_c) * 0.5 * ldk(g.udx2rm + kc)) + fabs((z_jp + z_c) * 0.5 * g.dxz));
          const double dv =
              ((t_ip - t_c) * g.dxt + (r_kp - r_c) * ldk(g.udx2m + kc)) * ldk(g.usrm + kc) + (z_jp - z_c) * g.dxz;
          v[0] = fmax(v[0], cfl);
          v[1] = fmax(v[1], fabs(dv));
          v[2] = fmax(v[2], fabs(t_c));
          v[3] = fmax(v[3], fabs(r_c));
          v[4] = fmax(v[4], fabs(z_c));
          const double tsum = t_c + t_ip;
          v[5] += tsum * tsum * ldk(g.pvol + kc) * pi * 0.25;
          const double u = r_c * ldk(g.usrc + kc) + r_kp * ldk(g.usrc + kc + 1);
          v[6] += u * u * ldk(g.pvol + kc) * pi * 0.25;
          const double w = z_c + z_jp;
          v[7] += w * w * ldk(g.pvol + kc) * pi * 0.25;
          if (kc == 2) {
            const double grtlow = ((t_c * g.usrm[2] + tpv[e] * g.usrm[1]) * 0.5 - virotint * g.usrc[1]) * del;
            v[8] += grtlow * (double)icyl[l + e];
          }
          if (kc == g.nrm) {
            const double grtup =
                (virotext * g.usrc[g.nr] - (tpv[e] * g.usrm[g.nrm - 1] + t_c * g.usrm[g.nrm]) * 0.5) * deln;
            v[9] += grtup * (double)ocyl[l + e];
          }
        }
      }
      tprev = tc;
    }
    dkm = d;
    d = dkp;
    rraw = rnext;
  }
  const int ops[10] = {1, 1, 1, 1, 1, 0, 0, 0, 0, 0};
  block_reduce<10>(v, ops, part + 10 * blk);
}

__global__ __launch_bounds__(256) void k_correct_diag(
    GridDev g, const double *__restrict__ qt, const double *__restrict__ qr,
    const double *__restrict__ qz, double *__restrict__ pr, double *__restrict__ tout,
    double *__restrict__ rout, double *__restrict__ zout, const double *__restrict__ dph,
    double dt, double al, double be, const unsigned char *__restrict__ icyl,
    const unsigned char *__restrict__ ocyl, double virotint, double virotext, double del,
    double deln, double pi, double *__restrict__ part) {
  // one-dimensional grid of (theta block, z block, r segment) tiles, theta
  // fastest, handed out XCD by XCD so that z-neighbouring tiles share an L2
  // (the rows of a block run unsynchronised: meeting every few planes, so
  // that neighbours' dph and qz are read while still cached, measured no
  // faster)
  const int nbx = (g.nthm / 2 + 63) / 64, nby = (g.nzm + 3) / 4;
  const int blk = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = blk % nbx, by = (blk / nbx) % nby, seg = blk / (nbx * nby);
  correct_diag_body(bx, by, seg, gridDim.x / (nbx * nby), g, qt, qr, qz, pr, tout, rout, zout, dph,
                    dt, al, be, icyl, ocyl, virotint, virotext, del, deln, pi, part, blk);
}

// Segments of r per column: enough blocks for about six per CU (at
// 512x512x385 three segments of 129 planes ran 1.46-1.51 ms against 1.81 ms
// for two and 1.56-1.61 ms for four to twelve) of at least 24 planes
// (256x256x193: 178 us with 8 segments, 195 with 12), or down to four planes
// while there are fewer than two blocks per CU (64x64x65: 19 us with 16
// segments, 24 with 8, 36 with 4), and the partials within the reduction
// buffer (TC_CDIAG_SEG overrides).
int correct_diag_segments(const tc_ctx *c) {
  const long long cols = (long long)((c->nthm / 2 + 63) / 64) * ((c->nzm + 3) / 4);
  static const int env = [] {
    const char *e = std::getenv("TC_CDIAG_SEG");
    return e ? std::atoi(e) : 0;
  }();
  long long s = env > 0 ? env : (CDIAG_TARGET + cols - 1) / cols;
  if (env <= 0) {
    s = std::min<long long>(s, std::max(1, c->nrm / 24));
    if (s * cols < 512) s = std::max<long long>(s, std::min<long long>(512 / cols, c->nrm / 4));
  }
  s = std::min<long long>(s, c->nrm);
  s = std::min<long long>(s, (long long)c->red_cap / (10 * cols));
  return (int)std::max<long long>(s, 1);
}

bool correct_diag_applies(const tc_ctx *c) { return c->nthm % 2 == 0 && c->nrm >= 3; }

// The corrected qt, qr, qz land in the spare arrays rhs, dq, qcap (free at
// the end of a substep), whose pointers then trade places with qt, qr, qz.
void launch_correct_diag(tc_ctx *c) {
  const int nseg = correct_diag_segments(c);
  const dim3 grid((unsigned)(((c->nthm / 2 + 63) / 64) * ((c->nzm + 3) / 4) * nseg));
  const double del = -1.0 / (c->g.rc[2] - c->g.rc[1]);
  const double deln = -1.0 / (c->g.rc[c->nr] - c->g.rc[c->nrm]);
  timer_begin(c, "correct_diag");
  hipLaunchKernelGGL(k_correct_diag, grid, dim3(64, 4), 0, c->stream, c->gd, c->f[TC_QT],
                     c->f[TC_QR], c->f[TC_QZ], c->f[TC_PR], c->f[TC_RHS], c->f[TC_DQ],
                     c->f[TC_QCAP], c->f[TC_DPH], c->dt, c->al, c->beta, c->mask, c->mask + c->P,
                     c->p.virotint, c->p.virotext, del, deln, c->g.pi, c->red);
  std::swap(c->f[TC_QT], c->f[TC_RHS]);
  std::swap(c->f[TC_QR], c->f[TC_DQ]);
  std::swap(c->f[TC_QZ], c->f[TC_QCAP]);
  hipLaunchKernelGGL(k_combine, dim3(10u), dim3(256), 0, c->stream, c->red, (int)grid.x, 10,
                     0x1Fu, c->red_host);
  timer_end(c);
}

// Plain streaming copy of one field (nr planes): the achievable-bandwidth
// reference and the calibration point for hardware byte counters.  One
// 16-byte element per thread over a grid that covers the field once.
__global__ __launch_bounds__(256) void k_copy(const double2 *__restrict__ src,
                                              double2 *__restrict__ dst, long long n2,
                                              const double *__restrict__ s1, double *__restrict__ d1,
                                              long long n) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n2) dst[q] = src[q];
  if (q == 0 && (n & 1)) d1[n - 1] = s1[n - 1];
}

void launch_copy(tc_ctx *c, int dst, int src) {
  timer_begin(c, "copy");
  const long long n2 = c->N / 2;
  const unsigned blocks = (unsigned)((n2 + 255) / 256 > 0 ? (n2 + 255) / 256 : 1);
  hipLaunchKernelGGL(k_copy, dim3(blocks), dim3(256), 0, c->stream, (const double2 *)c->f[src],
                     (double2 *)c->f[dst], n2, c->f[src], c->f[dst], c->N);
  timer_end(c);
}

// Fortran order (1:nr,1:nzm,1:nthm) to and from the device's [r][z][theta],
// for the theta columns i0 .. i0+ni-1, whose nr*nzm values each are
// contiguous in f.  A 32 x 32 (r x theta) tile of one z goes through LDS, so
// both sides move 256-byte runs; bound by HBM (16 bytes a value), behind the
// host copy that feeds it.
constexpr int TP = 32;
template <bool TO_DEVICE>
__global__ __launch_bounds__(256) void k_transpose(double *__restrict__ f, double *__restrict__ d,
                                                   int nr, int nzm, int nthm, int i0, int ni) {
  __shared__ double t[TP][TP + 1];
  const int x = threadIdx.x % TP, y = threadIdx.x / TP, j = blockIdx.z;
  const int ib = blockIdx.x * TP, kb = blockIdx.y * TP;
  auto at_f = [&](int k, int i) { return ((long long)i * nzm + j) * nr + k; };
  auto at_d = [&](int k, int i) { return ((long long)k * nzm + j) * nthm + i0 + i; };
#pragma unroll
  for (int q = 0; q < TP; q += 256 / TP) {
    if (TO_DEVICE) {
      if (kb + x < nr && ib + y + q < ni) t[y + q][x] = f[at_f(kb + x, ib + y + q)];
    } else {
      if (ib + x < ni && kb + y + q < nr) t[y + q][x] = d[at_d(kb + y + q, ib + x)];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < TP; q += 256 / TP) {
    if (TO_DEVICE) {
      if (ib + x < ni && kb + y + q < nr) d[at_d(kb + y + q, ib + x)] = t[x][y + q];
    } else {
      if (kb + x < nr && ib + y + q < ni) f[at_f(kb + x, ib + y + q)] = t[x][y + q];
    }
  }
}

void launch_transpose(tc_ctx *c, bool to_device, double *f, double *d, int i0, int ni) {
  const dim3 grid((unsigned)((ni + TP - 1) / TP), (unsigned)((c->nr + TP - 1) / TP), (unsigned)c->nzm);
  if (to_device)
    hipLaunchKernelGGL(k_transpose<true>, grid, dim3(256), 0, c->stream, f, d, c->nr, c->nzm,
                       c->nthm, i0, ni);
  else
    hipLaunchKernelGGL(k_transpose<false>, grid, dim3(256), 0, c->stream, f, d, c->nr, c->nzm,
                       c->nthm, i0, ni);
}

// STREAM triad a = b + s*c over whole fields, two doubles per thread.
__global__ __launch_bounds__(256) void k_triad(double2 *__restrict__ a, const double2 *__restrict__ b,
                                               const double2 *__restrict__ cc, double s, long long n2,
                                               double *__restrict__ a1, const double *__restrict__ b1,
                                               const double *__restrict__ c1, long long n) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n2) {
    const double2 x = b[q], y = cc[q];
    a[q] = make_double2(x.x + s * y.x, x.y + s * y.y);
  }
  if (q == 0 && (n & 1)) a1[n - 1] = b1[n - 1] + s * c1[n - 1];
}

void launch_triad(tc_ctx *c, int a, int b, int cc, double s) {
  timer_begin(c, "triad");
  const long long n2 = c->N / 2;
  const unsigned blocks = (unsigned)((n2 + 255) / 256 > 0 ? (n2 + 255) / 256 : 1);
  hipLaunchKernelGGL(k_triad, dim3(blocks), dim3(256), 0, c->stream, (double2 *)c->f[a],
                     (const double2 *)c->f[b], (const double2 *)c->f[cc], s, n2, c->f[a], c->f[b],
                     c->f[cc], c->N);
  timer_end(c);
}

// ---------------------------------------------------------------------------
// Grouped launches over the instances of one shape group
// ---------------------------------------------------------------------------

template <bool U, int LPT>
static void launch_rhs_g(tc_ctx *c, const StepDesc *tab, const BatchDyn *dyn, int ns, int n,
                         hipStream_t st, bool corr) {
  const int ntx = (c->nthm + FT_I - 1) / FT_I, ntz = (c->nzm + FT_J * LPT - 1) / (FT_J * LPT);
  const int nseg = helm_segments(c, LPT, corr, n);
  const dim3 grid((unsigned)(ntx * ntz * nseg), (unsigned)n);
  // (a corrected launch has an even nthm, defers_correction)
  auto *kernel = corr ? k_helm_rhs_g<U, LPT, true, true>
                      : (c->nthm % 2 == 0 ? k_helm_rhs_g<U, LPT, false, true>
                                          : k_helm_rhs_g<U, LPT, false, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(helm_threads(c, LPT)), 0, st, tab, dyn, ns, ntx, ntz, nseg);
}

template <bool U>
static void launch_solve_g(const SolveShape s, dim3 grid, hipStream_t st, const tc_ctx *c,
                           const StepDesc *tab, int comp0) {
  const dim3 block(64, (unsigned)s.ns);
  const size_t lds = solve_lds(s, c->nrm);
#define TC_SOLVE(R, CHUNKS) \
  hipLaunchKernelGGL((k_helm_solve_g<R, U, CHUNKS>), grid, block, lds, st, tab, comp0)
  switch (s.rows) {
    case 8: TC_SOLVE(8, false); break;
    case 25: TC_SOLVE(25, false); break;
    case 50: TC_SOLVE(50, false); break;
    default:
      if (s.chunks) TC_SOLVE(100, true);
      else TC_SOLVE(100, false);
  }
#undef TC_SOLVE
}

// corr: every instance's descriptor carries a deferred correction
void launch_helmholtz_fused_g(tc_ctx *c, const StepDesc *tab, const BatchDyn *dyn, int ns, int n,
                              hipStream_t st, bool corr) {
  if (c->masks_uniform_one) {
    if (c->helm_lpt == 2) launch_rhs_g<true, 2>(c, tab, dyn, ns, n, st, corr);
    else launch_rhs_g<true, 1>(c, tab, dyn, ns, n, st, corr);
  } else {
    if (c->helm_lpt == 2) launch_rhs_g<false, 2>(c, tab, dyn, ns, n, st, corr);
    else launch_rhs_g<false, 1>(c, tab, dyn, ns, n, st, corr);
  }
  const SolveShape s = solve_shape(c);
  const unsigned serial = c->lu_serial, ncomp = serial ? 1 : 3;
  const dim3 grid((unsigned)((c->P + 63) / 64), ncomp, (unsigned)n);
  for (int q = 0; q < 3; q += (int)ncomp) {
    if (serial >> q & 1)
      hipLaunchKernelGGL(k_helm_solve_serial_g, dim3(line_blocks(c), (unsigned)n), dim3(256), 0, st,
                         tab, q);
    else if (c->masks_uniform_one)
      launch_solve_g<true>(s, grid, st, c, tab, q);
    else
      launch_solve_g<false>(s, grid, st, c, tab, q);
  }
}

void launch_correct_both_g(tc_ctx *c, const StepDesc *tab, int n, hipStream_t st) {
  if (c->nthm % 2 == 0) {
    const dim3 grid((unsigned)((c->nthm / 2 + 63) / 64), (unsigned)((c->nzm + 3) / 4),
                    (unsigned)(c->nrm * n));
    hipLaunchKernelGGL(k_correct_both2_g, grid, dim3(64, 4), 0, st, tab, c->nrm);
  } else {
    const dim3 grid((unsigned)((c->nthm + 63) / 64), (unsigned)((c->nzm + 3) / 4),
                    (unsigned)(c->nrm * n));
    hipLaunchKernelGGL(k_correct_both_g, grid, dim3(64, 4), 0, st, tab, c->nrm);
  }
}

void launch_cfl_check_g(tc_ctx *c, const StepDesc *tab, const BatchDyn *dyn, BatchRes *res, int n,
                        hipStream_t st) {
  const int ns = red_segments(c);
  const unsigned nb = red_blocks(c) * ns;
  hipLaunchKernelGGL(k_pointmax_cfl_g, dim3(nb, (unsigned)n), dim3(RED_THREADS), 0, st, tab, ns);
  hipLaunchKernelGGL(k_combine_g, dim3(1, (unsigned)n), dim3(256), 0, st, tab,
                     (const BatchDyn *)nullptr, (int)nb, 1, 1u);
  hipLaunchKernelGGL(k_cfl_check_g, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st, tab, dyn, res,
                     n);
}

void launch_diagnostics_g(tc_ctx *c, const StepDesc *tab, const BatchDyn *dyn, BatchRes *res, int n,
                          hipStream_t st) {
  const int ns = red_segments(c);
  const unsigned nb = red_blocks(c) * ns;
  hipLaunchKernelGGL(k_diagnostics_g, dim3(nb, (unsigned)n), dim3(RED_THREADS), 0, st, tab, dyn, ns);
  hipLaunchKernelGGL(k_combine_g, dim3(10, (unsigned)n), dim3(256), 0, st, tab, dyn, (int)nb, 10,
                     0x1Fu);
  hipLaunchKernelGGL(k_diag_store_g, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st, tab, dyn,
                     res, n);
}

}  // namespace tc
