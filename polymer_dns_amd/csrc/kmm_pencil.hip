// Pencil-stage kernels of the KMM channel step (wall-normal direction).
//
// k_pencil_step fuses, per (kx,kz) pencil, the work the reference spreads
// over FFTW_DNS/code/src/dns/main_dns.f90:241-811 and the spectral half of
// vcw3dp: forward Chebyshev transform of the previous step's nonlinear terms
// (solvers.f90:3279-3416), smoothing (main_dns.f90:710-745), nonlin
// (solvers.f90:1497-1572), the scalar and phi/v/omega_y CN/AB2 solves
// (phirhs/solve/penta, main_dns.f90:324-484), the influence-matrix
// correction (main_dns.f90:433-466), the mean-flow solves (uzero,
// solvers.f90:1065-1176), veloc/vort/gradscl and the inverse Chebyshev
// transforms (solvers.f90:2241-2546).  Projections of ``norm`` that couple
// +kz and -kz are applied once per step in the plane stage (they commute
// with every pencil operation); the pencil-local ones are applied here.
// Products are contracted with additions within an expression only, so that
// the step's two forms (a wavefront per four pencils, four wavefronts on them)
// round alike whatever the compiler makes of their surroundings.
#pragma clang fp contract(on)
#include "kmm_kernels.h"
#include "kmm_pencil.h"
#include "kmm_row.h"

namespace kmm {

// ---------------------------------------------------------- 1/d tables --
// d recurrence of eqsolve/pntsolve (solvers.f90:500-553, 931-935) per pencil
// and parity; thread per pencil.
template <int NY>
__global__ void k_tau_tables(int P, int nz, double alpha, double beta, double dyde, double g,
                             const double* __restrict__ wnv, double2* __restrict__ tab) {
  constexpr int L = NY / 2;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  double wn;
  if (wnv) {
    wn = wnv[p];
  } else {
    const int kx = p / nz, kzi = p % nz;
    const int kzs = (kzi < nz / 2) ? kzi : kzi - nz;
    const double kxw = kx * alpha, kzw = kzs * beta;
    wn = kxw * kxw + kzw * kzw + g;
  }
  constexpr int TW = tab_width(NY);
  double2* t = tab + (size_t)p * TW;
  for (int i = 0; i < TW; ++i) t[i] = make_double2(0.0, 0.0);
  // even: m = L
  double a1, a2, a3, b1, b2, b3;
  coef_even<NY>(L, wn, dyde, a1, a2, a3);
  double d = a2;
  t[TW - 1].x = 1.0 / d;
  double dn = d;  // d_{i+1}
  for (int i = L - 1; i >= 1; --i) {
    coef_even<NY>(i, wn, dyde, a1, a2, a3);
    coef_even<NY>(i + 1, wn, dyde, b1, b2, b3);
    d = a2 - a3 * b1 / dn;
    t[i].x = 1.0 / d;
    dn = d;
  }
  // odd: m = L-1
  coef_odd<NY>(L - 1, wn, dyde, a1, a2, a3);
  d = a2;
  t[L - 1].y = 1.0 / d;
  dn = d;
  for (int i = L - 2; i >= 1; --i) {
    coef_odd<NY>(i, wn, dyde, a1, a2, a3);
    coef_odd<NY>(i + 1, wn, dyde, b1, b2, b3);
    d = a2 - a3 * b1 / dn;
    t[i].y = 1.0 / d;
    dn = d;
  }
}


// ------------------------------------------------- Green's functions --
// gfcn (solvers.f90:5-172) with real boundary data: the reference's complex
// data (pt,pt) only scales each pencil's solution by a constant that
// cancels in c1*gf1 + c2*gf2, so the real solution and real influence
// coefficients give the same composite v.
template <int NY>
__global__ __launch_bounds__(PW * 64) void k_green(PencilArgs A, double pb1, double pt1, double pb2, double pt2,
                                                   double2* __restrict__ G1, double2* __restrict__ G2,
                                                   double4* __restrict__ gk) {
  constexpr int L = NY / 2;
  using PF = PFN<NY>;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int p = blockIdx.x * PW + wv;
  if (p >= A.P) return;
  double kx, kz;
  int kxi, kzi;
  pencil_k(A, p, kx, kz, kxi, kzi);
  const double k2 = kx * kx + kz * kz;
  const double2* tH = A.tabH + (size_t)p * tab_width(NY);
  const double2* tP = A.tabP + (size_t)p * tab_width(NY);
  double2 gt[2], gb[2];
  for (int w = 0; w < 2; ++w) {
    const double pb = w ? pb2 : pb1, pt = w ? pt2 : pt1;
    PF z = pf_zero<NY>();
    PF phi = tau_solve<NY>(z, k2 + A.gH, A.dyde, tH, make_double2(pt, 0.0), make_double2(pb, 0.0), 0, lane);
    PF g = tau_solve<NY>(phi, k2, A.dyde, tP, czero(), czero(), 0, lane);
    g = pf_real(g);
    double2* G = (w ? G2 : G1) + (size_t)p * (L + 1);
#pragma unroll
    for (int q = 0; q < PLay<NY>::S; ++q) {
      const int gi = q * WAVE + lane;
      if (gi < L) G[gi] = make_double2(g.a[q].x, g.b[q].x);
    }
    if (lane == 0) G[L] = make_double2(g.e.x, 0.0);
    wall_derivs<NY>(g, A.dyde, lane, gt[w], gb[w]);
  }
  if (lane == 0) {
    const double g1b = gb[0].x, g1t = gt[0].x, g2b = gb[1].x, g2t = gt[1].x;
    const double den = g1t * g2b - g2t * g1b;
    // c1 = (vb g2t - vt g2b)/den, c2 = (vt g1b - vb g1t)/den
    gk[p] = make_double4(g2t / den, -g2b / den, -g1t / den, g1b / den);
  }
}

// ----------------------------------------------------------- the step --
// A real Green's function (pairs of values, NY/2 + 1 entries).
// G: the wavefront's first pencil's, o: the row's offset
template <int NY>
__device__ __forceinline__ void green_add(RP<NY>& v, double2 c, const double2* __restrict__ G, unsigned o, int l) {
  constexpr int L = RLay<NY>::L, K = RLay<NY>::K;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const int g = K * l + i;
    if (RLay<NY>::FULL || g < L) {
      const double2 q = G[o + g];
      v.a[i] = cfma(q.x, c, v.a[i]);
      v.b[i] = cfma(q.y, c, v.b[i]);
    }
  }
  v.e = cfma(G[o + L].x, c, v.e);
}

// MODE 0: full step (NL from buffers or FN/GN/SCN), MODE 1: startup
// (derived fields of the current state only), MODE 2: finish (NL -> FN, GN,
// SCN, h1n, h3n).  blk: the block's index along its channel's pencils (16 a
// block, four a wavefront, one per row of 16 lanes: kmm_row.h).
//
// Order: the scalar through to its transfer fields, then omega_y, then v, so
// that at most three pencils and a solve's temporaries are held at a time (two
// wavefronts per SIMD).  All walls are no-slip or moving walls
// (Dirichlet rows, checked by the launch), so the mean-flow solves (uzero,
// solvers.f90:1065-1176) are omega_y's of the (0,0) pencil: u0 and w0 as the
// real and imaginary part of its unknown.  The z-Nyquist pencil computes on
// zeros (norm zeroes it, helpers.f90:149-156).
// The transforms stand in loops that are not unrolled: one copy of their code
// for the nonlinear terms, one for the scalar's and one for the flow's fields.
template <int NY, bool SCALAR, int MODE, typename V>
__device__ __forceinline__ void pencil_body(const PencilArgs& A, int blk) {
  using RL = RLay<NY>;
  using PF = RP<NY>;
  extern __shared__ __align__(16) unsigned char smraw[];
  V* smem = reinterpret_cast<V*>(smraw);
  const V* tw = lds_twiddles<NY, V>(smem, static_cast<const V*>(A.twM));
  const int lane = threadIdx.x & 63, l = lane & 15, row = lane >> 4;
  const unsigned wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double2* wd = reinterpret_cast<double2*>(smraw + 2 * NY * sizeof(V)) + (size_t)wv * RPW * RL::BUF;
  V* w = reinterpret_cast<V*>(wd);          // the wavefront's lines in the transfer precision
  const unsigned P = (unsigned)A.P, p0 = (unsigned)(blk * RWV + wv) * RPW;
  constexpr unsigned TW = tab_width(NY);
  const unsigned rt = row * TW;             // the row's table entries from the wavefront's first
  V* const* TT = reinterpret_cast<V* const*>(A.T);
  V* const* TPD = reinterpret_cast<V* const*>(A.TPD);
  double kx, kz;
  int kxi, kzi;
  pencil_k(A, (int)p0 + row, kx, kz, kxi, kzi);
  const double k2 = kx * kx + kz * kz;
  const bool is00 = (kxi == 0 && kzi == 0), nyq = (kzi == A.nzh);
  const double dy = A.dyde, th = A.theta;
  const bool fromNL = MODE == 2 || (MODE == 0 && A.first_nl);
  const double sz = A.smooth ? A.smz[kzi] : 1.0;
  using RV = RowRaw<NY, V>;
  using RD = RowRaw<NY, double2>;
  // a nonlinear term's coefficients
  auto term = [&](const void* F, const double2* TF) -> PF {
    RV q;
    rows_fetch<NY, V>(q, static_cast<const V*>(F), P, p0, lane);
    PF h = rows_to_cheb<NY, V>(q, w, tw, lane);
    if (TF) h = pf_add(h, pm_load<NY>(TF, p0, wd, lane));  // subforce (helpers.f90:564-606), before smoothing
    if (A.smooth) r_smooth<NY>(h, A.smy, sz, l);
    rp_mask_imag(h, is00);
    rp_mask(h, nyq);
    return h;
  };

  // ---------------- scalar (main_dns.f90:324-358) ----------------------
  if (SCALAR) {
    PF sn, sc;
    if (MODE != 1) {
      if (fromNL) {
        sn = term(A.NLS, nullptr);
      } else {
        sn = pm_load<NY>(A.SCN, p0, wd, lane);
        rp_mask(sn, nyq);
      }
    }
    if (MODE == 2) {
      pm_store<NY>(A.SCN, p0, wd, lane, sn);
    } else {
      sc = pm_load<NY>(A.TH, p0, wd, lane);
      rp_mask(sc, nyq);
      if (MODE == 0) {
        RD qm;
        pm_fetch<NY>(qm, A.SCNM1, p0, lane);
        PF rhs = r_cderiv<NY>(r_cderiv<NY>(sc, dy, l), dy, l);
        PF old = pm_take<NY>(qm, wd, lane);
        rp_mask(old, nyq);
        rhs = r_phirhs(sc, rhs, sn, old, k2, A.re, A.diff, A.dt, th);
        pm_store<NY>(A.SCNM1, p0, wd, lane, sn);
        sc = r_solve<NY, true>(rhs, k2 + A.gS, dy, A.tabS + (size_t)p0 * TW, rt, czero(), czero(), l);
        rp_mask_imag(sc, is00);
        pm_store<NY>(A.TH, p0, wd, lane, sc);
      }
#pragma unroll 1
      for (int j = 0; j < 3; ++j) {
        PF o = pf_imul(sc, j == 0 ? kx : kz);
        if (j == 1) o = r_cderiv<NY>(sc, dy, l);
        cheb_to_rows<NY, V>(o, w, tw, lane, TT[6 + j], P, p0);
      }
    }
  }

  // ---------------- nonlinear terms -> fn, gn (spectral) ---------------
  // nonlin (solvers.f90:1497-1572); gn of the (0,0) pencil: the mean terms
  // h1 + i h3 (main_dns.f90:748-751)
  PF fn, gn;
  if (MODE != 1) {
    if (fromNL) {
#pragma unroll 1
      for (int j = 0; j < 3; ++j) {
        const PF h = term(j == 0 ? A.NL1 : j == 1 ? A.NL3 : A.NL2, j == 0 ? A.TF[0] : j == 1 ? A.TF[2] : A.TF[1]);
        if (j == 0) {
          fn = pf_imul(h, kx);
          gn = pf_imul(h, kz);
          if (is00) gn = h;
        } else if (j == 1) {
          fn = pf_add(fn, pf_imul(h, kz));
          gn = pf_sub(gn, pf_imul(h, is00 ? -1.0 : kx));
        } else {
          fn = pf_sub(pf_scale(h, -k2), r_cderiv<NY>(fn, dy, l));
        }
      }
      if (MODE == 2) {
        pm_store<NY>(A.FN, p0, wd, lane, fn);
        if (is00) mean_store<NY>(A.h1n, A.h3n, gn, l);
        rp_mask(gn, is00);
        pm_store<NY>(A.GN, p0, wd, lane, gn);
        return;
      }
    } else {
      fn = pm_load<NY>(A.FN, p0, wd, lane);
      gn = pm_load<NY>(A.GN, p0, wd, lane);
      if (is00) gn = mean_load<NY>(A.h1n, A.h3n, l);
      rp_mask(fn, nyq);
      rp_mask(gn, nyq);
    }
  }

  // ---------------- omega_y and the mean flow, v (main_dns.f90:360-502) --
  PF omy = pm_load<NY>(A.OMY, p0, wd, lane), v;
  rp_mask(omy, nyq || is00);
  if (MODE == 0) {
    {
      RD qg;
      pm_fetch<NY>(qg, A.GNM1, p0, lane);
      if (is00) omy = mean_load<NY>(A.u0, A.w0, l);
      PF rhs = r_cderiv<NY>(r_cderiv<NY>(omy, dy, l), dy, l);
      PF old = pm_take<NY>(qg, wd, lane);
      rp_mask(old, nyq);
      if (is00) {
        old = mean_load<NY>(A.h1nm1, A.h3nm1, l);
        mean_store<NY>(A.h1nm1, A.h3nm1, gn, l);
        mean_store<NY>(A.h1n, A.h3n, gn, l);
      }
      rhs = r_phirhs(omy, rhs, gn, old, k2, A.re, 1.0, A.dt, th);
      rp_mask(gn, is00);
      pm_store<NY>(A.GNM1, p0, wd, lane, gn);
      double2 be = czero(), bo = czero();
      if (is00) {
        be = make_double2(0.5 * (A.gtu + A.gbu), 0.5 * (A.gtw + A.gbw));
        bo = make_double2(0.5 * (A.gtu - A.gbu), 0.5 * (A.gtw - A.gbw));
      }
      omy = r_solve<NY, false>(rhs, k2 + A.gH, dy, A.tabH + (size_t)p0 * TW, rt, be, bo, l);
      if (A.cmf && p0 == 0) {
        // constant mass flux: u0 += f phi, phi = the response to a unit
        // forcing held over the step (rhs -re/theta, homogeneous wall data)
        rhs = rp_zero<NY>();
        if (l == 0) rhs.a[0] = make_double2(-A.re / th, 0.0);
        rhs = r_solve<NY, false>(rhs, k2 + A.gH, dy, A.tabH + (size_t)p0 * TW, rt, czero(), czero(), l);
        const double fc = (A.ubulk - r_bulk<NY>(omy, l)) / r_bulk<NY>(rhs, l);
        if (is00) {
          omy = pf_axpy(fc, rhs, omy);
          if (l == 0) *A.dpdx = *A.dpdx - fc;
        }
      }
      if (is00) mean_store<NY>(A.u0, A.w0, omy, l);
      rp_mask(omy, is00);
      pm_store<NY>(A.OMY, p0, wd, lane, omy);
    }
    RD qf;
    v = pm_load<NY>(A.V, p0, wd, lane);
    pm_fetch<NY>(qf, A.FNM1, p0, lane);
    rp_mask(v, nyq || is00);
    v = pf_axpy(-k2, v, r_cderiv<NY>(r_cderiv<NY>(v, dy, l), dy, l));  // phi
    {
      const PF d = r_cderiv<NY>(r_cderiv<NY>(v, dy, l), dy, l);
      PF old = pm_take<NY>(qf, wd, lane);
      rp_mask(old, nyq || is00);
      v = r_phirhs(v, d, fn, old, k2, A.re, 1.0, A.dt, th);
    }
    pm_store<NY>(A.FNM1, p0, wd, lane, fn);
#pragma unroll 1
    for (int s = 0; s < 2; ++s)  // phi, then v with homogeneous walls
      v = r_solve<NY, false>(v, s ? k2 : k2 + A.gH, dy, (s ? A.tabP : A.tabH) + (size_t)p0 * TW, rt, czero(), czero(), l);
    // influence matrix (main_dns.f90:433-466)
    double2 vt, vb;
    r_wall_derivs<NY>(v, dy, l, vt, vb);
    const double4 g = (A.gk + p0)[row];
    constexpr unsigned GW = NY / 2 + 1;
    green_add<NY>(v, cadd(cscale(vb, g.x), cscale(vt, g.y)), A.G1 + (size_t)p0 * GW, row * GW, l);
    green_add<NY>(v, cadd(cscale(vb, g.z), cscale(vt, g.w)), A.G2 + (size_t)p0 * GW, row * GW, l);
    rp_mask(v, is00 || nyq);
    pm_store<NY>(A.V, p0, wd, lane, v);
  } else {  // startup: the current state, its (0,0) pencils zeroed
    v = pm_load<NY>(A.V, p0, wd, lane);
    if (p0 == 0) {
      rp_mask(v, is00);
      pm_store<NY>(A.V, p0, wd, lane, v);
      PF o = pm_load<NY>(A.OMY, p0, wd, lane);
      rp_mask(o, is00);
      pm_store<NY>(A.OMY, p0, wd, lane, o);
    }
    rp_mask(v, is00 || nyq);
  }

  // ---------------- veloc / vort (solvers.f90:1576-1722) ---------------
  // D u, D v, D w (TPD) only for the velocity-gradient tensor (gradv,
  // derivatives.f90:6-86)
  PF d;
  const double ik2 = 1.0 / k2;
#pragma unroll 1
  for (int j = 0; j < 9; ++j) {
    PF o;
    V* dst;
    switch (j) {
      case 0: o = v; dst = TT[1]; break;
      case 1: o = omy; dst = TT[4]; break;
      case 2: o = r_cderiv<NY>(v, dy, l); dst = TPD[1]; break;
      case 3: case 6: {  // u, w
        const PF dv = r_cderiv<NY>(v, dy, l);
        o = pf_scale(pf_add(pf_imul(dv, j == 3 ? kx : kz), pf_imul(omy, j == 3 ? -kz : kx)), ik2);
        if (is00) {
          const PF m = mean_load<NY>(A.u0, A.w0, l);
          o = j == 3 ? m : pf_imul(m, -1.0);
          rp_mask_imag(o, true);
        }
        d = r_cderiv<NY>(o, dy, l);
        dst = TT[j == 3 ? 0 : 2];
        break;
      }
      case 4: o = d; dst = TPD[0]; break;
      case 5: o = pf_sub(pf_imul(v, kx), d); dst = TT[5]; break;  // omega_z
      case 7: o = d; dst = TPD[2]; break;
      default: o = pf_sub(d, pf_imul(v, kz)); dst = TT[3]; break;  // omega_x
    }
    if (dst) cheb_to_rows<NY, V>(o, w, tw, lane, dst, P, p0);
  }
}

// TV: occupancy variant picked by the autotuner (0: row_waves, 1: one instead
// of two wavefronts per SIMD and two instead of one; 128 x 129 x 128 FP64 0.122
// and 0.151 ms)
template <int NY, bool SCALAR, int MODE, typename V, int TV = 0>
__global__ __launch_bounds__(RWV * 64) __attribute__((amdgpu_waves_per_eu(TV ? 3 - row_waves<NY>() : row_waves<NY>()))) void k_pencil(PencilArgs A) {
  pencil_body<NY, SCALAR, MODE, V>(A, xcd_group(blockIdx.x, gridDim.x));
}

// The step with a block's four wavefronts on the same four pencils, where a
// channel has too few pencils to fill the chip with a wavefront each:
//   wavefront 0  h1; omega_y (and the mean flow); u, omega_z
//   wavefront 1  h2; v; v, D v
//   wavefront 2  h3; w, omega_x
//   wavefront 3  the scalar, or phi and its derivatives for wavefront 1; omega_y
// with block barriers after the nonlinear terms, after fn and gn have been
// formed from them and after the solves; what passes between wavefronts stands
// in LDS as the lanes hold it, omega_y and v in the place of h1 and h3 (at ny =
// 128 that lets two blocks share a CU: 2048 pencils 38 -> 27 us).  Bound by
// the chain of wavefront 1: one transform, two solves, the wall correction, two
// transforms, against the whole step's in pencil_body.
// h1, h3, then omega_y, v; without the scalar phi and D^2 phi beside them
template <int NY, bool SCALAR, typename V>
constexpr size_t team_lds() { return row_lds<NY, V>() + (SCALAR ? 2 : 4) * (size_t)lane_slots<NY>() * sizeof(double2); }
template <int NY, bool SCALAR, typename V>
__device__ __forceinline__ void team_body(const PencilArgs& A, int blk) {
  using RL = RLay<NY>;
  using PF = RP<NY>;
  extern __shared__ __align__(16) unsigned char smraw[];
  V* smem = reinterpret_cast<V*>(smraw);
  const V* tw = lds_twiddles<NY, V>(smem, static_cast<const V*>(A.twM));
  const int lane = threadIdx.x & 63, l = lane & 15, row = lane >> 4;
  const unsigned wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double2* wd = reinterpret_cast<double2*>(smraw + 2 * NY * sizeof(V)) + (size_t)wv * RPW * RL::BUF;
  V* w = reinterpret_cast<V*>(wd);
  double2* X = reinterpret_cast<double2*>(smraw + row_lds<NY, V>()) + lane;
  double2 *XH1 = X, *XH3 = X + lane_slots<NY>(), *XP = X + 2 * lane_slots<NY>(), *XD = X + 3 * lane_slots<NY>();
  double2 *const XO = XH1, *const XV = XH3;  // once these have been read
  const unsigned P = (unsigned)A.P, p0 = (unsigned)blk * RPW;
  constexpr unsigned TW = tab_width(NY);
  const unsigned rt = row * TW;
  V* const* TT = reinterpret_cast<V* const*>(A.T);
  V* const* TPD = reinterpret_cast<V* const*>(A.TPD);
  double kx, kz;
  int kxi, kzi;
  pencil_k(A, (int)p0 + row, kx, kz, kxi, kzi);
  const double k2 = kx * kx + kz * kz;
  const bool is00 = (kxi == 0 && kzi == 0), nyq = (kzi == A.nzh);
  const double dy = A.dyde, th = A.theta;
  const double sz = A.smooth ? A.smz[kzi] : 1.0;
  auto load = [&](const double2* F) -> PF {
    PF h = pm_load<NY>(F, p0, wd, lane);
    rp_mask(h, nyq);
    return h;
  };
  auto phi_parts = [&](PF& phi, PF& d) {
    phi = pm_load<NY>(A.V, p0, wd, lane);
    rp_mask(phi, nyq || is00);
    phi = pf_axpy(-k2, phi, r_cderiv<NY>(r_cderiv<NY>(phi, dy, l), dy, l));
    d = r_cderiv<NY>(r_cderiv<NY>(phi, dy, l), dy, l);
  };

  // nonlinear terms; a wavefront's own in h
  PF h = rp_zero<NY>();
  const bool scal = SCALAR && wv == 3;
  if (A.first_nl && (wv < 3 || scal)) {
    const void* F = wv == 0 ? A.NL1 : wv == 1 ? A.NL2 : wv == 2 ? A.NL3 : A.NLS;
    RowRaw<NY, V> q;
    rows_fetch<NY, V>(q, static_cast<const V*>(F), P, p0, lane);
    h = rows_to_cheb<NY, V>(q, w, tw, lane);
    if (wv < 3 && A.TF[wv]) h = pf_add(h, pm_load<NY>(A.TF[wv], p0, wd, lane));
    if (A.smooth) r_smooth<NY>(h, A.smy, sz, l);
    rp_mask_imag(h, is00);
    rp_mask(h, nyq);
    if (wv == 0) lane_put<NY>(XH1, h);
    if (wv == 2) lane_put<NY>(XH3, h);
  } else if (!SCALAR && wv == 3) {
    PF d;
    phi_parts(h, d);
    lane_put<NY>(XP, h);
    lane_put<NY>(XD, d);
  }
  __syncthreads();
  if (A.first_nl) {  // gn (the (0,0) pencil's: h1 + i h3) and fn from the terms
    if (wv == 0) {
      h = is00 ? h : pf_imul(h, kz);
      h = pf_sub(h, pf_imul(lane_get<NY>(XH3), is00 ? -1.0 : kx));
    } else if (wv == 1) {
      const PF f = pf_add(pf_imul(lane_get<NY>(XH1), kx), pf_imul(lane_get<NY>(XH3), kz));
      h = pf_sub(pf_scale(h, -k2), r_cderiv<NY>(f, dy, l));
    }
  }
  __syncthreads();

  if (wv == 0) {  // omega_y and the mean flow
    PF gn = h;
    if (!A.first_nl) {
      gn = load(A.GN);
      if (is00) gn = mean_load<NY>(A.h1n, A.h3n, l);
    }
    PF omy = load(A.OMY);
    rp_mask(omy, is00);
    if (is00) omy = mean_load<NY>(A.u0, A.w0, l);
    PF rhs = r_cderiv<NY>(r_cderiv<NY>(omy, dy, l), dy, l);
    PF old = load(A.GNM1);
    if (is00) {
      old = mean_load<NY>(A.h1nm1, A.h3nm1, l);
      mean_store<NY>(A.h1nm1, A.h3nm1, gn, l);
      mean_store<NY>(A.h1n, A.h3n, gn, l);
    }
    rhs = r_phirhs(omy, rhs, gn, old, k2, A.re, 1.0, A.dt, th);
    rp_mask(gn, is00);
    pm_store<NY>(A.GNM1, p0, wd, lane, gn);
    double2 be = czero(), bo = czero();
    if (is00) {
      be = make_double2(0.5 * (A.gtu + A.gbu), 0.5 * (A.gtw + A.gbw));
      bo = make_double2(0.5 * (A.gtu - A.gbu), 0.5 * (A.gtw - A.gbw));
    }
    omy = r_solve<NY, false>(rhs, k2 + A.gH, dy, A.tabH + (size_t)p0 * TW, rt, be, bo, l);
    if (A.cmf && p0 == 0) {  // constant mass flux, as in pencil_body
      rhs = rp_zero<NY>();
      if (l == 0) rhs.a[0] = make_double2(-A.re / th, 0.0);
      rhs = r_solve<NY, false>(rhs, k2 + A.gH, dy, A.tabH + (size_t)p0 * TW, rt, czero(), czero(), l);
      const double fc = (A.ubulk - r_bulk<NY>(omy, l)) / r_bulk<NY>(rhs, l);
      if (is00) {
        omy = pf_axpy(fc, rhs, omy);
        if (l == 0) *A.dpdx = *A.dpdx - fc;
      }
    }
    if (is00) mean_store<NY>(A.u0, A.w0, omy, l);
    rp_mask(omy, is00);
    lane_put<NY>(XO, omy);
    pm_store<NY>(A.OMY, p0, wd, lane, omy);
  } else if (wv == 1) {  // phi, v
    PF fn = h;
    if (!A.first_nl) fn = load(A.FN);
    PF v, d;
    if (SCALAR) {
      phi_parts(v, d);
    } else {
      v = lane_get<NY>(XP);
      d = lane_get<NY>(XD);
    }
    {
      PF old = load(A.FNM1);
      rp_mask(old, is00);
      v = r_phirhs(v, d, fn, old, k2, A.re, 1.0, A.dt, th);
    }
    pm_store<NY>(A.FNM1, p0, wd, lane, fn);
#pragma unroll 1
    for (int s = 0; s < 2; ++s)  // phi, then v with homogeneous walls
      v = r_solve<NY, false>(v, s ? k2 : k2 + A.gH, dy, (s ? A.tabP : A.tabH) + (size_t)p0 * TW, rt, czero(), czero(), l);
    double2 vt, vb;
    r_wall_derivs<NY>(v, dy, l, vt, vb);
    const double4 g = (A.gk + p0)[row];
    constexpr unsigned GW = NY / 2 + 1;
    green_add<NY>(v, cadd(cscale(vb, g.x), cscale(vt, g.y)), A.G1 + (size_t)p0 * GW, row * GW, l);
    green_add<NY>(v, cadd(cscale(vb, g.z), cscale(vt, g.w)), A.G2 + (size_t)p0 * GW, row * GW, l);
    rp_mask(v, is00 || nyq);
    lane_put<NY>(XV, v);
    pm_store<NY>(A.V, p0, wd, lane, v);
  } else if (scal) {
    PF sn = h;
    if (!A.first_nl) sn = load(A.SCN);
    PF sc = load(A.TH);
    PF rhs = r_cderiv<NY>(r_cderiv<NY>(sc, dy, l), dy, l);
    PF old = load(A.SCNM1);
    rhs = r_phirhs(sc, rhs, sn, old, k2, A.re, A.diff, A.dt, th);
    pm_store<NY>(A.SCNM1, p0, wd, lane, sn);
    sc = r_solve<NY, true>(rhs, k2 + A.gS, dy, A.tabS + (size_t)p0 * TW, rt, czero(), czero(), l);
    rp_mask_imag(sc, is00);
    pm_store<NY>(A.TH, p0, wd, lane, sc);
#pragma unroll 1
    for (int j = 0; j < 3; ++j) {
      PF o = pf_imul(sc, j == 0 ? kx : kz);
      if (j == 1) o = r_cderiv<NY>(sc, dy, l);
      cheb_to_rows<NY, V>(o, w, tw, lane, TT[6 + j], P, p0);
    }
  }
  __syncthreads();

  // veloc / vort: wavefronts 0 and 2 u and w, their D, omega_z and omega_x;
  // 1 v, D v; 3 omega_y
  const PF v = lane_get<NY>(XV);
  const bool uw = wv == 0 || wv == 2, isu = wv == 0;
  PF o, d;
  if (wv == 1) {
    o = v;
    d = r_cderiv<NY>(v, dy, l);
  } else {
    o = lane_get<NY>(XO);
    if (uw) {
      const double ik2 = 1.0 / k2;
      o = pf_scale(pf_add(pf_imul(r_cderiv<NY>(v, dy, l), isu ? kx : kz), pf_imul(o, isu ? -kz : kx)), ik2);
      if (is00) {
        const PF m = mean_load<NY>(A.u0, A.w0, l);
        o = isu ? m : pf_imul(m, -1.0);
        rp_mask_imag(o, true);
      }
      d = r_cderiv<NY>(o, dy, l);
    }
  }
#pragma unroll 1
  for (int j = 0; j < 3; ++j) {
    V* dst;
    if (j == 0) {
      dst = TT[wv == 3 ? 4 : wv];
    } else if (j == 1) {
      dst = wv == 3 ? nullptr : TPD[wv];
      o = d;
    } else {
      dst = uw ? TT[isu ? 5 : 3] : nullptr;
      o = isu ? pf_sub(pf_imul(v, kx), d) : pf_sub(d, pf_imul(v, kz));
    }
    if (dst) cheb_to_rows<NY, V>(o, w, tw, lane, dst, P, p0);
  }
}

template <int NY, bool SCALAR, typename V>
__global__ __launch_bounds__(RWV * 64) __attribute__((amdgpu_waves_per_eu(row_waves<NY>())))
void k_pencil_team(PencilArgs A) {
  team_body<NY, SCALAR, V>(A, xcd_group(blockIdx.x, gridDim.x));
}

// The step kernel of an ensemble of channels of one size in one launch:
// channel blockIdx.y takes its arguments from AA[blockIdx.y].
template <int NY, bool SCALAR, typename V, int TV>
__global__ __launch_bounds__(RWV * 64) __attribute__((amdgpu_waves_per_eu(TV ? 3 - row_waves<NY>() : row_waves<NY>())))
void k_pencil_batch(const PencilArgs* __restrict__ AA) {
  pencil_body<NY, SCALAR, 0, V>(AA[blockIdx.y], xcd_group(blockIdx.x, gridDim.x));
}

// -------------------------------------------------- parity kernels --
template <int NY>
__global__ __launch_bounds__(PW * 64) void k_cderiv(int P, double dyde, const double2* __restrict__ in,
                                                    double2* __restrict__ out) {
  using PF = PFN<NY>;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int p = blockIdx.x * PW + wv;
  if (p >= P) return;
  PF f = pf_load<NY>(in, P, p, lane);
  pf_store<NY>(out, P, p, lane, cderiv<NY>(f, dyde, lane));
}

// gradv (derivatives.f90:6-86): out[3 i + k] = d u_i / d x_k for i, k in
// x, y, z, out[9 + i] = Laplacian of u_i (D^2 - k^2); wave per pencil
template <int NY>
__global__ __launch_bounds__(PW * 64) void k_gradv(int P, int nz, int nzh, double alpha, double beta, double dyde,
                                                   const double2* __restrict__ u, const double2* __restrict__ v,
                                                   const double2* __restrict__ w, double2* const* __restrict__ out) {
  using PF = PFN<NY>;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int p = blockIdx.x * PW + wv;
  if (p >= P) return;
  const int kxi = p / nz, kzi = p % nz;
  const double kx = kxi * alpha, kz = ((kzi < nzh) ? kzi : kzi - nz) * beta;
  const double k2 = kx * kx + kz * kz;
  const double2* in[3] = {u, v, w};
#pragma unroll 1
  for (int i = 0; i < 3; ++i) {
    const PF f = pf_load<NY>(in[i], P, p, lane);
    const PF d = cderiv<NY>(f, dyde, lane);
    pf_store<NY>(out[3 * i + 0], P, p, lane, pf_imul(f, kx));
    pf_store<NY>(out[3 * i + 1], P, p, lane, d);
    pf_store<NY>(out[3 * i + 2], P, p, lane, pf_imul(f, kz));
    pf_store<NY>(out[9 + i], P, p, lane, pf_axpy(-k2, f, cderiv<NY>(d, dyde, lane)));
  }
}

// Laplacians of u, v, w for inertial particles (gradv's D^2 f - k^2 f,
// derivatives.f90:77-79, normed as in main_dns.f90:556-558) from the state v,
// omega_y, u0, w0 through veloc (u = -(-i kx Dv + i kz omy)/k2,
// w = -(-i kz Dv - i kx omy)/k2; u0, 0, w0 at kx = kz = 0), inverse Chebyshev
// transformed to physical y; one wave per pencil
template <int NY, typename V>
__global__ __launch_bounds__(PW * 64) void k_mr_lap(MrLapArgs A) {
  using PF = PFN<NY>;
  extern __shared__ __align__(16) unsigned char smraw[];
  V* smem = reinterpret_cast<V*>(smraw);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int p = blockIdx.x * PW + wv;
  const V* twl = lds_twiddles<NY, V>(smem, static_cast<const V*>(A.twM));
  if (p >= A.P) return;
  V* buf = wave_lds<NY, V>(smem, wv);
  V* scr = buf + FFTBuf<2 * NY>::len;
  const size_t P = (size_t)A.P;
  double kx, kz;
  int kxi, kzi;
  pencil_k(A, p, kx, kz, kxi, kzi);
  const double k2 = kx * kx + kz * kz;
  const double dy = A.dyde;
  const bool is00 = (kxi == 0 && kzi == 0);
  PF f[3] = {pf_zero<NY>(), pf_zero<NY>(), pf_zero<NY>()};
  if (kzi != A.nzh) {  // norm zeroes the z-Nyquist row
    if (is00) {
      f[0] = pf_load_real<NY>(A.u0, lane);
      f[2] = pf_load_real<NY>(A.w0, lane);
    } else {
      const PF v = pf_load_pm<NY>(A.V, p, lane);
      const PF omy = pf_load_pm<NY>(A.OMY, p, lane);
      const PF dv = cderiv<NY>(v, dy, lane);
      const double ik2 = 1.0 / k2;
      f[0] = pf_scale(pf_sub(pf_imul(dv, kx), pf_imul(omy, kz)), ik2);
      f[1] = v;
      f[2] = pf_scale(pf_add(pf_imul(dv, kz), pf_imul(omy, kx)), ik2);
    }
  }
#pragma unroll 1
  for (int i = 0; i < 3; ++i) {
    PF l = pf_axpy(-k2, f[i], cderiv<NY>(cderiv<NY>(f[i], dy, lane), dy, lane));
    if (is00) l = pf_real(l);
    cheb_to_phys_store<NY, V>(l, buf, scr, twl, lane, static_cast<V*>(A.LT[i]), P, p);
  }
}

// inverse: FP64 spectral in -> V physical-y out; forward: V in -> FP64 out
template <int NY, typename V>
__global__ __launch_bounds__(PW * 64) void k_cheb(int P, const V* __restrict__ tw, const void* in, void* out,
                                                  int inverse) {
  using PF = PFN<NY>;
  extern __shared__ __align__(16) unsigned char smraw[];
  V* smem = reinterpret_cast<V*>(smraw);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int p = blockIdx.x * PW + wv;
  const V* twl = lds_twiddles<NY, V>(smem, tw);
  if (p >= P) return;
  V* buf = wave_lds<NY, V>(smem, wv);
  if (inverse) {  // 2: the spectral input is stored pencil-major
    PF f = inverse == 2 ? pf_load_pm<NY>(static_cast<const double2*>(in), p, lane)
                        : pf_load<NY>(static_cast<const double2*>(in), P, p, lane);
    cheb_to_phys_store<NY, V>(f, buf, buf + FFTBuf<2 * NY>::len, twl, lane, static_cast<V*>(out), P, p);
  } else {
    PF r = phys_to_cheb_load<NY, V>(static_cast<const V*>(in), P, p, buf, buf + FFTBuf<2 * NY>::len, twl, lane);
    pf_store<NY>(static_cast<double2*>(out), P, p, lane, r);
  }
}

template <int NY>
__global__ __launch_bounds__(PW * 64) void k_solve(int P, double dyde, const double2* __restrict__ tab,
                                                   const double* __restrict__ wn, double2* __restrict__ u,
                                                   const double2* __restrict__ bct, const double2* __restrict__ bcb,
                                                   int ib, const int* __restrict__ kzero) {
  using PF = PFN<NY>;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int p = blockIdx.x * PW + wv;
  if (p >= P) return;
  PF f = pf_load<NY>(u, P, p, lane);
  PF r = tau_solve<NY>(f, wn[p], dyde, tab + (size_t)p * tab_width(NY), bct[p], bcb[p], ib, lane);
  if (kzero && kzero[p]) r = pf_zero<NY>();
  pf_store<NY>(u, P, p, lane, r);
}

template <int NY>
__global__ __launch_bounds__(PW * 64) void k_penta(int P, double dyde, const double2* __restrict__ tab,
                                                   const double* __restrict__ wn, double2* __restrict__ u,
                                                   double at, double bt, const double2* __restrict__ gtop,
                                                   double ab, double bb, const double2* __restrict__ gbot,
                                                   double bsign, const int* __restrict__ kzero) {
  using PF = PFN<NY>;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int p = blockIdx.x * PW + wv;
  if (p >= P) return;
  PF f = pf_load<NY>(u, P, p, lane);
  auto tt = [=](int n) -> double { return at + dyde * bt * (double)n * (double)n; };
  auto tb = [=](int n) -> double { double t = ab + bsign * dyde * bb * (double)n * (double)n; return (n & 1) ? -t : t; };
  PF r = tau_penta<NY>(f, wn[p], dyde, tab + (size_t)p * tab_width(NY), tt, tb, gtop[p], gbot[p], lane);
  if (kzero && kzero[p]) r = pf_zero<NY>();
  pf_store<NY>(u, P, p, lane, r);
}

// ------------------------------------------------------------ launchers --
hipError_t launch_tau_tables(int ny, const PencilArgs& a, double g, double2* tab, hipStream_t s) {
  KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_tau_tables<NY>), dim3((a.P + 127) / 128), dim3(128), 0, s, a.P, a.nz,
                                          a.alpha, a.beta, a.dyde, g, (const double*)nullptr, tab));
  return hipGetLastError();
}
hipError_t launch_tau_tables_wn(int ny, int P, double dyde, const double* wn, double2* tab, hipStream_t s) {
  KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_tau_tables<NY>), dim3((P + 127) / 128), dim3(128), 0, s, P, 1, 0.0,
                                          0.0, dyde, 0.0, wn, tab));
  return hipGetLastError();
}
hipError_t launch_green(int ny, const PencilArgs& a, double pb1, double pt1, double pb2, double pt2, double2* G1,
                        double2* G2, double4* gk, hipStream_t s) {
  KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_green<NY>), dim3(nblk(a.P)), dim3(PW * 64), 0, s, a, pb1, pt1, pb2,
                                          pt2, G1, G2, gk));
  return hipGetLastError();
}
// pencils come in blocks of 16 (nx/2 is a multiple of 8, nz even), the walls'
// rows are Dirichlet rows of weight 1
static bool row_ok(const PencilArgs& a) {
  return a.P % (RWV * RPW) == 0 && a.nz % RPW == 0 && a.atu == 1.0 && a.abu == 1.0 && a.atw == 1.0 && a.abw == 1.0 &&
         a.btu == 0.0 && a.bbu == 0.0 && a.btw == 0.0 && a.bbw == 0.0;
}
// Four wavefronts on the same pencils where that leaves the blocks about two
// rounds on the 256 CUs.  Measured, a wavefront per four pencils -> four (us):
//   512 pencils   ny 32 27 -> 12.7
//   2048 pencils  ny 64 34 -> 19 (mixed with scalar 40 -> 22), 128 46 -> 27
//                 (55 -> 30), 192 61 -> 51
//   4608 pencils  ny 48 40 -> 33 (FP64 with scalar 60 -> 48), 64 45 -> 36, 80
//                 mixed with scalar 66 -> 64, 128 73 -> 65, 192 138 -> 133
//   8192 pencils  ny 32 39 -> 43, 48 51 -> 55, 64 51 -> 55, 128 mixed with
//                 scalar 100 -> 123
static bool team_ok(int P) { return P <= 5120; }
template <int MODE, typename V, int TV>
static hipError_t launch_pencil_tv(int ny, const PencilArgs& a, hipStream_t s) {
  if (!row_ok(a)) return hipErrorInvalidValue;
  const dim3 grid(a.P / (RWV * RPW)), block(RWV * 64);
  if (MODE == 0 && TV == 0 && team_ok(a.P)) {
    const dim3 tgrid(a.P / RPW);
    if (a.scalar) {
      KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_pencil_team<NY, true, V>), tgrid, block, (team_lds<NY, true, V>()), s, a));
    } else {
      KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_pencil_team<NY, false, V>), tgrid, block, (team_lds<NY, false, V>()), s, a));
    }
    return hipGetLastError();
  }
  if (a.scalar) {
    KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_pencil<NY, true, MODE, V, TV>), grid, block, (row_lds<NY, V>()), s, a));
  } else {
    KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_pencil<NY, false, MODE, V, TV>), grid, block, (row_lds<NY, V>()), s, a));
  }
  return hipGetLastError();
}
template <int MODE, typename V>
static hipError_t launch_pencil_mode_v(int ny, const PencilArgs& a, hipStream_t s) {
  // only the step kernel has tuning variants
  if (MODE == 0 && a.tune == 1) return launch_pencil_tv<MODE, V, 1>(ny, a, s);
  return launch_pencil_tv<MODE, V, 0>(ny, a, s);
}
template <int MODE>
static hipError_t launch_pencil_mode(int ny, const PencilArgs& a, hipStream_t s) {
  return a.mixed ? launch_pencil_mode_v<MODE, float2>(ny, a, s) : launch_pencil_mode_v<MODE, double2>(ny, a, s);
}
hipError_t launch_pencil_step(int ny, const PencilArgs& a, hipStream_t s) { return launch_pencil_mode<0>(ny, a, s); }

template <typename V, int TV>
static hipError_t launch_pencil_batch_v(int ny, const PencilArgs& a0, const PencilArgs* dA, int nmem,
                                        hipStream_t s) {
  if (!row_ok(a0)) return hipErrorInvalidValue;
  const dim3 grid(a0.P / (RWV * RPW), nmem), block(RWV * 64);
  if (a0.scalar) {
    KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_pencil_batch<NY, true, V, TV>), grid, block, (row_lds<NY, V>()), s, dA));
  } else {
    KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_pencil_batch<NY, false, V, TV>), grid, block, (row_lds<NY, V>()), s, dA));
  }
  return hipGetLastError();
}
hipError_t launch_pencil_step_batch(int ny, const PencilArgs& a0, const PencilArgs* dA, int nmem, hipStream_t s) {
  if (nmem < 1) return hipErrorInvalidValue;
  if (a0.mixed)
    return a0.tune == 1 ? launch_pencil_batch_v<float2, 1>(ny, a0, dA, nmem, s)
                        : launch_pencil_batch_v<float2, 0>(ny, a0, dA, nmem, s);
  return a0.tune == 1 ? launch_pencil_batch_v<double2, 1>(ny, a0, dA, nmem, s)
                      : launch_pencil_batch_v<double2, 0>(ny, a0, dA, nmem, s);
}
hipError_t launch_pencil_startup(int ny, const PencilArgs& a, hipStream_t s) { return launch_pencil_mode<1>(ny, a, s); }
hipError_t launch_pencil_finish(int ny, const PencilArgs& a, hipStream_t s) { return launch_pencil_mode<2>(ny, a, s); }

hipError_t launch_gradv(int ny, int P, int nz, double alpha, double beta, double dyde, const double2* u,
                        const double2* v, const double2* w, double2* const* out, hipStream_t s) {
  KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_gradv<NY>), dim3(nblk(P)), dim3(PW * 64), 0, s, P, nz, nz / 2, alpha,
                                         beta, dyde, u, v, w, out));
  return hipGetLastError();
}
hipError_t launch_mr_lap_pencil(int ny, const MrLapArgs& a, hipStream_t s) {
  if (a.mixed) {
    KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_mr_lap<NY, float2>), dim3(nblk(a.P)), dim3(PW * 64),
                                           (lds_bytes<NY, float2>()), s, a));
  } else {
    KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_mr_lap<NY, double2>), dim3(nblk(a.P)), dim3(PW * 64),
                                           (lds_bytes<NY, double2>()), s, a));
  }
  return hipGetLastError();
}
hipError_t launch_cderiv(int ny, int P, double dyde, const double2* in, double2* out, hipStream_t s) {
  KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_cderiv<NY>), dim3(nblk(P)), dim3(PW * 64), 0, s, P, dyde, in, out));
  return hipGetLastError();
}
hipError_t launch_cheb(int ny, int P, const void* tw, const void* in, void* out, int inverse, int mixed,
                       hipStream_t s) {
  if (mixed) {
    KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_cheb<NY, float2>), dim3(nblk(P)), dim3(PW * 64),
                                           (lds_bytes<NY, float2>()), s, P, static_cast<const float2*>(tw), in, out,
                                           inverse));
  } else {
    KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_cheb<NY, double2>), dim3(nblk(P)), dim3(PW * 64),
                                           (lds_bytes<NY, double2>()), s, P, static_cast<const double2*>(tw), in,
                                           out, inverse));
  }
  return hipGetLastError();
}
hipError_t launch_solve(int ny, const PencilArgs& a, const double2* tab, const double* wn, double2* u,
                        const double2* bctop, const double2* bcbot, int ib, const int* kzero, hipStream_t s) {
  KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_solve<NY>), dim3(nblk(a.P)), dim3(PW * 64), 0, s, a.P, a.dyde, tab,
                                          wn, u, bctop, bcbot, ib, kzero));
  return hipGetLastError();
}
hipError_t launch_penta(int ny, const PencilArgs& a, const double2* tab, const double* wn, double2* u, double at,
                        double bt, const double2* gtop, double ab, double bb, const double2* gbot, int bottom_sign,
                        const int* kzero, hipStream_t s) {
  KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_penta<NY>), dim3(nblk(a.P)), dim3(PW * 64), 0, s, a.P, a.dyde, tab,
                                          wn, u, at, bt, gtop, ab, bb, gbot, (double)bottom_sign, kzero));
  return hipGetLastError();
}

}  // namespace kmm
