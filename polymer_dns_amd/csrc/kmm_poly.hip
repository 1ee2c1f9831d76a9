// Pencil stage of the FENE-P conformation tensor (POLYMER build of the
// reference), four (kx,kz) pencils per wavefront (kmm_row.h), the six
// independent components one after another:
//
//   part B  forward Chebyshev transform of the plane stage's c_n and str_n
//           (solvers.f90:3279-3416); the polymer force
//           t = div(qp), qp = zbeta1 str_n (polyforce, helpers.f90:498-560,
//           before smoothing as in main_dns.f90:674-680); the n -> n-1 copy
//           that the reference makes before smoothing (main_dns.f90:682-703);
//           smoothing (main_dns.f90:726-737)
//   init    C = diag(c11z, c22z, c33z) (main_dns.f90:206-236; the constant's
//           only Chebyshev-Fourier coefficient is the (0,0,0) one)
//   solve   polyNL (helpers.f90:610-674), phirhs with fn = cNL,
//           fnm1 = 2 cNL (main_dns.f90:249-261), n -> n-1 copy (:263-281)
//           and the Neumann penta solve with g = re diffpoly/(dt theta)
//           (:286-304)
//   evaluate  C and dC/dy to physical y for the plane stage (derivscji's
//           y-derivatives, derivatives.f90:148-254; the x and z derivatives
//           are taken in the plane stage).
//
// The conformation tensor, its histories (C, CNM1, ...) and the force TF are
// stored pencil-major, [pencil][y] (the reference's order of a spectral
// field).  The fields shared with the plane stage (the physical-y NLP and TP
// fields) keep the [y][pencil] layout of the transforms.
//
// MODE 0: step, MODE 1: startup (evaluate only), MODE 2: finish (part B only),
// MODE 3: C from the physical-y fields in NLP[0..5] (a conformation tensor
// rebuilt on the 3/2 grid and forward transformed in x and z), MODE 4: part B
// of a learned-closure stress (the force only: a closure stress is neither
// smoothed nor stored, and there is no conformation to transport).
#include "kmm_kernels.h"
#include "kmm_pencil.h"
#include "kmm_row.h"

namespace kmm {

// A force component that waits for its other terms is held in LDS where two
// wavefronts share a SIMD's registers, and in registers where one has them.
template <int NY> constexpr bool poly_park() { return row_waves<NY>() > 1; }
template <int NY, typename V>
constexpr size_t poly_lds() {
  return row_lds<NY, V>() + (poly_park<NY>() ? (size_t)RWV * lane_slots<NY>() * sizeof(double2) : 0);
}
template <int NY>
struct Parked {
  RP<NY> r;
  double2* q;
  __device__ __forceinline__ void put(const RP<NY>& f) {
    if (poly_park<NY>()) lane_put<NY>(q, f);
    else r = f;
  }
  __device__ __forceinline__ RP<NY> get() const { return poly_park<NY>() ? lane_get<NY>(q) : r; }
};

// The components run in the order 11, 12, 22, 23, 33, 13: two force
// components are open at a time (t1 until 13; t2 until 23, then t3), and each
// is stored as soon as it is complete, so that the registers hold one force,
// the component's two terms and, in the solve, C and the right-hand side.
//
// Bound by memory: a step reads 30 and writes 33 fields of 16 B a coefficient
// (2.4 GB at 192 x 129 x 192 FP64, 0.5 ms at the 4.8 TB/s of a large copy).
// Measured against one pencil a wavefront with CN and STRN stored as well (12
// fields more): 192 x 129 x 192 FP64 1.13 -> 0.74 ms (0.87 with them), mixed
// 0.98 -> 0.61 ms; 256 x 193 x 256 FP64, before in two passes of fewer
// registers each, 4.00 -> 1.60 ms (1.83 with them).  At ny = 128 one
// wavefront a SIMD with every value in registers is the same (0.71, mixed
// 0.64) and at ny = 64 slower (256 x 65 x 128 0.27 against 0.38 ms); loads
// issued a component ahead gave nothing at either.
template <int NY, int MODE, typename V>
__global__ __launch_bounds__(RWV * 64) __attribute__((amdgpu_waves_per_eu(row_waves<NY>())))
void k_poly_pencil(PolyArgs A) {
  using RL = RLay<NY>;
  using PF = RP<NY>;
  extern __shared__ __align__(16) unsigned char smraw[];
  V* smem = reinterpret_cast<V*>(smraw);
  const V* tw = lds_twiddles<NY, V>(smem, static_cast<const V*>(A.twM));
  const int lane = threadIdx.x & 63, l = lane & 15, row = lane >> 4;
  const unsigned wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double2* wd = reinterpret_cast<double2*>(smraw + 2 * NY * sizeof(V)) + (size_t)wv * RPW * RL::BUF;
  V* w = reinterpret_cast<V*>(wd);
  const unsigned P = (unsigned)A.P, p0 = (unsigned)(xcd_group(blockIdx.x, gridDim.x) * RWV + wv) * RPW;
  constexpr unsigned TW = tab_width(NY);
  double kx, kz;
  int kxi, kzi;
  pencil_k(A, (int)p0 + row, kx, kz, kxi, kzi);
  const double k2 = kx * kx + kz * kz;
  const bool is00 = (kxi == 0 && kzi == 0), nyq = (kzi == A.nzh);  // norm zeroes the z-Nyquist row
  const double dy = A.dyde;
  const double sz = A.smooth ? A.smz[kzi] : 1.0;
  const double ti = 1.0 / A.tpoly;
  const bool haveB = MODE == 2 || MODE == 4 || (MODE == 0 && A.partB);
  const bool force = MODE == 4 || (A.force && haveB);
  auto term = [&](const void* F) -> PF {
    RowRaw<NY, V> q;
    rows_fetch<NY, V>(q, static_cast<const V*>(F), P, p0, lane);
    PF h = rows_to_cheb<NY, V>(q, w, tw, lane);
    rp_mask_imag(h, is00);
    rp_mask(h, nyq);
    return h;
  };
  auto load = [&](const double2* F) -> PF {
    PF h = pm_load<NY>(F, p0, wd, lane);
    rp_mask(h, nyq);
    return h;
  };
  PF tA = rp_zero<NY>();
  Parked<NY> tB;
  tB.q = reinterpret_cast<double2*>(smraw + row_lds<NY, V>()) + (size_t)wv * lane_slots<NY>() + lane;
#pragma unroll 1
  for (int it = 0; it < 6; ++it) {
    const int c = (0x254310 >> (4 * it)) & 7;  // components 11, 12, 13, 22, 23, 33 as 0..5
    if (MODE == 3) {
      pm_store<NY>(A.C[c], p0, wd, lane, term(A.NLP[c]));
      continue;
    }
    PF cn, sn;
    if (haveB) {
      sn = term(A.NLP[6 + c]);
      if (force) {
        // t_i = d q_ik / d x_k with q = zbeta1 str (symmetric)
        const double z = A.zbeta1, zx = z * kx, zz = z * kz;
        PF d = sn;
        if (c == 1 || c == 3 || c == 4) d = r_cderiv<NY>(sn, z * dy, l);
        if (c < 3) tA = pf_add(tA, c == 1 ? d : pf_imul(sn, c == 0 ? zx : zz));
        if (c == 2) {
          rp_mask_imag(tA, is00);
          pm_store<NY>(A.TF[0], p0, wd, lane, tA);
        }
        if (c != 0) {
          PF t = c == 3 ? d : pf_imul(sn, c < 3 ? zx : zz);
          if (c != 1) t = pf_add(t, tB.get());
          if (c == 2 || c == 4) {
            rp_mask_imag(t, is00);
            pm_store<NY>(A.TF[c == 2 ? 2 : 1], p0, wd, lane, t);
            t = d;
          }
          tB.put(t);
        }
      }
      if (MODE == 4) continue;
      cn = rp_zero<NY>();
      if (!A.closure) cn = term(A.NLP[c]);
      if (A.copy) {
        pm_store<NY>(A.CNM1[c], p0, wd, lane, cn);
        pm_store<NY>(A.STRNM1[c], p0, wd, lane, sn);
        // the solve below reads them back through other lanes
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
      }
      // a closure stress feeds only the force: in a step its smoothed copy
      // in STRN has no reader (an explicit finish still stores it)
      const bool keep = !A.closure || MODE == 2;
      if (A.smooth && keep) {
        r_smooth<NY>(cn, A.smy, sz, l);
        r_smooth<NY>(sn, A.smy, sz, l);
      }
      // a solve stores them below as the next step's n-1 terms
      if (MODE == 2 || !A.solve) {
        if (!A.closure) pm_store<NY>(A.CN[c], p0, wd, lane, cn);
        if (keep) pm_store<NY>(A.STRN[c], p0, wd, lane, sn);
      }
      if (MODE == 2) continue;
    }
    PF C;
    if (MODE == 0 && A.solve) {
      // cNL = 3 (c_n - str_n/lambda) - (c_nm1 - str_nm1/lambda)
      if (!haveB) {
        cn = load(A.CN[c]);
        sn = load(A.STRN[c]);
      }
      {
        PF old = load(A.CNM1[c]);
        pm_store<NY>(A.CNM1[c], p0, wd, lane, cn);
        cn = pf_sub(pf_scale(pf_axpy(-ti, sn, cn), 3.0), old);
        old = load(A.STRNM1[c]);
        pm_store<NY>(A.STRNM1[c], p0, wd, lane, sn);
        cn = pf_axpy(ti, old, cn);
      }
    }
    if (MODE == 0 && A.init) {
      C = rp_zero<NY>();
      if (is00 && l == 0 && (c == 0 || c == 3 || c == 5)) C.a[0] = make_double2(A.c0[c == 0 ? 0 : (c == 3 ? 1 : 2)], 0.0);
    } else {
      C = load(A.C[c]);
    }
    if (MODE == 0 && A.solve) {
      // phirhs with fn = cNL, fnm1 = 2 cNL: 3 fn - fnm1 = cNL; Neumann rows
      const double c0 = -A.re * A.diffpoly / (A.dt * A.theta), c2 = (1.0 - A.theta) / A.theta;
      cn = pf_axpy(-A.re * A.diffpoly / (2.0 * A.theta), cn, pf_scale(C, c0 + c2 * k2));
#pragma unroll 1
      for (int h = 0; h < 2; ++h) C = r_cderiv<NY>(C, dy, l);
      C = pf_axpy(-c2, C, cn);
      C = r_solve<NY, true>(C, k2 + A.gC, dy, A.tabC + (size_t)p0 * TW, row * TW, czero(), czero(), l);
      rp_mask_imag(C, is00);
    }
    if (MODE == 0 && (A.init || A.solve)) pm_store<NY>(A.C[c], p0, wd, lane, C);
    if (A.evaluate) {
#pragma unroll 1
      for (int h = 0; h < 2; ++h) {
        cheb_to_rows<NY, V>(C, w, tw, lane, static_cast<V*>(A.TP[c + 6 * h]), P, p0);
        if (h == 0) C = r_cderiv<NY>(C, dy, l);
      }
    }
  }
}

template <int MODE, typename V>
static hipError_t launch_poly_v(int ny, const PolyArgs& a, hipStream_t s) {
  if (a.P % (RWV * RPW) != 0 || a.nz % RPW != 0) return hipErrorInvalidValue;
  KMM_NY_DISPATCH(ny, hipLaunchKernelGGL((k_poly_pencil<NY, MODE, V>), dim3(a.P / (RWV * RPW)), dim3(RWV * 64),
                                         (poly_lds<NY, V>()), s, a));
  return hipGetLastError();
}

hipError_t launch_poly_pencil(int ny, int mode, const PolyArgs& a, bool mixed, hipStream_t s) {
  switch (mode) {
    case 0: return mixed ? launch_poly_v<0, float2>(ny, a, s) : launch_poly_v<0, double2>(ny, a, s);
    case 1: return mixed ? launch_poly_v<1, float2>(ny, a, s) : launch_poly_v<1, double2>(ny, a, s);
    case 2: return mixed ? launch_poly_v<2, float2>(ny, a, s) : launch_poly_v<2, double2>(ny, a, s);
    case 3: return mixed ? launch_poly_v<3, float2>(ny, a, s) : launch_poly_v<3, double2>(ny, a, s);
    case 4: return mixed ? launch_poly_v<4, float2>(ny, a, s) : launch_poly_v<4, double2>(ny, a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace kmm
