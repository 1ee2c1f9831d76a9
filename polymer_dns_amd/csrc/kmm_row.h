// Wall-normal (Chebyshev) routines of the step kernels: four pencils per
// wavefront, one per row of 16 lanes.
//
// Lane l of a row holds K = ceil(NY / 32) consecutive coefficient pairs,
// n = 2 (K l) .. 2 (K l + K) - 1, and a copy of n = NY.  A recurrence in n
// (cderiv, the tau elimination and substitution) runs serially over the
// lane's K values and as a four-level scan over the row, all lane exchange
// being DPP moves inside the row: no lane reads, no selects.  With one
// pencil over the whole wavefront (K = 1, six levels in two stages) the
// cross-lane work was as large as the arithmetic: 8 760 vector instructions a
// pencil for the 128-point FP64 step with a scalar (counted), here 2 760.
//
// The Chebyshev transforms of a wavefront's four pencils run together: the
// even extension of NY + 1 values, length 16 R (R = NY / 8), in two register
// passes, 16 points on the lanes j = 0 .. R/2 and R points on the lanes
// k = 0 .. 8; the other residues follow from the symmetry of the data (even)
// and are never transformed, and no mirrored value is written or read.
//
// k_pencil (before -> after): 128 x 129 x 128 with the scalar FP64 0.240 ->
// 0.122, FP32 transforms 0.201 -> 0.101 ms; 96 x 81 x 96 with the scalar FP32
// 0.122 -> 0.065; 192 x 129 x 192 FP64 0.411 -> 0.276; 256 x 193 x 256 FP64
// 1.61 -> 0.73; 64 x 65 x 64 FP64 0.041 -> 0.034; 32 x 33 x 32 0.027 -> 0.027 ms
// (128 wavefronts, one instruction chain long).  At 128^3 the step moves 423
// MB (85 us at 5 TB/s) and issues 37 us of vector work per SIMD.
//
// A wavefront owns its LDS (four lines) and its pencils: there is no block
// barrier.  Fields laid out [y][pencil] move as rows of four pencils (64
// bytes in FP64), pencil-major ones as 16 lanes' contiguous values.
#pragma once
#include "kmm_pencil.h"
#include "kmm_xfft.h"

namespace kmm {

// Wavefronts per SIMD: two up to NY = 128 (256 registers hold the step without
// spills), one above, where a pencil takes half as many registers again (NY =
// 192, FP64: 0.73 ms; two with 1 KB a lane spilled 1.24 ms).
template <int NY> constexpr int row_waves() { return NY > 128 ? 1 : 2; }
constexpr int RLANES = 16, RPW = 4;   // lanes per pencil, pencils per wavefront
constexpr int RWV = 4;                // wavefronts per block

template <int NY>
struct RLay {
  static constexpr int L = NY / 2, K = (L + RLANES - 1) / RLANES, NV = 2 * K;
  static constexpr int M = 2 * NY, R = NY / 8, S = R | 1;
  static constexpr bool FULL = K * RLANES == L;
  // a line: NY + 1 values with one pad element every NV (a lane's own values
  // start NV + 1 apart: conflict-free), or the exchange [9][S]; 2 mod 8, so
  // that rows of four pencils spread over the banks
  static constexpr int RAW = 9 * S > NY + NY / NV + 1 ? 9 * S : NY + NY / NV + 1;
  static constexpr int BUF = RAW + (10 - RAW % 8) % 8;
  static_assert(NY % 16 == 0 && R % 2 == 0 && R / 2 < RLANES, "pencil length");
};
template <int NY> using RP = PFT<RLay<NY>::K>;
template <int NY> __device__ __forceinline__ constexpr int rpad(int n) { return n + n / RLay<NY>::NV; }

// The lane index as a value the compiler knows nothing about: what a routine
// derives from it (addresses, table entries, weights) is formed again in each
// use instead of being kept in registers from one to the next (a step held
// about 120 registers of such values).
__device__ __forceinline__ int fresh(int l) {
  asm volatile("" : "+v"(l));
  return l;
}

template <int NY>
__device__ __forceinline__ RP<NY> rp_zero() {
  RP<NY> f;
#pragma unroll
  for (int i = 0; i < RLay<NY>::K; ++i) f.a[i] = f.b[i] = czero();
  f.e = czero();
  return f;
}
template <int S>
__device__ __forceinline__ void rp_mask(PFT<S>& f, bool zero) {
  if (zero) {
#pragma unroll
    for (int i = 0; i < S; ++i) f.a[i] = f.b[i] = czero();
    f.e = czero();
  }
}
template <int S>
__device__ __forceinline__ void rp_mask_imag(PFT<S>& f, bool zero) {
  if (zero) {
#pragma unroll
    for (int i = 0; i < S; ++i) f.a[i].y = f.b[i].y = 0.0;
    f.e.y = 0.0;
  }
}

// ------------------------------------------------------------ row moves --
template <int N> __device__ __forceinline__ double row_bcast(double v) { return dpp<0x150 + N>(v); }
template <int N> __device__ __forceinline__ double2 row_bcast(double2 v) { return dpp<0x150 + N>(v); }
template <int N> __device__ __forceinline__ double row_ror(double v) { return dpp<0x120 + N>(v); }
__device__ __forceinline__ double row_sum(double v) {
  v += row_ror<8>(v);
  v += row_ror<4>(v);
  v += row_ror<2>(v);
  v += row_ror<1>(v);
  return v;
}
__device__ __forceinline__ double2 row_sum(double2 v) { return make_double2(row_sum(v.x), row_sum(v.y)); }
// values of pairs g + 1 and g - 1 (0 beyond the row)
template <int K, typename W>
__device__ __forceinline__ void row_next(const W (&v)[K], W (&r)[K]) {
#pragma unroll
  for (int i = 0; i + 1 < K; ++i) r[i] = v[i + 1];
  r[K - 1] = dpp<DPP_ROW_SHL | 1>(v[0]);
}
template <int K, typename W>
__device__ __forceinline__ void row_prev(const W (&v)[K], W (&r)[K]) {
#pragma unroll
  for (int i = 1; i < K; ++i) r[i] = v[i - 1];
  r[0] = dpp<DPP_ROW_SHR | 1>(v[K - 1]);
}
// pair G on every lane of the row
template <int G, int K, typename W>
__device__ __forceinline__ W row_pair(const W (&v)[K]) { return row_bcast<G / K>(v[G % K]); }

// r_g = sum_{g' >= g} v_g'
template <int K>
__device__ __forceinline__ void row_suffix_sum(const double2 (&v)[K], double2 (&r)[K]) {
  r[K - 1] = v[K - 1];
#pragma unroll
  for (int i = K - 2; i >= 0; --i) r[i] = cadd(v[i], r[i + 1]);
  double2 t = r[0];
  t = cadd(t, dpp<DPP_ROW_SHL | 1>(t));
  t = cadd(t, dpp<DPP_ROW_SHL | 2>(t));
  t = cadd(t, dpp<DPP_ROW_SHL | 4>(t));
  t = cadd(t, dpp<DPP_ROW_SHL | 8>(t));
  t = dpp<DPP_ROW_SHL | 1>(t);
#pragma unroll
  for (int i = 0; i < K; ++i) r[i] = cadd(r[i], t);
}
// y_g = w_g + c_g y_{g+1} (0 past the end).  A move reads 0 past the row's
// end, so the lanes whose map is complete gain nothing in the later levels
// whatever their factor.
template <int K, typename W>
__device__ __forceinline__ void row_suffix_affine(const double (&c)[K], const W (&w)[K], W (&y)[K]) {
  double C = c[K - 1];
  W Y = w[K - 1];
#pragma unroll
  for (int i = K - 2; i >= 0; --i) {
    Y = affine_apply(c[i], w[i], Y);
    C *= c[i];
  }
  Y = affine_apply(C, Y, dpp<DPP_ROW_SHL | 1>(Y));
  C *= dpp<DPP_ROW_SHL | 1>(C);
  Y = affine_apply(C, Y, dpp<DPP_ROW_SHL | 2>(Y));
  C *= dpp<DPP_ROW_SHL | 2>(C);
  Y = affine_apply(C, Y, dpp<DPP_ROW_SHL | 4>(Y));
  C *= dpp<DPP_ROW_SHL | 4>(C);
  Y = affine_apply(C, Y, dpp<DPP_ROW_SHL | 8>(Y));
  W in = dpp<DPP_ROW_SHL | 1>(Y);
#pragma unroll
  for (int i = K - 1; i >= 0; --i) {
    in = affine_apply(c[i], w[i], in);
    y[i] = in;
  }
}
// y_g = a_g + b_g y_{g-1} (0 before the start)
template <int K>
__device__ __forceinline__ void row_prefix_affine(const double (&b)[K], const double2 (&a)[K], double2 (&y)[K]) {
  double B = b[0];
  double2 Y = a[0];
#pragma unroll
  for (int i = 1; i < K; ++i) {
    Y = cfma(b[i], Y, a[i]);
    B *= b[i];
  }
  Y = cfma(B, dpp<DPP_ROW_SHR | 1>(Y), Y);
  B *= dpp<DPP_ROW_SHR | 1>(B);
  Y = cfma(B, dpp<DPP_ROW_SHR | 2>(Y), Y);
  B *= dpp<DPP_ROW_SHR | 2>(B);
  Y = cfma(B, dpp<DPP_ROW_SHR | 4>(Y), Y);
  B *= dpp<DPP_ROW_SHR | 4>(B);
  Y = cfma(B, dpp<DPP_ROW_SHR | 8>(Y), Y);
  double2 in = dpp<DPP_ROW_SHR | 1>(Y);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    in = cfma(b[i], in, a[i]);
    y[i] = in;
  }
}

// ------------------------------------------------ Chebyshev derivative --
// derivatives.f90:258-314 (cderiv of kmm_pencil.h)
template <int NY>
__device__ __forceinline__ RP<NY> r_cderiv(const RP<NY>& f, double dyde, int l) {
  l = fresh(l);
  constexpr int L = RLay<NY>::L, K = RLay<NY>::K;
  double2 go[K], ge[K], so[K], se[K], sx[K];
  const double g0 = (double)(K * l);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const double c = 4.0 * dyde * (g0 + i);         // 2 (2g) dyde
    ge[i] = cscale(f.a[i], c);
    go[i] = cscale(f.b[i], c + 2.0 * dyde);         // 2 (2g + 1) dyde
  }
  row_suffix_sum<K>(go, so);
  row_suffix_sum<K>(ge, se);
  row_next<K>(se, sx);
  RP<NY> d;
  const double ce = 2.0 * NY * dyde;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    d.a[i] = so[i];
    d.b[i] = cfma(ce, f.e, sx[i]);
    if (!RLay<NY>::FULL && K * l + i >= L) d.b[i] = czero();
  }
  d.e = czero();
  if (l == 0) d.a[0] = cscale(d.a[0], 0.5);
  return d;
}
// derivatives.f90:541-595 (y=+1) and 370-427 (y=-1)
template <int NY>
__device__ __forceinline__ void r_wall_derivs(const RP<NY>& f, double dyde, int l, double2& top, double2& bot) {
  constexpr int K = RLay<NY>::K;
  double2 ev = czero(), od = czero();
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const double n0 = 2.0 * (K * l + i), n1 = n0 + 1.0;
    ev = cfma(n0 * n0, f.a[i], ev);
    od = cfma(n1 * n1, f.b[i], od);
  }
  ev = cfma((double)NY * NY, f.e, row_sum(ev));
  od = row_sum(od);
  top = cscale(cadd(od, ev), dyde);
  bot = cscale(csub(od, ev), dyde);
}
// mean over y: sum over even n of a_n / (1 - n^2)
template <int NY>
__device__ __forceinline__ double r_bulk(const RP<NY>& f, int l) {
  constexpr int K = RLay<NY>::K;
  double v = 0.0;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const double n = 2.0 * (K * l + i);
    v += f.a[i].x / (1.0 - n * n);
  }
  return row_sum(v) + f.e.x / (1.0 - (double)NY * (double)NY);
}

// -------------------------------------------------------- tau systems --
// Row constants of evnc/oddc and evns/odds (solvers.f90:324-496) per pair g:
// even row coefficients of n - 2, n, n + 2, then the odd row's; the doubled
// n = 0 weight and the terms the truncation drops are folded in, and pairs
// without a row (0 and beyond NY/2 - 1) hold zeros.
template <int NY>
struct RowTau {
  static constexpr int L = RLay<NY>::L, N = RLay<NY>::K * RLANES;
  double c[N][6];
  constexpr RowTau() : c{} {
    for (int i = 1; i < L; ++i) {
      const double je = 2.0 * i, jo = je + 1.0;
      c[i][0] = (i == 1 ? 2.0 : 1.0) / (4.0 * je * (je - 1.0));
      c[i][1] = 1.0 / (2.0 * (je * je - 1.0));
      c[i][2] = i <= L - 2 ? 1.0 / (4.0 * je * (je + 1.0)) : 0.0;
      c[i][3] = 1.0 / (4.0 * jo * (jo - 1.0));
      c[i][4] = i <= L - 2 ? 1.0 / (2.0 * (jo * jo - 1.0)) : 0.0;
      c[i][5] = i <= L - 3 ? 1.0 / (4.0 * jo * (jo + 1.0)) : 0.0;
    }
  }
};
template <int NY> __device__ constexpr RowTau<NY> kRowTau{};

// One parity of eqsolve (solvers.f90:500-553): a1, a3 = wn c1, wn c3, RHS
// w, 1/d; boundary row of weights T(n) = 1 (Dirichlet) or dyde n^2 (Neumann).
// EVEN has the extra row (unknown n = NY).
template <int NY, bool EVEN, bool NEUMANN>
__device__ __forceinline__ void r_parity(const double (&c1)[RLay<NY>::K], const double (&c3)[RLay<NY>::K],
                                         const double (&invd)[RLay<NY>::K], double invdx, double wn, double dyde,
                                         const double2 (&w)[RLay<NY>::K], double2 wx, double2 bc, int l,
                                         double2 (&x)[RLay<NY>::K], double2& xx) {
  constexpr int L = RLay<NY>::L, K = RLay<NY>::K;
  double dn[K], nrho[K], k[K];
  double2 wp[K];
  row_next<K>(invd, dn);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    nrho[i] = -(wn * c3[i]) * dn[i];
    k[i] = -(wn * c1[i]) * invd[i];
  }
  row_suffix_affine<K, double2>(nrho, w, wp);
  constexpr double jx = (double)NY;
  const double a1x = EVEN ? wn * (1.0 / (4.0 * jx * (jx - 1.0))) : 0.0;
  // weight of unknown q (even: n = 2 (q-1), odd: n = 2q - 1)
  auto T = [&](double q) -> double {
    if (!NEUMANN) return 1.0;
    const double n = EVEN ? 2.0 * (q - 1.0) : 2.0 * q - 1.0;
    return dyde * n * n;
  };
  const double tx = T(L + 1);
  const double carry = EVEN ? T(L) - tx * a1x * invdx : T(L);
  double fc[K], fw[K], F[K], Fn[K];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    fc[i] = k[i];
    fw[i] = T((double)(K * l + i));
    if (K * l + i == L - 1) {
      fw[i] = fma(k[i], carry, fw[i]);
      fc[i] = 0.0;
    }
  }
  row_suffix_affine<K, double>(fc, fw, F);
  row_next<K>(F, Fn);
  double2 s = czero();
#pragma unroll
  for (int i = 0; i < K; ++i) {
    if (K * l + i == L - 1) Fn[i] = carry;
    s = cfma(Fn[i] * invd[i], wp[i], s);
  }
  s = row_sum(s);
  if (EVEN) s = cfma(tx * invdx, wx, s);
  const double F1 = row_pair<1, K>(F);
  const double2 x1 = cscale(csub(bc, s), 1.0 / F1);
  double2 a[K];
#pragma unroll
  for (int i = 0; i < K; ++i) a[i] = cscale(wp[i], invd[i]);
  if (l == 0) a[0] = x1;
  row_prefix_affine<K>(k, a, x);
  if (EVEN) {
    const double2 xl = row_pair<L - 1, K>(x);
    xx = cscale(cfma(-a1x, xl, wx), invdx);
  }
}

// solve (solvers.f90:174-283): (dyde^2 D^2 - wn) u = f with Dirichlet rows,
// sum of the even unknowns' bce and of the odd ones' bco, or Neumann rows
// (also penta's, :680-1061, whose two rows of equal weights up to the sign of
// the odd unknowns separate).  tab: the wavefront's first pencil's 1/d table,
// ot: the row's offset.
template <int NY, bool NEUMANN>
__device__ __forceinline__ RP<NY> r_solve(const RP<NY>& f, double wn, double dyde, const double2* __restrict__ tab,
                                          unsigned ot, double2 bce, double2 bco, int l) {
  l = fresh(l);
  constexpr int L = RLay<NY>::L, K = RLay<NY>::K;
  const double* c = kRowTau<NY>.c[K * l];
  double te[K], to[K];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const double2 t = tab[ot + K * l + i];
    te[i] = t.x;
    to[i] = t.y;
  }
  const double invdx = tab[ot + tab_width(NY) - 1].x;
  RP<NY> u;
  double2 w[K], m[K], p[K];
  double c1[K], c3[K];
  row_prev<K>(f.a, m);
  row_next<K>(f.a, p);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    c1[i] = c[6 * i];
    c3[i] = c[6 * i + 2];
    w[i] = cfma(-c3[i], p[i], cfma(c[6 * i + 1], f.a[i], cscale(m[i], -c1[i])));
  }
  constexpr double jx = (double)NY;
  const double2 wx = cscale(row_pair<L - 1, K>(f.a), -1.0 / (4.0 * jx * (jx - 1.0)));
  r_parity<NY, true, NEUMANN>(c1, c3, te, invdx, wn, dyde, w, wx, bce, l, u.a, u.e);
  row_prev<K>(f.b, m);
  row_next<K>(f.b, p);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    c1[i] = c[6 * i + 3];
    c3[i] = c[6 * i + 5];
    w[i] = cfma(-c3[i], p[i], cfma(c[6 * i + 4], f.b[i], cscale(m[i], -c1[i])));
  }
  double2 none;
  r_parity<NY, false, NEUMANN>(c1, c3, to, 0.0, wn, dyde, w, czero(), bco, l, u.b, none);
  return u;
}

// phirhs (solvers.f90:555-676) for theta <= 0.99
template <int S>
__device__ __forceinline__ PFT<S> r_phirhs(const PFT<S>& v, const PFT<S>& d2v, const PFT<S>& fn, const PFT<S>& fnm1,
                                           double k2, double re, double var, double dt, double th) {
  const double c0 = -re * var / (dt * th), c1 = -re * var / (2.0 * th), c2 = (1.0 - th) / th;
  PFT<S> r = pf_scale(v, c0);
  r = pf_axpy(3.0 * c1, fn, r);
  r = pf_axpy(-c1, fnm1, r);
  r = pf_axpy(c2 * k2, v, r);
  return pf_axpy(-c2, d2v, r);
}
template <int NY>
__device__ __forceinline__ void r_smooth(RP<NY>& f, const double* __restrict__ smy, double sz, int l) {
  l = fresh(l);
  constexpr int L = RLay<NY>::L, K = RLay<NY>::K;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const int g = RLay<NY>::FULL ? K * l + i : min(K * l + i, L - 1);
    f.a[i] = cscale(f.a[i], sz * smy[2 * g]);
    f.b[i] = cscale(f.b[i], sz * smy[2 * g + 1]);
  }
  f.e = cscale(f.e, sz * smy[NY]);
}

// -------------------------------------------------------- LDS and lines --
// LDS of a block: the 2 NY twiddles, then per wavefront RPW lines of double2
// (also used as lines of V at the same spacing)
template <int NY, typename V>
constexpr size_t row_lds() { return 2 * NY * sizeof(V) + (size_t)RWV * RPW * RLay<NY>::BUF * sizeof(double2); }

// twiddle w_M^k conjugated by SIGN
template <int NY, typename V>
__device__ __forceinline__ void row_fft(V* b, const V* __restrict__ tw, int l) {
  l = fresh(l);
  using RL = RLay<NY>;
  constexpr int R = RL::R, S = RL::S, NV = RL::NV;
  wave_sync();
  const bool on1 = l <= R / 2, on2 = l <= 8;
  V v[16];
  if (on1) {
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      if constexpr (R % NV == 0) {  // pads advance evenly: fixed offsets from two addresses
        v[m] = m < 8 ? b[rpad<NY>(l) + m * (R + R / NV)]
                     : b[(16 - m) * (R + R / NV) - l - (l + NV - 1) / NV];
      } else {
        v[m] = b[rpad<NY>(m < 8 ? l + R * m : R * (16 - m) - l)];
      }
    }
    dft<16, -1, V>(v);
  }
  wave_sync();
  if (on1) {
    const bool mir = l > 0 && l < R / 2;  // residue R - l by symmetry
    b[l] = v[0];
    if (mir) b[R - l] = v[0];
#pragma unroll
    for (int k = 1; k <= 8; ++k) {
      const V t = tw[l * k];
      b[k * S + l] = cmul(v[k], t);
      if (mir) b[k * S + R - l] = cmul(v[16 - k], cconj(t));
    }
  }
  wave_sync();
  V w[R];
  if (on2) {
#pragma unroll
    for (int j = 0; j < R; ++j) w[j] = b[l * S + j];
    dft<R, -1, V>(w);
  }
  wave_sync();
  if (on2) {  // outputs 16 k + l, those past NY as their mirror images
#pragma unroll
    for (int k = 0; k < R; ++k) {
      if constexpr (16 % NV == 0) {
        if (k < R / 2) b[rpad<NY>(l) + k * (16 + 16 / NV)] = w[k];
        else b[(R - k) * (16 + 16 / NV) - l - (l + NV - 1) / NV] = w[k];
      } else {
        b[rpad<NY>(k < R / 2 ? l + 16 * k : 16 * (R - k) - l)] = w[k];
      }
    }
  }
  wave_sync();
}

// Values of a field in flight, NY / 16 a lane and the last row's (parts as
// scalars: arrays of vector values stay in scratch memory).  p0, the
// wavefront's first pencil, is uniform (a scalar register), so that a fetch
// or a store needs one address register.
template <int NY, typename E>
struct RowRaw {
  static constexpr int N = NY / 16;
  typename Scal<E>::T x[N + 1], y[N + 1];
  __device__ __forceinline__ void set(int k, E v) { x[k] = v.x; y[k] = v.y; }
  __device__ __forceinline__ E get(int k) const { return mkv<E>(x[k], y[k]); }
};
// index of row y = r + 16 k of a line
template <int NY>
__device__ __forceinline__ int rline(int r, int k) {
  if constexpr (16 % RLay<NY>::NV == 0) return rpad<NY>(r) + k * (16 + 16 / RLay<NY>::NV);
  else return rpad<NY>(r + 16 * k);
}
// rows of the four pencils p0 .. p0 + 3 of a field [y][pencil]
template <int NY, typename E>
__device__ __forceinline__ void rows_fetch(RowRaw<NY, E>& q, const E* __restrict__ F, unsigned P, unsigned p0, int lane) {
  const unsigned o = (unsigned)(lane >> 2) * P + (lane & 3);
#pragma unroll
  for (int k = 0; k < NY / 16; ++k) q.set(k, (F + ((size_t)(16 * k) * P + p0))[o]);
  if (lane < 4) q.set(NY / 16, (F + ((size_t)NY * P + p0))[o]);
}
// w: the wavefront's first line
template <int NY, typename E>
__device__ __forceinline__ void rows_put(const RowRaw<NY, E>& q, E* w, int lane) {
  E* b = w + (lane & 3) * RLay<NY>::BUF;
#pragma unroll
  for (int k = 0; k < NY / 16; ++k) b[rline<NY>(lane >> 2, k)] = q.get(k);
  if (lane < 4) b[rpad<NY>(NY)] = q.get(NY / 16);
}
template <int NY, typename E>
__device__ __forceinline__ void rows_store(const E* w, E* __restrict__ F, unsigned P, unsigned p0, int lane) {
  const E* b = w + (lane & 3) * RLay<NY>::BUF;
  const unsigned o = (unsigned)(lane >> 2) * P + (lane & 3);
#pragma unroll
  for (int k = 0; k < NY / 16; ++k) (F + ((size_t)(16 * k) * P + p0))[o] = b[rline<NY>(lane >> 2, k)];
  if (lane < 4) (F + ((size_t)NY * P + p0))[o] = b[rpad<NY>(NY)];
}
// the rows' own pencils of a pencil-major field
template <int NY>
__device__ __forceinline__ void pm_fetch(RowRaw<NY, double2>& q, const double2* __restrict__ F, unsigned p0, int lane) {
  const double2* f = F + (size_t)p0 * (NY + 1);
  const unsigned o = (unsigned)(lane >> 4) * (NY + 1) + (lane & 15);
#pragma unroll
  for (int k = 0; k < NY / 16; ++k) q.set(k, f[o + 16 * k]);
  if ((lane & 15) == 0) q.set(NY / 16, f[o + NY]);
}
// a lane's own values of its line
template <int NY, typename V>
__device__ __forceinline__ RP<NY> line_take(const V* b, int l) {
  constexpr int L = RLay<NY>::L, K = RLay<NY>::K;
  RP<NY> f;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    f.a[i] = to_d(b[l * (RLay<NY>::NV + 1) + 2 * i]);
    f.b[i] = to_d(b[l * (RLay<NY>::NV + 1) + 2 * i + 1]);
    if (!RLay<NY>::FULL && K * l + i >= L) f.a[i] = f.b[i] = czero();
  }
  f.e = to_d(b[rpad<NY>(NY)]);
  return f;
}
template <int NY, typename V>
__device__ __forceinline__ void line_put(const RP<NY>& f, V* b, int l) {
  constexpr int L = RLay<NY>::L, K = RLay<NY>::K;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    if (RLay<NY>::FULL || K * l + i < L) {
      b[l * (RLay<NY>::NV + 1) + 2 * i] = to_v<V>(f.a[i]);
      b[l * (RLay<NY>::NV + 1) + 2 * i + 1] = to_v<V>(f.b[i]);
    }
  }
  if (l == 0) b[rpad<NY>(NY)] = to_v<V>(f.e);
}
// wd: the wavefront's first line
template <int NY>
__device__ __forceinline__ RP<NY> pm_take(const RowRaw<NY, double2>& q, double2* wd, int lane) {
  const int l = lane & 15;
  double2* b = wd + (lane >> 4) * RLay<NY>::BUF;
  wave_sync();
#pragma unroll
  for (int k = 0; k < NY / 16; ++k) b[rline<NY>(l, k)] = q.get(k);
  if (l == 0) b[rpad<NY>(NY)] = q.get(NY / 16);
  wave_sync();
  return line_take<NY, double2>(b, l);
}
template <int NY>
__device__ __forceinline__ RP<NY> pm_load(const double2* __restrict__ F, unsigned p0, double2* wd, int lane) {
  RowRaw<NY, double2> q;
  pm_fetch<NY>(q, F, p0, lane);
  return pm_take<NY>(q, wd, lane);
}
template <int NY>
__device__ __forceinline__ void pm_store(double2* __restrict__ F, unsigned p0, double2* wd, int lane, const RP<NY>& f) {
  const int l = lane & 15;
  double2* b = wd + (lane >> 4) * RLay<NY>::BUF;
  wave_sync();
  line_put<NY, double2>(f, b, l);
  wave_sync();
  double2* d = F + (size_t)p0 * (NY + 1);
  const unsigned o = (unsigned)(lane >> 4) * (NY + 1) + l;
#pragma unroll
  for (int k = 0; k < NY / 16; ++k) d[o + 16 * k] = b[rline<NY>(l, k)];
  if (l == 0) d[o + NY] = b[rpad<NY>(NY)];
}
// Chebyshev coefficients (solvers.f90:3279-3416) of rows fetched before
template <int NY, typename V>
__device__ __forceinline__ RP<NY> rows_to_cheb(const RowRaw<NY, V>& q, V* w, const V* tw, int lane) {
  const int l = lane & 15;
  V* b = w + (lane >> 4) * RLay<NY>::BUF;
  wave_sync();
  rows_put<NY, V>(q, w, lane);
  row_fft<NY, V>(b, tw, l);
  RP<NY> f = pf_scale(line_take<NY, V>(b, l), 1.0 / NY);
  if (l == 0) f.a[0] = cscale(f.a[0], 0.5);
  f.e = cscale(f.e, 0.5);
  return f;
}
// values at the Gauss-Lobatto points (solvers.f90:2241-2546), stored as rows
template <int NY, typename V>
__device__ __forceinline__ void cheb_to_rows(const RP<NY>& f, V* w, const V* tw, int lane, V* __restrict__ dst, unsigned P,
                                             unsigned p0) {
  const int l = lane & 15;
  V* b = w + (lane >> 4) * RLay<NY>::BUF;
  RP<NY> h = pf_scale(f, 0.5);
  if (l == 0) h.a[0] = f.a[0];
  h.e = f.e;
  wave_sync();
  line_put<NY, V>(h, b, l);
  row_fft<NY, V>(b, tw, l);
  rows_store<NY, V>(w, dst, P, p0, lane);
}
// a lane's values in LDS, as held (q: the field's [2 K + 1][64], from the lane on)
template <int NY> constexpr int lane_slots() { return 64 * (2 * RLay<NY>::K + 1); }
template <int NY>
__device__ __forceinline__ void lane_put(double2* q, const RP<NY>& f) {
  constexpr int K = RLay<NY>::K;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    q[64 * 2 * i] = f.a[i];
    q[64 * (2 * i + 1)] = f.b[i];
  }
  q[64 * 2 * K] = f.e;
}
template <int NY>
__device__ __forceinline__ RP<NY> lane_get(const double2* q) {
  constexpr int K = RLay<NY>::K;
  RP<NY> f;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    f.a[i] = q[64 * 2 * i];
    f.b[i] = q[64 * (2 * i + 1)];
  }
  f.e = q[64 * 2 * K];
  return f;
}
// real mean profiles u, w as the parts of one complex pencil
template <int NY>
__device__ __forceinline__ RP<NY> mean_load(const double* __restrict__ u, const double* __restrict__ w, int l) {
  constexpr int L = RLay<NY>::L, K = RLay<NY>::K;
  RP<NY> f = rp_zero<NY>();
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const int g = K * l + i;
    if (g < L) {
      f.a[i] = make_double2(u[2 * g], w[2 * g]);
      f.b[i] = make_double2(u[2 * g + 1], w[2 * g + 1]);
    }
  }
  f.e = make_double2(u[NY], w[NY]);
  return f;
}
template <int NY>
__device__ __forceinline__ void mean_store(double* __restrict__ u, double* __restrict__ w, const RP<NY>& f, int l) {
  constexpr int L = RLay<NY>::L, K = RLay<NY>::K;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const int g = K * l + i;
    if (g < L) {
      u[2 * g] = f.a[i].x; w[2 * g] = f.a[i].y;
      u[2 * g + 1] = f.b[i].x; w[2 * g + 1] = f.b[i].y;
    }
  }
  if (l == 0) { u[NY] = f.e.x; w[NY] = f.e.y; }
}

}  // namespace kmm
