// The x transforms of the plane kernels: one wavefront transforms NB lines
// of MX = R1 R2 complex values at a time in two register passes.
//
// Per line, L = max(R1, R2) lanes.  Inverse: R2 lanes each take the R1
// values n = j + R2 m (the middle third, the dealiasing band, is zero and is
// never read), transform them, multiply by the twiddles and pass them on
// through LDS; R1 lanes each take R2 of those and leave the points
// x = l + R1 m.  Forward: the same with the passes swapped, so that the
// outputs of the last pass that fall into the band are never formed.  Lines
// enter and leave in natural order in LDS, where the whole wavefront fills
// and reads them.
//
// With one line per wavefront and stages of radix 3 to 8, a line went through
// LDS four or five times (36 to 50 LDS instructions a line, idle lanes in the
// radix 6 and 8 stages); two passes over NB lines take 18 to 27, and a
// batch's lines share its three LDS latencies.  Measured (before -> after):
//   k_xplane       128 x 129 x 128, scalar  FP64 0.147 -> 0.135  FP32 0.102 -> 0.072 ms
//                  192 x 129 x 192          FP64 0.226 -> 0.189 ms
//                  96 x 81 x 96, scalar     FP32 0.037 -> 0.024 ms
//                  64 x 65 x 64             FP64 0.028 -> 0.019 ms
//                  256 x 193 x 256          FP64 0.451 -> 0.469 ms (24 points a lane)
//   k_xplane_poly  192 x 129 x 192          FP64 1.28  -> 0.83   FP32 0.68  -> 0.43 ms
//                  256 x 193 x 256          FP64 2.95  -> 2.91 ms
//                  64 x 65 x 64             FP64 0.124 -> 0.074 ms
// The FP64 kernels now divide their time between LDS (45 us of the 135 at
// 128 x 129 x 128, counted), the vector ALU (40 us) and memory (330 MB, 66 us
// at 5 TB/s), two wavefronts a SIMD; the FP32 ones run at memory rate.
#pragma once
#include "kmm_device.h"

namespace kmm {

// ------------------------------------------------------- register DFTs --
// dft<R>: R-point transform in registers, natural order, from the radix 2 to
// 8 butterflies: coprime factors A B (10 = 2 5, 12 = 3 4, 18 = 2 9, 24 = 3 8) by the
// Good-Thomas index maps (n = B a + A b mod AB in, k = k mod A, k mod B out:
// no twiddles), 9 and 16 as squares with constant twiddles.
template <int DIR, typename V>
__device__ __forceinline__ V crot(V a, double c, double s) {  // a (c - i s) forward, a (c + i s) backward
  using T = typename Scal<V>::T;
  return cmul(a, mkv<V>((T)c, (T)(DIR < 0 ? -s : s)));
}
template <int R, int DIR, typename V>
__device__ __forceinline__ void dft(V (&v)[R]);

template <int A, int B, int DIR, typename V>
__device__ __forceinline__ void dft_coprime(V (&v)[A * B]) {
  V t[A][B];
#pragma unroll
  for (int a = 0; a < A; ++a) {
#pragma unroll
    for (int b = 0; b < B; ++b) t[a][b] = v[(B * a + A * b) % (A * B)];
    dft<B, DIR, V>(t[a]);
  }
#pragma unroll
  for (int b = 0; b < B; ++b) {
    V c[A];
#pragma unroll
    for (int a = 0; a < A; ++a) c[a] = t[a][b];
    dft<A, DIR, V>(c);
#pragma unroll
    for (int a = 0; a < A; ++a) t[a][b] = c[a];
  }
#pragma unroll
  for (int k = 0; k < A * B; ++k) v[k] = t[k % A][k % B];
}

// W9^1, 2, 4 and W16^1, 2, 3 as (cos, sin)
constexpr double kC9[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, 0.0, -0.93969262078590838405};
constexpr double kS9[5] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.0, 0.34202014332566873304};
constexpr double kC16[10] = {1.0, 0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0, 0.0,
                             -0.70710678118654752440, 0.0, 0.0, -0.92387953251128675613};
constexpr double kS16[10] = {0.0, 0.38268343236508977173, 0.70710678118654752440, 0.92387953251128675613, 1.0, 0.0,
                             0.70710678118654752440, 0.0, 0.0, -0.38268343236508977173};

template <int R, int DIR, typename V>
__device__ __forceinline__ void dft(V (&v)[R]) {
  if constexpr (R == 2) dft2<DIR>(v[0], v[1]);
  else if constexpr (R == 3) dft3<DIR>(v[0], v[1], v[2]);
  else if constexpr (R == 4) dft4<DIR>(v[0], v[1], v[2], v[3]);
  else if constexpr (R == 5) dft5<DIR>(v[0], v[1], v[2], v[3], v[4]);
  else if constexpr (R == 6) dft_coprime<2, 3, DIR, V>(v);
  else if constexpr (R == 8) dft8<DIR>(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]);
  else if constexpr (R == 10) dft_coprime<2, 5, DIR, V>(v);
  else if constexpr (R == 12) dft_coprime<3, 4, DIR, V>(v);
  else if constexpr (R == 18) dft_coprime<2, 9, DIR, V>(v);
  else if constexpr (R == 24) dft_coprime<3, 8, DIR, V>(v);
  else {  // 9 and 16: n = Q a + b, k = a' + Q b'
    static_assert(R == 9 || R == 16, "radix");
    constexpr int Q = R == 9 ? 3 : 4;
    V t[Q][Q];
#pragma unroll
    for (int b = 0; b < Q; ++b) {
      V c[Q];
#pragma unroll
      for (int a = 0; a < Q; ++a) c[a] = v[Q * a + b];
      dft<Q, DIR, V>(c);
#pragma unroll
      for (int a = 0; a < Q; ++a) {
        const int e = a * b;
        if (e == 0) t[a][b] = c[a];
        else if (R == 16 && e == 4) t[a][b] = DIR < 0 ? mkv<V>(c[a].y, -c[a].x) : mkv<V>(-c[a].y, c[a].x);
        else t[a][b] = R == 9 ? crot<DIR, V>(c[a], kC9[e], kS9[e]) : crot<DIR, V>(c[a], kC16[e], kS16[e]);
      }
    }
#pragma unroll
    for (int a = 0; a < Q; ++a) {
      dft<Q, DIR, V>(t[a]);
#pragma unroll
      for (int b = 0; b < Q; ++b) v[a + Q * b] = t[a][b];
    }
  }
}

// ------------------------------------------------------------- the plan --
// R1 is divisible by 3: the band [MX/3, 2 MX/3) is then the middle third of
// every radix-R1 input or output.  S1, S2: odd strides of the two exchanges
// (conflict-free on both sides).
template <int MX>
struct XFft {
  static constexpr int R1 = MX == 48 ? 6 : MX == 288 ? 18 : MX == 384 ? 24 : 12;
  static constexpr int R2 = MX / R1;
  static constexpr int L = R1 > R2 ? R1 : R2;
  static constexpr int NB = 64 / L;
  static constexpr int S1 = R2 | 1, S2 = R1 | 1;
  static constexpr int BUF = R1 * S1 > R2 * S2 ? R1 * S1 : R2 * S2;
  static_assert(R1 * R2 == MX && R1 % 3 == 0, "x plan");
};

// v[k] *= w^(l k), k < R.  FP64 with 24 points: every fourth twiddle from the
// table, the others as products (16 of 23 LDS reads fewer; k_xplane at 384
// points 0.493 -> 0.469 ms at 256 x 193 x 256; with 12 to 18 points no gain)
template <int R, int DIR, typename V>
__device__ __forceinline__ void xtwiddle(V (&v)[R], const V* __restrict__ tw, int l) {
  if constexpr (sizeof(V) == 16 && R >= 24) {
    const V w1 = twid<DIR>(tw, l), w2 = twid<DIR>(tw, 2 * l), w3 = twid<DIR>(tw, 3 * l);
    v[1] = cmul(v[1], w1);
    v[2] = cmul(v[2], w2);
    v[3] = cmul(v[3], w3);
#pragma unroll
    for (int k = 4; k < R; k += 4) {
      const V wk = twid<DIR>(tw, l * k);
      v[k] = cmul(v[k], wk);
      if (k + 1 < R) v[k + 1] = cmul(v[k + 1], cmul(wk, w1));
      if (k + 2 < R) v[k + 2] = cmul(v[k + 2], cmul(wk, w2));
      if (k + 3 < R) v[k + 3] = cmul(v[k + 3], cmul(wk, w3));
    }
  } else {
#pragma unroll
    for (int k = 1; k < R; ++k) v[k] = cmul(v[k], twid<DIR>(tw, l * k));
  }
}

// NL <= NB lines at buf + g BUF, spectra in natural order (the band's values are
// not read, except n = 2 MX / 3, which must be zero) -> points, natural order
template <int MX, int NL, typename V>
__device__ __forceinline__ void xfft_inv(V* buf, const V* __restrict__ tw, int lane) {
  using P = XFft<MX>;
  constexpr int R1 = P::R1, R2 = P::R2;
  static_assert(NL <= P::NB, "lines per wavefront");
  const int g = lane / P::L, l = lane - g * P::L;
  V* b = buf + g * P::BUF;
  const bool on1 = g < NL && l < R2, on2 = g < NL && l < R1;
  wave_sync();
  V v[R1];
  if (on1) {
#pragma unroll
    for (int m = 0; m < R1; ++m) v[m] = (m >= R1 / 3 && m < 2 * R1 / 3) ? vzero<V>() : b[l + R2 * m];
    dft<R1, +1, V>(v);
    xtwiddle<R1, +1, V>(v, tw, l);
  }
  wave_sync();
  if (on1) {
#pragma unroll
    for (int k = 0; k < R1; ++k) b[k * P::S1 + l] = v[k];
  }
  wave_sync();
  V w[R2];
  if (on2) {
#pragma unroll
    for (int j = 0; j < R2; ++j) w[j] = b[l * P::S1 + j];
    dft<R2, +1, V>(w);
  }
  wave_sync();
  if (on2) {
#pragma unroll
    for (int k = 0; k < R2; ++k) b[l + R1 * k] = w[k];
  }
  wave_sync();
}

// NL <= NB lines of points, natural order -> spectra, natural order (values of the
// band are not formed)
template <int MX, int NL, typename V>
__device__ __forceinline__ void xfft_fwd(V* buf, const V* __restrict__ tw, int lane) {
  using P = XFft<MX>;
  constexpr int R1 = P::R1, R2 = P::R2;
  static_assert(NL <= P::NB, "lines per wavefront");
  const int g = lane / P::L, l = lane - g * P::L;
  V* b = buf + g * P::BUF;
  const bool on1 = g < NL && l < R1, on2 = g < NL && l < R2;
  wave_sync();
  V w[R2];
  if (on1) {
#pragma unroll
    for (int m = 0; m < R2; ++m) w[m] = b[l + R1 * m];
    dft<R2, -1, V>(w);
    xtwiddle<R2, -1, V>(w, tw, l);
  }
  wave_sync();
  if (on1) {
#pragma unroll
    for (int k = 0; k < R2; ++k) b[k * P::S2 + l] = w[k];
  }
  wave_sync();
  V v[R1];
  if (on2) {
#pragma unroll
    for (int j = 0; j < R1; ++j) v[j] = b[l * P::S2 + j];
    dft<R1, -1, V>(v);
  }
  wave_sync();
  if (on2) {
#pragma unroll
    for (int k = 0; k < R1; ++k)
      if (k < R1 / 3 || k >= 2 * R1 / 3) b[l + R2 * k] = v[k];
  }
  wave_sync();
}

// ------------------------------------------------- filling and reading --
// spectra a, b (modes k = lane + 64 q < MX / 3) of two real lines as one
// complex line a + i b: slot g
template <int MX, typename V>
__device__ __forceinline__ void xline_pack(V* buf, int g, const V (&a)[(MX / 3 + 63) / 64],
                                           const V (&b)[(MX / 3 + 63) / 64], int lane) {
  V* r = buf + g * XFft<MX>::BUF;
#pragma unroll
  for (int q = 0; q < (MX / 3 + 63) / 64; ++q) {
    const int k = lane + 64 * q;
    if (k >= MX / 3) continue;
    if (k == 0) {
      r[0] = mkv<V>(a[q].x, b[q].x);
      r[MX - MX / 3] = vzero<V>();
    } else {
      r[k] = mkv<V>(a[q].x - b[q].y, a[q].y + b[q].x);
      r[MX - k] = mkv<V>(a[q].x + b[q].y, b[q].x - a[q].y);
    }
  }
}
// points x = lane + 64 m of slot g (zero past MX)
template <int MX, typename V>
__device__ __forceinline__ void xline_read(const V* buf, int g, V (&p)[(MX + 63) / 64], int lane) {
  const V* r = buf + g * XFft<MX>::BUF;
#pragma unroll
  for (int m = 0; m < (MX + 63) / 64; ++m) {
    const int x = lane + 64 * m;
    p[m] = x < MX ? r[x] : vzero<V>();
  }
}
template <int MX, typename V>
__device__ __forceinline__ void xline_write(V* buf, int g, const V (&p)[(MX + 63) / 64], int lane) {
  V* r = buf + g * XFft<MX>::BUF;
#pragma unroll
  for (int m = 0; m < (MX + 63) / 64; ++m) {
    const int x = lane + 64 * m;
    if (x < MX) r[x] = p[m];
  }
}
// the kept modes of the two real lines transformed as line g
template <int MX, typename V>
__device__ __forceinline__ void xline_unpack(const V* buf, int g, V* __restrict__ oa, V* __restrict__ ob, int lane) {
  using T = typename Scal<V>::T;
  const V* r = buf + g * XFft<MX>::BUF;
#pragma unroll
  for (int q = 0; q < (MX / 3 + 63) / 64; ++q) {
    const int k = lane + 64 * q;
    if (k >= MX / 3) continue;
    const V zk = r[k], zm = r[k == 0 ? 0 : MX - k];
    oa[k] = mkv<V>((T)0.5 * (zk.x + zm.x), (T)0.5 * (zk.y - zm.y));
    ob[k] = mkv<V>((T)0.5 * (zk.y + zm.y), (T)-0.5 * (zk.x - zm.x));
  }
}
// Lines per batch of N transforms, at most CAP: batches as even as they come
template <int MX, int N, int CAP = 64>
constexpr int xlines() {
  const int nb = XFft<MX>::NB < CAP ? XFft<MX>::NB : CAP;
  const int count = (N + nb - 1) / nb;
  return (N + count - 1) / count;
}
// LDS of a block of wpb wavefronts: the MX twiddles, then nl line buffers each
template <int MX, typename V>
constexpr size_t xfft_lds(int wpb, int nl) { return (size_t)(MX + wpb * nl * XFft<MX>::BUF) * sizeof(V); }

}  // namespace kmm
