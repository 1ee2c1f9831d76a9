// Learned polymer-stress closure: a 22 -> 4 x 128 -> 6 multilayer
// perceptron with bfloat16 weights and FP32 accumulation (no reference
// counterpart); hidden activation ReLU, GELU as x sigma(1.702 x), or GELU with
// a polynomial in the sigmoid's place, chosen per network.
//
//   k_mlp_infer   inference on the matrix cores: v_mfma_f32_16x16x32_bf16
//                 with the weights as the A operand (staged once per block in
//                 LDS, input index permuted so that each layer's accumulators
//                 are the next layer's B operands) and the activations of
//                 kT tiles of 16 points in registers; 8 wavefronts per block,
//                 one block per CU, persistent over passes of 64 points.
//   k_mlp_fb, k_mlp_wgrad, k_mlp_reduce   training: forward + backward, the
//                 weight gradients and their sum (fixed order, no atomics)
//                 with Adam on the FP32 master parameters and the refresh of
//                 the bf16 copies.  mode 1 rounds weights and layer inputs
//                 to bf16 exactly where inference does; mode 0 is plain
//                 FP32 (gradient checks).
//
// Parameter vector (FP32 master, `kMlpParams` floats): for l = 0..4,
// W_l (n_out x n_in row-major) then b_l; sizes 22,128,128,128,128,6.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "kmm_kernels.h"
#include "kmm_device.h"

namespace kmm {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef short i16x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));  // eight packed bf16 (an MFMA operand)

constexpr int kIn = 22, kH = 128, kOut = 6, kNL = 5;
__host__ __device__ constexpr int lay_in(int l) { return l == 0 ? kIn : kH; }
__host__ __device__ constexpr int lay_out(int l) { return l == kNL - 1 ? kOut : kH; }
__host__ __device__ constexpr int w_off(int l) {
  int o = 0;
  for (int i = 0; i < l; ++i) o += lay_out(i) * lay_in(i) + lay_out(i);
  return o;
}
__host__ __device__ constexpr int b_off(int l) { return w_off(l) + lay_out(l) * lay_in(l); }
constexpr int kParams = w_off(kNL);

// padded bf16 layout for the matrix cores: K padded to 32, N to 16, rows of
// K + 8 elements
__host__ __device__ constexpr int kin_pad(int l) { return l == 0 ? 32 : kH; }
__host__ __device__ constexpr int nout_pad(int l) { return l == kNL - 1 ? 16 : kH; }
__host__ __device__ constexpr int wrow(int l) { return kin_pad(l) + 8; }
__host__ __device__ constexpr int wb_off(int l) {
  int o = 0;
  for (int i = 0; i < l; ++i) o += nout_pad(i) * wrow(i);
  return o;
}
constexpr int kWb = wb_off(kNL);  // bf16 elements of the padded weights
constexpr int kBias = 4 * kH + 16;

// activation: ReLU.  On the matrix-core path it is applied to the packed bf16
// pair after rounding (a negative bf16 is a negative int16, so one
// v_pk_max_i16 against 0 serves two activations; rounding and ReLU commute).
// On gfx950 the vector ALU and the matrix cores hardly overlap, so the
// activation's instruction count sets a large part of inference time.
__device__ __forceinline__ float act_f(float x) { return fmaxf(x, 0.0f); }
__device__ __forceinline__ float act_df(float x) { return x > 0.0f ? 1.0f : 0.0f; }
// GELU in the sigmoid form x sigma(1.702 x) (Hendrycks and Gimpel, "Gaussian
// Error Linear Units", 2016, section 2; within 0.02 of x Phi(x)): one
// exponential, one reciprocal, three multiply-adds per activation
constexpr float kGeluA = 1.702f;
__device__ __forceinline__ float gelu_sig(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __expf(-kGeluA * x));
}
__device__ __forceinline__ float gelu_f(float x) { return x * gelu_sig(x); }
__device__ __forceinline__ float gelu_df(float x) {
  const float sg = gelu_sig(x);
  return sg + kGeluA * x * sg * (1.0f - sg);
}
// GELU with a polynomial sigmoid (no exponential, no reciprocal: only
// full-rate vector operations): x s(t), t = clamp(1/2 + x/(2c), 0, 1),
// s(t) = t^3 (t (6 t - 15) + 10) (the quintic smoothstep, s' = 30 t^2 (t-1)^2
// vanishes at both clamps), c = 2.64: within 0.0195 of x Phi(x) (the sigmoid
// form above: 0.0204)
constexpr float kGpK = 1.0f / (2.0f * 2.64f);
__device__ __forceinline__ float gelup_t(float x) { return fminf(fmaxf(fmaf(x, kGpK, 0.5f), 0.0f), 1.0f); }
__device__ __forceinline__ float gelup_f(float x) {
  const float t = gelup_t(x);
  return x * (t * t * t * fmaf(t, fmaf(t, 6.0f, -15.0f), 10.0f));
}
__device__ __forceinline__ float gelup_df(float x) {
  const float t = gelup_t(x), u = t * (t - 1.0f);
  return t * t * t * fmaf(t, fmaf(t, 6.0f, -15.0f), 10.0f) + x * kGpK * 30.0f * u * u;
}
// activation a (0 ReLU, 1 GELU, 2 GELU with the polynomial sigmoid) and its derivative
__device__ __forceinline__ float act_a(int a, float x) {
  return a == 2 ? gelup_f(x) : (a ? gelu_f(x) : act_f(x));
}
__device__ __forceinline__ float act_da(int a, float x) {
  return a == 2 ? gelup_df(x) : (a ? gelu_df(x) : act_df(x));
}
// round to bfloat16 (nearest even) and back
__device__ __forceinline__ float bf16r(float x) {
  unsigned u = __float_as_uint(x);
  if ((u & 0x7f800000u) == 0x7f800000u) return x;
  u = (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u;
  return __uint_as_float(u);
}

}  // namespace

int mlp_param_count() { return kParams; }
int mlp_wb_count() { return kWb; }

// -------------------------------------------------------------- inference --
// Layout for the matrix cores.  One v_mfma_f32_16x16x32_bf16 computes
// D[m][n] = sum_k A[m][k] B[k][n] + C[m][n] with lane l holding A row l%16,
// B column l%16, both at k = 8 (l/16) + i (i < 8), and D column l%16, rows
// 4 (l/16) + i (i < 4).  Inference puts the weights in A (m = output neuron)
// and the activations in B (n = point), so a lane's D values for neuron tiles
// 2j and 2j+1 are exactly the eight B values it needs at k-step j of the next
// layer once the next layer's input index is permuted:
//   slot s = 32 j + 8 q + i  <->  neuron 32 j + 16 (i/4) + 4 q + i%4.
// The permutation is applied to the packed bf16 weights, so activations never
// leave registers between layers.  The first layer's slots hold the features
// in the order that lets lanes q = 0, 1 keep 2 h1 - h2 for the outputs they
// produce (rows 0-3 and 4-5 of the last layer):
//   q=0: h1[0..3], (h1-h2)[0..3]     q=1: h1[4,5], (h1-h2)[4,5], g[0..3]
//   q=2: g[4..8], wall distance, 0, 0     q=3: 0
__host__ __device__ constexpr int feat_of_slot(int s) {
  return s < 4 ? 10 + s : s < 8 ? 12 + s : s < 10 ? 6 + s : s < 12 ? 10 + s : s < 21 ? s - 12 : s == 21 ? 9 : -1;
}
__host__ __device__ constexpr int slot_of_feat(int k) {
  return k < 9 ? 12 + k : k == 9 ? 21 : k < 14 ? k - 10 : k < 16 ? k - 6 : k < 20 ? k - 12 : k - 10;
}
__host__ __device__ constexpr int neuron_of_slot(int s) {
  return (s & ~31) | ((s & 4) << 2) | ((s & 24) >> 1) | (s & 3);
}
__host__ __device__ constexpr int slot_of_neuron(int k) {
  return (k & ~31) | ((k & 12) << 1) | ((k & 16) >> 2) | (k & 3);
}
// packed position of input index k of layer l
__host__ __device__ constexpr int slot_of(int l, int k) { return l == 0 ? slot_of_feat(k) : slot_of_neuron(k); }
// input index of packed slot s of layer l (-1: padding)
__host__ __device__ constexpr int input_of(int l, int s) { return l == 0 ? feat_of_slot(s) : neuron_of_slot(s); }

constexpr int kT = 4;             // 16-point tiles per wavefront pass (each weight read feeds kT products)
constexpr int kChunk = 16 * kT;   // points per pass
constexpr int kInferThreads = 512;  // 8 wavefronts: 2 per SIMD

__device__ __forceinline__ float wall_feature(const MlpFieldIO& io, size_t p) {
  return (float)(1.0 - fabs(io.ycoord[(unsigned)p / (unsigned)io.plane_pts]) / io.half);
}

// feature k of point p from field-major captures (learned-closure layout)
__device__ __forceinline__ float field_feature(const MlpFieldIO& io, size_t p, int k) {
  if (k < 9) return io.g[(size_t)k * io.P + p];
  if (k == 9) return wall_feature(io, p);
  if (k < 16) return io.h1[(size_t)(k - 10) * io.P + p];
  // the last step's change, formed in FP32 before the bf16 rounding of the inputs
  return io.h1[(size_t)(k - 16) * io.P + p] - io.h2[(size_t)(k - 16) * io.P + p];
}

// activation of two FP32 values, rounded to a packed bf16 pair: ReLU after
// the rounding (ACT 0), GELU before it (ACT 1)
template <int ACT>
__device__ __forceinline__ unsigned act_pk(float a, float b) {
  if constexpr (ACT == 1) {
    const bf16x2 p = __builtin_convertvector(f32x2{gelu_f(a), gelu_f(b)}, bf16x2);
    return __builtin_bit_cast(unsigned, p);
  } else {
    const bf16x2 p = __builtin_convertvector(f32x2{a, b}, bf16x2);  // one v_cvt_pk_bf16_f32
    return __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(i16x2, p), i16x2{0, 0}));
  }
}

// Eight values that an instruction stream may not reorder around: what was
// asked for before is done for all eight first.
template <bool ON>
__device__ __forceinline__ void eight(float (&v)[8]) {
  if constexpr (ON)
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
}
// gelup_f of eight values side by side, rounded to packed bf16 pairs; ORD
// holds the compiler to that order (its own saves registers and has each
// instruction wait for the one before)
template <bool ORD>
__device__ __forceinline__ u32x4 gelup_pk8(const float (&x)[8]) {
  float t[8], u[8], y[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = gelup_t(x[i]);
  eight<ORD>(t);
#pragma unroll
  for (int i = 0; i < 8; ++i) u[i] = t[i] * t[i];
  eight<ORD>(u);
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = fmaf(t[i], 6.0f, -15.0f);
  eight<ORD>(y);
#pragma unroll
  for (int i = 0; i < 8; ++i) u[i] = u[i] * t[i];
  eight<ORD>(u);
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = fmaf(t[i], y[i], 10.0f);
  eight<ORD>(y);
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = u[i] * y[i];
  eight<ORD>(y);
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = x[i] * y[i];
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{y[2 * e], y[2 * e + 1]}, bf16x2));
  return o;
}

__device__ __forceinline__ u32x4 pack8(const float (&v)[8]) {
  bf16x8 o;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = (__bf16)v[i];
  return __builtin_bit_cast(u32x4, o);
}

// One layer with KS input k-steps and 128 outputs, eight neuron tiles of 16:
// A operands (weights, rows of wr bf16) from LDS, each read once per pass and
// used for kT point tiles; the bias enters as the accumulator of the first
// k-step; outputs activated, rounded to bf16 and laid out as the next layer's
// B operands (tile nt fills elements 4 (nt%2) .. 4 (nt%2) + 3 of out[nt/2]).
// Software pipelined: tile nt's products are interleaved with the activation
// of tile nt-1 and with the weight reads of tile nt+1, so that neither waits
// for the other's results.
//
// Bound by issue: vector and matrix instructions hardly overlap on gfx950, and
// a pass of 64 points takes 432 products of 16 cycles and, with ACT 2, 4265
// vector instructions of 4 (3840 of them the 512 activations' polynomial and
// rounding), together 112 % of its cycles (counted).  ACT 2 therefore gains
// from eight activations side by side (gelup_pk8), the others from the
// interleaving alone.  Measured
// with ACT 0, 1, 2 (us; the closure's step is 192 x 129 x 192, 10.7 M points):
//                                       10^6 rows       one row        closure's step
//   this form                           101  206  181   8.6 15.7 15.2  950 1820 1640
//   ACT 2's activations one by one      101  206  188   8.6 15.7 15.0  950 1820 1710
//   32x32x16 products, not interleaved  112  211  179  10.1 17.2 17.3 1000 1820 1660
// ORD, the order of the eight held (the field kernel), is 2 % there; one row
// takes 16.0 with it, 15.2 without, so the row kernel leaves it to the compiler.
template <int KS, int ACT, bool ORD>
__device__ __forceinline__ void mlp_layer(const u32x4 (&in)[KS][kT], u32x4 (&out)[4][kT], const __bf16* W, int wr,
                                          const float* bias, int r16, int kq) {
  const __bf16* wl = W + r16 * wr + kq * 8;  // this lane's A row in tile 0
  const float* bl = bias + 4 * kq;            // this lane's four accumulator rows in tile 0
  f32x4 acc[2][kT];
  bf16x8 a[2][KS];
  f32x4 bb[2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) a[0][ks] = *reinterpret_cast<const bf16x8*>(wl + ks * 32);
  bb[0] = *reinterpret_cast<const f32x4*>(bl);
#pragma unroll
  for (int nt = 0; nt <= 8; ++nt) {
    if (nt < 7) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        a[(nt + 1) & 1][ks] = *reinterpret_cast<const bf16x8*>(wl + (nt + 1) * 16 * wr + ks * 32);
      bb[(nt + 1) & 1] = *reinterpret_cast<const f32x4*>(bl + (nt + 1) * 16);
    }
    if (nt < 8) {
      const f32x4 b4 = bb[nt & 1];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int t = 0; t < kT; ++t)
          acc[nt & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a[nt & 1][ks], __builtin_bit_cast(bf16x8, in[ks][t]), ks == 0 ? b4 : acc[nt & 1][t], 0, 0, 0);
    }
    if (nt > 0) {
      const int m = nt - 1;
#pragma unroll
      for (int t = 0; t < kT; t += 2) {
        if constexpr (ACT == 2) {
          float x[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = acc[m & 1][t + i / 4][i % 4];
          const u32x4 y = gelup_pk8<ORD>(x);
          out[m >> 1][t][2 * (m & 1)] = y[0];
          out[m >> 1][t][2 * (m & 1) + 1] = y[1];
          out[m >> 1][t + 1][2 * (m & 1)] = y[2];
          out[m >> 1][t + 1][2 * (m & 1) + 1] = y[3];
        } else {
#pragma unroll
          for (int q = t; q < t + 2; ++q) {
            out[m >> 1][q][2 * (m & 1)] = act_pk<ACT>(acc[m & 1][q][0], acc[m & 1][q][1]);
            out[m >> 1][q][2 * (m & 1) + 1] = act_pk<ACT>(acc[m & 1][q][2], acc[m & 1][q][3]);
          }
        }
      }
    }
    if (nt > 0 && nt < 8) {
      // one product, then its share of the vector work
#pragma unroll
      for (int i = 0; i < KS * kT; ++i) {
        if (i <= KS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 64 / (KS * kT) > 4 ? 64 / (KS * kT) : 4, 0);
      }
    }
    // keep each stage's registers from being hoisted into the previous one
    __builtin_amdgcn_sched_barrier(0);
  }
}

// FIELD = false: X[n][22] -> Y[n][6]; FIELD = true: io fields -> io.out[6][P].
// Persistent: wavefront w takes passes w, w + (all wavefronts), ...
template <bool FIELD, int ACT>
__global__ __launch_bounds__(kInferThreads) void k_mlp_infer(int n, const float* __restrict__ X,
                                                             float* __restrict__ Y, MlpFieldIO io,
                                                             const __bf16* __restrict__ wb,
                                                             const float* __restrict__ par,
                                                             const float* __restrict__ norm) {
  extern __shared__ __align__(16) unsigned char smraw[];
  __bf16* sw = reinterpret_cast<__bf16*>(smraw);           // [kWb]
  float* sb = reinterpret_cast<float*>(sw + kWb);           // biases [kBias]
  float* sxs = sb + kBias;                                  // input scale per slot [32]
  float* sxo = sxs + 32;                                    // input shift per slot [32]
  const int tid = threadIdx.x, lane = tid & 63;
  // 2 h1 - h2 of the outputs this lane produces, kept here between the ends of
  // a pass: in registers ACT 2 spills 88 bytes a lane (1.73 against 1.64 ms)
  f32x4* exl = reinterpret_cast<f32x4*>(sxo + 32) + tid;
  {
    const uint4* src = reinterpret_cast<const uint4*>(wb);
    uint4* dst = reinterpret_cast<uint4*>(sw);
    for (int e = tid; e < kWb / 8; e += blockDim.x) dst[e] = src[e];
  }
  // biases: layer l at 128 l (the last layer's padded entries at 512)
  for (int l = 0; l < kNL; ++l)
    for (int j = tid; j < nout_pad(l); j += blockDim.x) sb[128 * l + j] = (j < lay_out(l)) ? par[b_off(l) + j] : 0.0f;
  if (tid < 32) {
    const int k = feat_of_slot(tid);
    sxs[tid] = k < 0 ? 0.0f : 1.0f / norm[kIn + k];
    sxo[tid] = k < 0 ? 0.0f : -norm[k] / norm[kIn + k];
  }
  __syncthreads();
  const float* mu_y = norm + 2 * kIn;
  const float* sd_y = norm + 2 * kIn + kOut;
  const int r16 = lane & 15, kq = lane >> 4;
  const int npass = (n + kChunk - 1) / kChunk;
  const int nwave = gridDim.x * (blockDim.x >> 6);
  for (int c = blockIdx.x * (blockDim.x >> 6) + (tid >> 6); c < npass; c += nwave) {
    const int p0 = c * kChunk;
    u32x4 x0[1][kT];
    // all of the pass's loads first, then one wait.  Every load instruction
    // reads one array for the whole wavefront (rows chosen per lane group,
    // always in range; the values a group does not need are discarded):
    // A = h1 rows 4q + j (q = 0: 0-3, q = 1: 4-5), B = h2 likewise,
    // G = g rows 4 (q >= 2) + j (q = 1: 0-3, q >= 2: 4-8).
    float A[kT][4], B[kT][4], G[kT][5];
    double yc[kT];
    const unsigned P = FIELD ? (unsigned)io.P : 0u;
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      const unsigned p = (unsigned)min(p0 + 16 * t + r16, n - 1);
      if (FIELD) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const unsigned row = (unsigned)min(4 * kq + j, 5);
          A[t][j] = io.h1[row * P + p];
          B[t][j] = io.h2[row * P + p];
        }
#pragma unroll
        for (int j = 0; j < 5; ++j) G[t][j] = io.g[(unsigned)min((kq >= 2 ? 4 : 0) + j, 8) * P + p];
        yc[t] = io.ycoord[p / (unsigned)io.plane_pts];
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int k = feat_of_slot(8 * kq + j);
          const float x = X[(size_t)p * kIn + (k < 0 ? 0 : k)];
          if (j < 4) A[t][j] = x;
          else B[t][j - 4] = x;
        }
      }
    }
    const bool q0 = kq == 0, q1 = kq == 1;
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      float v[8];
      if (FIELD) {
        // slots of this lane's group: q=0 h1[0..3], h1[0..3]-h2[0..3];
        // q=1 h1[4,5], h1[4,5]-h2[4,5], g[0..3]; q=2 g[4..8], wall, 0, 0
        const float wall = (float)(1.0 - fabs(yc[t]) / io.half);
        float d[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = A[t][i] - B[t][i];  // the last step's change, in FP32
        exl[t * kInferThreads] = f32x4{A[t][0] + d[0], A[t][1] + d[1], A[t][2] + d[2], A[t][3] + d[3]};
        v[0] = q0 || q1 ? A[t][0] : G[t][0];
        v[1] = q0 || q1 ? A[t][1] : G[t][1];
        v[2] = q0 ? A[t][2] : q1 ? d[0] : G[t][2];
        v[3] = q0 ? A[t][3] : q1 ? d[1] : G[t][3];
        v[4] = q0 ? d[0] : q1 ? G[t][0] : G[t][4];
        v[5] = q0 ? d[1] : q1 ? G[t][1] : wall;
        v[6] = q0 ? d[2] : q1 ? G[t][2] : 0.0f;
        v[7] = q0 ? d[3] : q1 ? G[t][3] : 0.0f;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = A[t][i];
          v[4 + i] = B[t][i];
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = fmaf(v[i], sxs[8 * kq + i], sxo[8 * kq + i]);
      x0[0][t] = pack8(v);
    }
    u32x4 a1[4][kT], a2[4][kT];
    mlp_layer<1, ACT, FIELD>(x0, a1, sw + wb_off(0), wrow(0), sb, r16, kq);
    mlp_layer<4, ACT, FIELD>(a1, a2, sw + wb_off(1), wrow(1), sb + 128, r16, kq);
    mlp_layer<4, ACT, FIELD>(a2, a1, sw + wb_off(2), wrow(2), sb + 256, r16, kq);
    mlp_layer<4, ACT, FIELD>(a1, a2, sw + wb_off(3), wrow(3), sb + 384, r16, kq);
    // output layer: one neuron tile (rows 0-5 used)
    f32x4 acc[kT];
    {
      const __bf16* W = sw + wb_off(4);
      const f32x4 b4 = *reinterpret_cast<const f32x4*>(sb + 512 + 4 * kq);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(W + r16 * wrow(4) + ks * 32 + kq * 8);
#pragma unroll
        for (int t = 0; t < kT; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, a2[ks][t]), ks == 0 ? b4 : acc[t],
                                                           0, 0, 0);
      }
    }
    if (kq < 2) {
      const int nout = kq == 0 ? 4 : 2;
#pragma unroll
      for (int t = 0; t < kT; ++t) {
        const int p = p0 + 16 * t + r16;
        if (p < n) {
          f32x4 ex = {};
          if (FIELD) ex = exl[t * kInferThreads];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int col = 4 * kq + i;
            if (i < nout) {
              const float yv = acc[t][i] * sd_y[col] + mu_y[col];
              // the closure network predicts the correction to linear
              // extrapolation of the two previous steps: out = 2 h1 - h2 + y
              if (FIELD) io.out[(size_t)col * io.P + p] = ex[i] + yv;
              else Y[(size_t)p * kOut + col] = yv;
            }
          }
        }
      }
    }
  }
}

static_assert((kWb * 2 + kBias * 4 + 64 * 4) % 16 == 0, "LDS layout");
constexpr size_t mlp_infer_lds(bool field) {
  return (size_t)kWb * 2 + (size_t)kBias * 4 + 64 * 4 + (field ? (size_t)kInferThreads * kT * 16 : 0);
}

static int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
                                              hipSuccess || cus <= 0)
    cus = 256;
  return cus;
}

template <bool FIELD, int ACT>
static hipError_t mlp_infer_launch_a(int n, const float* X, float* Y, const MlpFieldIO& io, const void* wb,
                                     const float* par, const float* norm, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int passes = (n + kChunk - 1) / kChunk;
  static const int cus = device_cus();
  const int blocks = std::min((passes + kInferThreads / 64 - 1) / (kInferThreads / 64), cus);
  static bool attr = false;  // > 64 KB of dynamic LDS (160 KB per CU on gfx950)
  if (!attr) {
    hipError_t e = hipFuncSetAttribute((const void*)k_mlp_infer<FIELD, ACT>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)mlp_infer_lds(FIELD));
    if (e != hipSuccess) return e;
    attr = true;
  }
  hipLaunchKernelGGL((k_mlp_infer<FIELD, ACT>), dim3(blocks), dim3(kInferThreads), mlp_infer_lds(FIELD), s, n, X, Y, io,
                     static_cast<const __bf16*>(wb), par, norm);
  return hipGetLastError();
}
template <bool FIELD>
static hipError_t mlp_infer_launch(int n, const float* X, float* Y, const MlpFieldIO& io, const void* wb,
                                   const float* par, const float* norm, int act, hipStream_t s) {
  if (act == 2) return mlp_infer_launch_a<FIELD, 2>(n, X, Y, io, wb, par, norm, s);
  return act ? mlp_infer_launch_a<FIELD, 1>(n, X, Y, io, wb, par, norm, s)
             : mlp_infer_launch_a<FIELD, 0>(n, X, Y, io, wb, par, norm, s);
}

hipError_t launch_mlp_infer(int n, const float* X, float* Y, const void* wb, const float* par, const float* norm,
                            int act, hipStream_t s) {
  MlpFieldIO io;
  std::memset(&io, 0, sizeof(io));
  return mlp_infer_launch<false>(n, X, Y, io, wb, par, norm, act, s);
}

hipError_t launch_mlp_field(const MlpFieldIO& io, const void* wb, const float* par, const float* norm, int act,
                            hipStream_t s) {
  // 32-bit point indices inside the kernel
  if (io.P >= (size_t)0x7fffffff || io.plane_pts <= 0) return hipErrorInvalidValue;
  return mlp_infer_launch<true>((int)io.P, nullptr, nullptr, io, wb, par, norm, act, s);
}

// SplitMix64 of (seed, i): point index of sample i
__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__global__ void k_mlp_sample(MlpFieldIO io, const float* __restrict__ t, int n, unsigned long long seed,
                             float* __restrict__ X, float* __restrict__ T) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t p = (size_t)(mix64(seed ^ mix64((unsigned long long)i)) % (unsigned long long)io.P);
  for (int k = 0; k < kIn; ++k) X[(size_t)i * kIn + k] = field_feature(io, p, k);
  for (int j = 0; j < kOut; ++j) {
    const size_t q = (size_t)j * io.P + p;
    T[(size_t)i * kOut + j] = (t[q] - io.h1[q]) - (io.h1[q] - io.h2[q]);
  }
}

hipError_t launch_mlp_sample(const MlpFieldIO& io, const float* t, int n, unsigned long long seed, float* X,
                             float* T, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_mlp_sample, dim3((n + 255) / 256), dim3(256), 0, s, io, t, n, seed, X, T);
  return hipGetLastError();
}

// -------------------------------------------------------------- training --
// One gradient is three launches:
//
//   k_mlp_fb     forward + backward of 16 samples per block of 8 waves: the
//                layers are products of 16 x 16 x 4 FP32 matrix instructions
//                (FP32 operands and sums; mode 1 rounds weights and layer
//                inputs to bf16 first), a wave one tile of 16 neurons, the
//                layer's weights and the samples from LDS, the next layer's
//                weights loaded into registers meanwhile.  Writes each
//                layer's inputs and deltas, sample-major, to the workspace.
//   k_mlp_wgrad  the weight gradients d^T a as products over the samples, a
//                wave one 16 x 16 tile of one layer.
//   k_mlp_reduce the sum over chunks of samples, Adam.
//
// Every sum keeps the order of plain loops (inputs, then 16 samples, then
// the blocks of 16), which the matrix instruction's four-term chain allows:
// training amplifies rounding (Adam divides by the gradient's size, weights
// are rounded to bf16), so a run keeps its history.  Storing layer inputs
// and deltas (4.2 KB a sample) in place of a 212 KB gradient per 16 samples
// takes that pass over memory away; the matrix instructions and one
// activation per neuron take the products and the activations (evaluated
// again for each product before) off the vector ALU.  A training step at
// 1024 samples: 1.98 ms on the GPU with a thread per output, 0.057 ms like
// this (k_mlp_fb 0.031 of it: 13 barriers and 200 dependent matrix products
// a block, on 64 of the CUs; k_mlp_wgrad 0.020, the latency of its operands).
constexpr int kBS = 16;         // samples per block
constexpr int kLd = kH + 4;     // LDS row (16-byte aligned, rows 4 banks apart)

// workspace (floats) for npad samples (a multiple of kBS): inputs of layer 0
// [npad][32] (zero past kIn), inputs of layers 1..4 [npad][kH], deltas of
// layers 0..3 [npad][kH], deltas of layer 4 [npad][16] (zero past kOut)
__host__ __device__ constexpr int a_row(int l) { return l == 0 ? 32 : kH; }
__host__ __device__ constexpr int d_row(int l) { return l == kNL - 1 ? 16 : kH; }
__host__ __device__ constexpr int a_ofs(int l) { return l == 0 ? 0 : 32 + (l - 1) * kH; }
__host__ __device__ constexpr int d_ofs(int l) { return 32 + 4 * kH + l * kH; }
constexpr int kWsRow = 32 + 4 * kH + 4 * kH + 16;

// D[m][n] += sum_k A[m][k] B[k][n], k = 0..3 in order: lane holds A row
// lane % 16 and B column lane % 16 at k = lane / 16, D column lane % 16 at
// rows 4 (lane / 16) + i
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr size_t mlp_fb_lds() { return (size_t)(kH + 2 * kBS) * kLd * sizeof(float); }

__global__ __launch_bounds__(512) void k_mlp_fb(int n, int npad, const float* __restrict__ X,
                                                const float* __restrict__ T, const float* __restrict__ par,
                                                const float* __restrict__ norm, int mode, float scale,
                                                float* __restrict__ ws, float* __restrict__ lpart) {
  extern __shared__ __align__(16) unsigned char smraw[];
  float* wl = reinterpret_cast<float*>(smraw);          // [kH][kLd] weights of the current layer
  float* ab = wl + kH * kLd;                            // [2][kBS][kLd] layer inputs, then deltas (ping-pong)
  __shared__ float zo[kBS * kOut], l2[kBS * kOut], w4[kOut * kLd];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int r16 = lane & 15, q = lane >> 4;
  const int k0 = 16 * wv + 4 * q;   // this lane's outputs of a layer: sample r16, neurons k0 .. k0 + 3
  const int s0 = blockIdx.x * kBS;
  const float* mu_x = norm;
  const float* sd_x = norm + kIn;
  const float* mu_y = norm + 2 * kIn;
  const float* sd_y = norm + 2 * kIn + kOut;
  const bool rb = (mode & 1) != 0;   // bf16 rounding where inference rounds
  const int act = (mode >> 1) & 3;    // 0 ReLU, 1 GELU, 2 GELU (polynomial sigmoid)
  auto rnd = [&](float v) -> float { return rb ? bf16r(v) : v; };
  auto wsa = [&](int l, int s) -> float* { return ws + (size_t)a_ofs(l) * npad + (size_t)(s0 + s) * a_row(l); };
  auto wsd = [&](int l, int s) -> float* { return ws + (size_t)d_ofs(l) * npad + (size_t)(s0 + s) * d_row(l); };
  // a hidden layer's 128 x 128 weights, 16 pairs per thread (8-byte aligned:
  // every W_l starts at an even offset)
  float2 pre[16];
  auto fetch = [&](int l) {
    const float2* W = reinterpret_cast<const float2*>(par + w_off(l));
#pragma unroll
    for (int i = 0; i < 16; ++i) pre[i] = W[tid + 512 * i];
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int e = tid + 512 * i;
      *reinterpret_cast<float2*>(&wl[(e >> 6) * kLd + 2 * (e & 63)]) = make_float2(rnd(pre[i].x), rnd(pre[i].y));
    }
  };
  {
    const int s = tid >> 5, k = tid & 31;  // 16 x 32 values
    float v = 0.0f;
    if (k < kIn && s0 + s < n) v = rnd((X[(size_t)(s0 + s) * kIn + k] - mu_x[k]) / sd_x[k]);
    ab[s * kLd + k] = v;
    wsa(0, s)[k] = v;
    for (int e = tid; e < kH * 24; e += 512) {
      const int j = e / 24, kk = e % 24;
      wl[j * kLd + kk] = kk < kIn ? rnd(par[w_off(0) + j * kIn + kk]) : 0.0f;
    }
  }
  for (int e = tid; e < kOut * kH; e += 512) w4[(e >> 7) * kLd + (e & 127)] = rnd(par[w_off(4) + e]);
  float bias[4][4];
#pragma unroll
  for (int l = 0; l < 4; ++l)
#pragma unroll
    for (int i = 0; i < 4; ++i) bias[l][i] = par[b_off(l) + k0 + i];
  fetch(1);
  __syncthreads();
  // forward, hidden layers
  float dact[4][4];  // act'(z) of this lane's neurons
  int cur = 0;
#pragma unroll
  for (int l = 0; l < kNL - 1; ++l) {
    f32x4 acc;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = bias[l][i];
    const float* wa = wl + (16 * wv + r16) * kLd + q;
    const float* xb = ab + (cur * kBS + r16) * kLd + q;
#pragma unroll
    for (int m = 0; m < (l == 0 ? 6 : kH / 4); ++m) acc = mfma4(wa[4 * m], xb[4 * m], acc);
    float4 a;
    a.x = rnd(act_a(act, acc[0]));
    a.y = rnd(act_a(act, acc[1]));
    a.z = rnd(act_a(act, acc[2]));
    a.w = rnd(act_a(act, acc[3]));
#pragma unroll
    for (int i = 0; i < 4; ++i) dact[l][i] = act_da(act, acc[i]);
    cur ^= 1;
    *reinterpret_cast<float4*>(&ab[(cur * kBS + r16) * kLd + k0]) = a;
    *reinterpret_cast<float4*>(wsa(l + 1, r16) + k0) = a;
    __syncthreads();
    if (l < 3) {
      stage();
      if (l < 2) fetch(l + 2);
      __syncthreads();
    }
  }
  fetch(2);  // for the backward pass (layer 3's weights are still in LDS)
  // output layer, loss and output delta: L = scale sum (yn - tn)^2
  if (tid < kBS * kOut) {
    const int s = tid / kOut, j = tid % kOut;
    float acc = par[b_off(4) + j];
    const float* x = ab + (cur * kBS + s) * kLd;
#pragma unroll 16
    for (int k = 0; k < kH; ++k) acc += x[k] * w4[j * kLd + k];
    float dv = 0.0f, r2 = 0.0f;
    if (s0 + s < n) {
      const float tn = (T[(size_t)(s0 + s) * kOut + j] - mu_y[j]) / sd_y[j];
      const float r = acc - tn;
      r2 = r * r;
      dv = 2.0f * scale * r;
    }
    zo[tid] = dv;
    l2[tid] = r2;
  }
  __syncthreads();
  if (tid < kBS * 16) {
    const int s = tid >> 4, j = tid & 15;
    wsd(4, s)[j] = j < kOut ? zo[s * kOut + j] : 0.0f;
  }
  if (tid == 511) {
    float t = 0.0f;
#pragma unroll 16
    for (int i = 0; i < kBS * kOut; ++i) t += l2[i];
    lpart[blockIdx.x] = t * scale;
  }
  // delta of layer 3: (d W_4) act'(z_3)
  cur ^= 1;
  {
    float4 d;
    float* dp = &d.x;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float acc = 0.0f;
#pragma unroll
      for (int j = 0; j < kOut; ++j) acc += zo[r16 * kOut + j] * w4[j * kLd + k0 + i];
      dp[i] = acc * dact[3][i];
    }
    *reinterpret_cast<float4*>(&ab[(cur * kBS + r16) * kLd + k0]) = d;
    *reinterpret_cast<float4*>(wsd(3, r16) + k0) = d;
  }
  __syncthreads();
  // deltas of layers 2, 1, 0 from those of layers 3, 2, 1
#pragma unroll
  for (int l = 3; l >= 1; --l) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const float* wa = wl + q * kLd + 16 * wv + r16;
    const float* xb = ab + (cur * kBS + r16) * kLd + q;
#pragma unroll
    for (int m = 0; m < kH / 4; ++m) acc = mfma4(wa[4 * m * kLd], xb[4 * m], acc);
    const float4 d = make_float4(acc[0] * dact[l - 1][0], acc[1] * dact[l - 1][1], acc[2] * dact[l - 1][2],
                                 acc[3] * dact[l - 1][3]);
    *reinterpret_cast<float4*>(wsd(l - 1, r16) + k0) = d;
    if (l > 1) {
      cur ^= 1;
      *reinterpret_cast<float4*>(&ab[(cur * kBS + r16) * kLd + k0]) = d;
      __syncthreads();
      stage();
      if (l > 2) fetch(1);
      __syncthreads();
    }
  }
}

// Weight gradients over one chunk of samples: unit u is one 16 x 16 tile
// (rows j: outputs, columns k: inputs) of a layer: layer 0 has 8 x 2 tiles,
// layers 1-3 8 x 8, layer 4 1 x 8.  A wave walks the samples 16 at a time
// (one chain of four products, added to the running sum), the next
// eight groups' operands in flight; the first column's wave also sums the deltas
// (the bias gradient, a product with ones).
constexpr int kUnits = 16 + 3 * 64 + 8;
__global__ __launch_bounds__(64) void k_mlp_wgrad(int npad, int chunk, const float* __restrict__ ws,
                                                  float* __restrict__ gpart) {
  const int lane = threadIdx.x, r16 = lane & 15, q = lane >> 4;
  const int u = blockIdx.x;
  const int l = u < 16 ? 0 : u < 208 ? 1 + (u - 16) / 64 : 4;
  const int v = u < 16 ? u : u < 208 ? (u - 16) % 64 : u - 208;
  const int j0 = l == 0 ? 16 * (v >> 1) : l < 4 ? 16 * (v >> 3) : 0;
  const int k0 = l == 0 ? 16 * (v & 1) : l < 4 ? 16 * (v & 7) : 16 * v;
  const int dr = d_row(l), ar = a_row(l);
  const int sb = blockIdx.y * chunk, ng = (min(sb + chunk, npad) - sb) / kBS;  // groups of 16 samples
  const float* D = ws + (size_t)d_ofs(l) * npad + (size_t)(sb + q) * dr + j0 + r16;
  const float* A = ws + (size_t)a_ofs(l) * npad + (size_t)(sb + q) * ar + k0 + r16;
  const bool bias = k0 == 0;
  constexpr int PF = 8;  // groups in flight
  float d[PF][4], a[PF][4];
  auto load = [&](int slot, int g) {
    const int gc = min(g, ng - 1);  // past the end: in range, not used
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      d[slot][m] = D[(size_t)(kBS * gc + 4 * m) * dr];
      a[slot][m] = A[(size_t)(kBS * gc + 4 * m) * ar];
    }
  };
#pragma unroll
  for (int s = 0; s < PF; ++s) load(s, s);
  f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f}, bsum = sum;
  for (int g = 0; g < ng; g += PF) {
#pragma unroll
    for (int s = 0; s < PF; ++s) {
      if (g + s >= ng) break;
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, b = acc;
#pragma unroll
      for (int m = 0; m < 4; ++m) acc = mfma4(d[s][m], a[s][m], acc);
      if (bias) {
#pragma unroll
        for (int m = 0; m < 4; ++m) b = mfma4(d[s][m], 1.0f, b);
      }
      sum += acc;
      bsum += b;
      load(s, g + s + PF);
    }
  }
  float* gp = gpart + (size_t)blockIdx.y * kParams;
  const int N = lay_out(l), K = lay_in(l);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = j0 + 4 * q + i, k = k0 + r16;
    if (j < N && k < K) gp[w_off(l) + j * K + k] = sum[i];
    if (bias && r16 == 0 && j < N) gp[b_off(l) + j] = bsum[i];
  }
}

// g[i] = sum over chunks of gpart[c][i] (fixed order); loss = sum of lpart.
// ADAM: the update of the FP32 master parameters and of their padded bf16
// copy follows in the same thread.
struct AdamArgs {
  float *par, *m, *v;
  float lr, b1, b2, eps, c1, c2;
  __bf16* wb;
};
template <bool ADAM>
__global__ void k_mlp_reduce(int nchunk, int nl, const float* __restrict__ gpart, const float* __restrict__ lpart,
                             float* __restrict__ g, float* __restrict__ loss, AdamArgs A) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == gridDim.x - 1) {  // the last block has no parameter: the loss, in order
    if (threadIdx.x == 0) {
      float t = 0.0f;
#pragma unroll 8
      for (int b = 0; b < nl; ++b) t += lpart[b];
      *loss = t;
    }
    return;
  }
  if (i >= kParams) return;
  float acc = 0.0f;
  for (int b = 0; b < nchunk; ++b) acc += gpart[(size_t)b * kParams + i];
  g[i] = acc;
  if constexpr (ADAM) {
    const float mi = A.b1 * A.m[i] + (1.0f - A.b1) * acc;
    const float vi = A.b2 * A.v[i] + (1.0f - A.b2) * acc * acc;
    A.m[i] = mi;
    A.v[i] = vi;
    const float p = A.par[i] - A.lr * (mi / A.c1) / (sqrtf(vi / A.c2) + A.eps);
    A.par[i] = p;
    for (int l = 0; l < kNL; ++l) {
      const int w0 = w_off(l), wn = lay_out(l) * lay_in(l);
      if (i >= w0 && i < w0 + wn) {
        const int j = (i - w0) / lay_in(l), k = (i - w0) % lay_in(l);
        A.wb[wb_off(l) + j * wrow(l) + slot_of(l, k)] = (__bf16)p;
      }
    }
  }
}

// rebuild the padded, slot-permuted bf16 weights (zero padding) from the
// master parameters
__global__ void k_mlp_pack(const float* __restrict__ par, __bf16* __restrict__ wb) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= kWb) return;
  int l = 0;
  while (l + 1 < kNL && e >= wb_off(l + 1)) ++l;
  const int r = (e - wb_off(l)) / wrow(l), s = (e - wb_off(l)) % wrow(l);
  const int k = s < kin_pad(l) ? input_of(l, s) : -1;
  float v = 0.0f;
  if (r < lay_out(l) && k >= 0 && k < lay_in(l)) v = par[w_off(l) + r * lay_in(l) + k];
  wb[e] = (__bf16)v;
}

hipError_t launch_mlp_pack(const float* par, void* wb, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_pack, dim3((kWb + 255) / 256), dim3(256), 0, s, par, static_cast<__bf16*>(wb));
  return hipGetLastError();
}

// Samples per chunk of the weight gradient: one chain of sums up to 4096
// samples (0.020 ms for a batch of 1024, bit for bit the sum in sample
// order); beyond, the chunks' sums are added by k_mlp_reduce.
static int wgrad_chunk(int npad) { return std::min(npad, 4096); }
static int pad_samples(int n) { return (n + kBS - 1) / kBS * kBS; }

size_t mlp_train_ws(int n) {
  const int npad = pad_samples(n), chunk = wgrad_chunk(npad);
  return (size_t)npad * kWsRow + (size_t)((npad + chunk - 1) / chunk) * kParams + (size_t)npad / kBS;
}

// ws: mlp_train_ws(n) floats
static hipError_t mlp_grad_launch(int n, const float* X, const float* T, const float* par, const float* norm, int mode,
                                  float* ws, float* g, float* loss, const AdamArgs* adam, hipStream_t s) {
  const int npad = pad_samples(n), chunk = wgrad_chunk(npad), nc = (npad + chunk - 1) / chunk, nb = npad / kBS;
  float* gpart = ws + (size_t)npad * kWsRow;
  float* lpart = gpart + (size_t)nc * kParams;
  static bool attr = false;  // > 64 KB of dynamic LDS (160 KB per CU on gfx950)
  if (!attr) {
    hipError_t e = hipFuncSetAttribute((const void*)k_mlp_fb, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)mlp_fb_lds());
    if (e != hipSuccess) return e;
    attr = true;
  }
  hipLaunchKernelGGL(k_mlp_fb, dim3(nb), dim3(512), mlp_fb_lds(), s, n, npad, X, T, par, norm, mode, 1.0f / (float)n, ws, lpart);
  hipLaunchKernelGGL(k_mlp_wgrad, dim3(kUnits, nc), dim3(64), 0, s, npad, chunk, ws, gpart);
  const dim3 rg((kParams + 63) / 64 + 1);
  if (adam)
    hipLaunchKernelGGL((k_mlp_reduce<true>), rg, dim3(64), 0, s, nc, nb, gpart, lpart, g, loss, *adam);
  else
    hipLaunchKernelGGL((k_mlp_reduce<false>), rg, dim3(64), 0, s, nc, nb, gpart, lpart, g, loss, AdamArgs{});
  return hipGetLastError();
}

hipError_t launch_mlp_grad(int n, const float* X, const float* T, const float* par, const float* norm, int mode,
                           float* ws, float* g, float* loss, hipStream_t s) {
  return mlp_grad_launch(n, X, T, par, norm, mode, ws, g, loss, nullptr, s);
}

hipError_t launch_mlp_train_step(int n, const float* X, const float* T, float* par, const float* norm, int mode,
                                 float* ws, float* g, float* loss, float* m, float* v, float lr, int t, void* wb,
                                 hipStream_t s) {
  const float b1 = 0.9f, b2 = 0.999f;
  const AdamArgs A{par, m, v, lr, b1, b2, 1e-8f, 1.0f - powf(b1, (float)t), 1.0f - powf(b2, (float)t),
                   static_cast<__bf16*>(wb)};
  return mlp_grad_launch(n, X, T, par, norm, mode, ws, g, loss, &A, s);
}

}  // namespace kmm
