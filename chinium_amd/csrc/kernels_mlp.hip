// Learned stand-in for the meta-GGA functional kernel: a small MLP on the
// spin-restricted descriptors (ln rho, s, alpha) that predicts the enhancement
// factor F = e_xc / e_x^unif(rho); e_xc's rho / sigma / tau derivatives come
// from the network's own input gradient. Trained on the GPU by the kernels
// below (forward + backward with the weight gradient, Adam); evaluated with
// FP32 weights (split into two BF16 terms for the MFMA products) and FP32
// arithmetic. With an analytic base (MlpBox::base, e.g. Slater + VWN5) the
// network predicts F - F_base and the base is added back. Points outside the
// training box, and the low-density tail, take the analytic functional
// (FP64). No reference
// counterpart: the reference evaluates functionals through libxc
// (src/ExchangeCorrelation.cpp:86-163), whose result this replaces.
//
// Network: 3 -> 64 -> 64 -> 64 -> 1, tanh hidden units, linear output. One
// wave handles 64 samples (lane = sample); the raw forward pass runs the network
// per lane in FP32 with the weights uniform across the wave, read through the
// constant address space (scalar loads) from a run copy that holds W2 transposed,
// so that every weight row a loop walks is contiguous. Training runs forward and
// backward as FP32 MFMA products over 64 samples per block. Inference (Evaluate and
// point evaluation) runs the three hidden products and the two backward ones
// as transposed split-BF16 MFMA GEMMs over the wave's 64 points.
#include "internal.hpp"
#include "device_common.hpp"
#include "xc_functionals.hpp"

namespace chx {

namespace {

constexpr int kLanes = 64;
constexpr double kCxUnif = -0.7385587663820224;  // e_x^unif = kCxUnif rho^(4/3) = -(3/4)(3/pi)^(1/3) rho^(4/3)
constexpr double kSFac = 0.16162045967399548;    // s = kSFac |grad rho| / rho^(4/3); 1 / (2 (3 pi^2)^(1/3))
constexpr double kTauUnif = 2.8712340001881915;  // tau_unif = kTauUnif rho^(5/3); (3/10) (3 pi^2)^(2/3)

__device__ __forceinline__ float ldp(const float* P, int i) {
  using cf = const __attribute__((address_space(4))) float;
  return ((cf*)P)[i];
}

// Network value and input gradient of one sample, activations in registers.
// Forward: a = tanh(W1 u + b1), b = tanh(W2 a + b2), h = tanh(W3 b + b3),
// y = w4 . h + b4. Backward from dy = 1: d3 = w4 (1 - h^2),
// d2 = (W3^T d3)(1 - b^2), d1 = (W2^T d2)(1 - a^2), du = W1^T d1. Layer-1
// activations are recomputed in the backward loop rather than held.
__device__ __forceinline__ float mlp_value_grad(const float* R, const float u[3], float du[3]) {
  float z2[kMlpH];
#pragma unroll
  for (int i = 0; i < kMlpH; ++i) z2[i] = ldp(R, kMlpB2 + i);
  for (int j = 0; j < kMlpH; ++j) {  // z2 += W2[:, j] a_j (row j of W2^T)
    const float aj = ::tanhf(ldp(R, kMlpB1 + j) + ldp(R, kMlpW1 + 3 * j) * u[0] + ldp(R, kMlpW1 + 3 * j + 1) * u[1] +
                             ldp(R, kMlpW1 + 3 * j + 2) * u[2]);
#pragma unroll
    for (int i = 0; i < kMlpH; ++i) z2[i] += ldp(R, kMlpW2 + kMlpH * j + i) * aj;
  }
#pragma unroll
  for (int i = 0; i < kMlpH; ++i) z2[i] = ::tanhf(z2[i]);  // b
  float acc[kMlpH];
#pragma unroll
  for (int j = 0; j < kMlpH; ++j) acc[j] = 0.f;
  float y = ldp(R, kMlpB4);
  for (int i = 0; i < kMlpH; ++i) {  // row i of W3: forward dot, then W3^T d3 as an axpy with the same row
    float z = ldp(R, kMlpB3 + i);
#pragma unroll
    for (int j = 0; j < kMlpH; ++j) z += ldp(R, kMlpW3 + kMlpH * i + j) * z2[j];
    const float h = ::tanhf(z), w = ldp(R, kMlpW4 + i);
    y += w * h;
    const float d3 = w * (1.f - h * h);
#pragma unroll
    for (int j = 0; j < kMlpH; ++j) acc[j] += ldp(R, kMlpW3 + kMlpH * i + j) * d3;
  }
#pragma unroll
  for (int j = 0; j < kMlpH; ++j) acc[j] *= 1.f - z2[j] * z2[j];  // d2
  du[0] = du[1] = du[2] = 0.f;
  for (int k = 0; k < kMlpH; ++k) {  // (W2^T d2)_k: row k of the transposed copy
    float t = 0.f;
#pragma unroll
    for (int j = 0; j < kMlpH; ++j) t += ldp(R, kMlpW2 + kMlpH * k + j) * acc[j];
    const float w0 = ldp(R, kMlpW1 + 3 * k), w1 = ldp(R, kMlpW1 + 3 * k + 1), w2 = ldp(R, kMlpW1 + 3 * k + 2);
    const float ak = ::tanhf(ldp(R, kMlpB1 + k) + w0 * u[0] + w1 * u[1] + w2 * u[2]);
    const float d1 = t * (1.f - ak * ak);
    du[0] += w0 * d1;
    du[1] += w1 * d1;
    du[2] += w2 * d1;
  }
  return y;
}

// ---- MFMA inference (one wave = 64 points) -------------------------------
// Every layer is computed transposed, C[unit][point] = W X, on
// v_mfma_f32_16x16x32_bf16 (operand layout: A[m = l%16][k = 8(l/16)+e],
// B[k = 8(l/16)+e][n = l%16], C register r = C[4(l/16)+r][l%16]). Lane
// l = 16 g + c holds X[mt][nt][r] = activation of unit 16 mt + 4 g + r at
// point 16 nt + c: the C registers of a layer. The K slots of every product
// are permuted so that these registers are also the next product's B operand:
// K step ks, slot 8 g + e carries unit U(ks, 8g+e) = 16 (2 ks + e/4) + 4 g + e%4,
// i.e. B element e of (nt, ks) is X[2 ks + e/4][nt][e%4]. The packed weights
// (k_mlp_pack_mx) hold A[m][slot] in that order, split in two BF16 terms
// (hi = bf16(w), lo = bf16(w - hi)), and activations enter split the same way,
// so each tile is three MFMAs per K step (lo.hi, hi.lo, then hi.hi): FP32-level
// products with FP32 accumulation. Forward: W2, W3; backward for dF/du: W3^T, W2^T.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float fast_tanh(float x) {  // 1 - 2 / (e^(2x) + 1)
  return 1.f - 2.f * __builtin_amdgcn_rcpf(__expf(2.f * x) + 1.f);
}
__device__ __forceinline__ unsigned short bf_bits(float x) { return __builtin_bit_cast(unsigned short, (__bf16)x); }
__device__ __forceinline__ float bf_val(unsigned short h) { return __builtin_bit_cast(float, (unsigned)h << 16); }

// B operand of K step ks for point tile nt, split: hi and lo halves.
__device__ __forceinline__ void pack_b(const float (&X)[4][4][4], int nt, int ks, u32x4_t& hi, u32x4_t& lo) {
  unsigned h[4], l[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float x0 = X[2 * ks + (2 * q) / 4][nt][(2 * q) % 4], x1 = X[2 * ks + (2 * q + 1) / 4][nt][(2 * q + 1) % 4];
    const unsigned short h0 = bf_bits(x0), h1 = bf_bits(x1);
    const unsigned short l0 = bf_bits(x0 - bf_val(h0)), l1 = bf_bits(x1 - bf_val(h1));
    h[q] = (unsigned)h0 | ((unsigned)h1 << 16);
    l[q] = (unsigned)l0 | ((unsigned)l1 << 16);
  }
  hi = u32x4_t{h[0], h[1], h[2], h[3]};
  lo = u32x4_t{l[0], l[1], l[2], l[3]};
}

// acc = W_mat X (64 x 64 times 64 x 64 points), packed weights Wpk.
__device__ __forceinline__ void mx_layer(const u32x4_t* __restrict__ Wpk, int mat, const float (&X)[4][4][4],
                                         f32x4_t (&acc)[4][4], int lane) {
  u32x4_t bh[4][2], bl[4][2];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) pack_b(X, nt, ks, bh[nt][ks], bl[nt][ks]);
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    // fragment (mat, mt, ks, hl): Wpk[(((mat * 4 + mt) * 2 + ks) * 2 + hl) * 64 + lane]
    const int f0 = ((mat * 4 + mt) * 2) * 2;
    const bf16x8_t a0h = __builtin_bit_cast(bf16x8_t, Wpk[(f0 + 0) * 64 + lane]);
    const bf16x8_t a0l = __builtin_bit_cast(bf16x8_t, Wpk[(f0 + 1) * 64 + lane]);
    const bf16x8_t a1h = __builtin_bit_cast(bf16x8_t, Wpk[(f0 + 2) * 64 + lane]);
    const bf16x8_t a1l = __builtin_bit_cast(bf16x8_t, Wpk[(f0 + 3) * 64 + lane]);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      f32x4_t c = f32x4_t{0.f, 0.f, 0.f, 0.f};  // the small terms first
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0l, __builtin_bit_cast(bf16x8_t, bh[nt][0]), c, 0, 0, 0);
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1l, __builtin_bit_cast(bf16x8_t, bh[nt][1]), c, 0, 0, 0);
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0h, __builtin_bit_cast(bf16x8_t, bl[nt][0]), c, 0, 0, 0);
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1h, __builtin_bit_cast(bf16x8_t, bl[nt][1]), c, 0, 0, 0);
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0h, __builtin_bit_cast(bf16x8_t, bh[nt][0]), c, 0, 0, 0);
      acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1h, __builtin_bit_cast(bf16x8_t, bh[nt][1]), c, 0, 0, 0);
    }
  }
}

// Network value and input gradient of the wave's 64 points (lane = point);
// every lane of the wave must call it. R: run parameters (FP32, for W1,
// biases, w4); Wpk: packed split-BF16 W2, W3, W3^T, W2^T fragments.
__device__ __forceinline__ float mlp_value_grad_mx(const u32x4_t* __restrict__ Wpk, const float* __restrict__ R,
                                                   const float u[3], float du[3]) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  float un[4][3];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int k = 0; k < 3; ++k) un[nt][k] = __shfl(u[k], 16 * nt + c);
  float X1[4][4][4], X2[4][4][4];
  f32x4_t acc[4][4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int unit = 16 * mt + 4 * g + r;
      const float w0 = R[kMlpW1 + 3 * unit], w1 = R[kMlpW1 + 3 * unit + 1], w2 = R[kMlpW1 + 3 * unit + 2];
      const float b = R[kMlpB1 + unit];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) X1[mt][nt][r] = fast_tanh(b + w0 * un[nt][0] + w1 * un[nt][1] + w2 * un[nt][2]);
    }
  mx_layer(Wpk, 0, X1, acc, lane);  // W2
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float b = R[kMlpB2 + 16 * mt + 4 * g + r];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) X2[mt][nt][r] = fast_tanh(acc[mt][nt][r] + b);
    }
  mx_layer(Wpk, 1, X2, acc, lane);  // W3
  float yp[4] = {0.f, 0.f, 0.f, 0.f};
  float D[4][4][4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int unit = 16 * mt + 4 * g + r;
      const float b = R[kMlpB3 + unit], w = R[kMlpW4 + unit];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const float h = fast_tanh(acc[mt][nt][r] + b);
        yp[nt] += w * h;
        D[mt][nt][r] = w * (1.f - h * h);  // d3
      }
    }
  mx_layer(Wpk, 2, D, acc, lane);  // W3^T d3
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) D[mt][nt][r] = acc[mt][nt][r] * (1.f - X2[mt][nt][r] * X2[mt][nt][r]);  // d2
  mx_layer(Wpk, 3, D, acc, lane);  // W2^T d2
  float dp[4][3] = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int unit = 16 * mt + 4 * g + r;
      const float w0 = R[kMlpW1 + 3 * unit], w1 = R[kMlpW1 + 3 * unit + 1], w2 = R[kMlpW1 + 3 * unit + 2];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const float d1 = acc[mt][nt][r] * (1.f - X1[mt][nt][r] * X1[mt][nt][r]);
        dp[nt][0] += w0 * d1;
        dp[nt][1] += w1 * d1;
        dp[nt][2] += w2 * d1;
      }
    }
  // sums over the four lane groups (units 4 g + r); lane 16 g + c then reads point tile nt = g
  float y = 0.f;
  du[0] = du[1] = du[2] = 0.f;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    float v = yp[nt];
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    float d[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      d[k] = dp[nt][k];
      d[k] += __shfl_xor(d[k], 16);
      d[k] += __shfl_xor(d[k], 32);
    }
    if (nt == g) {
      y = v;
      du[0] = d[0];
      du[1] = d[1];
      du[2] = d[2];
    }
  }
  return y + R[kMlpB4];
}

// Descriptors t = (ln rho, s/(1+s), alpha/(1+alpha)) and their derivatives
// dt[k] = (dt_k/drho, dt_k/dsigma, dt_k/dtau). s and alpha are formed as the
// analytic meta-GGA sees them: tau floored at 1e-20, sigma floored at 1e-40
// and capped at 8 rho tau (where the cap binds alpha = 0 and sigma follows
// 8 rho tau).
__device__ __forceinline__ void mlp_descriptors(double rho, double sigma, double tau, double t[3], double dt[3][3]) {
  const double r = rho;
  const double r13 = ::cbrt(r);
  const bool tfloor = tau < 1e-20;
  const double tk = tfloor ? 1e-20 : tau;
  const double sfl = 1e-40;
  double sg = sigma > sfl ? sigma : sfl;
  double dsg[3] = {0.0, sigma > sfl ? 1.0 : 0.0, 0.0};  // d sigma_eff / d(rho, sigma, tau)
  if (sg > 8.0 * r * tk) {
    sg = 8.0 * r * tk;
    dsg[0] = 8.0 * tk;
    dsg[1] = 0.0;
    dsg[2] = tfloor ? 0.0 : 8.0 * r;
  }
  const double dtk = tfloor ? 0.0 : 1.0;
  t[0] = ::log(r);
  dt[0][0] = 1.0 / r;
  dt[0][1] = dt[0][2] = 0.0;
  const double s = kSFac * ::sqrt(sg) / (r * r13);
  const double ds_dsg = s / (2.0 * sg), ds_dr = -4.0 / 3.0 * s / r;
  const double ps = 1.0 / ((1.0 + s) * (1.0 + s));
  t[1] = s / (1.0 + s);
  dt[1][0] = ps * (ds_dr + ds_dsg * dsg[0]);
  dt[1][1] = ps * ds_dsg * dsg[1];
  dt[1][2] = ps * ds_dsg * dsg[2];
  const double tu = kTauUnif * r * r13 * r13;
  double al = (tk - sg / (8.0 * r)) / tu;
  double dal[3];
  dal[0] = (sg / (8.0 * r * r) - dsg[0] / (8.0 * r)) / tu - 5.0 / 3.0 * al / r;
  dal[1] = -dsg[1] / (8.0 * r * tu);
  dal[2] = (dtk - dsg[2] / (8.0 * r)) / tu;
  if (al < 0.0) {  // rounding below the cap
    al = 0.0;
    dal[0] = dal[1] = dal[2] = 0.0;
  }
  const double pa = 1.0 / ((1.0 + al) * (1.0 + al));
  t[2] = al / (1.0 + al);
  for (int k = 0; k < 3; ++k) dt[2][k] = pa * dal[k];
}

// Surrogate at one point: eps (per particle) and v_rho, v_sigma, v_tau, or the
// analytic functional where the point is below rho_min or outside the box
// (returns false then). Every lane runs the network.
template <bool MX>
__device__ __forceinline__ bool mlp_point(const float* R, const u32x4_t* Wpk, const MlpBox& box, const int* codes,
                                          int ncodes, double rho, double sigma, double tau, double* eps, double* vr,
                                          double* vs, double* vt) {
  const double r = rho > 1e-300 ? rho : 1e-300;
  double t[3], dt[3][3];
  mlp_descriptors(r, sigma, tau, t, dt);
  bool in = rho >= box.rho_min;
  float u[3];
  double hinv[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double lo = box.lo[k], hi = box.hi[k];
    in = in && t[k] >= lo && t[k] <= hi;
    hinv[k] = 2.0 / (hi - lo);
    u[k] = (float)((t[k] - 0.5 * (lo + hi)) * hinv[k]);
  }
  float du[3];
  const float F = MX ? mlp_value_grad_mx(Wpk, R, u, du) : mlp_value_grad(R, u, du);
  if (in) {
    double g[3];  // dF/dt
#pragma unroll
    for (int k = 0; k < 3; ++k) g[k] = (double)du[k] * hinv[k];
    const double r13 = ::cbrt(r);
    const double eu = kCxUnif * r * r13;
    double dF[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) dF[c] = g[0] * dt[0][c] + g[1] * dt[1][c] + g[2] * dt[2][c];
    double e0 = 0.0, r0 = 0.0, s0 = 0.0, t0 = 0.0;  // the analytic base, if any
    if (box.nbase > 0) eval_codes(box.base, box.nbase, rho, sigma, tau, &e0, &r0, &s0, &t0);
    *eps = e0 + eu * (double)F / r;
    *vr = r0 + (4.0 / 3.0) * kCxUnif * r13 * (double)F + eu * dF[0];
    *vs = s0 + eu * dF[1];
    *vt = t0 + eu * dF[2];
    return true;
  }
  eval_codes(codes, ncodes, rho, sigma, tau, eps, vr, vs, vt);
  return false;
}

__device__ __forceinline__ int run_index(int k) {
  if (k >= kMlpW2 && k < kMlpW2 + kMlpH * kMlpH) {
    const int o = k - kMlpW2;
    return kMlpW2 + kMlpH * (o % kMlpH) + o / kMlpH;
  }
  return k;
}

__device__ __forceinline__ float bf16_round(float x) {
  return __builtin_bit_cast(float, (unsigned)__builtin_bit_cast(unsigned short, (__bf16)x) << 16);
}

}  // namespace

// Run copies of a canonical parameter block: FP32 (training) and BF16-rounded
// (inference), both with W2 transposed.
__global__ void k_mlp_pack(const float* __restrict__ P, float* __restrict__ Prun, float* __restrict__ Pinf) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= kMlpParams) return;
  const float p = P[k];
  Prun[run_index(k)] = p;
  Pinf[run_index(k)] = bf16_round(p);
}

// Raw network on normalised inputs U (n x 3): F (n) and dF/dU (n x 3); the
// per-lane FP32 network, or with Wpk the MFMA network of the inference path.
__global__ __launch_bounds__(64) void k_mlp_forward(long n, const float* __restrict__ U, const float* R,
                                                    const u32x4_t* __restrict__ Wpk, float* __restrict__ F,
                                                    float* __restrict__ dF) {
  const long i0 = (long)blockIdx.x * kLanes + threadIdx.x;
  const long i = i0 < n ? i0 : n - 1;  // the MFMA network needs every lane of the wave
  const float u[3] = {U[3 * i], U[3 * i + 1], U[3 * i + 2]};
  float du[3];
  const float y = Wpk ? mlp_value_grad_mx(Wpk, R, u, du) : mlp_value_grad(R, u, du);
  if (i0 >= n) return;
  F[i] = y;
  if (dF) {
    dF[3 * i] = du[0];
    dF[3 * i + 1] = du[1];
    dF[3 * i + 2] = du[2];
  }
}

// Packed split-BF16 A-operand fragments of the MFMA network: for matrix mat
// (0 W2, 1 W3, 2 W3^T, 3 W2^T), m tile mt, K step ks, term hl (0 hi, 1 lo),
// lane l = 16 g + c, element e: A[m = 16 mt + c][slot 8 g + e] with the slot's
// unit U = 16 (2 ks + e/4) + 4 g + e%4.
__global__ void k_mlp_pack_mx(const float* __restrict__ P, unsigned short* __restrict__ Wpk) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;  // ((((mat * 4 + mt) * 2 + ks) * 2 + hl) * 64 + lane) * 8 + e
  if (idx >= 4 * 4 * 2 * 2 * 64 * 8) return;
  const int e = idx & 7, lane = (idx >> 3) & 63, hl = (idx >> 9) & 1, ks = (idx >> 10) & 1, mt = (idx >> 11) & 3,
            mat = idx >> 13;
  const int g = lane >> 4, c = lane & 15;
  const int m = 16 * mt + c, un = 16 * (2 * ks + e / 4) + 4 * g + e % 4;
  float w;
  switch (mat) {
    case 0: w = P[kMlpW2 + kMlpH * m + un]; break;
    case 1: w = P[kMlpW3 + kMlpH * m + un]; break;
    case 2: w = P[kMlpW3 + kMlpH * un + m]; break;
    default: w = P[kMlpW2 + kMlpH * un + m]; break;
  }
  const unsigned short h = bf_bits(w);
  Wpk[idx] = hl ? bf_bits(w - bf_val(h)) : h;
}

// Loss L = cs sum_i C_i (y_i - T_i)^2 over the samples [0, n) (C_i = 1 when C
// is null) and its gradient with respect to the canonical parameters P: block b
// writes its samples' sums to Gpart[b] and losspart[b] (k_mlp_update adds them up).
//
// A block of 4 waves takes 64 samples at a time; every layer is a product on
// v_mfma_f32_16x16x4_f32 (FP32 operands and sums, as the per-lane loops it
// replaces): Z = W H (units x samples), dW = D H^T, and W^T D. Wave w owns the
// units 16 w..+15 of a layer's result: lane (g = lane / 16, c = lane % 16) holds
// units 16 w + 4 g + r at samples 16 nt + c. The K order of every product is 16
// ks + 4 g + e (step 4 ks + e, lane group g), so an operand is read four steps at
// a time as 16 bytes along K: activations and deltas lie in LDS both [sample]
// [unit] (K = units) and [unit][sample] (K = samples), with a pitch of 68 floats
// that spreads a wave's 16-byte reads over the banks; the weights of the wave's
// units stay in registers. One wave per 64 samples (the per-lane network) left
// most of the chip idle: 23.5 us for a minibatch of 16384 (500 before), the update 7.6.
constexpr int kGp = 68;
struct MlpGradSmem {
  float Hs1[kLanes][kGp], Hu1[kMlpH][kGp];  // layer-1 activations [sample][unit], [unit][sample]
  float Hs2[kLanes][kGp], Hu2[kMlpH][kGp];
  float Ds[kLanes][kGp], Du[kMlpH][kGp];    // deltas of the layer at hand
  float U[kLanes][4];
  float y[4][kLanes];
};

// acc[nt] += sum_k A[m][k] B[k][n] over 64 K values: a (4 ks + e) the wave's A
// operand, B read from rows[n = 16 nt + c][k].
__device__ __forceinline__ void mlp_gemm(const float (&a)[16], const float (*rows)[kGp], int g, int c,
                                         f32x4_t (&acc)[4]) {
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const f32x4_t b = *reinterpret_cast<const f32x4_t*>(&rows[16 * nt + c][16 * ks + 4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[4 * ks + e], b[e], acc[nt], 0, 0, 0);
    }
}

__global__ __launch_bounds__(256) void k_mlp_grad(long n, const float* __restrict__ U, const float* __restrict__ T,
                                                  const float* __restrict__ C, float cs, const float* __restrict__ P,
                                                  float* __restrict__ Gpart, float* __restrict__ losspart) {
  __shared__ __attribute__((aligned(16))) MlpGradSmem sm;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int u0 = 16 * w + 4 * g;  // the lane's first unit
  // operands of the wave's 16 rows: W2, W3 (row 16 w + c) and their transposes (column 16 w + c)
  float a2[16], a3[16], t2[16], t3[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int k = 16 * (q >> 2) + 4 * g + (q & 3);
    a2[q] = P[kMlpW2 + kMlpH * (16 * w + c) + k];
    a3[q] = P[kMlpW3 + kMlpH * (16 * w + c) + k];
    t2[q] = P[kMlpW2 + kMlpH * k + 16 * w + c];
    t3[q] = P[kMlpW3 + kMlpH * k + 16 * w + c];
  }
  float w1[4][3], b1[4], b2[4], b3[4], w4[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int k = 0; k < 3; ++k) w1[r][k] = P[kMlpW1 + 3 * (u0 + r) + k];
    b1[r] = P[kMlpB1 + u0 + r];
    b2[r] = P[kMlpB2 + u0 + r];
    b3[r] = P[kMlpB3 + u0 + r];
    w4[r] = P[kMlpW4 + u0 + r];
  }
  const float b4 = P[kMlpB4];
  f32x4_t gW2[4], gW3[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) gW2[j] = gW3[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float gW1[4][3] = {}, gb1[4] = {}, gb2[4] = {}, gb3[4] = {}, gw4[4] = {}, gb4 = 0.f, lsum = 0.f;
  // a layer's result at the lane's units and samples, into both layouts
  auto put = [&](float (*Sm)[kGp], float (*Um)[kGp], const f32x4_t (&v)[4]) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      *reinterpret_cast<f32x4_t*>(&Sm[16 * nt + c][u0]) = v[nt];
#pragma unroll
      for (int r = 0; r < 4; ++r) Um[u0 + r][16 * nt + c] = v[nt][r];
    }
  };
  // dW (rows 16 w.., 64 columns) += D H^T over the chunk's samples
  auto outer = [&](const float (*Um)[kGp], f32x4_t (&dW)[4]) {
    float a[16];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(&sm.Du[16 * w + c][16 * ks + 4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[4 * ks + e] = v[e];
    }
    mlp_gemm(a, Um, g, c, dW);
  };
  const long nchunks = (n + kLanes - 1) / kLanes;
  for (long ch = blockIdx.x; ch < nchunks; ch += gridDim.x) {
    __syncthreads();  // the previous chunk's readers are done
    if (tid < 3 * kLanes) {
      const long i = ch * kLanes + tid / 3;
      sm.U[tid / 3][tid % 3] = U[3 * (i < n ? i : n - 1) + tid % 3];
    }
    __syncthreads();
    f32x4_t h1[4], h2[4], h3[4], d[4];
    float us[4][3];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
#pragma unroll
      for (int k = 0; k < 3; ++k) us[nt][k] = sm.U[16 * nt + c][k];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        h1[nt][r] = ::tanhf(b1[r] + w1[r][0] * us[nt][0] + w1[r][1] * us[nt][1] + w1[r][2] * us[nt][2]);
    }
    put(sm.Hs1, sm.Hu1, h1);
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) h2[nt] = f32x4_t{b2[0], b2[1], b2[2], b2[3]};
    mlp_gemm(a2, sm.Hs1, g, c, h2);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) h2[nt][r] = ::tanhf(h2[nt][r]);
    put(sm.Hs2, sm.Hu2, h2);
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) h3[nt] = f32x4_t{b3[0], b3[1], b3[2], b3[3]};
    mlp_gemm(a3, sm.Hs2, g, c, h3);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      float y = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        h3[nt][r] = ::tanhf(h3[nt][r]);
        y += w4[r] * h3[nt][r];
      }
      y += __shfl_xor(y, 16);
      y += __shfl_xor(y, 32);
      if (g == 0) sm.y[w][16 * nt + c] = y;
    }
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int s = 16 * nt + c;
      const long i = ch * kLanes + s;
      const bool live = i < n;
      const float y = b4 + ((sm.y[0][s] + sm.y[1][s]) + (sm.y[2][s] + sm.y[3][s]));
      const float cw = live ? cs * (C ? C[i] : 1.f) : 0.f, e = live ? y - T[i] : 0.f;
      const float gy = 2.f * cw * e;  // dL/dy
      lsum += cw * e * e;
      gb4 += gy;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        gw4[r] += gy * h3[nt][r];
        d[nt][r] = gy * w4[r] * (1.f - h3[nt][r] * h3[nt][r]);
        gb3[r] += d[nt][r];
      }
    }
    put(sm.Ds, sm.Du, d);
    __syncthreads();
    outer(sm.Hu2, gW3);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) d[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    mlp_gemm(t3, sm.Ds, g, c, d);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        d[nt][r] *= 1.f - h2[nt][r] * h2[nt][r];
        gb2[r] += d[nt][r];
      }
    __syncthreads();  // layer 3's deltas are read
    put(sm.Ds, sm.Du, d);
    __syncthreads();
    outer(sm.Hu1, gW2);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) d[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    mlp_gemm(t2, sm.Ds, g, c, d);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float d1 = d[nt][r] * (1.f - h1[nt][r] * h1[nt][r]);
        gb1[r] += d1;
#pragma unroll
        for (int k = 0; k < 3; ++k) gW1[r][k] += d1 * us[nt][k];
      }
  }
  float* __restrict__ G = Gpart + (size_t)blockIdx.x * kMlpParams;
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      G[kMlpW2 + kMlpH * (u0 + r) + 16 * j + c] = gW2[j][r];
      G[kMlpW3 + kMlpH * (u0 + r) + 16 * j + c] = gW3[j][r];
    }
  auto sum16 = [](float v) {  // over the 16 lanes of a group: the samples
    for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o);
    return v;
  };
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float s1 = sum16(gb1[r]), s2 = sum16(gb2[r]), s3 = sum16(gb3[r]), s4 = sum16(gw4[r]);
    const float q0 = sum16(gW1[r][0]), q1 = sum16(gW1[r][1]), q2 = sum16(gW1[r][2]);
    if (c == 0) {
      G[kMlpB1 + u0 + r] = s1;
      G[kMlpB2 + u0 + r] = s2;
      G[kMlpB3 + u0 + r] = s3;
      G[kMlpW4 + u0 + r] = s4;
      G[kMlpW1 + 3 * (u0 + r)] = q0;
      G[kMlpW1 + 3 * (u0 + r) + 1] = q1;
      G[kMlpW1 + 3 * (u0 + r) + 2] = q2;
    }
  }
  gb4 = sum16(gb4);  // the same in every group
  lsum = sum16(lsum);
  if (tid == 0) {
    G[kMlpB4] = gb4;
    losspart[blockIdx.x] = lsum;
  }
}

// The gradient and loss from the blocks' sums, 64 parameters per block, 16
// partial sums each; ADAM: one step of Adam (Kingma and Ba, ICLR 2015) on the
// canonical FP32 weights, else the gradient goes to G. *loss gets the loss added.
template <bool ADAM>
__global__ __launch_bounds__(1024) void k_mlp_update(int nparts, const float* __restrict__ Gpart,
                                                     const float* __restrict__ losspart, float* __restrict__ P,
                                                     float* __restrict__ G, float* __restrict__ M,
                                                     float* __restrict__ V, float* __restrict__ loss, float lr,
                                                     float b1, float b2, float eps, float c1, float c2) {
  __shared__ float red[16][64];
  const int p = threadIdx.x & 63, s = threadIdx.x >> 6, k = blockIdx.x * 64 + p;
  float t = 0.f;
  if (k < kMlpParams)
    for (int b = s; b < nparts; b += 16) t += Gpart[(size_t)b * kMlpParams + k];
  red[s][p] = t;
  __syncthreads();
  if (s == 0 && k < kMlpParams) {
    float g = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) g += red[i][p];
    if (ADAM) {
      const float m = b1 * M[k] + (1.f - b1) * g, v = b2 * V[k] + (1.f - b2) * g * g;
      M[k] = m;
      V[k] = v;
      P[k] -= lr * (m / c1) / (::sqrtf(v / c2) + eps);
    } else {
      G[k] = g;
    }
  }
  if (blockIdx.x == 0 && s == 1) {
    float l = 0.f;
    for (int b = p; b < nparts; b += 64) l += losspart[b];
    for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o);
    if (p == 0) *loss += l;
  }
}

// Training samples: descriptors t (n x 3) and target F = e_xc / e_x^unif of
// the analytic functional (codes) at each (rho, sigma, tau).
__global__ void k_mlp_features(long n, const double* __restrict__ rho, const double* __restrict__ sigma,
                               const double* __restrict__ tau, const int* __restrict__ codes, int ncodes,
                               float* __restrict__ tout, float* __restrict__ Fout) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double r = rho[i] > 1e-300 ? rho[i] : 1e-300;
  double t[3], dt[3][3];
  mlp_descriptors(r, sigma[i], tau[i], t, dt);
  tout[3 * i] = (float)t[0];
  tout[3 * i + 1] = (float)t[1];
  tout[3 * i + 2] = (float)t[2];
  double e, vr, vs, vt;
  eval_codes(codes, ncodes, rho[i], sigma[i], tau[i], &e, &vr, &vs, &vt);
  Fout[i] = (float)(e / (kCxUnif * ::cbrt(r)));  // (rho eps) / (kCxUnif rho^(4/3))
}

// Surrogate at n arbitrary points; *nfall counts the analytic fallbacks.
__global__ __launch_bounds__(64) void k_mlp_eval(long n, const float* R, const u32x4_t* __restrict__ Wpk, MlpBox box,
                                                 const int* __restrict__ codes,
                                                 int ncodes, const double* __restrict__ rho,
                                                 const double* __restrict__ sigma, const double* __restrict__ tau,
                                                 double* __restrict__ exc, double* __restrict__ vrho,
                                                 double* __restrict__ vsigma, double* __restrict__ vtau,
                                                 int* __restrict__ nfall) {
  const long i0 = (long)blockIdx.x * kLanes + threadIdx.x;
  const bool live = i0 < n;
  const long i = live ? i0 : n - 1;  // tail lanes run a copy of the last point and store nothing
  double e, vr, vs, vt;
  const bool net = mlp_point<true>(R, Wpk, box, codes, ncodes, rho[i], sigma[i], tau[i], &e, &vr, &vs, &vt);
  if (live) {
    exc[i] = e;
    vrho[i] = vr;
    vsigma[i] = vs;
    vtau[i] = vt;
    if (!net) atomicAdd(nfall, 1);
  }
}

// The Evaluate step of a meta-GGA grid with the surrogate (the counterpart of
// k_functional): rho, grad rho and tau from the density partials, the network
// (or the analytic fallback) per point, the Vxc integrand coefficients, and
// per-block sums of E = sum w rho eps and N = sum w rho.
__global__ __launch_bounds__(64) void k_functional_mlp(int nslots, const int* __restrict__ grp_off,
                                                       const double* __restrict__ part,
                                                       const double* __restrict__ part_tau,
                                                       const double* __restrict__ bw, const float* R,
                                                       const u32x4_t* __restrict__ Wpk, MlpBox box,
                                                       const int* __restrict__ codes, int ncodes, int want_e,
                                                       int want_v, double* __restrict__ rho_out,
                                                       double* __restrict__ coef, double* __restrict__ en_part,
                                                       int* __restrict__ nfall) {
  const int slot0 = blockIdx.x * kLanes + threadIdx.x;
  const bool live = slot0 < nslots;
  const int slot = live ? slot0 : nslots - 1;
  const int b = slot / kBatch, g = slot % kBatch;
  double rho = 0, gx = 0, gy = 0, gz = 0, tau = 0;
  for (int k = grp_off[b]; k < grp_off[b + 1]; ++k) {
    const double* p = part + (size_t)k * 4 * kBatch;
    rho += p[g];
    gx += p[kBatch + g];
    gy += p[2 * kBatch + g];
    gz += p[3 * kBatch + g];
    const double* q = part_tau + (size_t)k * 3 * kBatch;
    tau += q[g] + q[kBatch + g] + q[2 * kBatch + g];
  }
  gx *= 2; gy *= 2; gz *= 2;
  tau *= 0.5;
  const double w = bw[slot];
  const double sigma = gx * gx + gy * gy + gz * gz;
  double eps, vr, vs, vt;
  const bool net = mlp_point<true>(R, Wpk, box, codes, ncodes, rho, sigma, tau, &eps, &vr, &vs, &vt);
  double e_acc = 0, n_acc = 0;
  if (live) {
    rho_out[slot] = rho;
    if (want_v) {
      coef[kCoef * (size_t)slot + 0] = 0.5 * w * vr;
      const double f = 2.0 * w * vs;
      coef[kCoef * (size_t)slot + 1] = f * gx;
      coef[kCoef * (size_t)slot + 2] = f * gy;
      coef[kCoef * (size_t)slot + 3] = f * gz;
      coef[kCoef * (size_t)slot + 4] = 0.25 * w * vt;
    }
    if (want_e) e_acc = w * rho * eps;
    n_acc = w * rho;
    if (!net && rho >= kDensThreshold && w != 0.0) atomicAdd(nfall, 1);
  }
  for (int o = 32; o > 0; o >>= 1) {
    e_acc += __shfl_xor(e_acc, o);
    n_acc += __shfl_xor(n_acc, o);
  }
  if (threadIdx.x == 0) {
    en_part[2 * blockIdx.x] = e_acc;
    en_part[2 * blockIdx.x + 1] = n_acc;
  }
}

// Per-point density of a grid after getDensity: rho, sigma, tau, weight (slot order).
__global__ void k_point_density(int nslots, const int* __restrict__ grp_off, const double* __restrict__ part,
                                const double* __restrict__ part_tau, int has_tau, const double* __restrict__ bw,
                                double* __restrict__ rho_o, double* __restrict__ sig_o, double* __restrict__ tau_o,
                                double* __restrict__ w_o) {
  const int slot = blockIdx.x * blockDim.x + threadIdx.x;
  if (slot >= nslots) return;
  const int b = slot / kBatch, g = slot % kBatch;
  double rho = 0, gx = 0, gy = 0, gz = 0, tau = 0;
  for (int k = grp_off[b]; k < grp_off[b + 1]; ++k) {
    const double* p = part + (size_t)k * 4 * kBatch;
    rho += p[g];
    gx += p[kBatch + g];
    gy += p[2 * kBatch + g];
    gz += p[3 * kBatch + g];
    if (has_tau) {
      const double* q = part_tau + (size_t)k * 3 * kBatch;
      tau += q[g] + q[kBatch + g] + q[2 * kBatch + g];
    }
  }
  rho_o[slot] = rho;
  sig_o[slot] = 4.0 * (gx * gx + gy * gy + gz * gz);
  tau_o[slot] = 0.5 * tau;
  w_o[slot] = bw[slot];
}

// ---- launchers
void launch_mlp_pack(hipStream_t st, const float* P, float* Prun, float* Pinf) {
  hipLaunchKernelGGL(k_mlp_pack, dim3((kMlpParams + 255) / 256), dim3(256), 0, st, P, Prun, Pinf);
  CHX_HIP(hipGetLastError());
}

void launch_mlp_forward(hipStream_t st, long n, const float* U, const float* R, const unsigned* Wpk, float* F,
                        float* dF) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)((n + kLanes - 1) / kLanes)), dim3(kLanes), 0, st, n, U, R,
                     reinterpret_cast<const u32x4_t*>(Wpk), F, dF);
  CHX_HIP(hipGetLastError());
}

void launch_mlp_pack_mx(hipStream_t st, const float* P, unsigned* Wpk) {
  hipLaunchKernelGGL(k_mlp_pack_mx, dim3(4 * 4 * 2 * 2 * 64 * 8 / 256), dim3(256), 0, st, P,
                     reinterpret_cast<unsigned short*>(Wpk));
  CHX_HIP(hipGetLastError());
}

int launch_mlp_grad(hipStream_t st, long n, const float* U, const float* T, const float* C, float cs, const float* P,
                    float* Gpart, float* losspart) {
  if (n <= 0) return 0;
  const long nchunks = (n + kLanes - 1) / kLanes;
  const int nb = (int)(nchunks < kMlpGradBlocks ? nchunks : kMlpGradBlocks);
  hipLaunchKernelGGL(k_mlp_grad, dim3(nb), dim3(256), 0, st, n, U, T, C, cs, P, Gpart, losspart);
  CHX_HIP(hipGetLastError());
  return nb;
}

void launch_mlp_adam(hipStream_t st, int nparts, const float* Gpart, const float* losspart, float* P, float* M,
                     float* V, float* loss, float lr, int step) {
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - std::pow(b1, (float)step), c2 = 1.f - std::pow(b2, (float)step);
  hipLaunchKernelGGL(k_mlp_update<true>, dim3((kMlpParams + 63) / 64), dim3(1024), 0, st, nparts, Gpart, losspart, P,
                     nullptr, M, V, loss, lr, b1, b2, eps, c1, c2);
  CHX_HIP(hipGetLastError());
}

void launch_mlp_reduce(hipStream_t st, int nparts, const float* Gpart, const float* losspart, float* G, float* loss) {
  hipLaunchKernelGGL(k_mlp_update<false>, dim3((kMlpParams + 63) / 64), dim3(1024), 0, st, nparts, Gpart, losspart,
                     nullptr, G, nullptr, nullptr, loss, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f);
  CHX_HIP(hipGetLastError());
}

void launch_mlp_features(hipStream_t st, long n, const double* rho, const double* sigma, const double* tau,
                         const int* codes, int ncodes, float* t, float* F) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mlp_features, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, rho, sigma, tau, codes,
                     ncodes, t, F);
  CHX_HIP(hipGetLastError());
}

void launch_mlp_eval(hipStream_t st, long n, const float* R, const unsigned* Wpk, const MlpBox& box, const int* codes,
                     int ncodes, const double* rho, const double* sigma, const double* tau, double* exc, double* vrho,
                     double* vsigma, double* vtau, int* nfall) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mlp_eval, dim3((unsigned)((n + kLanes - 1) / kLanes)), dim3(kLanes), 0, st, n, R,
                     reinterpret_cast<const u32x4_t*>(Wpk), box, codes, ncodes, rho, sigma, tau, exc, vrho, vsigma,
                     vtau, nfall);
  CHX_HIP(hipGetLastError());
}

void launch_functional_mlp(hipStream_t st, int nbatches, const int* grp_off, const double* part,
                           const double* part_tau, const double* bw, const float* R, const unsigned* Wpk,
                           const MlpBox& box, const int* codes, int ncodes, int want_e, int want_v, double* rho_out,
                           double* coef, double* en_part, int* nfall) {
  const int nslots = nbatches * kBatch;
  if (nslots == 0) return;
  hipLaunchKernelGGL(k_functional_mlp, dim3((unsigned)((nslots + kLanes - 1) / kLanes)), dim3(kLanes), 0, st, nslots,
                     grp_off, part, part_tau, bw, R, reinterpret_cast<const u32x4_t*>(Wpk), box, codes, ncodes, want_e,
                     want_v, rho_out, coef, en_part, nfall);
  CHX_HIP(hipGetLastError());
}

void launch_point_density(hipStream_t st, int nbatches, const int* grp_off, const double* part,
                          const double* part_tau, int has_tau, const double* bw, double* rho, double* sigma,
                          double* tau, double* w) {
  const int nslots = nbatches * kBatch;
  if (nslots == 0) return;
  hipLaunchKernelGGL(k_point_density, dim3((nslots + 255) / 256), dim3(256), 0, st, nslots, grp_off, part, part_tau,
                     has_tau, bw, rho, sigma, tau, w);
  CHX_HIP(hipGetLastError());
}

}  // namespace chx
