// Learned face flux: the encoding shared by the data dump, the training kernels and the
// surrogate-assisted step.
//
// A face is described in its normal frame after the floors and the GLM pair
// (glm_physics.jl:317-323): L, R = (rho, un, ua, ub, p, bn*, ba, bb). The network never
// sees raw left/right values (bfloat16 keeps ~3 significant digits, and the quantity of
// interest is a 2% difference); each of the 8 primitives enters as its face mean and its
// jump, both normalised by the local fast-speed scale a = sqrt((gamma p + |B|^2)/rho) of
// the mean state, and jumps are divided by the gate threshold so that gated faces give
// O(1) inputs:
//   x[2v]   = mean_v / scale_v,   x[2v+1] = (R_v - L_v) / (2 scale_v thr)
// with scale = (rho, a, a, a, rho a^2, a sqrt(rho), a sqrt(rho), a sqrt(rho)) of the mean.
// The network predicts the HLLD dissipation relative to the central flux,
//   y_k = (F_HLLD,k - (F(L)_k + F(R)_k)/2) / (thr s_k),
//   s = (rho a, rho a^2, rho a^2, rho a^2, rho a^3, -, a^2 sqrt(rho), a^2 sqrt(rho), -),
// so the flux is F = (F(L)+F(R))/2 + thr s y. The GLM slots (normal B and psi) are not
// learned: they are the exact glm_pair values.
// Gate (the jump detector): |drho|/rho and |dp|/p below thr, the jump of |B| relative to
// its mean at most thr (so that unmagnetised faces pass), and the low-density LLF switch
// not triggered.
#pragma once
#include "mhd_device.hpp"

namespace pmf {

constexpr int SURR_IN = 16, SURR_H = 64, SURR_OUT = 9;

struct SurrScales {
  float s[9];
};

// Encodes a normal-frame face (8 primitives each side, common bn). Returns the gate.
template <class T>
__device__ __forceinline__ bool surr_encode(const T* L, const T* R, T gamma, T thr, T* x, T* s) {
  const T rho = T(0.5) * (L[0] + R[0]);
  const T ir = rcp(rho);
  const T p = T(0.5) * (L[4] + R[4]);
  const T by = T(0.5) * (L[6] + R[6]), bz = T(0.5) * (L[7] + R[7]), bn = L[5];
  const T b2 = bn * bn + by * by + bz * bz;
  const T a2 = (gamma * p + b2) * ir;
  const T ia = rsq(a2);
  const T a = a2 * ia;
  const T sr = dsqrt(rho);
  const T isr = rcp(sr);
  const T sc[8] = {rho, a, a, a, rho * a2, a * sr, a * sr, a * sr};
  const T isc[8] = {ir, ia, ia, ia, ir * ia * ia, ia * isr, ia * isr, ia * isr};
  const T ith = rcp(T(2) * thr);
  (void)sc;
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    x[2 * v] = T(0.5) * (L[v] + R[v]) * isc[v];
    x[2 * v + 1] = (R[v] - L[v]) * isc[v] * ith;
  }
  s[0] = thr * rho * a;
  s[1] = s[2] = s[3] = thr * rho * a2;
  s[4] = thr * rho * a2 * a;
  s[5] = T(0);
  s[6] = s[7] = thr * a2 * sr;
  s[8] = T(0);
  const T bL = dsqrt(bn * bn + L[6] * L[6] + L[7] * L[7]);
  const T bR = dsqrt(bn * bn + R[6] * R[6] + R[7] * R[7]);
  const bool smooth = dabs(R[0] - L[0]) < thr * rho && dabs(R[4] - L[4]) < thr * p &&
                      dabs(bR - bL) <= thr * T(0.5) * (bL + bR);  // <=: unmagnetised faces pass
  return smooth;
}

// Central flux (F(L)+F(R))/2 in the normal frame (phys_flux_x, glm_physics.jl:28-34).
template <class T>
__device__ __forceinline__ void surr_central(const T* L, const T* R, T igm1, T* fc) {
  T qL[9] = {L[0], L[1], L[2], L[3], L[4], L[5], L[6], L[7], T(0)};
  T qR[9] = {R[0], R[1], R[2], R[3], R[4], R[5], R[6], R[7], T(0)};
  T fL[9], fR[9];
  dflux<0>(qL, fL, igm1);
  dflux<0>(qR, fR, igm1);
#pragma unroll
  for (int k = 0; k < 9; ++k) fc[k] = T(0.5) * (fL[k] + fR[k]);
}

// Normal-frame states after the floors and the GLM pair, and the exact GLM flux slots
// (the first part of riemann, glm_physics.jl:317-324). Returns the low-density switch.
template <class T>
__device__ __forceinline__ bool surr_prepare(T* L, T* R, const StepParams<T>& P, T& fbn, T& fpsi) {
  L[0] = dmax(L[0], P.smallr);
  L[4] = dmax(L[4], P.pfl);
  R[0] = dmax(R[0], P.smallr);
  R[4] = dmax(R[4], P.pfl);
  T bns;
  {
    // the GLM pair exactly as riemann_n evaluates it (no contraction)
#pragma clang fp contract(off)
    bns = T(0.5) * (L[5] + R[5]) - T(0.5) * (R[8] - L[8]) * P.ich;
    fbn = T(0.5) * (L[8] + R[8]) - T(0.5) * P.ch * (R[5] - L[5]);
    fpsi = P.ch2 * bns;
  }
  L[5] = bns;
  R[5] = bns;
  return (P.llf_dmin > T(0) && dmin(L[0], R[0]) < P.llf_dmin) ||
         (P.llf_pmin > T(0) && dmin(L[4], R[4]) < P.llf_pmin);
}

// tanh-form GELU, 0.5 z (1 + tanh(u)) with u = k0 (z + k1 z^3), evaluated as
// z * sigmoid(2u) = z / (1 + exp(-2u)) (one exp2, one reciprocal), and its derivative
// sigma + 2 z sigma (1 - sigma) k0 (1 + 3 k1 z^2); used identically in training and
// inference.
__device__ __forceinline__ float gelu(float z) {
  const float c1 = -2.0f * 1.4426950408889634f * 0.7978845608028654f, c3 = c1 * 0.044715f;
  const float e = __builtin_amdgcn_exp2f(z * __builtin_fmaf(c3, z * z, c1));  // exp(-2u)
  return z * __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float gelu_grad(float z) {
  const float k0 = 0.7978845608028654f, k1 = 0.044715f;
  const float c1 = -2.0f * 1.4426950408889634f * k0, c3 = c1 * k1;
  const float z2 = z * z;
  const float e = __builtin_amdgcn_exp2f(z * __builtin_fmaf(c3, z2, c1));
  const float sg = __builtin_amdgcn_rcpf(1.0f + e);
  return sg + 2.0f * z * sg * (1.0f - sg) * k0 * (1.0f + 3.0f * k1 * z2);
}

// float -> bfloat16, round to nearest even (the hardware v_cvt_pk_bf16_f32).
__device__ __forceinline__ unsigned short bf16_bits(float f) {
  return __builtin_bit_cast(unsigned short, (__bf16)f);
}

}  // namespace pmf

namespace pmf {

// LDS image of the network for wave-level inference: transposed weights W_l^T [out][in]
// in bfloat16 with rows padded by 4 (bank spread, 8-byte aligned MFMA A fragments), then the
// float32 biases (the output layer's padded to 32).
constexpr int SIMG_S1 = 16 + 4, SIMG_S2 = 64 + 4;
constexpr int SIMG_W1 = 0;                       // 64 x 20
constexpr int SIMG_W2 = SIMG_W1 + 64 * SIMG_S1;  // 64 x 68
constexpr int SIMG_W3 = SIMG_W2 + 64 * SIMG_S2;  // 64 x 68
constexpr int SIMG_W4 = SIMG_W3 + 64 * SIMG_S2;  // 9 x 68
constexpr int SIMG_NW = SIMG_W4 + SURR_OUT * SIMG_S2 + 4;  // bf16 entries, to a multiple of 16 bytes: 10600
constexpr int SIMG_NB = 64 * 3 + 32;             // float biases (output padded)
constexpr int SIMG_BYTES = SIMG_NW * 2 + SIMG_NB * 4;
static_assert(SIMG_NW * 2 % 16 == 0 && SIMG_W4 % 4 == 0, "aligned fragments and biases");

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef float sf32x16 __attribute__((ext_vector_type(16)));

// Eight bfloat16 weights of one row of the LDS image: four at column c0, four at c1.
__device__ __forceinline__ bf16x8 lds_frag8(const unsigned short* row, int c0, int c1) {
  const u16x4 a = *reinterpret_cast<const u16x4*>(row + c0);
  const u16x4 b = *reinterpret_cast<const u16x4*>(row + c1);
  s16x8 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    v[q] = (short)a[q];
    v[4 + q] = (short)b[q];
  }
  return __builtin_bit_cast(bf16x8, v);
}

// Accumulator initialised with the layer's biases: register r of lane half h holds unit
// 32 mb + 8 (r / 4) + 4 h + r % 4 (the 32x32 MFMA output layout).
__device__ __forceinline__ sf32x16 bias_acc(const float* b, int mb, int lh) {
  sf32x16 d;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float4 v = *reinterpret_cast<const float4*>(b + 32 * mb + 8 * r + 4 * lh);
    d[4 * r] = v.x;
    d[4 * r + 1] = v.y;
    d[4 * r + 2] = v.z;
    d[4 * r + 3] = v.w;
  }
  return d;
}

}  // namespace pmf


namespace pmf {

// The gated face flux in two halves around a batched network pass (the surrogate-assisted
// fused step queues the smooth faces of a whole tile plane and evaluates them in dense
// batches of 64, so waves whose faces are mostly rough do not run the network).
// surr_face_begin: lab-frame states in; in the normal frame, f is the exact flux of a
// rough face (HLLD, or LLF under the low-density switch) or the central flux of a smooth
// one with the exact GLM slots, s the output scales and x the 16 network inputs. Returns
// whether the face is smooth. Lanes with active false compute nothing of use.
template <int D>
__device__ __forceinline__ bool surr_face_begin(const float* Lq, const float* Rq, const StepParams<float>& P,
                                                float thr, bool active, float* f, float* s, float* x) {
  constexpr int N = D, A = (D + 1) % 3, B = (D + 2) % 3;
  float L[9] = {Lq[0], Lq[1 + N], Lq[1 + A], Lq[1 + B], Lq[4], Lq[5 + N], Lq[5 + A], Lq[5 + B], Lq[8]};
  float R[9] = {Rq[0], Rq[1 + N], Rq[1 + A], Rq[1 + B], Rq[4], Rq[5 + N], Rq[5 + A], Rq[5 + B], Rq[8]};
  float fbn, fpsi;
  const bool uself = surr_prepare(L, R, P, fbn, fpsi);
  const bool smooth = surr_encode(L, R, P.gamma, thr, x, s) && !uself && active;
  const bool rough = active && !smooth;
  if (rough) {
    if (uself) llf_n(L, R, P.ch, fbn, fpsi, f, P);
    else hlld_n(L, R, L[5], fbn, fpsi, f, P);
  }
  if (smooth) {
    surr_central(L, R, P.igm1, f);
    f[5] = fbn;
    f[8] = fpsi;
  }
  return smooth;
}

// surr_face_end: adds the learned dissipation y (smooth faces) and rotates to the lab frame.
template <int D>
__device__ __forceinline__ void surr_face_end(float* f, const float* s, const float* y, bool smooth, float* F) {
  constexpr int N = D, A = (D + 1) % 3, B = (D + 2) % 3;
  if (smooth) {
#pragma unroll
    for (int k = 0; k < 9; ++k)
      if (k != 5 && k != 8) f[k] = f[k] + s[k] * y[k];
  }
  F[0] = f[0];
  F[1 + N] = f[1];
  F[1 + A] = f[2];
  F[1 + B] = f[3];
  F[4] = f[4];
  F[5 + N] = f[5];
  F[5 + A] = f[6];
  F[5 + B] = f[7];
  F[8] = f[8];
}

// LDS queue of the smooth faces of one tile plane: one 32-byte slot per face holding its
// 16 network inputs as bfloat16 (the precision the network reads them in), which the
// network pass overwrites with the seven learned outputs in float32 (the GLM slots 5 and
// 8 are exact and not learned).
constexpr int SURR_QOUT = 7;
__device__ __forceinline__ constexpr int surr_qk(int j) { return j < 5 ? j : j + 1; }  // output slot j -> k

template <int CAP>
struct SurrQueue {
  unsigned n;
  unsigned pad[3];
  uint4 slot[CAP * 2];  // 32 bytes per face
};

// Appends the calling lanes' faces that want a slot (one LDS atomic per wave); returns
// the slot, or -1.
template <int CAP>
__device__ __forceinline__ int surr_enqueue(bool want, const float* x, SurrQueue<CAP>& Q) {
  const unsigned long long b = __ballot(want);
  if (b == 0ull) return -1;
  const int lane = threadIdx.x & 63;
  const int leader = __builtin_ctzll(b);
  unsigned base = 0;
  if (lane == leader) base = atomicAdd(&Q.n, (unsigned)__popcll(b));
  base = __shfl(base, leader, 64);
  if (!want) return -1;
  const int slot = int(base) + __popcll(b & ((1ull << lane) - 1ull));
  unsigned w[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) w[k] = (unsigned)bf16_bits(x[2 * k]) | ((unsigned)bf16_bits(x[2 * k + 1]) << 16);
  Q.slot[2 * slot] = make_uint4(w[0], w[1], w[2], w[3]);
  Q.slot[2 * slot + 1] = make_uint4(w[4], w[5], w[6], w[7]);
  return slot;
}

// One batch of up to 32 queued faces (slots b .. b+31 below nq), evaluated by the calling wave;
// all its lanes must call it. img: the network's image, in LDS. Units are the MFMA rows and
// faces the columns; v_mfma_f32_32x32x16_bf16 contracts 16 units per step. A slot's 32 bytes
// are the two lane halves' B fragments of the first layer as they stand; the hidden layers'
// contraction order is permuted so that accumulator registers 8s..8s+7 of a lane are its B
// fragment for step s of the next layer (lane half h then holds units 16s + 4h + {0..3} and
// 16s + 8 + 4h + {0..3}; the weight fragments read the same units); and the outputs leave from
// the registers they arrive in (lane half 0: 0..3, half 1: 4..7, 5 not learned). So
// activations never leave registers and no lane exchanges anything. The two accumulators'
// chains alternate and a layer's weights are read before the activations that they wait for.
// Bound: the 96 GELUs a lane (two quarter-rate and five full-rate operations each) at two
// waves per SIMD. Through arrays in scratch memory, lane shuffles, biases in global memory
// and one accumulator after the other a 192^3 step with 0.90 / 0.31 / 0.11 of its faces in the
// network took 2.71 / 1.53 / 1.11 ms, now 2.19 / 1.31 / 0.99. A function of its own, for one
// batch: inlined, with the loop inside, or for two batches at once its registers push the
// step's own carries into scratch (a step without network faces 0.56 -> 1.39 / 0.64 / 1.07 ms).
template <int CAP>
__device__ __attribute__((noinline)) void surr_batch(int b, int nq, SurrQueue<CAP>& Q, const unsigned short* img) {
  const int lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5;
  const float* bias = reinterpret_cast<const float*>(img + SIMG_NW);
  const int slot = min(b + li, nq - 1);  // lanes past the end repeat the last face
  bf16x8 w[2][4], f[4];
  f[0] = __builtin_bit_cast(bf16x8, Q.slot[2 * slot + lh]);
  sf32x16 d[2];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
    d[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        lds_frag8(img + SIMG_W1 + (mb * 32 + li) * SIMG_S1, 8 * lh, 8 * lh + 4), f[0], bias_acc(bias, mb, lh), 0, 0, 0);
#pragma unroll 1
  for (int layer = 1; layer < 3; ++layer) {
    const unsigned short* row = img + (layer == 1 ? SIMG_W2 : SIMG_W3) + li * SIMG_S2;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int st = 0; st < 4; ++st)
        w[mb][st] = lds_frag8(row + mb * 32 * SIMG_S2, 16 * st + 4 * lh, 16 * st + 8 + 4 * lh);
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int q = 0; q < 8; ++q) f[st][q] = (__bf16)gelu(d[st >> 1][8 * (st & 1) + q]);
    d[0] = bias_acc(bias + 64 * layer, 0, lh);
    d[1] = bias_acc(bias + 64 * layer, 1, lh);
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) d[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[mb][st], f[st], d[mb], 0, 0, 0);
  }
  // output layer: rows past the nine outputs are never read
  const unsigned short* row = img + SIMG_W4 + min(li, SURR_OUT - 1) * SIMG_S2;
#pragma unroll
  for (int st = 0; st < 4; ++st) w[0][st] = lds_frag8(row, 16 * st + 4 * lh, 16 * st + 8 + 4 * lh);
#pragma unroll
  for (int st = 0; st < 4; ++st)
#pragma unroll
    for (int q = 0; q < 8; ++q) f[st][q] = (__bf16)gelu(d[st >> 1][8 * (st & 1) + q]);
  sf32x16 o = bias_acc(bias + 192, 0, lh);
#pragma unroll
  for (int st = 0; st < 4; ++st) o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[0][st], f[st], o, 0, 0, 0);
  // the slots' inputs were read above by this wave, the only one that touches them
  if (b + li < nq) {
    float4 v = make_float4(o[0], o[1], o[2], o[3]);
    if (lh) v = make_float4(o[0], o[2], o[3], 0.f);
    *reinterpret_cast<float4*>(&Q.slot[2 * slot + lh]) = v;
  }
}

// The learned outputs of queue slot q (zeros for q < 0), after the network pass.
template <int CAP>
__device__ __forceinline__ void surr_result(const SurrQueue<CAP>& Q, int q, float* y) {
#pragma unroll
  for (int k = 0; k < SURR_OUT; ++k) y[k] = 0.f;
  if (q >= 0) {
    const float* in = reinterpret_cast<const float*>(&Q.slot[2 * q]);
#pragma unroll
    for (int j = 0; j < SURR_QOUT; ++j) y[surr_qk(j)] = in[j];
  }
}

}  // namespace pmf
