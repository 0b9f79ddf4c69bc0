// The learned face flux: data dump from the plain solver, training kernels (bfloat16
// operands on MFMA with float32 accumulation, float32 master weights, Adam), batch
// evaluation, and the host entry points (declared in include/pmfmhd.h).
//
// Network: 16 -> 64 -> 64 -> 64 -> 9, tanh-form GELU, y = W4^T g(W3^T g(W2^T g(W1^T x +
// b1) + b2) + b3) + b4. Weights are stored W_l[in][out] row-major; the flat parameter
// vector is [W1 b1 W2 b2 W3 b3 W4 b4] (9993 floats). Encoding of x and y: surrogate.hpp.
#include <cmath>
#include <cstring>
#include <random>

#include "cellpredict.hpp"
#include "state.hpp"
#include "surrogate.hpp"

namespace pmf {

constexpr int NPARAM = 16 * 64 + 64 + 64 * 64 + 64 + 64 * 64 + 64 + 64 * 9 + 9;  // 9993
constexpr int LAYER_IN[4] = {16, 64, 64, 64};
constexpr int LAYER_OUT[4] = {64, 64, 64, 9};

__host__ __device__ constexpr int w_off(int l) {
  return l == 0 ? 0 : l == 1 ? 16 * 64 + 64 : l == 2 ? 16 * 64 + 64 + 64 * 64 + 64 : 16 * 64 + 64 + 2 * (64 * 64 + 64);
}
__host__ __device__ constexpr int b_off(int l) { return w_off(l) + LAYER_IN[l] * LAYER_OUT[l]; }

// ---------------------------------------------------------------------------
// The network over a batch: forward pass, and for training the loss and the whole gradient,
// in one kernel. A workgroup (four waves) takes tiles of 32 samples; wave w owns units
// 16w..16w+15 of each hidden layer, so a layer is four 16x16 MFMA tiles' worth of latency
// and eight activations a lane. Products have units as rows and samples as columns
// (W^T x, W dz) and, for the weight gradients, contract the tile's 32 samples in one MFMA.
// Activations and dz go through LDS twice, as [sample][unit] for the next layer's product
// and as [unit][sample] for the weight gradient; the weights sit there as [out][in] and
// [in][out]. Weight gradients stay in registers over a workgroup's tiles (40 a lane) and
// leave as one partial per workgroup; k_net_update folds the partials.
//
// Bound: latency (a chain of eight layers with a barrier each). Layer by layer through
// global memory, the weight gradients' 64x64 results left one workgroup walking all
// samples: 6.9 ms a step at batch 8192 (27 launches); this kernel and the update: see
// pmf_surrogate_train.
//
// BF16: operands rounded to bfloat16 (v_mfma_f32_16x16x32_bf16), otherwise float32
// (v_mfma_f32_16x16x4_f32, eight per 32 of the contraction); accumulation in float32, bias
// gradients and the loss in float64. Lane layout (16x16, wave64): A[i][k] and B[k][j] from
// lane (i or j) + 16 g with k = 8 g + q, q = 0..7 (any order of k serves, as A and B share
// it); D[i][j] in lane j + 16 (i / 4), register i % 4.
constexpr int NET_TILE = 32, NET_THREADS = 256, NET_MAX_WG = 256;
constexpr int NET_DSLOTS = 3 * 64 + 2 * 16 + 2;  // float64 partials: three bias layers, the output layer and loss by wave

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <bool BF16> struct NetOps;
template <> struct NetOps<true> {
  typedef unsigned short E;
  typedef bf16x8 Frag;
  static constexpr int S64 = 72, S16 = 24, ST = 40;  // row strides: 16-byte aligned, spread over the banks
  static __device__ __forceinline__ E put(float v) { return bf16_bits(v); }
  static __device__ __forceinline__ Frag load(const E* p) { return __builtin_bit_cast(Frag, *reinterpret_cast<const uint4*>(p)); }
  static __device__ __forceinline__ Frag zero() { return __builtin_bit_cast(Frag, make_uint4(0, 0, 0, 0)); }
  static __device__ __forceinline__ f32x4 mma(Frag a, Frag b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ void put4(E* p, const float* v) {
    *reinterpret_cast<uint2*>(p) = make_uint2((unsigned)put(v[0]) | ((unsigned)put(v[1]) << 16),
                                              (unsigned)put(v[2]) | ((unsigned)put(v[3]) << 16));
  }
};
template <> struct NetOps<false> {
  typedef float E;
  struct Frag {
    float4 a, b;
  };
  static constexpr int S64 = 68, S16 = 20, ST = 36;
  static __device__ __forceinline__ E put(float v) { return v; }
  static __device__ __forceinline__ Frag load(const E* p) {
    const float4* v = reinterpret_cast<const float4*>(p);
    return Frag{v[0], v[1]};
  }
  static __device__ __forceinline__ Frag zero() { return Frag{make_float4(0, 0, 0, 0), make_float4(0, 0, 0, 0)}; }
  static __device__ __forceinline__ f32x4 mma(const Frag& a, const Frag& b, f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.a.x, b.a.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.a.y, b.a.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.a.z, b.a.z, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.a.w, b.a.w, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.b.x, b.b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.b.y, b.b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.b.z, b.b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.b.w, b.b.w, c, 0, 0, 0);
  }
  static __device__ __forceinline__ void put4(E* p, const float* v) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  }
};

template <bool BF16, bool TRAIN> struct __attribute__((aligned(16))) NetLds {
  typedef NetOps<BF16> O;
  typename O::E f1[64 * O::S16], f2[64 * O::S64], f3[64 * O::S64], f4[16 * O::S64];           // weights [out][in]
  typename O::E b2[TRAIN ? 64 * O::S64 : 8], b3[TRAIN ? 64 * O::S64 : 8], b4[TRAIN ? 64 * O::S16 : 8];  // [in][out]
  typename O::E f[2][NET_TILE * O::S64];                                                      // [sample][unit]
  typename O::E tx[TRAIN ? 16 * O::ST : 8], ta[TRAIN ? 3 : 1][TRAIN ? 64 * O::ST : 8];        // inputs [unit][sample]
  typename O::E td[TRAIN ? 2 : 1][TRAIN ? 64 * O::ST : 8];                                    // dz [unit][sample]
  float bias[3 * 64 + 16];
};

// Sample of minibatch row r: hashed, with replacement.
__device__ __forceinline__ int64_t batch_sample(unsigned long long key, int64_t r, int64_t n) {
  unsigned long long z = key + (unsigned long long)r * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (int64_t)(z % (unsigned long long)n);
}

// rows samples of X (16 each): the rows themselves, or with pick the hashed minibatch of ndata
// samples. TRAIN: targets Tg (9 each); per-workgroup gradient partials part (NPARAM floats)
// and dpart (NET_DSLOTS doubles). Otherwise the outputs Y (9 each).
template <bool BF16, bool TRAIN>
__global__ __launch_bounds__(NET_THREADS) void k_net(const float* __restrict__ w, const float* __restrict__ X,
                                                     const float* __restrict__ Tg, int64_t ndata, int pick,
                                                     unsigned long long key, int64_t rows, float* __restrict__ Y,
                                                     float* __restrict__ part, double* __restrict__ dpart) {
  typedef NetOps<BF16> O;
  typedef typename O::Frag Frag;
  __shared__ NetLds<BF16, TRAIN> S;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int lj = lane & 15, lg = lane >> 4;
  const int u0 = 16 * wave + 4 * lg;  // first of this lane's four units in a hidden layer
  // weights (all loads in flight together) and biases
  {
    float4 v[9];
    v[0] = reinterpret_cast<const float4*>(w + w_off(0))[t];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[1 + k] = reinterpret_cast<const float4*>(w + w_off(1))[t + k * NET_THREADS];
      v[5 + k] = reinterpret_cast<const float4*>(w + w_off(2))[t + k * NET_THREADS];
    }
    // element e of a layer is W[i = e / out][o = e % out]
    auto spread = [&](float4 x, int e, typename O::E* fw, int st, typename O::E* bw) {
      const float c[4] = {x.x, x.y, x.z, x.w};
      const int i = e >> 6, o = e & 63;
#pragma unroll
      for (int q = 0; q < 4; ++q) fw[(o + q) * st + i] = O::put(c[q]);
      if (bw) O::put4(bw + i * O::S64 + o, c);
    };
    spread(v[0], 4 * t, S.f1, O::S16, nullptr);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int e = 4 * (t + k * NET_THREADS);
      spread(v[1 + k], e, S.f2, O::S64, TRAIN ? S.b2 : nullptr);
      spread(v[5 + k], e, S.f3, O::S64, TRAIN ? S.b3 : nullptr);
    }
  }
#pragma unroll
  for (int k = 0; k < 64 * 16 / NET_THREADS; ++k) {
    const int e = t + k * NET_THREADS, i = e >> 4, o = e & 15;
    const typename O::E v = O::put(o < 9 ? w[w_off(3) + i * 9 + o] : 0.f);
    S.f4[o * O::S64 + i] = v;
    if constexpr (TRAIN) S.b4[i * O::S16 + o] = v;
  }
  if (t < 192) S.bias[t] = w[b_off(t >> 6) + (t & 63)];
  else if (t < 208) S.bias[t] = t - 192 < 9 ? w[b_off(3) + t - 192] : 0.f;

  f32x4 g1 = {0, 0, 0, 0}, g2[4], g3[4], g4 = {0, 0, 0, 0};  // weight gradients
  double db[3][4], db4[4], loss = 0.0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    g2[q] = g3[q] = f32x4{0, 0, 0, 0};
    db[0][q] = db[1][q] = db[2][q] = db4[q] = 0.0;
  }
  const float scale = float(rows * 7);
  const int64_t ntiles = (rows + NET_TILE - 1) / NET_TILE;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t r0 = tile * NET_TILE;
    {
      const int s = t >> 3, c = (t & 7) * 2;
      float2 x = make_float2(0.f, 0.f);
      if (r0 + s < rows) {
        const int64_t i = pick ? batch_sample(key, r0 + s, ndata) : r0 + s;
        x = *reinterpret_cast<const float2*>(X + i * 16 + c);
      }
      S.f[0][s * O::S64 + c] = O::put(x.x);
      S.f[0][s * O::S64 + c + 1] = O::put(x.y);
      if constexpr (TRAIN) {
        S.tx[c * O::ST + s] = O::put(x.x);
        S.tx[(c + 1) * O::ST + s] = O::put(x.y);
      }
    }
    // the output layer's lanes (waves 0 and 1, one block of 16 samples each) take their targets early
    const int64_t row = r0 + 16 * wave + lj;
    const bool live = wave < 2 && row < rows;
    float tg[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (TRAIN) {
      if (live) {
        const int64_t i = pick ? batch_sample(key, row, ndata) : row;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (4 * lg + q < 9) tg[q] = Tg[i * 9 + 4 * lg + q];
      }
    }
    __syncthreads();
    float gp[3][2][4];  // GELU'(z) of this lane's units
    // hidden layer l from [sample][unit] buffer in to buffer out
    auto hidden = [&](int l, const typename O::E* W, int nk, const typename O::E* in, typename O::E* out) {
      Frag a[2], b[2][2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if (k >= nk) break;
        const bool in16 = nk == 1;  // 16 inputs: the upper half of the contraction is zero
        const int st = in16 ? O::S16 : O::S64;
        a[k] = in16 && lg >= 2 ? O::zero() : O::load(W + (16 * wave + lj) * st + 32 * k + 8 * lg);
#pragma unroll
        for (int fb = 0; fb < 2; ++fb)
          b[fb][k] = in16 && lg >= 2 ? O::zero() : O::load(in + (16 * fb + lj) * O::S64 + 32 * k + 8 * lg);
      }
#pragma unroll
      for (int fb = 0; fb < 2; ++fb) {
        f32x4 d = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          if (k >= nk) break;
          d = O::mma(a[k], b[fb][k], d);
        }
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float z = d[q] + S.bias[64 * l + u0 + q];
          v[q] = gelu(z);
          if constexpr (TRAIN) gp[l][fb][q] = gelu_grad(z);
        }
        O::put4(out + (16 * fb + lj) * O::S64 + u0, v);
        if constexpr (TRAIN) {
#pragma unroll
          for (int q = 0; q < 4; ++q) S.ta[l][(u0 + q) * O::ST + 16 * fb + lj] = O::put(v[q]);
        }
      }
      __syncthreads();
    };
    hidden(0, S.f1, 1, S.f[0], S.f[1]);
    hidden(1, S.f2, 2, S.f[1], S.f[0]);
    hidden(2, S.f3, 2, S.f[0], S.f[1]);
    // output layer
    if (wave < 2) {
      f32x4 d = {0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < 2; ++k)
        d = O::mma(O::load(S.f4 + lj * O::S64 + 32 * k + 8 * lg),
                   O::load(S.f[1] + (16 * wave + lj) * O::S64 + 32 * k + 8 * lg), d);
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int o = 4 * lg + q;
        const float y = d[q] + S.bias[192 + o];
        if constexpr (TRAIN) {
          // loss gradient 2 (y - target) / (rows * 7) on the learned slots (0-4, 6, 7)
          const float e = live && o < 8 && o != 5 ? y - tg[q] : 0.f;
          v[q] = 2.f * e / scale;
          loss += (double)e * e;
          db4[q] += (double)v[q];
          S.td[0][o * O::ST + 16 * wave + lj] = O::put(v[q]);
        } else if (live && o < 9) {
          Y[row * 9 + o] = y;
        }
      }
      if constexpr (TRAIN) O::put4(S.f[0] + (16 * wave + lj) * O::S64 + 4 * lg, v);
    }
    if constexpr (TRAIN) {
      __syncthreads();
      // dz of hidden layer l from the layer above (W: [in][out], dz in buffer in, 16 of them
      // or 64), to buffer out and td[o]
      auto back = [&](int l, const typename O::E* W, int nk, const typename O::E* in, typename O::E* out, int o) {
#pragma unroll
        for (int fb = 0; fb < 2; ++fb) {
          f32x4 d = {0, 0, 0, 0};
          const bool in16 = nk == 1;
          const int st = in16 ? O::S16 : O::S64;
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            if (k >= nk) break;
            const Frag a = in16 && lg >= 2 ? O::zero() : O::load(W + (16 * wave + lj) * st + 32 * k + 8 * lg);
            const Frag b = in16 && lg >= 2 ? O::zero() : O::load(in + (16 * fb + lj) * O::S64 + 32 * k + 8 * lg);
            d = O::mma(a, b, d);
          }
          float v[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            v[q] = d[q] * gp[l][fb][q];
            db[l][q] += (double)v[q];
            S.td[o][(u0 + q) * O::ST + 16 * fb + lj] = O::put(v[q]);
          }
          if (out) O::put4(out + (16 * fb + lj) * O::S64 + u0, v);
        }
      };
      // one 16x16 block of a weight gradient: input units from A, output units from row n of td
      auto grad = [&](const typename O::E* A, int k, const typename O::E* D, int n, f32x4 g) {
        return O::mma(O::load(A + (k + lj) * O::ST + 8 * lg), O::load(D + (n + lj) * O::ST + 8 * lg), g);
      };
      back(2, S.b4, 1, S.f[0], S.f[1], 1);
      g4 = grad(S.ta[2], 16 * wave, S.td[0], 0, g4);
      __syncthreads();
      back(1, S.b3, 2, S.f[1], S.f[0], 0);
#pragma unroll
      for (int n = 0; n < 4; ++n) g3[n] = grad(S.ta[1], 16 * wave, S.td[1], 16 * n, g3[n]);
      __syncthreads();
      back(0, S.b2, 2, S.f[0], nullptr, 1);
#pragma unroll
      for (int n = 0; n < 4; ++n) g2[n] = grad(S.ta[0], 16 * wave, S.td[0], 16 * n, g2[n]);
      __syncthreads();
      g1 = grad(S.tx, 0, S.td[1], 16 * wave, g1);
    }
    __syncthreads();  // the next tile overwrites the buffers
  }
  if constexpr (TRAIN) {
    float* p = part + (int64_t)blockIdx.x * NPARAM;
    double* dp = dpart + (int64_t)blockIdx.x * NET_DSLOTS;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      p[w_off(0) + (4 * lg + q) * 64 + 16 * wave + lj] = g1[q];
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        p[w_off(1) + (u0 + q) * 64 + 16 * n + lj] = g2[n][q];
        p[w_off(2) + (u0 + q) * 64 + 16 * n + lj] = g3[n][q];
      }
      if (lj < 9) p[w_off(3) + (u0 + q) * 9 + lj] = g4[q];
#pragma unroll
      for (int m = 1; m < 16; m <<= 1) {
#pragma unroll
        for (int l = 0; l < 3; ++l) db[l][q] += __shfl_xor(db[l][q], m, 64);
        db4[q] += __shfl_xor(db4[q], m, 64);
      }
      if (lj == 0) {
#pragma unroll
        for (int l = 0; l < 3; ++l) dp[64 * l + u0 + q] = db[l][q];
        if (wave < 2) dp[192 + 16 * wave + 4 * lg + q] = db4[q];
      }
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) loss += __shfl_xor(loss, m, 64);
    if (lane == 0 && wave < 2) dp[224 + wave] = loss;
  }
}

// Folds the nwg gradient partials in float64 (64 parameters a block, 16 waves share the
// partials) into g and, with adam, takes one Adam step; the entry past the last parameter
// is the loss. Reads 40 KB a partial: 7 us for 256, 2.4 us for one.
__global__ __launch_bounds__(1024) void k_net_update(const float* __restrict__ part, const double* __restrict__ dpart,
                                                     int nwg, float* __restrict__ g, double* __restrict__ loss,
                                                     double loss_scale, int adam, float* __restrict__ w,
                                                     float* __restrict__ m, float* __restrict__ v, float lr, float b1, float b2, float eps,
                                                     float c1, float c2) {
  __shared__ double sh[16][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int e = blockIdx.x * 64 + lane;
  int slot = -1;  // float64 partial of a bias or of the loss (the output layer's and the loss have two)
#pragma unroll
  for (int l = 0; l < 4; ++l)
    if (e >= b_off(l) && e < b_off(l) + LAYER_OUT[l]) slot = 64 * l + e - b_off(l);
  if (e == NPARAM) slot = 224;
  const int twin = slot >= 224 ? 1 : slot >= 192 ? 16 : 0;
  double s = 0.0;
  if (e <= NPARAM) {
    if (slot < 0) {
      // NET_MAX_WG / 16 partials a wave, all loads in flight together
      float v[NET_MAX_WG / 16];
#pragma unroll
      for (int k = 0; k < NET_MAX_WG / 16; ++k) v[k] = part[min(wave + 16 * k, nwg - 1) * NPARAM + e];
#pragma unroll
      for (int k = 0; k < NET_MAX_WG / 16; ++k) s += wave + 16 * k < nwg ? (double)v[k] : 0.0;
    } else {
      for (int p = wave; p < nwg; p += 16) {
        const double* d = dpart + (int64_t)p * NET_DSLOTS + slot;
        s += d[0];
        if (twin) s += d[twin];
      }
    }
  }
  sh[wave][lane] = s;
  __syncthreads();
  if (wave != 0 || e > NPARAM) return;
#pragma unroll
  for (int k = 1; k < 16; ++k) s += sh[k][lane];
  if (e == NPARAM) {
    *loss = s * loss_scale;
    return;
  }
  const float gi = (float)s;
  g[e] = gi;
  if (adam) {
    const float mi = b1 * m[e] + (1.f - b1) * gi;
    const float vi = b2 * v[e] + (1.f - b2) * gi * gi;
    m[e] = mi;
    v[e] = vi;
    w[e] -= lr * (mi * c1) / (__builtin_sqrtf(vi * c2) + eps);
  }
}

// ---------------------------------------------------------------------------
// Face dump: every lower face of every cell (x, y, z) of the current state, predicted
// exactly as the per-cell step does; gated faces are kept with probability keep and
// appended as (x[16], y[9], state[18]) where state = normal-frame L[8], R[8], fbn, fpsi.
__global__ __launch_bounds__(256) void k_dump_faces(Fields<const float> U, Grid G, StepParams<float> P, float thr,
                                                    float keep, unsigned long long key, float* __restrict__ X,
                                                    float* __restrict__ Y, float* __restrict__ S,
                                                    unsigned long long* __restrict__ count, int64_t cap) {
  int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= G.nc) return;
  const int i = (int)(c % G.nx), j = (int)((c / G.nx) % G.ny), k = (int)(c / ((int64_t)G.nx * G.ny));
  float mh[9], dL[3][9], dR[3][9], mhn[9], dLn[3][9], dRn[3][9];
  predict_cell<RECON_PLM_MINMOD>(U, G, i, j, k, P, mh, dL, dR);
  for (int d = 0; d < 3; ++d) {
    unsigned long long z = key ^ ((unsigned long long)c * 3 + d) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    if ((float)(z >> 40) * (1.0f / 16777216.0f) >= keep) continue;
    predict_cell<RECON_PLM_MINMOD>(U, G, i - (d == 0), j - (d == 1), k - (d == 2), P, mhn, dLn, dRn);
    float Lq[9], Rq[9];
    for (int v = 0; v < 9; ++v) {
      Lq[v] = mhn[v] + dRn[d][v];
      Rq[v] = mh[v] + dL[d][v];
    }
    const int N = d, A = (d + 1) % 3, B = (d + 2) % 3;
    float L[9] = {Lq[0], Lq[1 + N], Lq[1 + A], Lq[1 + B], Lq[4], Lq[5 + N], Lq[5 + A], Lq[5 + B], Lq[8]};
    float R[9] = {Rq[0], Rq[1 + N], Rq[1 + A], Rq[1 + B], Rq[4], Rq[5 + N], Rq[5 + A], Rq[5 + B], Rq[8]};
    float fbn, fpsi;
    bool uself = surr_prepare(L, R, P, fbn, fpsi);
    float x[16], s[9];
    bool smooth = surr_encode(L, R, P.gamma, thr, x, s);
    if (!smooth || uself) continue;
    float fh[9], fc[9];
    hlld_n(L, R, L[5], fbn, fpsi, fh, P);
    surr_central(L, R, P.igm1, fc);
    unsigned long long slot = atomicAdd(count, 1ull);
    if ((int64_t)slot >= cap) continue;
    for (int q = 0; q < 16; ++q) X[slot * 16 + q] = x[q];
    for (int q = 0; q < 9; ++q) Y[slot * 9 + q] = (q == 5 || q == 8) ? 0.f : (fh[q] - fc[q]) / s[q];
    for (int q = 0; q < 8; ++q) {
      S[slot * 18 + q] = L[q];
      S[slot * 18 + 8 + q] = R[q];
    }
    S[slot * 18 + 16] = fbn;
    S[slot * 18 + 17] = fpsi;
  }
}

// Face fluxes of dumped states: mode 0 = HLLD, 1 = central + thr s y (surrogate), 2 =
// central only (the method without the learned correction).
__global__ __launch_bounds__(256) void k_face_flux(const float* __restrict__ S, const float* __restrict__ Yp, int64_t n,
                                                   StepParams<float> P, float thr, int mode, float* __restrict__ F) {
  int64_t f = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (f >= n) return;
  float L[9], R[9];
  for (int q = 0; q < 8; ++q) {
    L[q] = S[f * 18 + q];
    R[q] = S[f * 18 + 8 + q];
  }
  L[8] = R[8] = 0.f;
  const float fbn = S[f * 18 + 16], fpsi = S[f * 18 + 17];
  float out[9];
  if (mode == 0) {
    hlld_n(L, R, L[5], fbn, fpsi, out, P);
  } else {
    float x[16], s[9], fc[9];
    surr_encode(L, R, P.gamma, thr, x, s);
    surr_central(L, R, P.igm1, fc);
    for (int q = 0; q < 9; ++q) out[q] = fc[q] + (mode == 1 ? s[q] * Yp[f * 9 + q] : 0.f);
    out[5] = fbn;
    out[8] = fpsi;
  }
  for (int q = 0; q < 9; ++q) F[f * 9 + q] = out[q];
}

// The network's LDS image for the surrogate-assisted step (layout in surrogate.hpp):
// transposed bfloat16 weights with padded rows, then the float32 biases.
__global__ __launch_bounds__(256) void k_surr_image(const float* __restrict__ w, unsigned char* __restrict__ img) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  unsigned short* W = reinterpret_cast<unsigned short*>(img);
  float* B = reinterpret_cast<float*>(img + SIMG_NW * 2);
  if (e < SIMG_NW) {
    float val = 0.f;
    if (e < SIMG_W2) {
      int r = e / SIMG_S1, c = e % SIMG_S1;
      if (c < 16) val = w[w_off(0) + c * 64 + r];
    } else if (e < SIMG_W4) {
      int l = e < SIMG_W3 ? 1 : 2, o = e - (l == 1 ? SIMG_W2 : SIMG_W3);
      int r = o / SIMG_S2, c = o % SIMG_S2;
      if (c < 64) val = w[w_off(l) + c * 64 + r];
    } else {
      int o = e - SIMG_W4, r = o / SIMG_S2, c = o % SIMG_S2;
      if (r < 9 && c < 64) val = w[w_off(3) + c * 9 + r];
    }
    W[e] = bf16_bits(val);
  }
  if (e < SIMG_NB) {
    float val = 0.f;
    if (e < 192) val = w[b_off(e / 64) + e % 64];
    else if (e - 192 < 9) val = w[b_off(3) + e - 192];
    B[e] = val;
  }
}

__global__ void k_zero_u64(unsigned long long* p) { *p = 0ull; }

}  // namespace pmf

// ---------------------------------------------------------------------------
// Host side.
using namespace pmf;

struct pmf_surrogate {
  pmf_state* s = nullptr;  // parameters and stream (not owned)
  float* w = nullptr;      // NPARAM master weights
  float* g = nullptr;      // gradient
  float* m = nullptr;      // Adam moments
  float* v = nullptr;
  int64_t adam_t = 0;
  // dataset
  float *X = nullptr, *Y = nullptr, *S = nullptr;
  int64_t cap = 0, n = 0;
  unsigned long long* dcount = nullptr;
  float* part = nullptr;  // gradient partials of NET_MAX_WG workgroups
  double* dpart = nullptr;
  float *Yb = nullptr, *Fb = nullptr;  // outputs and fluxes of out_rows samples
  int64_t out_rows = 0;
  double* dloss = nullptr;  // one loss per step, loss_steps of them
  int64_t loss_steps = 0;
  unsigned char* img = nullptr;         // LDS image for the surrogate-assisted step
  unsigned long long* nsmooth = nullptr;  // faces solved by the network in the last step
};

namespace {

// At least `want` elements of `each` T. The old buffer goes only when the new one is there: if the
// device has no room, p stays what it was (later calls rely on one loss).
template <class T> void grow(T*& p, int64_t& have, int64_t want, int64_t each) {
  if (want <= have) return;
  T* q = nullptr;
  hip_check(hipMalloc(&q, sizeof(T) * each * want), "hipMalloc");
  (void)hipFree(p);
  p = q;
  have = want;
}

void ensure_outputs(pmf_surrogate* n, int64_t rows) {
  if (rows <= n->out_rows) return;
  int64_t have = 0;
  (void)hipFree(n->Fb);
  n->Fb = nullptr;
  n->out_rows = 0;
  (void)hipFree(n->Yb);
  n->Yb = nullptr;
  grow(n->Yb, have, rows, 9);
  have = 0;
  grow(n->Fb, have, rows, 9);
  n->out_rows = rows;
}

unsigned blocks(int64_t n) { return (unsigned)((n + 255) / 256); }

// Outputs Yb of rows samples X (row-major rows x 16).
void forward(pmf_surrogate* n, const float* X, int64_t rows, bool bf16) {
  const int64_t tiles = (rows + NET_TILE - 1) / NET_TILE;
  const dim3 grd((unsigned)std::min<int64_t>(tiles, 4 * NET_MAX_WG)), blk(NET_THREADS);
  hipStream_t st = n->s->st;
#define PMF_NET(B) \
  hipLaunchKernelGGL((k_net<B, false>), grd, blk, 0, st, n->w, X, nullptr, 0, 0, 0ull, rows, n->Yb, nullptr, nullptr)
  if (bf16) PMF_NET(true);
  else PMF_NET(false);
#undef PMF_NET
}

struct Adam {
  int on = 0;  // 0: gradient only
  float lr = 0.f, b1 = 0.f, b2 = 0.f, eps = 0.f, c1 = 0.f, c2 = 0.f;
};

// Gradient of the mean-squared loss over rows samples (pick: the hashed minibatch of key, of the
// whole dataset) into n->g, the loss into *loss, and the Adam step.
void learn(pmf_surrogate* n, const float* X, const float* Tg, int64_t rows, bool pick, unsigned long long key,
           bool bf16, double* loss, const Adam& a) {
  const int64_t tiles = (rows + NET_TILE - 1) / NET_TILE;
  const int nwg = (int)std::min<int64_t>(tiles, NET_MAX_WG);
  const dim3 grd(nwg), blk(NET_THREADS);
  hipStream_t st = n->s->st;
#define PMF_NET(B)                                                                                                  \
  hipLaunchKernelGGL((k_net<B, true>), grd, blk, 0, st, n->w, X, Tg, n->n, pick ? 1 : 0, key, rows, nullptr, n->part, \
                     n->dpart)
  if (bf16) PMF_NET(true);
  else PMF_NET(false);
#undef PMF_NET
  hipLaunchKernelGGL(k_net_update, dim3((NPARAM + 64) / 64), dim3(1024), 0, st, n->part, n->dpart, nwg, n->g, loss,
                     1.0 / double(rows * 7), a.on, n->w, n->m, n->v, a.lr, a.b1, a.b2, a.eps, a.c1, a.c2);
}

}  // namespace

extern "C" {

int pmf_surrogate_create(pmf_state* s, uint64_t seed, pmf_surrogate** out) {
  return guard([&] {
    check_state(s);
    if (!out) throw Error("null argument");
    if (s->p.precision != PMF_F32) throw Error("the flux surrogate runs on float32 states");
    auto* n = new pmf_surrogate();
    try {
      n->s = s;
      hip_check(hipMalloc(&n->w, sizeof(float) * NPARAM), "hipMalloc");
      hip_check(hipMalloc(&n->g, sizeof(float) * NPARAM), "hipMalloc");
      hip_check(hipMalloc(&n->m, sizeof(float) * NPARAM), "hipMalloc");
      hip_check(hipMalloc(&n->v, sizeof(float) * NPARAM), "hipMalloc");
      hip_check(hipMalloc(&n->part, sizeof(float) * NPARAM * NET_MAX_WG), "hipMalloc");
      hip_check(hipMalloc(&n->dpart, sizeof(double) * NET_DSLOTS * NET_MAX_WG), "hipMalloc");
      grow(n->dloss, n->loss_steps, 1, 1);
      hip_check(hipMalloc(&n->dcount, sizeof(unsigned long long)), "hipMalloc");
      hip_check(hipMalloc(&n->img, SIMG_BYTES), "hipMalloc");
      hip_check(hipMalloc(&n->nsmooth, sizeof(unsigned long long)), "hipMalloc");
      // He-style uniform init of the weights, zero biases
      std::vector<float> h(NPARAM, 0.f);
      std::mt19937_64 rng(seed);
      for (int l = 0; l < 4; ++l) {
        float lim = std::sqrt(6.0f / float(LAYER_IN[l] + LAYER_OUT[l])) * (l < 3 ? 1.0f : 0.1f);
        std::uniform_real_distribution<float> u(-lim, lim);
        for (int e = 0; e < LAYER_IN[l] * LAYER_OUT[l]; ++e) h[w_off(l) + e] = u(rng);
      }
      hip_check(hipMemcpy(n->w, h.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice), "copy");
      hip_check(hipMemset(n->m, 0, sizeof(float) * NPARAM), "memset");
      hip_check(hipMemset(n->v, 0, sizeof(float) * NPARAM), "memset");
      // null-stream work: the state's non-blocking stream does not wait for it
      hip_check(hipDeviceSynchronize(), "hipDeviceSynchronize");
    } catch (...) {
      pmf_surrogate_destroy(n);
      throw;
    }
    *out = n;
  });
}

int pmf_surrogate_destroy(pmf_surrogate* n) {
  return guard([&] {
    if (!n) return;
    if (n->s) (void)hipStreamSynchronize(n->s->st);
    (void)hipFree(n->part);
    (void)hipFree(n->dpart);
    (void)hipFree(n->Yb);
    (void)hipFree(n->Fb);
    (void)hipFree(n->w);
    (void)hipFree(n->g);
    (void)hipFree(n->m);
    (void)hipFree(n->v);
    (void)hipFree(n->X);
    (void)hipFree(n->Y);
    (void)hipFree(n->S);
    (void)hipFree(n->dloss);
    (void)hipFree(n->dcount);
    (void)hipFree(n->img);
    (void)hipFree(n->nsmooth);
    delete n;
  });
}

int pmf_surrogate_nparams(void) { return NPARAM; }

int pmf_surrogate_get_weights(pmf_surrogate* n, float* host, int64_t count) {
  return guard([&] {
    if (!n || !host || count != NPARAM) throw Error("weights array must hold pmf_surrogate_nparams() floats");
    hip_check(hipMemcpyAsync(host, n->w, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, n->s->st), "copy");
    sync(n->s);
  });
}

int pmf_surrogate_set_weights(pmf_surrogate* n, const float* host, int64_t count) {
  return guard([&] {
    if (!n || !host || count != NPARAM) throw Error("weights array must hold pmf_surrogate_nparams() floats");
    hip_check(hipMemcpyAsync(n->w, host, sizeof(float) * NPARAM, hipMemcpyHostToDevice, n->s->st), "copy");
    sync(n->s);
  });
}

int pmf_surrogate_reserve(pmf_surrogate* n, int64_t cap) {
  return guard([&] {
    if (!n || cap < 1) throw Error("bad arguments");
    (void)hipFree(n->X);
    (void)hipFree(n->Y);
    (void)hipFree(n->S);
    n->X = n->Y = n->S = nullptr;
    hip_check(hipMalloc(&n->X, sizeof(float) * 16 * cap), "hipMalloc(dataset)");
    hip_check(hipMalloc(&n->Y, sizeof(float) * 9 * cap), "hipMalloc(dataset)");
    hip_check(hipMalloc(&n->S, sizeof(float) * 18 * cap), "hipMalloc(dataset)");
    n->cap = cap;
    n->n = 0;
  });
}

int pmf_surrogate_dump(pmf_surrogate* n, pmf_state* s, double dt, double ch, double thr, double keep, uint64_t seed,
                       int64_t* total) {
  return guard([&] {
    if (!n || !n->X) throw Error("reserve the dataset first (pmf_surrogate_reserve)");
    check_fields(s);
    if (s->p.precision != PMF_F32) throw Error("the flux surrogate runs on float32 states");
    if (!(ch > 0)) throw Error("step! needs the GLM cleaning speed `ch` (GLM states)");
    unsigned long long c0 = (unsigned long long)n->n;
    hip_check(hipMemcpyAsync(n->dcount, &c0, sizeof(c0), hipMemcpyHostToDevice, s->st), "copy");
    StepParams<float> P = make_params<float>(s, dt, ch, 1.0);
    hipLaunchKernelGGL(k_dump_faces, dim3(blocks(s->nc)), dim3(256), 0, s->st, cfields_at<float>(s->U, s->nc), s->G,
                       P, float(thr), float(keep), (unsigned long long)seed, n->X, n->Y, n->S, n->dcount, n->cap);
    hip_check(hipGetLastError(), "dump launch");
    unsigned long long c1 = 0;
    hip_check(hipMemcpyAsync(&c1, n->dcount, sizeof(c1), hipMemcpyDeviceToHost, s->st), "copy");
    sync(s);
    n->n = std::min<int64_t>((int64_t)c1, n->cap);
    if (total) *total = n->n;
  });
}

int pmf_surrogate_dataset(pmf_surrogate* n, int64_t first, int64_t count, float* X, float* Y, float* S) {
  return guard([&] {
    if (!n || first < 0 || count < 0 || first + count > n->n) throw Error("dataset range out of bounds");
    hipStream_t st = n->s->st;
    if (X) hip_check(hipMemcpyAsync(X, n->X + first * 16, sizeof(float) * 16 * count, hipMemcpyDeviceToHost, st), "copy");
    if (Y) hip_check(hipMemcpyAsync(Y, n->Y + first * 9, sizeof(float) * 9 * count, hipMemcpyDeviceToHost, st), "copy");
    if (S) hip_check(hipMemcpyAsync(S, n->S + first * 18, sizeof(float) * 18 * count, hipMemcpyDeviceToHost, st), "copy");
    sync(n->s);
  });
}

int pmf_surrogate_upload(pmf_surrogate* n, const float* X, const float* Y, const float* S, int64_t count) {
  return guard([&] {
    if (!n || !X || !Y || count < 1) throw Error("bad arguments");
    if (count > n->cap) throw Error("dataset capacity exceeded");
    hipStream_t st = n->s->st;
    hip_check(hipMemcpyAsync(n->X, X, sizeof(float) * 16 * count, hipMemcpyHostToDevice, st), "copy");
    hip_check(hipMemcpyAsync(n->Y, Y, sizeof(float) * 9 * count, hipMemcpyHostToDevice, st), "copy");
    if (S) hip_check(hipMemcpyAsync(n->S, S, sizeof(float) * 18 * count, hipMemcpyHostToDevice, st), "copy");
    sync(n->s);
    n->n = count;
  });
}

int pmf_surrogate_grad(pmf_surrogate* n, int64_t first, int64_t count, int32_t bf16, float* grad, double* loss) {
  return guard([&] {
    if (!n || first < 0 || count < 1 || first + count > n->n) throw Error("dataset range out of bounds");
    learn(n, n->X + first * 16, n->Y + first * 9, count, false, 0ull, bf16 != 0, n->dloss, Adam{});
    hip_check(hipGetLastError(), "surrogate launch");
    if (grad) hip_check(hipMemcpyAsync(grad, n->g, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, n->s->st), "copy");
    if (loss) hip_check(hipMemcpyAsync(loss, n->dloss, sizeof(double), hipMemcpyDeviceToHost, n->s->st), "copy");
    sync(n->s);
  });
}

int pmf_surrogate_predict(pmf_surrogate* n, int64_t first, int64_t count, int32_t bf16, float* Yhost) {
  return guard([&] {
    if (!n || first < 0 || count < 1 || first + count > n->n) throw Error("dataset range out of bounds");
    ensure_outputs(n, count);
    forward(n, n->X + first * 16, count, bf16 != 0);
    hip_check(hipGetLastError(), "surrogate launch");
    hip_check(hipMemcpyAsync(Yhost, n->Yb, sizeof(float) * 9 * count, hipMemcpyDeviceToHost, n->s->st), "copy");
    sync(n->s);
  });
}

int pmf_surrogate_train(pmf_surrogate* n, int32_t batch, int32_t steps, double lr, uint64_t seed, int32_t bf16,
                        double* losses) {
  return guard([&] {
    if (!n || n->n < 1) throw Error("the dataset is empty");
    if (batch < 1 || steps < 0) throw Error("bad arguments");
    // Two launches a step and no wait between steps: the losses stay on the device until the
    // end. Batch 8192: 6.9 ms a step layer by layer, now 27 us of 128 or more in a call, 31 of eight
    // (4096: 20 and 24, 1024: 15 and 19).
    grow(n->dloss, n->loss_steps, std::max<int64_t>(steps, 1), 1);
    Adam a;
    a.on = 1;
    a.lr = float(lr);
    a.b1 = 0.9f;
    a.b2 = 0.999f;
    a.eps = 1e-8f;
    for (int it = 0; it < steps; ++it) {
      unsigned long long key = seed * 0xD1B54A32D192ED03ull + (unsigned long long)(n->adam_t + 1) * 0x9E3779B97F4A7C15ull;
      ++n->adam_t;
      a.c1 = 1.f / (1.f - std::pow(a.b1, (float)n->adam_t));
      a.c2 = 1.f / (1.f - std::pow(a.b2, (float)n->adam_t));
      learn(n, n->X, n->Y, batch, true, key, bf16 != 0, n->dloss + it, a);
    }
    hip_check(hipGetLastError(), "surrogate launch");
    if (losses && steps > 0)
      hip_check(hipMemcpyAsync(losses, n->dloss, sizeof(double) * steps, hipMemcpyDeviceToHost, n->s->st), "copy");
    sync(n->s);
  });
}

int pmf_surrogate_face_flux(pmf_surrogate* n, int64_t first, int64_t count, int32_t mode, double thr, float* Fhost) {
  return guard([&] {
    if (!n || first < 0 || count < 1 || first + count > n->n) throw Error("dataset range out of bounds");
    if (mode < 0 || mode > 2) throw Error("mode must be 0 (HLLD), 1 (surrogate) or 2 (central)");
    ensure_outputs(n, count);
    hipStream_t st = n->s->st;
    if (mode == 1) forward(n, n->X + first * 16, count, true);
    float* F = n->Fb;
    StepParams<float> P = make_params<float>(n->s, 0.0, 1.0, 1.0);
    hipLaunchKernelGGL(k_face_flux, dim3(blocks(count)), dim3(256), 0, st, n->S + first * 18,
                       mode == 1 ? n->Yb : (const float*)nullptr, count, P, float(thr), mode, F);
    hip_check(hipGetLastError(), "face flux launch");
    hip_check(hipMemcpyAsync(Fhost, F, sizeof(float) * 9 * count, hipMemcpyDeviceToHost, st), "copy");
    sync(n->s);
  });
}

int pmf_step_surrogate(pmf_state* s, pmf_surrogate* n, double dt, double ch, double glm_cr, double thr,
                       int64_t* nsmooth) {
  return guard([&] {
    check_fields(s);
    if (!n) throw Error("null surrogate");
    if (s->p.precision != PMF_F32) throw Error("the flux surrogate runs on float32 states");
    if (s->p.solver != PMF_SOLVER_GLM) throw Error("the flux surrogate replaces the GLM-HLLD flux (GLM states only)");
    if (s->p.riemann != PMF_RIEMANN_HLLD) throw Error("the flux surrogate stands in for HLLD (riemann=:hlld)");
    if (!(ch > 0.0)) throw Error("step! needs the GLM cleaning speed `ch` (GLM states)");
    if (!surrogate_grid(s->G))
      throw Error("the surrogate step needs an all-periodic grid whose nx is a multiple of 16");
    const double decay = decay_of(s, dt, ch, glm_cr);
    hipLaunchKernelGGL(k_surr_image, dim3((SIMG_NW + 255) / 256), dim3(256), 0, s->st, n->w, n->img);
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, s->st, n->nsmooth);
    mark(s);
    bool ok = launch_step_fused_surr(cfields_at<float>(s->U, s->nc), fields_at<float>(s->S, s->nc), s->G,
                                     make_params<float>(s, dt, ch, decay), s->red, s->dval, n->img, float(thr),
                                     n->nsmooth, s->st, s->hval);
    mark(s);
    if (!ok) throw Error("surrogate step unavailable for this configuration");
    hip_check(hipGetLastError(), "surrogate step launch");
    std::swap(s->U, s->S);
    s->smax_valid = true;
    if (nsmooth) {
      unsigned long long c = 0;
      hip_check(hipMemcpyAsync(&c, n->nsmooth, sizeof(c), hipMemcpyDeviceToHost, s->st), "copy");
      sync(s);
      *nsmooth = (int64_t)c;
    }
  });
}

}  // extern "C"
