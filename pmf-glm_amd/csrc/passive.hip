// Passive species transport after the MHD step (lib/MHDKernels/src/passive_transport.jl):
// conserved species densities to bounded mass fractions, and the semi-Lagrangian
// backtrace of fractions (or of an unconstrained scalar) with the post-step cell velocity,
// sampled trilinearly on the periodic cubic grid and restored to mass densities with the
// new gas density.
#include <limits>

#include "launch.hpp"

namespace pmf {

template <class T> __device__ __forceinline__ T clampT(T x, T lo, T hi) { return x < lo ? lo : (x > hi ? hi : x); }

// passive_transport.jl:5-25
template <class T>
__global__ __launch_bounds__(256) void k_species_to_fractions(T* __restrict__ s1, T* __restrict__ s2,
                                                              const T* __restrict__ rho, int64_t nc, T maxt) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= nc) return;
  const T d = dmax(rho[c], std::numeric_limits<T>::epsilon());
  if (s2) {
    const T q2 = clampT(s2[c] / d, T(0), maxt);
    const T q1 = clampT(s1[c] / d, T(0), maxt - q2);
    s1[c] = q1;
    s2[c] = q2;
  } else {
    s1[c] = clampT(s1[c] / d, T(0), maxt);
  }
}

// passive_transport.jl:40-54: muladd(f, r - l, l) along x, then y, then z, as one fused
// multiply-add in the field's own precision
__device__ __forceinline__ float lerp(float l, float r, float f) { return __builtin_fmaf(f, r - l, l); }
__device__ __forceinline__ double lerp(double l, double r, double f) { return __builtin_fma(f, r - l, l); }

// The cells l and l + 1 of one axis, wrapped (passive_transport.jl:27-32, 0-based). A cell
// moves a fraction of a cell per step, so the wrap is a compare; a far one takes the
// non-negative modulo.
__device__ __forceinline__ void wrap2(int l, int n, int& a, int& b) {
  if (__builtin_expect((unsigned)(l + n) >= 2u * (unsigned)n, 0)) {
    l %= n;
  }
  a = l < 0 ? l + n : l;
  b = a + 1 == n ? 0 : a + 1;
}

// The eight corners of a cell's box: rows r[0..3] (y, z low and high: 00, 10, 01, 11), columns
// i0, i1; and their trilinear interpolation.
template <bool NARROW, class T, class I>
__device__ __forceinline__ void corners(const T* __restrict__ a, const I* r, int i0, int i1, T* p) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    p[2 * q] = *cell_at<NARROW>(a, r[q] + i0);
    p[2 * q + 1] = *cell_at<NARROW>(a, r[q] + i1);
  }
}
template <class T> __device__ __forceinline__ T trilinear(const T* p, T fx, T fy, T fz) {
  const T x00 = lerp(p[0], p[1], fx), x10 = lerp(p[2], p[3], fx);
  const T x01 = lerp(p[4], p[5], fx), x11 = lerp(p[6], p[7], fx);
  return lerp(lerp(x00, x10, fy), lerp(x01, x11, fy), fz);
}

// passive_transport.jl:78-190. MODE 0: one fraction, 1: two fractions (the second
// bounds the first), 2: unconstrained scalar. NARROW: 32-bit byte offsets (fields below 4
// GiB). The neighbouring lanes' gas comes from different rows and planes, and gathers that
// spread over them held the kernel at 90 us (192^3, two fractions, 2.5 TB/s), whatever the
// address arithmetic, the block order and the cells in flight. So a block of 64 x 16 cells
// stages the fields' planes k-1 .. k+1 with their halo in LDS, in whole rows, and the corners
// are gathered there: 59 us. A cell whose gas came from farther away reads the fields.
constexpr int kBtX = 64, kBtRows = 4, kBtY = 4 * kBtRows;  // a thread's cells: kBtRows rows
constexpr int kBtW = kBtX + 2, kBtH = kBtY + 2;
template <class T, int MODE, bool NARROW>
__global__ __launch_bounds__(256) void k_backtrace(T* __restrict__ o1, T* __restrict__ o2, const T* __restrict__ a1,
                                                   const T* __restrict__ a2, const T* __restrict__ rho,
                                                   const T* __restrict__ mx, const T* __restrict__ my,
                                                   const T* __restrict__ mz, int n, T dtdx, T maxt) {
  typedef typename std::conditional<NARROW, uint32_t, int64_t>::type I;
  constexpr int NF = MODE == 1 ? 2 : 1;
  __shared__ T S[NF][3 * kBtH * kBtW];
  const int nx = (n + kBtX - 1) / kBtX, ny = (n + kBtY - 1) / kBtY, w = xcd_tile();
  const int x0 = w % nx * kBtX, y0 = w / nx % ny * kBtY, k = w / (nx * ny);
  const int i = x0 + (threadIdx.x & 63), j = y0 + (threadIdx.x >> 6) * kBtRows;
  // the staged cells: -1 .. n of each axis (the ends wrapped), as far as the block reaches
  auto wrap1 = [n](int v) { return v < 0 ? v + n : (v >= n ? v - n : v); };
  constexpr int NE = 3 * kBtH * kBtW, NL = (NE + 255) / 256;
  T st[NL][NF];  // all loads in flight together
#pragma unroll
  for (int q = 0; q < NL; ++q) {
    const int e = threadIdx.x + 256 * q;
    const int x = x0 - 1 + e % kBtW, y = y0 - 1 + e / kBtW % kBtH, z = k - 1 + e / (kBtW * kBtH);
    if (e < NE && x <= n && y <= n) {
      const I c = ((I)wrap1(z) * n + wrap1(y)) * n + wrap1(x);
      st[q][0] = *cell_at<NARROW>(a1, c);
      if constexpr (MODE == 1) st[q][NF - 1] = *cell_at<NARROW>(a2, c);
    }
  }
  const int lim_x = min(kBtX, n - x0), lim_y = min(kBtY, n - y0);  // last staged low corner
  T d[kBtRows], m[kBtRows][3];
#pragma unroll
  for (int q = 0; q < kBtRows; ++q) {
    const I c = ((I)k * n + min(j + q, n - 1)) * n + min(i, n - 1);
    d[q] = *cell_at<NARROW>(rho, c);
    m[q][0] = *cell_at<NARROW>(mx, c);
    m[q][1] = *cell_at<NARROW>(my, c);
    m[q][2] = *cell_at<NARROW>(mz, c);
  }
#pragma unroll
  for (int q = 0; q < NL; ++q) {
    const int e = threadIdx.x + 256 * q;
    if (e < NE) {
      S[0][e] = st[q][0];
      if constexpr (MODE == 1) S[NF - 1][e] = st[q][NF - 1];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kBtRows; ++q) {
    if (i >= n || j + q >= n) break;
    const T dq = dmax(d[q], std::numeric_limits<T>::epsilon());
    const T x = T(i) - dtdx * m[q][0] / dq;
    const T y = T(j + q) - dtdx * m[q][1] / dq;
    const T z = T(k) - dtdx * m[q][2] / dq;
    const int il = (int)__builtin_floor(x), jl = (int)__builtin_floor(y), kl = (int)__builtin_floor(z);
    const T fx = x - T(il), fy = y - T(jl), fz = z - T(kl);
    const int lx = il - x0 + 1, ly = jl - y0 + 1, lz = kl - k + 1;  // low corner in the staged box
    T p1[8], p2[8];
    if ((unsigned)lx <= (unsigned)lim_x && (unsigned)ly <= (unsigned)lim_y && (unsigned)lz <= 1u) {
      const int e = (lz * kBtH + ly) * kBtW + lx;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int at = e + (r & 1) + ((r >> 1) & 1) * kBtW + (r >> 2) * kBtH * kBtW;
        p1[r] = S[0][at];
        if constexpr (MODE == 1) p2[r] = S[NF - 1][at];
      }
    } else {
      int i0, i1, j0, j1, k0, k1;
      wrap2(il, n, i0, i1);
      wrap2(jl, n, j0, j1);
      wrap2(kl, n, k0, k1);
      const I r[4] = {((I)k0 * n + j0) * n, ((I)k0 * n + j1) * n, ((I)k1 * n + j0) * n, ((I)k1 * n + j1) * n};
      corners<NARROW>(a1, r, i0, i1, p1);
      if constexpr (MODE == 1) corners<NARROW>(a2, r, i0, i1, p2);
    }
    const I c = ((I)k * n + j + q) * n + i;
    const T s1 = trilinear(p1, fx, fy, fz);
    if constexpr (MODE == 2) {
      *cell_at<NARROW>(o1, c) = s1;
    } else if constexpr (MODE == 1) {
      const T q2 = clampT(trilinear(p2, fx, fy, fz), T(0), maxt);
      const T q1 = clampT(s1, T(0), maxt - q2);
      *cell_at<NARROW>(o1, c) = dq * q1;
      *cell_at<NARROW>(o2, c) = dq * q2;
    } else {
      *cell_at<NARROW>(o1, c) = dq * clampT(s1, T(0), maxt);
    }
  }
}

template <class T>
void launch_species_to_fractions(T* s1, T* s2, const T* rho, int64_t nc, T maxt, hipStream_t st) {
  hipLaunchKernelGGL(k_species_to_fractions<T>, dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, st, s1, s2, rho, nc,
                     maxt);
}

template <class T>
void launch_backtrace(T* o1, T* o2, const T* a1, const T* a2, Fields<const T> U, int n, T dtdx, T maxt, int mode,
                      hipStream_t st) {
  const dim3 grd((unsigned)((n + kBtX - 1) / kBtX * ((n + kBtY - 1) / kBtY) * n)), blk(256);
  const bool narrow = (uint64_t)n * n * n * sizeof(T) < (1ull << 32);
#define PMF_BT(M, N)                                                                                              \
  hipLaunchKernelGGL((k_backtrace<T, M, N>), grd, blk, 0, st, o1, o2, a1, a2, U.v[0], U.v[1], U.v[2], U.v[3], n, \
                     dtdx, maxt)
  if (narrow) {
    if (mode == 1) PMF_BT(1, true);
    else if (mode == 2) PMF_BT(2, true);
    else PMF_BT(0, true);
  } else {
    if (mode == 1) PMF_BT(1, false);
    else if (mode == 2) PMF_BT(2, false);
    else PMF_BT(0, false);
  }
#undef PMF_BT
}

template void launch_species_to_fractions<float>(float*, float*, const float*, int64_t, float, hipStream_t);
template void launch_species_to_fractions<double>(double*, double*, const double*, int64_t, double, hipStream_t);
template void launch_backtrace<float>(float*, float*, const float*, const float*, Fields<const float>, int, float,
                                      float, int, hipStream_t);
template void launch_backtrace<double>(double*, double*, const double*, const double*, Fields<const double>, int,
                                       double, double, int, hipStream_t);

}  // namespace pmf
