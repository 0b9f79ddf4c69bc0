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

// Where the gas of cell (i, j, k) came from: the low corner's cell and the fractions beyond it.
template <class T> struct Foot {
  int i, j, k;
  T fx, fy, fz;
};
template <class T> __device__ __forceinline__ Foot<T> foot(int i, int j, int k, T d, const T* m, T dtdx) {
  const T x = T(i) - dtdx * m[0] / d, y = T(j) - dtdx * m[1] / d, z = T(k) - dtdx * m[2] / d;
  Foot<T> f;
  f.i = (int)__builtin_floor(x);
  f.j = (int)__builtin_floor(y);
  f.k = (int)__builtin_floor(z);
  f.fx = x - T(f.i);
  f.fy = y - T(f.j);
  f.fz = z - T(f.k);
  return f;
}

// The corners of the foot's box, read from the fields.
template <int MODE, bool NARROW, class I, class T>
__device__ __forceinline__ void gather(const T* __restrict__ a1, const T* __restrict__ a2, const Foot<T>& f, int n,
                                       T* p1, T* p2) {
  int i0, i1, j0, j1, k0, k1;
  wrap2(f.i, n, i0, i1);
  wrap2(f.j, n, j0, j1);
  wrap2(f.k, n, k0, k1);
  const I r[4] = {((I)k0 * n + j0) * n, ((I)k0 * n + j1) * n, ((I)k1 * n + j0) * n, ((I)k1 * n + j1) * n};
  corners<NARROW>(a1, r, i0, i1, p1);
  if constexpr (MODE == 1) corners<NARROW>(a2, r, i0, i1, p2);
}

// passive_transport.jl:78-190 for one cell. MODE 0: one fraction, 1: two fractions (the second
// bounds the first), 2: unconstrained scalar.
template <int MODE, bool NARROW, class I, class T>
__device__ __forceinline__ void put_cell(T* __restrict__ o1, T* __restrict__ o2, I c, T d, const Foot<T>& f,
                                         const T* p1, const T* p2, T maxt) {
  const T s1 = trilinear(p1, f.fx, f.fy, f.fz);
  if constexpr (MODE == 2) {
    *cell_at<NARROW>(o1, c) = s1;
  } else if constexpr (MODE == 1) {
    const T q2 = clampT(trilinear(p2, f.fx, f.fy, f.fz), T(0), maxt);
    const T q1 = clampT(s1, T(0), maxt - q2);
    *cell_at<NARROW>(o1, c) = d * q1;
    *cell_at<NARROW>(o2, c) = d * q2;
  } else {
    *cell_at<NARROW>(o1, c) = d * clampT(s1, T(0), maxt);
  }
}

// The backtrace, a cell a thread. NARROW: 32-bit byte offsets (fields below 4 GiB).
template <class T, int MODE, bool NARROW>
__global__ __launch_bounds__(256) void k_backtrace_cells(T* __restrict__ o1, T* __restrict__ o2,
                                                         const T* __restrict__ a1, const T* __restrict__ a2,
                                                         const T* __restrict__ rho, const T* __restrict__ mx,
                                                         const T* __restrict__ my, const T* __restrict__ mz, int n,
                                                         T dtdx, T maxt) {
  typedef typename std::conditional<NARROW, uint32_t, int64_t>::type I;
  const I c = (I)blockIdx.x * 256 + threadIdx.x, nn = (I)n * n;
  if (c >= nn * n) return;
  const int k = (int)(c / nn), j = (int)(c % nn / n), i = (int)(c % n);
  const T d = dmax(*cell_at<NARROW>(rho, c), std::numeric_limits<T>::epsilon());
  const T m[3] = {*cell_at<NARROW>(mx, c), *cell_at<NARROW>(my, c), *cell_at<NARROW>(mz, c)};
  const Foot<T> f = foot(i, j, k, d, m, dtdx);
  T p1[8], p2[8];
  gather<MODE, NARROW, I>(a1, a2, f, n, p1, p2);
  put_cell<MODE, NARROW>(o1, o2, c, d, f, p1, p2, maxt);
}

// The same from LDS. The neighbouring lanes' gas comes from different rows and planes, and gathers that
// spread over them held the kernel above at 90 us (192^3, two fractions, 2.5 TB/s), whatever the
// address arithmetic, the block order and the cells in flight. So a block of 64 x 16 cells
// stages the fields' planes k-1 .. k+1 with their halo in LDS, in whole rows, and the corners
// are gathered there: 59 us. A cell whose gas came from farther away reads the fields.
constexpr int kBtX = 64, kBtRows = 4, kBtY = 4 * kBtRows;  // a thread's cells: kBtRows rows
constexpr int kBtW = kBtX + 2, kBtH = kBtY + 2;
template <class T, int MODE, bool NARROW>
__global__ __launch_bounds__(256) void k_backtrace_tiles(T* __restrict__ o1, T* __restrict__ o2, const T* __restrict__ a1,
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
    const Foot<T> f = foot(i, j + q, k, dq, m[q], dtdx);
    const int lx = f.i - x0 + 1, ly = f.j - y0 + 1, lz = f.k - k + 1;  // low corner in the staged box
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
      gather<MODE, NARROW, I>(a1, a2, f, n, p1, p2);
    }
    const I c = ((I)k * n + j + q) * n + i;
    put_cell<MODE, NARROW>(o1, o2, c, dq, f, p1, p2, maxt);
  }
}

template <class T>
void launch_species_to_fractions(T* s1, T* s2, const T* rho, int64_t nc, T maxt, hipStream_t st) {
  hipLaunchKernelGGL(k_species_to_fractions<T>, dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, st, s1, s2, rho, nc,
                     maxt);
}

// Whether the fields' planes are staged. On small grids the tiles are few and part empty, and what
// counts is one cell's chain of loads, to which staging adds a barrier. us, cells and tiles, float32
// two fractions (one): 32^3 19.6, 21.8 (16.8, 18.2); 65^3 23.3, 26.0 (18.0, 21.8); 72^3 25.9, 26.8;
// 76^3 27.2, 25.6; (84^3 22.6, 22.7; 96^3 25.7, 24.7); 129^3 51, 43 (36, 35); 192^3 118, 72 (73, 54).
// float64 within 4% of the same line: 80^3 34.5, 33.3 (24.0, 25.9); 192^3 196, 161 (104, 92).
static bool backtrace_tiles(int n, int mode) { return n >= (mode == 1 ? 75 : 85); }

template <class T>
void launch_backtrace(T* o1, T* o2, const T* a1, const T* a2, Fields<const T> U, int n, T dtdx, T maxt, int mode,
                      hipStream_t st) {
  const bool narrow = (uint64_t)n * n * n * sizeof(T) < (1ull << 32), tiles = backtrace_tiles(n, mode);
  const unsigned nb = tiles ? (unsigned)((n + kBtX - 1) / kBtX * ((n + kBtY - 1) / kBtY) * n)
                            : (unsigned)(((int64_t)n * n * n + 255) / 256);
#define PMF_BT_N(M, N)                                                                                             \
  if (tiles)                                                                                                       \
    hipLaunchKernelGGL((k_backtrace_tiles<T, M, N>), dim3(nb), dim3(256), 0, st, o1, o2, a1, a2, U.v[0], U.v[1],  \
                       U.v[2], U.v[3], n, dtdx, maxt);                                                             \
  else                                                                                                             \
    hipLaunchKernelGGL((k_backtrace_cells<T, M, N>), dim3(nb), dim3(256), 0, st, o1, o2, a1, a2, U.v[0], U.v[1],  \
                       U.v[2], U.v[3], n, dtdx, maxt)
#define PMF_BT(M)            \
  if (narrow) {              \
    PMF_BT_N(M, true);       \
  } else {                   \
    PMF_BT_N(M, false);      \
  }
  if (mode == 1) {
    PMF_BT(1)
  } else if (mode == 2) {
    PMF_BT(2)
  } else {
    PMF_BT(0)
  }
#undef PMF_BT_N
#undef PMF_BT
}

template void launch_species_to_fractions<float>(float*, float*, const float*, int64_t, float, hipStream_t);
template void launch_species_to_fractions<double>(double*, double*, const double*, int64_t, double, hipStream_t);
template void launch_backtrace<float>(float*, float*, const float*, const float*, Fields<const float>, int, float,
                                      float, int, hipStream_t);
template void launch_backtrace<double>(double*, double*, const double*, const double*, Fields<const double>, int,
                                       double, double, int, hipStream_t);

}  // namespace pmf
