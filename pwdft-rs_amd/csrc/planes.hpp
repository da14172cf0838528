// One z-plane of the sphere-pruned FFT in LDS, shared by the H·ψ plane pass (hpsi.hip) and the band
// density (density.hip).
//
// A workgroup works on SLOTS planes at once (the same i3 of SLOTS bands), so that the y-lines (only
// the nx1 rows that carry sticks, about half of them) and the x-lines of a plane fill whole waves: a
// 60-point plane alone has 29 y-lines for 64 lanes, two planes have 58. Or on one (ONE): H·ψ of wider spheres,
// and of few planes (hpsi_sphere.hip).
//
// A plane's LDS image holds only the rows that carry sticks when these are the two runs i1 < ra and
// i1 >= nx - rb (a sphere's columns), followed by a zero row that stands for every other row; grids
// whose columns are not two such runs hold all rows (ra = nx, rb = 0). pl_src (setup_basis) gives the
// stick of every element of that image, -1 for zeros: one pass of coalesced loads fills it, without
// clearing it first and without a barrier in between.
#pragma once

#include "common.hpp"
#include "fft_pfa.hpp"
#include "fft_reg.hpp"

namespace pwk {

template <typename T>
struct V2t;
template <>
struct V2t<double> {
  using t = double2;
};
template <>
struct V2t<float> {
  using t = float2;
};

// Waves and planes per workgroup of a square N × N plane pass. Cost of a workgroup's passes in
// wave-wide line transforms, per plane: ceil(SLOTS·N / 64) waves run x-lines, ceil(SLOTS·(N/2) / 64)
// run y-lines; the cheapest of 1-4 waves is taken, fewer waves on a tie, whose planes fit 72 KB of
// LDS (two workgroups per CU) with the rows of a sphere, and the 160 KB of a CU with all rows. ACC:
// an FP64 sum per point and plane in LDS as well.
template <typename T, int N, bool ACC = false, bool ONE = false>
struct PlaneShape {
  static constexpr int LD = N + 1;  // one element of padding against bank conflicts on row access
  static constexpr int slots(int w) { return 64 * w / N; }
  static constexpr size_t lds(int w, int rows) {
    return (size_t)slots(w) * (rows * LD * sizeof(typename V2t<T>::t) + (ACC ? N * N * sizeof(double) : 0));
  }
  static constexpr int cost(int w) {  // in 1/720 of a wave-wide transform per plane (720: all slot counts divide)
    return ((slots(w) * N + 63) / 64 + (slots(w) * (N / 2) + 63) / 64) * 720 / slots(w);
  }
  static constexpr int best() {
    int w = (N + 63) / 64;
    for (int v = w + 1; v <= 4; ++v)
      if (lds(v, N / 2 + 3) <= 72 * 1024 && lds(v, N + 2) <= 160 * 1024 && cost(v) < cost(w)) w = v;
    return w;
  }
  static constexpr int W = ONE ? (N + 63) / 64 : best(), NT = 64 * W, SLOTS = ONE ? 1 : slots(W);
};

// loads of a thread in flight while NT threads move n elements: no more than it has, up to 16 (FP64 8)
template <typename T, int NT>
constexpr int in_flight(int n) {
  const int most = 16 / (int)(sizeof(T) / 4), need = (n + NT - 1) / NT;
  return need < most ? need : most;
}

// the plane row j in the held image (`absent` for a row without sticks)
struct PlaneRows {
  int ra, rb;
};
template <int N>
__device__ __forceinline__ int plane_row(const PlaneRows& pr, int j, int absent) {
  return j < pr.ra ? j : (j >= N - pr.rb ? j - (N - pr.rb) + pr.ra : absent);
}

// fills `nsl` images (stride `image` elements) from the stick rows tp0 + p·band_stride; n elements each
template <typename T, int N, int NT, int U>
__device__ __forceinline__ void plane_fill(typename V2t<T>::t* P, int image,
                                           const typename V2t<T>::t* tp0, size_t band_stride, int nsl,
                                           const int* __restrict__ src, int n) {
  using V2 = typename V2t<T>::t;
  for (int e0 = threadIdx.x; e0 < n; e0 += U * NT) {
    int s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) s[u] = src[min(e0 + u * NT, n - 1)];
    for (int p = 0; p < nsl; ++p) {
      const V2* tp = tp0 + (size_t)p * band_stride;
      V2 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = tp[max(s[u], 0)];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * NT;
        if (e < n) {
          V2 x;
          x.x = s[u] >= 0 ? v[u].x : (T)0;
          x.y = s[u] >= 0 ? v[u].y : (T)0;
          P[p * image + e] = x;
        }
      }
    }
  }
}

// the y-lines of the rows that carry sticks: row r of an image, or (x1list non-null: all rows held)
// row x1list[r]
template <typename T, int N, int NT, int SIGN>
__device__ __forceinline__ void plane_ylines(typename V2t<T>::t* P, int image, int nsl, int nx1,
                                             const int* __restrict__ x1list) {
  constexpr int LD = N + 1;
  for (int t = threadIdx.x; t < nsl * nx1; t += NT) {
    const int p = t / nx1, r = t - p * nx1;
    typename V2t<T>::t* row = P + p * image + (x1list ? x1list[r] : r) * LD;
    T re[N], im[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      re[j] = row[j].x;
      im[j] = row[j].y;
    }
    fft_dif<T, N, SIGN>(re, im);
#pragma unroll
    for (int f = 0; f < N; ++f) {
      row[f].x = re[FftOrder<N>::pos(f)];
      row[f].y = im[FftOrder<N>::pos(f)];
    }
  }
}

// ---- spheres within a quarter of the axes ------------------------------------------------
// On a grid of at least 4·max|n| + 1 points per axis (ecutrho = 4·ecutwfc, the default) every index that
// carries plane waves is i < PA or i >= N - PB. Knowing that at compile time, the line transforms load
// only those inputs and store only those outputs (the arithmetic on the others drops out), the held rows
// sit at constant offsets and no zero or discard row is needed.
template <int N>
struct Quarter {
  static constexpr int PB = (N - 1) / 4, PA = PB + 1, R = PA + PB;  // held indices
  static constexpr int LD = N | 1;                                   // odd row stride: no bank conflicts
  static constexpr bool has(int i) { return i < PA || i >= N - PB; }
  static constexpr int at(int i) { return i < PA ? i : i - (N - R); }  // held index -> row of the image
  __host__ __device__ static constexpr int index(int r) { return r < PA ? r : r + (N - R); }
};

// fills nsl images of R rows: src[r·R + c] is the stick of held row r and held column c, -1 for zero
template <typename T, int N, int NT, int U>
__device__ __forceinline__ void quarter_fill(typename V2t<T>::t* P, const typename V2t<T>::t* tp0, size_t band_stride,
                                             int nsl, const int* __restrict__ src) {
  using V2 = typename V2t<T>::t;
  using Q = Quarter<N>;
  constexpr int n = Q::R * Q::R;
  for (int e0 = threadIdx.x; e0 < n; e0 += U * NT) {
    int s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) s[u] = src[min(e0 + u * NT, n - 1)];
    for (int p = 0; p < nsl; ++p) {
      const V2* tp = tp0 + (size_t)p * band_stride;
      V2 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = tp[max(s[u], 0)];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * NT;
        if (e < n) {
          const int r = e / Q::R, c = e - r * Q::R;
          V2 x;
          x.x = s[u] >= 0 ? v[u].x : (T)0;
          x.y = s[u] >= 0 ? v[u].y : (T)0;
          P[(p * Q::R + r) * Q::LD + Q::index(c)] = x;
        }
      }
    }
  }
}

// y-lines of the held rows: inverse (held columns in, all out) or forward (all in, held columns out)
template <typename T, int N, int NT, int SIGN>
__device__ __forceinline__ void quarter_ylines(typename V2t<T>::t* P, int nsl) {
  using Q = Quarter<N>;
  for (int t = threadIdx.x; t < nsl * Q::R; t += NT) {
    typename V2t<T>::t* row = P + t * Q::LD;
    T re[N], im[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const bool in = SIGN < 0 || Q::has(j);
      re[j] = in ? row[j].x : (T)0;
      im[j] = in ? row[j].y : (T)0;
    }
    fft_line<T, N, SIGN>(re, im);
#pragma unroll
    for (int f = 0; f < N; ++f)
      if (SIGN > 0 || Q::has(f)) {
        row[f].x = re[LineOrder<N>::pos(f)];
        row[f].y = im[LineOrder<N>::pos(f)];
      }
  }
}

// one x-line (column i2 of an image) from the held rows: inverse transform, frequency f at pos(f)
template <typename T, int N>
__device__ __forceinline__ void quarter_xline(const typename V2t<T>::t* col, T (&re)[N], T (&im)[N]) {
  using Q = Quarter<N>;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    re[j] = Q::has(j) ? col[Q::at(j) * Q::LD].x : (T)0;
    im[j] = Q::has(j) ? col[Q::at(j) * Q::LD].y : (T)0;
  }
  fft_line<T, N, 1>(re, im);
}

}  // namespace pwk
