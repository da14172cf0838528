// Local part of H·ψ and the z-inverse of the density on spheres within a quarter of the axes
// (planes.hpp, Quarter): the three passes of hpsi.hip with the transforms pruned at compile time.
//   z-inverse: the sticks of a workgroup (64) are one contiguous range of ψ, which goes through LDS so
//              that ψ is read coalesced; a lane transforms one stick.
//   plane:     SLOTS planes per workgroup in LDS: y-inverse, x-inverse, × V(r), x-forward, y-forward.
//   z-forward: a lane per stick; Hψ = T_kin ψ + (1/N)·(...) is formed in LDS in place of ψ, so that ψ, the
//              kinetic energies and Hψ are read and written coalesced.
// Bounds: the plane pass by vector arithmetic, the z passes by the stick buffer's traffic (144 bands on
// 60³: 49 MB each way, 10 us at the rate of a copy).
#include <algorithm>

#include "common.hpp"
#include "fft_sizes.hpp"
#include "planes.hpp"

namespace pwk {

namespace {

constexpr int ZS = 64;  // sticks (lanes) per workgroup of the z passes

// the basis range of the workgroup's sticks [s0, s1)
struct StickRange {
  int w0, n;
};
__device__ __forceinline__ StickRange stick_range(int s0, int s1, const int* __restrict__ st_pw0,
                                                  const int* __restrict__ st_cnt) {
  const int w0 = st_pw0[s0];
  return {w0, st_pw0[s1 - 1] + st_cnt[s1 - 1] - w0};
}

template <typename V, int U>
__device__ __forceinline__ void range_to_lds(V* dst, const V* __restrict__ src, int n) {
  for (int e0 = threadIdx.x; e0 < n; e0 += U * ZS) {
    V v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = src[min(e0 + u * ZS, n - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e0 + u * ZS < n) dst[e0 + u * ZS] = v[u];
  }
}

// FP32 60³ × 144 bands 18 us -> 16 us, FP64 45³ × 160 bands 18 us -> 17 us (against k_zinv).
template <typename T, int NZ>
__global__ void __launch_bounds__(ZS) k_zinv_q(const typename V2t<T>::t* __restrict__ psi,
                                               typename V2t<T>::t* __restrict__ tbuf, int npw, int S,
                                               const int* __restrict__ st_pw0, const int* __restrict__ st_cnt,
                                               const int* __restrict__ st_lo, const int* __restrict__ list) {
  using V2 = typename V2t<T>::t;
  using Q = Quarter<NZ>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  V2* L = reinterpret_cast<V2*>(smem_raw);
  const int s0 = blockIdx.x * ZS, s1 = min(S, s0 + ZS), b = blockIdx.y;
  const StickRange rg = stick_range(s0, s1, st_pw0, st_cnt);
  range_to_lds<V2, 8>(L, psi + (size_t)(list ? list[b] : b) * npw + rg.w0, rg.n);
  const int s = s0 + threadIdx.x;
  __syncthreads();
  if (s >= s1) return;
  const int cnt = st_cnt[s], lo = st_lo[s], o = st_pw0[s] - rg.w0 - lo;
  T re[NZ], im[NZ];
#pragma unroll
  for (int i3 = 0; i3 < NZ; ++i3) {
    re[i3] = im[i3] = 0;
    if (Q::has(i3)) {
      const int n3 = i3 < Q::PA ? i3 : i3 - NZ, j = n3 - lo;
      const bool in = j >= 0 && j < cnt;
      const V2 v = L[in ? o + n3 : 0];
      re[i3] = in ? v.x : (T)0;
      im[i3] = in ? v.y : (T)0;
    }
  }
  fft_line<T, NZ, 1>(re, im);
  V2* dst = tbuf + (size_t)b * NZ * S;  // uniform row pointers, one lane offset
  const unsigned us = (unsigned)s;
#pragma unroll
  for (int f = 0; f < NZ; ++f) {
    V2 v;
    v.x = re[LineOrder<NZ>::pos(f)];
    v.y = im[LineOrder<NZ>::pos(f)];
    (dst + (size_t)f * S)[us] = v;
  }
}

// FP32 60³ × 144 bands 38 us -> 21.6 us, FP64 45³ × 160 bands 36 us -> 30 us (against k_zfwd, which gathers
// and stores the sphere with strided accesses).
template <typename T, int NZ, class Entries>
__global__ void __launch_bounds__(ZS) k_zfwd_q(const typename V2t<T>::t* __restrict__ tbuf,
                                               const typename V2t<T>::t* __restrict__ psi,
                                               typename V2t<T>::t* __restrict__ hpsi, const T* __restrict__ kin, int npw,
                                               int S, const int* __restrict__ st_pw0, const int* __restrict__ st_cnt,
                                               const int* __restrict__ st_lo, T inv_n, int nbk, int b0,
                                               const Entries entries) {
  using V2 = typename V2t<T>::t;
  using Q = Quarter<NZ>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  V2* L = reinterpret_cast<V2*>(smem_raw);
  T* K = reinterpret_cast<T*>(L + ZS * (Q::R + 1));
  const int s0 = blockIdx.x * ZS, s1 = min(S, s0 + ZS), b = blockIdx.y;
  const StickRange rg = stick_range(s0, s1, st_pw0, st_cnt);
  const int s = min(s0 + (int)threadIdx.x, s1 - 1);  // lanes past the last stick repeat it and store nothing
  const V2* src = tbuf + (size_t)b * NZ * S;  // uniform row pointers, one lane offset
  const unsigned us = (unsigned)s;
  T re[NZ], im[NZ];
#pragma unroll
  for (int i3 = 0; i3 < NZ; ++i3) {
    const V2 v = (src + (size_t)i3 * S)[us];
    re[i3] = v.x;
    im[i3] = v.y;
  }
  range_to_lds<V2, 8>(L, psi + (size_t)b * npw + rg.w0, rg.n);
  range_to_lds<T, 8>(K, band_kin(entries, kin, npw, nbk, b0 + b) + rg.w0, rg.n);
  __syncthreads();
  fft_line<T, NZ, -1>(re, im);
  // a slot of the line that the stick does not reach goes to a discard element of the lane's own: without
  // a branch, which would draw the transform's last stages into it and double its registers
  const int cnt = s0 + (int)threadIdx.x < s1 ? st_cnt[s] : 0, lo = st_lo[s], o = st_pw0[s] - rg.w0 - lo;
  const int none = ZS * Q::R + threadIdx.x;
#pragma unroll
  for (int i3 = 0; i3 < NZ; ++i3) {
    if (!Q::has(i3)) continue;
    const int n3 = i3 < Q::PA ? i3 : i3 - NZ, j = n3 - lo;
    const int e = j >= 0 && j < cnt ? o + n3 : none;
    const V2 ps = L[e];
    const T tk = K[e];
    V2 x;
    x.x = tk * ps.x + re[LineOrder<NZ>::pos(i3)] * inv_n;
    x.y = tk * ps.y + im[LineOrder<NZ>::pos(i3)] * inv_n;
    L[e] = x;
  }
  __syncthreads();
  V2* h = hpsi + (size_t)b * npw + rg.w0;
  for (int e = threadIdx.x; e < rg.n; e += ZS) h[e] = L[e];
}

// Against the passes over every held row (126 us with one plane per workgroup, 96 us with two; 59 us of
// those were the vector instructions alone, which is why half of them are pruned): FP32 60³ × 144 bands
// 67 us, FP64 45³ × 160 bands 151 us -> 103 us.
// Up to 81 points in FP32 a line's registers leave room for two waves per SIMD, which 64 points does not
// get unasked: 64³ × 144 bands 111 us -> 71 us. FP64 lines spill under that bound.
template <typename T, int N, bool ONE>
__global__ void __launch_bounds__((PlaneShape<T, N, false, ONE>::NT), (sizeof(T) == 4 && N <= 81 ? 2 : 1))
    k_plane_q(typename V2t<T>::t* tbuf, int nb, const T* __restrict__ vr, int S, int nz, const int* __restrict__ src,
              const int* __restrict__ st_off) {
  using V2 = typename V2t<T>::t;
  using Sh = PlaneShape<T, N, false, ONE>;
  using Q = Quarter<N>;
  constexpr int NT = Sh::NT, SLOTS = Sh::SLOTS, IMG = Q::R * Q::LD;
  constexpr int U = in_flight<T, NT>(Q::R * Q::R);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  V2* P = reinterpret_cast<V2*>(smem_raw);
  const int i3 = blockIdx.x, b0 = blockIdx.y * SLOTS, nsl = min(SLOTS, nb - b0);
  const size_t stride = (size_t)nz * S;
  V2* tp0 = tbuf + (size_t)b0 * stride + (size_t)i3 * S;
  quarter_fill<T, N, NT, U>(P, tp0, stride, nsl, src);
  __syncthreads();
  quarter_ylines<T, N, NT, 1>(P, nsl);
  __syncthreads();
  const int slot = threadIdx.x / N, i2 = threadIdx.x - slot * N;
  if (slot < nsl) {
    const T* v = vr + (size_t)i3 * N * N;
    const unsigned ui2 = (unsigned)i2;
    V2* col = P + slot * IMG + i2;
    T re[N], im[N];
    quarter_xline<T, N>(col, re, im);
    T r2[N], m2[N];
#pragma unroll
    for (int f = 0; f < N; ++f) {
      const T vv = (v + f * N)[ui2];
      r2[f] = re[LineOrder<N>::pos(f)] * vv;
      m2[f] = im[LineOrder<N>::pos(f)] * vv;
    }
    fft_line<T, N, -1>(r2, m2);
#pragma unroll
    for (int f = 0; f < N; ++f)
      if (Q::has(f)) {
        V2 x;
        x.x = r2[LineOrder<N>::pos(f)];
        x.y = m2[LineOrder<N>::pos(f)];
        col[Q::at(f) * Q::LD] = x;
      }
  }
  __syncthreads();
  quarter_ylines<T, N, NT, -1>(P, nsl);
  __syncthreads();
  for (int e0 = threadIdx.x; e0 < S; e0 += U * NT) {
    int off[U];
#pragma unroll
    for (int u = 0; u < U; ++u) off[u] = st_off[min(e0 + u * NT, S - 1)];
    for (int p = 0; p < nsl; ++p) {
      V2* tp = tp0 + (size_t)p * stride;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (e0 + u * NT < S) tp[e0 + u * NT] = P[p * IMG + off[u]];
    }
  }
}

// ---- grids with nx != ny ------------------------------------------------------------------
// The plane pass in three launches, so that each axis has its own compiled length: y-lines of the held rows
// (sticks -> U[band][i3][held row][i2]), x-lines with the potential between (a lane per (i3, i2), its line
// read and written along i2), y-lines back to the sticks. Only the held rows move between the launches.
// 50 × 25 × 25, 40 bands FP32: a whole H·ψ 60 us -> 25 us; the whole-grid transforms that this replaces took
// nine launches over all points. Bound: launches and the latency of one short wave each.
constexpr int RT = 64;

template <typename T, int NY, int SIGN>
__global__ void __launch_bounds__(RT) k_rows_q(typename V2t<T>::t* __restrict__ tbuf, typename V2t<T>::t* __restrict__ U,
                                               int S, int nz, int rx, const int* __restrict__ src,
                                               const int* __restrict__ st_off) {
  using V2 = typename V2t<T>::t;
  using Q = Quarter<NY>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  V2* P = reinterpret_cast<V2*>(smem_raw);  // [held row][LD]
  const size_t pl = (size_t)blockIdx.y * nz + blockIdx.x;
  V2* tp = tbuf + pl * S;
  V2* up = U + pl * rx * NY;
  if (SIGN > 0) {
    const int n = rx * Q::R;
    for (int e0 = threadIdx.x; e0 < n; e0 += 8 * RT) {
      int s[8];
      V2 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) s[u] = src[min(e0 + u * RT, n - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = tp[max(s[u], 0)];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int e = e0 + u * RT, r = e / Q::R;
        V2 x;
        x.x = s[u] >= 0 ? v[u].x : (T)0;
        x.y = s[u] >= 0 ? v[u].y : (T)0;
        if (e < n) P[r * Q::LD + Q::index(e - r * Q::R)] = x;
      }
    }
  } else {
#pragma unroll 8
    for (int e = threadIdx.x; e < rx * NY; e += RT) P[e / NY * Q::LD + e % NY] = up[e];
  }
  __syncthreads();
  for (int r = threadIdx.x; r < rx; r += RT) {
    V2* row = P + r * Q::LD;
    T re[NY], im[NY];
#pragma unroll
    for (int j = 0; j < NY; ++j) {
      const bool in = SIGN < 0 || Q::has(j);
      re[j] = in ? row[j].x : (T)0;
      im[j] = in ? row[j].y : (T)0;
    }
    fft_line<T, NY, SIGN>(re, im);
#pragma unroll
    for (int f = 0; f < NY; ++f)
      if (SIGN > 0 || Q::has(f)) {
        row[f].x = re[LineOrder<NY>::pos(f)];
        row[f].y = im[LineOrder<NY>::pos(f)];
      }
  }
  __syncthreads();
  if (SIGN > 0) {
#pragma unroll 8
    for (int e = threadIdx.x; e < rx * NY; e += RT) up[e] = P[e / NY * Q::LD + e % NY];
  } else {
#pragma unroll 8
    for (int s = threadIdx.x; s < S; s += RT) tp[s] = P[st_off[s]];
  }
}

template <typename T, int NX>
__global__ void __launch_bounds__(RT) k_cols_q(typename V2t<T>::t* U, const T* __restrict__ vr, int ny, int nz,
                                               int nlines) {
  using V2 = typename V2t<T>::t;
  using Q = Quarter<NX>;
  const int l = blockIdx.x * RT + threadIdx.x;  // i3·ny + i2
  if (l >= nlines) return;
  const int i3 = l / ny, i2 = l - i3 * ny;
  V2* up = U + ((size_t)blockIdx.y * nz + i3) * Q::R * ny + i2;
  const T* v = vr + (size_t)i3 * NX * ny + i2;
  T re[NX], im[NX];
#pragma unroll
  for (int j = 0; j < NX; ++j) {
    V2 x;
    x.x = x.y = 0;
    if (Q::has(j)) x = up[Q::at(j) * ny];
    re[j] = x.x;
    im[j] = x.y;
  }
  fft_line<T, NX, 1>(re, im);
  T r2[NX], m2[NX];
#pragma unroll
  for (int f = 0; f < NX; ++f) {
    const T vv = v[f * ny];
    r2[f] = re[LineOrder<NX>::pos(f)] * vv;
    m2[f] = im[LineOrder<NX>::pos(f)] * vv;
  }
  fft_line<T, NX, -1>(r2, m2);
#pragma unroll
  for (int f = 0; f < NX; ++f)
    if (Q::has(f)) {
      V2 x;
      x.x = r2[LineOrder<NX>::pos(f)];
      x.y = m2[LineOrder<NX>::pos(f)];
      up[Q::at(f) * ny] = x;
    }
}

template <typename T, int N, int SIGN>
void rows_q(Context& c, int nb, typename V2t<T>::t* tbuf, typename V2t<T>::t* U) {
  const int rx = 2 * ((c.dims[0] - 1) / 4) + 1;
  const size_t sh = (size_t)rx * Quarter<N>::LD * sizeof(typename V2t<T>::t);
  ensure_lds_limit((const void*)k_rows_q<T, N, SIGN>, sh);
  k_rows_q<T, N, SIGN><<<dim3((unsigned)c.dims[2], (unsigned)nb), RT, sh, c.stream>>>(
      tbuf, U, c.nsticks, c.dims[2], rx, c.q_src.as<int>(), c.q_off.as<int>());
}

template <typename T, int SIGN>
void rows_any(Context& c, int nb, typename V2t<T>::t* tbuf, typename V2t<T>::t* U) {
  switch (c.dims[1]) {
#define PWK_CASE(L) \
  case L:           \
    rows_q<T, L, SIGN>(c, nb, tbuf, U); \
    break;
    PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
    default:
      throw Error(PWK_E_UNSUPPORTED, "ny has no compiled kernel");
  }
  PWK_HIP(hipGetLastError());
}

template <typename T, int N, bool ONE>
void plane_q(Context& c, typename V2t<T>::t* tbuf, int nb, const T* vr) {
  using Sh = PlaneShape<T, N, false, ONE>;
  const size_t sh = (size_t)Sh::SLOTS * Quarter<N>::R * Quarter<N>::LD * sizeof(typename V2t<T>::t);
  ensure_lds_limit((const void*)k_plane_q<T, N, ONE>, sh);
  k_plane_q<T, N, ONE><<<dim3((unsigned)c.dims[2], blocks_for((size_t)nb, Sh::SLOTS)), Sh::NT, sh, c.stream>>>(
      tbuf, nb, vr, c.nsticks, c.dims[2], c.q_src.as<int>(), c.q_off.as<int>());
}

// One plane per workgroup where the form with more than two would leave SIMDs without a wave (FP32: fewer
// waves than the 1024 of the chip; half of that in FP64, whose planes take twice as long): a whole H·ψ of 16
// FP32 bands on 25³ 18.2 us -> 15.9 us, of 60 19.2 -> 17.2, of 140 22.1 against 23.0; 8 bands on 36³ 21.6 ->
// 17.9, 140 bands 34.0 against 36.7. A single band has the waves of the larger form to itself (FP64 45³ 26.5
// against 27.6), and two planes (54 points and more) stay together: 60³ x 1 band 25.8 us against 28.7.
template <typename T, int N>
void plane_any(Context& c, typename V2t<T>::t* tbuf, int nb, const T* vr) {
  using Sh = PlaneShape<T, N>;
  if constexpr (Sh::SLOTS > 2) {
    const long waves = (long)c.dims[2] * ((nb + Sh::SLOTS - 1) / Sh::SLOTS) * Sh::W;
    if (nb > 1 && waves < (sizeof(T) == 4 ? 1024 : 512)) {
      plane_q<T, N, true>(c, tbuf, nb, vr);
      return;
    }
  }
  plane_q<T, N, false>(c, tbuf, nb, vr);
}

template <typename T, int N, class Entries>
void zfwd_q(Context& c, const typename V2t<T>::t* tbuf, int nb, const T* kin, int nbk, int b0, const Entries& entries,
            const void* psi, void* hpsi) {
  using V2 = typename V2t<T>::t;
  const size_t sh = (size_t)ZS * (Quarter<N>::R + 1) * (sizeof(V2) + sizeof(T));
  ensure_lds_limit((const void*)k_zfwd_q<T, N, Entries>, sh);
  k_zfwd_q<T, N, Entries><<<dim3(blocks_for((size_t)c.nsticks, ZS), (unsigned)nb), ZS, sh, c.stream>>>(
      tbuf, (const V2*)psi, (V2*)hpsi, kin, c.npw, c.nsticks, c.st_pw0.as<int>(), c.st_cnt.as<int>(),
      c.st_n3lo.as<int>(), (T)(1.0 / (double)c.N), nbk, b0, entries);
}

template <typename T, int N>
void zinv_q(Context& c, int nb, const void* psi, typename V2t<T>::t* tbuf, const int* list) {
  using V2 = typename V2t<T>::t;
  const size_t sh = (size_t)ZS * Quarter<N>::R * sizeof(V2);
  ensure_lds_limit((const void*)k_zinv_q<T, N>, sh);
  k_zinv_q<T, N><<<dim3(blocks_for((size_t)c.nsticks, ZS), (unsigned)nb), ZS, sh, c.stream>>>(
      (const V2*)psi, tbuf, c.npw, c.nsticks, c.st_pw0.as<int>(), c.st_cnt.as<int>(), c.st_n3lo.as<int>(), list);
}

}  // namespace

template <typename T>
void sphere_zinv(Context& c, int nb, const void* psi, void* out, const int* list) {
  auto* tbuf = (typename V2t<T>::t*)out;
  switch (c.dims[2]) {
#define PWK_CASE(L) \
  case L:           \
    zinv_q<T, L>(c, nb, psi, tbuf, list); \
    break;
    PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
    default:
      throw Error(PWK_E_UNSUPPORTED, "nz has no compiled kernel");
  }
  PWK_HIP(hipGetLastError());
}

size_t sphere_rows_elems(const Context& c, int nb) {
  return (size_t)nb * c.dims[2] * (2 * ((c.dims[0] - 1) / 4) + 1) * c.dims[1];
}

int stick_chunk(const Context& c, int nb, size_t es) {
  if (c.dims[0] == c.dims[1]) return nb;
  const size_t per = ((size_t)c.dims[2] * c.nsticks + sphere_rows_elems(c, 1)) * es;
  return (int)std::max<size_t>(1, std::min<size_t>(std::min<size_t>((size_t)nb, 32768), ((size_t)256 << 20) / per));
}

template <typename T>
void sphere_rows_inverse(Context& c, int nb, void* buf, void* rows) {
  rows_any<T, 1>(c, nb, (typename V2t<T>::t*)buf, (typename V2t<T>::t*)rows);
}

template <typename T>
void sphere_plane(Context& c, int nb, void* buf, const T* vr, void* rows) {
  auto* tbuf = (typename V2t<T>::t*)buf;
  if (c.dims[0] != c.dims[1]) {
    auto* U = (typename V2t<T>::t*)rows;
    const int nlines = c.dims[1] * c.dims[2];
    const dim3 g(blocks_for((size_t)nlines, RT), (unsigned)nb);
    rows_any<T, 1>(c, nb, tbuf, U);
    switch (c.dims[0]) {
#define PWK_CASE(L) \
  case L:           \
    k_cols_q<T, L><<<g, RT, 0, c.stream>>>(U, vr, c.dims[1], c.dims[2], nlines); \
    break;
      PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
      default:
        throw Error(PWK_E_UNSUPPORTED, "nx has no compiled kernel");
    }
    PWK_HIP(hipGetLastError());
    rows_any<T, -1>(c, nb, tbuf, U);
    return;
  }
  switch (c.dims[0]) {
#define PWK_CASE(L) \
  case L:           \
    plane_any<T, L>(c, tbuf, nb, vr); \
    break;
    PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
    default:
      throw Error(PWK_E_UNSUPPORTED, "nx has no compiled kernel");
  }
  PWK_HIP(hipGetLastError());
}

template <typename T, class Entries>
void sphere_zfwd(Context& c, int nb, const void* buf, const T* kin, int nbk, int b0, const Entries& entries,
                 const void* psi, void* hpsi) {
  auto* tbuf = (const typename V2t<T>::t*)buf;
  switch (c.dims[2]) {
#define PWK_CASE(L) \
  case L:           \
    zfwd_q<T, L>(c, tbuf, nb, kin, nbk, b0, entries, psi, hpsi); \
    break;
    PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
    default:
      throw Error(PWK_E_UNSUPPORTED, "nz has no compiled kernel");
  }
  PWK_HIP(hipGetLastError());
}

template void sphere_zinv<float>(Context&, int, const void*, void*, const int*);
template void sphere_zinv<double>(Context&, int, const void*, void*, const int*);
template void sphere_rows_inverse<float>(Context&, int, void*, void*);
template void sphere_rows_inverse<double>(Context&, int, void*, void*);
template void sphere_plane<float>(Context&, int, void*, const float*, void*);
template void sphere_plane<double>(Context&, int, void*, const double*, void*);
#define PWK_INST(T)                                                                                                  \
  template void sphere_zfwd(Context&, int, const void*, const T*, int, int, const NoBatch&, const void*, void*);      \
  template void sphere_zfwd(Context&, int, const void*, const T*, int, int, const BatchKin<FEW_BATCH_ENTRIES>&,       \
                            const void*, void*);                                                                      \
  template void sphere_zfwd(Context&, int, const void*, const T*, int, int, const BatchKin<MAX_BATCH_ENTRIES>&,       \
                            const void*, void*);
PWK_INST(float)
PWK_INST(double)
#undef PWK_INST

}  // namespace pwk
