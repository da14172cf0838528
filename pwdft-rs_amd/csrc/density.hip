// Band density on the sphere-pruned FFT: ρ(r) += Σ_b fw_b |ψ_b(r)|²
// (src/scf/density.rs:59-97).
//
// Three launches: the z-inverse of the bands that carry weight (launch_zinv), the plane pass
// k_plane_density on (z-plane, band group), and k_density_sum, which adds the groups' FP64 partial
// sums in group order, so the result does not depend on scheduling; two where a small grid has one group.
#include <algorithm>
#include <vector>

#include "common.hpp"
#include "fft_sizes.hpp"
#include "planes.hpp"

namespace pwk {

namespace {

// Whether a thread keeps the FP64 sums of its x-line in registers: the line and its sums in at most
// 280 32-bit registers; longer lines keep them in LDS.
template <typename T, int N>
constexpr bool acc_in_regs() {
  return 2 * N * (int)(sizeof(T) / 4) + 2 * N <= 280;
}
template <int N, bool QUARTER>
struct LineTable : LineOrder<N> {};
template <int N>
struct LineTable<N, false> : FftOrder<N> {};
template <typename T, int N>
using DensityShape = PlaneShape<T, N, !acc_in_regs<T, N>()>;

// One z-plane of `per` batches of SLOTS bands per workgroup: y- and x-inverse of each, then the sums
// of fw·|ψ|² over the workgroup's bands to part[group][i3][i1][i2]. A thread owns one x-line of one
// slot throughout, so its sums stay in registers over all its bands and are added across the slots
// once, at the end.
// Bound: vector arithmetic of the line transforms (a band's plane enters LDS once and never
// returns). One workgroup per plane that loops over every band, as before, left 60 of 256 CUs with
// one wave each: 144 FP32 bands on 60³ 1741 us -> 72 us;
// 540 FP64 bands on 25³, the whole density beside other work, 901 us -> 31 us.
// QUARTER: a sphere within a quarter of the axes (planes.hpp); otherwise the held rows come from the
// basis' tables. DIRECT: the one group adds its sums to ρ itself.
template <typename T, int N, bool QUARTER, bool DIRECT>
__global__ void __launch_bounds__((DensityShape<T, N>::NT))
    k_plane_density(const typename V2t<T>::t* __restrict__ tbuf, int nb, int per, const double* __restrict__ fw,
                    double* __restrict__ part, int S, int nz, const int* __restrict__ src, int image,
                    PlaneRows pr, int nx1, const int* __restrict__ x1list, int overwrite) {
  using V2 = typename V2t<T>::t;
  using Sh = DensityShape<T, N>;
  constexpr int LD = Sh::LD, NT = Sh::NT, SLOTS = Sh::SLOTS;
  constexpr bool REGS = acc_in_regs<T, N>();
  constexpr int U = 16 / (int)(sizeof(T) / 4);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  V2* P = reinterpret_cast<V2*>(smem_raw);
  double* acc_lds = reinterpret_cast<double*>(smem_raw + (size_t)SLOTS * image * sizeof(V2));  // !REGS
  const int i3 = blockIdx.x, g = blockIdx.y, t = threadIdx.x;
  const int slot = t / N, i2 = t - slot * N;
  double acc[REGS ? N : 1];
#pragma unroll
  for (int q = 0; q < (REGS ? N : 1); ++q) acc[q] = 0.0;
  if (!REGS)
    for (int i = t; i < SLOTS * N * N; i += NT) acc_lds[i] = 0.0;
  const int b_end = min(nb, (g + 1) * per * SLOTS);
  for (int b0 = g * per * SLOTS; b0 < b_end; b0 += SLOTS) {
    const int nsl = min(SLOTS, b_end - b0);
    const V2* tp0 = tbuf + ((size_t)b0 * nz + i3) * S;
    if constexpr (QUARTER)
      quarter_fill<T, N, NT, U>(P, tp0, (size_t)nz * S, nsl, src);
    else
      plane_fill<T, N, NT, U>(P, image, tp0, (size_t)nz * S, nsl, src, image);
    __syncthreads();
    if constexpr (QUARTER)
      quarter_ylines<T, N, NT, 1>(P, nsl);
    else
      plane_ylines<T, N, NT, 1>(P, image, nsl, nx1, x1list);
    __syncthreads();
    const double f = slot < nsl ? fw[b0 + slot] : 0.0;
    if (!(f < 1e-15)) {  // src/scf/density.rs:14,72
      const V2* col = P + slot * image + i2;
      T re[N], im[N];
      if constexpr (QUARTER) {
        quarter_xline<T, N>(col, re, im);
      } else {
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const V2 v = col[plane_row<N>(pr, j, nx1) * LD];
          re[j] = v.x;
          im[j] = v.y;
        }
        fft_dif<T, N, 1>(re, im);
      }
#pragma unroll
      for (int q = 0; q < N; ++q) {
        const int o = LineTable<N, QUARTER>::pos(q);
        const double x = (double)re[o], y = (double)im[o];
        if constexpr (REGS)
          acc[q] += f * (x * x + y * y);
        else
          acc_lds[(slot * N + q) * N + i2] += f * (x * x + y * y);
      }
    }
    __syncthreads();  // the image is filled again
  }
  // add the slots in order and write the plane
  double* sum = REGS ? reinterpret_cast<double*>(smem_raw) : acc_lds;  // [N][N]
  if constexpr (REGS) {
    const int used = DIRECT ? min(SLOTS, nb) : SLOTS;
    for (int p = 0; p < used; ++p) {
      if (slot == p) {
#pragma unroll
        for (int q = 0; q < N; ++q) sum[q * N + i2] = p == 0 ? acc[q] : sum[q * N + i2] + acc[q];
      }
      __syncthreads();
    }
  }
  double* out = part + ((size_t)g * nz + i3) * N * N;
  for (int i = t; i < N * N; i += NT) {
    double s = sum[i];
    if (!REGS)
      for (int p = 1; p < SLOTS; ++p) s += sum[p * N * N + i];
    if constexpr (DIRECT) {
      double* d = &part[(size_t)i * nz + i3];
      *d = overwrite ? s : *d + s;
    } else {
      out[i] = s;
    }
  }
}

// The same for grids with nx != ny, whose y-lines have been taken already (rows[band][i3][held row][i2],
// sphere_rows_inverse): a lane per (i3, i2) transforms its x-line of every band of the group.
template <typename T, int NX>
__global__ void __launch_bounds__(64) k_cols_density(const typename V2t<T>::t* __restrict__ rows, int nb, int per,
                                                     const double* __restrict__ fw, double* __restrict__ part, int ny,
                                                     int nz) {
  using V2 = typename V2t<T>::t;
  using Q = Quarter<NX>;
  const int l = blockIdx.x * 64 + threadIdx.x, g = blockIdx.y;
  if (l >= ny * nz) return;
  const int i3 = l / ny, i2 = l - i3 * ny;
  double acc[NX];
#pragma unroll
  for (int q = 0; q < NX; ++q) acc[q] = 0.0;
  const int b_end = min(nb, (g + 1) * per);
  for (int b = g * per; b < b_end; ++b) {
    const V2* up = rows + ((size_t)b * nz + i3) * Q::R * ny + i2;
    const double f = fw[b];
    if (f < 1e-15) continue;
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
#pragma unroll
    for (int q = 0; q < NX; ++q) {
      const double x = (double)re[LineOrder<NX>::pos(q)], y = (double)im[LineOrder<NX>::pos(q)];
      acc[q] += f * (x * x + y * y);
    }
  }
  double* out = part + ((size_t)g * nz + i3) * NX * ny + i2;
#pragma unroll
  for (int q = 0; q < NX; ++q) out[q * ny] = acc[q];
}

// rho[i1][i2][i3] (+)= Σ_g part[g][i3][i1][i2] in group order; a 32 × 32 (i2, i3) tile per workgroup
// goes through LDS, so that both sides are read and written along their contiguous axis. Bound: the
// partials' traffic (groups·N·8 bytes; 60³ in 15 groups 26 MB, 8.5 us).
__global__ void __launch_bounds__(256) k_density_sum(int ngroups, int nx, int ny, int nz, const double* __restrict__ part,
                                                     double* __restrict__ rho, int overwrite) {
  __shared__ double tile[32][33];
  const int i1 = blockIdx.z, i20 = blockIdx.x * 32, i30 = blockIdx.y * 32;
  const int c = threadIdx.x & 31, r = threadIdx.x >> 5;
  const size_t n = (size_t)nx * ny * nz;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  const int i2 = min(i20 + c, ny - 1);
  size_t o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = ((size_t)min(i30 + r + 8 * k, nz - 1) * nx + i1) * ny + i2;
#pragma unroll 4
  for (int g = 0; g < ngroups; ++g)
#pragma unroll
    for (int k = 0; k < 4; ++k) s[k] += part[(size_t)g * n + o[k]];
#pragma unroll
  for (int k = 0; k < 4; ++k) tile[r + 8 * k][c] = s[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int y = i20 + r + 8 * k, z = i30 + c;
    if (y < ny && z < nz) {
      double* d = &rho[((size_t)i1 * ny + y) * nz + z];
      const double v = tile[c][r + 8 * k];
      *d = overwrite ? v : *d + v;
    }
  }
}

template <typename T, int N, bool QUARTER, bool DIRECT>
void plane_density(Context& c, const void* tbuf, int nb, int per, int groups, const double* fw, double* part,
                   int overwrite) {
  using V2 = typename V2t<T>::t;
  using Sh = DensityShape<T, N>;
  const int image = QUARTER ? Quarter<N>::R * Quarter<N>::LD : c.pl_rows * Sh::LD;
  size_t sh = (size_t)Sh::SLOTS * image * sizeof(V2);
  if (acc_in_regs<T, N>())
    sh = std::max(sh, (size_t)N * N * sizeof(double));
  else
    sh += (size_t)Sh::SLOTS * N * N * sizeof(double);
  PWK_REQUIRE(sh <= 160 * 1024, PWK_E_UNSUPPORTED, "density plane exceeds the LDS");
  ensure_lds_limit((const void*)k_plane_density<T, N, QUARTER, DIRECT>, sh);
  const PlaneRows pr{c.pl_ra, c.pl_rb};
  k_plane_density<T, N, QUARTER, DIRECT><<<dim3((unsigned)c.dims[2], (unsigned)groups), Sh::NT, sh, c.stream>>>(
      (const V2*)tbuf, nb, per, fw, part, c.nsticks, c.dims[2], QUARTER ? c.q_src.as<int>() : c.pl_src.as<int>(), image,
      pr, c.nx1, c.x1_runs ? nullptr : c.x1list.as<int>(), overwrite);
  PWK_HIP(hipGetLastError());
}

constexpr int DIRECT_MAX = 27;  // the longest axis of grids whose one group adds to ρ itself
template <typename T, int N>
void plane_density_any(Context& c, int nb, int per, int groups, const double* fw, double* part, double* rho,
                       int overwrite, bool direct) {
  if constexpr (N <= DIRECT_MAX) {
    if (direct) {
      if (c.quarter)
        plane_density<T, N, true, true>(c, c.work_a.p, nb, per, 1, fw, rho, overwrite);
      else
        plane_density<T, N, false, true>(c, c.work_a.p, nb, per, 1, fw, rho, overwrite);
      return;
    }
  }
  if (c.quarter)
    plane_density<T, N, true, false>(c, c.work_a.p, nb, per, groups, fw, part, 0);
  else
    plane_density<T, N, false, false>(c, c.work_a.p, nb, per, groups, fw, part, 0);
}

template <typename T>
int plane_slots(int n) {
  switch (n) {
#define PWK_CASE(L) \
  case L:           \
    return DensityShape<T, L>::SLOTS;
    PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
    default:
      throw Error(PWK_E_UNSUPPORTED, "nx has no compiled kernel");
  }
}

template <typename T>
void density_sticks_t(Context& c, int nb, const void* psi, const double* fw_host, double* rho, bool overwrite) {
  using V2 = typename V2t<T>::t;
  // the bands that carry weight (src/scf/density.rs:14,72), their weights first. While the stream is captured
  // every band is transformed and the weights are the caller's own at each replay: the kernels skip the
  // bands without weight.
  const bool captured = c.capturing();
  std::vector<double>& h = c.dens_host;
  int live = nb;
  if (!captured) {
    h.clear();
    for (int b = 0; b < nb; ++b)
      if (!(fw_host[b] < 1e-15)) h.push_back(fw_host[b]);
    live = (int)h.size();
    h.resize((size_t)live + (size_t)(live + 1) / 2);
    int32_t* list = reinterpret_cast<int32_t*>(h.data() + live);
    for (int b = 0, i = 0; b < nb; ++b)
      if (!(fw_host[b] < 1e-15)) list[i++] = b;
  }
  const int nx = c.dims[0], ny = c.dims[1], nz = c.dims[2];
  // about 1024 workgroups (four per CU): more only adds partial sums to store and read, fewer leave
  // CUs idle (60³ × 144 bands: 72 batches × 60 planes in 15 groups).
  const bool square = nx == ny;
  const int slots = square ? plane_slots<T>(nx) : 1;
  const long wgs = square ? nz : (ny * nz + 63) / 64;  // workgroups per group
  // The workspaces are sized for all nb bands, whatever their weights: a captured call transforms every band
  // and cannot allocate, and its first run outside the graph may have had bands without weight. One z-inverse
  // buffer (of a chunk), then the groups' partial sums, of which any number of live bands makes at most
  // max_groups.
  const int chunk = stick_chunk(c, nb, sizeof(V2));
  const size_t ns = (size_t)chunk * nz * c.nsticks, held = square ? 0 : sphere_rows_elems(c, chunk);
  const size_t tb = ((ns + held) * sizeof(V2) + 255) & ~(size_t)255;
  const long max_groups = std::min<long>((chunk + slots - 1) / slots, (1024 + wgs - 1) / wgs);
  c.workspace(c.work_a, tb + (size_t)max_groups * c.N * sizeof(double));
  c.workspace(c.work_b, ((size_t)nb + (size_t)(nb + 1) / 2) * sizeof(double));
  if (live > 0) {
    const size_t wbytes = (captured ? (size_t)nb : h.size()) * sizeof(double);
    PWK_HIP(hipMemcpyAsync(c.work_b.p, captured ? fw_host : h.data(), wbytes, hipMemcpyHostToDevice, c.stream));
    const double* weights = c.work_b.as<double>();
    double* part = reinterpret_cast<double*>(c.work_a.as<unsigned char>() + tb);
    V2* rows = c.work_a.as<V2>() + ns;
    for (int b0 = 0; b0 < live; b0 += chunk) {
      const int n = std::min(chunk, live - b0);
      const double* fw = weights + b0;
      const int batches = (n + slots - 1) / slots;
      const int per = std::max(1, (int)((batches * wgs + 1023) / 1024));
      const int groups = (batches + per - 1) / per;
      const int ow = overwrite && b0 == 0 ? 1 : 0;
      // one group on a small grid: the plane pass adds to ρ itself, at strides of nz, and the third launch goes
      // (15 x 15 x 16, 1 band 16.1 us -> 11.2, 20 x 20 x 24 14.9 -> 11.3; on 32³ 18.5 against 17.8, and
      // 60³ 45.1 against 29.6)
      const bool direct = square && groups == 1 && nx <= DIRECT_MAX && c.N <= 20000;
      launch_zinv(c, n, captured ? (const V2*)psi + (size_t)b0 * c.npw : psi, c.work_a.p,
                  std::is_same<T, double>::value ? PWK_FP64 : PWK_FP32,
                  captured ? nullptr : reinterpret_cast<const int*>(weights + live) + b0);
      if (!square) sphere_rows_inverse<T>(c, n, c.work_a.p, rows);
      switch (nx) {
#define PWK_CASE(L)                                                                                                   \
  case L:                                                                                                             \
    if (!square)                                                                                                      \
      k_cols_density<T, L><<<dim3((unsigned)wgs, (unsigned)groups), 64, 0, c.stream>>>(rows, n, per, fw, part, ny, nz); \
    else                                                                                                              \
      plane_density_any<T, L>(c, n, per, groups, fw, part, rho, ow, direct);                                          \
    break;
        PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
        default:
          throw Error(PWK_E_UNSUPPORTED, "nx has no compiled kernel");
      }
      PWK_HIP(hipGetLastError());
      if (direct) continue;
      const dim3 gs(blocks_for((size_t)ny, 32), blocks_for((size_t)nz, 32), (unsigned)nx);
      k_density_sum<<<gs, 256, 0, c.stream>>>(groups, nx, ny, nz, part, rho, ow);
      PWK_HIP(hipGetLastError());
    }
  } else if (overwrite) {
    const dim3 gs(blocks_for((size_t)ny, 32), blocks_for((size_t)nz, 32), (unsigned)nx);
    k_density_sum<<<gs, 256, 0, c.stream>>>(0, nx, ny, nz, nullptr, rho, 1);
    PWK_HIP(hipGetLastError());
  }
}

}  // namespace

void launch_density_sticks(Context& c, int nb, const void* psi, const double* fw_host, void* rho, int precision,
                           bool overwrite) {
  if (precision == PWK_FP64)
    density_sticks_t<double>(c, nb, psi, fw_host, (double*)rho, overwrite);
  else
    density_sticks_t<float>(c, nb, psi, fw_host, (double*)rho, overwrite);
}

}  // namespace pwk
