// Local part of H·ψ on the sphere-pruned FFT.
//
// The plane-wave sphere occupies S z-sticks (distinct (n1, n2)); the
// reference enumerates the basis n1 -> n2 -> n3 (src/basis.rs:47-59), so the
// coefficients of one stick are contiguous. One H·ψ is three kernels:
//   k_zinv   : per (band, stick) scatter ψ along z, inverse FFT along z
//              -> stick buffer T[band][i3][stick]            (S·nz values)
//   k_plane  : per (band, z-plane) in LDS: y-inverse on the rows carrying
//              sticks, x-inverse, × V(r), x-forward, y-forward -> T
//   k_zfwd   : per (band, stick) forward FFT along z, gather the sphere,
//              Hψ = T_kin ψ + (1/N)·(...)                  (src/scf/potentials.rs:163-190)
// which equals the dense fill_hamiltonian_with_v_eff product because the
// wrapped Miller difference there is a circular convolution.
// Bases within a quarter of every axis (the default ecutrho = 4·ecutwfc) take the same passes pruned at
// compile time (hpsi_sphere.hip); the kernels here serve the other bases on nx = ny, and the whole-grid
// transforms below the rest. The band density (density.hip) shares the z-inverse and the planes' layout.
#include <algorithm>

#include "common.hpp"
#include "fft_reg.hpp"
#include "fft_sizes.hpp"
#include "planes.hpp"
#include "sticks.hpp"

namespace pwk {

namespace {

// index of n3 ≡ i3 (mod nz) inside a stick starting at n3 = lo, or >= cnt if absent
__device__ __forceinline__ int stick_slot(int i3, int lo, int nz) {
  int j = i3 - lo;
  if (j < 0) j += nz;
  if (j >= nz) j -= nz;
  return j;
}

template <typename T, int NZ>
__global__ void __launch_bounds__(64) k_zinv(const typename V2t<T>::t* __restrict__ psi,
                                             typename V2t<T>::t* __restrict__ tbuf, int npw, int S,
                                             const int* __restrict__ st_pw0, const int* __restrict__ st_cnt,
                                             const int* __restrict__ st_lo, const int* __restrict__ list) {
  int s = blockIdx.x * 64 + threadIdx.x;
  int b = blockIdx.y;
  if (s >= S) return;
  int pw0 = st_pw0[s], cnt = st_cnt[s], lo = st_lo[s];
  const typename V2t<T>::t* src = psi + (size_t)(list ? list[b] : b) * npw + pw0;
  T re[NZ], im[NZ];
#pragma unroll
  for (int i3 = 0; i3 < NZ; ++i3) {
    int j = stick_slot(i3, lo, NZ);
    typename V2t<T>::t v;
    v.x = 0;
    v.y = 0;
    if (j < cnt) v = src[j];
    re[i3] = v.x;
    im[i3] = v.y;
  }
  fft_dif<T, NZ, 1>(re, im);
  typename V2t<T>::t* dst = tbuf + (size_t)b * NZ * S + s;
#pragma unroll
  for (int f = 0; f < NZ; ++f) {
    typename V2t<T>::t v;
    v.x = re[FftOrder<NZ>::pos(f)];
    v.y = im[FftOrder<NZ>::pos(f)];
    dst[(size_t)f * S] = v;
  }
}

template <typename T, int NZ, class Entries>
__global__ void __launch_bounds__(64) k_zfwd(const typename V2t<T>::t* __restrict__ tbuf,
                                             const typename V2t<T>::t* __restrict__ psi,
                                             typename V2t<T>::t* __restrict__ hpsi, const T* __restrict__ kin,
                                             int npw, int S, const int* __restrict__ st_pw0,
                                             const int* __restrict__ st_cnt, const int* __restrict__ st_lo,
                                             T inv_n, int nbk, const Entries entries) {
  int s = blockIdx.x * 64 + threadIdx.x;
  int b = blockIdx.y;
  const T* tb = nullptr;  // the entry's kinetic diagonal, by all lanes before any leaves
  if constexpr (Entries::batch) tb = band_kin(entries, kin, npw, nbk, b);
  if (s >= S) return;
  int pw0 = st_pw0[s], cnt = st_cnt[s], lo = st_lo[s];
  const typename V2t<T>::t* src = tbuf + (size_t)b * NZ * S + s;
  T re[NZ], im[NZ];
#pragma unroll
  for (int i3 = 0; i3 < NZ; ++i3) {
    typename V2t<T>::t v = src[(size_t)i3 * S];
    re[i3] = v.x;
    im[i3] = v.y;
  }
  fft_dif<T, NZ, -1>(re, im);
  if constexpr (sizeof(T) == 8 && NZ > 50) {
    // lines that fill the registers are complete here: drawn into the branches below, their last stages keep
    // twice the registers and spill (60 points 748 bytes a lane; shorter lines gain by the earlier loads)
#pragma unroll
    for (int f = 0; f < NZ; ++f) asm volatile("" : "+v"(re[f]), "+v"(im[f]));
  }
  const typename V2t<T>::t* p = psi + (size_t)b * npw + pw0;
  typename V2t<T>::t* h = hpsi + (size_t)b * npw + pw0;
  if constexpr (!Entries::batch) tb = kin + (size_t)(b / nbk) * npw;
  const T* t = tb + pw0;
#pragma unroll
  for (int i3 = 0; i3 < NZ; ++i3) {
    int j = stick_slot(i3, lo, NZ);
    if (j < cnt) {
      typename V2t<T>::t ps = p[j];
      T tk = t[j];
      typename V2t<T>::t o;
      o.x = tk * ps.x + re[FftOrder<NZ>::pos(i3)] * inv_n;
      o.y = tk * ps.y + im[FftOrder<NZ>::pos(i3)] * inv_n;
      h[j] = o;
    }
  }
}

// H·ψ plane pass: one z-plane of one band per workgroup (planes.hpp): y-inverse on the rows with
// sticks, x-inverse, × V(r), x-forward, y-forward, back to the sticks. The rows without sticks are zero
// through the y passes and their x output is never gathered: the x-lines read them from the image's
// zero row and write them to a discard row after it, so the loads and stores need no branch. Bound: the
// vector arithmetic of the line transforms; the traffic is the stick buffer in and out.
// Several planes per workgroup fill its waves better, but an image of a wide sphere's rows lets fewer waves
// on a CU and fewer workgroups start: a whole H·ψ with radius 9 on 25³, 16 FP32 bands 22.5 us against 18.8,
// radius 17 on 45³, 60 bands 77.6 against 60.2, radius 12 on 27³, 140 FP64 bands 73.4 against 63.2.
template <typename T, int N>
__global__ void __launch_bounds__((PlaneShape<T, N, false, true>::NT))
    k_plane_hpsi(typename V2t<T>::t* tbuf, const T* __restrict__ vr, int S, int nz, const int* __restrict__ src, int nsrc,
                 const int* __restrict__ st_off, PlaneRows pr, int nx1, const int* __restrict__ x1list) {
  using V2 = typename V2t<T>::t;
  constexpr int LD = N + 1, NT = PlaneShape<T, N, false, true>::NT;
  constexpr int UI = in_flight<T, NT>(N * LD), UO = in_flight<T, NT>(N * N / 2);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  V2* P = reinterpret_cast<V2*>(smem_raw);
  const int i3 = blockIdx.x, b = blockIdx.y, i2 = threadIdx.x;
  V2* tp = tbuf + ((size_t)b * nz + i3) * S;
  plane_fill<T, N, NT, UI>(P, 0, tp, 0, 1, src, nsrc);
  __syncthreads();
  plane_ylines<T, N, NT, 1>(P, 0, 1, nx1, x1list);
  __syncthreads();
  if (i2 < N) {
    const T* v = vr + (size_t)i3 * N * N + i2;
    V2* col = P + i2;
    T re[N], im[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const V2 x = col[plane_row<N>(pr, j, nx1) * LD];
      re[j] = x.x;
      im[j] = x.y;
    }
    fft_dif<T, N, 1>(re, im);
    T r2[N], m2[N];
#pragma unroll
    for (int f = 0; f < N; ++f) {
      const T vv = v[f * N];
      r2[f] = re[FftOrder<N>::pos(f)] * vv;
      m2[f] = im[FftOrder<N>::pos(f)] * vv;
    }
    fft_dif<T, N, -1>(r2, m2);
#pragma unroll
    for (int f = 0; f < N; ++f) {
      V2 x;
      x.x = r2[FftOrder<N>::pos(f)];
      x.y = m2[FftOrder<N>::pos(f)];
      col[plane_row<N>(pr, f, nx1 + 1) * LD] = x;
    }
  }
  __syncthreads();
  plane_ylines<T, N, NT, -1>(P, 0, 1, nx1, x1list);
  __syncthreads();
  for (int s0 = threadIdx.x; s0 < S; s0 += UO * NT) {
    int off[UO];
#pragma unroll
    for (int u = 0; u < UO; ++u) off[u] = st_off[min(s0 + u * NT, S - 1)];
#pragma unroll
    for (int u = 0; u < UO; ++u)
      if (s0 + u * NT < S) tp[s0 + u * NT] = P[off[u]];
  }
}

template <typename T, int N>
void plane_hpsi(Context& c, typename V2t<T>::t* tbuf, int nb, const T* vr) {
  const int nz = c.dims[2], rows = c.x1_runs ? c.pl_rows + 1 : c.pl_rows;
  const size_t sh = (size_t)rows * (N + 1) * sizeof(typename V2t<T>::t);
  PWK_REQUIRE(sh <= 160 * 1024, PWK_E_UNSUPPORTED, "plane exceeds the LDS");
  ensure_lds_limit((const void*)k_plane_hpsi<T, N>, sh);
  k_plane_hpsi<T, N><<<dim3((unsigned)nz, (unsigned)nb), PlaneShape<T, N, false, true>::NT, sh, c.stream>>>(
      tbuf, vr, c.nsticks, nz, c.pl_src.as<int>(), c.pl_rows * (N + 1), c.st_off.as<int>(),
      PlaneRows{c.pl_ra, c.pl_rb}, c.nx1, c.x1_runs ? nullptr : c.x1list.as<int>());
  PWK_HIP(hipGetLastError());
}

// V(r) = Re IFFT_unnorm(V_eff(G)) re-ordered to plane-major [i3][i1][i2] (stick path), and in
// grid order (fused small-grid path)
__global__ void __launch_bounds__(256) k_vr_reorder(const double2* __restrict__ vg_r, double* __restrict__ v64,
                                                    float* __restrict__ v32, double* __restrict__ n64,
                                                    float* __restrict__ n32, int nx, int ny, int nz) {
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t n = (size_t)nx * ny * nz;
  if (idx >= n) return;
  // idx in plane-major order
  int i2 = (int)(idx % ny);
  int i1 = (int)((idx / ny) % nx);
  int i3 = (int)(idx / ((size_t)nx * ny));
  const size_t g = ((size_t)i1 * ny + i2) * nz + i3;
  double v = vg_r[g].x;
  v64[idx] = v;
  v32[idx] = (float)v;
  n64[g] = v;
  n32[g] = (float)v;
}

// ---- full-grid path (an axis beyond the register lengths, or nx != ny with a wide sphere) --------
// the stick path's plane and z kernels hold whole lines in registers: square planes, every axis
// one of the register lengths; other grids of register lengths when the pruned passes apply (in FP64 up
// to x-lines of 64 points: longer ones do not fit the registers of the x passes)
bool stick_path_ok(const Context& c, bool f64) {
  return (c.quarter && (c.dims[0] == c.dims[1] || !f64 || c.dims[0] <= 64)) || (c.dims[0] == c.dims[1] && fft_len_compiled(c.dims[0]) && fft_len_compiled(c.dims[2]));
}

// ψ scattered on the whole grid of each band of a chunk, batched 3D FFTs (one compiled
// line length per axis), V(r) multiply and gather. Slower than the stick path but valid
// for every grid shape the line kernels compile.
template <typename T>
__global__ void __launch_bounds__(256) k_grid_zero(size_t n, typename V2t<T>::t* __restrict__ grid) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  typename V2t<T>::t z;
  z.x = 0;
  z.y = 0;
  grid[i] = z;
}

template <typename T>
__global__ void __launch_bounds__(256) k_grid_put(size_t n, size_t N, int npw, const typename V2t<T>::t* psi,
                                                  const int* __restrict__ g2fft, typename V2t<T>::t* __restrict__ grid) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;  // band · npw + g
  if (i >= n) return;
  const size_t b = i / npw, g = i % npw;
  grid[b * N + g2fft[g]] = psi[i];
}

template <typename T>
__global__ void __launch_bounds__(256) k_grid_mulv(size_t n, size_t N, const T* __restrict__ v,
                                                   typename V2t<T>::t* __restrict__ grid) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const T vv = v[i % N];
  grid[i].x *= vv;
  grid[i].y *= vv;
}

template <typename T>
__global__ void __launch_bounds__(256) k_grid_get(size_t n, size_t N, int npw, int nbk, int b0,
                                                  const typename V2t<T>::t* __restrict__ grid,
                                                  const int* __restrict__ g2fft,
                                                  const typename V2t<T>::t* __restrict__ psi, const T* __restrict__ kin,
                                                  typename V2t<T>::t* __restrict__ hpsi, T inv_n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;  // chunk band · npw + g
  if (i >= n) return;
  const size_t bl = i / npw, g = i % npw;
  const size_t b = (size_t)b0 + bl;
  const typename V2t<T>::t w = grid[bl * N + g2fft[g]], ps = psi[b * npw + g];
  const T tk = kin[(b / nbk) * npw + g];
  typename V2t<T>::t o;
  o.x = tk * ps.x + w.x * inv_n;
  o.y = tk * ps.y + w.y * inv_n;
  hpsi[b * npw + g] = o;
}

// ρ(r) += Σ_b fw_b |ψ_b(r)|² over the bands of a chunk in band order (src/scf/density.rs:59-97)
template <typename T>
__global__ void __launch_bounds__(256) k_grid_density(size_t N, int nbc, const typename V2t<T>::t* __restrict__ grid,
                                                      const double* __restrict__ fw, double* __restrict__ rho) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= N) return;
  double acc = rho[i];
  for (int b = 0; b < nbc; ++b) {
    const double f = fw[b];
    if (f < 1e-15) continue;  // src/scf/density.rs:14,72
    const typename V2t<T>::t v = grid[(size_t)b * N + i];
    const double x = (double)v.x, y = (double)v.y;
    acc += f * (x * x + y * y);
  }
  rho[i] = acc;
}

// bands per chunk of the full-grid path: at most 256 MiB of grids
template <typename T>
int grid_chunk(const Context& c, int nb) {
  const size_t per = c.N * sizeof(typename V2t<T>::t);
  return (int)std::max<size_t>(1, std::min<size_t>(std::min<size_t>((size_t)nb, 32768), ((size_t)256 << 20) / per));
}

template <typename T>
void hpsi_fullgrid(Context& c, const T* kin, int nb, int nbk, const void* psi, void* hpsi) {
  using V2 = typename V2t<T>::t;
  const int prec = std::is_same<T, double>::value ? PWK_FP64 : PWK_FP32;
  const T* vr = std::is_same<T, double>::value ? (const T*)c.vrn64.p : (const T*)c.vrn32.p;
  const size_t N = c.N;
  const int chunk = grid_chunk<T>(c, nb);
  c.workspace(c.work_a, (size_t)chunk * N * sizeof(V2));
  V2* grid = c.work_a.as<V2>();
  TimedScope ts(c, "hpsi_fullgrid");
  for (int b0 = 0; b0 < nb; b0 += chunk) {
    const int nbc = std::min(chunk, nb - b0);
    const size_t ng = (size_t)nbc * N, np = (size_t)nbc * c.npw;
    k_grid_zero<T><<<blocks_for(ng, 256), 256, 0, c.stream>>>(ng, grid);
    k_grid_put<T><<<blocks_for(np, 256), 256, 0, c.stream>>>(np, N, c.npw, (const V2*)psi + (size_t)b0 * c.npw,
                                                             c.g2fft.as<int>(), grid);
    PWK_HIP(hipGetLastError());
    launch_fft3d(c, grid, nbc, +1, prec);
    k_grid_mulv<T><<<blocks_for(ng, 256), 256, 0, c.stream>>>(ng, N, vr, grid);
    PWK_HIP(hipGetLastError());
    launch_fft3d(c, grid, nbc, -1, prec);
    k_grid_get<T><<<blocks_for(np, 256), 256, 0, c.stream>>>(np, N, c.npw, nbk, b0, grid, c.g2fft.as<int>(),
                                                             (const V2*)psi, kin, (V2*)hpsi,
                                                             (T)(1.0 / (double)N));
    PWK_HIP(hipGetLastError());
  }
}

template <typename T>
void density_fullgrid(Context& c, int nb, const void* psi, const double* fw_host, void* rho) {
  using V2 = typename V2t<T>::t;
  const int prec = std::is_same<T, double>::value ? PWK_FP64 : PWK_FP32;
  const size_t N = c.N;
  const int chunk = grid_chunk<T>(c, nb);
  c.workspace(c.work_a, (size_t)chunk * N * sizeof(V2));
  c.workspace(c.work_b, (size_t)nb * sizeof(double));
  PWK_HIP(hipMemcpyAsync(c.work_b.p, fw_host, (size_t)nb * sizeof(double), hipMemcpyHostToDevice, c.stream));
  V2* grid = c.work_a.as<V2>();
  for (int b0 = 0; b0 < nb; b0 += chunk) {
    const int nbc = std::min(chunk, nb - b0);
    const size_t ng = (size_t)nbc * N, np = (size_t)nbc * c.npw;
    k_grid_zero<T><<<blocks_for(ng, 256), 256, 0, c.stream>>>(ng, grid);
    k_grid_put<T><<<blocks_for(np, 256), 256, 0, c.stream>>>(np, N, c.npw, (const V2*)psi + (size_t)b0 * c.npw,
                                                             c.g2fft.as<int>(), grid);
    PWK_HIP(hipGetLastError());
    launch_fft3d(c, grid, nbc, +1, prec);
    k_grid_density<T><<<blocks_for(N, 256), 256, 0, c.stream>>>(N, nbc, grid, c.work_b.as<double>() + b0,
                                                                (double*)rho);
    PWK_HIP(hipGetLastError());
  }
}

// ---- dispatch ------------------------------------------------------------------
template <typename T>
void zinv_t(Context& c, int nb, const void* psi, typename V2t<T>::t* out, const int* list) {
  using V2 = typename V2t<T>::t;
  PWK_REQUIRE(nb <= 65535, PWK_E_UNSUPPORTED, "too many bands in one launch");
  if (c.quarter) {
    sphere_zinv<T>(c, nb, psi, out, list);
    return;
  }
  const dim3 gz(blocks_for((size_t)c.nsticks, 64), (unsigned)nb);
  switch (c.dims[2]) {
#define PWK_CASE(L)                                                                                             \
  case L:                                                                                                       \
    k_zinv<T, L><<<gz, 64, 0, c.stream>>>((const V2*)psi, out, c.npw, c.nsticks, c.st_pw0.as<int>(),            \
                                          c.st_cnt.as<int>(), c.st_n3lo.as<int>(), list);                       \
    break;
    PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
    default:
      throw Error(PWK_E_UNSUPPORTED, "nz has no compiled kernel");
  }
  PWK_HIP(hipGetLastError());
}

// Local part of H·ψ for nb bands; band b uses the kinetic diagonal kin + (b / nbk)·npw,
// so consecutive groups of nbk bands may belong to different k-points.
template <typename T, class Entries = NoBatch>
void hpsi_local(Context& c, const T* kin, int nb, int nbk, const void* psi, void* hpsi,
                const Entries& entries = Entries()) {
  using V2 = typename V2t<T>::t;
  int nx = c.dims[0], nz = c.dims[2];
  PWK_REQUIRE(c.have_v, PWK_E_STATE, "V_eff not set (pwk_set_veff)");
  if (!stick_path_ok(c, std::is_same<T, double>::value)) {
    hpsi_fullgrid<T>(c, kin, nb, nbk, psi, hpsi);
    return;
  }
  const int chunk = stick_chunk(c, nb, sizeof(V2));
  PWK_REQUIRE(chunk <= 65535, PWK_E_UNSUPPORTED, "too many bands in one H·psi launch");
  const size_t ns = (size_t)chunk * nz * c.nsticks, rows = nx == c.dims[1] ? 0 : sphere_rows_elems(c, chunk);
  c.workspace(c.work_a, (ns + rows) * sizeof(V2));
  V2* T_ = c.work_a.as<V2>();
  const T* vr = std::is_same<T, double>::value ? (const T*)c.vr64.p : (const T*)c.vr32.p;
  for (int b0 = 0; b0 < nb; b0 += chunk) {
    const int nbc = std::min(chunk, nb - b0);
    const V2* in = (const V2*)psi + (size_t)b0 * c.npw;
    V2* out = (V2*)hpsi + (size_t)b0 * c.npw;
    {
      TimedScope ts(c, "hpsi_zinv");
      zinv_t<T>(c, nbc, in, T_, nullptr);
    }
    {
      TimedScope ts(c, "hpsi_plane");
      // (the pruned FP64 plane pass of 81 points does not fit the registers)
      if (c.quarter && !(std::is_same<T, double>::value && nx > 80 && nx == c.dims[1])) {
        sphere_plane<T>(c, nbc, T_, vr, T_ + ns);
      } else {
        switch (nx) {
#define PWK_CASE(L)                    \
  case L:                              \
    plane_hpsi<T, L>(c, T_, nbc, vr);  \
    break;
          PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
          default:
            throw Error(PWK_E_UNSUPPORTED, "nx has no compiled kernel");
        }
      }
    }
    TimedScope ts(c, "hpsi_zfwd");
    if (c.quarter) {
      sphere_zfwd<T>(c, nbc, T_, kin, nbk, b0, entries, in, out);
      continue;
    }
    const T inv_n = (T)(1.0 / (double)c.N);
    const dim3 gz(blocks_for((size_t)c.nsticks, 64), (unsigned)nbc);  // (nx = ny: one chunk)
    switch (nz) {
#define PWK_CASE(L)                                                                                     \
  case L:                                                                                               \
    k_zfwd<T, L, Entries><<<gz, 64, 0, c.stream>>>(T_, in, out, kin, c.npw, c.nsticks,                  \
                                          c.st_pw0.as<int>(), c.st_cnt.as<int>(), c.st_n3lo.as<int>(),  \
                                          inv_n, nbk, entries);                                         \
    break;
      PWK_FOR_EACH_FFT_SIZE(PWK_CASE)
#undef PWK_CASE
      default:
        throw Error(PWK_E_UNSUPPORTED, "nz has no compiled kernel");
    }
    PWK_HIP(hipGetLastError());
  }
}

}  // namespace

void setup_basis(Context& c, int npw, const int32_t* m) {
  c.check_grid();
  PWK_REQUIRE(npw > 0 && m != nullptr, PWK_E_INVALID, "empty basis");
  const char* why = nullptr;
  const StickTables t = stick_tables(c.dims, npw, m, &why);
  PWK_REQUIRE(!why, PWK_E_UNSUPPORTED, why);
  c.npw = npw;
  c.nsticks = (int)t.pw0.size();
  c.nx1 = (int)t.x1list.size();
  c.x1_runs = t.x1_runs;
  c.x1_ra = t.x1_ra;
  c.x1_rb = t.x1_rb;
  c.pl_rows = t.pl_rows;
  c.pl_ra = t.pl_ra;
  c.pl_rb = t.pl_rb;
  c.quarter = t.quarter;
  auto up = [&](DevBuf& d, const void* h, size_t bytes) {
    d.ensure(bytes);
    PWK_HIP(hipMemcpyAsync(d.p, h, bytes, hipMemcpyHostToDevice, c.stream));
  };
  up(c.miller, m, (size_t)npw * 3 * sizeof(int32_t));
  auto table = [&](DevBuf& d, const std::vector<int32_t>& h) { up(d, h.data(), h.size() * sizeof(int32_t)); };
  table(c.g2fft, t.g2fft);
  table(c.st_pw0, t.pw0);
  table(c.st_cnt, t.cnt);
  table(c.st_n3lo, t.lo);
  table(c.x1list, t.x1list);
  table(c.pl_src, t.pl_src);
  table(c.st_off, t.st_off);
  if (c.quarter) {
    table(c.q_src, t.q_src);
    table(c.q_off, t.q_off);
  }
  c.sync();  // the host tables go out of scope here
}

void reserve_veff_slots(Context& c, int nslots) {
  c.check_grid();
  const size_t n = c.N * (size_t)std::max(1, nslots);
  c.vr64.ensure(n * sizeof(double));
  c.vr32.ensure(n * sizeof(float));
  c.vrn64.ensure(n * sizeof(double));
  c.vrn32.ensure(n * sizeof(float));
}

void set_veff_device(Context& c, const void* veff_g_dev, int slot, bool need_g) {
  c.check_grid();
  size_t n = c.N;
  PWK_REQUIRE(slot >= 0 && slot <= 1, PWK_E_INVALID, "V_eff slot must be 0 or 1");
  if (slot == 0) {
    reserve_veff_slots(c, 1);
    if (need_g) {
      c.veffg64.ensure(n * sizeof(double2));
      PWK_HIP(hipMemcpyAsync(c.veffg64.p, veff_g_dev, n * sizeof(double2), hipMemcpyDeviceToDevice, c.stream));
    }
  } else {
    PWK_REQUIRE(c.vrn64.bytes >= 2 * n * sizeof(double), PWK_E_STATE, "second V_eff slot not reserved");
  }
  c.workspace(c.work_b, n * sizeof(double2));
  launch_fft3d_copy(c, veff_g_dev, c.work_b.p, +1);
  const size_t o = (size_t)slot * n;
  k_vr_reorder<<<blocks_for(n, 256), 256, 0, c.stream>>>(c.work_b.as<double2>(), c.vr64.as<double>() + o,
                                                         c.vr32.as<float>() + o, c.vrn64.as<double>() + o,
                                                         c.vrn32.as<float>() + o, c.dims[0], c.dims[1], c.dims[2]);
  PWK_HIP(hipGetLastError());
  if (slot == 0) c.have_v = true;
}

void launch_zinv(Context& c, int nb, const void* psi, void* out, int precision, const int* list) {
  if (precision == PWK_FP64)
    zinv_t<double>(c, nb, psi, (double2*)out, list);
  else
    zinv_t<float>(c, nb, psi, (float2*)out, list);
}

void launch_hpsi(Context& c, int ik, int nb, const void* psi, void* hpsi, int precision) {
  c.check_basis();
  PWK_REQUIRE(nb > 0, PWK_E_INVALID, "nb must be positive");
  KData& kd = c.k(ik);
  PWK_REQUIRE(kd.have_kin, PWK_E_STATE, "kinetic diagonal of this k-point not set (pwk_set_kinetic)");
  if (precision != PWK_SPLIT_BF16 && c.have_v && hpsi_small_supported(c, precision, kd.nch) &&
      (kd.nch == 0 || (precision == PWK_FP64 ? kd.B64.p && kd.DBH64.p : kd.B32.p && kd.DBH32.p))) {
    const bool f64 = precision == PWK_FP64;
    launch_hpsi_small(c, nb, nb, psi, hpsi, precision, f64 ? kd.kin64.p : kd.kin32.p, kd.nch,
                      f64 ? kd.B64.p : kd.B32.p, f64 ? kd.DBH64.p : kd.DBH32.p);
    return;
  }
  if (precision == PWK_FP64) {
    hpsi_local<double>(c, kd.kin64.as<double>(), nb, nb, psi, hpsi);
  } else {
    hpsi_local<float>(c, kd.kin32.as<float>(), nb, nb, psi, hpsi);
  }
  if (kd.nch > 0) {
    // P = (D·B^H)·ψ  (nch × nb), then Hψ += B·P   (src/potential/nonlocal.rs:432-450)
    size_t es = precision == PWK_FP64 ? sizeof(double2) : sizeof(float2);
    c.workspace(c.proj, (size_t)kd.nch * nb * es);
    const void* dbh = precision == PWK_FP64 ? kd.DBH64.p : kd.DBH32.p;
    const void* bm = precision == PWK_FP64 ? kd.B64.p : kd.B32.p;
    {
      TimedScope ts(c, "hpsi_nl_project");
      launch_zgemm_mfma(c, kd.nch, nb, c.npw, dbh, kd.nch, psi, c.npw, c.proj.p, kd.nch, false, precision);
    }
    TimedScope ts(c, "hpsi_nl_expand");
    launch_zgemm_mfma(c, c.npw, nb, kd.nch, bm, c.npw, c.proj.p, kd.nch, hpsi, c.npw, true, precision);
  }
}

// H·ψ of nb bands at each of nk k-points in one pass: psi and hpsi hold nk blocks of
// npw × nb (band-major), kin nk × npw in the precision of psi, B / D·B^H nk blocks of
// npw × nch / nch × npw. The local part runs as one launch sequence over nk·nb bands,
// the projector GEMMs as strided batches.
void launch_hpsi_multi(Context& c, int nk, int nb, const void* psi, void* hpsi, int precision, const void* kin,
                       int nch, const void* B, const void* DBH, void* proj) {
  c.check_basis();
  PWK_REQUIRE(nk > 0 && nb > 0, PWK_E_INVALID, "nk and nb must be positive");
  if (precision != PWK_SPLIT_BF16 && c.have_v && hpsi_small_supported(c, precision, nch)) {
    launch_hpsi_small(c, nk * nb, nb, psi, hpsi, precision, kin, nch, B, DBH);
    return;
  }
  const long long npw = c.npw;
  if (precision == PWK_FP64)
    hpsi_local<double>(c, (const double*)kin, nk * nb, nb, psi, hpsi);
  else
    hpsi_local<float>(c, (const float*)kin, nk * nb, nb, psi, hpsi);
  if (nch > 0) {
    {
      TimedScope ts(c, "hpsi_nl_project");
      launch_zgemm_mfma_batched(c, nch, nb, (int)npw, DBH, nch, (long long)nch * npw, psi, (int)npw, npw * nb, proj,
                                nch, (long long)nch * nb, nk, false, precision);
    }
    TimedScope ts(c, "hpsi_nl_expand");
    launch_zgemm_mfma_batched(c, (int)npw, nb, nch, B, (int)npw, npw * nch, proj, nch, (long long)nch * nb, hpsi,
                              (int)npw, npw * nb, nk, true, precision);
  }
}

namespace {

size_t batch_bands(Context& c, int nent, const int32_t* ik, const int32_t* nbands) {
  PWK_REQUIRE(nent >= 1 && ik && nbands, PWK_E_INVALID, "empty or null k-point batch");
  size_t total = 0;
  for (int e = 0; e < nent; ++e) {
    PWK_REQUIRE(nbands[e] >= 1, PWK_E_INVALID, "every batch entry needs at least one band");
    const KData& kd = c.k(ik[e]);
    PWK_REQUIRE(kd.have_kin, PWK_E_STATE, "kinetic diagonal of a batch k-point not set (pwk_set_kinetic)");
    total += (size_t)nbands[e];
  }
  PWK_REQUIRE(total <= (size_t)0x7fffffff, PWK_E_INVALID, "batch too large");
  return total;
}

}  // namespace

namespace {

// The entries [e0, e1) of a batch on the stick path: one launch sequence over the bands of all of them, each
// with its entry's kinetic diagonal, and the entries' projector products as one grouped launch each.
// 27 k-points of about 24 bands (1189 plane waves, 25³) took 162 launches one entry at a time.
template <typename T, int CAP>
void hpsi_batch_sticks(Context& c, int e0, int e1, const int32_t* ik, const int32_t* nbands, const void* psi,
                       void* hpsi, int precision) {
  const bool f64 = std::is_same<T, double>::value;
  const int nch = c.k(ik[e0]).nch;
  BatchKin<CAP> kin;
  GemmGroups<CAP> project, expand;
  project.n = expand.n = e1 - e0;
  int total = 0, nmax = 0;
  for (int e = 0; e < e1 - e0; ++e) {
    const KData& kd = c.k(ik[e0 + e]);
    project.A[e] = f64 ? kd.DBH64.p : kd.DBH32.p;
    expand.A[e] = f64 ? kd.B64.p : kd.B32.p;
    project.col[e] = expand.col[e] = total;
    project.cols[e] = expand.cols[e] = nbands[e0 + e];
    total += nbands[e0 + e];
    nmax = std::max(nmax, (int)nbands[e0 + e]);
    kin.end[e] = total;
    kin.kin[e] = f64 ? kd.kin64.p : kd.kin32.p;
  }
  hpsi_local<T>(c, nullptr, total, 1, psi, hpsi, kin);
  if (nch > 0) {
    c.workspace(c.proj, (size_t)nch * total * sizeof(typename V2t<T>::t));
    {
      TimedScope ts(c, "hpsi_nl_project");
      launch_zgemm_mfma_groups(c, nch, nmax, c.npw, project, nch, psi, c.npw, c.proj.p, nch, false, precision);
    }
    TimedScope ts(c, "hpsi_nl_expand");
    launch_zgemm_mfma_groups(c, c.npw, nmax, nch, expand, c.npw, c.proj.p, nch, hpsi, c.npw, true, precision);
  }
}

// the same in the one launch of the fused small grids
template <int CAP>
void hpsi_batch_small(Context& c, int e0, int e1, const int32_t* ik, const int32_t* nbands, const void* psi,
                      void* hpsi, int precision) {
  const bool f64 = precision == PWK_FP64;
  BatchSmall<CAP> entries;
  int total = 0;
  for (int e = 0; e < e1 - e0; ++e) {
    const KData& kd = c.k(ik[e0 + e]);
    entries.end[e] = total += nbands[e0 + e];
    entries.kin[e] = f64 ? kd.kin64.p : kd.kin32.p;
    entries.B[e] = f64 ? kd.B64.p : kd.B32.p;
    entries.DBH[e] = f64 ? kd.DBH64.p : kd.DBH32.p;
  }
  launch_hpsi_small_batch(c, entries, total, psi, hpsi, precision, c.k(ik[e0]).nch);
}

template <int CAP>
void hpsi_batch_run(Context& c, int e0, int e1, const int32_t* ik, const int32_t* nbands, const void* psi, void* hpsi,
                    int precision, bool small) {
  if (small)
    hpsi_batch_small<CAP>(c, e0, e1, ik, nbands, psi, hpsi, precision);
  else if (precision == PWK_FP64)
    hpsi_batch_sticks<double, CAP>(c, e0, e1, ik, nbands, psi, hpsi, precision);
  else
    hpsi_batch_sticks<float, CAP>(c, e0, e1, ik, nbands, psi, hpsi, precision);
}

// The entries from e0 on that share their launches: as many as one launch takes, with one channel count, and
// off the small grids at most 256 MiB of sticks (a chunk of the whole-grid path; entries beyond it fill the
// chip by themselves).
int batch_run(Context& c, int nent, int e0, const int32_t* ik, const int32_t* nbands, bool small, bool f64) {
  const size_t per_band = small ? 0
                                : ((size_t)c.dims[2] * c.nsticks + (c.dims[0] == c.dims[1] ? 0 : sphere_rows_elems(c, 1))) *
                                      (f64 ? sizeof(double2) : sizeof(float2));
  const size_t most = small ? 0x7fffffff : 65535;
  const int nch = c.k(ik[e0]).nch;
  size_t total = 0;
  int e = e0;
  for (; e < nent && e - e0 < MAX_BATCH_ENTRIES; ++e) {
    const KData& kd = c.k(ik[e]);
    total += (size_t)nbands[e];
    if (total > most || total * per_band > ((size_t)256 << 20)) break;
    if (kd.nch != nch || (nch > 0 && !(f64 ? kd.B64.p && kd.DBH64.p : kd.B32.p && kd.DBH32.p))) break;
  }
  return std::max(e, e0 + 1);
}

}  // namespace

// H·ψ of a k × band batch with a band count per entry: entry e holds nbands[e] bands of k-point
// ik[e], the entries' bands packed back to back in psi and hpsi. Consecutive entries with the same channel
// count share each launch on the stick path, and are one fused launch on small cubic grids; elsewhere one H·ψ
// per entry.
void launch_hpsi_batch(Context& c, int nent, const int32_t* ik, const int32_t* nbands, const void* psi, void* hpsi,
                       int precision) {
  c.check_basis();
  batch_bands(c, nent, ik, nbands);
  const bool f64 = precision == PWK_FP64;
  const size_t es = f64 ? sizeof(double2) : sizeof(float2);
  for (int e = 0; e < nent;) {
    const int nch = c.k(ik[e]).nch;
    const bool small = precision != PWK_SPLIT_BF16 && c.have_v && hpsi_small_supported(c, precision, nch);
    const int end = small || stick_path_ok(c, f64) ? batch_run(c, nent, e, ik, nbands, small, f64) : e + 1;
    if (end == e + 1) {
      launch_hpsi(c, ik[e], nbands[e], psi, hpsi, precision);
    } else if (end - e <= FEW_BATCH_ENTRIES) {
      hpsi_batch_run<FEW_BATCH_ENTRIES>(c, e, end, ik, nbands, psi, hpsi, precision, small);
    } else {
      hpsi_batch_run<MAX_BATCH_ENTRIES>(c, e, end, ik, nbands, psi, hpsi, precision, small);
    }
    for (; e < end; ++e) {
      psi = (const char*)psi + (size_t)nbands[e] * c.npw * es;
      hpsi = (char*)hpsi + (size_t)nbands[e] * c.npw * es;
    }
  }
}

// ρ += Σ_b fw_b |ψ_b(r)|² over every band of a k × band batch (fw per band, occupation × k
// weight, entries back to back): the density does not depend on k, so all bands go through one
// density launch.
void launch_density_batch(Context& c, int nent, const int32_t* ik, const int32_t* nbands, const void* psi,
                          const double* fw_host, void* rho, int precision) {
  c.check_basis();
  const size_t total = batch_bands(c, nent, ik, nbands);
  launch_density(c, (int)total, psi, fw_host, rho, precision);
}

void launch_density(Context& c, int nb, const void* psi, const double* fw_host, void* rho, int precision,
                    bool overwrite) {
  c.check_basis();
  PWK_REQUIRE(nb > 0, PWK_E_INVALID, "nb must be positive");
  const int dprec = precision == PWK_FP64 ? PWK_FP64 : PWK_FP32;
  if (density_small_supported(c, dprec)) {
    c.workspace(c.work_b, (size_t)nb * sizeof(double));
    PWK_HIP(hipMemcpyAsync(c.work_b.p, fw_host, (size_t)nb * sizeof(double), hipMemcpyHostToDevice, c.stream));
    launch_density_small(c, nb, psi, c.work_b.as<double>(), rho, dprec, overwrite);
    return;
  }
  if (stick_path_ok(c, dprec == PWK_FP64)) {
    launch_density_sticks(c, nb, psi, fw_host, rho, dprec, overwrite);
    return;
  }
  if (overwrite) PWK_HIP(hipMemsetAsync(rho, 0, c.N * sizeof(double), c.stream));
  if (precision == PWK_FP64)
    density_fullgrid<double>(c, nb, psi, fw_host, rho);
  else
    density_fullgrid<float>(c, nb, psi, fw_host, rho);
}

}  // namespace pwk
