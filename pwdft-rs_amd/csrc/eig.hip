// Batched dense Hermitian eigensolver, FP64, one workgroup per matrix: the
// lowest nb eigenpairs of each n×n matrix, eigenvalues ascending, as
// diagonalize_lowest (src/eigensolver/dense.rs:87-98), which keeps the first
// n_bands pairs of a full self-adjoint decomposition.
//
//   1. Householder reduction to Hermitian tridiagonal form; the reflectors are
//      kept below the diagonal of the (overwritten) input, the trailing
//      rank-2 updates are spread over the workgroup.
//   2. A diagonal unitary D makes the sub-diagonal real: T = D·T_r·D^H.
//   3. The nb lowest eigenvalues of T_r by Sturm-count multisection, lane
//      groups of one wavefront per eigenvalue, one probe point per lane.
//   4. Their eigenvectors by inverse iteration (tridiagonal LU with partial
//      pivoting, one lane per vector, three solves from a fixed pseudo-random
//      start; factors in LDS when they fit), then modified Gram-Schmidt inside
//      clusters of close eigenvalues.
//   5. Back-transformation V = Q·D·Z through the reflectors in reverse order.
// Matrices of at most 32 rows (the Rayleigh-Ritz problems of the filtered
// eigensolver) take a different route: a one-wavefront cyclic Jacobi solver
// with the matrix and the eigenvectors in LDS (round-robin ordering, n/2
// disjoint complex rotations per round, at most 30 sweeps).
// Every loop has a fixed bound; nothing waits on data.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "jacobi.hpp"

namespace pwk {

namespace {

// Two workgroup shapes: 16 waves (memory-level parallelism for the latency-bound passes
// of larger matrices) and one wave for matrices of at most 64 rows, where barriers
// dominate and a single wave needs none of its reductions in LDS.
constexpr int EIG_NT = 1024;
constexpr int EIG_WAVES = EIG_NT / 64;  // LDS is sized for the larger shape

__host__ __device__ inline size_t eig_stride(int n, int nb) {
  // ecx (2n) | dph (2n) | z (n·nb) | LU factors (5·n·nb)
  size_t s = 4 * (size_t)n + 6 * (size_t)n * nb;
  return (s + 1) & ~(size_t)1;
}

template <int NT>
__device__ double block_sum(double v, double* red) {
  constexpr int EIG_WAVES = NT / 64;
  const int t = threadIdx.x;
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if (NT == 64) return __shfl(v, 0, 64);
  __syncthreads();
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  if (t == 0) {
    double s = 0.0;
    for (int w = 0; w < EIG_WAVES; ++w) s += red[w];
    red[EIG_WAVES] = s;
  }
  __syncthreads();
  return red[EIG_WAVES];
}

// 1/x to the last bit or two: the hardware estimate and two Newton steps, a third of the latency of a
// division (the Sturm recurrences and the LU sweeps are chains of them)
__device__ __forceinline__ double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

// Number of eigenvalues of the real symmetric tridiagonal (d, e) below x.
__device__ int sturm_count(int n, const double* d, const double* e2, double x, double pivmin) {
  int cnt = 0;
  double q = d[0] - x;
  if (fabs(q) < pivmin) q = -pivmin;
  cnt += q < 0.0;
  double dn = n > 1 ? d[1] - x : 0.0, en = e2[0];
  for (int i = 1; i < n; ++i) {
    const double di = dn, ei = en;
    dn = d[min(i + 1, n - 1)] - x;  // the next entries, in flight
    en = e2[i];
    q = fma(-ei, recip(q), di);
    if (fabs(q) < pivmin) q = -pivmin;
    cnt += q < 0.0;
  }
  return cnt;
}

// Deterministic start vector entry in [-1, 1).
__device__ double start_entry(int i, int j) {
  uint32_t h = (uint32_t)i * 0x9E3779B1u ^ ((uint32_t)j + 0x7F4A7C15u) * 0x85EBCA77u;
  h ^= h >> 15;
  h *= 0x2C1B3C6Du;
  h ^= h >> 12;
  h *= 0x297A2D39u;
  h ^= h >> 15;
  return (double)h * (2.0 / 4294967296.0) - 1.0;
}

// Steps 2-4 on the tridiagonal form (d in LDS, the complex sub-diagonal in ecx): eigenvalues to lam,
// the phases to dph, eigenvectors of the real tridiagonal to Z. lu holds 6·n·nb doubles (Z first).
template <int NT>
__device__ __forceinline__ void tri_pairs(int n, int nb, double* d, double* e, double* e2, double* lam, double* red, double* s_bounds,
                          const double2* ecx, double2* dph, double* Z) {
  constexpr int EIG_NT = NT;
  constexpr int EIG_WAVES = NT / 64;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  double* U0 = Z + (size_t)n * nb;                     // LU factors, interleaved by vector like Z
  double* U1 = U0 + (size_t)n * nb;
  double* U2 = U1 + (size_t)n * nb;
  double* ML = U2 + (size_t)n * nb;
  double* PV = ML + (size_t)n * nb;

  // ---- 2. real sub-diagonal, phases, Gershgorin bounds -------------------------------
  // moduli and unit phases by all threads (the unit phases into Z), then the running product of the
  // phases by one, which is all that is serial
  double2* unit = reinterpret_cast<double2*>(Z);
  for (int k = t; k < n; k += EIG_NT) {
    double ab = 0.0;
    double2 u = make_double2(1.0, 0.0);
    if (k + 1 < n) {
      const double2 ek = ecx[k];
      ab = sqrt(ek.x * ek.x + ek.y * ek.y);
      if (ab > 0.0) u = make_double2(ek.x / ab, ek.y / ab);
    }
    e[k] = ab;
    e2[k] = ab * ab;
    unit[k] = u;
  }
  __syncthreads();
  // (fmin and fmax leave NaNs out: the bounds are NaN, and with them every eigenvalue, if all entries are)
  double lo = __builtin_nan(""), hi = lo;
  for (int k = t; k < n; k += EIG_NT) {
    const double r = e[k] + (k > 0 ? e[k - 1] : 0.0);
    lo = fmin(lo, d[k] - r);
    hi = fmax(hi, d[k] + r);
  }
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_down(lo, off, 64));
    hi = fmax(hi, __shfl_down(hi, off, 64));
  }
  if (lane == 0) red[wave] = lo;
  __syncthreads();
  if (t == 0) {
    for (int w = 0; w < EIG_WAVES; ++w) lo = fmin(lo, red[w]);
    s_bounds[0] = lo;
  }
  __syncthreads();
  if (lane == 0) red[wave] = hi;
  __syncthreads();
  if (t == 0) {
    for (int w = 0; w < EIG_WAVES; ++w) hi = fmax(hi, red[w]);
    const double tnorm = fmax(fabs(lo), fabs(hi));
    const double pad = 2.220446049250313e-16 * tnorm * (double)n + 1e-300;
    s_bounds[0] = lo - pad;
    s_bounds[1] = hi + pad;
    s_bounds[2] = fmax(tnorm, 1e-300);
  }
  if (wave == EIG_WAVES - 1 && lane == 0) {
    double2 ph = make_double2(1.0, 0.0), u = unit[0];
    dph[0] = ph;
    for (int k = 0; k + 1 < n; ++k) {
      const double2 un = unit[k + 1];  // the next factor, in flight
      ph = make_double2(ph.x * u.x - ph.y * u.y, ph.x * u.y + ph.y * u.x);
      dph[k + 1] = ph;
      u = un;
    }
  }
  __syncthreads();
  const double tnorm = s_bounds[2];
  const double pivmin = 1e-290 * fmax(1.0, tnorm * tnorm);

  // ---- 3. eigenvalues by multisection: groups of G lanes per eigenvalue, each lane one
  // probe; the groups of all waves cover as many eigenvalues at once as there are groups
  {
    int gpw = 1;  // groups per wave: the smallest power of two with NW·gpw >= nb (at most 64)
    while (gpw < 64 && gpw * EIG_WAVES < nb) gpw <<= 1;
    const int G = 64 / gpw, g = lane / G, sub = lane % G;
    const unsigned long long gmask = G == 64 ? ~0ull : ((1ull << G) - 1ull);
    const int per_round = EIG_WAVES * gpw;
    for (int j0 = 0; j0 < nb; j0 += per_round) {
      const int j = j0 + wave * gpw + g;
      const bool active = j < nb;
      double a = s_bounds[0], bb = s_bounds[1];
      bool done = !active;
      for (int it = 0; it < 64; ++it) {
        if (__ballot(!done) == 0ull) break;  // wave-uniform exit
        const double x = a + (bb - a) * ((double)(sub + 1) / (double)(G + 1));
        const int cnt = done ? 0 : sturm_count(n, d, e2, x, pivmin);
        const unsigned long long le = (__ballot(cnt <= j) >> (g * G)) & gmask;
        // first probe of the group above the j-th eigenvalue
        const int k = (~le & gmask) == 0ull ? G : __builtin_ctzll(~le & gmask);
        const double na = __shfl(x, g * G + (k > 0 ? k - 1 : 0), 64);
        const double nbv = __shfl(x, g * G + (k < G ? k : G - 1), 64);
        if (!done) {
          const double a2 = k > 0 ? na : a, b2 = k < G ? nbv : bb;
          // converged to the precision the tridiagonal form carries: eps relative to the
          // eigenvalue or eps·|T| absolute, whichever is larger
          done = (a2 == a && b2 == bb) ||
                 b2 - a2 <= 4.440892098500626e-16 * fmax(fmax(fabs(a2), fabs(b2)), tnorm);
          a = a2;
          bb = b2;
        }
      }
      if (active && sub == 0) lam[j] = 0.5 * (a + bb);
    }
  }
  __syncthreads();

  // ---- 4. inverse iteration, one lane per eigenvector ------------------------------------
  const double tiny = 2.220446049250313e-16 * tnorm;
  for (int j = t; j < nb; j += EIG_NT) {
    const double lj = lam[j];
    // LU of T_r - lj I with row interchanges (upper factor has two super-diagonals)
    // U0 holds the pivots' reciprocals; each loop loads the next step's entries before it uses this one's
    double cd = d[0] - lj, cs = n > 1 ? e[0] : 0.0;
    double sub = cs, an = n > 1 ? d[1] - lj : 0.0, bn = n > 2 ? e[1] : 0.0;
    for (int i = 0; i + 1 < n; ++i) {
      const double dn2 = d[min(i + 2, n - 1)], en1 = e[min(i + 1, n - 1)], en2 = e[min(i + 2, n - 1)];
      const bool swap = !(fabs(cd) >= fabs(sub));
      if (!swap && fabs(cd) < tiny) cd = cd < 0.0 ? -tiny : tiny;
      const double ru = recip(swap ? sub : cd), ml = (swap ? cd : sub) * ru;
      const size_t o = (size_t)i * nb + j;
      U0[o] = ru;
      U1[o] = swap ? an : cs;
      U2[o] = swap ? bn : 0.0;
      ML[o] = ml;
      PV[o] = swap ? 1.0 : 0.0;
      const double cd2 = swap ? cs - ml * an : an - ml * cs;
      cs = swap ? -ml * bn : bn;
      cd = cd2;
      sub = en1;
      an = dn2 - lj;
      bn = i + 3 < n ? en2 : 0.0;
    }
    if (fabs(cd) < tiny) cd = cd < 0.0 ? -tiny : tiny;
    {
      const size_t o = (size_t)(n - 1) * nb + j;
      U0[o] = recip(cd);
      U1[o] = 0.0;
      U2[o] = 0.0;
      ML[o] = 0.0;
      PV[o] = 0.0;
    }
    // start vector
    double nrm = 0.0;
    for (int i = 0; i < n; ++i) {
      const double s = start_entry(i, j);
      Z[(size_t)i * nb + j] = s;
      nrm += s * s;
    }
    for (int sweep = 0; sweep < 3; ++sweep) {
      const double sc = 1.0 / sqrt(nrm);
      // forward: row interchanges and multipliers
      double carry = Z[j] * sc;
      double pv = PV[j], ml = ML[j], zn = Z[(size_t)min(1, n - 1) * nb + j];
      for (int i = 0; i + 1 < n; ++i) {
        const size_t o = (size_t)i * nb + j, o1 = o + nb, o2 = (size_t)min(i + 2, n - 1) * nb + j;
        const double pv1 = PV[o1], ml1 = ML[o1], zn1 = Z[o2];
        const double yn = zn * sc;
        const bool swap = pv != 0.0;
        const double yi = swap ? yn : carry;
        carry = (swap ? carry : yn) - ml * yi;
        Z[o] = yi;
        pv = pv1;
        ml = ml1;
        zn = zn1;
      }
      Z[(size_t)(n - 1) * nb + j] = carry;
      // backward substitution
      double x2 = 0.0, x1 = 0.0;
      nrm = 0.0;
      size_t ol = (size_t)(n - 1) * nb + j;
      double zi = carry, r0 = U0[ol], r1 = U1[ol], r2 = U2[ol];
      for (int i = n - 1; i >= 0; --i) {
        const size_t o = (size_t)i * nb + j, om = (size_t)max(i - 1, 0) * nb + j;
        const double zm = Z[om], m0 = U0[om], m1 = U1[om], m2 = U2[om];
        const double xi = (zi - r1 * x1 - r2 * x2) * r0;
        Z[o] = xi;
        nrm += xi * xi;
        x2 = x1;
        x1 = xi;
        zi = zm;
        r0 = m0;
        r1 = m1;
        r2 = m2;
      }
      if (!(nrm > 0.0) || !isfinite(nrm)) nrm = 1.0;
    }
    const double sc = 1.0 / sqrt(nrm);
    for (int i = 0; i < n; ++i) Z[(size_t)i * nb + j] *= sc;
  }
  __syncthreads();
  // modified Gram-Schmidt inside clusters (gap below 1e-3·|T|)
  const double ortol = 1e-3 * tnorm;
  for (int j = 1; j < nb; ++j) {
    int first = j;
    while (first > 0 && lam[first] - lam[first - 1] <= ortol) --first;
    if (first == j) continue;
    for (int i = first; i < j; ++i) {
      double part = 0.0;
      for (int r = t; r < n; r += EIG_NT) part += Z[(size_t)r * nb + i] * Z[(size_t)r * nb + j];
      const double dp = block_sum<NT>(part, red);
      for (int r = t; r < n; r += EIG_NT) Z[(size_t)r * nb + j] -= dp * Z[(size_t)r * nb + i];
      __syncthreads();
    }
    double part = 0.0;
    for (int r = t; r < n; r += EIG_NT) part += Z[(size_t)r * nb + j] * Z[(size_t)r * nb + j];
    const double nn = block_sum<NT>(part, red);
    const double sc = nn > 0.0 ? 1.0 / sqrt(nn) : 0.0;
    for (int r = t; r < n; r += EIG_NT) Z[(size_t)r * nb + j] *= sc;
    __syncthreads();
  }
}

template <int NT>
__global__ void __launch_bounds__(NT) k_heev(int n, int nb, int a_in_lds, int lu_in_lds, double2* __restrict__ Hb,
                                             double* __restrict__ work, double* __restrict__ w_out,
                                             double2* __restrict__ V_out, int* __restrict__ status) {
  constexpr int EIG_NT = NT;
  constexpr int EIG_WAVES = NT / 64;
  extern __shared__ unsigned char smem[];
  double2* v = reinterpret_cast<double2*>(smem);      // n
  double2* wv = v + n;                                // n
  double* d = reinterpret_cast<double*>(wv + n);      // n: diagonal of T_r
  double* e = d + n;                                  // n: sub-diagonal of T_r
  double* e2 = e + n;                                 // n: e²
  double* lam = e2 + n;                               // nb: eigenvalues
  double* red = lam + nb;                             // EIG_WAVES + 2
  // EIG_WAVES × 64 matvec partials, 16-byte aligned
  const size_t pp_off = ((size_t)(reinterpret_cast<unsigned char*>(red + EIG_WAVES + 2) - smem) + 15) & ~(size_t)15;
  double2* pp = reinterpret_cast<double2*>(smem + pp_off);
  double2* lds_a = pp + 16 * 64;                                          // n·n when a_in_lds
  double* lds_lu = reinterpret_cast<double*>(lds_a + (a_in_lds ? (size_t)n * n : 0));  // 6·n·nb when lu_in_lds
  __shared__ double s_bounds[3];

  const int b = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  double2* A = Hb + (size_t)b * n * n;
  if (a_in_lds) {  // small matrices live in LDS for the whole solve (the input is not written back)
    for (int i = t; i < n * n; i += EIG_NT) lds_a[i] = A[i];
    __syncthreads();
    A = lds_a;
  }
  double* base = work + (size_t)b * eig_stride(n, nb);
  double2* ecx = reinterpret_cast<double2*>(base);    // n
  double2* dph = ecx + n;                              // n
  double* Z = lu_in_lds ? lds_lu : reinterpret_cast<double*>(dph + n);  // Z[i*nb + j]

  // ---- 1. Householder tridiagonalisation --------------------------------------------
  for (int k = 0; k + 2 < n; ++k) {
    const int m = n - k - 1;
    double2* col = A + (size_t)k * n + k + 1;
    double part = 0.0;
    for (int i = t; i < m; i += EIG_NT) part += col[i].x * col[i].x + col[i].y * col[i].y;
    const double xn = sqrt(block_sum<NT>(part, red));
    if (xn == 0.0) {
      for (int i = t; i < m; i += EIG_NT) col[i] = make_double2(0.0, 0.0);  // identity reflector
      if (t == 0) ecx[k] = make_double2(0.0, 0.0);
      __syncthreads();
      continue;
    }
    const double2 x0 = col[0];
    const double ax0 = sqrt(x0.x * x0.x + x0.y * x0.y);
    const double2 ph = ax0 > 0.0 ? make_double2(x0.x / ax0, x0.y / ax0) : make_double2(1.0, 0.0);
    const double2 alpha = make_double2(-ph.x * xn, -ph.y * xn);
    // v = (x - alpha e1) / |x - alpha e1|;  |x - alpha e1|² = 2(|x|² + |x||x0|)
    const double vn = sqrt(2.0 * (xn * xn + xn * ax0));
    for (int i = t; i < m; i += EIG_NT) {
      double2 x = col[i];
      if (i == 0) {
        x.x -= alpha.x;
        x.y -= alpha.y;
      }
      v[i] = make_double2(x.x / vn, x.y / vn);
    }
    __syncthreads();
    // p = A_sub v: rows in chunks of 64 lanes, the columns split over the waves, then a
    // fixed-order sum of the per-wave partials
    for (int i0 = 0; i0 < m; i0 += 64) {
      const int i = i0 + lane;
      double pr = 0.0, pi = 0.0;
      if (i < m) {
        const double2* arow = A + (size_t)(k + 1) * n + k + 1 + i;
        for (int j = wave; j < m; j += EIG_WAVES) {
          const double2 a = arow[(size_t)j * n];
          const double2 vj = v[j];
          pr += a.x * vj.x - a.y * vj.y;
          pi += a.x * vj.y + a.y * vj.x;
        }
      }
      pp[wave * 64 + lane] = make_double2(pr, pi);
      __syncthreads();
      if (wave == 0 && i < m) {
        double sr = 0.0, si = 0.0;
        for (int w = 0; w < EIG_WAVES; ++w) {
          sr += pp[w * 64 + lane].x;
          si += pp[w * 64 + lane].y;
        }
        wv[i] = make_double2(sr, si);
      }
      __syncthreads();
    }
    part = 0.0;
    for (int i = t; i < m; i += EIG_NT) part += v[i].x * wv[i].x + v[i].y * wv[i].y;  // v^H p (real)
    const double K = block_sum<NT>(part, red);
    for (int i = t; i < m; i += EIG_NT) {
      wv[i].x -= K * v[i].x;
      wv[i].y -= K * v[i].y;
    }
    __syncthreads();
    // A_sub -= 2 (v w^H + w v^H)
    for (int idx = t; idx < m * m; idx += EIG_NT) {
      const int i = idx % m, j = idx / m;
      const double2 vi = v[i], wi = wv[i], vj = v[j], wj = wv[j];
      const double re = (vi.x * wj.x + vi.y * wj.y) + (wi.x * vj.x + wi.y * vj.y);
      const double im = (vi.y * wj.x - vi.x * wj.y) + (wi.y * vj.x - wi.x * vj.y);
      double2* a = &A[(size_t)(k + 1 + j) * n + k + 1 + i];
      a->x -= 2.0 * re;
      a->y -= 2.0 * im;
    }
    __syncthreads();
    for (int i = t; i < m; i += EIG_NT) col[i] = v[i];
    if (t == 0) ecx[k] = alpha;
    __syncthreads();
  }
  if (t == 0 && n >= 2) ecx[n - 2] = A[(size_t)(n - 2) * n + n - 1];
  for (int i = t; i < n; i += EIG_NT) d[i] = A[(size_t)i * n + i].x;
  __syncthreads();

  tri_pairs<NT>(n, nb, d, e, e2, lam, red, s_bounds, ecx, dph, Z);

  // ---- 5. V = Q·D·Z --------------------------------------------------------------------
  double2* V = V_out + (size_t)b * n * nb;
  for (int idx = t; idx < n * nb; idx += EIG_NT) {
    const int r = idx % n, jj = idx / n;
    const double zr = Z[(size_t)r * nb + jj];
    const double2 p = dph[r];
    V[(size_t)jj * n + r] = make_double2(p.x * zr, p.y * zr);
  }
  for (int jj = t; jj < nb; jj += EIG_NT) w_out[(size_t)b * nb + jj] = lam[jj];
  __syncthreads();
  double2* sv = wv;  // nb ≤ n projections
  for (int k = n - 3; k >= 0; --k) {
    const int m = n - k - 1;
    const double2* vk = A + (size_t)k * n + k + 1;
    // one wave per vector, lanes over the reflector
    for (int jj = wave; jj < nb; jj += EIG_WAVES) {
      double sr = 0.0, si = 0.0;
      const double2* x = V + (size_t)jj * n + k + 1;
      for (int i = lane; i < m; i += 64) {
        const double2 a = vk[i], xi = x[i];
        sr += a.x * xi.x + a.y * xi.y;  // conj(v)·x
        si += a.x * xi.y - a.y * xi.x;
      }
      for (int off = 32; off > 0; off >>= 1) {
        sr += __shfl_down(sr, off, 64);
        si += __shfl_down(si, off, 64);
      }
      if (lane == 0) sv[jj] = make_double2(sr, si);
    }
    __syncthreads();
    for (int idx = t; idx < m * nb; idx += EIG_NT) {
      const int i = idx % m, jj = idx / m;
      const double2 a = vk[i], s = sv[jj];
      double2* x = &V[(size_t)jj * n + k + 1 + i];
      x->x -= 2.0 * (a.x * s.x - a.y * s.y);
      x->y -= 2.0 * (a.x * s.y + a.y * s.x);
    }
    __syncthreads();
  }
  if (t == 0 && status) status[b] = 0;
}

// ---- matrices of 65 to 256 rows ------------------------------------------------------------------
// The same steps with the Householder reduction arranged around one pass over the matrix per reflector:
//  - wave w owns the columns j ≡ w mod 8 and a lane the rows lane + 64r of them for the whole reduction, so
//    the matrix (in L2) is read and written by the threads that own it and needs no barrier;
//  - pass k applies the rank-2 update of reflector k - 1 to the columns behind k and multiplies the updated
//    entries with v_k on the way (rows in registers, the column factors broadcast from LDS); the eight waves
//    partial products go through LDS, and column k + 1 is left there for the next reflector;
//  - one wave then forms w and the next reflector in its registers (wave sums by lane moves; all waves doing so
//    redundantly took four times as long, they share the vector units) while the others' first loads are
//    in flight: three barriers per reflector.
// Back-transformation: one wave per vector, its rows in registers, no barrier.
// Bound: the chain of reflectors, each with a pass of about 13k cycles of issue by two waves per SIMD (the
// loads and stores hide behind it). 8 matrices of 169 rows, 8 pairs: 5.0 ms in the form above (15 barriers and
// an integer division per entry and reflector), 2.5 with the column factors read from LDS per column, 1.9 by
// lane moves; 4 or 16 waves per matrix, or more columns in flight, took longer. The form above is slower over
// the whole range, also where the matrix fits the LDS (up to 90 rows): 65 rows 0.78 -> 0.45 ms, 90 rows 1.58 ->
// 0.65, 128 rows 2.56 -> 1.00, 256 rows 14.8 -> 3.8 (8 pairs, 1 to 64 matrices), 300 matrices of 65 rows
// 1.56 -> 0.65, of 144 rows 6.9 -> 3.2.
constexpr int ROW_NT = 512, ROW_WAVES = 8, ROW_GROUPS = 2;

template <int CTRL>
__device__ __forceinline__ double dpp_add(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
  return x + __hiloint2double(hi, lo);
}
// the sum over a wave, in every lane: within rows of 16 lanes by lane moves, then the four rows
__device__ __forceinline__ double wave_sum(double x) {
  x = dpp_add<0xB1>(x);   // quad_perm [1,0,3,2]
  x = dpp_add<0x4E>(x);   // quad_perm [2,3,0,1]
  x = dpp_add<0x141>(x);  // row_half_mirror
  x = dpp_add<0x140>(x);  // row_mirror
  double s = 0.0;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    s += __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), 16 * r),
                          __builtin_amdgcn_readlane(__double2loint(x), 16 * r));
  return s;
}

__host__ __device__ inline size_t rows_lds_vectors(int n) { return (size_t)(4 + ROW_GROUPS) * n * sizeof(double2); }
// LDS of k_heev_rows: vectors v, w, x, column, p sums (complex) | d, e, e2, lam, red | the waves' partial
// products, later the tridiagonal's vectors and LU factors when they fit
inline size_t rows_lds_head(int n, int nb) {
  return rows_lds_vectors(n) + ((((size_t)3 * n + nb + 32) * sizeof(double) + 15) & ~(size_t)15);
}

constexpr unsigned kNoRow = 0x80000000u;  // an offset past every matrix of 256 rows
typedef unsigned u4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ double2 buf_load(__amdgpu_buffer_rsrc_t r, unsigned off, int soff) {
  const u4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0);
  return make_double2(__hiloint2double((int)v.y, (int)v.x), __hiloint2double((int)v.w, (int)v.z));
}
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t r, unsigned off, int soff, double2 x) {
  u4 v;
  v.x = (unsigned)__double2loint(x.x);
  v.y = (unsigned)__double2hiint(x.x);
  v.z = (unsigned)__double2loint(x.y);
  v.w = (unsigned)__double2hiint(x.y);
  __builtin_amdgcn_raw_buffer_store_b128(v, r, off, soff, 0);
}

// the value of lane l (uniform) in every lane
__device__ __forceinline__ double2 lane_of(const double2& x, int l) {
  return make_double2(__hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x.x), l),
                                       __builtin_amdgcn_readlane(__double2loint(x.x), l)),
                      __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x.y), l),
                                       __builtin_amdgcn_readlane(__double2loint(x.y), l)));
}

// z -= 2(v_i conj(w_j) + w_i conj(v_j)), the factor 2 in w
__device__ __forceinline__ void rank2(double2& z, const double2& vi, const double2& wi, const double2& vj,
                                      const double2& wj) {
  z.x = fma(-vi.x, wj.x, fma(-vi.y, wj.y, fma(-wi.x, vj.x, fma(-wi.y, vj.y, z.x))));
  z.y = fma(-vi.y, wj.x, fma(vi.x, wj.y, fma(-wi.y, vj.x, fma(wi.x, vj.y, z.y))));
}

// R = rows per lane
template <int R>
__global__ void __launch_bounds__(ROW_NT) k_heev_rows(int n, int nb, int lu_in_lds, double2* __restrict__ Hb,
                                                      double* __restrict__ work, double* __restrict__ w_out,
                                                      double2* __restrict__ V_out, int* __restrict__ status) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  double2* sv = reinterpret_cast<double2*>(smem);  // reflector k - 1, its w, reflector k
  double2* sw = sv + n;
  double2* sx = sw + n;
  double2* scol = sx + n;  // column k, reflectors up to k - 2 applied
  double2* psum = scol + n;  // A·v of reflector k - 1, two partial sums
  double* d = reinterpret_cast<double*>(psum + ROW_GROUPS * n);
  double* e = d + n;
  double* e2 = e + n;
  double* lam = e2 + n;
  double* red = lam + nb;
  double2* part = reinterpret_cast<double2*>(
      smem + (((size_t)(reinterpret_cast<unsigned char*>(red + 32) - smem) + 15) & ~(size_t)15));  // [wave][n]
  __shared__ double s_bounds[3];
  const int b = blockIdx.x, t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // uniform: column addresses stay in scalar registers
  double2* A = Hb + (size_t)b * n * n;
  double* base = work + (size_t)b * eig_stride(n, nb);
  double2* ecx = reinterpret_cast<double2*>(base);
  double2* dph = ecx + n;
  double* Z = lu_in_lds ? reinterpret_cast<double*>(part) : reinterpret_cast<double*>(dph + n);

  const __amdgpu_buffer_rsrc_t Ar = __builtin_amdgcn_make_buffer_rsrc(A, 0, n * n * 16, 0x00027000);
  double2 x[R];  // wave 0: its rows of the last reflector
#pragma unroll
  for (int r = 0; r < R; ++r) x[r] = make_double2(0.0, 0.0);
  for (int i = t; i < n; i += ROW_NT) scol[i] = A[i];
  for (int i = t; i < ROW_GROUPS * n; i += ROW_NT) psum[i] = make_double2(0.0, 0.0);
  __syncthreads();
  for (int k = 0; k + 1 < n; ++k) {
    const int j0 = k + 1 + ((wave - (k + 1)) & (ROW_WAVES - 1));  // the wave's first column behind k
    // A column's rows through buffer accesses: rows that are not behind k get an offset past the buffer, so
    // their loads give zero and their stores are dropped without a branch, which would hide from the
    // compiler how many accesses are in flight and make every wait one for all of them.
    unsigned row[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + 64 * r;
      row[r] = i > k && i < n ? (unsigned)i * 16u : kNoRow;
    }
    auto load = [&](double2(&a)[R], int j) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (64 * r + 63 > k) a[r] = buf_load(Ar, j < n ? row[r] : kNoRow, min(j, n - 1) * n * 16);
    };
    double2 a0[R], a1[R];  // two columns in flight
    load(a0, j0);  // in flight during the vector phase
    if (wave == 0) {
      // w of reflector k - 1, column k, reflector k
      double2 p[R], v[R], w[R];
      double kk = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int i = lane + 64 * r;
        v[r] = x[r];
        p[r] = make_double2(0.0, 0.0);
        x[r] = i < n && i >= k ? scol[i] : make_double2(0.0, 0.0);
#pragma unroll
        for (int g = 0; g < ROW_GROUPS; ++g) {
          const double2 y = psum[g * n + min(i, n - 1)];
          p[r].x += y.x;
          p[r].y += y.y;
        }
        kk += v[r].x * p[r].x + v[r].y * p[r].y;  // v^H p (real); v is zero past the matrix
      }
      kk = wave_sum(kk);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        w[r] = make_double2(2.0 * (p[r].x - kk * v[r].x), 2.0 * (p[r].y - kk * v[r].y));
        if (lane + 64 * r < n) {
          sv[lane + 64 * r] = v[r];
          sw[lane + 64 * r] = w[r];
        }
      }
      const double2 vk = sv[k], wk = sw[k];  // (the wave's own stores)
      double xx = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int i = lane + 64 * r;
        rank2(x[r], v[r], w[r], vk, wk);
        if (i > k && i < n) xx += x[r].x * x[r].x + x[r].y * x[r].y;
        if (i == k) d[k] = x[r].x;
        if (i == k + 1) sx[i] = x[r];
      }
      xx = wave_sum(xx);
      const double2 x0 = sx[k + 1];
      // the last column has no reflector: its sub-diagonal entry stays as it is
      const bool last = k + 2 >= n;
      const double xn = sqrt(xx), ax0 = sqrt(x0.x * x0.x + x0.y * x0.y);
      const double2 ph = ax0 > 0.0 ? make_double2(x0.x / ax0, x0.y / ax0) : make_double2(1.0, 0.0);
      const double2 alpha = make_double2(-ph.x * xn, -ph.y * xn);
      // v = (x - alpha e1) / |x - alpha e1|;  |x - alpha e1|² = 2(|x|² + |x||x0|)
      const double vn = sqrt(2.0 * (xn * xn + xn * ax0));
      // a column without weight takes no reflector; one with a NaN or an infinity does, and spreads it over
      // the matrix as the general form does
      const bool reflect = !last && xn != 0.0;
      const double rv = reflect ? 1.0 / vn : 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int i = lane + 64 * r;
        double2 y = make_double2(0.0, 0.0);
        if (i > k && i < n && reflect) {
          y = x[r];
          if (i == k + 1) {
            y.x -= alpha.x;
            y.y -= alpha.y;
          }
          y.x *= rv;
          y.y *= rv;
        }
        x[r] = y;
        if (i < n) {
          sx[i] = y;
          if (i > k && !last) A[(size_t)k * n + i] = y;  // the reflector, for the back-transformation
        }
      }
      if (lane == 0) ecx[k] = last ? x0 : alpha;
    }
    __syncthreads();
    // the column factors of this wave's columns, a column per lane (32 at most): a lane move each per use
    // instead of an LDS read with its latency
    double2 cv = make_double2(0.0, 0.0), cw = cv, cx = cv;
    {
      const int j = j0 + ROW_WAVES * lane;
      if (j < n) {
        cv = sv[j];
        cw = sw[j];
        cx = sx[j];
      }
    }
    double2 vv[R], ww[R];  // of the rows behind k
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + 64 * r;
      const double2 z = make_double2(0.0, 0.0);
      vv[r] = i > k && i < n ? sv[i] : z;
      ww[r] = i > k && i < n ? sw[i] : z;
    }
    // pass k: the next columns' loads go out before this batch's stores
    double2 q[R];
#pragma unroll
    for (int r = 0; r < R; ++r) q[r] = make_double2(0.0, 0.0);
    // RLO: the first row group with rows behind k (the groups before it are not touched)
    auto run = [&](auto rlo) {
      constexpr int RLO = decltype(rlo)::value;
      auto next = [&](double2(&a)[R], int j) {
#pragma unroll
        for (int r = RLO; r < R; ++r) a[r] = buf_load(Ar, j < n ? row[r] : kNoRow, min(j, n - 1) * n * 16);
      };
      auto pass = [&](double2(&a)[R], int j) {
        const int jc = min(j, n - 1), l = min((j - j0) / ROW_WAVES, 63);
        const double2 vj = lane_of(cv, l), wj = lane_of(cw, l), xj = lane_of(cx, l);
#pragma unroll
        for (int r = RLO; r < R; ++r) {
          double2& z = a[r];
          rank2(z, vv[r], ww[r], vj, wj);
          buf_store(Ar, j < n ? row[r] : kNoRow, jc * n * 16, z);
          q[r].x = fma(z.x, xj.x, fma(-z.y, xj.y, q[r].x));
          q[r].y = fma(z.x, xj.y, fma(z.y, xj.x, q[r].y));
        }
        if (j == k + 1) {
#pragma unroll
          for (int r = RLO; r < R; ++r)
            if (lane + 64 * r < n) scol[lane + 64 * r] = a[r];
        }
      };
      constexpr int S = ROW_WAVES;
      for (int jb = j0; jb < n; jb += 2 * S) {
        next(a1, jb + S);
        pass(a0, jb);
        next(a0, jb + 2 * S);
        pass(a1, jb + S);
      }
    };
    const int rlo = (k + 1) >> 6;
    if (rlo == 0)
      run(std::integral_constant<int, 0>{});
    else if (rlo == 1)
      run(std::integral_constant<int, 1>{});
    else if (R > 2 && rlo == 2)
      run(std::integral_constant<int, (R > 2 ? 2 : 1)>{});
    else if (R > 3)
      run(std::integral_constant<int, (R > 3 ? 3 : 1)>{});
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (lane + 64 * r < n) part[(size_t)wave * n + lane + 64 * r] = q[r];
    __syncthreads();
    // the waves' products in two stages: four by four here, the two sums in the vector phase
    if ((t & 255) < n) {
      double2 s = make_double2(0.0, 0.0);
#pragma unroll
      for (int u = 0; u < ROW_WAVES / ROW_GROUPS; ++u) {
        const double2 y = part[(size_t)((t >> 8) * (ROW_WAVES / ROW_GROUPS) + u) * n + (t & 255)];
        s.x += y.x;
        s.y += y.y;
      }
      psum[(t >> 8) * n + (t & 255)] = s;
    }
    __syncthreads();
  }
  if (t == 0) d[n - 1] = scol[n - 1].x;
  __syncthreads();

  tri_pairs<ROW_NT>(n, nb, d, e, e2, lam, red, s_bounds, ecx, dph, Z);

  // ---- V = Q·D·Z, a wave per vector ------------------------------------------------------------
  double2* V = V_out + (size_t)b * n * nb;
  for (int jj = t; jj < nb; jj += ROW_NT) w_out[(size_t)b * nb + jj] = lam[jj];
  for (int jj = wave; jj < nb; jj += ROW_WAVES) {
    double2 y[R], h[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + 64 * r;
      y[r] = h[r] = make_double2(0.0, 0.0);
      if (i < n) {
        const double z = Z[(size_t)i * nb + jj];
        const double2 pz = dph[i];
        y[r] = make_double2(pz.x * z, pz.y * z);
      }
    }
    auto load = [&](double2(&g)[R], int k) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int i = lane + 64 * r;
        g[r] = make_double2(0.0, 0.0);
        if (k >= 0 && i > k && i < n) g[r] = A[(size_t)k * n + i];
      }
    };
    double2 g[R];
    load(h, n - 3);
    for (int k = n - 3; k >= 0; --k) {
      load(g, k - 1);  // the next reflector, in flight
      double sr = 0.0, si = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        sr += h[r].x * y[r].x + h[r].y * y[r].y;  // conj(v)·x
        si += h[r].x * y[r].y - h[r].y * y[r].x;
      }
      sr = 2.0 * wave_sum(sr);
      si = 2.0 * wave_sum(si);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        y[r].x -= h[r].x * sr - h[r].y * si;
        y[r].y -= h[r].x * si + h[r].y * sr;
        h[r] = g[r];
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (lane + 64 * r < n) V[(size_t)jj * n + lane + 64 * r] = y[r];
  }
  if (t == 0 && status) status[b] = 0;
}

// One wavefront per matrix, n <= JMAX: cyclic Jacobi with the matrix and the vectors in LDS.
__global__ void __launch_bounds__(64) k_jacobi(int n, int nb, const double2* __restrict__ Hb, double* __restrict__ w_out,
                                               double2* __restrict__ V_out) {
  __shared__ JacobiLds J;
  const int b = blockIdx.x, lane = threadIdx.x;
  const double2* H = Hb + (size_t)b * n * n;
  for (int e = lane; e < n * n; e += 64) {
    const int r = e % n, col = e / n;
    J.A[r][col] = H[e];
    J.V[r][col] = make_double2(r == col ? 1.0 : 0.0, 0.0);
  }
  __syncthreads();
  jacobi_lds(n, J);
  for (int jj = lane; jj < nb; jj += 64) w_out[(size_t)b * nb + jj] = J.A[J.order[jj]][J.order[jj]].x;
  for (int e = lane; e < n * nb; e += 64) {
    const int r = e % n, jj = e / n;
    V_out[(size_t)b * n * nb + e] = J.V[r][J.order[jj]];
  }
}

size_t heev_lds_base(int n, int nb) {
  size_t b = (size_t)2 * n * sizeof(double2) + ((size_t)3 * n + nb + EIG_WAVES + 2) * sizeof(double);
  b = (b + 15) & ~(size_t)15;
  return b + (size_t)16 * 64 * sizeof(double2);
}
constexpr size_t kLdsCap = 150 * 1024;
size_t a_bytes(int n) { return (size_t)n * n * sizeof(double2); }
size_t lu_bytes(int n, int nb) { return (size_t)6 * n * nb * sizeof(double); }
bool a_fits_lds(int n, int nb) { return heev_lds_base(n, nb) + a_bytes(n) <= kLdsCap; }
bool lu_fits_lds(int n, int nb) {
  return heev_lds_base(n, nb) + (a_fits_lds(n, nb) ? a_bytes(n) : 0) + lu_bytes(n, nb) <= kLdsCap;
}
// k_heev_rows: the partial products' area, or the tridiagonal's vectors and factors when they fit
bool rows_lu_in_lds(int n, int nb) { return rows_lds_head(n, nb) + lu_bytes(n, nb) <= kLdsCap; }
size_t rows_lds_bytes(int n, int nb) {
  const size_t part = (size_t)ROW_WAVES * n * sizeof(double2);
  return rows_lds_head(n, nb) + std::max(part, rows_lu_in_lds(n, nb) ? lu_bytes(n, nb) : (size_t)0);
}
template <int R>
void heev_rows(Context& c, int n, int nb, int nk, void* H, void* work, double* w, void* V, int* status) {
  const size_t sh = rows_lds_bytes(n, nb);
  ensure_lds_limit((const void*)k_heev_rows<R>, sh);
  k_heev_rows<R><<<(unsigned)nk, ROW_NT, sh, c.stream>>>(n, nb, rows_lu_in_lds(n, nb) ? 1 : 0, (double2*)H,
                                                         (double*)work, w, (double2*)V, status);
}
size_t heev_lds_bytes(int n, int nb) {
  return heev_lds_base(n, nb) + (a_fits_lds(n, nb) ? a_bytes(n) : 0) + (lu_fits_lds(n, nb) ? lu_bytes(n, nb) : 0);
}

}  // namespace

size_t heev_work_doubles(int n, int nb, int nk) { return (size_t)nk * eig_stride(n, nb); }

// ---- the allocation-free form -----------------------------------------------------------
// Workspace of pwk_dev_dense_eigh_noalloc: one static device array per GPU (16 MiB, held from
// the first use of the library on that GPU until the process ends). Host code never passes the
// array's name to a kernel: its device address is looked up once per device, with that device
// current, when a context is created on it, and only that address is used afterwards. Every
// call on one GPU shares the array; the eigensolver writes each workspace entry before reading
// it, so nothing needs clearing between calls, and calls that overlap on one GPU race.
constexpr size_t kNoAllocEigDoubles = (size_t)1 << 21;
static __device__ __align__(256) double scratch[kNoAllocEigDoubles];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

void init_noalloc_scratch(int device) {
  PWK_REQUIRE(device >= 0 && device < kMaxDevices, PWK_E_NO_DEVICE, "device ordinal above 63");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return;
  void* p = nullptr;
  PWK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  PWK_REQUIRE(p != nullptr, PWK_E_DEVICE, "static eigensolver workspace has no device address");
  g_scratch_ptr[device] = static_cast<double*>(p);
}

size_t noalloc_heev_capacity_doubles() { return kNoAllocEigDoubles; }

void launch_heev_noalloc(Context& c, int n, int nb, int nk, void* H, double* w, void* V) {
  PWK_REQUIRE(n >= 1 && nb >= 1 && nb <= n && nk >= 1, PWK_E_INVALID, "bad eigensolver shape");
  PWK_REQUIRE(heev_work_doubles(n, nb, nk) <= kNoAllocEigDoubles, PWK_E_INVALID,
              "batch needs more than the 16 MiB static workspace (nk*(4n + 6n*nb) doubles above 2^21)");
  double* ws = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (c.device >= 0 && c.device < kMaxDevices) ws = g_scratch_ptr[c.device];
  }
  PWK_REQUIRE(ws != nullptr, PWK_E_STATE, "static eigensolver workspace not set up on this device");
  launch_heev_batched(c, n, nb, nk, H, ws, w, V, nullptr);
}

bool heev_supported(int n, int nb) { return n >= 1 && nb >= 1 && nb <= n && heev_lds_base(n, nb) <= kLdsCap; }

void launch_heev_batched(Context& c, int n, int nb, int nk, void* H, void* work, double* w, void* V, int* status) {
  PWK_REQUIRE(n >= 1 && nb >= 1 && nb <= n && nk >= 1, PWK_E_INVALID, "bad eigensolver shape");
  PWK_REQUIRE(heev_supported(n, nb), PWK_E_UNSUPPORTED, "matrix too large for the batched eigensolver");
  const size_t sh = heev_lds_bytes(n, nb);
  TimedScope ts(c, "dense_eigh");
  if (n <= JMAX) {
    k_jacobi<<<(unsigned)nk, 64, 0, c.stream>>>(n, nb, (const double2*)H, w, (double2*)V);
    PWK_HIP(hipGetLastError());
    if (status) PWK_HIP(hipMemsetAsync(status, 0, (size_t)nk * sizeof(int), c.stream));
    return;
  }
  const int al = a_fits_lds(n, nb) ? 1 : 0, lu = lu_fits_lds(n, nb) ? 1 : 0;
  if (n <= 64) {
    ensure_lds_limit((const void*)k_heev<64>, sh);
    k_heev<64><<<(unsigned)nk, 64, sh, c.stream>>>(n, nb, al, lu, (double2*)H, (double*)work, w, (double2*)V,
                                                   status);
  } else if (n <= 256 && rows_lds_bytes(n, nb) <= kLdsCap) {
    if (n <= 128)
      heev_rows<2>(c, n, nb, nk, H, work, w, V, status);
    else if (n <= 192)
      heev_rows<3>(c, n, nb, nk, H, work, w, V, status);
    else
      heev_rows<4>(c, n, nb, nk, H, work, w, V, status);
  } else {
    ensure_lds_limit((const void*)k_heev<EIG_NT>, sh);
    k_heev<EIG_NT><<<(unsigned)nk, EIG_NT, sh, c.stream>>>(n, nb, al, lu, (double2*)H, (double*)work, w,
                                                           (double2*)V, status);
  }
  PWK_HIP(hipGetLastError());
}

}  // namespace pwk
