// Cyclic complex Jacobi eigensolver for small Hermitian matrices held in LDS,
// shared by the batched eigensolver (n <= 32) and the fused Rayleigh-Ritz
// kernel. Every thread of the block calls it; the rotations of one
// round-robin round are independent, so the block applies them together.
#pragma once

#include <hip/hip_runtime.h>

namespace pwk {

constexpr int JMAX = 32;

// LDS of the solver for matrices up to JM × JM
template <int JM>
struct JacobiLdsT {
  double2 A[JM][JM + 1];  // matrix (row, column); one padding column against bank conflicts
  double2 V[JM][JM + 1];  // accumulated rotations
  double rc[JM / 2], rs[JM / 2];
  double2 rph[JM / 2];
  int rp[JM / 2], rq[JM / 2], order[JM];
  double red[32];  // per-wave partial sums (off, total) for up to 16 waves
};
using JacobiLds = JacobiLdsT<JMAX>;

// Block-wide sum of (a, b) over all threads, in wave order (same result on every thread).
__device__ inline void jacobi_sum2(double& a, double& b, double* red) {
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  const int w = threadIdx.x >> 6, nw = (int)(blockDim.x >> 6);
  if ((threadIdx.x & 63) == 0) {
    red[2 * w] = a;
    red[2 * w + 1] = b;
  }
  __syncthreads();
  a = 0.0;
  b = 0.0;
  for (int i = 0; i < nw; ++i) {
    a += red[2 * i];
    b += red[2 * i + 1];
  }
  __syncthreads();
}

// J.order from the diagonal of J.A
template <int JM>
__device__ __forceinline__ void jacobi_order(int n, JacobiLdsT<JM>& J) {
  const int t = threadIdx.x;
  // ascending order by rank (ties by index). The order is total even for a NaN diagonal (NaNs
  // after every number, among themselves by index), so the ranks are always a permutation and
  // every entry of J.order is written.
  if (t < n) {
    const double di = J.A[t][t].x;
    const bool ni = di != di;
    int rank = 0;
    for (int j = 0; j < n; ++j) {
      const double dj = J.A[j][j].x;
      const bool nj = dj != dj;
      const bool before = (ni || nj) ? (nj == ni ? j < t : ni) : (dj < di || (dj == di && j < t));
      rank += before ? 1 : 0;
    }
    J.order[rank] = t;
  }
  __syncthreads();
}

// Diagonalises J.A (n <= JMAX) in place: on return the diagonal of J.A holds the eigenvalues,
// J.V = V_in · (product of the rotations), J.order[r] the index of the r-th smallest eigenvalue
// (ties by index). Sweeps stop when the off-diagonal weight falls below 1e-30 of the total.
template <int JM>
__device__ inline void jacobi_lds(int n, JacobiLdsT<JM>& J) {
  const int t = threadIdx.x, nt = blockDim.x;
  const int N = n + (n & 1);
  for (int sweep = 0; sweep < 30; ++sweep) {
    double off = 0.0, tot = 0.0;
    for (int e = t; e < n * n; e += nt) {
      const int r = e % n, col = e / n;
      const double2 a = J.A[r][col];
      const double m2 = a.x * a.x + a.y * a.y;
      tot += m2;
      if (r != col) off += m2;
    }
    jacobi_sum2(off, tot, J.red);
    if (off <= 1e-30 * tot || off < 1e-300) break;  // block-uniform
    for (int round = 0; round < N - 1; ++round) {
      // round-robin pairing: position 0 stays, positions 1..N-1 have rotated `round` times
      if (t < N / 2) {
        const int u = N - 1 - t;
        // (t - 1 - round) and (u - 1 - round) lie in (-(N - 1), N - 1): one wrap is enough
        int p = 0;
        if (t != 0) {
          p = t - 1 - round;
          p += p < 0 ? N - 1 : 0;
          p += 1;
        }
        int q = u - 1 - round;
        q += q < 0 ? N - 1 : 0;
        q += 1;
        if (p > q) {
          const int tt = p;
          p = q;
          q = tt;
        }
        double c = 1.0, sn = 0.0;
        double2 ph = make_double2(1.0, 0.0);
        if (q < n) {
          // with d = (A_qq - A_pp)/2, g = |A_pq|: tan θ = sign(d)·g/(|d| + sqrt(d² + g²)), so
          // c = den/sqrt(den² + g²), s = sign(d)·g/sqrt(den² + g²) with den = |d| + sqrt(d² + g²),
          // and the phase A_pq/g: one sqrt and two reciprocal square roots on the chain
          const double a = J.A[p][p].x, bq = J.A[q][q].x;
          const double2 apq = J.A[p][q];
          const double g2 = apq.x * apq.x + apq.y * apq.y;
          if (g2 > 1e-300) {  // |A_pq| above 1e-150: no denormal reaches rsqrt
            const double ig = rsqrt(g2);
            ph = make_double2(apq.x * ig, apq.y * ig);
            const double d = 0.5 * (bq - a);
            const double den = fabs(d) + sqrt(d * d + g2);
            const double inv = rsqrt(den * den + g2);
            c = den * inv;
            sn = (d >= 0.0 ? 1.0 : -1.0) * (g2 * ig) * inv;
          }
        }
        J.rp[t] = p;
        J.rq[t] = q < n ? q : -1;
        J.rc[t] = c;
        J.rs[t] = sn;
        J.rph[t] = ph;
      }
      __syncthreads();
      // A ← Wᴴ·A·W block by block: the entries in the rows of pair kr and the columns of pair kc
      // change only through rotations kr and kc, so each (kr, kc) block is updated by one thread
      // (the column rotation, then the row rotation, as a column pass followed by a row pass
      // would); V ← V·W column pairs alongside. W = [[c, s], [-s e, c e]], e = conj(ph).
      const int NP = N / 2;
      for (int it = t; it < NP * NP + NP * n; it += nt) {
        if (it < NP * NP) {
          const int kr = it / NP, kc = it % NP;
          const int pr = J.rp[kr], qr = J.rq[kr], pc = J.rp[kc], qc = J.rq[kc];
          double2 a00 = J.A[pr][pc], a01 = qc >= 0 ? J.A[pr][qc] : make_double2(0.0, 0.0);
          double2 a10 = qr >= 0 ? J.A[qr][pc] : make_double2(0.0, 0.0);
          double2 a11 = (qr >= 0 && qc >= 0) ? J.A[qr][qc] : make_double2(0.0, 0.0);
          if (qc >= 0) {  // columns (pc, qc)
            const double c = J.rc[kc], sn = J.rs[kc];
            const double2 e = make_double2(J.rph[kc].x, -J.rph[kc].y);
            double2 ey = make_double2(e.x * a01.x - e.y * a01.y, e.x * a01.y + e.y * a01.x);
            const double2 n00 = make_double2(c * a00.x - sn * ey.x, c * a00.y - sn * ey.y);
            const double2 n01 = make_double2(sn * a00.x + c * ey.x, sn * a00.y + c * ey.y);
            a00 = n00;
            a01 = n01;
            if (qr >= 0) {
              ey = make_double2(e.x * a11.x - e.y * a11.y, e.x * a11.y + e.y * a11.x);
              const double2 n10 = make_double2(c * a10.x - sn * ey.x, c * a10.y - sn * ey.y);
              const double2 n11 = make_double2(sn * a10.x + c * ey.x, sn * a10.y + c * ey.y);
              a10 = n10;
              a11 = n11;
            }
          }
          if (qr >= 0) {  // rows (pr, qr), Wᴴ = [[c, -s conj(e)], [s, c conj(e)]]
            const double c = J.rc[kr], sn = J.rs[kr];
            const double2 ce = J.rph[kr];
            double2 ey = make_double2(ce.x * a10.x - ce.y * a10.y, ce.x * a10.y + ce.y * a10.x);
            const double2 n00 = make_double2(c * a00.x - sn * ey.x, c * a00.y - sn * ey.y);
            const double2 n10 = make_double2(sn * a00.x + c * ey.x, sn * a00.y + c * ey.y);
            a00 = n00;
            a10 = n10;
            if (qc >= 0) {
              ey = make_double2(ce.x * a11.x - ce.y * a11.y, ce.x * a11.y + ce.y * a11.x);
              const double2 n01 = make_double2(c * a01.x - sn * ey.x, c * a01.y - sn * ey.y);
              const double2 n11 = make_double2(sn * a01.x + c * ey.x, sn * a01.y + c * ey.y);
              a01 = n01;
              a11 = n11;
            }
          }
          J.A[pr][pc] = a00;
          if (qc >= 0) J.A[pr][qc] = a01;
          if (qr >= 0) J.A[qr][pc] = a10;
          if (qr >= 0 && qc >= 0) J.A[qr][qc] = a11;
        } else {
          const int rem = it - NP * NP, k = rem / n, r = rem % n, q = J.rq[k];
          if (q < 0) continue;
          const int p = J.rp[k];
          const double c = J.rc[k], sn = J.rs[k];
          const double2 e = make_double2(J.rph[k].x, -J.rph[k].y);
          const double2 x = J.V[r][p], y = J.V[r][q];
          const double2 ey = make_double2(e.x * y.x - e.y * y.y, e.x * y.y + e.y * y.x);
          J.V[r][p] = make_double2(c * x.x - sn * ey.x, c * x.y - sn * ey.y);
          J.V[r][q] = make_double2(sn * x.x + c * ey.x, sn * x.y + c * ey.y);
        }
      }
      __syncthreads();
    }
  }
  jacobi_order(n, J);
}

// 1/sqrt(x) for normal x > 0: v_rsq_f64 (2^-23) and one step of third order, e³ < 2^-66, so the result
// carries the rounding of the step alone. The library's function and its sqrt handle denormals and
// infinities as well, which the rotations never pass; they were half of a rotation's serial chain.
__device__ __forceinline__ double jacobi_rsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// The rotation W = [[c, σ], [-conj(σ), c]] of columns (p, q) that makes (Wᴴ·A·W)_pq zero. With
// d = (A_qq - A_pp)/2 and h = sqrt(d² + |A_pq|²): cos 2θ = |d|/h, so c² = (1 + |d|/h)/2, in [1/2, 1]
// without cancellation, and σ = sign(d)·A_pq/(2·h·c): two reciprocal square roots on the chain and no
// separate phase.
__device__ __forceinline__ void jacobi_rotation(double app, double aqq, double2 apq, double& c, double2& s) {
  const double g2 = apq.x * apq.x + apq.y * apq.y;
  c = 1.0;
  s = make_double2(0.0, 0.0);
  if (g2 > 1e-300) {  // |A_pq| above 1e-150: no denormal reaches the reciprocal roots
    const double d = 0.5 * (aqq - app);
    const double ih = jacobi_rsqrt(fma(d, d, g2));
    const double c2 = fma(0.5 * fabs(d), ih, 0.5);
    const double ic = jacobi_rsqrt(c2);
    c = c2 * ic;
    const double f = (d >= 0.0 ? 0.5 : -0.5) * ih * ic;
    s = make_double2(apq.x * f, apq.y * f);
  }
}

// (x, y) <- (c·x - conj(s)·y, s·x + c·y): the rotation on two columns
__device__ __forceinline__ void jacobi_cols(double c, double2 s, double2& x, double2& y) {
  const double2 u = make_double2(c * x.x - (s.x * y.x + s.y * y.y), c * x.y - (s.x * y.y - s.y * y.x));
  y = make_double2(c * y.x + (s.x * x.x - s.y * x.y), c * y.y + (s.x * x.y + s.y * x.x));
  x = u;
}

// pair k of a round: position 0 stays, positions 1..N-1 have rotated `round` times
__device__ __forceinline__ void jacobi_pair(int N, int round, int k, int& p, int& q) {
  const int u = N - 1 - k;
  // (k - 1 - round) and (u - 1 - round) lie in (-(N - 1), N - 1): one wrap is enough
  int a = k - 1 - round, b = u - 1 - round;
  a += (a < 0 ? N - 1 : 0) + 1;
  b += (b < 0 ? N - 1 : 0) + 1;
  if (k == 0) a = 0;
  p = min(a, b);
  q = max(a, b);
}

// The same for a workgroup of NT >= (JM/2)² threads, with a second image A2 of A (any contents): a thread
// per 2 × 2 block (kr, kc), which computes both of its rotations itself and writes the block to the other
// image, so that a round has one barrier and no rotation goes through LDS. A round is a serial chain (LDS
// read, two reciprocal roots, the updates, barrier), not work: what is computed twice costs less than the
// exchange. An odd n is padded with a zero row and column, whose rotations are the identity.
template <int JM, int NT>
__device__ inline void jacobi_block(int n, JacobiLdsT<JM>& J, double2 (*A2)[JM + 1]) {
  constexpr int HB = JM / 2;
  static_assert(NT >= HB * HB, "a thread per block of two pairs");
  // rows of V: on threads that hold no block where they are enough, beside the blocks elsewhere
  constexpr bool APART = NT >= HB * HB + HB * JM;
  const int t = threadIdx.x, N = n + (n & 1), NP = N / 2;
  const int kc = t % HB, kr = t / HB;
  const bool on = kc < NP, blk = on && kr < NP;
  const int v0 = APART ? kr - HB : kr;
  if (n < N && t < N) {
    J.A[n][t] = J.A[t][n] = make_double2(0.0, 0.0);
    J.V[n][t] = J.V[t][n] = make_double2(0.0, 0.0);
  }
  double2(*A)[JM + 1] = J.A;
  double2(*B)[JM + 1] = A2;
  for (int sweep = 0; sweep < 30; ++sweep) {
    double off = 0.0, tot = 0.0;
    for (int e = t; e < JM * JM; e += NT) {
      const int r = e / JM, col = e % JM;
      if (r < n && col < n) {
        const double2 a = A[r][col];
        const double m2 = a.x * a.x + a.y * a.y;
        tot += m2;
        if (r != col) off += m2;
      }
    }
    jacobi_sum2(off, tot, J.red);
    if (off <= 1e-30 * tot || off < 1e-300) break;  // block-uniform
    for (int round = 0; round < N - 1; ++round) {
      if (on) {
        int pc, qc;
        jacobi_pair(N, round, kc, pc, qc);
        double cc;
        double2 sc;
        if (blk) {
          int pr, qr;
          jacobi_pair(N, round, kr, pr, qr);
          double2 a00 = A[pr][pc], a01 = A[pr][qc], a10 = A[qr][pc], a11 = A[qr][qc];
          const double rp = A[pr][pr].x, rq = A[qr][qr].x;
          const double2 rpq = A[pr][qr];
          double cr;
          double2 sr;
          jacobi_rotation(A[pc][pc].x, A[qc][qc].x, A[pc][qc], cc, sc);
          jacobi_rotation(rp, rq, rpq, cr, sr);
          jacobi_cols(cc, sc, a00, a01);
          jacobi_cols(cc, sc, a10, a11);
          sr.y = -sr.y;  // rows: the conjugate rotation
          jacobi_cols(cr, sr, a00, a10);
          jacobi_cols(cr, sr, a01, a11);
          B[pr][pc] = a00;
          B[pr][qc] = a01;
          B[qr][pc] = a10;
          B[qr][qc] = a11;
        } else {
          jacobi_rotation(A[pc][pc].x, A[qc][qc].x, A[pc][qc], cc, sc);
        }
        // the threads of pair kc share its columns of V by rows
#pragma unroll
        for (int r = v0; r < (APART ? v0 + 1 : JM); r += HB)
          if (r >= 0 && r < n) {
            double2 x = J.V[r][pc], y = J.V[r][qc];
            jacobi_cols(cc, sc, x, y);
            J.V[r][pc] = x;
            J.V[r][qc] = y;
          }
      }
      __syncthreads();
      double2(*T)[JM + 1] = A;
      A = B;
      B = T;
    }
  }
  if (A != J.A) {  // block-uniform
    if (t < n) J.A[t][t] = A[t][t];
    __syncthreads();
  }
  jacobi_order(n, J);
}

}  // namespace pwk
