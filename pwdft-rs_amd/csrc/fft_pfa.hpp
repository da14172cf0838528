// Register-resident FFT of compile-time length N without twiddles between coprime factors.
//
// N = Π q_i with q_i powers of 2, 3 and 5 (Good 1958, Thomas 1963): with the input index written
// n = Σ n_i·(N/q_i) mod N, X[k] = Σ x[n] e^{∓2πi nk/N} separates into plain q_i-point transforms over
// n_i at frequency k mod q_i. Each runs in place by decimation in frequency (radices 4, 2, 3, 5,
// twiddles only inside a prime power), so every index is a constant after unrolling and the values stay
// in VGPRs; LineOrder<N>::pos(f) is where frequency f ends up. Inputs that are literal zeros and
// outputs that are never read drop out of the arithmetic at compile time.
//
// A 60-point transform takes 912 vector instructions instead of the 1250 of the mixed-radix form of
// fft_reg.hpp, a 45-point one 764 instead of 950: the plane and stick passes are bound by them.
#pragma once

#include "fft_reg.hpp"

namespace pwk {

template <typename T, int SIGN>
__device__ __forceinline__ void pfa_bfly3(T& r0, T& i0, T& r1, T& i1, T& r2, T& i2) {
  const T h = (T)((double)SIGN * 0.86602540378443864676);
  const T tr = r1 + r2, ti = i1 + i2, dr = r1 - r2, di = i1 - i2;
  const T mr = r0 - (T)0.5 * tr, mi = i0 - (T)0.5 * ti;
  r0 += tr;
  i0 += ti;
  r1 = mr - h * di;
  i1 = mi + h * dr;
  r2 = mr + h * di;
  i2 = mi - h * dr;
}

template <typename T, int SIGN>
__device__ __forceinline__ void pfa_bfly5(T (&r)[5], T (&i)[5]) {
  const T k = (T)0.55901699437494742410;  // √5/4
  const T s1 = (T)((double)SIGN * 0.95105651629515357212), s2 = (T)((double)SIGN * 0.58778525229247312917);
  const T t1r = r[1] + r[4], t1i = i[1] + i[4], t2r = r[2] + r[3], t2i = i[2] + i[3];
  const T d1r = r[1] - r[4], d1i = i[1] - i[4], d2r = r[2] - r[3], d2i = i[2] - i[3];
  const T tr = t1r + t2r, ti = t1i + t2i, ur = t1r - t2r, ui = t1i - t2i;
  const T mr = r[0] - (T)0.25 * tr, mi = i[0] - (T)0.25 * ti;
  const T ar = mr + k * ur, ai = mi + k * ui, br = mr - k * ur, bi = mi - k * ui;
  const T e1r = s1 * d1r + s2 * d2r, e1i = s1 * d1i + s2 * d2i;
  const T e2r = s2 * d1r - s1 * d2r, e2i = s2 * d1i - s1 * d2i;
  r[0] += tr;
  i[0] += ti;
  r[1] = ar - e1i;
  i[1] = ai + e1r;
  r[4] = ar + e1i;
  i[4] = ai - e1r;
  r[2] = br - e2i;
  i[2] = bi + e2r;
  r[3] = br + e2i;
  i[3] = bi - e2r;
}

// x·e^{SIGN·2πi·e/M}; multiples of a quarter turn without arithmetic
template <typename T, int M, int SIGN>
__device__ __forceinline__ void pfa_twiddle(T& xr, T& xi, int e) {
  const T r = xr, i = xi;
  if ((4 * e) % M == 0) {
    const int q = (((4 * e) / M) * (SIGN > 0 ? 1 : 3)) % 4;
    xr = q == 0 ? r : q == 1 ? -i : q == 2 ? -r : i;
    xi = q == 0 ? i : q == 1 ? r : q == 2 ? -i : -r;
  } else {
    const T wc = (T)Twiddle<M, SIGN>::tab.c[e], ws = (T)Twiddle<M, SIGN>::tab.s[e];
    xr = r * wc - i * ws;
    xi = r * ws + i * wc;
  }
}

// in-place decimation in frequency of the Q values r[b + ·] (Q a power of 2, 3 or 5), then of its blocks
template <typename T, int Q, int M, int SIGN>
__device__ __forceinline__ void pfa_stages(T (&r)[Q], T (&i)[Q]) {
  if constexpr (M > 1) {
    constexpr int p = first_radix(M), m = M / p;
#pragma unroll
    for (int b = 0; b < Q; b += M) {
#pragma unroll
      for (int k = 0; k < m; ++k) {
        const int o = b + k;
        if constexpr (p == 2) {
          bfly2<T, SIGN>(r, i, o, o + m);
        } else if constexpr (p == 4) {
          bfly4<T, SIGN>(r, i, o, o + m, o + 2 * m, o + 3 * m);
        } else if constexpr (p == 3) {
          pfa_bfly3<T, SIGN>(r[o], i[o], r[o + m], i[o + m], r[o + 2 * m], i[o + 2 * m]);
        } else {
          T xr[5] = {r[o], r[o + m], r[o + 2 * m], r[o + 3 * m], r[o + 4 * m]};
          T xi[5] = {i[o], i[o + m], i[o + 2 * m], i[o + 3 * m], i[o + 4 * m]};
          pfa_bfly5<T, SIGN>(xr, xi);
#pragma unroll
          for (int q = 0; q < 5; ++q) {
            r[o + q * m] = xr[q];
            i[o + q * m] = xi[q];
          }
        }
#pragma unroll
        for (int q = 1; q < p; ++q) pfa_twiddle<T, M, SIGN>(r[o + q * m], i[o + q * m], (q * k) % M);
      }
    }
    pfa_stages<T, Q, m, SIGN>(r, i);
  }
}

constexpr int pfa_part(int n, int p) {  // the power of p in n
  int q = 1;
  while (n % p == 0) {
    n /= p;
    q *= p;
  }
  return q;
}

// index of element t of line l of the Q-point transforms inside N: the lines are the residues modulo
// N/Q, each started at its multiple of Q (coordinate 0)
template <int N, int Q>
struct PfaLines {
  struct Table {
    int p[N / Q][Q];
  };
  static constexpr Table make() {
    Table t{};
    constexpr int s = N / Q;
    for (int l = 0; l < s; ++l) {
      int b = l;
      while (b % Q != 0) b += s;
      for (int e = 0; e < Q; ++e) t.p[l][e] = (b + e * s) % N;
    }
    return t;
  }
  static constexpr Table tab = make();
};

template <typename T, int N, int Q, int SIGN>
__device__ __forceinline__ void pfa_factor(T (&re)[N], T (&im)[N]) {
  if constexpr (Q > 1) {
#pragma unroll
    for (int l = 0; l < N / Q; ++l) {
      T r[Q], i[Q];
#pragma unroll
      for (int e = 0; e < Q; ++e) {
        r[e] = re[PfaLines<N, Q>::tab.p[l][e]];
        i[e] = im[PfaLines<N, Q>::tab.p[l][e]];
      }
      pfa_stages<T, Q, Q, SIGN>(r, i);
#pragma unroll
      for (int e = 0; e < Q; ++e) {
        re[PfaLines<N, Q>::tab.p[l][e]] = r[e];
        im[PfaLines<N, Q>::tab.p[l][e]] = i[e];
      }
    }
  }
}

template <int N>
struct LineOrder {
  struct Table {
    int p[N];
  };
  static constexpr Table make() {
    Table t{};
    constexpr int q2 = pfa_part(N, 2), q3 = pfa_part(N, 3), q5 = pfa_part(N, 5);
    for (int f = 0; f < N; ++f)
      t.p[f] = (FftOrder<q2>::pos_rec(f % q2, q2) * (N / q2) + FftOrder<q3>::pos_rec(f % q3, q3) * (N / q3) +
                FftOrder<q5>::pos_rec(f % q5, q5) * (N / q5)) % N;
    return t;
  }
  static constexpr Table tab = make();
  static constexpr int pos(int f) { return tab.p[f]; }
};

// In-place FFT; frequency f ends at LineOrder<N>::pos(f). The factor of 2 first: with the middle half of
// the input zero, its butterflies simplify most.
template <typename T, int N, int SIGN>
__device__ __forceinline__ void fft_line(T (&re)[N], T (&im)[N]) {
  pfa_factor<T, N, pfa_part(N, 2), SIGN>(re, im);
  pfa_factor<T, N, pfa_part(N, 3), SIGN>(re, im);
  pfa_factor<T, N, pfa_part(N, 5), SIGN>(re, im);
}

}  // namespace pwk
