// Complex GEMM on the matrix cores, column-major: C (+)= A·B, A M×K, B K×N.
//
// A wave owns 16 complex rows and all columns of its tile. Its complex product is two real products with
// the same B operand (interleaved re, im along k): the rows of real parts (re, -im, ...) and the rows of
// imaginary parts (im, re, ...) of A, so a lane holds the real and the imaginary part of each of its C
// entries. In a 16×16 MFMA step over 32 real k a lane holds row l mod 16 and the 8 real k of group l / 16,
// which are 4 whole complex entries of A: a lane loads them from global memory into registers (a wave's
// load is four runs of 16 consecutive rows) and A never passes through LDS. B, which the four waves of a
// workgroup share, is staged in LDS (split to bf16 on the way in), double-buffered with one barrier per
// 16 complex k; the loads of the next steps are in flight during the MFMAs of the current one.
//   MODE_F32 : v_mfma_f32_16x16x4_f32, 8 steps of 4 real k (lane group g supplies k = 8g + step)
//   MODE_F64 : v_mfma_f64_16x16x4_f64, likewise
//   MODE_BF16X3 : v_mfma_f32_16x16x32_bf16 on the split x = hi + lo,
//                 hi = bf16(x), lo = bf16(x - hi); C += Alo·Bhi + Ahi·Blo + Ahi·Bhi (FP32 accumulate)
// Split-K partial sums are reduced in a fixed order (deterministic).
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace pwk {

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));
typedef double d4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));

enum { MODE_F32 = 0, MODE_F64 = 1, MODE_BF16X3 = 2 };

constexpr int BMC = 64;  // complex rows per block
constexpr int BKC = 16;  // complex K per step
constexpr int BKR = 32;  // real K per step

template <int MODE>
struct Traits {
  using T = float;
  using V2 = float2;
  using acc_t = f4v;
};
template <>
struct Traits<MODE_F64> {
  using T = double;
  using V2 = double2;
  using acc_t = d4v;
};

__device__ __forceinline__ __bf16 to_bf16(float x) { return (__bf16)x; }

// LDS row stride of a B column (elements): its 32 real k, padded so that the 16-byte reads of the 16
// columns of a fragment fall on distinct banks
template <int MODE>
constexpr int b_stride() {
  return MODE == MODE_BF16X3 ? BKR + 8 : MODE == MODE_F32 ? BKR + 4 : BKR + 2;
}

// a barrier that waits for LDS traffic only: global loads stay in flight across it
__device__ __forceinline__ void lds_only_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// the A fragments of one step from a lane's 4 complex entries: [0] real rows, [1] imaginary rows
template <int MODE>
struct AFrag {
  using T = typename Traits<MODE>::T;
  T v[2][8];
  __device__ __forceinline__ void make(const typename Traits<MODE>::V2 (&a)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[0][2 * k] = a[k].x;
      v[0][2 * k + 1] = -a[k].y;
      v[1][2 * k] = a[k].y;
      v[1][2 * k + 1] = a[k].x;
    }
  }
};
template <>
struct AFrag<MODE_BF16X3> {
  bf8v hi[2], lo[2];
  __device__ __forceinline__ void make(const float2 (&a)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const __bf16 hx = to_bf16(a[k].x), hy = to_bf16(a[k].y);
      const __bf16 lx = to_bf16(a[k].x - (float)hx), ly = to_bf16(a[k].y - (float)hy);
      hi[0][2 * k] = hx;
      hi[0][2 * k + 1] = -hy;
      hi[1][2 * k] = hy;
      hi[1][2 * k + 1] = hx;
      lo[0][2 * k] = lx;
      lo[0][2 * k + 1] = -ly;
      lo[1][2 * k] = ly;
      lo[1][2 * k + 1] = lx;
    }
  }
};

// Widest column tile (blocks of 16) and workgroups per CU that split K aims at. Two or three narrow tiles
// per CU hide each other's loads, conversions and barriers better than one wide tile, and A re-read by the
// column tiles comes from L2: Si64 split-bf16 512 × 144 × 13133, 3 blocks and 32 chunks 46 us, 9 blocks 53-60;
// 13133 × 144 × 512 47 against 58; FP64 256 × 160 × 6859, 2 blocks 51 us, 5 blocks 57.
template <int MODE>
struct Tile {
  static constexpr int W = MODE == MODE_F64 ? 2 : 3, PER_CU = MODE == MODE_F64 ? 2 : 3;
};

// Bound: the matrix cores; per step a workgroup issues 4·NB16·{6, 16} MFMAs (split-bf16, FP32/FP64).
// Against the form with A and B in LDS behind two barriers per step and one wide tile per CU (projection with
// its partial sums, expansion): split-bf16 512 × 144 × 13133 75 and 79 us -> 51 and 47 us; FP64
// 256 × 160 × 6859 133 and 90 us -> 57 and 56 us.
template <int MODE, int NB16, class Groups>
__global__ void __launch_bounds__(256, 2) k_zgemm_mfma(int M, int N, int K, int kchunk, int nsplit, long long sA,
                                                    long long sB, long long sC,
                                                    const typename Traits<MODE>::V2* __restrict__ A, int lda,
                                                    const typename Traits<MODE>::V2* __restrict__ B, int ldb,
                                                    typename Traits<MODE>::V2* __restrict__ C, int ldc, int accumulate,
                                                    typename Traits<MODE>::V2* __restrict__ partial,
                                                    const Groups groups) {
  using V2 = typename Traits<MODE>::V2;
  using T = typename Traits<MODE>::T;
  using acc_t = typename Traits<MODE>::acc_t;
  constexpr int BN = 16 * NB16, BKS = b_stride<MODE>();
  constexpr bool SPLIT = MODE == MODE_BF16X3;
  using ldsT = typename std::conditional<SPLIT, __bf16, T>::type;
  constexpr int NPART = SPLIT ? 2 : 1;
  __shared__ __attribute__((aligned(16))) ldsT Bs[2][NPART][BN * BKS];

  const int tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, li = lane & 15, lk = lane >> 4;
  // One-dimensional grid over (row tile, column tile, batch · nsplit + split). Workgroup i runs on
  // XCD i mod 8, and each XCD takes a contiguous range of tiles in an order where neighbours
  // share an operand in that XCD's L2: with split K, the row and column tiles of one K chunk
  // (they read the same B rows); without, the column tiles of one row tile (the same A rows).
  const int mt = (M + BMC - 1) / BMC, nt = (N + BN - 1) / BN, plane = mt * nt;
  const int total = (int)gridDim.x, xcd = (int)blockIdx.x & 7;
  const int lg = xcd * (total >> 3) + min(xcd, total & 7) + ((int)blockIdx.x >> 3);
  const int bz = lg / plane, rem = lg % plane;
  const int bx = nsplit > 1 ? rem % mt : rem / nt, by = nsplit > 1 ? rem / mt : rem % nt;
  const int m0 = bx * BMC + w * 16, n0 = by * BN;
  // bz = batch · nsplit + split
  const int zb = bz / nsplit, zs = bz % nsplit;
  if (partial) partial += (size_t)(zb * nsplit + zs) * M * N;
  if constexpr (Groups::batch) {  // products of their own A and column count; N is the widest
    A = (const V2*)groups.A[zb];
    B += (size_t)groups.col[zb] * ldb;
    C += (size_t)groups.col[zb] * ldc;
    N = groups.cols[zb];
    if (n0 >= N) return;
  } else {
    A += (size_t)zb * sA;
    B += (size_t)zb * sB;
    C += (size_t)zb * sC;
  }
  const int kbeg = zs * kchunk;
  const int kend = min(K, kbeg + kchunk);

  acc_t acc[NB16][2];
#pragma unroll
  for (int cb = 0; cb < NB16; ++cb)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[cb][h][q] = 0;

  // Rows and columns past the matrix repeat its last one (never stored); k past the chunk is zero in A and B.
  const V2* a_row = A + min(m0 + li, M - 1);
  constexpr int NBV = (BKC * BN + 255) / 256;
  V2 ra[2][4], rb[2][NBV];
  const int kk = tid & (BKC - 1);  // this thread's k within a step of B, for every column it loads
  const V2* b_col[NBV];
#pragma unroll
  for (int e = 0; e < NBV; ++e) b_col[e] = B + (size_t)min(n0 + min(tid / BKC + 16 * e, BN - 1), N - 1) * ldb;
  auto load_a = [&](V2(&r)[4], int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = a_row[(size_t)min(k0 + 4 * lk + i, kend - 1) * lda];
  };
  auto load_b = [&](V2(&r)[NBV], int k0) {
    const int k = min(k0 + kk, kend - 1);
#pragma unroll
    for (int e = 0; e < NBV; ++e) r[e] = b_col[e][k];
  };
  auto store_b = [&](const V2(&r)[NBV], int buf, int k0) {
    const bool in = k0 + kk < kend;
#pragma unroll
    for (int e = 0; e < NBV; ++e) {
      const int nn = tid / BKC + 16 * e;
      const T x = in ? r[e].x : (T)0, y = in ? r[e].y : (T)0;
      ldsT* p = &Bs[buf][0][nn * BKS + 2 * kk];
      if constexpr (SPLIT) {
        const __bf16 hx = to_bf16(x), hy = to_bf16(y);
        p[0] = hx;
        p[1] = hy;
        ldsT* q = &Bs[buf][1][nn * BKS + 2 * kk];
        q[0] = to_bf16(x - (float)hx);
        q[1] = to_bf16(y - (float)hy);
      } else {
        p[0] = x;
        p[1] = y;
      }
    }
  };
  auto step = [&](V2(&a)[4], V2(&b)[NBV], int k0, int buf) {
    if (k0 + BKC > kend) {  // the chunk's last, shorter step
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (k0 + 4 * lk + i >= kend) a[i].x = a[i].y = 0;
    }
    AFrag<MODE> f;
    f.make(a);
    store_b(b, buf, k0);
    // the loads of the step after next, unconditionally (clamped), so that the waits count them exactly
    load_b(b, k0 + 2 * BKC);
    load_a(a, k0 + 2 * BKC);
    lds_only_barrier();
    // all columns of one product term in turn: independent MFMA chains hide their latency
    if constexpr (SPLIT) {
      bf8v bhi[NB16], blo[NB16];
#pragma unroll
      for (int c = 0; c < NB16; ++c) {
        const int o = (c * 16 + li) * BKS + lk * 8;
        bhi[c] = *reinterpret_cast<const bf8v*>(&Bs[buf][0][o]);
        blo[c] = *reinterpret_cast<const bf8v*>(&Bs[buf][1][o]);
      }
#pragma unroll
      for (int c = 0; c < NB16; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[c][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.lo[h], bhi[c], acc[c][h], 0, 0, 0);
#pragma unroll
      for (int c = 0; c < NB16; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[c][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.hi[h], blo[c], acc[c][h], 0, 0, 0);
#pragma unroll
      for (int c = 0; c < NB16; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[c][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.hi[h], bhi[c], acc[c][h], 0, 0, 0);
    } else {
      typedef T v16 __attribute__((ext_vector_type(16 / sizeof(T))));  // 16-byte LDS reads
      constexpr int V = 16 / (int)sizeof(T);
      T bv[NB16][8];
#pragma unroll
      for (int c = 0; c < NB16; ++c)
#pragma unroll
        for (int i = 0; i < 8; i += V) {
          const v16 x = *reinterpret_cast<const v16*>(&Bs[buf][0][(c * 16 + li) * BKS + lk * 8 + i]);
#pragma unroll
          for (int j = 0; j < V; ++j) bv[c][i + j] = x[j];
        }
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
#pragma unroll
        for (int c = 0; c < NB16; ++c)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if constexpr (MODE == MODE_F32)
              acc[c][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.v[h][ks], bv[c][ks], acc[c][h], 0, 0, 0);
            else
              acc[c][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.v[h][ks], bv[c][ks], acc[c][h], 0, 0, 0);
          }
    }
  };
  if (kbeg < kend) {
    load_b(rb[0], kbeg);
    load_a(ra[0], kbeg);
    load_b(rb[1], kbeg + BKC);
    load_a(ra[1], kbeg + BKC);
    // two steps per turn: the registers and the LDS buffers alternate at constant indices (a step past
    // the chunk adds zeros)
    for (int k0 = kbeg; k0 < kend; k0 += 2 * BKC) {
      step(ra[0], rb[0], k0, 0);
      step(ra[1], rb[1], k0 + BKC, 1);
    }
  }
  // Store. Result rows of a lane: 4·(l/16) + q, or l/16 + 4q in FP64 (measured on gfx950); column l mod 16.
#pragma unroll
  for (int cb = 0; cb < NB16; ++cb) {
    const int gn = n0 + cb * 16 + li;
    if (gn >= N) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int gm = m0 + (MODE == MODE_F64 ? lk + 4 * q : 4 * lk + q);
      if (gm >= M) continue;
      V2 o;
      o.x = acc[cb][0][q];
      o.y = acc[cb][1][q];
      if (partial) {
        partial[(size_t)gn * M + gm] = o;
      } else {
        V2* c = &C[(size_t)gn * ldc + gm];
        if (accumulate) {
          const V2 old = *c;
          o.x += old.x;
          o.y += old.y;
        }
        *c = o;
      }
    }
  }
}

template <typename V2, class Groups>
__global__ void __launch_bounds__(256) k_splitk_sum(int M, int N, int nsplit, const V2* __restrict__ partial,
                                                    V2* __restrict__ C, int ldc, long long sC, int accumulate,
                                                    const Groups groups) {
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)M * N) return;
  partial += (size_t)blockIdx.y * nsplit * M * N;
  int gm = (int)(idx % M), gn = (int)(idx / M);
  if constexpr (Groups::batch) {
    if (gn >= groups.cols[blockIdx.y]) return;
    C += (size_t)groups.col[blockIdx.y] * ldc;
  } else {
    C += (size_t)blockIdx.y * sC;
  }
  V2 s;
  s.x = 0;
  s.y = 0;
#pragma unroll 8
  for (int z = 0; z < nsplit; ++z) {
    V2 p = partial[(size_t)z * M * N + idx];
    s.x += p.x;
    s.y += p.y;
  }
  V2* c = &C[(size_t)gn * ldc + gm];
  if (accumulate) {
    V2 old = *c;
    s.x += old.x;
    s.y += old.y;
  }
  *c = s;
}

struct Batch {
  int count = 1;
  long long sA = 0, sB = 0, sC = 0;  // element strides between consecutive products
};

template <int MODE, int NB16, class Groups>
void launch_nb(Context& c, dim3 grid, int M, int N, int K, int kchunk, int nsplit, const Batch& bt, const void* A,
               int lda, const void* B, int ldb, void* C, int ldc, int acc, void* part, const Groups& groups) {
  using V2 = typename Traits<MODE>::V2;
  k_zgemm_mfma<MODE, NB16, Groups><<<grid, 256, 0, c.stream>>>(M, N, K, kchunk, nsplit, bt.sA, bt.sB, bt.sC, (const V2*)A,
                                                        lda, (const V2*)B, ldb, (V2*)C, ldc, acc, (V2*)part, groups);
}

template <int MODE, class Groups>
void zgemm_mfma_t(Context& c, int M, int N, int K, const void* A, int lda, const void* B, int ldb, void* C, int ldc,
                  bool accumulate, const Batch& bt, const Groups& groups) {
  using V2 = typename Traits<MODE>::V2;
  const int cus = c.cu_count > 0 ? c.cu_count : 256;
  // Column blocks of equal width. Without split K the width whose tiles, dealt to the CUs, take the fewest
  // steps on the busiest CU (half a block stands for what a tile costs besides its MFMAs), narrower on a tie.
  const int n16 = (N + 15) / 16, mt = (M + BMC - 1) / BMC;
  auto balanced = [&](int w) {
    const int blocks = (n16 + w - 1) / w;
    return (n16 + blocks - 1) / blocks;
  };
  auto tiles_of = [&](int w) { return (long)mt * ((n16 + w - 1) / w) * bt.count; };
  auto cost = [&](int w) { return (double)((tiles_of(w) + cus - 1) / cus) * (w + 0.5); };
  int nb16 = balanced(Tile<MODE>::W), nsplit = 1;
  // split K only for K >= 256 (short reductions are cheaper than the extra partial-sum pass) and
  // when the tiles fill less than half the CUs (above that the partial-sum round trip costs
  // more than the idle CUs), into chunks of at least 4 steps and no more workgroups than run at once;
  // tiles narrower where even so the CUs are not all busy (64 × 40 × 1921: 10 us instead of 15)
  if (tiles_of(nb16) < cus / 2 && K >= 16 * BKC) {
    const int most = std::max(1, K / (4 * BKC));
    while (nb16 > 1 && tiles_of(nb16) * most < cus) nb16 = balanced(nb16 - 1);
    nsplit = (int)std::min<long>(std::max<long>(1, cus * Tile<MODE>::PER_CU / tiles_of(nb16)), most);
  } else {
    for (int w = Tile<MODE>::W; w >= 1; --w)
      if (cost(balanced(w)) <= cost(nb16)) nb16 = balanced(w);
  }
  const int BN = 16 * nb16, nt = (N + BN - 1) / BN;
  int kchunk = (K + nsplit - 1) / nsplit;
  kchunk = ((kchunk + 2 * BKC - 1) / (2 * BKC)) * (2 * BKC);
  nsplit = (K + kchunk - 1) / kchunk;
  PWK_REQUIRE((long)nsplit * bt.count <= 65535, PWK_E_UNSUPPORTED, "GEMM batch too large");
  PWK_REQUIRE((long)mt * nt * nsplit * bt.count <= 0x7fffffffL, PWK_E_UNSUPPORTED, "GEMM grid too large");
  dim3 grid((unsigned)((long)mt * nt * nsplit * bt.count));
  void* part = nullptr;
  if (nsplit > 1) {
    c.workspace(c.gemm_ws, (size_t)bt.count * nsplit * M * N * sizeof(V2));
    part = c.gemm_ws.p;
  }
  int acc = (nsplit == 1 && accumulate) ? 1 : 0;
  switch (nb16) {
    case 1:
      launch_nb<MODE, 1>(c, grid, M, N, K, kchunk, nsplit, bt, A, lda, B, ldb, C, ldc, acc, part, groups);
      break;
    case 2:
      launch_nb<MODE, 2>(c, grid, M, N, K, kchunk, nsplit, bt, A, lda, B, ldb, C, ldc, acc, part, groups);
      break;
    default:
      launch_nb<MODE, Tile<MODE>::W>(c, grid, M, N, K, kchunk, nsplit, bt, A, lda, B, ldb, C, ldc, acc, part, groups);
      break;
  }
  PWK_HIP(hipGetLastError());
  if (nsplit > 1) {
    dim3 g(blocks_for((size_t)M * N, 256), (unsigned)bt.count);
    k_splitk_sum<V2, Groups><<<g, 256, 0, c.stream>>>(M, N, nsplit, (const V2*)part, (V2*)C, ldc, bt.sC,
                                              accumulate ? 1 : 0, groups);
    PWK_HIP(hipGetLastError());
  }
}

}  // namespace

void launch_zgemm_mfma(Context& c, int M, int N, int K, const void* A, int lda, const void* B, int ldb, void* C,
                       int ldc, bool accumulate, int precision) {
  launch_zgemm_mfma_batched(c, M, N, K, A, lda, 0, B, ldb, 0, C, ldc, 0, 1, accumulate, precision);
}

void launch_zgemm_mfma_batched(Context& c, int M, int N, int K, const void* A, int lda, long long sA, const void* B,
                               int ldb, long long sB, void* C, int ldc, long long sC, int batch, bool accumulate,
                               int precision) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  if (K <= 0) {
    PWK_REQUIRE(accumulate, PWK_E_INVALID, "zgemm with K = 0 and no accumulation");
    return;
  }
  Batch bt;
  bt.count = batch;
  bt.sA = sA;
  bt.sB = sB;
  bt.sC = sC;
  if (precision == PWK_FP64)
    zgemm_mfma_t<MODE_F64>(c, M, N, K, A, lda, B, ldb, C, ldc, accumulate, bt, NoBatch{});
  else if (precision == PWK_SPLIT_BF16)
    zgemm_mfma_t<MODE_BF16X3>(c, M, N, K, A, lda, B, ldb, C, ldc, accumulate, bt, NoBatch{});
  else
    zgemm_mfma_t<MODE_F32>(c, M, N, K, A, lda, B, ldb, C, ldc, accumulate, bt, NoBatch{});
}

template <int CAP>
void launch_zgemm_mfma_groups(Context& c, int M, int Nmax, int K, const GemmGroups<CAP>& groups, int lda, const void* B,
                              int ldb, void* C, int ldc, bool accumulate, int precision) {
  if (M <= 0 || Nmax <= 0 || K <= 0 || groups.n <= 0) return;
  Batch bt;
  bt.count = groups.n;
  if (precision == PWK_FP64)
    zgemm_mfma_t<MODE_F64>(c, M, Nmax, K, nullptr, lda, B, ldb, C, ldc, accumulate, bt, groups);
  else if (precision == PWK_SPLIT_BF16)
    zgemm_mfma_t<MODE_BF16X3>(c, M, Nmax, K, nullptr, lda, B, ldb, C, ldc, accumulate, bt, groups);
  else
    zgemm_mfma_t<MODE_F32>(c, M, Nmax, K, nullptr, lda, B, ldb, C, ldc, accumulate, bt, groups);
}

template void launch_zgemm_mfma_groups(Context&, int, int, int, const GemmGroups<FEW_BATCH_ENTRIES>&, int, const void*, int,
                                       void*, int, bool, int);
template void launch_zgemm_mfma_groups(Context&, int, int, int, const GemmGroups<MAX_BATCH_ENTRIES>&, int, const void*, int,
                                       void*, int, bool, int);

}  // namespace pwk
