// Batched task kernels of the H-LLt factorisation and the H-triangular solves.
// Each launch processes the tasks of one type in one dependency wave; the
// tasks of a launch are independent.  GEMM, LDLt, acaFull and the elementwise
// tasks run in the storage type T (FP64 or FP32); POTRF and GETRF of leaves of up
// to 128 rows, TRSM and the QR / SVD of the recompressions in FP64.
#include "dev_linalg.hpp"
#include "dev_panel.hpp"
#include "factor_kernels.hpp"

namespace hmx {

namespace {

__device__ inline int eff(const Dim& d) {
  if (d.d == nullptr) return d.s;
  const int v = *d.d;
  return v < d.s ? v : d.s;
}
__device__ inline int rank_of(const RkRef& r) {
  const int v = *r.rank;
  return v < r.cap ? v : r.cap;
}

// 16 x 16 x 4 matrix-core products in FP64 and FP32.  D[i][j] is returned to
// lane j + 16 (i mod 4) as element i / 4 in FP64, to lane j + 16 (i / 4) as
// element i mod 4 in FP32.
template <typename T>
struct MfmaAcc;
template <>
struct MfmaAcc<double> {
  typedef double type __attribute__((ext_vector_type(4)));
  __device__ static int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <>
struct MfmaAcc<float> {
  typedef float type __attribute__((ext_vector_type(4)));
  __device__ static int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};
__device__ inline MfmaAcc<double>::type mfma16x16x4(double a, double b, MfmaAcc<double>::type c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline MfmaAcc<float>::type mfma16x16x4(float a, float b, MfmaAcc<float>::type c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// f(0), ..., f(N - 1) with compile-time indices (register arrays)
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// ---------------------------------------------------------------------------
// GEMM: C (m x n, ldc) = beta C + alpha op(A) op(B), 64 x 64 tiles.  Bound in the
// factorisation's launches (98-row leaves, some 200 tiles): latency, of the
// flag, tile, task and operands and then of each k-step.  With C read entry by
// entry after the products, its columns across the lanes, and transposed
// operands gathered, a launch averaged 13.0 us (40,000 points, FP32) and 16.3 us
// (8,000 points), now 10.8 and 12.4 us.
// ---------------------------------------------------------------------------
constexpr int TM = 64, TN = 64, TK = 32;
static_assert(TM == TN, "one tile side");

// Products with a side of at most 32 (the right-hand sides of a solve, a rank) or
// all of a leaf's size, in launches of few tiles, are bound by the latency of
// their loads: a workgroup takes a 32 x 32 tile, its wavefronts a quarter of the
// inner dimension each with 32 or 64 steps' operands in flight straight into the
// matrix-core layout, and the four partial tiles meet in LDS.  Larger products
// and launches share operands through LDS (k_gemm's 64 x 64 tiles).
// Where the line lies, 64 x 64 tiles against these, by the launch's number of
// 64 x 64 tiles: up to 16 9.8 against 5.3 us (6,000 points, FP64), 65 to 128
// 10.2 against 6.9 us, 513 to 1,024 17.6 against 15.1 us, 1,025 to 2,048 24.4
// against 27.6 us, above 4,096 71 against 142 us (40,000 points, FP32).
constexpr int kThin = 32, kThinSide = 256, kThinLaunch = 1024;
inline bool gemm_is_thin(const FTask& t) {
  const int m = t.m.s, n = t.n.s;
  return m <= kThin || n <= kThin || (m <= kThinSide && n <= kThinSide && t.p.s <= kThinSide);
}

// sh: 4096 entries
template <typename T>
__device__ __forceinline__ void gemm_thin(const FTask& t, int i0, int j0, int M, int N, int P, T* sh) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const long sia = t.ta ? (long)t.lda : 1L, ska = t.ta ? 1L : (long)t.lda;
  const long sib = t.tb ? 1L : (long)t.ldb, skb = t.tb ? (long)t.ldb : 1L;
  const int mi = M - i0 < kThin ? M - i0 : kThin, nj = N - j0 < kThin ? N - j0 : kThin;
  const bool two_a = mi > 16, two_b = nj > 16;
  cgptr<T> pa[2], pb[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int i = 16 * a + li;
    pa[a] = (cgptr<T>)t.A + (i0 + (i < mi ? i : mi - 1)) * sia;
    pb[a] = (cgptr<T>)t.B + (j0 + (i < nj ? i : nj - 1)) * sib;
  }
  // thread (w, lane) finishes entry (16 a + li, 16 b + row(lane, w)) of each 16 x 16
  // tile: C in flight during the products
  const auto C0 = (gptr<T>)t.C + i0 + (size_t)j0 * t.ldc;
  const bool add = t.mode != 0;
  const int jr = MfmaAcc<T>::row(lane, w);
  T old[2][2];
  if (add) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int i = 16 * a + li, j = 16 * b + jr;
        old[a][b] = C0[(i < mi ? i : mi - 1) + (size_t)(j < nj ? j : nj - 1) * t.ldc];
      }
  }
  using Acc = typename MfmaAcc<T>::type;
  Acc acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = Acc{0, 0, 0, 0};
  // lane group lk takes the inner indices 16 s + 4 lk + e, e = 0..3: a lane's four
  // loads are neighbours where the inner index runs along memory
  constexpr int kB = sizeof(T) == 4 ? 4 : 2;  // groups of 16 in flight
  const int chunk = (P + 63) / 64 * 16;
  const int lo = w * chunk, hi = lo + chunk < P ? lo + chunk : P;
  for (int k0 = lo; k0 < hi; k0 += 16 * kB) {
    T fa[2][4 * kB], fb[2][4 * kB];
#pragma unroll
    for (int q = 0; q < 4 * kB; ++q) {
      const int k = k0 + 16 * (q / 4) + 4 * lk + q % 4, kc = k < hi ? k : hi - 1;
      fa[0][q] = pa[0][kc * ska];
      fb[0][q] = pb[0][kc * skb];
    }
    if (two_a) {
#pragma unroll
      for (int q = 0; q < 4 * kB; ++q) {
        const int k = k0 + 16 * (q / 4) + 4 * lk + q % 4;
        fa[1][q] = pa[1][(k < hi ? k : hi - 1) * ska];
      }
    }
    if (two_b) {
#pragma unroll
      for (int q = 0; q < 4 * kB; ++q) {
        const int k = k0 + 16 * (q / 4) + 4 * lk + q % 4;
        fb[1][q] = pb[1][(k < hi ? k : hi - 1) * skb];
      }
    }
#pragma unroll
    for (int q = 0; q < 4 * kB; ++q) {
      const bool in = k0 + 16 * (q / 4) + 4 * lk + q % 4 < hi;
      const T a0 = in ? fa[0][q] : (T)0, b0 = in ? fb[0][q] : (T)0;
      acc[0][0] = mfma16x16x4(b0, a0, acc[0][0]);
      if (two_a) acc[1][0] = mfma16x16x4(b0, in ? fa[1][q] : (T)0, acc[1][0]);
      if (two_b) {
        const T b1 = in ? fb[1][q] : (T)0;
        acc[0][1] = mfma16x16x4(b1, a0, acc[0][1]);
        if (two_a) acc[1][1] = mfma16x16x4(b1, in ? fa[1][q] : (T)0, acc[1][1]);
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v) sh[((w * 2 + a) * 2 + b) * 256 + v * 64 + lane] = acc[a][b][v];
  __syncthreads();
  const T alpha = (T)t.alpha;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      T x = (T)0;
#pragma unroll
      for (int q = 0; q < 4; ++q) x += sh[((q * 2 + a) * 2 + b) * 256 + threadIdx.x];
      x *= alpha;
      const int i = 16 * a + li, j = 16 * b + jr;
      if (i < mi && j < nj) C0[i + (size_t)j * t.ldc] = add ? old[a][b] + x : x;
    }
}

template <typename T>
__global__ void __launch_bounds__(256) k_gemm(const FTask* tasks, const GemmTile* tiles,
                                              const int* fail) {
  __shared__ T sh[2 * TK * (TM + 1)];
  auto& As = *(T(*)[TK][TM + 1])sh;
  auto& Bs = *(T(*)[TK][TN + 1])(sh + TK * (TM + 1));
  const int failed = *fail;  // in flight together with the tile and the task
  const GemmTile tl = tiles[blockIdx.x];
  const FTask& t = tasks[tl.task];
  const int M = eff(t.m), N = eff(t.n), P = eff(t.p);
  const bool thin = tl.tm < 0;
  const int i0 = thin ? ~tl.tm * kThin : tl.tm * TM, j0 = tl.tn * (thin ? kThin : TN);
  if ((failed != 0) | (i0 >= M) | (j0 >= N)) return;
  if (thin) {
    gemm_thin<T>(t, i0, j0, M, N, P, sh);
    return;
  }
  const auto A = (cgptr<T>)t.A;
  const auto B = (cgptr<T>)t.B;
  const auto C = (gptr<T>)t.C;
  // wavefront w computes the 32 x 32 quadrant (w & 1, w >> 1) of the tile as
  // 2 x 2 matrix-core tiles of 16 x 16, transposed (op(B)^T is the A operand), so
  // that 16 lanes hold 16 rows of a column of C
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int qi = (w & 1) * 32, qj = (w >> 1) * 32;
  using Acc = typename MfmaAcc<T>::type;
  Acc acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = Acc{0, 0, 0, 0};
  // As[kk][ii] = op(A)(i0 + ii, k0 + kk), Bs[kk][jj] = op(B)(k0 + kk, j0 + jj):
  // each thread loads 8 + 8 entries of a k-step into registers; the loads of
  // step k0 + TK are in flight while step k0 is multiplied (two steps ahead cost
  // a wavefront per SIMD and made large launches 2.5 times slower).  Consecutive lanes
  // take consecutive addresses: rows of the tile, or its k when the stored
  // matrix is the transpose.  The loads read a clamped entry and select.
  constexpr int kPer = TM * TK / 256;
  const int mi = M - i0 < TM ? M - i0 : TM, nj = N - j0 < TN ? N - j0 : TN;
  const bool ka = t.ta, kb = !t.tb;  // k runs along the lanes
  const int ia = ka ? threadIdx.x / TK : threadIdx.x % TM, ja = ka ? threadIdx.x % TK : threadIdx.x / TM;
  const int ib = kb ? threadIdx.x / TK : threadIdx.x % TN, jb = kb ? threadIdx.x % TK : threadIdx.x / TN;
  const int dia = ka ? 256 / TK : 0, dja = ka ? 0 : 256 / TM;
  const int dib = kb ? 256 / TK : 0, djb = kb ? 0 : 256 / TN;
  const long la = t.lda, lb = t.ldb;
  const long sia = ka ? la : 1, ska = ka ? 1 : la, sib = kb ? lb : 1, skb = kb ? 1 : lb;
  const auto A0 = A + i0 * sia;
  const auto B0 = B + j0 * sib;
  T ra[kPer], rb[kPer];
  auto load_step = [&](int k0) __attribute__((always_inline)) {
    const int pk = P - k0 < TK ? P - k0 : TK;
    const auto Ak = A0 + k0 * ska;
    const auto Bk = B0 + k0 * skb;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = ia + u * dia, j = ja + u * dja;
      ra[u] = Ak[(i < mi ? i : mi - 1) * sia + (j < pk ? j : pk - 1) * ska];
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = ib + u * dib, j = jb + u * djb;
      rb[u] = Bk[(i < nj ? i : nj - 1) * sib + (j < pk ? j : pk - 1) * skb];
    }
  };
  if (P > 0) load_step(0);
  // C is in flight during the products
  const auto C0 = C + i0 + (size_t)j0 * t.ldc;
  const bool add = t.mode != 0;
  T old[2][2][4];
  if (add) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = qi + 16 * a + li, j = qj + 16 * b + MfmaAcc<T>::row(lane, v);
          old[a][b][v] = C0[(i < mi ? i : mi - 1) + (size_t)(j < nj ? j : nj - 1) * t.ldc];
        }
  }
  for (int k0 = 0; k0 < P; k0 += TK) {
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = ia + u * dia, j = ja + u * dja, ii = ib + u * dib, jj = jb + u * djb;
      As[j][i] = i < mi && k0 + j < P ? ra[u] : (T)0;
      Bs[jj][ii] = ii < nj && k0 + jj < P ? rb[u] : (T)0;
    }
    __syncthreads();
    if (k0 + TK < P) load_step(k0 + TK);
#pragma unroll
    for (int kk = 0; kk < TK; kk += 4) {
      T fa[2], fb[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) fa[a] = As[kk + lk][qi + 16 * a + li];
#pragma unroll
      for (int b = 0; b < 2; ++b) fb[b] = Bs[kk + lk][qj + 16 * b + li];
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = mfma16x16x4(fb[b], fa[a], acc[a][b]);
    }
    __syncthreads();
  }
  const T alpha = (T)t.alpha;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = qi + 16 * a + li, j = qj + 16 * b + MfmaAcc<T>::row(lane, v);
        const T x = alpha * acc[a][b][v];
        if (i < mi && j < nj) C0[i + (size_t)j * t.ldc] = add ? old[a][b][v] + x : x;
      }
}

// ---------------------------------------------------------------------------
// POTRF (lower).  Leaves of up to kLdsDense rows are factorised in LDS in FP64
// (potrf_lds), larger ones and the HODLR node blocks in global memory in the
// type they have (potrf_body).
// ---------------------------------------------------------------------------
constexpr int kLdsDense = 128;

constexpr int kNb = 16;  // panel width of the blocked POTRF / TRSM
constexpr int kTrsmCols = 64;  // independent rows / columns of a TRSM tile: 16 per wavefront
// entries of a tile of the elementwise tasks (ZERO, AXPY, SUMK): one workgroup
// per task left a 2,048 x 2,048 identity at 590 us and the sum of 8 slices of
// 2,048 x 65 at 535 us, with 255 CUs idle
constexpr int kElemsPerTile = 2048;

// Right-looking blocked Cholesky in global memory: each 16-column panel is
// factorised left-looking (one thread per row, short dots over the panel only, two
// barriers per column), then the trailing lower triangle gets the panel's rank-16
// update with all threads.
template <typename T>
__device__ void potrf_body(T* L, int ld, int n, int* info) {
  for (int jb = 0; jb < n; jb += kNb) {
    const int je = jb + kNb < n ? jb + kNb : n;
    for (int j = jb; j < je; ++j) {
      for (int i = j + threadIdx.x; i < n; i += kBlock) {
        // the panel's earlier columns: a fixed 16 terms with a mask, so that
        // their loads issue together (column indices clamped into the matrix)
        T s = L[i + (size_t)j * ld];
#pragma unroll
        for (int q = 0; q < kNb; ++q) {
          const int l = jb + q < n ? jb + q : n - 1;
          const T a = L[i + (size_t)l * ld], b = L[j + (size_t)l * ld];
          s -= (jb + q < j) ? a * b : (T)0;
        }
        L[i + (size_t)j * ld] = s;
      }
      __syncthreads();
      const T d = L[j + (size_t)j * ld];
      const T piv = sqrt(d);
      for (int i = j + 1 + threadIdx.x; i < n; i += kBlock) L[i + (size_t)j * ld] /= piv;
      __syncthreads();
      if (threadIdx.x == 0) {
        if (!(d > (T)0)) atomicOr(info, 1);
        L[j + (size_t)j * ld] = piv;
      }
    }
    __syncthreads();
    const int r = n - je;
    for (int e = threadIdx.x; e < r * r; e += kBlock) {
      const int i = je + e % r, c = je + e / r;
      if (c > i) continue;
      T s = 0;
#pragma unroll
      for (int q = 0; q < kNb; ++q) {
        const int l = jb + q < n ? jb + q : n - 1;
        const T a = L[i + (size_t)l * ld], b = L[c + (size_t)l * ld];
        s += (jb + q < je) ? a * b : (T)0;
      }
      L[i + (size_t)c * ld] -= s;
    }
    __syncthreads();
  }
}

// Reciprocal, quotient and square root for the serial chains of the leaf
// factorisations: hardware estimates with Newton / Goldschmidt steps and
// Markstein's final corrections (P. Markstein, IBM J. Res. Dev. 34, 1990), a
// power of two taken out first.  About a third of the dependent steps of the
// library forms.
__device__ inline double chain_rcp(double d) {
  const int e = __builtin_amdgcn_frexp_exp(d);
  const double s = __builtin_amdgcn_ldexp(d, -e);
  double y = __builtin_amdgcn_rcp(s);
  y = fma(fma(-s, y, 1.0), y, y);
  y = fma(fma(-s, y, 1.0), y, y);
  return fabs(d) <= 1.79e308 ? __builtin_amdgcn_ldexp(y, -e) : 1.0 / d;
}
// A power of two that brings a divisor whose reciprocal is above the largest
// finite number (below 5.6e-309) into range: a / d = (a up) / (d up).
__device__ inline double chain_up(double d) { return fabs(d) < 0x1p-1000 ? 0x1p+500 : 1.0; }
// a / d with y = 1 / d: the product corrected by its remainder (a == d gives 1)
__device__ inline double chain_div(double a, double d, double y) {
  const double q = a * y;
  return fabs(d) <= 1.79e308 ? fma(fma(-q, d, a), y, q) : q;
}
// sqrt(d)
__device__ inline double chain_sqrt(double d) {
  const int e = __builtin_amdgcn_frexp_exp(d) & ~1;
  const double s = __builtin_amdgcn_ldexp(d, -e);
  const double y = __builtin_amdgcn_rsq(s);
  double g = s * y, h = 0.5 * y;
  double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  g = fma(fma(-g, g, s), h, g);
  return (d > 0.0 && d <= 1.79e308) ? __builtin_amdgcn_ldexp(g, e >> 1) : d;
}

// The 16 x 16 tiles t = w, w + 4, ... < count of a trailing update by 16
// columns, four at a time so that their LDS reads and products overlap:
// tile(t, x0, y0) gives the tile's offsets, A(i, k) and B(k, j) the operands'
// entries, and the block itself (ld ld, n x n) is the accumulator.
template <typename FT, typename FA, typename FB>
__device__ inline void panel_update(double* P, int ld, int n, int count, FT tile, FA A, FB B) {
  constexpr int kBatch = 4;
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave, ii = lane & 15, kk = lane >> 4;
  for (int t0 = w; t0 < count; t0 += kBatch * kWaves) {
    int x0[kBatch], y0[kBatch];
    double a[kBatch][4], b[kBatch][4];
    hmx_double4 acc[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int t = t0 + u * kWaves;
      tile(t < count ? t : t0, x0[u], y0[u]);
      const int xr = x0[u] + ii < n ? x0[u] + ii : n - 1, yc = y0[u] + ii < n ? y0[u] + ii : n - 1;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        a[u][q] = -A(xr, 4 * q + kk);
        b[u][q] = B(4 * q + kk, yc);
        const int i = x0[u] + kk + 4 * q;
        acc[u][q] = P[(i < n ? i : n - 1) + yc * ld];
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int u = 0; u < kBatch; ++u) acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][q], b[u][q], acc[u], 0, 0, 0);
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = x0[u] + kk + 4 * v, j = y0[u] + ii;
        if (t0 + u * kWaves < count && i < n && j < n) P[i + j * ld] = acc[u][v];
      }
  }
}

// n x n (n <= 128) between global memory (ld lda) and LDS (ld n): a wavefront
// per column, no index divisions, 16 columns' loads in flight.
template <typename T>
__device__ inline void leaf_in(double* L, cgptr<T> A, int lda, int n) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  constexpr int kC = 16;
  const int i1 = lane < n ? lane : n - 1, i2 = lane + kWave < n ? lane + kWave : n - 1;
  for (int j0 = w; j0 < n; j0 += kC * kWaves) {
    T v[kC][2];
#pragma unroll
    for (int c = 0; c < kC; ++c) {
      const int j = j0 + kWaves * c < n ? j0 + kWaves * c : n - 1;
      v[c][0] = A[(size_t)j * lda + i1];
      v[c][1] = A[(size_t)j * lda + i2];
    }
#pragma unroll
    for (int c = 0; c < kC; ++c) {
      const int j = j0 + kWaves * c;
      if (j >= n) continue;
      if (lane < n) L[j * n + lane] = (double)v[c][0];
      if (lane + kWave < n) L[j * n + lane + kWave] = (double)v[c][1];
    }
  }
}
template <typename T>
__device__ inline void leaf_out(gptr<T> A, int lda, const double* L, int n, bool lower) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll 4
  for (int j = w; j < n; j += kWaves)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int i = lane + kWave * h;
      if (i < n) A[(size_t)j * lda + i] = (lower && i < j) ? (T)0 : (T)L[j * n + i];
    }
}

// Blocked Cholesky of a leaf of at most 128 rows in LDS (FP64).  Per 16
// columns: the diagonal block on one wavefront with a row per lane in registers
// (the other lanes' entries by readlane: no LDS round trip and no barrier in its
// 16 steps), in the square-root-free form, so that a step's chain is one
// reciprocal, the roots being taken for all 16 columns at once; the rows below
// by one thread each with the block's multipliers; the trailing lower triangle
// on the matrix cores.  Bound: the chain of reciprocals and rank-1 steps of the
// diagonal blocks.  125 rows: 244 us (FP64) and 167 us (FP32 storage) with a column
// per step of the whole workgroup, 90 us now.
__device__ void potrf_lds(double* L, int ld, int n, int* info) {
  __shared__ double mult[kNb * kNb];  // a_cj / d_j at c + 16 j
  __shared__ double root[kNb], rroot[kNb];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave, i = lane & 15;
  for (int r0 = 0; r0 < n; r0 += kNb) {
    const int bs = n - r0 < kNb ? n - r0 : kNb;
    if (w == 0) {
      double a[kNb];
      const int ir = r0 + (i < bs ? i : bs - 1);
#pragma unroll
      for (int c = 0; c < kNb; ++c) {
        const double v = L[ir + (r0 + (c < bs ? c : bs - 1)) * ld];
        a[c] = (i < bs && c < bs) ? v : (i == c ? 1.0 : 0.0);
      }
      bool bad = false;
      double diag = 1.0;
      static_for<0, kNb>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        const double d = lane_read(a[j], j);
        bad |= !(d > 0.0);
        diag = i == j ? a[j] : diag;
        const double up = chain_up(d);
        const double m = (a[j] * up) * chain_rcp(d * up);
        if (lane < kNb) mult[i + kNb * j] = m;
#pragma unroll
        for (int c = j + 1; c < kNb; ++c) a[c] -= m * lane_read(a[j], c);
      });
      if (bad && lane == 0) atomicOr(info, 1);
      const double p = chain_sqrt(diag), y = chain_rcp(p);
      if (lane < kNb) {
        root[i] = p;
        rroot[i] = y;
      }
#pragma unroll
      for (int c = 0; c < kNb; ++c) {
        const double pc = lane_read(p, c), l = i == c ? pc : chain_div(a[c], pc, lane_read(y, c));
        if (lane < bs && c <= i) L[r0 + i + (r0 + c) * ld] = l;
      }
    }
    __syncthreads();
    const int below = n - r0 - kNb;
    if (below <= 0) break;
    if ((int)threadIdx.x < below) {
      double* row = L + r0 + kNb + threadIdx.x + r0 * ld;
      double x[kNb];
#pragma unroll
      for (int c = 0; c < kNb; ++c) x[c] = row[c * ld];
      static_for<0, kNb>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
#pragma unroll
        for (int c = j + 1; c < kNb; ++c) x[c] -= x[j] * mult[c + kNb * j];
      });
#pragma unroll
      for (int c = 0; c < kNb; ++c) row[c * ld] = chain_div(x[c], root[c], rroot[c]);
    }
    __syncthreads();
    const int nt = (below + kNb - 1) / kNb;
    panel_update(
        L, ld, n, nt * (nt + 1) / 2,
        [&](int t, int& x0, int& y0) {
          int tj = 0;
          while (t >= nt - tj) t -= nt - tj++;
          x0 = r0 + kNb * (tj + t + 1);
          y0 = r0 + kNb * (tj + 1);
        },
        [&](int r, int k) { return L[r + (r0 + k) * ld]; }, [&](int k, int c) { return L[c + (r0 + k) * ld]; });
    __syncthreads();
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_potrf(const FTask* tasks, int* info) {
  __shared__ double lds[kLdsDense * kLdsDense];
  const FTask& t = tasks[blockIdx.x];
  const int n = t.m.s;
  T* A = (T*)t.A;
  const int lda = t.lda;
  if (n <= kLdsDense) {
    leaf_in<T>(lds, (cgptr<T>)A, lda, n);
    __syncthreads();
    potrf_lds(lds, n, n, info);
    __syncthreads();
    leaf_out<T>((gptr<T>)A, lda, lds, n, true);
  } else {
    potrf_body(A, lda, n, info);
    for (int e = threadIdx.x; e < n * n; e += kBlock) {
      const int i = e % n, j = e / n;
      if (i < j) A[i + (size_t)j * lda] = (T)0;
    }
  }
}

// ---------------------------------------------------------------------------
// LDLt of a diagonal leaf (ScalarArray::ldltDecomposition scalar_array.cpp:
// 737-779): A = L D L^T in place, L unit lower with its diagonal set to 1 and
// the upper triangle zeroed, D into d.  Left-looking, one column per step:
// d_j = a_jj - sum_l l_jl^2 d_l, l_ij = (a_ij - sum_l l_il l_jl d_l) / d_j.
// A zero or non-finite pivot sets info (the reference throws).
// ---------------------------------------------------------------------------
template <typename T>
__device__ void ldlt_body(T* L, int ld, int n, T* d, int* info) {
  for (int j = 0; j < n; ++j) {
    for (int i = j + threadIdx.x; i < n; i += kBlock) {
      T s = L[i + (size_t)j * ld];
      for (int l = 0; l < j; ++l) s -= L[i + (size_t)l * ld] * (L[j + (size_t)l * ld] * d[l]);
      L[i + (size_t)j * ld] = s;
    }
    __syncthreads();
    const T dj = L[j + (size_t)j * ld];
    const T inv = (T)1 / dj;
    for (int i = j + 1 + threadIdx.x; i < n; i += kBlock) L[i + (size_t)j * ld] *= inv;
    __syncthreads();
    if (threadIdx.x == 0) {
      if (!(dj != (T)0) || !isfinite((double)dj)) atomicOr(info, 1);
      d[j] = dj;
      L[j + (size_t)j * ld] = (T)1;
    }
    __syncthreads();
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_ldlt(const FTask* tasks, int* info) {
  __shared__ T lds[kLdsDense * kLdsDense];
  __shared__ T dl[kLdsDense];
  const FTask& t = tasks[blockIdx.x];
  const int n = t.m.s;
  T* A = (T*)t.A;
  T* D = (T*)t.B;
  const int lda = t.lda;
  if (n <= kLdsDense) {
    stage_in(lds, n, (cgptr<T>)A, 1L, (long)lda, n, n);
    __syncthreads();
    ldlt_body(lds, n, n, dl, info);
    for (int e = threadIdx.x; e < n * n; e += kBlock) {
      const int i = e % n, j = e / n;
      A[i + (size_t)j * lda] = (i >= j) ? lds[i + j * n] : (T)0;
    }
    for (int i = threadIdx.x; i < n; i += kBlock) D[i] = dl[i];
  } else {
    ldlt_body(A, lda, n, D, info);
    for (int e = threadIdx.x; e < n * n; e += kBlock) {
      const int i = e % n, j = e / n;
      if (i < j) A[i + (size_t)j * lda] = (T)0;
    }
  }
}

// C = A times a diagonal (ScalarArray::multiplyWithDiagOrDiagInv
// scalar_array.cpp:1434-1470): the columns (kDscaleCols) or the rows of A
// scaled by d or, with kDscaleInv, by 1 / d.  A may be C.  kDscaleSplit
// workgroups share a task.
constexpr int kDscaleSplit = 8;
template <typename T>
__global__ void k_dscale(const FTask* tasks, const int* fail) {
  if (*fail) return;
  const FTask& t = tasks[blockIdx.x / kDscaleSplit];
  const int part = blockIdx.x % kDscaleSplit;
  const auto A = (cgptr<T>)t.A;
  const auto d = (cgptr<T>)t.B;
  const auto C = (gptr<T>)t.C;
  const int m = eff(t.m), n = eff(t.n);
  const bool cols = t.mode & kDscaleCols, inv = t.mode & kDscaleInv;
  const int64_t total = (int64_t)m * n;
  for (int64_t e = part * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)kDscaleSplit * blockDim.x) {
    const int i = (int)(e % m), j = (int)(e / m);
    const T f = d[cols ? j : i];
    C[i + (size_t)j * t.ldc] = A[i + (size_t)j * t.lda] * (inv ? (T)1 / f : f);
  }
}

// ---------------------------------------------------------------------------
// GETRF of a diagonal leaf (ScalarArray::luDecomposition, scalar_array.cpp:
// 694-705): A = P L U in place, L unit lower, U upper, partial pivoting as
// LAPACK getrf (pivot = first row of largest |a_ij| in the column), 0-based
// interchanges into piv[0..n).  A zero or non-finite pivot sets info (the
// reference throws on getrf's info > 0).  Right-looking, one column per step.
// ---------------------------------------------------------------------------
template <typename T>
__device__ void getrf_body(T* P, int ld, int n, int* piv, int* info) {
  __shared__ int pv;
  const int lane = threadIdx.x & (kWave - 1);
  for (int j = 0; j < n; ++j) {
    if (threadIdx.x < kWave) {
      double best = -1.0;
      int bi = n;
      for (int i = j + lane; i < n; i += kWave) {
        const double v = fabs((double)P[i + (size_t)j * ld]);
        if (v > best) {
          best = v;
          bi = i;
        }
      }
      for (int o = kWave / 2; o > 0; o >>= 1) {
        const double ob = __shfl_xor(best, o, kWave);
        const int oi = __shfl_xor(bi, o, kWave);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      if (bi >= n) bi = j;  // column of NaNs: keep the row, the pivot test below fails
      if (lane == 0) {
        pv = bi;
        piv[j] = bi;
      }
    }
    __syncthreads();
    const int p = pv;
    if (p != j)
      for (int c = threadIdx.x; c < n; c += kBlock) {
        const T a = P[j + (size_t)c * ld];
        P[j + (size_t)c * ld] = P[p + (size_t)c * ld];
        P[p + (size_t)c * ld] = a;
      }
    __syncthreads();
    const double d = (double)P[j + (size_t)j * ld];
    if (d == 0.0 || !isfinite(d)) {
      if (threadIdx.x == 0) atomicOr(info, 1);
      return;
    }
    for (int i = j + 1 + threadIdx.x; i < n; i += kBlock) P[i + (size_t)j * ld] = (T)((double)P[i + (size_t)j * ld] / d);
    __syncthreads();
    const int r = n - j - 1;
    for (int e = threadIdx.x; e < r * r; e += kBlock) {
      const int i = j + 1 + e % r, c = j + 1 + e / r;
      P[i + (size_t)c * ld] -= P[i + (size_t)j * ld] * P[j + (size_t)c * ld];
    }
    __syncthreads();
  }
}

// Blocked LU of a leaf of at most 128 rows in LDS (FP64), the same pivots.  Per
// 16 columns: the panel on one wavefront with two rows per lane in registers;
// rows stay where they are and carry their position (the interchanges move
// positions), the pivot row reaches the others by readlane, so a step has no
// barrier.  Then the interchanges on the other columns and the 16 rows of U by
// one thread per column, and the trailing block on the matrix cores.  Bound:
// the chain of pivot searches and divisions.  94 rows in FP64: 231 us with a
// column per step of the whole workgroup, 127 us now.
__device__ void getrf_lds(double* P, int ld, int n, int* piv, int* info) {
  __shared__ int swap[kNb];
  __shared__ int from[2 * kWave];  // the row that the panel's interchanges bring to a position
  __shared__ int stop;
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  if (threadIdx.x == 0) stop = 0;
  __syncthreads();
  for (int r0 = 0; r0 < n; r0 += kNb) {
    const int bs = n - r0 < kNb ? n - r0 : kNb, rows = n - r0;
    if (w == 0) {
      // rows r0 + lane + 64 h, columns r0 .. r0 + bs
      double a[2][kNb];
      int pos[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        pos[h] = lane + kWave * h;
        const int r = r0 + (pos[h] < rows ? pos[h] : rows - 1);
#pragma unroll
        for (int c = 0; c < kNb; ++c) a[h][c] = P[r + (r0 + (c < bs ? c : bs - 1)) * ld];
      }
      bool fail = false;
      static_for<0, kNb>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        if (j >= bs || fail) return;
        // largest |a_ij| among the rows at positions >= j, the first of equals
        double v[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const bool in = pos[h] >= j && pos[h] < rows;
          const double x = fabs(a[h][j]);
          v[h] = (in && x == x) ? x : -1.0;
        }
        double m = v[0] > v[1] ? v[0] : v[1];
        m = fmax(m, dpp_swap<0xB1>(m));
        m = fmax(m, dpp_swap<0x4E>(m));
        m = fmax(m, dpp_swap<0x141>(m));
        m = fmax(m, dpp_swap<0x140>(m));
        m = fmax(fmax(lane_read(m, 0), lane_read(m, 16)), fmax(lane_read(m, 32), lane_read(m, 48)));
        int pp = 0x7fffffff;  // its position
        uint64_t at0 = __ballot(m >= 0.0 && v[0] == m), at1 = __ballot(m >= 0.0 && v[1] == m);
        if (__popcll(at0) + __popcll(at1) == 1) {
          pp = at0 ? __builtin_amdgcn_readlane(pos[0], __builtin_ctzll(at0))
                   : __builtin_amdgcn_readlane(pos[1], __builtin_ctzll(at1));
        } else {
          for (uint64_t b = at0; b; b &= b - 1) pp = min(pp, __builtin_amdgcn_readlane(pos[0], __builtin_ctzll(b)));
          for (uint64_t b = at1; b; b &= b - 1) pp = min(pp, __builtin_amdgcn_readlane(pos[1], __builtin_ctzll(b)));
          if (pp == 0x7fffffff) pp = j;  // a column of NaNs: the pivot test below fails
        }
        // the lane and half that hold position pp
        const uint64_t w0 = __ballot(pos[0] == pp), w1 = __ballot(pos[1] == pp);
        const bool second = w0 == 0;
        const int src = __builtin_ctzll(second ? w1 : w0);
        double u[kNb];
#pragma unroll
        for (int c = j; c < kNb; ++c) u[c] = second ? lane_read(a[1][c], src) : lane_read(a[0][c], src);
        if (lane == 0) swap[j] = pp;
        const double d = u[j];
        if (d == 0.0 || !isfinite(d)) {
          fail = true;
          return;
        }
        // a quotient and not a product with 1 / d: the multiplier of a row equal to
        // the pivot's is then exactly 1, and a singular leaf ends on an exact zero
        const double up = chain_up(d), du = d * up, y = chain_rcp(du);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // interchange of the positions j and pp
          pos[h] = pos[h] == pp ? j : (pos[h] == j ? pp : pos[h]);
          if (pos[h] > j) {
            const double l = chain_div(a[h][j] * up, du, y);
            a[h][j] = l;
#pragma unroll
            for (int c = j + 1; c < kNb; ++c) a[h][c] -= l * u[c];
          }
        }
      });
      if (fail) {
        if (lane == 0) {
          atomicOr(info, 1);
          stop = 1;
        }
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (lane + kWave * h < rows)
#pragma unroll
            for (int c = 0; c < kNb; ++c)
              if (c < bs) P[r0 + pos[h] + (r0 + c) * ld] = a[h][c];
        if (lane < bs) piv[r0 + lane] = r0 + swap[lane];
        from[pos[0]] = lane;
        from[pos[1]] = lane + kWave;
      }
    }
    __syncthreads();
    if (stop) return;
    // the interchanges on the other columns; right of the panel also
    // U12 = L11^{-1} A12
    const int c = threadIdx.x;
    if (c < n && (c < r0 || c >= r0 + bs)) {
      double* col = P + c * ld + r0;
      // the rows that move are those at positions j < 16 and swap[j]: all loads
      // first, then the stores (equal positions get equal values)
      double x[kNb], z[kNb];
      int at[kNb];
#pragma unroll
      for (int j = 0; j < kNb; ++j) {
        at[j] = swap[j < bs ? j : bs - 1];
        x[j] = col[from[j < bs ? j : bs - 1]];
        z[j] = col[from[at[j]]];
      }
#pragma unroll
      for (int j = 0; j < kNb; ++j) {
        col[at[j]] = z[j];
        if (j < bs) col[j] = x[j];
      }
      if (c >= r0 + bs) {
        // (bs == 16 here)
        const double* blk = P + r0 + r0 * ld;
        static_for<1, kNb>([&](auto J) __attribute__((always_inline)) {
          constexpr int j = decltype(J)::value;
#pragma unroll
          for (int l = 0; l < j; ++l) x[j] -= blk[j + l * ld] * x[l];
          col[j] = x[j];
        });
      }
    }
    __syncthreads();
    const int rest = n - r0 - kNb;
    if (rest <= 0) break;
    const int nt = (rest + kNb - 1) / kNb;
    // an entry takes its 16 terms one after the other, as in the panel and in U:
    // a row that equals an earlier pivot's ends on exact zeros here too
    panel_update(
        P, ld, n, nt * nt,
        [&](int t, int& x0, int& y0) {
          x0 = r0 + kNb * (t % nt + 1);
          y0 = r0 + kNb * (t / nt + 1);
        },
        [&](int r, int k) { return P[r + (r0 + k) * ld]; }, [&](int k, int c) { return P[r0 + k + c * ld]; });
    __syncthreads();
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_getrf(const FTask* tasks, int* info) {
  __shared__ double lds[kLdsDense * kLdsDense];
  const FTask& t = tasks[blockIdx.x];
  const int n = t.m.s;
  T* A = (T*)t.A;
  const int lda = t.lda;
  int* piv = (int*)t.B;
  if (n <= kLdsDense) {
    leaf_in<T>(lds, (cgptr<T>)A, lda, n);
    __syncthreads();
    getrf_lds(lds, n, n, piv, info);
    __syncthreads();
    leaf_out<T>((gptr<T>)A, lda, lds, n, false);
  } else {
    getrf_body(A, lda, n, piv, info);
  }
}

// ---------------------------------------------------------------------------
// The r x r blocks of a symmetric HODLR node (computeSymX11 + computeSymKK,
// hodlr.cpp:163-219, the Gram form the reference selects with
// HMAT_HODLR_NOQR; its default QR form is the same in exact arithmetic).
// With G = a^T a and P = b^T b of the node's transformed Rk block a b^T:
//   La La^T = G,  M11 M11^T = I - La^T P La,  log det M11 into tgt.b,
//   X11 = La^-T (M11 - I) La^-1 into C,  KK = (I + X11 G)^-1 X11 into tgt.a.
// FP64 in the task's workspace (5 r^2 + r values), one workgroup per node.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(kBlock) k_hodlr(const FTask* tasks, double* ws_base, int* info) {
  const FTask& t = tasks[blockIdx.x];
  const int n = eff(t.m), ld = t.lda;
  const T* G = (const T*)t.A;
  const T* P = (const T*)t.B;
  T* X11 = (T*)t.C;
  T* KK = (T*)t.tgt.a;
  double* logdet = (double*)t.tgt.b;
  if (n == 0) {
    if (threadIdx.x == 0) *logdet = 0.0;
    return;
  }
  const size_t nn = (size_t)n * n;
  double* la = ws_base + t.ws;
  double* x = la + nn;
  double* tmp = x + nn;
  double* g = tmp + nn;
  double* y = g + nn;
  int* piv = (int*)(y + nn);
  for (size_t e = threadIdx.x; e < nn; e += kBlock) {
    const int i = (int)(e % n), j = (int)(e / n);
    g[e] = (double)G[i + (size_t)j * ld];
    la[e] = g[e];
    tmp[e] = (double)P[i + (size_t)j * ld];
  }
  __syncthreads();
  potrf_body<double>(la, n, n, info);
  __syncthreads();
  for (size_t e = threadIdx.x; e < nn; e += kBlock)
    if ((int)(e % n) < (int)(e / n)) la[e] = 0.0;
  __syncthreads();
  // x = -P La (La lower)
  for (size_t e = threadIdx.x; e < nn; e += kBlock) {
    const int i = (int)(e % n), j = (int)(e / n);
    double s = 0.0;
    for (int k = j; k < n; ++k) s += tmp[i + (size_t)k * n] * la[k + (size_t)j * n];
    x[e] = -s;
  }
  __syncthreads();
  // tmp = I + La^T x
  for (size_t e = threadIdx.x; e < nn; e += kBlock) {
    const int i = (int)(e % n), j = (int)(e / n);
    double s = 0.0;
    for (int k = i; k < n; ++k) s += la[k + (size_t)i * n] * x[k + (size_t)j * n];
    tmp[e] = s + (i == j ? 1.0 : 0.0);
  }
  __syncthreads();
  potrf_body<double>(tmp, n, n, info);  // M11 in the lower triangle
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int i = 0; i < n; ++i) s += log(tmp[i + (size_t)i * n]);
    *logdet = s;
  }
  // x = M11 - I (lower)
  for (size_t e = threadIdx.x; e < nn; e += kBlock) {
    const int i = (int)(e % n), j = (int)(e / n);
    x[e] = i >= j ? tmp[e] - (i == j ? 1.0 : 0.0) : 0.0;
  }
  __syncthreads();
  // x <- x La^-1 (each row on its own)
  for (int i = threadIdx.x; i < n; i += kBlock)
    for (int j = n - 1; j >= 0; --j) {
      double s = x[i + (size_t)j * n];
      for (int k = j + 1; k < n; ++k) s -= x[i + (size_t)k * n] * la[k + (size_t)j * n];
      x[i + (size_t)j * n] = s / la[j + (size_t)j * n];
    }
  __syncthreads();
  // x <- La^-T x (each column on its own)
  for (int j = threadIdx.x; j < n; j += kBlock)
    for (int i = n - 1; i >= 0; --i) {
      double s = x[i + (size_t)j * n];
      for (int k = i + 1; k < n; ++k) s -= la[k + (size_t)i * n] * x[k + (size_t)j * n];
      x[i + (size_t)j * n] = s / la[i + (size_t)i * n];
    }
  __syncthreads();
  // X11 out; tmp = I + X11 G; y = X11
  for (size_t e = threadIdx.x; e < nn; e += kBlock) {
    const int i = (int)(e % n), j = (int)(e / n);
    X11[i + (size_t)j * ld] = (T)x[e];
    double s = 0.0;
    for (int k = 0; k < n; ++k) s += x[i + (size_t)k * n] * g[k + (size_t)j * n];
    tmp[e] = s + (i == j ? 1.0 : 0.0);
    y[e] = x[e];
  }
  __syncthreads();
  getrf_body<double>(tmp, n, n, piv, info);
  __syncthreads();
  // KK = tmp^-1 X11: interchanges, unit lower, upper
  for (int j = 0; j < n; ++j) {
    const int p = piv[j];
    if (p != j && p >= 0 && p < n)
      for (int c = threadIdx.x; c < n; c += kBlock) {
        const double a = y[j + (size_t)c * n];
        y[j + (size_t)c * n] = y[p + (size_t)c * n];
        y[p + (size_t)c * n] = a;
      }
    __syncthreads();
  }
  for (int c = threadIdx.x; c < n; c += kBlock) {
    for (int i = 0; i < n; ++i) {
      double s = y[i + (size_t)c * n];
      for (int k = 0; k < i; ++k) s -= tmp[i + (size_t)k * n] * y[k + (size_t)c * n];
      y[i + (size_t)c * n] = s;
    }
    for (int i = n - 1; i >= 0; --i) {
      double s = y[i + (size_t)c * n];
      for (int k = i + 1; k < n; ++k) s -= tmp[i + (size_t)k * n] * y[k + (size_t)c * n];
      y[i + (size_t)c * n] = s / tmp[i + (size_t)i * n];
    }
    for (int i = 0; i < n; ++i) KK[i + (size_t)c * ld] = (T)y[i + (size_t)c * n];
  }
}

// ---------------------------------------------------------------------------
// TRSM with a lower-triangular leaf L (n x n):
//   mode 0: X (m x n) <- X L^{-T}     (solveUpperTriangularRight, LLt)
//   mode 1: X (n x k) <- L^{-1} X     (solveLowerTriangularLeft)
//   mode 2: X (n x k) <- L^{-T} X     (solveUpperTriangularLeft, Uplo LOWER)
// Flags (ftask.hpp): kTrsmTransA reads L as the transpose of an upper
// triangle U (so 0 is X U^{-1}, 1 is U^{-T} X, 2 is U^{-1} X: the LU cases of
// scalar_array.cpp:852-874), kTrsmUnit assumes a unit diagonal, kTrsmPiv
// applies getrf's row interchanges to X first (laswp, scalar_array.cpp:855).
// Rows (mode 0) / columns (modes 1, 2) of X are independent: a task is cut
// into tiles of kTrsmCols of them, one workgroup each.
// ---------------------------------------------------------------------------
constexpr int kShDoubles = 19456;  // 152 KiB of LDS per workgroup

// A wavefront solves 16 independent rows / columns of X on its own: X^T (mode
// 0) or X is cut into 16 x 16 blocks that stay in registers in the layout in
// which v_mfma_f64_16x16x4f64 returns a tile, which is also its B operand's,
// so a solved block is the operand of the next products without passing
// through LDS:
//   X_p <- inv(L_pp) (X_p - sum_{c < p} L_pc X_c)   (p from the last block in mode 2)
// The blocks of L come from the L2 (one 128-byte run per 16 lanes, shorter
// runs for transposed operands), eight of them in flight.  Only the inverted
// diagonal blocks pass through LDS.  Eight blocks (128 rows) are solved at a
// time: above that the solved blocks are read back by the lanes that wrote
// them.
// Bound: the serial chain of nb (nb + 1) / 2 block products; no barrier after
// the inversions.  The earlier form kept L and X in LDS, two workgroups per
// task: leaves above 100 rows did not fit beside X and were substituted row by
// row, and a block of 2,000 columns had two CUs.  The N = 4,000 system (leaves
// of 125 rows, inverses of its 2,000-row diagonal blocks for the solve) went
// from 138.9 to 24.4 ms with this, the tiles of the elementwise tasks and the
// skipped zero half of the inverses.
// With the masks and the conversion at the use and not at the load (which made
// every load wait), the interchanges followed backwards and the diagonal's loads
// together, an average launch went from 32.4 to 18.3 us (94 rows, FP64, with
// interchanges), 29 to 20 us (125 rows, FP32) and 16 to 12.8 us (78 rows, FP32).
constexpr int kTrsmBlocks = 8;              // blocks solved in registers at a time
constexpr int kTrsmInvLd = kNb * kNb + 8;   // diagonal blocks in LDS: spread over the banks

// row p of the s-th pair (p, c), c < p, in row order
constexpr int trsm_pair_row(int s) {
  int p = 1;
  while (p * (p + 1) / 2 <= s) ++p;
  return p;
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_trsm(const FTask* tasks, const GemmTile* tiles, const int* fail) {
  __shared__ double inv[kTrsmBlocks * kTrsmInvLd];
  __shared__ double rdiag[kTrsmBlocks * kNb];
  __shared__ int perm[kTrsmBlocks * kNb];
  constexpr int NB = kTrsmBlocks;
  const int failed = *fail;  // in flight together with the tile and the task
  const GemmTile tl = tiles[blockIdx.x];
  const FTask& t = tasks[tl.task];
  const int other = eff(t.m), col0 = tl.tm * kTrsmCols, n = t.n.s;
  if ((failed != 0) | (col0 >= other) | (n <= 0)) return;
  const int nb = (n + kNb - 1) / kNb;
  const int mode = t.mode & kTrsmBase;
  const bool transa = (t.mode & kTrsmTransA) != 0, unit = (t.mode & kTrsmUnit) != 0;
  const bool back = mode == 2, pivot = (t.mode & kTrsmPiv) && mode != 0;
  const auto Lg = (cgptr<T>)t.A;
  const auto X = (gptr<T>)t.C;
  const long li = transa ? (long)t.lda : 1L, lk = transa ? 1L : (long)t.lda;  // strides of L(i, k)
  const long ai = back ? lk : li, ak = back ? li : lk;  // of the operand: L, or L^T in mode 2
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const int ii = lane & 15, kk = lane >> 4;
  // this wavefront's 16 columns of X (rows in mode 0): element (row r, column
  // ii) at Xc[r * xr]
  const int j = col0 + kNb * w + ii, jc = j < other ? j : other - 1;
  const bool mine = col0 + kNb * w < other;
  const long xr = mode == 0 ? (long)t.ldc : 1L;
  const auto Xc = X + (mode == 0 ? (size_t)jc : (size_t)jc * t.ldc);
  const bool permuted = pivot && nb <= NB;
  if (permuted && w == 0) {
    // the interchanges as one permutation: the lane follows the content of rows
    // lane + 64 q back through them (steps of two compares, no chain of exchanges)
    const auto piv = (cgptr<int>)t.B;
    constexpr int kQ = NB / 4;
    int src[kQ], pv[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int r = lane + kWave * q;
      src[q] = r;
      const int p = piv[r < n ? r : n - 1];
      pv[q] = p < 0 ? 0 : (p >= n ? n - 1 : p);
    }
#pragma unroll
    for (int h = kQ - 1; h >= 0; --h)
      for (int i = (n - kWave * h < kWave ? n - kWave * h : kWave) - 1; i >= 0; --i) {
        const int p = __builtin_amdgcn_readlane(pv[h], i), g = i + kWave * h;
#pragma unroll
        for (int q = 0; q < kQ; ++q) src[q] = src[q] == g ? p : (src[q] == p ? g : src[q]);
      }
#pragma unroll
    for (int q = 0; q < kQ; ++q) perm[lane + kWave * q] = src[q];
  } else if (pivot && !permuted) {
    // wide leaves: each thread replays the interchanges on its own column
    const auto piv = (cgptr<int>)t.B;
    if (threadIdx.x < kTrsmCols && col0 + (int)threadIdx.x < other) {
      const auto xc = X + (size_t)(col0 + threadIdx.x) * t.ldc;
      for (int i = 0; i < n; ++i) {
        int p = piv[i];
        p = p < 0 ? 0 : (p >= n ? n - 1 : p);
        if (p != i) {
          const T a = xc[i];
          xc[i] = xc[p];
          xc[p] = a;
        }
      }
    }
  }
  for (int p0 = 0; p0 < nb; p0 += NB) {
    const int np = nb - p0 < NB ? nb - p0 : NB;
    auto block_of = [&](int p) { return back ? nb - 1 - p : p; };
    __syncthreads();
    // the diagonal blocks (lower triangles) and the reciprocals of the diagonal
    {
      static_assert(kNb * kNb == kBlock, "an entry of each block per thread");
      const int r = threadIdx.x % kNb, l = threadIdx.x / kNb;
      T v[NB];
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int gr = block_of(p0 + (q < np ? q : np - 1)) * kNb + r, gl = gr - r + l;
        v[q] = Lg[(gr < n ? gr : n - 1) * li + (gl < n ? gl : n - 1) * lk];
      }
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        if (q >= np) break;
        const int gr = block_of(p0 + q) * kNb + r;
        const bool in = gr < n && l <= r;
        inv[q * kTrsmInvLd + r + l * kNb] = in ? (double)v[q] : 0.0;
        if (r == l) rdiag[q * kNb + r] = (unit || !in) ? 1.0 : 1.0 / (double)v[q];
      }
    }
    __syncthreads();
    // thread (q, c): column c of the inverse of block q by forward
    // substitution, in registers; written over the block once all are done
    const int iq = threadIdx.x / kNb, ic = threadIdx.x % kNb;
    double xi[kNb];
    if (iq < np) {
      const double* blk = inv + iq * kTrsmInvLd;
#pragma unroll
      for (int r = 0; r < kNb; ++r) {
        double s = r == ic ? 1.0 : 0.0;
#pragma unroll
        for (int l = 0; l < r; ++l) s -= blk[r + l * kNb] * xi[l];
        xi[r] = r < ic ? 0.0 : s * rdiag[iq * kNb + r];
      }
    }
    __syncthreads();
    if (iq < np) {
      double* blk = inv + iq * kTrsmInvLd;
      const int g0 = block_of(p0 + iq) * kNb;
#pragma unroll
      for (int r = 0; r < kNb; ++r) {
        const double v = (g0 + ic >= n || g0 + r >= n) ? 0.0 : xi[r];
        blk[back ? ic + r * kNb : r + ic * kNb] = v;  // mode 2 applies the transposed inverse
      }
    }
    __syncthreads();
    if (!mine) continue;
    // (all loads of X and of the operand blocks issue before anything waits for
    // one: the conversion and the masks come at the use)
    T xin[NB][4];
#pragma unroll
    for (int p = 0; p < NB; ++p) {
      const int r0 = kNb * block_of(p0 + (p < np ? p : np - 1));
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = r0 + kk + 4 * v, rc = r < n ? r : n - 1;
        xin[p][v] = Xc[(permuted ? perm[rc] : rc) * xr];
      }
    }
    // operand blocks in the order in which they are used, (1, 0), (2, 0),
    // (2, 1), ...: kAhead of them in flight.  Past the last row they repeat it: such
    // inner indices meet zeros of x, and such rows of the sum are cleared.
    constexpr int kAhead = 8, kPairs = NB * (NB - 1) / 2;
    T a[kAhead][4];
    auto load_block = [&](auto S) __attribute__((always_inline)) {
      constexpr int s = decltype(S)::value, p = trsm_pair_row(s), c = s - p * (p - 1) / 2;
      if (p >= np) return;
      const int r = kNb * block_of(p0 + p) + ii, rc = r < n ? r : n - 1;
      const int k0 = kNb * block_of(p0 + c) + kk;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = k0 + 4 * q, kc = k < n ? k : n - 1;
        a[s % kAhead][q] = Lg[rc * ai + kc * ak];
      }
    };
    static_for<0, kAhead < kPairs ? kAhead : kPairs>(load_block);
    hmx_double4 x[NB];
#pragma unroll
    for (int p = 0; p < NB; ++p) {
      const int r0 = kNb * block_of(p0 + p) + kk;
#pragma unroll
      for (int v = 0; v < 4; ++v) x[p][v] = p < np && r0 + 4 * v < n ? (double)xin[p][v] : 0.0;
    }
    // the blocks solved before these eight
    for (int c = 0; c < p0; ++c) {
      const int c0 = kNb * block_of(c) + kk;
      double xs[4], as[NB][4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = c0 + 4 * q, kc = k < n ? k : n - 1;
        const double y = (double)Xc[kc * xr];
        xs[q] = k < n ? -y : 0.0;
#pragma unroll
        for (int p = 0; p < NB; ++p) {
          const int r = kNb * block_of(p0 + (p < np ? p : np - 1)) + ii, rc = r < n ? r : n - 1;
          const double v = (double)Lg[rc * ai + kc * ak];
          as[p][q] = (r < n && k < n) ? v : 0.0;
        }
      }
#pragma unroll
      for (int p = 0; p < NB; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) x[p] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[p][q], xs[q], x[p], 0, 0, 0);
    }
    static_for<0, NB>([&](auto P) __attribute__((always_inline)) {
      constexpr int p = decltype(P)::value;
      if (p >= np) return;
      hmx_double4 s0 = x[p], s1 = {0.0, 0.0, 0.0, 0.0};
      // x of the solved blocks holds the negated result
      static_for<0, p>([&](auto C) __attribute__((always_inline)) {
        constexpr int c = decltype(C)::value, s = p * (p - 1) / 2 + c;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if constexpr (c & 1)
            s1 = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[s % kAhead][q], x[c][q], s1, 0, 0, 0);
          else
            s0 = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[s % kAhead][q], x[c][q], s0, 0, 0, 0);
        }
        if constexpr (s + kAhead < kPairs) load_block(std::integral_constant<int, s + kAhead>{});
      });
      const int r0 = kNb * block_of(p0 + p) + kk;
      const double* blk = inv + p * kTrsmInvLd;
      hmx_double4 y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q)
        y = __builtin_amdgcn_mfma_f64_16x16x4f64(blk[q * kWave + lane], r0 + 4 * q < n ? s0[q] + s1[q] : 0.0, y, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (r0 + 4 * v < n && j < other) Xc[(r0 + 4 * v) * xr] = (T)y[v];
        x[p][v] = -y[v];
      }
    });
  }
}

// ---------------------------------------------------------------------------
// SUMK: C (m x n) = (mode ? C : 0) + sum_q W_q, the partial products of a
// GEMM split along its inner dimension, added in a fixed order.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void k_sumk(const FTask* tasks, const GemmTile* tiles, const int* fail) {
  if (*fail) return;
  const GemmTile tl = tiles[blockIdx.x];
  const FTask& t = tasks[tl.task];
  const int M = eff(t.m), N = eff(t.n), S = t.p.s;
  const auto W = (cgptr<T>)t.A;
  const auto C = (gptr<T>)t.C;
  const int64_t hi = std::min<int64_t>((int64_t)M * N, (int64_t)(tl.tm + 1) * kElemsPerTile);
  for (int64_t e = (int64_t)tl.tm * kElemsPerTile + threadIdx.x; e < hi; e += blockDim.x) {
    const int i = (int)(e % M), j = (int)(e / M);
    const auto pc = C + i + (size_t)j * t.ldc;
    const auto w = W + i + (size_t)j * t.lda;
    double s = t.mode ? (double)*pc : 0.0;
#pragma unroll 8
    for (int q = 0; q < S; ++q) s += (double)w[(size_t)q * t.ldb];
    *pc = (T)s;
  }
}

// ---------------------------------------------------------------------------
// zero fill and axpy
// ---------------------------------------------------------------------------
template <typename T>
__global__ void k_zero(const FTask* tasks, const GemmTile* tiles, const int* fail) {
  if (*fail) return;
  const GemmTile tl = tiles[blockIdx.x];
  const FTask& t = tasks[tl.task];
  const auto C = (gptr<T>)t.C;
  const int m = t.m.s, n = t.n.s;
  // mode 1: the identity
  const int64_t hi = std::min<int64_t>((int64_t)m * n, (int64_t)(tl.tm + 1) * kElemsPerTile);
  for (int64_t e = (int64_t)tl.tm * kElemsPerTile + threadIdx.x; e < hi; e += blockDim.x) {
    const int i = (int)(e % m), j = (int)(e / m);
    C[i + (size_t)j * t.ldc] = (t.mode == 1 && i == j) ? (T)1 : (T)0;
  }
}

template <typename T>
__global__ void k_axpy(const FTask* tasks, const GemmTile* tiles, const int* fail) {
  if (*fail) return;
  const GemmTile tl = tiles[blockIdx.x];
  const FTask& t = tasks[tl.task];
  const auto C = (gptr<T>)t.C;
  const auto A = (cgptr<T>)t.A;
  const int m = eff(t.m), n = eff(t.n);
  const T al = (T)t.alpha;
  const int64_t hi = std::min<int64_t>((int64_t)m * n, (int64_t)(tl.tm + 1) * kElemsPerTile);
  for (int64_t e = (int64_t)tl.tm * kElemsPerTile + threadIdx.x; e < hi; e += blockDim.x) {
    const int i = (int)(e % m), j = (int)(e / m);
    const T v = t.ta ? A[j + (size_t)i * t.lda] : A[i + (size_t)j * t.lda];
    if (t.mode)
      C[i + (size_t)j * t.ldc] = al * v;
    else
      C[i + (size_t)j * t.ldc] += al * v;
  }
}

// ---------------------------------------------------------------------------
// Recompression helpers (FP64; operands in LDS when they fit)
// ---------------------------------------------------------------------------
// G (gr x gc, ld gr) holds D (tr == false) or D^T (tr == true) of the dense
// block to compress; V, sig, order scratch (gc^2, gc, gc).  Truncated SVD at
// eps into out (A = U sqrt(S) on the row side of D).
template <typename T>
__device__ int dense_to_rk(double* G, bool in_lds, int gr, int gc, bool tr, double* V, double* sig, int* order,
                           double eps, RkRef out, int* overflow, int* flag) {
  if (in_lds)
    jacobi_svd<true>((lptr<double>)G, gr, gr, gc, (lptr<double>)V, gc, flag);
  else
    jacobi_svd<true>((gptr<double>)G, gr, gr, gc, (gptr<double>)V, gc, flag);
  sorted_norms(G, gr, gr, gc, sig, order);
  int k = find_k(sig, order, gc, eps);
  if (k > out.cap) {
    if (threadIdx.x == 0) atomicOr(overflow, 1);
    k = out.cap;
  }
  T* A = (T*)out.a;
  T* B = (T*)out.b;
  for (int e = threadIdx.x; e < k * gr; e += kBlock) {
    const int i = e % gr, c = e / gr, j = order[c];
    const double v = G[i + (size_t)j * gr] / sqrt(sig[j]);
    if (tr)
      B[i + (size_t)c * out.lb] = (T)v;
    else
      A[i + (size_t)c * out.la] = (T)v;
  }
  for (int e = threadIdx.x; e < k * gc; e += kBlock) {
    const int i = e % gc, c = e / gc, j = order[c];
    const double v = V[i + (size_t)j * gc] * sqrt(sig[j]);
    if (tr)
      A[i + (size_t)c * out.la] = (T)v;
    else
      B[i + (size_t)c * out.lb] = (T)v;
  }
  __syncthreads();
  if (threadIdx.x == 0) *out.rank = k;
  return k;
}

// Scratch of the QR recompression (all K x K blocks ld K).
// (P double pointers, PI int pointers: LDS or global)
template <typename P, typename PI>
struct QrScratch {
  P taua, taub;  // K each
  P g, v;        // core SVD: G = Ra Rb^T -> U Sigma, and its input
  P ta, tb;      // block-reflector factors of the two panels
  P x, w;        // K x nk work blocks of the back-transformation
  P sig, scale;  // K each
  PI order;      // K
};
using LdsScratch = QrScratch<lptr<double>, lptr<int>>;
using GlobalScratch = QrScratch<gptr<double>, gptr<int>>;

// doubles of the scratch above.  The core SVD of up to kCoreMax columns works in
// x and w, which are free then; where they are too small (K below 10, and 17) it
// goes past their end.
__device__ inline int64_t qr_core(int K) {
  const int64_t K2 = (int64_t)K * K;
  const int64_t past = K <= kCoreMax ? core_work(K, K) - 2 * K2 : 0;
  return 6 * K2 + 5 * (int64_t)K + (past > 0 ? past : 0);
}

template <typename W, typename P>
__device__ inline W carve_qr(P core, int K) {
  const size_t K2 = (size_t)K * K;
  W w;
  w.taua = core;
  w.taub = core + K;
  w.sig = core + 2 * K;
  w.scale = core + 3 * K;
  w.order = (decltype(w.order))(core + 4 * K);
  w.g = core + 5 * K;
  w.v = w.g + K2;
  w.ta = w.v + K2;
  w.tb = w.ta + K2;
  w.x = w.tb + K2;
  w.w = w.x + K2;
  return w;
}

// Rows of one side of the formatted sum, concatenated: the target's panel
// followed by every live part's panel placed at its row offset (zero
// elsewhere); alpha_i scales the A side.  dst is rows x K, ld ld.
template <typename T, typename PD>
__device__ void concat_side(PD dst, int ld, int rows, bool bside, const FTask& t, int kt) {
  const RkRef& tg = t.tgt;
  const auto src = (cgptr<T>)(bside ? tg.b : tg.a);
  const int lds = bside ? tg.lb : tg.la;
  stage_in(dst, ld, src, 1L, (long)lds, rows, kt);
  int off = kt;
  for (int q = 0; q < t.nparts; ++q) {
    const Part& p = t.parts[q];
    const int kq = rank_of(p.rk);
    if (!(kq > 0 && p.alpha != 0.0 && p.rk.m > 0 && p.rk.n > 0)) continue;
    const auto P = (cgptr<T>)(bside ? p.rk.b : p.rk.a);
    const int ldp = bside ? p.rk.lb : p.rk.la;
    const int o = bside ? p.coff : p.roff, pr = bside ? p.rk.n : p.rk.m;
    const double f = bside ? 1.0 : p.alpha;
    // the part covers rows [o, o + pr) of the target; zero elsewhere
    const int r_lo = o > 0 ? o : 0, r_hi = o + pr < rows ? o + pr : rows;
    const PD col0 = dst + (size_t)off * ld;
    if (r_hi > r_lo)
      stage_in(col0 + r_lo, ld, P + (r_lo - o), 1L, (long)ldp, r_hi - r_lo, kq, r_hi - r_lo, kq, f);
    const int nz = rows - (r_hi > r_lo ? r_hi - r_lo : 0);
    for (int e = threadIdx.x; e < nz * kq; e += kBlock) {
      int i = e % nz;
      const int c = e / nz;
      if (r_hi > r_lo && i >= r_lo) i += r_hi - r_lo;
      col0[i + (size_t)c * ld] = 0.0;
    }
    off += kq;
  }
}

// Both sides at once for K <= kColsMax: a lane builds each column's descriptor,
// then every wavefront copies four columns at a time, their loads in flight
// together and no index divided.
constexpr int kColsMax = 32;
constexpr int kColDoubles = 6 * kColsMax;  // LDS for the descriptors (2 K of three doubles)

template <typename T, typename PD>
__device__ void concat_both(PD da, int lda, PD db, int ldb, int K, const FTask& t, int kt, lptr<double> desc) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const RkRef& tg = t.tgt;
  const auto base = (lptr<long>)desc;            // address of the column's row 0
  const auto span = (lptr<int>)(desc + 2 * K);   // offset and rows
  const auto scale = desc + 4 * K;
  const int c = threadIdx.x;
  if (c < 2 * K) {
    const bool bside = c >= K;
    int cc = bside ? c - K : c;
    const T* p = (const T*)(bside ? tg.b : tg.a);
    int ld = bside ? tg.lb : tg.la, o = 0, pr = bside ? tg.n : tg.m;
    double f = 1.0;
    if (cc >= kt) {
      cc -= kt;
      for (int q = 0; q < t.nparts; ++q) {
        const Part& x = t.parts[q];
        const int kq = rank_of(x.rk);
        if (!(kq > 0 && x.alpha != 0.0 && x.rk.m > 0 && x.rk.n > 0)) continue;
        if (cc < kq) {
          p = (const T*)(bside ? x.rk.b : x.rk.a);
          ld = bside ? x.rk.lb : x.rk.la;
          o = bside ? x.coff : x.roff;
          pr = bside ? x.rk.n : x.rk.m;
          f = bside ? 1.0 : x.alpha;
          break;
        }
        cc -= kq;
      }
    }
    base[c] = (long)(p + (size_t)cc * ld);
    span[2 * c] = o;
    span[2 * c + 1] = pr;
    scale[c] = f;
  }
  __syncthreads();
  constexpr int kC = 4, kR = 2;
  for (int c0 = kC * w; c0 < 2 * K; c0 += kC * kWaves) {
    cgptr<T> p[kC];
    int o[kC], pr[kC], len[kC], most = 0;
    double f[kC];
    PD dst[kC];
#pragma unroll
    for (int b = 0; b < kC; ++b) {
      const int cb = c0 + b < 2 * K ? c0 + b : 2 * K - 1;
      p[b] = (cgptr<T>)base[cb];
      o[b] = span[2 * cb];
      pr[b] = span[2 * cb + 1];
      f[b] = scale[cb];
      len[b] = c0 + b >= 2 * K ? 0 : (cb < K ? tg.m : tg.n);
      dst[b] = cb < K ? da + (size_t)cb * lda : db + (size_t)(cb - K) * ldb;
      most = len[b] > most ? len[b] : most;
    }
    for (int r0 = lane; r0 < most; r0 += kR * kWave) {
      T x[kR][kC];
#pragma unroll
      for (int u = 0; u < kR; ++u)
#pragma unroll
        for (int b = 0; b < kC; ++b) {
          const int r = r0 + u * kWave - o[b];
          x[u][b] = p[b][r < 0 ? 0 : (r < pr[b] ? r : pr[b] - 1)];
        }
#pragma unroll
      for (int u = 0; u < kR; ++u)
#pragma unroll
        for (int b = 0; b < kC; ++b) {
          const int r = r0 + u * kWave;
          if (r < len[b]) dst[b][r] = (r >= o[b] && r < o[b] + pr[b]) ? f[b] * (double)x[u][b] : 0.0;
        }
    }
  }
  __syncthreads();
}

// G (K x K) = Ra Rb^T with Ra, Rb the upper triangles of two panels.
template <typename PA, typename PB, typename PG>
__device__ inline void core_product(PA Ra, int lra, PB Rb, int lrb, int K, PG G) {
  for (int e = threadIdx.x; e < K * K; e += kBlock) {
    const int i = e % K, j = e / K;
    double s = 0.0;
    const int lo = i > j ? i : j;
    for (int l = lo; l < K; ++l) s += Ra[i + (size_t)l * lra] * Rb[j + (size_t)l * lrb];
    G[i + (size_t)j * K] = s;
  }
}

// out (rows x nk, ld ldo) = Q [U; 0] with Q = I - V Tq V^T (rows x K panel of
// reflectors V, ld ldv) and U[i, c] = src[i, order[c]] * scale[c] (K x nk,
// ld K): X = V1^T U, W = Tq X (K x nk, from the unit lower K x K top V1 of V
// staged in w.w), then out = [U; 0] - V W with each thread owning rows and
// streaming a row of V once per eight output columns.
template <typename T, typename PV, typename PS, typename W>
__device__ void wy_apply_out(PV V, int ldv, int rows, int K, PS Tq, PS src, const W& w, int nk, gptr<T> out,
                             int ldo) {
  for (int e = threadIdx.x; e < K * K; e += kBlock) {
    const int i = e % K, l = e / K;
    w.w[e] = i > l ? V[i + (size_t)l * ldv] : (i == l ? 1.0 : 0.0);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < K * nk; e += kBlock) {
    const int l = e % K, c = e / K;
    const PS u = src + (size_t)w.order[c] * K;
    const PS vl = w.w + (size_t)l * K;
    double s = 0.0;
    for (int i = l; i < K; ++i) s += vl[i] * u[i];
    w.x[l + (size_t)c * K] = s * w.scale[c];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < K * nk; e += kBlock) {
    const int l = e % K, c = e / K;
    double s = 0.0;
    for (int r = l; r < K; ++r) s += Tq[l + (size_t)r * K] * w.x[r + (size_t)c * K];
    w.w[l + (size_t)c * K] = s;  // the staged V1 is no longer read
  }
  __syncthreads();
  constexpr int kC = 8;
  for (int c0 = 0; c0 < nk; c0 += kC) {
    PS wc[kC];
#pragma unroll
    for (int b = 0; b < kC; ++b) wc[b] = w.w + (size_t)(c0 + b < nk ? c0 + b : nk - 1) * K;
    // two rows per thread at a time (the second one kBlock further), so that
    // 16 loads of V are in flight per round; rows past the panel read a
    // clamped row and are not stored
    for (int i0 = threadIdx.x; i0 < rows; i0 += 2 * kBlock) {
      const int ia = i0, ib = i0 + kBlock < rows ? i0 + kBlock : rows - 1;
      const bool has_b = i0 + kBlock < rows;
      double acc[2][kC];
#pragma unroll
      for (int b = 0; b < kC; ++b) acc[0][b] = acc[1][b] = 0.0;
      // entries strictly below the unit diagonal: l < min(i, K)
      const int la = ia < K ? ia : K, lb = ib < K ? ib : K, lmax = la > lb ? la : lb;
      const PV va = V + ia;
      const PV vb = V + ib;
      int l = 0;
      for (; l + 8 <= lmax; l += 8) {
        double xa[8], xb[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          xa[q] = va[(size_t)(l + q) * ldv];
          xb[q] = vb[(size_t)(l + q) * ldv];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const double ya = l + q < la ? xa[q] : 0.0, yb = l + q < lb ? xb[q] : 0.0;
#pragma unroll
          for (int b = 0; b < kC; ++b) {
            acc[0][b] += ya * wc[b][l + q];
            acc[1][b] += yb * wc[b][l + q];
          }
        }
      }
      for (; l < lmax; ++l) {
        const double ya = l < la ? va[(size_t)l * ldv] : 0.0, yb = l < lb ? vb[(size_t)l * ldv] : 0.0;
#pragma unroll
        for (int b = 0; b < kC; ++b) {
          acc[0][b] += ya * wc[b][l];
          acc[1][b] += yb * wc[b][l];
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (h == 1 && !has_b) break;
        const int i = h == 0 ? ia : ib;
#pragma unroll
        for (int b = 0; b < kC; ++b) {
          if (c0 + b >= nk) break;
          double y = -acc[h][b];
          if (i < K) y += src[i + (size_t)w.order[c0 + b] * K] * w.scale[c0 + b] - wc[b][i];
          out[i + (size_t)(c0 + b) * ldo] = (T)y;
        }
      }
    }
  }
  __syncthreads();
}

// After QR of both panels (reflectors Va, Vb, factors ta, tb) and G = Ra Rb^T
// in w.g: SVD of G, cut at eps, write Qa U sqrt(S) and Qb V sqrt(S) to out.
// stage: free LDS of kShDoubles doubles when the core lives in global memory:
// a core of at most kShDoubles entries is rotated there.
template <typename T, typename PV, typename P, typename PI>
__device__ void qr_finish(PV Va, int lda, int m, PV Vb, int ldb, int n, int K, const QrScratch<P, PI>& w,
                          double eps, RkRef out, int* overflow, int* flag, lptr<double> stage) {
  constexpr bool kInLds = std::is_same_v<P, lptr<double>>;
  __shared__ int core_cut;
  // one-sided Jacobi on G without V: G_in (kept in w.v) gives the right side
  // afterwards as G_in^T U, so the rounds only rotate G
  for (int e = threadIdx.x; e < K * K; e += kBlock) w.v[e] = w.g[e];
  __syncthreads();
  bool cut = false;
  if constexpr (kInLds) {
    if (K <= kCoreMax) {
      if (threadIdx.x < kWave) {
        const int c = wave_core_svd(w.g, K, K, K, w.x, 1e-26);
        const int k = wave_sorted_cut(w.g, K, K, c, w.sig, w.order, eps);
        if (threadIdx.x == 0) core_cut = k;
      }
      __syncthreads();
      cut = true;
    } else {
      jacobi_svd<false>(w.g, K, K, K, w.g, K, flag);
    }
  } else if (K * K <= kShDoubles) {
    // the rounds' loads and stores hit LDS instead of the L2
    for (int e = threadIdx.x; e < K * K; e += kBlock) stage[e] = w.g[e];
    __syncthreads();
    jacobi_svd<false>(stage, K, K, K, stage, K, flag);
    for (int e = threadIdx.x; e < K * K; e += kBlock) w.g[e] = stage[e];
    __syncthreads();
  } else {
    jacobi_svd<false>(w.g, K, K, K, w.g, K, flag);
    __syncthreads();
  }
  int nk;
  if (cut) {
    nk = core_cut;
  } else {
    sorted_norms(w.g, K, K, K, w.sig, w.order);
    nk = find_k(w.sig, w.order, K, eps);
  }
  if (nk > out.cap) {
    if (threadIdx.x == 0) atomicOr(overflow, 1);
    nk = out.cap;
  }
  // A = Qa U sqrt(S): column j of the rotated G is sigma_j u_j
  for (int c = threadIdx.x; c < nk; c += kBlock) w.scale[c] = 1.0 / sqrt(w.sig[w.order[c]]);
  __syncthreads();
  wy_apply_out<T>(Va, lda, m, K, w.ta, w.g, w, nk, (gptr<T>)out.a, out.la);
  // B = Qb V sqrt(S) with v_j sigma_j = G_in^T u_j, u_j = g_j / sigma_j: column j
  // of w.ta (the A side's block factor is done) gets G_in^T u_j, and the same
  // scale 1 / sqrt(sigma_j) as the A side applies
  for (int e = threadIdx.x; e < K * nk; e += kBlock) {
    const int i = e % K, j = w.order[e / K];
    const P gi = w.v + (size_t)i * K;
    const P gj = w.g + (size_t)j * K;
    double s = 0.0;
    for (int l = 0; l < K; ++l) s += gi[l] * gj[l];
    w.ta[i + (size_t)j * K] = s / w.sig[j];
  }
  __syncthreads();
  wy_apply_out<T>(Vb, ldb, n, K, w.tb, w.ta, w, nk, (gptr<T>)out.b, out.lb);
  if (threadIdx.x == 0) *out.rank = nk;
}

// QR form with both concatenated panels in global memory (Va m x K, Vb n x K);
// part: part_size doubles of free LDS.
template <typename T, typename W>
__device__ void qr_global(gptr<double> Va, int m, gptr<double> Vb, int n, int K, const W& w, lptr<double> part,
                          int64_t part_size, double eps, RkRef out, int* overflow, int* flag, lptr<double> stage) {
  // V^T V of the global panels on the matrix cores when its LDS staging fits
  const bool mfma_gram = K <= 64 && gram_part(K) <= part_size;
  // both panels at once, one per half of the workgroup, when each has at
  // most 16 rows per thread
  const bool pair = m <= 16 * (kBlock / 2) && n <= 16 * (kBlock / 2);
  if (pair)
    house_qr_pair(Va, m, m, w.taua, Vb, n, n, w.taub, K);
  else
    house_qr(Va, m, m, K, w.taua);
  if (mfma_gram) {
    wg_reflector_gram_any(Va, m, m, K, w.x, part);
    larft_recurrence<kBlock>(K, w.taua, w.x, w.ta);
  } else {
    team_larft<kBlock>(Va, m, m, K, w.taua, w.x, w.ta);
  }
  if (!pair) house_qr(Vb, n, n, K, w.taub);
  if (mfma_gram) {
    wg_reflector_gram_any(Vb, n, n, K, w.x, part);
    larft_recurrence<kBlock>(K, w.taub, w.x, w.tb);
  } else {
    team_larft<kBlock>(Vb, n, n, K, w.taub, w.x, w.tb);
  }
  core_product(Va, m, Vb, n, K, w.g);
  __syncthreads();
  qr_finish<T>(Va, m, m, Vb, n, n, K, w, eps, out, overflow, flag, stage);
}

// ---------------------------------------------------------------------------
// Gram recompression of single-precision panels.  The formatted sum is
// [A] [B]^T with A (m x K), B (n x K) the concatenated panels (FP64 copies).
// Instead of Householder QR of each panel (one column step at a time), the
// Grams A^T A and B^T B are formed on the FP64 matrix cores in one pass over
// the panels and factored by pivoted Cholesky, A P = Q [R11 R12] with Q =
// A P1 R11^-1, stopping where the remaining diagonal falls below 1e-13 of the
// largest (columns below 3e-7 of the largest norm, far under the FP32 data's
// own rounding relative to eps).  The core R~a R~b^T (R with its columns back
// in panel order) gets the same Jacobi SVD and eps cut as the QR form of
// RkMatrix::truncate (rk_matrix.cpp:490-585), and the new panels are
// A' = A P1 R11^-1 U sqrt(S), B' = B P1 R11^-1 V sqrt(S).  Q is orthonormal to
// about 1e-16 / 1e-13 = 1e-3, so the truncated product stays within eps.
// ---------------------------------------------------------------------------
// Widest sum in this form.  Squaring the panels' condition costs accuracy that
// wider sums, which come with tight cuts, do not have: with 33 to 40 columns and
// eps = 1e-7 the result was 3.5e-7 off instead of 1e-7, two ranks short (at 1e-8
// 18 to 36 times the best error, against 5 to 7 times through Householder QR;
// 256 sums of 33 columns and 100 rows take 620 us that way, 570 in this form).
constexpr int kGramMaxK = kColsMax;
constexpr double kGramTol = 1e-13;
constexpr double kGramJacobiTol2 = 1e-16;

// Pivoted Cholesky of G (K x K, ld K, symmetric, K <= kN) by one wavefront, lane
// c holding column c of the factor in registers (left-looking: row j is G's row
// of the pivot less the rows above, the pivot's entries by readlane): G = R^T R
// with R (rank x K, ld K, columns in G's order, zeros in columns already
// pivoted), piv[j] the pivot of row j, rinv[j] = 1 / R[j, piv[j]].  Returns the
// rank.  Bound: its K^2 / 2 steps of two readlanes and an FMA.
template <int kN>
__device__ inline int wave_pchol(lptr<double> G, int K, lptr<double> R, lptr<int> piv, lptr<double> rinv) {
  const int lane = threadIdx.x & (kWave - 1), lc = lane < K ? lane : K - 1;
  double d = lane < K ? G[lc + lc * K] : -1.0;
  const double tol = kGramTol * wave_max(d);
  double row[kN];
  int r = 0;
  bool go = true;
  static_for<0, kN>([&](auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    if (go && j < K) {
      const double m = wave_max(d);
      if (m > tol) {
        const int p = __builtin_ctzll(__ballot(d == m));
        double v = G[lc + p * K];
        static_for<0, j>([&](auto ic) __attribute__((always_inline)) {
          constexpr int i = decltype(ic)::value;
          v -= lane_read(row[i], p) * row[i];
        });
        const double root = chain_sqrt(m), inv = chain_rcp(root);
        const bool done = !(d >= 0.0) && lane != p;  // pivoted before (or past K)
        const double x = lane == p ? root : (done ? 0.0 : v * inv);
        row[j] = x;
        d = lane == p || done ? -1.0 : fmax(d - x * x, 0.0);
        if (lane < K) R[j + lane * K] = x;
        if (lane == 0) {
          piv[j] = p;
          rinv[j] = inv;
        }
        r = j + 1;
      } else {
        go = false;
      }
    }
  });
  __builtin_amdgcn_wave_barrier();
  return r;
}

// out (K, rows piv[i] = solution, zero elsewhere) = P1 R11^-1 x for one column x
// (r entries) on this thread: R as wave_pchol leaves it.  Column-oriented, x in
// registers, so that a step's products are independent.
template <int kN>
__device__ inline void pchol_solve(lptr<double> R, int K, lptr<int> piv, lptr<double> rinv, int r, lptr<double> x,
                                   lptr<double> out) {
  double v[kN];
#pragma unroll
  for (int i = 0; i < kN; ++i) v[i] = i < r ? x[i] : 0.0;
  for (int i = 0; i < K; ++i) out[i] = 0.0;
  static_for<0, kN>([&](auto ic) __attribute__((always_inline)) {
    constexpr int i = kN - 1 - decltype(ic)::value;
    if (i < r) {
      const int p = piv[i];
      const lptr<double> col = R + p * K;
      const double y = v[i] * rinv[i];
      out[p] = y;
#pragma unroll
      for (int l = 0; l < i; ++l) v[l] -= col[l] * y;
    }
  });
}

// LDS doubles of gram_recompress for K columns, beside the panels
__device__ inline int gram_lds(int K) {
  const int nb = (K + 15) / 16;
  const int part = 512 * nb * (nb + 1);
  return 6 * K * K + 6 * K + (part > kColDoubles ? part : kColDoubles);
}

// The panels Va (m x K, ld lda) and Vb in LDS or global memory (PV).  With an
// index division per entry, both panels in global memory and the Cholesky, the
// sort and the triangular solve through LDS, a block of up to 256 rows took 55 us
// (19 of them the core SVD) and an average launch of FADD 147 us (40,000 points)
// and 159 us (8,000 points); now 104 and 120 us.  Bound: the serial steps of the
// core SVD, in long panels the reads of the Gram products.
template <typename T, typename PV>
__device__ void gram_recompress(PV Va, int lda, PV Vb, int ldb, const FTask& t, int kt, int K, lptr<double> sh,
                                double eps, int* overflow) {
  __shared__ int ranks[3];
  const RkRef tg = t.tgt;
  const int m = tg.m, n = tg.n;
  const int K2 = K * K;
  const lptr<double> Ga = sh;
  const lptr<double> Gb = Ga + K2;
  const lptr<double> Cm = Gb + K2;
  const lptr<double> Cin = Cm + K2;
  const lptr<double> Ra = Cin + K2;
  const lptr<double> Rb = Ra + K2;
  const lptr<double> sig = Rb + K2;
  const lptr<double> scale = sig + K, ia = scale + K, ib = ia + K;
  const lptr<int> order = (lptr<int>)(ib + K), pa = order + K, pb = pa + K;
  const lptr<double> part = sig + 6 * K;
  concat_both<T>(Va, lda, Vb, ldb, K, t, kt, part);
  constexpr bool kInLds = std::is_same_v<PV, lptr<double>>;
  constexpr int kU = kInLds ? 4 : 8;
  if (K <= 16) {
    wg_gram<1, kU>(Va, lda, K, m, Ga, K, part);
    wg_gram<1, kU>(Vb, ldb, K, n, Gb, K, part);
  } else {
    wg_gram<2, kU / 2>(Va, lda, K, m, Ga, K, part);
    wg_gram<2, kU / 2>(Vb, ldb, K, n, Gb, K, part);
  }
  const int wid = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  if (wid < 2) {
    const lptr<double> G = wid ? Gb : Ga, R = wid ? Rb : Ra, inv = wid ? ib : ia;
    const lptr<int> piv = wid ? pb : pa;
    const int r = K <= 16 ? wave_pchol<16>(G, K, R, piv, inv) : wave_pchol<kGramMaxK>(G, K, R, piv, inv);
    if (lane == 0) ranks[wid] = r;
  }
  __syncthreads();
  const int ra = ranks[0], rb = ranks[1];
  if (ra == 0 || rb == 0) {
    if (threadIdx.x == 0) *tg.rank = 0;
    return;
  }
  // core (ra x rb, ld ra) = Ra Rb^T, kept in Cin for the right side
  for (int e = threadIdx.x; e < ra * rb; e += kBlock) {
    const int x = e % ra, y = e / ra;
    double s = 0.0;
    for (int c = 0; c < K; ++c) s += Ra[x + c * K] * Rb[y + c * K];
    Cm[e] = s;
    Cin[e] = s;
  }
  __syncthreads();
  // columns orthogonal to 1e-8 of their norms: far below the FP32 data's
  // rounding once scaled by the eps cut
  // (core_work(32, 32) is less than the Gram tiles' part, core_work(16, 16) too)
  static_assert(kGramMaxK <= kCoreMax, "the core SVD of one wavefront");
  if (wid == 0) {
    const int c = wave_core_svd(Cm, ra, ra, rb, part, kGramJacobiTol2);
    const int k = wave_sorted_cut(Cm, ra, ra, c, sig, order, eps);
    if (lane < c) scale[lane] = 1.0 / sqrt(sig[lane]);
    if (lane == 0) ranks[2] = k;
  }
  __syncthreads();
  int nk = ranks[2];
  if (nk > tg.cap) {
    if (threadIdx.x == 0) atomicOr(overflow, 1);
    nk = tg.cap;
  }
  // left U sqrt(S) (ra x nk, into Ga) and right V sqrt(S) = Cin^T U / sqrt(S)
  // (rb x nk, into Gb), ld K
  for (int e = threadIdx.x; e < ra * nk; e += kBlock) {
    const int x = e % ra, c = e / ra, oc = order[c];
    Ga[x + c * K] = Cm[x + oc * ra] * scale[oc];
  }
  for (int e = threadIdx.x; e < rb * nk; e += kBlock) {
    const int y = e % rb, c = e / rb, oc = order[c];
    double s = 0.0;
    for (int x = 0; x < ra; ++x) s += Cin[x + y * ra] * Cm[x + oc * ra];
    Gb[y + c * K] = s * scale[oc] / sig[oc];
  }
  __syncthreads();
  // P1 R11^-1 of each side into Cm / Cin (K x nk, ld K), one column per thread
  if (wid < 2 && lane < nk) {
    const lptr<double> R = wid ? Rb : Ra, inv = wid ? ib : ia;
    const lptr<double> x = (wid ? Gb : Ga) + lane * K, out = (wid ? Cin : Cm) + lane * K;
    const lptr<int> piv = wid ? pb : pa;
    const int r = wid ? rb : ra;
    if (K <= 16)
      pchol_solve<16>(R, K, piv, inv, r, x, out);
    else
      pchol_solve<kGramMaxK>(R, K, piv, inv, r, x, out);
  }
  __syncthreads();
  rows_times_small<T>(Va, lda, m, K, Cm, K, nk, (gptr<T>)tg.a, tg.la);
  rows_times_small<T>(Vb, ldb, n, K, Cin, K, nk, (gptr<T>)tg.b, tg.lb);
  if (threadIdx.x == 0) *tg.rank = nk;
}

// ---------------------------------------------------------------------------
// FADD: RkMatrix::formattedAddParts (rk_matrix.cpp:846-981)
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(kBlock) k_fadd(const FTask* tasks, double* wsbase, int* overflow) {
  __shared__ double sh[kShDoubles];
  __shared__ int flag;
  if (overflow[1]) return;
  const FTask& t = tasks[blockIdx.x];
  const RkRef tg = t.tgt;
  const int m = tg.m, n = tg.n;
  const int kt = rank_of(tg);
  int K = kt, np = 0, last = -1;
  // the ranks' loads in flight together
  int kqs[kMaxParts];
#pragma unroll
  for (int q = 0; q < kMaxParts; ++q) kqs[q] = q < t.nparts ? rank_of(t.parts[q].rk) : 0;
#pragma unroll
  for (int q = 0; q < kMaxParts; ++q) {
    const int kq = kqs[q];
    if (kq > 0 && t.parts[q].alpha != 0.0 && t.parts[q].rk.m > 0 && t.parts[q].rk.n > 0) {
      K += kq;
      ++np;
      last = q;
    }
  }
  // mode 1 recompresses the target alone (RkMatrix::truncate)
  if (np == 0 && !(t.mode == 1 && kt > 0)) return;
  T* TA = (T*)tg.a;
  T* TB = (T*)tg.b;
  if (kt == 0 && np == 1) {
    // single part: copy (scaled), no recompression
    const Part& p = t.parts[last];
    int k = rank_of(p.rk);
    if (k > tg.cap) {
      if (threadIdx.x == 0) atomicOr(overflow, 1);
      k = tg.cap;
    }
    const T* PA = (const T*)p.rk.a;
    const T* PB = (const T*)p.rk.b;
    for (int e = threadIdx.x; e < m * k; e += kBlock) {
      const int i = e % m, c = e / m;
      const int ii = i - p.roff;
      TA[i + (size_t)c * tg.la] =
          (ii >= 0 && ii < p.rk.m) ? (T)(p.alpha * (double)PA[ii + (size_t)c * p.rk.la]) : (T)0;
    }
    for (int e = threadIdx.x; e < n * k; e += kBlock) {
      const int i = e % n, c = e / n;
      const int ii = i - p.coff;
      TB[i + (size_t)c * tg.lb] = (ii >= 0 && ii < p.rk.n) ? PB[ii + (size_t)c * p.rk.lb] : (T)0;
    }
    __syncthreads();
    if (threadIdx.x == 0) *tg.rank = k;
    return;
  }
  double* gws = wsbase + t.ws;
  const int mn = m < n ? m : n;
  if (K >= mn) {
    // dense path: eval everything (oriented so that the Jacobi works on min(m,n) columns)
    const bool tr = m < n;
    const int gr = tr ? n : m, gc = mn;
    const int64_t need = (int64_t)m * n + (int64_t)gc * gc + 2 * gc;
    double* G = need <= kShDoubles ? sh : gws;
    for (int e = threadIdx.x; e < m * n; e += kBlock) {
      const int i = e % m, j = e / m;
      double s = 0.0;
      for (int l = 0; l < kt; ++l) s += (double)TA[i + (size_t)l * tg.la] * (double)TB[j + (size_t)l * tg.lb];
      for (int q = 0; q < t.nparts; ++q) {
        const Part& p = t.parts[q];
        const int ii = i - p.roff, jj = j - p.coff;
        if (ii < 0 || ii >= p.rk.m || jj < 0 || jj >= p.rk.n || p.alpha == 0.0) continue;
        const int kq = rank_of(p.rk);
        const T* PA = (const T*)p.rk.a;
        const T* PB = (const T*)p.rk.b;
        double sp = 0.0;
        for (int l = 0; l < kq; ++l) sp += (double)PA[ii + (size_t)l * p.rk.la] * (double)PB[jj + (size_t)l * p.rk.lb];
        s += p.alpha * sp;
      }
      if (tr)
        G[j + (size_t)i * gr] = s;
      else
        G[i + (size_t)j * gr] = s;
    }
    __syncthreads();
    double* V = G + (size_t)m * n;
    dense_to_rk<T>(G, G == sh, gr, gc, tr, V, V + (size_t)gc * gc, (int*)(V + (size_t)gc * gc + gc),
                   fabs(t.eps), tg, overflow, &flag);
    return;
  }
  if constexpr (sizeof(T) == 4) {
    if (K <= kGramMaxK) {
      // panels in LDS (odd ld: strided lane accesses spread over the banks) when
      // they fit beside the small matrices, else in the workspace
      const int64_t small = gram_lds(K);
      const auto s3 = (lptr<double>)sh;
      if (small + (int64_t)((m | 1) + (n | 1)) * K <= kShDoubles) {
        const lptr<double> Pa = s3 + small, Pb = Pa + (m | 1) * K;
        gram_recompress<T>(Pa, m | 1, Pb, n | 1, t, kt, K, s3, fabs(t.eps), overflow);
      } else {
        const auto Pa = (gptr<double>)gws;
        gram_recompress<T>(Pa, m, Pa + (size_t)m * K, n, t, kt, K, s3, fabs(t.eps), overflow);
      }
      return;
    }
  }
  // QR path (truncate, rk_matrix.cpp:490-585) on the concatenated panels
  // [target, alpha_i parts].  Three placements:
  //  fast   both panels and the scratch in LDS; wavefront 0 reduces A while
  //         wavefront 1 reduces B;
  //  staged one panel at a time in LDS (workgroup QR), reflectors parked in
  //         the workspace;
  //  global panels in the workspace, scratch in LDS when it fits.
  // Odd leading dimensions in LDS keep the strided lane accesses spread over
  // the banks.
  const int64_t core = qr_core(K);
  const int ldAf = m | 1, ldBf = n | 1, ldM = (m > n ? m : n) | 1;
  const double eps = fabs(t.eps);
  const auto s3 = (lptr<double>)sh;
  const auto Va = (gptr<double>)gws;
  const auto Vb = Va + (size_t)m * K;
  if ((int64_t)(ldAf + ldBf) * K + core <= kShDoubles) {
    const lptr<double> Pa = s3, Pb = Pa + ldAf * K;
    const auto w = carve_qr<LdsScratch>(Pb + ldBf * K, K);
    concat_side<T>(Pa, ldAf, m, false, t, kt);
    concat_side<T>(Pb, ldBf, n, true, t, kt);
    __syncthreads();
    const int wid = threadIdx.x / kWave;
    if (wid == 0) {
      wave_house_qr(Pa, ldAf, m, K, w.taua);
      team_larft<kWave>(Pa, ldAf, m, K, w.taua, w.x, w.ta);
    } else if (wid == 1) {
      wave_house_qr(Pb, ldBf, n, K, w.taub);
      team_larft<kWave>(Pb, ldBf, n, K, w.taub, w.w, w.tb);
    }
    __syncthreads();
    core_product(Pa, ldAf, Pb, ldBf, K, w.g);
    __syncthreads();
    qr_finish<T>(Pa, ldAf, m, Pb, ldBf, n, K, w, eps, tg, overflow, &flag, lptr<double>(nullptr));
    return;
  }
  if ((int64_t)ldM * K + core <= kShDoubles) {
    const lptr<double> P = s3;
    const auto w = carve_qr<LdsScratch>(P + ldM * K, K);
    concat_side<T>(P, ldM, m, false, t, kt);
    __syncthreads();
    house_qr(P, ldM, m, K, w.taua);
    team_larft<kBlock>(P, ldM, m, K, w.taua, w.x, w.ta);
    for (int e = threadIdx.x; e < m * K; e += kBlock) {
      const int i = e % m, c = e / m;
      Va[i + (size_t)c * m] = P[i + c * ldM];
      if (i < K) w.w[i + c * K] = P[i + c * ldM];  // Ra
    }
    __syncthreads();
    concat_side<T>(P, ldM, n, true, t, kt);
    __syncthreads();
    house_qr(P, ldM, n, K, w.taub);
    team_larft<kBlock>(P, ldM, n, K, w.taub, w.x, w.tb);
    for (int e = threadIdx.x; e < n * K; e += kBlock) {
      const int i = e % n, c = e / n;
      Vb[i + (size_t)c * n] = P[i + c * ldM];
    }
    core_product(w.w, K, P, ldM, K, w.g);
    __syncthreads();
    qr_finish<T>(Va, m, m, Vb, n, n, K, w, eps, tg, overflow, &flag, lptr<double>(nullptr));
    return;
  }
  concat_side<T>(Va, m, m, false, t, kt);
  concat_side<T>(Vb, n, n, true, t, kt);
  __syncthreads();
  if (core <= kShDoubles)
    qr_global<T>(Va, m, Vb, n, K, carve_qr<LdsScratch>(s3, K), s3 + core, kShDoubles - core, eps, tg, overflow,
                 &flag, lptr<double>(nullptr));
  else
    qr_global<T>(Va, m, Vb, n, K, carve_qr<GlobalScratch>(Va + (size_t)(m + n) * K, K), s3, kShDoubles, eps, tg,
                 overflow, &flag, s3);
}

// FADD_DENSE: RkMatrix::formattedAddParts with a full part (rk_matrix.cpp:984-1010)
template <typename T>
__global__ void __launch_bounds__(kBlock) k_fadd_dense(const FTask* tasks, double* wsbase, int* overflow) {
  __shared__ double sh[kShDoubles];
  __shared__ int flag;
  if (overflow[1]) return;
  const FTask& t = tasks[blockIdx.x];
  const RkRef tg = t.tgt;
  // mode 1 replaces the target (its current panels are ignored)
  const int m = tg.m, n = tg.n, kt = t.mode ? 0 : rank_of(tg);
  const T* TA = (const T*)tg.a;
  const T* TB = (const T*)tg.b;
  const T* P = (const T*)t.A;
  const int roff = t.parts[0].roff, coff = t.parts[0].coff;
  const int pm = t.m.s, pn = t.n.s;
  const bool tr = m < n;
  const int mn = tr ? m : n, gr = tr ? n : m, gc = mn;
  const int64_t need = (int64_t)m * n + (int64_t)gc * gc + 2 * gc;
  double* G = need <= kShDoubles ? sh : wsbase + t.ws;
  for (int e = threadIdx.x; e < m * n; e += kBlock) {
    const int i = e % m, j = e / m;
    double s = 0.0;
    for (int l = 0; l < kt; ++l) s += (double)TA[i + (size_t)l * tg.la] * (double)TB[j + (size_t)l * tg.lb];
    const int ii = i - roff, jj = j - coff;
    if (ii >= 0 && ii < pm && jj >= 0 && jj < pn) s += t.alpha * (double)P[ii + (size_t)jj * t.lda];
    if (tr)
      G[j + (size_t)i * gr] = s;
    else
      G[i + (size_t)j * gr] = s;
  }
  __syncthreads();
  double* V = G + (size_t)m * n;
  dense_to_rk<T>(G, G == sh, gr, gc, tr, V, V + (size_t)gc * gc, (int*)(V + (size_t)gc * gc + gc), t.eps, tg,
                 overflow, &flag);
}

// ---------------------------------------------------------------------------
// RKRK: RkMatrix::multiplyRkRk (rk_matrix.cpp:1245-1333)
//   parts[0] = (A1, B1) op-applied left factor, parts[1] = (A2, B2) right factor
//   tmp = B1^T A2, truncated SVD, newA = A1 U sqrt(S), newB = B2 V sqrt(S)
// ---------------------------------------------------------------------------
// ws: the scratch (LDS or global); part: free LDS (part_size doubles), which may
// be where the output factors go afterwards.
template <typename T, typename P, typename PI>
__device__ void rkrk_body(const FTask& t, int k1, int k2, P ws, lptr<double> part, int64_t part_size, int* overflow,
                          int* flag) {
  const RkRef r1 = t.parts[0].rk, r2 = t.parts[1].rk, out = t.tgt;
  const int p = r1.n;  // common dimension (rows of B1 == rows of A2)
  const bool tr = k1 < k2;
  const int gr = tr ? k2 : k1, gc = tr ? k1 : k2;
  const P G = ws, V = G + (size_t)gr * gc, sig = V + (size_t)gc * gc;
  const PI order = (PI)(sig + gc);
  const auto A1 = (cgptr<T>)r1.a;
  const auto B1 = (cgptr<T>)r1.b;
  const auto A2 = (cgptr<T>)r2.a;
  const auto B2 = (cgptr<T>)r2.b;
  // core B1^T A2 (k1 x k2; stored transposed when tr): on the matrix cores
  // when both ranks are <= 32 and the LDS staging fits, else a wavefront per
  // entry
  const bool mfma = k1 <= 32 && k2 <= 32 && xty_part(k1, k2) <= part_size &&
                    wg_xty_any(B1, r1.lb, k1, A2, r2.la, k2, p, G, gr, tr, part);
  if (!mfma) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    for (int e = w; e < k1 * k2; e += kWaves) {
      const int i = e % k1, j = e / k1;
      double s = 0.0;
      for (int r = lane; r < p; r += kWave) s += (double)B1[r + (size_t)i * r1.lb] * (double)A2[r + (size_t)j * r2.la];
      s = wave_sum(s);
      if (lane == 0) G[tr ? j + (size_t)i * gr : i + (size_t)j * gr] = s;
    }
    __syncthreads();
  }
  int r = gc;
  bool done = false;
  if constexpr (std::is_same_v<P, lptr<double>>)
    if (gr <= kCoreMax) {
      // V (gc x r) = G_in^T U with the copy of G kept behind the output factors,
      // and behind it the core SVD's work
      const P Gin = sig + gc + gc + (gc & 1) + (size_t)(gr + gc) * gc, W = Gin + gr * gc;
      for (int e = threadIdx.x; e < gr * gc; e += kBlock) Gin[e] = G[e];
      __syncthreads();
      if (threadIdx.x < kWave) {
        const int c = wave_core_svd(G, gr, gr, gc, W, 1e-26);
        const int k = wave_sorted_cut(G, gr, gr, c, sig, order, t.eps);
        if (threadIdx.x == 0) {
          flag[0] = c;
          flag[1] = k;
        }
      }
      __syncthreads();
      r = flag[0];
      for (int e = threadIdx.x; e < gc * r; e += kBlock) {
        const int i = e % gc, j = e / gc;
        double s = 0.0;
        for (int l = 0; l < gr; ++l) s += Gin[l + i * gr] * G[l + j * gr];
        V[i + (size_t)j * gc] = sig[j] > 0.0 ? s / (sig[j] * sig[j]) : 0.0;
      }
      __syncthreads();
      done = true;
    }
  if (!done) {
    jacobi_svd<true>(G, gr, gr, gc, V, gc, flag);
    sorted_norms(G, gr, gr, gc, sig, order);
  }
  int nk = done ? flag[1] : find_k(sig, order, r, t.eps);
  if (nk > out.cap) {
    if (threadIdx.x == 0) atomicOr(overflow, 1);
    nk = out.cap;
  }
  // tmp = U S V^T with U = G(:,j)/sig (k1 side), V (k2 side); swapped when tr.
  // The small factors Uc (k1 x nk) = U sqrt(S) and Vc (k2 x nk) = V sqrt(S)
  // go after the SVD scratch, then the outputs stream A1 and B2 once per
  // eight columns.
  const P Uc = sig + gc + gc + (gc & 1), Vc = Uc + (size_t)k1 * nk;
  for (int e = threadIdx.x; e < k1 * nk; e += kBlock) {
    const int l = e % k1, c = e / k1, j = order[c];
    const double sq = sqrt(sig[j]);
    Uc[e] = tr ? V[l + (size_t)j * gc] * sq : G[l + (size_t)j * gr] / sq;
  }
  for (int e = threadIdx.x; e < k2 * nk; e += kBlock) {
    const int l = e % k2, c = e / k2, j = order[c];
    const double sq = sqrt(sig[j]);
    Vc[e] = tr ? G[l + (size_t)j * gr] / sq : V[l + (size_t)j * gc] * sq;
  }
  __syncthreads();
  const int m = r1.m, n = r2.n;
  rows_times_small<T>(A1, r1.la, m, k1, Uc, k1, nk, (gptr<T>)out.a, out.la);
  rows_times_small<T>(B2, r2.lb, n, k2, Vc, k2, nk, (gptr<T>)out.b, out.lb);
  if (threadIdx.x == 0) *out.rank = nk;
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_rkrk(const FTask* tasks, double* wsbase, int* overflow) {
  __shared__ double sh[kShDoubles];
  __shared__ int flag[2];
  if (overflow[1]) return;
  const FTask& t = tasks[blockIdx.x];
  const int k1 = rank_of(t.parts[0].rk), k2 = rank_of(t.parts[1].rk);
  if (k1 == 0 || k2 == 0) {
    if (threadIdx.x == 0) *t.tgt.rank = 0;
    return;
  }
  const int gr = k1 > k2 ? k1 : k2, gc = k1 < k2 ? k1 : k2;
  const int64_t need = (int64_t)gr * gc + (int64_t)gc * gc + 2 * gc + 1;
  // SVD scratch, then the output factors (at most (gr + gc) x gc)
  const auto s3 = (lptr<double>)sh;
  const int64_t core = gr <= kCoreMax ? (int64_t)gr * gc + core_work(gr, gc) : 0;
  if (need + (int64_t)(gr + gc) * gc + core <= kShDoubles)
    rkrk_body<T, lptr<double>, lptr<int>>(t, k1, k2, s3, s3 + need, kShDoubles - need, overflow, flag);
  else
    rkrk_body<T, gptr<double>, gptr<int>>(t, k1, k2, (gptr<double>)(wsbase + t.ws), s3, kShDoubles, overflow, flag);
}

// ---------------------------------------------------------------------------
// ACAFULL: acaFull (compression.cpp:270-355) on a dense temp (modified)
// ---------------------------------------------------------------------------
// entries of the LDS copy: blocks of more than 128 rows or columns (up to that
// they are kept in registers) with at most this many entries
constexpr int kAcaLds = 16384;
// acaFull's stopping estimate after term nu (the reference sums l < nu - 1):
// est += 2 sum_l (a_nu . a_l)(b_nu . b_l) + |a_nu|^2 |b_nu|^2; true when the new
// term is below eps of it.  Each wavefront takes the terms l = w, w + 4, ...
// with wavefront sums, then one workgroup sum.
template <typename T>
__device__ inline bool acafull_converged(const RkRef& out, int m, int n, int nu, double eps, double& est) {
  __shared__ double red[3][kWaves];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const auto OA = (gptr<T>)out.a;
  const auto OB = (gptr<T>)out.b;
  const auto va = OA + (size_t)nu * out.la;
  const auto vb = OB + (size_t)nu * out.lb;
  double part = 0.0, an = 0.0, bn = 0.0;
  for (int l = wv; l + 1 < nu; l += kWaves) {
    double da = 0.0, db = 0.0;
    for (int r = lane; r < m; r += kWave) da += (double)va[r] * (double)OA[r + (size_t)l * out.la];
    for (int c = lane; c < n; c += kWave) db += (double)vb[c] * (double)OB[c + (size_t)l * out.lb];
    part += wave_sum(da) * wave_sum(db);
  }
  for (int r = threadIdx.x; r < m; r += kBlock) an += (double)va[r] * (double)va[r];
  for (int c = threadIdx.x; c < n; c += kBlock) bn += (double)vb[c] * (double)vb[c];
  an = wave_sum(an);
  bn = wave_sum(bn);
  __syncthreads();
  if (lane == 0) {
    red[0][wv] = part;
    red[1][wv] = an;
    red[2][wv] = bn;
  }
  __syncthreads();
  double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int i = 0; i < kWaves; ++i) v[q] += red[q][i];
  const double ab = v[1] * v[2];
  est += 2.0 * v[0] + ab;
  return ab < eps * eps * est;
}

// Blocks of at most 128 x 128: threads 2 c and 2 c + 1 hold the halves of column
// c in registers (storage precision), so a step is one pass over them for the
// update and the next maximum; the pivot column goes through LDS, the pivot
// row's entry of a column is picked by its own thread.  Bound: those passes
// (64 entries per thread).  125 x 125 blocks, ten terms: 170 us in LDS with an index
// division per entry, 56 (FP32) to 71 us (FP64) now.
constexpr int kAcaRows = 64;  // rows per thread
template <typename T>
__device__ void acafull_regs(const FTask& t) {
  __shared__ T col[2 * kAcaRows];
  __shared__ double rv[kWaves];
  __shared__ int ri[kWaves];
  const RkRef out = t.tgt;
  const int m = t.m.s, n = t.n.s;
  const auto D = (cgptr<T>)t.A;
  const int c = threadIdx.x >> 1, h = threadIdx.x & 1, r0 = h * kAcaRows;
  const bool live = c < n;
  T g[kAcaRows];
#pragma unroll
  for (int r = 0; r < kAcaRows; ++r) {
    const int i = r0 + r < m ? r0 + r : m - 1;
    const T v = D[i + (size_t)(live ? c : n - 1) * t.lda];
    g[r] = (live && r0 + r < m) ? v : (T)0;
  }
  int maxk = m < n ? m : n;
  if (maxk > out.cap) maxk = out.cap;
  double est = 0.0;
  int nu = 0;
  for (; nu < maxk; ++nu) {
    // the largest |entry|, the first of equals in column-major order (NaNs lose)
    T best = (T)-1;
    int at = -1;
#pragma unroll
    for (int r = 0; r < kAcaRows; ++r) {
      const T v = g[r] < (T)0 ? -g[r] : g[r];
      if (v > best && live && r0 + r < m) {
        best = v;
        at = r;
      }
    }
    ArgMax a{(double)best, at < 0 ? -1 : r0 + at + c * m};
    a = block_argmax(a, rv, ri);
    if (a.i < 0) break;  // all-NaN block
    const int i = a.i % m, j = a.i / m;
    const auto va = (gptr<T>)out.a + (size_t)nu * out.la;
    const auto vb = (gptr<T>)out.b + (size_t)nu * out.lb;
    if (c == j) {
#pragma unroll
      for (int r = 0; r < kAcaRows; ++r) col[r0 + r] = g[r];
    }
    // the entry of row i in this column (held by one half)
    T x = (T)0;
    const int ir = i - r0;
#pragma unroll
    for (int r = 0; r < kAcaRows; ++r) x = r == ir ? g[r] : x;
    const T y = dpp_swap<0xB1>(x);
    x = (ir >= 0 && ir < kAcaRows) ? x : y;
    __syncthreads();
    const double delta = (double)col[i];
    if (delta == 0.0) break;
    const T b = (T)((double)x / delta);
    if (live && h == 0) vb[c] = b;
    if ((int)threadIdx.x < m) va[threadIdx.x] = col[threadIdx.x];
#pragma unroll
    for (int r = 0; r < kAcaRows; ++r) g[r] -= col[r0 + r] * b;
    __syncthreads();
    if (acafull_converged<T>(out, m, n, nu, t.eps, est)) break;
  }
  __syncthreads();
  if (threadIdx.x == 0) *out.rank = nu;
}

// Other shapes: the dense block is a temporary, so the steps work on it (or on
// its LDS copy) in place.
template <typename T, typename PD>
__device__ void acafull_body(const FTask& t, PD D, int ld) {
  __shared__ double rv[kWaves];
  __shared__ int ri[kWaves];
  const RkRef out = t.tgt;
  const int m = t.m.s, n = t.n.s;
  int maxk = m < n ? m : n;
  if (maxk > out.cap) maxk = out.cap;
  double est = 0.0;
  int nu = 0;
  for (; nu < maxk; ++nu) {
    ArgMax a{-1.0, -1};
    for (int e = threadIdx.x; e < m * n; e += kBlock)
      a = better_max(a, ArgMax{fabs((double)D[e % m + (size_t)(e / m) * ld]), e});
    a = block_argmax(a, rv, ri);
    if (a.i < 0) break;  // all-NaN block
    const int i = a.i % m, j = a.i / m;
    const double delta = (double)D[i + (size_t)j * ld];
    if (delta == 0.0) break;
    const auto va = (gptr<T>)out.a + (size_t)nu * out.la;
    const auto vb = (gptr<T>)out.b + (size_t)nu * out.lb;
    for (int r = threadIdx.x; r < m; r += kBlock) va[r] = D[r + (size_t)j * ld];
    for (int c = threadIdx.x; c < n; c += kBlock) vb[c] = (T)((double)D[i + (size_t)c * ld] / delta);
    __syncthreads();
    for (int e = threadIdx.x; e < m * n; e += kBlock) {
      const int r = e % m, c = e / m;
      D[r + (size_t)c * ld] -= va[r] * vb[c];
    }
    if (acafull_converged<T>(out, m, n, nu, t.eps, est)) break;
  }
  __syncthreads();
  if (threadIdx.x == 0) *out.rank = nu;
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_acafull(const FTask* tasks, const int* fail) {
  __shared__ T dl[kAcaLds];
  if (*fail) return;
  const FTask& t = tasks[blockIdx.x];
  const int m = t.m.s, n = t.n.s;
  if (m <= 2 * kAcaRows && n <= kBlock / 2) {
    acafull_regs<T>(t);
  } else if ((int64_t)m * n <= kAcaLds) {
    stage_in((lptr<T>)dl, m, (cgptr<T>)t.A, 1L, (long)t.lda, m, n);
    __syncthreads();
    acafull_body<T>(t, (lptr<T>)dl, m);
  } else {
    acafull_body<T>(t, (gptr<T>)t.A, t.lda);
  }
}

}  // namespace

bool task_has_tiles(int type) {
  return type == T_GEMM || type == T_TRSM || type == T_ZERO || type == T_AXPY || type == T_SUMK;
}
void append_tiles(const FTask* tasks, int count, std::vector<GemmTile>& tiles) {
  if (count == 0 || !task_has_tiles(tasks[0].type)) return;
  auto parts = [](int n, int side) { return (n + side - 1) / side; };
  bool few = false;
  if (tasks[0].type == T_GEMM) {
    int64_t wide = 0;
    for (int q = 0; q < count; ++q) wide += (int64_t)parts(tasks[q].m.s, TM) * parts(tasks[q].n.s, TN);
    few = wide <= kThinLaunch;
  }
  for (int q = 0; q < count; ++q) {
    const FTask& t = tasks[q];
    switch (t.type) {
      case T_GEMM: {
        const bool thin = few && gemm_is_thin(t);
        const int side = thin ? kThin : TM;
        for (int a = 0; a < parts(t.m.s, side); ++a)
          for (int b = 0; b < parts(t.n.s, side); ++b) tiles.push_back(GemmTile{q, thin ? ~a : a, b});
        break;
      }
      case T_TRSM:
        for (int a = 0; a < parts(t.m.s, kTrsmCols); ++a) tiles.push_back(GemmTile{q, a, 0});
        break;
      default: {  // T_ZERO, T_AXPY, T_SUMK
        const int64_t e = (int64_t)t.m.s * t.n.s;
        for (int64_t a = 0; a * kElemsPerTile < e; ++a) tiles.push_back(GemmTile{q, (int)a, 0});
        break;
      }
    }
  }
}

int64_t fadd_workspace(int m, int n, int K) {
  // dense path only when K >= min(m, n); QR path otherwise (K actual < min)
  const int mn = m < n ? m : n;
  int64_t dense = K >= mn ? (int64_t)m * n + (int64_t)mn * mn + 2 * (int64_t)mn : 0;
  const int kq = K < mn ? K : mn - 1;
  int64_t qr = (int64_t)(m + n) * kq + 6 * (int64_t)kq * kq + 5 * (int64_t)kq;
  return (std::max(dense, qr) + 127) / 64 * 64;
}
int64_t fadd_dense_workspace(int m, int n) {
  const int mn = m < n ? m : n;
  return ((int64_t)m * n + (int64_t)mn * mn + 2 * (int64_t)mn + 127) / 64 * 64;
}
int64_t hodlr_workspace(int cap) { return ((int64_t)5 * cap * cap + cap + 127) / 64 * 64; }
int64_t rkrk_workspace(int k1, int k2) {
  const int64_t a = k1 > k2 ? k1 : k2, b = k1 < k2 ? k1 : k2;
  // G, V, sig, order (+ pad), then the two output factors (a + b) x b
  return (a * b + b * b + 2 * b + 1 + (a + b) * b + 127) / 64 * 64;
}

namespace {
__global__ void k_fill_int(int* p, size_t n, int v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = v;
}
}  // namespace

void launch_fill_int(int* p, size_t n, int v, hipStream_t s) {
  if (n == 0) return;
  const size_t blocks = std::min<size_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_fill_int, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
  HMX_CHECK(hipGetLastError());
}

template <typename T>
void launch_task_kernel(int type, const FTask* tasks, int count, const GemmTile* tiles,
                        int ntiles, double* ws, int* flags, hipStream_t s) {
  if (count == 0 || (task_has_tiles(type) && ntiles == 0)) return;
  switch (type) {
    case T_GEMM:
      hipLaunchKernelGGL(k_gemm<T>, dim3(ntiles), dim3(256), 0, s, tasks, tiles, flags + 1);
      break;
    case T_POTRF:
      hipLaunchKernelGGL(k_potrf<T>, dim3(count), dim3(kBlock), 0, s, tasks, flags + 1);
      break;
    case T_TRSM:
      hipLaunchKernelGGL(k_trsm<T>, dim3(ntiles), dim3(kBlock), 0, s, tasks, tiles, flags + 1);
      break;
    case T_FADD:
      hipLaunchKernelGGL(k_fadd<T>, dim3(count), dim3(kBlock), 0, s, tasks, ws, flags);
      break;
    case T_FADD_DENSE:
      hipLaunchKernelGGL(k_fadd_dense<T>, dim3(count), dim3(kBlock), 0, s, tasks, ws, flags);
      break;
    case T_RKRK:
      hipLaunchKernelGGL(k_rkrk<T>, dim3(count), dim3(kBlock), 0, s, tasks, ws, flags);
      break;
    case T_ACAFULL:
      hipLaunchKernelGGL(k_acafull<T>, dim3(count), dim3(kBlock), 0, s, tasks, flags + 1);
      break;
    case T_ZERO:
      hipLaunchKernelGGL(k_zero<T>, dim3(ntiles), dim3(256), 0, s, tasks, tiles, flags + 1);
      break;
    case T_AXPY:
      hipLaunchKernelGGL(k_axpy<T>, dim3(ntiles), dim3(256), 0, s, tasks, tiles, flags + 1);
      break;
    case T_GETRF:
      hipLaunchKernelGGL(k_getrf<T>, dim3(count), dim3(kBlock), 0, s, tasks, flags + 1);
      break;
    case T_SUMK:
      hipLaunchKernelGGL(k_sumk<T>, dim3(ntiles), dim3(256), 0, s, tasks, tiles, flags + 1);
      break;
    case T_LDLT:
      hipLaunchKernelGGL(k_ldlt<T>, dim3(count), dim3(kBlock), 0, s, tasks, flags + 1);
      break;
    case T_DSCALE:
      hipLaunchKernelGGL(k_dscale<T>, dim3(count * kDscaleSplit), dim3(256), 0, s, tasks, flags + 1);
      break;
    case T_HODLR:
      hipLaunchKernelGGL(k_hodlr<T>, dim3(count), dim3(kBlock), 0, s, tasks, ws, flags + 1);
      break;
    default:
      throw std::runtime_error("unknown task type");
  }
  HMX_CHECK(hipGetLastError());
}

template void launch_task_kernel<double>(int, const FTask*, int, const GemmTile*, int, double*, int*, hipStream_t);
template void launch_task_kernel<float>(int, const FTask*, int, const GemmTile*, int, double*, int*, hipStream_t);

}  // namespace hmx
