// Leaf-level H-gemv (h_matrix.cpp:792-857, rk_matrix.cpp:156-206) as
// deterministic passes over HBM-resident leaves:
//   zpass   : z = B^T x[cols] (and z' = A^T x[rows] for mirrored Rk) per panel
//             chunk of at most kZChunk rows, by a wavefront or a workgroup
//   zreduce : sums the chunks of the panels that have more than one
//   ypass   : one workgroup per run of a destination range's contributions: full
//             leaves (M x, plus M^T x into a slot when mirrored), Rk A z and
//             mirrored Rk B z' restricted to the range's rows; its sums go to a
//             slot of its own
//   yfinal  : y = beta y + alpha (sum of the range's slots), fixed order
// A destination range is a leaf cluster, cut into pieces of at most kYRows
// rows.  Accumulation is in FP64 whatever the storage type.
//
// Bound: HBM (the stored leaves, Rk panels twice: a panel can only be applied
// once all of it is reduced).  The wavefronts are independent: each streams its
// own columns from memory to registers, with no LDS staging and no barrier
// before the one sum at the end of its workgroup, and the plan cuts the
// contributions into runs of similar size, so that small and large matrices
// alike have several workgroups per CU.  One right-hand side is vector
// arithmetic; more of them are products on the FP64 matrix cores, 16 at a time.
//
// Measured against one y workgroup per leaf cluster with its leaves staged in
// LDS, and one z workgroup per chunk: FP64, one right-hand side, N = 2,000:
// y pass 46.6 -> 7.1 us (16 -> 173 workgroups); N = 200,000: z 182 + 40 (its
// sums) -> 163 + 22, y 414 -> 336 us (2.4 GB read at 4.6 TB/s); complex
// N = 20,000: y 855 -> 272 us; 8 right-hand sides, N = 50,021: z 185 -> 76,
// y 263 -> 197 us; 65 right-hand sides, N = 8,000: y 2,564 -> 475 us.
#include <algorithm>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "kernels.hpp"

namespace hmx {

namespace {

constexpr int kYMfma = 16;            // right-hand sides of a matrix-core tile
constexpr int kYv = kYRows / kWave;   // rows per lane
constexpr int kYb = kYRows / 16;      // 16-row blocks of a destination range

typedef double gv_double4 __attribute__((ext_vector_type(4)));

__device__ inline gv_double4 mfma4(double a, double b, gv_double4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ inline int64_t lane_read64(int64_t v, int lane) {
  const int lo = __builtin_amdgcn_readlane((int)(uint32_t)v, lane);
  const int hi = __builtin_amdgcn_readlane((int)(v >> 32), lane);
  return ((int64_t)hi << 32) | (uint32_t)lo;
}

// Sum of v over each row of 16 lanes, in all of them.
__device__ inline double row_sum(double v) {
  v += dpp_swap<0xB1>(v);
  v += dpp_swap<0x4E>(v);
  v += dpp_swap<0x141>(v);
  v += dpp_swap<0x140>(v);
  return v;
}
__device__ inline double sum_rows(double v) {  // over the four rows of 16 lanes
  v += __shfl_xor(v, 16, kWave);
  v += __shfl_xor(v, 32, kWave);
  return v;
}

// Column sums of a stream of columns, 16 at a time: add() takes the lanes'
// partial sums of column l, and after 16 columns (or the last one) lane i < 16
// holds the total of column (l & ~15) + i.
struct ColumnSums {
  double t = 0.0;
  __device__ void add(int l, double s) {
    s = row_sum(s);
    t = (int)(threadIdx.x & 15) == (l & 15) ? s : t;
  }
  __device__ double total() { return sum_rows(t); }
};

// z = P^T x of one chunk, one right-hand side.  A lane keeps its entries of x
// (rows lane + 64 v) in registers; the loads of 16 / kR64 columns are issued
// together (clamped to the chunk and the rank).
template <typename T, int kR64>
__device__ void zpass1_chunk(const T* P, int ld, const T* xs, int rows, int k, double* z) {
  constexpr int kC = 16 / kR64;
  const int lane = threadIdx.x & (kWave - 1);
  const int rm = rows - 1;
  double xr[kR64];
#pragma unroll
  for (int v = 0; v < kR64; ++v) {
    const int i = lane + kWave * v;
    const double t = (double)xs[i < rm ? i : rm];
    xr[v] = i < rows ? t : 0.0;
  }
  for (int l16 = 0; l16 < k; l16 += 16) {
    ColumnSums sums;
    const int lend = l16 + 16 < k ? l16 + 16 : k;
    for (int l0 = l16; l0 < lend; l0 += kC) {
      double p[kC][kR64];
#pragma unroll
      for (int c = 0; c < kC; ++c) {
        const T* col = P + (size_t)(l0 + c < k ? l0 + c : k - 1) * ld;
#pragma unroll
        for (int v = 0; v < kR64; ++v) {
          const int i = lane + kWave * v;
          p[c][v] = (double)col[i < rm ? i : rm];
        }
      }
#pragma unroll
      for (int c = 0; c < kC; ++c) {
        double s = 0.0;
#pragma unroll
        for (int v = 0; v < kR64; ++v) s += p[c][v] * xr[v];
        sums.add(l0 + c, s);
      }
    }
    const double t = sums.total();
    if (lane < 16 && l16 + lane < k) z[l16 + lane] = t;
  }
}

template <typename T>
__device__ void zpass1_rows(const T* P, int ld, const T* xs, int rows, int k, double* z) {
  if (rows <= 64) zpass1_chunk<T, 1>(P, ld, xs, rows, k, z);
  else if (rows <= 128) zpass1_chunk<T, 2>(P, ld, xs, rows, k, z);
  else zpass1_chunk<T, 4>(P, ld, xs, rows, k, z);
}

// The first nlong items (more than kZShort rows) take a workgroup each, a
// quarter of the rows per wavefront; the others a wavefront each.
constexpr int kZShort = kZChunk / kWaves;
constexpr int kZCols = 64;  // columns summed over the wavefronts at a time

template <typename T>
__global__ void __launch_bounds__(kBlock) k_zpass1(const int* ranks, const T* arena, const ZItem* items, int nlong,
                                                   int count, const T* x, double* zpart, double* z) {
  __shared__ double part[kWaves][kZCols];
  const int w = threadIdx.x / kWave;
  const bool shared_item = (int)blockIdx.x < nlong;
  const int q = shared_item ? (int)blockIdx.x : nlong + ((int)blockIdx.x - nlong) * kWaves + w;
  if (q >= count) return;
  const ZItem it = items[q];
  const int k = ranks[it.leaf];
  const T* P = arena + it.p;
  const T* xs = x + it.x0;
  double* out = (it.part ? zpart : z) + it.z;
  if (!shared_item) {
    zpass1_rows<T>(P, it.ld, xs, it.rows, k, out);
    return;
  }
  const int per = (it.rows + kWaves - 1) / kWaves, r0 = w * per, rows = it.rows - r0 < per ? it.rows - r0 : per;
  for (int l0 = 0; l0 < k; l0 += kZCols) {
    const int kc = k - l0 < kZCols ? k - l0 : kZCols;
    zpass1_rows<T>(P + r0 + (size_t)l0 * it.ld, it.ld, xs + r0, rows, kc, part[w]);
    __syncthreads();
    if ((int)threadIdx.x < kc)
      out[l0 + threadIdx.x] = (part[0][threadIdx.x] + part[1][threadIdx.x]) + (part[2][threadIdx.x] + part[3][threadIdx.x]);
    __syncthreads();
  }
}

// Four consecutive entries p[0..3]; those at or past n count as zero.
template <typename T>
__device__ inline void load4(const T* p, int n, double (&v)[4]) {
  if (n >= 4) {
    typedef T vec __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    const vec t = *(const vec*)p;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = (double)t[q];
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double t = n > 0 ? (double)p[q < n ? q : n - 1] : 0.0;
      v[q] = q < n ? t : 0.0;
    }
  }
}

// z = P^T X of one chunk for the right-hand sides [16 kT y, ...) of block row y:
// lane i + 16 kk holds rows 4 kk .. 4 kk + 3 of a 16-row slab, of panel column
// i (A operand) and of right-hand side i (B operand); MFMA q of a slab takes
// their q-th rows.
template <typename T, int kT>
__global__ void __launch_bounds__(kBlock) k_zpass(const int* ranks, const T* arena, const ZItem* items, int nlong,
                                                  int count, const T* x, int ldx, int nrhs, double* zpart, double* z) {
  __shared__ double part[kWaves][kT][4][kWave];
  const int w = threadIdx.x / kWave;
  const bool shared_item = (int)blockIdx.x < nlong;
  const int q = shared_item ? (int)blockIdx.x : nlong + ((int)blockIdx.x - nlong) * kWaves + w;
  if (q >= count) return;
  const ZItem it = items[q];
  const int k = ranks[it.leaf];
  // this wavefront's rows: all of a short item, a quarter (whole slabs) of a long one
  const int per = shared_item ? ((it.rows + 16 * kWaves - 1) / (16 * kWaves)) * 16 : it.rows;
  const int rbeg = shared_item ? w * per : 0, rend = rbeg + per < it.rows ? rbeg + per : it.rows;
  const int lane = threadIdx.x & (kWave - 1), ii = lane & 15, kk = lane >> 4;
  const int rhs0 = blockIdx.y * kYMfma * kT;
  double* out = (it.part ? zpart : z) + it.z * nrhs;
  const T* xs = x + it.x0;
  for (int l0 = 0; l0 < k; l0 += 16) {
    const bool in = l0 + ii < k;
    const T* col = arena + it.p + (size_t)(in ? l0 + ii : k - 1) * it.ld;
    gv_double4 acc[kT];
#pragma unroll
    for (int t = 0; t < kT; ++t) acc[t] = gv_double4{0.0, 0.0, 0.0, 0.0};
    constexpr int kU = 4;  // slabs in flight
    for (int r0 = rbeg; r0 < rend; r0 += 16 * kU) {
      double a[kU][4], b[kU][kT][4];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int r = r0 + 16 * u + 4 * kk, rc = r < rend ? r : 0;
        load4<T>(col + rc, in ? rend - r : 0, a[u]);
#pragma unroll
        for (int t = 0; t < kT; ++t) {
          const int j = rhs0 + kYMfma * t + ii;
          load4<T>(xs + rc + (size_t)(j < nrhs ? j : 0) * ldx, j < nrhs ? rend - r : 0, b[u][t]);
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
#pragma unroll
        for (int t = 0; t < kT; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t] = mfma4(a[u][e], b[u][t][e], acc[t]);
    }
    if (shared_item) {
#pragma unroll
      for (int t = 0; t < kT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) part[w][t][v][lane] = acc[t][v];
      __syncthreads();
      // wavefront w sums element w of the lanes
#pragma unroll
      for (int t = 0; t < kT; ++t) {
        const int j = rhs0 + kYMfma * t + ii, l = l0 + kk + 4 * w;
        const double s = (part[0][t][w][lane] + part[1][t][w][lane]) + (part[2][t][w][lane] + part[3][t][w][lane]);
        if (l < k && j < nrhs) out[l + (size_t)j * it.cap] = s;
      }
      __syncthreads();
      continue;
    }
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      const int j = rhs0 + kYMfma * t + ii;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int l = l0 + kk + 4 * v;
        if (l < k && j < nrhs) out[l + (size_t)j * it.cap] = acc[t][v];
      }
    }
  }
}

__global__ void k_zreduce(const ZReduce* red, const int* ranks, const double* zpart, int nrhs, double* z) {
  const ZReduce rd = red[blockIdx.x];
  const int k = ranks[rd.leaf];
  for (int e = threadIdx.x; e < k * nrhs; e += blockDim.x) {
    const int l = e % k, r = e / k;
    double s = 0.0;
    for (int q = 0; q < rd.count; ++q) s += zpart[(rd.part + (int64_t)q * rd.cap) * nrhs + l + (size_t)r * rd.cap];
    z[rd.z * nrhs + l + (size_t)r * rd.cap] = s;
  }
}

// The records of up to 64 contributions of a wavefront, one per lane.
struct YRecords {
  int64_t p, z;
  int leaf, ld, n, x0, cap, col0;
  __device__ YRecords(const YContrib* c, const int* ranks) {
    const YContrib r = *c;
    p = r.p;
    z = r.z;
    leaf = r.leaf;
    ld = r.ld;
    x0 = r.x0;
    cap = r.cap;
    col0 = r.col0;
    n = leaf >= 0 ? ranks[leaf] : r.n;
  }
};

// One right-hand side: a lane owns rows lane + 64 v of the range.
template <typename T>
__global__ void __launch_bounds__(kBlock) k_ypass1(const int* ranks, const T* arena, const YItem* items,
                                                   const YContrib* contrib, const double* z, double* slots,
                                                   const T* x) {
  __shared__ double part[kWaves][kYRows];
  const YItem it = items[blockIdx.x];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  int row[kYv];
  double xi[kYv], acc[kYv];
#pragma unroll
  for (int v = 0; v < kYv; ++v) {
    const int i = lane + kWave * v;
    row[v] = i < it.len ? i : it.len - 1;
    xi[v] = 0.0;
    acc[v] = 0.0;
  }
  // x_I of mirrored leaves: the rows' numbering is x's in symmetric storage
  // only (with other column trees it may reach past x)
  if (it.mirrored)
#pragma unroll
    for (int v = 0; v < kYv; ++v) {
      const double t = (double)x[it.x0 + row[v]];
      xi[v] = lane + kWave * v < it.len ? t : 0.0;
    }
  constexpr int kC = 8;  // columns in flight
  const int cnt = it.end - it.beg;
  for (int u0 = w; u0 < cnt; u0 += kWaves * kWave) {
    const int mu = u0 + kWaves * lane;
    const YRecords rec(contrib + it.beg + (mu < cnt ? mu : u0), ranks);
    const int left = (cnt - u0 + kWaves - 1) / kWaves, nu = left < kWave ? left : kWave;
    for (int u = 0; u < nu; ++u) {
      const T* P = arena + lane_read64(rec.p, u);
      const int64_t zo = lane_read64(rec.z, u);
      const int leaf = __builtin_amdgcn_readlane(rec.leaf, u), ld = __builtin_amdgcn_readlane(rec.ld, u);
      const int n = __builtin_amdgcn_readlane(rec.n, u), x0 = __builtin_amdgcn_readlane(rec.x0, u);
      if (leaf >= 0) {
        for (int l64 = 0; l64 < n; l64 += kWave) {
          const int m = n - l64 < kWave ? n - l64 : kWave;
          const double zl = z[zo + l64 + (lane < m ? lane : m - 1)];
          for (int l0 = 0; l0 < m; l0 += kC) {
            double p[kC][kYv];
#pragma unroll
            for (int c = 0; c < kC; ++c)
#pragma unroll
              for (int v = 0; v < kYv; ++v)
                p[c][v] = (double)P[(size_t)(l64 + (l0 + c < m ? l0 + c : m - 1)) * ld + row[v]];
#pragma unroll
            for (int c = 0; c < kC; ++c) {
              const double b = l0 + c < m ? lane_read(zl, l0 + c < m ? l0 + c : 0) : 0.0;
#pragma unroll
              for (int v = 0; v < kYv; ++v) acc[v] += p[c][v] * b;
            }
          }
        }
        continue;
      }
      // a full leaf's columns (at most kYCols of them)
      const double xl = (double)x[x0 + (lane < n ? lane : n - 1)];
      const int col0 = __builtin_amdgcn_readlane(rec.col0, u);
      for (int l16 = 0; l16 < n; l16 += 16) {
        ColumnSums sums;
        const int lend = l16 + 16 < n ? l16 + 16 : n;
        for (int l0 = l16; l0 < lend; l0 += kC) {
          double p[kC][kYv];
#pragma unroll
          for (int c = 0; c < kC; ++c)
#pragma unroll
            for (int v = 0; v < kYv; ++v)
              p[c][v] = (double)P[(size_t)(l0 + c < n ? l0 + c : n - 1) * ld + row[v]];
#pragma unroll
          for (int c = 0; c < kC; ++c) {
            const double b = l0 + c < n ? lane_read(xl, l0 + c < n ? l0 + c : 0) : 0.0;
            double s = 0.0;
#pragma unroll
            for (int v = 0; v < kYv; ++v) {
              acc[v] += p[c][v] * b;
              s += p[c][v] * xi[v];
            }
            if (zo >= 0) sums.add(l0 + c, s);
          }
        }
        if (zo >= 0) {
          const double t = sums.total();
          if (lane < 16 && l16 + lane < n) slots[zo + col0 + l16 + lane] = t;
        }
      }
    }
  }
#pragma unroll
  for (int v = 0; v < kYv; ++v) part[w][lane + kWave * v] = acc[v];
  __syncthreads();
  for (int i = threadIdx.x; i < it.len; i += kBlock)
    slots[it.out + i] = (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]);
}

// Right-hand sides [16 kT y, ...) of block row y on the matrix cores.  A
// wavefront takes 16 columns of a contribution at a time: coalesced loads into
// registers (issued while the previous 16 columns are multiplied), from there
// to its own part of LDS, where both operand layouts of the 16 x 16 blocks are
// read: rows across lanes for P Z (Z the rows of X or of z that belong to the
// columns), columns across lanes for M^T X of a mirrored full leaf.  Row r of
// column c sits at c kYRows + (r ^ 4 c), which spreads both reads over the
// banks.  Wavefronts meet only in the sum at the end.
template <typename T, int kT>
__global__ void __launch_bounds__(kBlock, kT == 1 ? 2 : 1) k_ypass(const int* ranks, const T* arena, const YItem* items,
                                                  const YContrib* contrib, const double* z, double* slots,
                                                  const T* x, int ldx, int nrhs) {
  constexpr int kNr = kYMfma * kT;
  __shared__ double buf[kYRows * kNr];  // X_I (ld kYRows), then the sums
  __shared__ double tile[kWaves][16 * kYRows];
  const YItem it = items[blockIdx.x];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave, ii = lane & 15, kk = lane >> 4;
  const int rhs0 = blockIdx.y * kNr, nr = nrhs - rhs0 < kNr ? nrhs - rhs0 : kNr;
  const int nb = (it.len + 15) / 16;
  double* tl = tile[w];
  if (it.mirrored)
    for (int e = threadIdx.x; e < kYRows * kNr; e += kBlock) {
      const int i = e % kYRows, r = e / kYRows;
      const double t = (double)x[it.x0 + (i < it.len ? i : it.len - 1) + (size_t)(rhs0 + (r < nr ? r : nr - 1)) * ldx];
      buf[e] = (i < it.len && r < nr) ? t : 0.0;
    }
  __syncthreads();
  unsigned row[kYv];
#pragma unroll
  for (int v = 0; v < kYv; ++v) row[v] = lane + kWave * v < it.len ? lane + kWave * v : it.len - 1;
  gv_double4 acc[kYb][kT];
#pragma unroll
  for (int b = 0; b < kYb; ++b)
#pragma unroll
    for (int t = 0; t < kT; ++t) acc[b][t] = gv_double4{0.0, 0.0, 0.0, 0.0};
  const int cnt = it.end - it.beg;
  for (int u0 = w; u0 < cnt; u0 += kWaves * kWave) {
    const int mu = u0 + kWaves * lane;
    const YRecords rec(contrib + it.beg + (mu < cnt ? mu : u0), ranks);
    const int left = (cnt - u0 + kWaves - 1) / kWaves, nu = left < kWave ? left : kWave;
    // as loaded: converted and masked only where they are used, so that
    // nothing waits for them before
    T p[16][kYv];
    uint64_t zb[kT][4];
    // columns [c0, c0 + 16) of contribution u, and rows of Z: element e of lane
    // i + 16 kk is row c0 + 4 e + kk, right-hand side i
    auto load = [&](int u, int c0) __attribute__((always_inline)) {
      const T* P = arena + lane_read64(rec.p, u);
      const int64_t zo = lane_read64(rec.z, u);
      const int leaf = __builtin_amdgcn_readlane(rec.leaf, u), ld = __builtin_amdgcn_readlane(rec.ld, u);
      const int n = __builtin_amdgcn_readlane(rec.n, u), x0 = __builtin_amdgcn_readlane(rec.x0, u);
      const int cap = __builtin_amdgcn_readlane(rec.cap, u);
      auto columns = [&](auto H) __attribute__((always_inline)) {
        constexpr int h = decltype(H)::value;
#pragma unroll
        for (int c = h; c < h + 8; ++c)
#pragma unroll
          for (int v = 0; v < kYv; ++v) p[c][v] = (P + (size_t)(c0 + c < n ? c0 + c : n - 1) * ld)[row[v]];
      };
      columns(std::integral_constant<int, 0>{});
      if (n - c0 > 8) columns(std::integral_constant<int, 8>{});
#pragma unroll
      for (int t = 0; t < kT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = kYMfma * t + ii, jc = j < nr ? j : nr - 1;
          const int l = c0 + 4 * e + kk, lc = l < n ? l : n - 1;
          if (leaf >= 0)
            zb[t][e] = __double_as_longlong(z[zo * nrhs + lc + (size_t)(rhs0 + jc) * cap]);
          else if constexpr (sizeof(T) == 8)
            zb[t][e] = __double_as_longlong(x[x0 + lc + (size_t)(rhs0 + jc) * ldx]);
          else
            zb[t][e] = __float_as_uint(x[x0 + lc + (size_t)(rhs0 + jc) * ldx]);
        }
    };
    int u = 0, c0 = 0, n = __builtin_amdgcn_readlane(rec.n, 0);
    while (u < nu && n <= 0) n = ++u < nu ? __builtin_amdgcn_readlane(rec.n, u) : 0;  // empty panels
    if (u < nu) load(u, 0);
    while (u < nu) {
      const int n16 = n - c0 < 16 ? n - c0 : 16, cu = u, cc = c0;
      const bool rk = __builtin_amdgcn_readlane(rec.leaf, u) >= 0;
      double zc[kT][4];
#pragma unroll
      for (int t = 0; t < kT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          double b = __longlong_as_double(zb[t][e]);
          if constexpr (sizeof(T) == 4)
            if (!rk) b = (double)__uint_as_float((uint32_t)zb[t][e]);
          zc[t][e] = (4 * e + kk < n16 && kYMfma * t + ii < nr) ? b : 0.0;
        }
      __builtin_amdgcn_wave_barrier();
      auto store = [&](auto H) __attribute__((always_inline)) {
        constexpr int h = decltype(H)::value;
#pragma unroll
        for (int c = h; c < h + 8; ++c)
#pragma unroll
          for (int v = 0; v < kYv; ++v)
            tl[c * kYRows + ((lane + kWave * v) ^ (4 * c))] = (c < n16 && lane + kWave * v < it.len) ? (double)p[c][v] : 0.0;
      };
      store(std::integral_constant<int, 0>{});
      if (n16 > 8) store(std::integral_constant<int, 8>{});
      // the next 16 columns
      c0 += 16;
      while (c0 >= n && u < nu) {
        c0 = 0;
        n = ++u < nu ? __builtin_amdgcn_readlane(rec.n, u) : 0;
      }
      if (u < nu) load(u, c0);
      __builtin_amdgcn_wave_barrier();
      const int64_t zo = lane_read64(rec.z, cu);
      const bool mir = !rk && zo >= 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (4 * e >= n16) continue;
        const int c = 4 * e + kk;
#pragma unroll
        for (int q = 0; q < kYb; ++q) {
          if (q >= nb) continue;
          const double a = tl[c * kYRows + ((16 * q + ii) ^ (4 * c))];
#pragma unroll
          for (int t = 0; t < kT; ++t) acc[q][t] = mfma4(a, zc[t][e], acc[q][t]);
        }
      }
      if (mir) {
        if (n16 <= 8) {
          // columns 8 .. 15 of the tile hold an earlier contribution's
#pragma unroll
          for (int c = 8; c < 16; ++c)
#pragma unroll
            for (int v = 0; v < kYv; ++v) tl[c * kYRows + lane + kWave * v] = 0.0;
          __builtin_amdgcn_wave_barrier();
        }
        gv_double4 tr[kT];
#pragma unroll
        for (int t = 0; t < kT; ++t) tr[t] = gv_double4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < kYb; ++q) {
          if (q >= nb) continue;
          const double* at = tl + ii * kYRows + ((16 * q + 4 * kk) ^ (4 * ii));
#pragma unroll
          for (int t = 0; t < kT; ++t) {
            const double* xi = buf + (kYMfma * t + ii) * kYRows + 16 * q + 4 * kk;
#pragma unroll
            for (int e = 0; e < 4; ++e) tr[t] = mfma4(at[e], xi[e], tr[t]);
          }
        }
        const int cap = __builtin_amdgcn_readlane(rec.cap, cu);
        double* out = slots + zo * nrhs + (size_t)rhs0 * cap + __builtin_amdgcn_readlane(rec.col0, cu) + cc;
#pragma unroll
        for (int t = 0; t < kT; ++t)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int c = kk + 4 * v, j = kYMfma * t + ii;
            if (c < n16 && j < nr) out[c + (size_t)j * cap] = tr[t][v];
          }
      }
    }
  }
  // the wavefronts' sums, one after the other
  for (int s = 0; s < kWaves; ++s) {
    __syncthreads();
    if (s != w) continue;
#pragma unroll
    for (int q = 0; q < kYb; ++q)
#pragma unroll
      for (int t = 0; t < kT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          double* o = buf + (16 * q + kk + 4 * v) + (kYMfma * t + ii) * kYRows;
          *o = s == 0 ? acc[q][t][v] : *o + acc[q][t][v];
        }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kYRows * nr; e += kBlock) {
    const int i = e % kYRows, r = e / kYRows;
    if (i < it.len) slots[it.out * nrhs + i + (size_t)(rhs0 + r) * it.len] = buf[e];
  }
}

// one right-hand side per block row
template <typename T>
__global__ void __launch_bounds__(kYRows) k_yfinal(const YFinal* items, const int64_t* slot_list, const double* slots,
                                                   T* y, int ldy, int nrhs, double alpha, double beta) {
  const YFinal it = items[blockIdx.x];
  const int r = blockIdx.y;
  for (int i = threadIdx.x; i < it.len; i += kYRows) {
    double s = 0.0;
    int q = it.beg;
    for (; q + 4 <= it.end; q += 4) {
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = slots[slot_list[q + u] * nrhs + i + (size_t)r * it.len];
#pragma unroll
      for (int u = 0; u < 4; ++u) s += v[u];
    }
    for (; q < it.end; ++q) s += slots[slot_list[q] * nrhs + i + (size_t)r * it.len];
    T* py = y + it.r0 + i + (size_t)r * ldy;
    const double old = (beta == 0.0) ? 0.0 : beta * (double)(*py);
    *py = (T)(old + alpha * s);
  }
}

template <typename S, typename D>
__global__ void k_convert(const S* src, D* dst, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    dst[i] = (D)src[i];
}

}  // namespace

template <typename S, typename D>
void launch_convert(const S* src, D* dst, size_t n, hipStream_t s) {
  if (n == 0) return;
  size_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL((k_convert<S, D>), dim3((unsigned)blocks), dim3(256), 0, s, src, dst, n);
  HMX_CHECK(hipGetLastError());
}
template void launch_convert<double, float>(const double*, float*, size_t, hipStream_t);

namespace {
__global__ void k_add_f2d(double* x, const float* d, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    x[i] += (double)d[i];
}
__global__ void k_col_sumsq(const double* v, int n, double* out) {
  __shared__ double red[kWaves];
  const double* c = v + (size_t)blockIdx.x * n;
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += kBlock) s += c[i] * c[i];
  s = block_sum(s, red);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}
}  // namespace

void launch_vec_add_f2d(double* x, const float* d, size_t n, hipStream_t s) {
  size_t blocks = std::min<size_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_add_f2d, dim3((unsigned)blocks), dim3(256), 0, s, x, d, n);
  HMX_CHECK(hipGetLastError());
}
void launch_col_sumsq(const double* v, int n, int nrhs, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_col_sumsq, dim3(nrhs), dim3(kBlock), 0, s, v, n, out);
  HMX_CHECK(hipGetLastError());
}

// ---- conjugate-gradient steps on n x nrhs column blocks (one system per column)
namespace {
__global__ void k_col_dot(const double* a, const double* b, int n, double* out) {
  __shared__ double red[kWaves];
  const double* ca = a + (size_t)blockIdx.x * n;
  const double* cb = b + (size_t)blockIdx.x * n;
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += kBlock) s += ca[i] * cb[i];
  s = block_sum(s, red);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}
// alpha_j = rz_j / pq_j (0 when pq_j is 0): x += alpha p, r -= alpha q
__global__ void k_cg_xr(double* x, double* r, const double* p, const double* q, const double* rz,
                        const double* pq, int n, int nrhs) {
  const size_t cnt = (size_t)n * nrhs;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < cnt; e += (size_t)gridDim.x * blockDim.x) {
    const int j = (int)(e / n);
    const double a = pq[j] != 0.0 ? rz[j] / pq[j] : 0.0;
    x[e] += a * p[e];
    r[e] -= a * q[e];
  }
}
// beta_j = rz_new_j / rz_old_j (0 when rz_old_j is 0): p = z + beta p
__global__ void k_cg_p(double* p, const double* z, const double* rz_new, const double* rz_old, int n, int nrhs) {
  const size_t cnt = (size_t)n * nrhs;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < cnt; e += (size_t)gridDim.x * blockDim.x) {
    const int j = (int)(e / n);
    const double b = rz_old[j] != 0.0 ? rz_new[j] / rz_old[j] : 0.0;
    p[e] = z[e] + b * p[e];
  }
}
unsigned grid_for(size_t cnt) { return (unsigned)std::min<size_t>((cnt + 255) / 256, 65536); }
}  // namespace

namespace {
__global__ void k_vec_add(double* x, const double* d, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    x[i] += d[i];
}
}  // namespace
void launch_vec_add(double* x, const double* d, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_vec_add, dim3(grid_for(n)), dim3(256), 0, s, x, d, n);
  HMX_CHECK(hipGetLastError());
}
void launch_col_dot(const double* a, const double* b, int n, int nrhs, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_col_dot, dim3(nrhs), dim3(kBlock), 0, s, a, b, n, out);
  HMX_CHECK(hipGetLastError());
}
void launch_cg_xr(double* x, double* r, const double* p, const double* q, const double* rz, const double* pq,
                  int n, int nrhs, hipStream_t s) {
  hipLaunchKernelGGL(k_cg_xr, dim3(grid_for((size_t)n * nrhs)), dim3(256), 0, s, x, r, p, q, rz, pq, n, nrhs);
  HMX_CHECK(hipGetLastError());
}
void launch_cg_p(double* p, const double* z, const double* rz_new, const double* rz_old, int n, int nrhs,
                 hipStream_t s) {
  hipLaunchKernelGGL(k_cg_p, dim3(grid_for((size_t)n * nrhs)), dim3(256), 0, s, p, z, rz_new, rz_old, n, nrhs);
  HMX_CHECK(hipGetLastError());
}
template void launch_convert<float, double>(const float*, double*, size_t, hipStream_t);

// One right-hand side takes the vector kernels, two and more the matrix cores,
// whose tiles are 16 wide: a whole product of 1 / 2 / 4 / 8 / 16 right-hand sides
// measured 97 / 258 / 262 / 273 / 288 us (N = 50,021, FP64), 27 / 93 / 94 / 96 / 98
// (N = 10,007, leaves of 100 rows), 54 / 190 / 192 / 197 / 204 (N = 30,011, FP32,
// non-symmetric) and 92 / 244 / 248 / 255 / 244 us (N = 8,000, complex).  Below
// the line a tile is mostly zeros: two right-hand sides cost more than two
// products of one each, three about as much as three; with a vector form for
// several right-hand sides at once (eight at a time, leaves in LDS) two took 326,
// 158, 275 and 811 us.
template <typename T>
void launch_gemv_zpass(const int* ranks, const T* arena, const ZItem* items, int nlong, int count,
                       const T* x, int ldx, int nrhs, double* zpart, double* z, hipStream_t s) {
  if (count == 0) return;
  const unsigned blocks = (unsigned)(nlong + (count - nlong + kWaves - 1) / kWaves);
  if (nrhs == 1)
    hipLaunchKernelGGL(k_zpass1<T>, dim3(blocks), dim3(kBlock), 0, s, ranks, arena, items, nlong, count, x,
                       zpart, z);
  else if (nrhs <= kYMfma)
    hipLaunchKernelGGL((k_zpass<T, 1>), dim3(blocks), dim3(kBlock), 0, s, ranks, arena, items, nlong, count, x,
                       ldx, nrhs, zpart, z);
  else
    // more than one tile of right-hand sides: two per wavefront, so that the
    // panels are read half as often
    hipLaunchKernelGGL((k_zpass<T, 2>), dim3(blocks, (nrhs + 2 * kYMfma - 1) / (2 * kYMfma)), dim3(kBlock), 0,
                       s, ranks, arena, items, nlong, count, x, ldx, nrhs, zpart, z);
  HMX_CHECK(hipGetLastError());
}

void launch_gemv_zreduce(const ZReduce* red, int count, const int* ranks, const double* zpart, int nrhs,
                         double* z, hipStream_t s) {
  if (count == 0) return;
  hipLaunchKernelGGL(k_zreduce, dim3(count), dim3(128), 0, s, red, ranks, zpart, nrhs, z);
  HMX_CHECK(hipGetLastError());
}

template <typename T>
void launch_gemv_ypass(const int* ranks, const T* arena, const YItem* items, int count,
                       const YContrib* contrib, const double* z, double* slots, const T* x, int ldx,
                       int nrhs, hipStream_t s) {
  if (count == 0) return;
  if (nrhs == 1)
    hipLaunchKernelGGL(k_ypass1<T>, dim3(count), dim3(kBlock), 0, s, ranks, arena, items, contrib, z,
                       slots, x);
  else if (nrhs <= kYMfma)
    hipLaunchKernelGGL((k_ypass<T, 1>), dim3(count), dim3(kBlock), 0, s, ranks, arena, items, contrib, z,
                       slots, x, ldx, nrhs);
  else
    hipLaunchKernelGGL((k_ypass<T, 2>), dim3(count, (nrhs + 2 * kYMfma - 1) / (2 * kYMfma)), dim3(kBlock), 0,
                       s, ranks, arena, items, contrib, z, slots, x, ldx, nrhs);
  HMX_CHECK(hipGetLastError());
}

template <typename T>
void launch_gemv_yfinal(const YFinal* items, int count, const int64_t* slot_list, const double* slots,
                        T* y, int ldy, int nrhs, double alpha, double beta, hipStream_t s) {
  if (count == 0) return;
  hipLaunchKernelGGL(k_yfinal<T>, dim3(count, nrhs), dim3(kYRows), 0, s, items, slot_list, slots, y, ldy,
                     nrhs, alpha, beta);
  HMX_CHECK(hipGetLastError());
}

#define HMX_INST(T)                                                                                 \
  template void launch_gemv_zpass<T>(const int*, const T*, const ZItem*, int, int, const T*, int, int, \
                                     double*, double*, hipStream_t);                                 \
  template void launch_gemv_ypass<T>(const int*, const T*, const YItem*, int, const YContrib*,      \
                                     const double*, double*, const T*, int, int, hipStream_t);       \
  template void launch_gemv_yfinal<T>(const YFinal*, int, const int64_t*, const double*, T*, int,   \
                                      int, double, double, hipStream_t);
HMX_INST(double)
HMX_INST(float)

// Device scratch of the allocation-free H-gemv entry point: a fixed array in
// the code object, so each GPU that loads the library holds its own copy (at
// its own address) until the process ends.  Every call on one GPU shares it
// and leaves its contents behind; the H-gemv passes write every scratch entry
// they read, so nothing needs clearing between calls.  Host code must not use
// the array's name as a device address: noalloc_gemv_scratch() returns the
// device address looked up with hipGetSymbolAddress, once per device.
static __device__ __align__(256) double scratch[kNoAllocScratchBytes / sizeof(double)];

double* noalloc_gemv_scratch(size_t* elems) {
  static std::mutex mu;
  static std::vector<double*> ptr;
  int dev = 0;
  HMX_CHECK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  if ((int)ptr.size() <= dev) ptr.resize(dev + 1, nullptr);
  if (!ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      throw std::runtime_error(std::string("hipGetSymbolAddress(scratch) failed: ") +
                               hipGetErrorString(e));
    ptr[dev] = static_cast<double*>(p);
  }
  *elems = kNoAllocScratchBytes / sizeof(double);
  return ptr[dev];
}

}  // namespace hmx
