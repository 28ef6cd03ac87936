// One-workgroup dense linear algebra used inside the batched task kernels:
// Householder QR of a tall panel, application of its Q, one-sided (Hestenes)
// Jacobi SVD, and the singular-value ordering / truncation rule.
//
// The routines work on column-major matrices that may live in LDS or in
// global memory (generic pointers) and end with a synchronisation of the
// threads that ran them.  Arithmetic is FP64; callers convert at the boundary.
#pragma once
#include "dev_common.hpp"

namespace hmx {

constexpr int kQrChunk = 16;  // size factor of the reduction scratch kept by callers

// The routines below are written for a "team" of kLanes threads: one
// wavefront (kLanes == kWave, synchronised by wave_barrier: LDS accesses of
// one wavefront complete in program order) or the whole workgroup
// (kLanes == kBlock, __syncthreads).  Work items (columns, column pairs) are
// spread over aligned groups of g lanes, g as large as the item count allows;
// a group reduces its partial sums with group_sum, so a reduction costs
// log2(g) register exchanges instead of a round trip through LDS.

template <int kLanes>
__device__ inline void team_sync() {
  if constexpr (kLanes == kWave)
    __builtin_amdgcn_wave_barrier();
  else
    __syncthreads();
}

// Thread index within its team; teams are aligned groups of kLanes threads
// (a power of two: a wavefront, half or all of the workgroup).  Teams
// smaller than the workgroup but larger than a wavefront synchronise with
// workgroup barriers, so all teams must pass the same number of them.
template <int kLanes>
__device__ inline int team_tid() {
  return (int)(threadIdx.x & (kLanes - 1));
}

// Largest power of two g <= kWave with g * items <= lanes (at least 1).
__device__ inline int group_lanes(int items, int lanes) {
  int g = kWave;
  while (g > 1 && g * items > lanes) g >>= 1;
  return g;
}

// sum_{i = i0, i0+g, ... < m} x[i] y[i]; four loads in flight per operand.
template <typename PX, typename PY>
__device__ inline double strided_dot(PX x, PY y, int i0, int m, int g) {
  double s0 = 0.0, s1 = 0.0;
  int i = i0;
  for (; i + 3 * g < m; i += 4 * g) {
    const double x0 = x[i], x1 = x[i + g], x2 = x[i + 2 * g], x3 = x[i + 3 * g];
    const double y0 = y[i], y1 = y[i + g], y2 = y[i + 2 * g], y3 = y[i + 3 * g];
    s0 += x0 * y0;
    s1 += x1 * y1;
    s0 += x2 * y2;
    s1 += x3 * y3;
  }
  for (; i < m; i += g) s0 += x[i] * y[i];
  return s0 + s1;
}

// y[i] -= f x[i] for i = i0, i0+g, ... < m (x and y distinct columns).
template <typename PY, typename PX>
__device__ inline void strided_axpy(PY y, double f, PX x, int i0, int m, int g) {
  int i = i0;
  for (; i + 3 * g < m; i += 4 * g) {
    const double x0 = x[i], x1 = x[i + g], x2 = x[i + 2 * g], x3 = x[i + 3 * g];
    const double y0 = y[i], y1 = y[i + g], y2 = y[i + 2 * g], y3 = y[i + 3 * g];
    y[i] = y0 - f * x0;
    y[i + g] = y1 - f * x1;
    y[i + 2 * g] = y2 - f * x2;
    y[i + 3 * g] = y3 - f * x3;
  }
  for (; i < m; i += g) y[i] -= f * x[i];
}

// Sum over the whole team; every thread gets the same value.  'red' holds
// kWaves doubles (workgroup team only).
template <int kLanes>
__device__ inline double team_sum(double v, lptr<double> red) {
  v = wave_sum(v);
  if constexpr (kLanes == kWave) {
    return v;
  } else {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) s += red[q];
    return s;
  }
}

// Householder QR, LAPACK dgeqrf conventions (dlarfg: beta = -sign(alpha)*norm,
// tau = (beta - alpha) / beta, v = x / (alpha - beta), v[0] = 1 implicit).
// On exit R is in the upper triangle, v_j below the diagonal, tau[j] set.
// The whole team forms each reflector (norm, scaling); trailing column c
// belongs to lane group c mod (kLanes / g), which applies the reflector to it.
template <int kLanes, typename PA, typename PT>
__device__ inline void team_house_qr(PA A, int lda, int m, int k, PT tau) {
  __shared__ double red[kWaves];
  const int tid = team_tid<kLanes>();
  const int steps = m < k ? m : k;
  const int g = group_lanes(k, kLanes), ngrp = kLanes / g, grp = tid / g, sub = tid % g;
  for (int j = 0; j < steps; ++j) {
    const PA v = A + (size_t)j * lda;
    double s = strided_dot(v, v, j + 1 + tid, m, kLanes);
    s = team_sum<kLanes>(s, (lptr<double>)red);
    const double alpha = v[j];
    double t = 0.0, beta = alpha;
    if (s != 0.0) {
      beta = -copysign(sqrt(alpha * alpha + s), alpha);
      t = (beta - alpha) / beta;
      const double scal = 1.0 / (alpha - beta);
      for (int i = j + 1 + tid; i < m; i += kLanes) v[i] *= scal;
    }
    team_sync<kLanes>();
    if (tid == 0) {
      tau[j] = t;
      v[j] = beta;
    }
    team_sync<kLanes>();
    if (t != 0.0) {
      int c = j + 1 + ((grp - (j + 1) % ngrp) + ngrp) % ngrp;
      for (; c < k; c += ngrp) {
        const PA a = A + (size_t)c * lda;
        double d = strided_dot(v, a, j + 1 + sub, m, g);
        d = group_sum(d, g) + a[j];
        const double f = t * d;
        strided_axpy(a, f, v, j + 1 + sub, m, g);
        if (sub == 0) a[j] -= f;
      }
    }
    team_sync<kLanes>();
  }
  if (tid == 0)
    for (int j = steps; j < k; ++j) tau[j] = 0.0;
  team_sync<kLanes>();
}

// Householder QR as team_house_qr with row ownership: thread t of the team
// keeps rows t + kLanes * r (r < kQrRows) of the current column in registers,
// and trailing columns are updated four at a time, their loads issued
// together and their four dot products reduced in one exchange.  A step thus
// costs a few memory round trips whether the panel lives in LDS or in global
// memory.  Requires m <= R * kLanes; 'red' holds 4 * kWaves doubles of
// shared scratch (workgroup team only).
constexpr int kQrRows = 8;

template <int kLanes, int kC>
__device__ inline void team_sum_n(double (&v)[kC], lptr<double> red) {
#pragma unroll
  for (int c = 0; c < kC; ++c) v[c] = wave_sum(v[c]);
  if constexpr (kLanes != kWave) {
    constexpr int kTeamWaves = kLanes / kWave;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int w0 = w - w % kTeamWaves;  // first wavefront of the team
    __syncthreads();
    if (lane == 0)
#pragma unroll
      for (int c = 0; c < kC; ++c) red[w * kC + c] = v[c];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kC; ++c) {
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < kTeamWaves; ++q) s += red[(w0 + q) * kC + c];
      v[c] = s;
    }
  }
}

// (one array for all instantiations in a kernel; wavefronts use their own part)
__device__ inline lptr<double> qr_red() {
  __shared__ double red[4 * kWaves];
  return (lptr<double>)red;
}

template <int kLanes, int R, typename PA, typename PT>
__device__ inline void team_house_qr_rows(PA A, int lda, int m, int k, PT tau) {
  const lptr<double> red = qr_red();
  const int tid = team_tid<kLanes>();
  const int steps = m < k ? m : k;
  // rows of this thread; loads use a clamped row and a select instead of a
  // branch, so all of them are in flight together
  int row[R], rc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    row[r] = tid + kLanes * r;
    rc[r] = row[r] < m ? row[r] : m - 1;
  }
  for (int j = 0; j < steps; ++j) {
    const PA vcol = A + (size_t)j * lda;
    double v[R];
    double s1[1] = {0.0};
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double x = vcol[rc[r]];
      v[r] = (row[r] > j && row[r] < m) ? x : 0.0;
      s1[0] += v[r] * v[r];
    }
    team_sum_n<kLanes, 1>(s1, red);
    const double s = s1[0];
    const double alpha = vcol[j];
    double t = 0.0, beta = alpha;
    if (s != 0.0) {
      beta = -copysign(sqrt(alpha * alpha + s), alpha);
      t = (beta - alpha) / beta;
      const double scal = 1.0 / (alpha - beta);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        v[r] *= scal;
        if (row[r] > j && row[r] < m) vcol[row[r]] = v[r];
      }
    }
    team_sync<kLanes>();
    if (tid == 0) {
      tau[j] = t;
      vcol[j] = beta;
    }
    {
      // also when t == 0 (a no-op then), so that every team passes the same barriers
      for (int c0 = j + 1; c0 < k; c0 += 4) {
        double a[4][R];
        double d[4], aj[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int cc = c0 + c < k ? c0 + c : k - 1;
          const PA ac = A + (size_t)cc * lda;
          aj[c] = ac[j];  // read by all before thread 0 rewrites it
#pragma unroll
          for (int r = 0; r < R; ++r) a[c][r] = ac[rc[r]];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          d[c] = 0.0;
#pragma unroll
          for (int r = 0; r < R; ++r) d[c] += v[r] * a[c][r];  // v is 0 outside rows (j, m)
        }
        team_sum_n<kLanes, 4>(d, red);
        team_sync<kLanes>();
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if (c0 + c >= k) continue;
          const PA ac = A + (size_t)(c0 + c) * lda;
          const double f = t * (d[c] + aj[c]);
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (row[r] > j && row[r] < m) ac[row[r]] = a[c][r] - f * v[r];
          if (tid == 0) ac[j] = aj[c] - f;
        }
      }
    }
    team_sync<kLanes>();
  }
  if (tid == 0)
    for (int j = steps; j < k; ++j) tau[j] = 0.0;
  team_sync<kLanes>();
}

// Picks the rows-per-thread count for m (m <= kQrRows * kLanes for a
// wavefront, 2 * kQrRows * kLanes for larger teams).
template <int kLanes, typename PA, typename PT>
__device__ inline void team_house_qr_any_rows(PA A, int lda, int m, int k, PT tau) {
  if (m <= 2 * kLanes)
    team_house_qr_rows<kLanes, 2>(A, lda, m, k, tau);
  else if (m <= 4 * kLanes)
    team_house_qr_rows<kLanes, 4>(A, lda, m, k, tau);
  else if (kLanes == kWave || m <= 8 * kLanes)
    team_house_qr_rows<kLanes, kQrRows>(A, lda, m, k, tau);
  else
    team_house_qr_rows<kLanes, 2 * kQrRows>(A, lda, m, k, tau);
}

// Householder QR of two global panels at once, one per half of the
// workgroup (rows <= 16 * 128 each, k columns each, k <= min(m, n)).  Both
// halves take the same k steps, so their workgroup barriers pair up.
template <typename PT>
__device__ inline void house_qr_pair(gptr<double> A, int lda, int m, PT tau_a, gptr<double> B, int ldb, int n,
                                     PT tau_b, int k) {
  if (threadIdx.x < kBlock / 2)
    team_house_qr_any_rows<kBlock / 2>(A, lda, m, k, tau_a);
  else
    team_house_qr_any_rows<kBlock / 2>(B, ldb, n, k, tau_b);
  __syncthreads();
}

// Y (m x r, ldy) <- Q Y with Q = H_0 ... H_{nref-1} from team_house_qr;
// column c of Y belongs to lane group c mod (kLanes / g).
template <int kLanes>
__device__ inline void team_apply_q(const double* V, int ldv, int m, int nref, const double* tau,
                                    double* Y, int ldy, int r) {
  const int tid = team_tid<kLanes>();
  const int g = group_lanes(r, kLanes), ngrp = kLanes / g, grp = tid / g, sub = tid % g;
  for (int c = grp; c < r; c += ngrp) {
    double* y = Y + (size_t)c * ldy;
    for (int j = nref - 1; j >= 0; --j) {
      const double t = tau[j];
      if (t == 0.0) continue;
      const double* v = V + (size_t)j * ldv;
      double d = strided_dot(v, y, j + 1 + sub, m, g);
      d = group_sum(d, g) + y[j];
      const double f = t * d;
      strided_axpy(y, f, v, j + 1 + sub, m, g);
      if (sub == 0) y[j] -= f;
      if (g > 1) __builtin_amdgcn_wave_barrier();
    }
  }
  team_sync<kLanes>();
}

// T of team_larft from the strict upper triangle of S = V^T V: T[j, j] = tau_j,
// T[l, j] = -tau_j sum_{r=l}^{j-1} T[l, r] S[r, j].  The recurrence runs on
// the team's first wavefront; row l of T is written by lane l mod 64 only.
template <int kLanes, typename PT>
__device__ inline void larft_recurrence(int k, PT tau, PT S, PT T) {
  const int tid = team_tid<kLanes>();
  if (tid < kWave) {
    for (int j = 0; j < k; ++j) {
      const double tj = tau[j];
      for (int l = tid; l < j; l += kWave) {
        double a = 0.0;
        for (int r = l; r < j; ++r) a += T[l + (size_t)r * k] * S[r + (size_t)j * k];
        T[l + (size_t)j * k] = -tj * a;
      }
      if (tid == (j & (kWave - 1))) T[j + (size_t)j * k] = tj;
    }
  }
  team_sync<kLanes>();
}

// Triangular factor T (k x k, ld k, upper) of the block reflector
// H_0 H_1 ... H_{k-1} = I - V T V^T of team_house_qr (LAPACK dlarft, forward,
// columnwise): S = V^T V (strict upper part, into S, k x k), then
// T[l, j] = -tau_j sum_{r=l}^{j-1} T[l, r] S[r, j], T[j, j] = tau_j.
// The recurrence runs on the team's first wavefront; row l of T is written
// by lane l mod 64 only, so its steps need no cross-lane exchange.
template <int kLanes, typename PV, typename PT>
__device__ inline void team_larft(PV V, int ldv, int m, int k, PT tau, PT S, PT T) {
  const int tid = team_tid<kLanes>();
  const int npairs = k * (k - 1) / 2;
  if (npairs > 0) {
    const int g = group_lanes(npairs, kLanes), ngrp = kLanes / g, grp = tid / g, sub = tid % g;
    for (int p = grp; p < npairs; p += ngrp) {
      int j = (int)((1.0 + sqrt(1.0 + 8.0 * p)) * 0.5);
      while (j * (j - 1) / 2 > p) --j;
      while ((j + 1) * j / 2 <= p) ++j;
      const int l = p - j * (j - 1) / 2;
      const PV vl = V + (size_t)l * ldv;
      const PV vj = V + (size_t)j * ldv;
      double d = strided_dot(vl, vj, j + 1 + sub, m, g);
      d = group_sum(d, g) + vl[j];
      if (sub == 0) S[l + (size_t)j * k] = d;
    }
  }
  team_sync<kLanes>();
  larft_recurrence<kLanes>(k, tau, S, T);
}

// Workgroup-wide wrappers.
template <typename PA, typename PT>
__device__ inline void house_qr(PA A, int lda, int m, int k, PT tau) {
  if (m <= 2 * kQrRows * kBlock)
    team_house_qr_any_rows<kBlock>(A, lda, m, k, tau);
  else
    team_house_qr<kBlock>(A, lda, m, k, tau);
}
__device__ inline void apply_q(const double* V, int ldv, int m, int nref, const double* tau,
                               double* Y, int ldy, int r, double* = nullptr, double* = nullptr) {
  team_apply_q<kBlock>(V, ldv, m, nref, tau, Y, ldy, r);
}
// Single-wavefront version.
template <typename PA, typename PT>
__device__ inline void wave_house_qr(PA A, int lda, int m, int k, PT tau) {
  if (m <= kQrRows * kWave)
    team_house_qr_any_rows<kWave>(A, lda, m, k, tau);
  else
    team_house_qr<kWave>(A, lda, m, k, tau);
}

constexpr int kJacobiMaxCols = 256;  // columns whose norms the Jacobi keeps in scratch

// One-sided (Hestenes) Jacobi SVD of G (rows x cols, ldg): on exit G = U Sigma
// (columns mutually orthogonal, unsorted) and V (cols x cols, ldv) holds the
// accumulated rotations so that G_in = (U Sigma) V^T.  Round-robin ordering:
// the cols/2 pairs of a round are independent and each belongs to one lane
// group.  Squared column norms are kept in 'nrm' (cols doubles of shared
// scratch), recomputed at the start of every sweep and updated exactly by
// each rotation (a' = a - t g, b' = b + t g), so a pair costs one reduction.
// A pair is rotated while g^2 > tol2 a b (tol2 1e-26 by default) and
// |g| > 1e-30 ||G||_F^2 (columns
// at rounding level of ||G|| carry nothing for the truncation thresholds used
// here).  Returns the number of sweeps.  'sh2' is 2 + kWaves shared doubles of
// scratch (workgroup team only); 'nrm' holds kJacobiMaxCols doubles.
// Rotation of one-sided Jacobi zeroing the inner product c2 of two columns
// with squared norms a and b: t = tan = sign(d) 2 c2 / (|d| + sqrt(d^2 + 4 c2^2))
// with d = b - a, c = 1 / sqrt(1 + t^2), s = c t.  d and 2 c2 are first
// scaled by a power of two (exact); the square roots and the quotient start
// from the hardware reciprocal and reciprocal square root and take Newton
// steps (two for c, so that c^2 + s^2 = 1 to a few ulp).
__device__ inline void jacobi_rot(double a, double b, double c2, double& t, double& c, double& s) {
  const double d = b - a, e = 2.0 * c2;
  const int ex = __builtin_amdgcn_frexp_exp(fmax(fabs(d), fabs(e)));
  const double ds = __builtin_amdgcn_ldexp(d, -ex), es = __builtin_amdgcn_ldexp(e, -ex);
  const double q = ds * ds + es * es;  // in [0.25, 2)
  double r = __builtin_amdgcn_rsq(q);
  r = r * (1.5 - 0.5 * q * r * r);
  const double den = fabs(ds) + q * r;  // |d| + sqrt(d^2 + e^2), scaled
  double inv = __builtin_amdgcn_rcp(den);
  inv = inv * (2.0 - den * inv);
  t = (d < 0.0 ? -es : es) * inv;
  const double w = 1.0 + t * t;  // in [1, 2]
  double y = __builtin_amdgcn_rsq(w);
  y = y * (1.5 - 0.5 * w * y * y);
  y = y * (1.5 - 0.5 * w * y * y);
  c = y;
  s = y * t;
}

// (kV and 'track' and not null pointers: the address of an LDS array can be 0,
// which is what a null LDS pointer is.  The norms' array sits there in FADD, and
// while it was tested against null the untracked loop ran: 98 x 98 sums of 64
// columns took 4.0 ms instead of 2.9)
template <int kLanes, bool kV, typename PG>
__device__ inline int team_jacobi(PG G, int ldg, int rows, int cols, PG V, int ldv,
                                  lptr<double> sh2, lptr<double> nrm, int max_sweeps, double tol2 = 1e-26) {
  const int tid = team_tid<kLanes>();
  if constexpr (kV)
    for (int e = tid; e < cols * cols; e += kLanes) {
      const int i = e % cols, j = e / cols;
      V[i + (size_t)j * ldv] = (i == j) ? 1.0 : 0.0;
    }
  if (cols < 2) {
    team_sync<kLanes>();
    return 0;
  }
  const int np = (cols + 1) & ~1, rounds = np - 1, half = np / 2;
  // long columns: at least 16 lanes per pair, so that a pair's loads are
  // coalesced and split 16 ways (fewer pairs side by side, each much faster
  // than a pair walked by one or two lanes)
  int g0 = group_lanes(half, kLanes);
  if (kLanes >= kWave && rows >= 128 && g0 < 16) g0 = 16;
  const int g = g0, ngrp = kLanes / g, grp = tid / g, sub = tid % g;
  // without scratch for every column the norms are recomputed pair by pair
  const bool track = cols <= kJacobiMaxCols;
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
    // column norms (and the Frobenius floor) afresh each sweep
    team_sync<kLanes>();
    double f = 0.0;
    if (track) {
      for (int c = grp; c < cols; c += ngrp) {
        double a = 0.0;
        for (int i = sub; i < rows; i += g) a += G[i + (size_t)c * ldg] * G[i + (size_t)c * ldg];
        a = group_sum(a, g);
        if (sub == 0) nrm[c] = a;
      }
      team_sync<kLanes>();
      for (int c = 0; c < cols; ++c) f += nrm[c];
    } else {
      for (int e = tid; e < rows * cols; e += kLanes) {
        const double x = G[e % rows + (size_t)(e / rows) * ldg];
        f += x * x;
      }
      f = team_sum<kLanes>(f, sh2 + 2);
    }
    const double floor2 = 1e-30 * f;
    int rotated = 0;
    for (int rd = 0; rd < rounds; ++rd) {
      for (int pk = grp; pk < half; pk += ngrp) {
        int p, q;
        if (pk == 0) {
          p = np - 1;
          q = rd;
        } else {
          p = rd + pk;
          if (p >= np - 1) p -= np - 1;
          q = rd - pk + (np - 1);
          if (q >= np - 1) q -= np - 1;
        }
        if (p > q) {
          const int tmp = p;
          p = q;
          q = tmp;
        }
        if (q >= cols) continue;
        const PG gp = G + (size_t)p * ldg;
        const PG gq = G + (size_t)q * ldg;
        double c2 = 0.0, a, b;
        if (track) {
          c2 = group_sum(strided_dot(gp, gq, sub, rows, g), g);
          a = nrm[p];
          b = nrm[q];
        } else {
          a = 0.0;
          b = 0.0;
          for (int i = sub; i < rows; i += g) {
            a += gp[i] * gp[i];
            b += gq[i] * gq[i];
            c2 += gp[i] * gq[i];
          }
          a = group_sum(a, g);
          b = group_sum(b, g);
          c2 = group_sum(c2, g);
        }
        if (!(c2 * c2 > tol2 * a * b) || !(fabs(c2) > floor2)) continue;
        // t = tan(theta) of the rotation zeroing the pair's inner product
        double t, c, s;
        jacobi_rot(a, b, c2, t, c, s);
        for (int i = sub; i < rows; i += g) {
          const double x = gp[i], y = gq[i];
          gp[i] = c * x - s * y;
          gq[i] = s * x + c * y;
        }
        if constexpr (kV) {
          const PG vp = V + (size_t)p * ldv;
          const PG vq = V + (size_t)q * ldv;
          for (int i = sub; i < cols; i += g) {
            const double x = vp[i], y = vq[i];
            vp[i] = c * x - s * y;
            vq[i] = s * x + c * y;
          }
        }
        if (track && sub == 0) {
          nrm[p] = a - t * c2;
          nrm[q] = b + t * c2;
        }
        rotated = 1;
      }
      team_sync<kLanes>();
    }
    int any;
    if constexpr (kLanes == kWave) {
      any = __ballot(rotated) != 0;
    } else {
      if (threadIdx.x == 0) sh2[1] = 0.0;
      __syncthreads();
      if (rotated) sh2[1] = 1.0;
      __syncthreads();
      any = sh2[1] != 0.0;
      __syncthreads();
    }
    if (!any) {
      ++sweep;
      break;
    }
  }
  team_sync<kLanes>();
  return sweep;
}

// Sum over aligned groups of kG lanes (compile-time kG <= 16, see group_sum).
template <int kG>
__device__ inline double group_sum_c(double v) {
  if constexpr (kG >= 2) v += dpp_swap<0xB1>(v);
  if constexpr (kG >= 4) v += dpp_swap<0x4E>(v);
  if constexpr (kG >= 8) v += dpp_swap<0x141>(v);
  if constexpr (kG >= 16) v += dpp_swap<0x140>(v);
  return v;
}

// team_jacobi with the pair's rows held in registers and a compile-time
// group of kG lanes per pair: lane 'sub' of a group owns rows sub + kG r
// (r < R) of G (and of V when kV); the loads use clamped rows and a select,
// the columns are read once per round and written back after the rotation.
// Requires rows (and cols when kV) <= R kG, kG == group_lanes(pairs, kLanes)
// and tracked norms.  Without V (kV false) the caller recovers the right
// singular vectors from the input, as G_in^T U.
template <int kLanes, int R, int kG, bool kV, typename PG>
__device__ inline int team_jacobi_rows(PG G, int ldg, int rows, int cols, PG V, int ldv,
                                       lptr<double> sh2, lptr<double> nrm, int max_sweeps, double tol2 = 1e-26) {
  const int tid = team_tid<kLanes>();
  if constexpr (kV) {
    for (int e = tid; e < cols * cols; e += kLanes) {
      const int i = e % cols, j = e / cols;
      V[i + (size_t)j * ldv] = (i == j) ? 1.0 : 0.0;
    }
  }
  if (cols < 2) {
    team_sync<kLanes>();
    return 0;
  }
  const int np = (cols + 1) & ~1, rounds = np - 1, half = np / 2;
  constexpr int ngrp = kLanes / kG;
  const int grp = tid / kG, sub = tid % kG;
  int rg[R], rgc[R], rvc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    rg[r] = sub + kG * r;
    rgc[r] = rg[r] < rows ? rg[r] : rows - 1;
    rvc[r] = rg[r] < cols ? rg[r] : cols - 1;
  }
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
    team_sync<kLanes>();
    for (int c = grp; c < cols; c += ngrp) {
      double a = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double x = G[rgc[r] + (size_t)c * ldg];
        a += rg[r] < rows ? x * x : 0.0;
      }
      a = group_sum_c<kG>(a);
      if (sub == 0) nrm[c] = a;
    }
    team_sync<kLanes>();
    double f = 0.0;
    for (int c = 0; c < cols; ++c) f += nrm[c];
    const double floor2 = 1e-30 * f;
    int rotated = 0;
    for (int rd = 0; rd < rounds; ++rd) {
      for (int pk = grp; pk < half; pk += ngrp) {
        int p, q;
        if (pk == 0) {
          p = np - 1;
          q = rd;
        } else {
          p = rd + pk;
          if (p >= np - 1) p -= np - 1;
          q = rd - pk + (np - 1);
          if (q >= np - 1) q -= np - 1;
        }
        if (p > q) {
          const int tmp = p;
          p = q;
          q = tmp;
        }
        if (q >= cols) continue;
        const PG gp = G + (size_t)p * ldg;
        const PG gq = G + (size_t)q * ldg;
        // all loads of the pair issued before the first wait
        double xp[R], xq[R], up[R], uq[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          xp[r] = gp[rgc[r]];
          xq[r] = gq[rgc[r]];
        }
        if constexpr (kV) {
          const PG vp = V + (size_t)p * ldv;
          const PG vq = V + (size_t)q * ldv;
#pragma unroll
          for (int r = 0; r < R; ++r) {
            up[r] = vp[rvc[r]];
            uq[r] = vq[rvc[r]];
          }
        }
        const double a = nrm[p], b = nrm[q];
        double c2 = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) c2 += rg[r] < rows ? xp[r] * xq[r] : 0.0;
        c2 = group_sum_c<kG>(c2);
        if (!(c2 * c2 > tol2 * a * b) || !(fabs(c2) > floor2)) continue;
        double t, c, s;
        jacobi_rot(a, b, c2, t, c, s);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (rg[r] < rows) {
            gp[rg[r]] = c * xp[r] - s * xq[r];
            gq[rg[r]] = s * xp[r] + c * xq[r];
          }
        }
        if constexpr (kV) {
          const PG vp = V + (size_t)p * ldv;
          const PG vq = V + (size_t)q * ldv;
#pragma unroll
          for (int r = 0; r < R; ++r) {
            if (rg[r] < cols) {
              vp[rg[r]] = c * up[r] - s * uq[r];
              vq[rg[r]] = s * up[r] + c * uq[r];
            }
          }
        }
        if (sub == 0) {
          nrm[p] = a - t * c2;
          nrm[q] = b + t * c2;
        }
        rotated = 1;
      }
      team_sync<kLanes>();
    }
    int any;
    if constexpr (kLanes == kWave) {
      any = __ballot(rotated) != 0;
    } else {
      if (threadIdx.x == 0) sh2[1] = 0.0;
      __syncthreads();
      if (rotated) sh2[1] = 1.0;
      __syncthreads();
      any = sh2[1] != 0.0;
      __syncthreads();
    }
    if (!any) {
      ++sweep;
      break;
    }
  }
  team_sync<kLanes>();
  return sweep;
}

// Dispatch on the group size and rows per lane; without kV the accumulation of
// V is left out.  Shapes outside the instantiated ones use team_jacobi.
template <int kLanes, bool kV, typename PG>
__device__ inline int team_jacobi_any(PG G, int ldg, int rows, int cols, PG V, int ldv,
                                      lptr<double> sh2, lptr<double> nrm, int max_sweeps, double tol2 = 1e-26) {
  if (cols <= kJacobiMaxCols && cols >= 2 && rows >= 1) {
    const int half = ((cols + 1) & ~1) / 2;
    const int g = group_lanes(half, kLanes);
    const int span = kV ? (rows > cols ? rows : cols) : rows;
    const int need = (span + g - 1) / g;
#define HMX_JR(G_, R_)                                                                             \
  if (g == G_ && need <= R_)                                                                       \
    return team_jacobi_rows<kLanes, R_, G_, kV>(G, ldg, rows, cols, V, ldv, sh2, nrm, max_sweeps, tol2);
    HMX_JR(16, 2)
    HMX_JR(8, 8)
#undef HMX_JR
  }
  return team_jacobi<kLanes, kV>(G, ldg, rows, cols, V, ldv, sh2, nrm, max_sweeps, tol2);
}

// The norms of the workgroup's Jacobi: one array for every instantiation.
__device__ inline lptr<double> jacobi_norms() {
  __shared__ double nrm[kJacobiMaxCols];
  return (lptr<double>)nrm;
}

// Workgroup version (cols <= kJacobiMaxCols); without kV, V is not touched.
template <bool kV, typename PG>
__device__ inline void jacobi_svd(PG G, int ldg, int rows, int cols, PG V, int ldv,
                                  int* /*flag*/, int max_sweeps = 40, double tol2 = 1e-26) {
  __shared__ double sh2[2 + kWaves];
  team_jacobi_any<kBlock, kV>(G, ldg, rows, cols, V, ldv, (lptr<double>)sh2, jacobi_norms(), max_sweeps, tol2);
}

// ---------------------------------------------------------------------------
// Core SVD of the recompressions: G (rows x cols, both at most kCoreMax) on one
// wavefront.  A one-sided Jacobi on the core itself took 7 to 14 sweeps of
// rounds whose index arithmetic, masks and branches cost 2,000 cycles each (88 us
// for 13 columns, the larger part of a recompression: an average launch of FADD
// went from 166 to 147 us in a 40,000-point FP32 Cholesky and from 137 to 110 us
// in a 6,000-point FP64 LU, RKRK from 53 to 41 and from 41 to 34 us).  Here:
//  1. Pivoted Gram-Schmidt of the rows of G in registers (lane c holds row c):
//     G = W Q^T, the columns of W graded, their number the numerical rank (cut at
//     1e-15 of the norm, the level below which the Jacobi rotates nothing).
//  2. Jacobi on the columns of W, which being graded needs about half the
//     sweeps, in a tournament whose columns move between fixed slots: every lane
//     reads and writes the same LDS addresses in every round, rows are padded
//     with zeros, a pair below the threshold gets the identity rotation, and the
//     norms come from the registers.
// On exit the first r columns of G hold sigma_j u_j; returns r.
// Bound: the instructions of one wavefront (about 100 per round).
// ---------------------------------------------------------------------------
constexpr int kCoreMax = 32;

// doubles of W for a core of rows x cols: odd leading dimensions spread the
// columns' rows over the banks; an even number of columns
__host__ __device__ constexpr int core_ld(int rows) { return rows <= 16 ? 17 : 33; }
__host__ __device__ constexpr int core_work(int rows, int cols) {
  const int c = rows < cols ? rows : cols;
  return core_ld(rows) * (c + (c & 1));
}

// kG lanes per pair, kR rows per lane (rows <= kG kR), cols <= 128 / kG; W has
// cols rounded up to even columns, ld rows >= kG kR, zero outside the matrix.
template <int kG, int kR>
__device__ inline void slot_jacobi(lptr<double> W, int ld, int cols, double tol2) {
  const int lane = threadIdx.x & (kWave - 1);
  const int h = (cols + 1) / 2, rounds = 2 * h - 1;
  const int i = lane / kG, sub = lane % kG;
  const bool act = i < h;
  const int ic = act ? i : 0;
  // slots: top column i of pair i, bottom column h + i.  The top of pair 0 stays,
  // the others move up through the tops and back through the bottoms.
  const int top_to = ic == 0 ? 0 : (ic < h - 1 ? ic + 1 : 2 * h - 1);
  const int bot_to = ic == 0 ? (h > 1 ? 1 : h) : h + ic - 1;
  const lptr<double> xt = W + ic * ld + sub, xb = W + (h + ic) * ld + sub;
  const lptr<double> yt = W + top_to * ld + sub, yb = W + bot_to * ld + sub;
  double floor2 = 0.0;
  for (int sweep = 0; sweep < 40; ++sweep) {
    bool rotated = false;
    for (int rd = 0; rd < rounds; ++rd) {
      double x[kR], y[kR];
#pragma unroll
      for (int r = 0; r < kR; ++r) {
        x[r] = xt[kG * r];
        y[r] = xb[kG * r];
      }
      double a = 0.0, b = 0.0, c2 = 0.0;
#pragma unroll
      for (int r = 0; r < kR; ++r) {
        a += x[r] * x[r];
        b += y[r] * y[r];
        c2 += x[r] * y[r];
      }
      a = group_sum_c<kG>(a);
      b = group_sum_c<kG>(b);
      c2 = group_sum_c<kG>(c2);
      if (sweep == 0 && rd == 0) floor2 = 1e-30 * wave_sum(act && sub == 0 ? a + b : 0.0);
      const bool turn = c2 * c2 > tol2 * a * b && fabs(c2) > floor2;
      double t, c, s;
      jacobi_rot(a, b, c2, t, c, s);
      c = turn ? c : 1.0;
      s = turn ? s : 0.0;
      rotated |= turn && act;
      __builtin_amdgcn_wave_barrier();
      if (act) {
#pragma unroll
        for (int r = 0; r < kR; ++r) {
          yt[kG * r] = c * x[r] - s * y[r];
          yb[kG * r] = s * x[r] + c * y[r];
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (__ballot(rotated) == 0) break;
  }
}

template <int kN>
__device__ inline int core_rows(lptr<double> G, int ldg, int rows, int cols, lptr<double> W, int ld) {
  const int lane = threadIdx.x & (kWave - 1);
  const int lc = lane < rows ? lane : rows - 1;
  double g[kN];
  double n2 = 0.0;
#pragma unroll
  for (int r = 0; r < kN; ++r) {
    const double v = G[lc + (r < cols ? r : cols - 1) * ldg];
    g[r] = (lane < rows && r < cols) ? v : 0.0;
    n2 += g[r] * g[r];
  }
  const double total = wave_sum(n2);
  if (!(total < __builtin_inf())) {  // infinities and NaN go on as NaN
    if (lane < ld) W[lane] = __builtin_nan("");
    return 1;
  }
  const double stop = 1e-30 * total;
  const int most = rows < cols ? rows : cols;
  int s = 0;
  for (; s < most; ++s) {
    const double m = wave_max(n2);
    if (!(m > stop)) break;
    const int p = __builtin_ctzll(__ballot(n2 == m));
    const double inv = 1.0 / sqrt(m);
    double q[kN], d = 0.0;
#pragma unroll
    for (int r = 0; r < kN; ++r) {
      q[r] = lane_read(g[r], p) * inv;
      d += q[r] * g[r];
    }
    if (lane < ld) W[lane + s * ld] = d;
    n2 = 0.0;
#pragma unroll
    for (int r = 0; r < kN; ++r) {
      g[r] = lane == p ? 0.0 : g[r] - d * q[r];  // what is left of the pivot is rounding
      n2 += g[r] * g[r];
    }
  }
  if ((s & 1) && lane < ld) W[lane + s * ld] = 0.0;
  return s;
}

// (one wavefront; rows, cols <= kCoreMax; W: core_work(rows, cols) doubles)
__device__ inline int wave_core_svd(lptr<double> G, int ldg, int rows, int cols, lptr<double> W, double tol2) {
  const int lane = threadIdx.x & (kWave - 1), ld = core_ld(rows);
  int r;
  if (rows <= 16) {
    r = cols <= 16 ? core_rows<16>(G, ldg, rows, cols, W, ld) : core_rows<32>(G, ldg, rows, cols, W, ld);
    __builtin_amdgcn_wave_barrier();
    if (r > 1) slot_jacobi<8, 2>(W, ld, r, tol2);
  } else {
    r = cols <= 24 ? core_rows<24>(G, ldg, rows, cols, W, ld) : core_rows<32>(G, ldg, rows, cols, W, ld);
    __builtin_amdgcn_wave_barrier();
    if (r > 1) slot_jacobi<4, 8>(W, ld, r, tol2);
  }
  __builtin_amdgcn_wave_barrier();
  for (int e = lane; e < rows * r; e += kWave) G[e % rows + e / rows * ldg] = W[e % rows + e / rows * ld];
  __builtin_amdgcn_wave_barrier();
  return r;
}

// Column norms of G into sig[0..cols), then order[] = permutation sorting
// sig descending (ties by index).  Returns nothing; ends with a barrier.
template <typename PG, typename PS, typename PI>
__device__ inline void sorted_norms(PG G, int ldg, int rows, int cols, PS sig, PI order) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  for (int j = w; j < cols; j += kWaves) {
    const PG g = G + (size_t)j * ldg;
    double s = 0.0;
    for (int i = lane; i < rows; i += kWave) s += g[i] * g[i];
    s = wave_sum(s);
    // a non-finite norm (NaN input) is ordered as zero so that 'order' is
    // always a permutation of [0, cols)
    if (lane == 0) sig[j] = (s >= 0.0 && s <= 1.79e308) ? sqrt(s) : 0.0;
  }
  __syncthreads();
  for (int j = threadIdx.x; j < cols; j += kBlock) {
    const double sj = sig[j];
    int pos = 0;
    for (int i = 0; i < cols; ++i) {
      const double si = sig[i];
      pos += (si > sj) || (si == sj && i < j);
    }
    order[pos] = j;
  }
  __syncthreads();
}

// findK scalar_array.cpp:98-116: number of sigma (descending) with
// sigma[i] > eps * sigma[0].
template <typename PS, typename PI>
__device__ inline int find_k(PS sig, PI order, int n, double eps) {
  if (n == 0) return 0;
  const double thr = sig[order[0]] * eps;
  int k = 0;
  while (k < n && !(sig[order[k]] <= thr)) ++k;
  return k;
}

// sorted_norms and find_k of at most kCoreMax columns by one wavefront: a lane
// per column, the order by counting.  Returns find_k's number.
__device__ inline int wave_sorted_cut(lptr<double> G, int ldg, int rows, int cols, lptr<double> sig,
                                      lptr<int> order, double eps) {
  const int lane = threadIdx.x & (kWave - 1);
  const lptr<double> g = G + (lane < cols ? lane : 0) * ldg;
  double s = 0.0;
  for (int i = 0; i < rows; ++i) s += g[i] * g[i];
  s = (s >= 0.0 && s <= 1.79e308) ? sqrt(s) : 0.0;
  int pos = 0;
  double top = 0.0;
  for (int i = 0; i < cols; ++i) {
    const double si = lane_read(s, i);
    pos += (si > s) || (si == s && i < lane);
    top = fmax(top, si);
  }
  if (lane < cols) {
    sig[lane] = s;
    order[pos] = lane;
  }
  __builtin_amdgcn_wave_barrier();
  return __popcll(__ballot(lane < cols && !(s <= top * eps)));
}

}  // namespace hmx
