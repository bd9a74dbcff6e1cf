// k_precond.hip — near-field sparse approximate inverse (SPAI) preconditioner.
//
// The reference preconditions GMRES with the LU factors of the near-field
// matrix Z_nf (entries whose RWG centres are within a cutoff,
// src/solver/NearFieldPreconditioner.jl:670-717).  A sparse LU is a serial,
// fill-in driven factorisation; the GPU form here instead minimises
// || Z M - I ||_F column by column over the same kind of geometric near-field
// pattern (Frobenius-norm minimisation, as used for EFIE by Alleon, Benzi and
// Giraud 1997 / Carpentieri et al. 2000):
//   m_j = argmin || Z[I_j, J_j] m - e_j ||_2,
// J_j = bases within cutJ of basis j (the columns' support), I_j = bases within
// cutI >= cutJ (the rows that carry the significant part of Z[:, J_j]).
// Each column is an independent small least-squares problem solved through the
// normal equations (G = A^H A, Cholesky in LDS, FP64) by one workgroup; the
// result is applied as a CSR SpMV, y_n = sum_{j in J(n)} M[n, j] x_j.
#include <hip/hip_runtime.h>

#include "dm_common.h"
#include "k_linalg.h"

namespace {

constexpr int SPAI_MAXJ = 80;  // columns per least-squares problem
constexpr int SPAI_CHUNK = 8;  // rows of A staged per pass

// One column per workgroup of NT threads; thread t owns one 4 x 4 block (A, B)
// of the lower triangle of the Gram matrix, held in registers from the first row
// of A to the solution:
//   Gram: chunks of SPAI_CHUNK rows staged in LDS (two buffers; the next chunk's
//     entries are on their way while this one's products are formed); per row a
//     thread reads 8 values for 16 complex products.
//   Cholesky, right-looking by block columns: the diagonal block's thread
//     factors it, the blocks below solve against it and put their result in LDS
//     while it solves its entries of L y = rhs, the blocks to the right subtract
//     their products while those below take theirs out of the right-hand side.
//   Backward: per block column the diagonal's thread solves its four entries and
//     the blocks to its left in that row take them out of y.
// Every entry is rounded in the order of the plain column-by-column form, so the
// workgroup's size and the blocks change no bit of the result.
// The largest NT is bound by FP64 arithmetic in the Gram part, the small ones by
// the serial steps, of which several workgroups per CU overlap.
// 4720 columns, supports of 80 and about 200 rows: 1.56 ms (Gram matrix in LDS,
// factorization and solves by one wave: 3.2); 30720 of 49: 2.6 ms (2.8).
// Blocks are numbered down block columns, so that the waves of finished columns
// drop out of the later steps.
template <int NT>
struct SpaiShape;  // NB: block rows (NB (NB + 1) / 2 <= NT)
template <>
struct SpaiShape<64> {
  static constexpr int NB = 10;
};
template <>
struct SpaiShape<128> {
  static constexpr int NB = 15;
};
template <>
struct SpaiShape<256> {
  static constexpr int NB = 20;
};

// b -= l y, and b -= conj(l) m (a product rounded once, then taken away)
__device__ inline void csub_fwd(double2& b, double2 l, double2 y) {
  b.x -= fma(l.x, y.x, -(l.y * y.y));
  b.y -= fma(l.x, y.y, l.y * y.x);
}
__device__ inline void csub_bwd(double2& b, double2 l, double2 m) {
  b.x -= fma(l.x, m.x, l.y * m.y);
  b.y -= fma(l.x, m.y, -(l.y * m.x));
}
// a -= p conj(q)
__device__ inline void csub_pq(double2& a, double2 p, double2 q) {
  a.x = fma(-p.x, q.x, a.x);
  a.x = fma(-p.y, q.y, a.x);
  a.y = fma(-p.y, q.x, a.y);
  a.y = fma(p.x, q.y, a.y);
}
// a += conj(p) q
__device__ inline void cacc_pq(double2& a, double2 p, double2 q) {
  a.x = fma(p.x, q.x, a.x);
  a.x = fma(p.y, q.y, a.x);
  a.y = fma(p.x, q.y, a.y);
  a.y = fma(-p.y, q.x, a.y);
}

template <int NT>
__global__ __launch_bounds__(NT, 2) void k_spai_build(int n, int per, ZRef z, const int* __restrict__ jptr,
                                                      const int* __restrict__ jidx, const int* __restrict__ iptr,
                                                      const int* __restrict__ iidx, double2* __restrict__ vals,
                                                      int* __restrict__ status) {
  constexpr int NB = SpaiShape<NT>::NB;
  constexpr int kPre = (4 * NB * SPAI_CHUNK + NT - 1) / NT;  // staged entries per thread
  static_assert(NB * (NB + 1) / 2 <= NT && NT % SPAI_CHUNK == 0, "one block per thread");
  // XCD-aware order: workgroup w runs on XCD w % 8, which takes the columns
  // [x per, (x + 1) per) in order, so the columns in flight on one XCD are
  // neighbours whose rows of Z overlap and are read through the same L2.
  const int j = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (j >= n) return;
  const int j0 = jptr[j], nJ = jptr[j + 1] - j0;
  const int i0 = iptr[j], nI = iptr[j + 1] - i0;
  // staged rows, column c of row r at [r][c % 4][c / 4] (a wave's block rows are
  // consecutive); the factorization's panel at [v][u][A] in the same place
  __shared__ double2 st[2][SPAI_CHUNK][4][NB];
  __shared__ double2 dl[4][4];
  __shared__ double dil[4];
  __shared__ double2 ys[4 * NB];
  double2(*panel)[4][NB] = st[0];
  const int tid = threadIdx.x;
  const int nb = (nJ + 3) / 4;  // block rows
  int A = -1, B = -1;
  if (tid < nb * (nb + 1) / 2) {
    int e = tid;
    for (B = 0; e >= nb - B; ++B) e -= nb - B;
    A = B + e;
  }
  // staging: this thread's row of every chunk, its columns
  const int sr = tid % SPAI_CHUNK;
  int sc[kPre], col[kPre];
#pragma unroll
  for (int q = 0; q < kPre; ++q) {
    sc[q] = tid / SPAI_CHUNK + q * (NT / SPAI_CHUNK);
    col[q] = jidx[j0 + min(sc[q], nJ - 1)];
  }
  double2 pre[kPre];
  auto row_of = [&](int r0) { return iidx[i0 + min(r0 + sr, nI - 1)]; };
  auto fetch = [&](int r0, int row) {
#pragma unroll
    for (int q = 0; q < kPre; ++q) {
      pre[q] = zat(z, row, col[q]);
      if (r0 + sr >= nI || sc[q] >= nJ) pre[q] = make_double2(0.0, 0.0);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int q = 0; q < kPre; ++q)
      if (sc[q] < 4 * nb) st[buf][sr][sc[q] & 3][sc[q] >> 2] = pre[q];
  };
  double2 acc[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[u][v] = make_double2(0.0, 0.0);
  fetch(0, row_of(0));
  int row = row_of(SPAI_CHUNK);
  stage(0);
  __syncthreads();
  for (int r0 = 0, buf = 0; r0 < nI; r0 += SPAI_CHUNK, buf ^= 1) {
    const bool more = r0 + SPAI_CHUNK < nI;
    if (more) {
      fetch(r0 + SPAI_CHUNK, row);
      row = row_of(r0 + 2 * SPAI_CHUNK);
    }
    if (A >= 0) {
      // a chunk's sums are formed apart and added
      double2 sum[4][4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) sum[u][v] = make_double2(0.0, 0.0);
#pragma unroll 2
      for (int r = 0; r < SPAI_CHUNK; ++r) {
        double2 p[4], q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          p[u] = st[buf][r][u][A];
          q[u] = st[buf][r][u][B];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) cacc_pq(sum[u][v], p[u], q[v]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          acc[u][v].x += sum[u][v].x;
          acc[u][v].y += sum[u][v].y;
        }
    }
    if (more) stage(buf ^ 1);
    __syncthreads();
  }
  // the identity past the last column, and the right-hand side A^H e_j =
  // conj(Z[j, J]) (row j of Z restricted to the pattern)
  if (A == nb - 1 && B == A) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (4 * A + u >= nJ) acc[u][u] = make_double2(1.0, 0.0);
  }
  for (int b = tid; b < 4 * nb; b += NT) {
    double2 v = zat(z, j, jidx[j0 + min(b, nJ - 1)]);
    ys[b] = b < nJ ? make_double2(v.x, -v.y) : make_double2(0.0, 0.0);
  }
  bool bad = false;
  for (int K = 0; K < nb; ++K) {
    if (A == K && B == K) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        double d = acc[v][v].x;
#pragma unroll
        for (int w = 0; w < v; ++w) d = fma(-acc[v][w].y, acc[v][w].y, fma(-acc[v][w].x, acc[v][w].x, d));
        if (!(d > 0.0)) {
          bad = true;
          d = 1e-300;
        }
        const double il = 1.0 / sqrt(d);
        dil[v] = il;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (u <= v) continue;
          double2 x = acc[u][v];
#pragma unroll
          for (int w = 0; w < v; ++w) csub_pq(x, acc[u][w], acc[v][w]);
          acc[u][v] = make_double2(x.x * il, x.y * il);
          dl[u][v] = acc[u][v];
        }
        acc[v][v] = make_double2(il, 0.0);  // 1 / L[v][v]
      }
    }
    __syncthreads();
    if (B == K && A > K) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const double il = dil[v];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          double2 x = acc[u][v];
#pragma unroll
          for (int w = 0; w < v; ++w) csub_pq(x, acc[u][w], dl[v][w]);
          acc[u][v] = make_double2(x.x * il, x.y * il);
          panel[v][u][A] = acc[u][v];
        }
      }
    }
    if (A == K && B == K) {
      // its four entries of y, while the others solve
      double2 y[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) y[v] = ys[4 * K + v];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        y[v] = make_double2(y[v].x * acc[v][v].x, y[v].y * acc[v][v].x);
#pragma unroll
        for (int u = v + 1; u < 4; ++u) csub_fwd(y[u], acc[u][v], y[v]);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) ys[4 * K + v] = y[v];
    }
    __syncthreads();
    if (B == K && A > K) {
      // the block's share out of the right-hand side, beside the updates
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        double2 b = ys[4 * A + u];
#pragma unroll
        for (int v = 0; v < 4; ++v) csub_fwd(b, acc[u][v], ys[4 * K + v]);
        ys[4 * A + u] = b;
      }
    }
    if (B > K) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        double2 p[4], q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          p[u] = panel[v][u][A];
          q[u] = panel[v][u][B];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int w = 0; w < 4; ++w) csub_pq(acc[u][w], p[u], q[w]);
      }
    }
  }
  for (int K = nb - 1; K >= 0; --K) {
    __syncthreads();
    if (A == K && B == K) {
      // L(K, K)^H m = y
      double2 m[4];
#pragma unroll
      for (int v = 3; v >= 0; --v) {
        double2 x = ys[4 * K + v];
#pragma unroll
        for (int u = 3; u > v; --u) csub_bwd(x, acc[u][v], m[u]);
        const double il = acc[v][v].x;
        m[v] = make_double2(x.x * il, x.y * il);
        ys[4 * K + v] = m[v];
      }
    }
    __syncthreads();
    if (A == K && B < K) {
      double2 m[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) m[u] = ys[4 * K + u];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        double2 x = ys[4 * B + v];
#pragma unroll
        for (int u = 3; u >= 0; --u) csub_bwd(x, acc[u][v], m[u]);
        ys[4 * B + v] = x;
      }
    }
  }
  __syncthreads();
  for (int a = tid; a < nJ; a += NT) vals[j0 + a] = ys[a];
  if (bad) status[0] = j + 1;
}

// y = M x with M in CSR form (row n: columns colidx[rowptr[n]..], values csrval).
// Eight lanes per row: lane j of a row's group takes nonzeros j, j + 8, ...
// (coalesced 128-byte reads of the row's values), then a 3-step xor reduction
// inside the group.  blockIdx.y selects one of several right-hand sides.
constexpr int kSpmvLanes = 8;

__global__ __launch_bounds__(256) void k_spmv(i64 n, const int* __restrict__ rowptr, const int* __restrict__ colidx,
                                              const double2* __restrict__ val, const double2* __restrict__ x,
                                              double2* __restrict__ y) {
  x += (i64)blockIdx.y * n;
  y += (i64)blockIdx.y * n;
  const i64 r = (blockIdx.x * (i64)blockDim.x + threadIdx.x) / kSpmvLanes;
  const int j = threadIdx.x % kSpmvLanes;
  double ar = 0, ai = 0;
  if (r < n) {
    const int p1 = rowptr[r + 1];
#pragma unroll 4
    for (int p = rowptr[r] + j; p < p1; p += kSpmvLanes) {
      double2 a = val[p], v = x[colidx[p]];
      ar += a.x * v.x - a.y * v.y;
      ai += a.x * v.y + a.y * v.x;
    }
  }
#pragma unroll
  for (int o = kSpmvLanes / 2; o > 0; o >>= 1) {
    ar += __shfl_xor(ar, o, kSpmvLanes);
    ai += __shfl_xor(ai, o, kSpmvLanes);
  }
  if (r < n && j == 0) y[r] = make_double2(ar, ai);
}

// Y[:, c] = M X[:, c] for kSpmmCols columns per workgroup row (blockIdx.y
// selects the column group): the row's values and column indices are read once
// per group instead of once per column.  Lanes take nonzeros as in k_spmv; the
// 8-lane reduction is a reduce-scatter (offsets 4, 2, 1, each lane keeping half
// of its remaining columns), which adds the same partial sums in the same
// order as k_spmv's butterfly and leaves lane j with columns 2j and 2j + 1.
// Bound by the gathers' cache lines; all 16 are issued together (a column past
// R reads the last one), 30720 rows, 128 columns: 255 us (388 when each column's
// load sat behind its range test).
constexpr int kSpmmCols = 2 * kSpmvLanes;

__global__ __launch_bounds__(256) void k_spmm(i64 n, int R, const int* __restrict__ rowptr,
                                              const int* __restrict__ colidx, const double2* __restrict__ val,
                                              const double2* __restrict__ X, double2* __restrict__ Y) {
  const int c0 = blockIdx.y * kSpmmCols;
  const int nc = min(kSpmmCols, R - c0);
  const i64 r = (blockIdx.x * (i64)blockDim.x + threadIdx.x) / kSpmvLanes;
  const int j = threadIdx.x % kSpmvLanes;
  const double2* xb = X + (i64)c0 * n;
  double ar[kSpmmCols], ai[kSpmmCols];
#pragma unroll
  for (int c = 0; c < kSpmmCols; ++c) ar[c] = ai[c] = 0.0;
  if (r < n) {
    const int p1 = rowptr[r + 1];
    for (int p = rowptr[r] + j; p < p1; p += kSpmvLanes) {
      const double2 a = val[p];
      const double2* xc = xb + colidx[p];
      double2 v[kSpmmCols];
#pragma unroll
      for (int c = 0; c < kSpmmCols; ++c) v[c] = xc[(i64)min(c, nc - 1) * n];
#pragma unroll
      for (int c = 0; c < kSpmmCols; ++c) {
        ar[c] += a.x * v[c].x - a.y * v[c].y;
        ai[c] += a.x * v[c].y + a.y * v[c].x;
      }
    }
  }
#pragma unroll
  for (int o = kSpmvLanes / 2, m = kSpmmCols; o > 0; o >>= 1, m >>= 1) {
    const bool hi = (j & o) != 0;
#pragma unroll
    for (int i = 0; i < m / 2; ++i) {
      const double sr = hi ? ar[i] : ar[i + m / 2], si = hi ? ai[i] : ai[i + m / 2];
      const double kr = hi ? ar[i + m / 2] : ar[i], ki = hi ? ai[i + m / 2] : ai[i];
      ar[i] = kr + __shfl_xor(sr, o, kSpmvLanes);
      ai[i] = ki + __shfl_xor(si, o, kSpmvLanes);
    }
  }
  if (r < n) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = 2 * j + i;
      if (c < nc) Y[(i64)(c0 + c) * n + r] = make_double2(ar[i], ai[i]);
    }
  }
}

__global__ void k_gather_vals(i64 nnz, const int* __restrict__ map, const double2* __restrict__ src,
                              double2* __restrict__ dst) {
  i64 p = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (p < nnz) dst[p] = src[map[p]];
}

}  // namespace

namespace dmp {

int spai_max_cols() { return SPAI_MAXJ; }

void spai_build(i64 n, const ZRef& z, int maxJ, const int* jptr, const int* jidx, const int* iptr, const int* iidx,
                double* vals, int* status, hipStream_t s) {
  DM_REQUIRE(maxJ >= 1 && maxJ <= SPAI_MAXJ, DM_ERR_ARGUMENT, "near-field preconditioner: support width out of range");
  DM_REQUIRE(n < (1LL << 31) - 8, DM_ERR_ARGUMENT, "near-field preconditioner: too many bases for one launch");
  const int per = (int)((n + 7) / 8), nb = (maxJ + 3) / 4;
  double2* v = reinterpret_cast<double2*>(vals);
  // the fewest threads that give every block of the widest support one
  if (nb <= SpaiShape<64>::NB)
    k_spai_build<64><<<8u * (unsigned)per, 64, 0, s>>>((int)n, per, z, jptr, jidx, iptr, iidx, v, status);
  else if (nb <= SpaiShape<128>::NB)
    k_spai_build<128><<<8u * (unsigned)per, 128, 0, s>>>((int)n, per, z, jptr, jidx, iptr, iidx, v, status);
  else
    k_spai_build<256><<<8u * (unsigned)per, 256, 0, s>>>((int)n, per, z, jptr, jidx, iptr, iidx, v, status);
  HIP_OK(hipGetLastError());
}

void csr_from_csc(i64 nnz, const int* map, const double* cscval, double* csrval, hipStream_t s) {
  k_gather_vals<<<(unsigned)((nnz + 255) / 256), 256, 0, s>>>(nnz, map, reinterpret_cast<const double2*>(cscval),
                                                               reinterpret_cast<double2*>(csrval));
  HIP_OK(hipGetLastError());
}

void spmv(i64 n, const int* rowptr, const int* colidx, const double* val, const double* x, double* y, hipStream_t s) {
  k_spmv<<<(unsigned)((n * kSpmvLanes + 255) / 256), 256, 0, s>>>(
      n, rowptr, colidx, reinterpret_cast<const double2*>(val), reinterpret_cast<const double2*>(x),
      reinterpret_cast<double2*>(y));
  HIP_OK(hipGetLastError());
}

void spmm(i64 n, int R, const int* rowptr, const int* colidx, const double* val, const double* X, double* Y,
          hipStream_t s) {
  if (R <= 0) return;
  DM_REQUIRE(R <= 65535, DM_ERR_ARGUMENT, "too many right-hand sides for one sparse product");
  dim3 g((unsigned)((n * kSpmvLanes + 255) / 256), (unsigned)((R + kSpmmCols - 1) / kSpmmCols));
  k_spmm<<<g, 256, 0, s>>>(n, R, rowptr, colidx, reinterpret_cast<const double2*>(val),
                           reinterpret_cast<const double2*>(X), reinterpret_cast<double2*>(Y));
  HIP_OK(hipGetLastError());
}

}  // namespace dmp
