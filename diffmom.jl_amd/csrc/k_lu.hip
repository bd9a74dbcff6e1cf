// k_lu.hip — dense LU with partial pivoting and the triangular solves of the
// direct method (solve_forward :direct, src/solver/Solve.jl:1124-1198).
//
// Right-looking, panels of kLuW columns, three launches per panel:
//   k_lu_panel   one workgroup factors the panel (see below),
//   k_lu_top     every other column: the panel's row exchanges, and for the
//                columns right of the panel U12 = L11^-1 A12,
//   k_lu_update  A22 -= L21 U12 on the FP64 matrix cores.
// Right-hand sides are carried as further columns of the matrix, so the
// factorization leaves L^-1 P B in them and only U x = y remains
// (k_lu_back: every workgroup solves its own columns).  n = 1976 with 64
// right-hand sides: 8.2 + 0.61 ms; with a memory-resident panel and the
// solves column by column it took 25 + 64 x 3.4 ms.
// Pivots: the largest |a|^2 in the column, the smallest row among equal ones.
#include <hip/hip_runtime.h>

#include "dm_common.h"
#include "k_linalg.h"

#include <algorithm>

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int kLuW = 32;

__device__ inline double2 cmul2(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
// c - a b
__device__ inline double2 cfms(double2 c, double2 a, double2 b) {
  c.x = fma(-a.x, b.x, c.x);
  c.x = fma(a.y, b.y, c.x);
  c.y = fma(-a.x, b.y, c.y);
  c.y = fma(-a.y, b.x, c.y);
  return c;
}
// 1 / d.  Where |d|^2 and its reciprocal are normal numbers, by |d|^2; else
// (|d| beyond 2^-511 or 2^511) the same for d scaled by a power of two.
__device__ inline bool plain_range(double dn) { return dn >= 0x1p-1022 && dn <= 0x1p1022; }
__device__ inline double2 crecip_scaled(double2 d) {
  const int e = ilogb(fmax(fabs(d.x), fabs(d.y)));
  d = make_double2(scalbn(d.x, -e), scalbn(d.y, -e));
  const double dn = d.x * d.x + d.y * d.y;
  return make_double2(scalbn(d.x / dn, -e), scalbn(-d.y / dn, -e));
}
__device__ inline double2 crecip(double2 d) {
  const double dn = d.x * d.x + d.y * d.y;
  if (!plain_range(dn)) return crecip_scaled(d);
  return make_double2(d.x / dn, -d.y / dn);
}
// the same by one reciprocal of |d|^2 (hardware estimate, two Newton steps)
__device__ inline double2 crecip_fast(double2 d) {
  const double dn = fma(d.x, d.x, d.y * d.y);
  if (!plain_range(dn)) return crecip_scaled(d);
  double r = __builtin_amdgcn_rcp(dn);
  r = fma(fma(-dn, r, 1.0), r, r);
  r = fma(fma(-dn, r, 1.0), r, r);
  return make_double2(d.x * r, -d.y * r);
}
__device__ inline double rl_f64(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b & 0xffffffffLL), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (long long)lo);
}

template <int CTRL, int ROWS>
__device__ inline int dpp_max(int v) {
  return max(v, __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xF, false));
}
// max over the first LANES (4, 8 or 64) lanes
template <int LANES>
__device__ inline int lanes_max(int v) {
  v = dpp_max<0xB1, 0xF>(v);  // quad_perm 1,0,3,2
  v = dpp_max<0x4E, 0xF>(v);  // quad_perm 2,3,0,1
  if (LANES == 4) return __builtin_amdgcn_readlane(v, 0);
  v = dpp_max<0x141, 0xF>(v);  // row_half_mirror
  if (LANES == 8) return __builtin_amdgcn_readlane(v, 0);
  v = dpp_max<0x140, 0xF>(v);  // row_mirror
  v = dpp_max<0x142, 0xA>(v);  // row_bcast15
  v = dpp_max<0x143, 0xC>(v);  // row_bcast31
  return __builtin_amdgcn_readlane(v, 63);
}
// The lane (of the first LANES) with the largest v (>= 0, or -1 where there is
// none), the smallest row among equal ones: the high words of the doubles
// order like integers, so one integer reduction decides nearly always.
template <int LANES>
__device__ inline int lane_of_max(double v, int row) {
  const long long bits = __double_as_longlong(v);
  const int hi = (int)(bits >> 32);
  const unsigned long long in = LANES == 64 ? ~0ull : (1ull << LANES) - 1;
  const int hm = lanes_max<LANES>(hi);
  unsigned long long win = __ballot(hi == hm) & in;
  if (win & (win - 1)) {
    // equal high words: the low words (sign bit flipped, unsigned order)
    const int lo = (int)((unsigned)(bits & 0xffffffffLL) ^ 0x80000000u);
    const int lm = lanes_max<LANES>(hi == hm ? lo : (int)0x80000000);
    win = __ballot(hi == hm && lo == lm) & in;
    if (win & (win - 1)) {  // equal values: the smallest row
      const int rm = lanes_max<LANES>(hi == hm && lo == lm ? ~row : (int)0x80000000);
      win = __ballot(hi == hm && lo == lm && ~row == rm) & in;
    }
  }
  return __ffsll(win) - 1;
}

// The lanes of one wave see each other's earlier LDS writes after this point.
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The row exchanges piv[0..w) (exchange j: rows j and piv[j] >= j, in order)
// as one gather, built by one wave: lane i < w stands for row i, further
// lanes for the other rows touched; afterwards row pos of a column takes the
// value its row src had.  Returns how many lanes are in use (<= 2 w <= 64).
__device__ inline int exchange_map(int w, const int* piv, int lane, int& pos, int& src) {
  pos = lane < w ? lane : -1;
  src = pos;
  int cnt = w;
  const int pv = piv[min(lane, w - 1)];  // lane j: exchange j
  for (int j = 0; j < w; ++j) {
    const int p = __builtin_amdgcn_readlane(pv, j);
    const unsigned long long hit = __ballot(pos == p);
    int b;
    if (hit) {
      b = __ffsll((unsigned long long)hit) - 1;
    } else {
      b = cnt++;
      if (lane == b) pos = src = p;
    }
    const int sj = __builtin_amdgcn_readlane(src, j), sb = __builtin_amdgcn_readlane(src, b);
    if (lane == j) src = sb;
    if (lane == b) src = sj;
  }
  return cnt;
}

// lane j of every row of 16 lanes, in all lanes of that row
template <int J>
__device__ inline double row_bcast(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)(b & 0xffffffffLL), 0x150 + J, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x150 + J, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
template <int W, int J>
__device__ inline void solve_steps(double2 (&x)[W / 4], const double2 (&l)[W]) {
  if constexpr (J < W) {
#pragma unroll
    for (int c = 0; c < W / 4; ++c) x[c] = cfms(x[c], l[J], make_double2(row_bcast<J>(x[c].x), row_bcast<J>(x[c].y)));
    solve_steps<W, J + 1>(x, l);
  }
}
// U = L^-1 U in LDS by one wave, L unit lower triangular (lt[column][row]):
// lane = row (lane % 16 < W) x a quarter of the columns, its row of L in
// registers, the solved row of each step broadcast by DPP.
template <int W>
__device__ inline void solve_unit_lower(const double2 (&lt)[W][W], double2 (&u)[W][W], int lane) {
  const int i = min(lane & 15, W - 1), g = lane >> 4;
  double2 l[W], x[W / 4];
#pragma unroll
  for (int j = 0; j < W; ++j) l[j] = lt[j][i];
#pragma unroll
  for (int c = 0; c < W / 4; ++c) x[c] = u[i][g * (W / 4) + c];
#pragma unroll
  for (int j = 0; j < W; ++j)
    if (i <= j) l[j] = make_double2(0.0, 0.0);
  solve_steps<W, 0>(x, l);
#pragma unroll
  for (int c = 0; c < W / 4; ++c) u[i][g * (W / 4) + c] = x[c];
}

// One workgroup factors the panel of w columns at k0.  Each thread keeps RPT
// rows x W columns (RPT W <= 32 complex values; local row l = thread + NT r) of
// a sub-panel in registers.  A column step: every wave's largest |a|^2 (an
// integer DPP reduction) to LDS, a barrier, every wave finds the winner among
// the candidates, the winner's thread puts the pivot row into LDS, a barrier,
// every wave takes the row with one LDS read and lane broadcasts, and the rows
// are scaled and updated in registers (exchanged rows stay in theirs; only
// their places change).  Sub-panels are left-looking: the
// columns of the earlier ones are applied W at a time when a sub-panel is
// loaded; its row exchanges reach the panel's other columns in one gather at
// its end.
// What bounds it: the chain of column steps, one workgroup's dependent
// instructions (1.6 us a column with 256 rows, 2.6 us with 1024, 3.8 us with
// 2048).  With the panel in global memory and three barriers a column it took
// 5.7 us at 96 rows, 8.7 us at 1976.  Exchanging the rows in registers through
// LDS, and every wave writing its whole candidate row before one barrier, were
// slower (an LDS write of one lane costs as much as a full one).
template <int NT, int RPT, int W>
__global__ __launch_bounds__(NT) void k_lu_panel(i64 n, i64 ld, int k0, int w, double2* __restrict__ A,
                                                 int* __restrict__ ipiv, int* __restrict__ status) {
  constexpr int NWV = NT / 64, kLv = RPT >= 8 ? 1 : RPT >= 4 ? 2 : 4;
  __shared__ double cval[NWV];  // each wave's candidate
  __shared__ int crow[NWV];
  __shared__ double2 prow[W];          // the pivot row
  __shared__ double2 tri[kLuW / W][W][W];  // diagonal triangles of L, [column][row]
  __shared__ double2 ut[W][W];             // U rows of one earlier sub-panel
  __shared__ int piv[kLuW];
  __shared__ int xpos[2 * W], xsrc[2 * W], xcnt;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = (int)(n - k0);
  static_assert(NWV == 4 || NWV == 8, "lane_of_max<NWV>");
  int zero = 0;  // thread 0: 1 + the first column without a pivot
  double2* P = A + k0 + (i64)k0 * ld;  // local row l, panel column c: P[l + c ld]
  for (int c0 = 0; c0 < w; c0 += W) {
    const int wc = min(W, w - c0);
    double2 a[RPT][W];
    int pos[RPT];  // the row's current place
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      // clamped, unconditional loads (all in flight together)
      const int l = tid + NT * r;
      pos[r] = l;
      const double2* p = P + min(l, m - 1);
#pragma unroll
      for (int c = 0; c < W; ++c) a[r][c] = p[(i64)min(c0 + c, w - 1) * ld];
#pragma unroll
      for (int c = 0; c < W; ++c)
        if (l >= m || c >= wc) a[r][c] = make_double2(0.0, 0.0);
    }
    // apply the earlier sub-panels: W rows of U from the triangle, then
    // a -= L U for the rows below them
    for (int q0 = 0; q0 < c0; q0 += W) {
      const int q = q0 / W;
#pragma unroll
      for (int r = 0; r < RPT; ++r) {
        const int l = tid + NT * r;
        if (l >= q0 && l < q0 + W) {
#pragma unroll
          for (int c = 0; c < W; ++c) ut[l - q0][c] = a[r][c];
        }
      }
      __syncthreads();
      if (wave == 0) solve_unit_lower<W>(tri[q], ut, lane);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < RPT; ++r) {
        const int l = tid + NT * r;
        if (l >= q0 && l < q0 + W) {
#pragma unroll
          for (int c = 0; c < W; ++c) a[r][c] = ut[l - q0][c];
        }
      }
      // kLv columns of L at a time (registers)
#pragma unroll 1
      for (int j0 = 0; j0 < W; j0 += kLv) {
        double2 lv[RPT][kLv], ul[kLv];
#pragma unroll
        for (int j = 0; j < kLv; ++j) ul[j] = ut[j0 + j][lane & (W - 1)];
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
          const double2* p = P + min(tid + NT * r, m - 1);
#pragma unroll
          for (int j = 0; j < kLv; ++j) lv[r][j] = p[(i64)(q0 + j0 + j) * ld];
        }
        // rows above (and past the end) are multiplied by zero
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
          const int l = tid + NT * r;
          if (l < q0 + W || l >= m) {
#pragma unroll
            for (int j = 0; j < kLv; ++j) lv[r][j] = make_double2(0.0, 0.0);
          }
        }
#pragma unroll
        for (int j = 0; j < kLv; ++j)
#pragma unroll
          for (int c = 0; c < W; ++c) {
            const double2 u = make_double2(rl_f64(ul[j].x, c), rl_f64(ul[j].y, c));
#pragma unroll
            for (int r = 0; r < RPT; ++r) a[r][c] = cfms(a[r][c], lv[r][j], u);
          }
      }
      __syncthreads();  // ut is rewritten by the next sub-panel's rows
    }
    // column steps: column c0 + j is a[.][0], and every step rotates the row
    // registers by one column as it updates them, so the loop stays rolled
    // (unrolled, its instructions were fetched anew for every panel: 2.4 us a
    // column) and W steps leave the columns in their places
#pragma unroll 1
    for (int j = 0; j < W; ++j) {
      const int lc = c0 + j;
      bool elim = false;
      double2 pr[W], inv = make_double2(0.0, 0.0);
#pragma unroll
      for (int c = 0; c < W; ++c) pr[c] = make_double2(0.0, 0.0);
      if (j < wc) {
        double best = -1.0;
        int bpos = 0, br = 0;
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
          const double2 v = a[r][0];
          const double q = v.x * v.x + v.y * v.y;
          if (pos[r] >= lc && pos[r] < m && (q > best || (q == best && pos[r] < bpos))) {
            best = q;
            bpos = pos[r];
            br = r;
          }
        }
        if (lane == lane_of_max<64>(best, bpos)) {
          cval[wave] = best;
          crow[wave] = bpos;
        }
        __syncthreads();
        const double cv = cval[lane & (NWV - 1)];
        const int cr = crow[lane & (NWV - 1)];
        const int bw = lane_of_max<NWV>(cv, cr) & (NWV - 1);
        elim = rl_f64(cv, bw) > 0.0;
        const int pv = elim ? __builtin_amdgcn_readlane(cr, bw) : lc;
        // (no global stores here: the next barrier would wait for them)
        if (tid == 0) {
          piv[lc] = pv;
          if (!elim && zero == 0) zero = lc + 1;
        }
        // the rows exchange places, not registers
        const bool mine = best >= 0.0 && bpos == pv;
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
          if (pos[r] == lc)
            pos[r] = pv;
          else if (pos[r] == pv)
            pos[r] = lc;
        }
        if (elim && mine) {
#pragma unroll
          for (int r = 0; r < RPT; ++r)
            if (r == br) {
#pragma unroll
              for (int c = 0; c < W; ++c) prow[c] = a[r][c];
            }
        }
        // also without a pivot: the next column's candidates overwrite these
        __syncthreads();
        if (elim) {
          // one LDS read for the whole row, its entries broadcast by lane
          // reads; columns already done (rotated to the end) are not updated
          const double2 pl = prow[lane & (W - 1)];
#pragma unroll
          for (int c = 0; c < W; ++c) {
            pr[c].x = c < W - j ? rl_f64(pl.x, c) : 0.0;
            pr[c].y = c < W - j ? rl_f64(pl.y, c) : 0.0;
          }
          inv = crecip_fast(pr[0]);
        }
      }
#pragma unroll
      for (int r = 0; r < RPT; ++r) {
        const bool below = elim && pos[r] > lc;
        const double2 a0 = a[r][0], q = cmul2(a0, inv);
        const double2 f = below ? q : make_double2(0.0, 0.0);
#pragma unroll
        for (int c = 1; c < W; ++c) a[r][c - 1] = cfms(a[r][c], f, pr[c]);
        a[r][W - 1] = below ? q : a0;
      }
    }
    // results to memory, the sub-panel's triangle to LDS
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int l = pos[r];
      if (l < m) {
#pragma unroll
        for (int c = 0; c < W; ++c)
          if (c < wc) P[l + (i64)(c0 + c) * ld] = a[r][c];
      }
      if (l >= c0 && l < c0 + W) {
#pragma unroll
        for (int c = 0; c < W; ++c) tri[c0 / W][c][l - c0] = a[r][c];
      }
    }
    __syncthreads();
    // the row exchanges on the panel's other columns
    if (wave == 0) {
      int pos, src;
      // exchanges relative to row c0
      __shared__ int rel[W];
      if (lane < W) rel[lane] = lane < wc ? piv[c0 + lane] - c0 : lane;
      wave_sync();
      const int cnt = exchange_map(wc, rel, lane, pos, src);
      if (lane < cnt) {
        xpos[lane] = c0 + pos;
        xsrc[lane] = c0 + src;
      }
      if (lane == 0) xcnt = cnt;
    }
    __syncthreads();
    const int cnt = xcnt, others = w - wc;
    // items (column, place): all reads of a round of NT items come before its
    // writes, and a round holds whole columns
    const int per = NT / (2 * W);  // columns per round
    for (int o0 = 0; o0 < others; o0 += per) {
      const int o = o0 + tid / (2 * W), i = tid % (2 * W);
      const bool act = o < others && tid / (2 * W) < per && i < cnt;
      const int c = o < c0 ? o : o + wc;
      double2 v = make_double2(0.0, 0.0);
      if (act) v = P[xsrc[i] + (i64)c * ld];
      __syncthreads();
      if (act && xsrc[i] != xpos[i]) P[xpos[i] + (i64)c * ld] = v;
    }
    __syncthreads();
  }
  if (tid < w) ipiv[k0 + tid] = k0 + piv[tid];
  if (zero && status[0] == 0) status[0] = k0 + zero;
}

// The same for panels of more than 4096 rows: the panel stays in memory,
// column by column with three barriers each.
__global__ __launch_bounds__(1024) void k_lu_panel_mem(i64 n, i64 ld, int k0, int w, double2* __restrict__ A,
                                                       int* __restrict__ ipiv, int* __restrict__ status) {
  __shared__ double wbest[16];
  __shared__ int widx[16];
  __shared__ double2 prow[kLuW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int j = 0; j < w; ++j) {
    const i64 c = (i64)k0 + j;
    double m = -1;
    int p = (int)c;
    for (i64 i = c + tid; i < n; i += 1024) {
      const double2 v = A[i + c * ld];
      const double a = v.x * v.x + v.y * v.y;
      if (a > m) {
        m = a;
        p = (int)i;
      }
    }
    // largest |a|^2, smallest row among equal ones: within the wave, then
    // over the 16 waves (every thread reduces the same 16 values)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const double om = __shfl_xor(m, o, 64);
      const int op = __shfl_xor(p, o, 64);
      if (om > m || (om == m && op < p)) {
        m = om;
        p = op;
      }
    }
    if (lane == 0) {
      wbest[wave] = m;
      widx[wave] = p;
    }
    __syncthreads();
    double bm = wbest[0];
    int bp = widx[0];
    for (int q = 1; q < 16; ++q) {
      if (wbest[q] > bm || (wbest[q] == bm && widx[q] < bp)) {
        bm = wbest[q];
        bp = widx[q];
      }
    }
    const bool sing = !(bm > 0.0);
    const int pv = sing ? (int)c : bp;
    if (tid == 0) {
      ipiv[c] = pv;
      if (sing && status[0] == 0) status[0] = (int)c + 1;
    }
    // swap rows c and pv inside the panel; the pivot row to LDS
    if (tid < w) {
      const i64 col = (i64)k0 + tid;
      const double2 rc = A[c + col * ld];
      double2 pr = rc;
      if (pv != c) {
        pr = A[pv + col * ld];
        A[c + col * ld] = pr;
        A[pv + col * ld] = rc;
      }
      prow[tid] = pr;
    }
    __syncthreads();
    if (!sing) {
      const double2 inv = crecip(prow[j]);
      for (i64 i = c + 1 + tid; i < n; i += 1024) {
        const double2 l = cmul2(A[i + c * ld], inv);
        A[i + c * ld] = l;
        double2* row = A + i + (i64)k0 * ld;
        // the row's entries past column j, eight loads issued together per round
#pragma unroll 1
        for (int q0 = 0; q0 < kLuW; q0 += 8) {
          if (q0 + 7 <= j || q0 >= w) continue;
          double2 e[8];
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (q0 + u > j && q0 + u < w) e[u] = row[(i64)(q0 + u) * ld];
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (q0 + u > j && q0 + u < w) row[(i64)(q0 + u) * ld] = cfms(e[u], l, prow[q0 + u]);
        }
      }
    }
    __syncthreads();
  }
}

// Columns outside the panel at k0 (w columns): the panel's row exchanges
// (swap), and for the columns >= solve_from U = L11^-1 T of their top w rows.
// T, ldt: the matrix the columns belong to (the factored one, with the panel's
// own columns skipped, or a block of right-hand sides, own = 0).  64 columns
// per workgroup; L11^-1 is formed in LDS by every workgroup (diagonal blocks of
// 8, then two doublings) while the columns load, and multiplied on the FP64
// matrix cores.  13 us a launch, most of it the block inversions' LDS
// latency (17 with L11 read after the exchange map, the map's exchanges read
// from LDS one by one and the exchanged rows kept in scratch).  (One thread per column substituting through L11 waited ~100 cycles
// for each LDS read: 47 us.)
__global__ __launch_bounds__(256) void k_lu_top(i64 ld, int k0, int w, const double2* __restrict__ A,
                                                const int* __restrict__ ipiv, double2* __restrict__ T, i64 ldt,
                                                i64 ncols, i64 solve_from, int own, int swap) {
  constexpr int LP = kLuW + 1;
  __shared__ double2 L[kLuW][LP];    // [row][column] of L11
  __shared__ double2 V[kLuW][LP];    // L11^-1
  __shared__ double2 H[kLuW][kLuW / 2];
  __shared__ double Br[kLuW][65], Bi[kLuW][65];
  __shared__ int xpos[64], xsrc[64], rel[kLuW], xcnt;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const i64 c0 = blockIdx.x * (i64)64;
  const bool solves = c0 + 64 > solve_from;
  // L11 is on its way while the first wave turns the exchanges into a gather
  double2 l11[kLuW * kLuW / 256];
  if (solves)
#pragma unroll
    for (int q = 0; q < kLuW * kLuW / 256; ++q) {
      const int e = tid + 256 * q;
      l11[q] = A[k0 + min(e % kLuW, w - 1) + (i64)(k0 + min(e / kLuW, w - 1)) * ld];
    }
  if (wave == 0) {
    int pos = lane, src = lane, cnt = w;
    if (swap) {
      if (lane < w) rel[lane] = ipiv[k0 + lane] - k0;
      wave_sync();
      cnt = exchange_map(w, rel, lane, pos, src);
    }
    xpos[lane] = pos;
    xsrc[lane] = src;
    if (lane == 0) xcnt = cnt;
  }
  if (solves)
#pragma unroll
    for (int q = 0; q < kLuW * kLuW / 256; ++q) {
      const int e = tid + 256 * q, c = e / kLuW, r = e % kLuW;
      L[r][c] = (c < w && r < w && r > c) ? l11[q] : make_double2(0.0, 0.0);
      V[r][c] = make_double2(r == c ? 1.0 : 0.0, 0.0);
    }
  __syncthreads();
  const int cnt = xcnt;
  auto valid = [&](i64 col) { return col < ncols && !(own && col >= k0 && col < (i64)k0 + w); };
  // all reads of a column before its writes: the top rows to LDS, the rows
  // exchanged with them to registers (thread (i, v): place i of columns v, v + 8, ...)
  const int i = tid & 31, v0 = tid >> 5;
  // (clamped, unconditional loads: all in flight together)
  double2 x[8], y[8];
  const int sx = xsrc[min(i, w - 1)], sy = xsrc[min(w + i, cnt - 1)];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const double2* t = T + k0 + min(c0 + v0 + 8 * q, ncols - 1) * ldt;
    x[q] = t[sx];
    y[q] = t[sy];
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const bool in = i < w;
    Br[i][v0 + 8 * q] = in ? x[q].x : 0.0;
    Bi[i][v0 + 8 * q] = in ? x[q].y : 0.0;
  }
  if (solves) {
    // diagonal blocks of 8: thread (block, column) substitutes e_column
    if (tid < 32) {
      const int b = tid & ~7, c = tid & 7;
      double2 x[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) x[r] = make_double2(r == c ? 1.0 : 0.0, 0.0);
#pragma unroll
      for (int j = 0; j < 7; ++j)
#pragma unroll
        for (int r = j + 1; r < 8; ++r) x[r] = cfms(x[r], L[b + r][b + j], x[j]);
#pragma unroll
      for (int r = 0; r < 8; ++r) V[b + r][b + c] = x[r];
    }
    __syncthreads();
    // doublings: V21 = -V22 L21 V11 for blocks of 8, then of 16
    for (int h = 8; h < kLuW; h *= 2) {
      const int items = kLuW / (2 * h) * h * h;
      for (int e = tid; e < items; e += 256) {
        const int b = e / (h * h) * 2 * h, r = e % (h * h) / h, c = e % h;
        double2 t = make_double2(0.0, 0.0);
#pragma unroll 8
        for (int j = 0; j < h; ++j) t = cfms(t, L[b + h + r][b + j], V[b + j][b + c]);
        H[b / 2 + r][c] = t;  // -L21 V11
      }
      __syncthreads();
      for (int e = tid; e < items; e += 256) {
        const int b = e / (h * h) * 2 * h, r = e % (h * h) / h, c = e % h;
        double2 t = make_double2(0.0, 0.0);
#pragma unroll 8
        for (int j = 0; j < h; ++j) t = cfms(t, V[b + h + r][b + h + j], H[b / 2 + j][c]);
        V[b + h + r][b + c] = make_double2(-t.x, -t.y);
      }
      __syncthreads();
    }
    // wave: real rows 16 wave .. of the interleaved V (complex rows 8 wave ..),
    // all 64 columns
    v4d accP[4], accQ[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) accP[b] = accQ[b] = (v4d){0.0, 0.0, 0.0, 0.0};
    const double* vr = reinterpret_cast<const double*>(&V[8 * wave + ((lane & 15) >> 1)][0]) + (lane & 1);
#pragma unroll
    for (int kq = 0; kq < kLuW / 4; ++kq) {
      const int kk = 4 * kq + (lane >> 4);
      const double a = vr[2 * kk];
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        accP[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, Br[kk][16 * cb + (lane & 15)], accP[cb], 0, 0, 0);
        accQ[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, Bi[kk][16 * cb + (lane & 15)], accQ[cb], 0, 0, 0);
      }
    }
    __syncthreads();  // every wave has read all rows of Br, Bi
    const bool odd = (lane >> 4) & 1;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const int c = 16 * cb + (lane & 15);
      const v4d p = accP[cb], q = accQ[cb];
      double po[4], qo[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        po[r] = __shfl_xor(p[r], 16, 64);
        qo[r] = __shfl_xor(q[r], 16, 64);
      }
      // columns left of solve_from keep their exchanged values
      if (c0 + c < solve_from) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = (16 * wave + ((lane >> 4) & ~1) + 4 * (odd ? 2 + h : h)) >> 1;
        const double pre = odd ? po[2 + h] : p[h], pim = odd ? p[2 + h] : po[h];
        const double qre = odd ? qo[2 + h] : q[h], qim = odd ? q[2 + h] : qo[h];
        Br[row][c] = pre - qim;
        Bi[row][c] = qre + pim;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const i64 col = c0 + v0 + 8 * q;
    const bool ok = valid(col);
    double2* t = T + k0 + min(col, ncols - 1) * ldt;
    const double2 ex = y[q];
    if (ok && i < w) t[i] = make_double2(Br[i][v0 + 8 * q], Bi[i][v0 + 8 * q]);
    if (ok && w + i < cnt) t[xpos[w + i]] = ex;
  }
}

// T (mr x ncols, ldt) -= L (mr x kLuW, ld) U (kLuW x ncols, leading dimension
// ldu) on the FP64 matrix cores: 64 x 64 complex per workgroup, the whole
// inner dimension staged at once (67 KB of LDS, two workgroups a CU), each
// wave 32 real rows of the interleaved L (see k_zx.hip for the real form and
// the output layout).  20 us on average over the panels of 1976 columns (26
// with each load behind its range test and T read last); the matrix cores and
// the read-modify-write of T (from the last-level cache) take about the same
// time.
constexpr int LU_T = 64;
__global__ __launch_bounds__(256, 2) void k_lu_update(i64 mr, i64 ncols, const double2* __restrict__ L, i64 ld,
                                                      const double2* __restrict__ U, i64 ldu,
                                                      double2* __restrict__ T, i64 ldt) {
  __shared__ double As[kLuW][2 * LU_T + 2];
  __shared__ double Br[kLuW][LU_T + 1];
  __shared__ double Bi[kLuW][LU_T + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4;
  const i64 m0 = (i64)blockIdx.x * LU_T, c0 = (i64)blockIdx.y * LU_T;
  // all loads clamped and unconditional, so that they are in flight together:
  // L and U tiles, then the entries this lane updates (places past the end
  // repeat the last row or column; their products are not stored)
  double2 lv[8], uv[8], ev[2][4][2];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int idx = tid + 256 * q;
    lv[q] = L[min(m0 + (idx & 63), mr - 1) + (i64)(idx >> 6) * ld];
    uv[q] = U[(idx & 31) + min(c0 + (idx >> 5), ncols - 1) * ldu];
  }
  // lanes with even g hold rows r = 0, 1, odd g rows r = 2, 3 of a pair
  auto row_at = [&](int r2, int h) {
    return m0 + ((32 * wave + 16 * r2 + (g & ~1) + 4 * ((g & 1) ? 2 + h : h)) >> 1);
  };
#pragma unroll
  for (int r2 = 0; r2 < 2; ++r2)
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        ev[r2][cb][h] = T[min(row_at(r2, h), mr - 1) + min(c0 + 16 * cb + (lane & 15), ncols - 1) * ldt];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int idx = tid + 256 * q;
    As[idx >> 6][2 * (idx & 63)] = lv[q].x;
    As[idx >> 6][2 * (idx & 63) + 1] = lv[q].y;
    Br[idx & 31][idx >> 5] = uv[q].x;
    Bi[idx & 31][idx >> 5] = uv[q].y;
  }
  __syncthreads();
  v4d accP[2][4], accQ[2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      accP[a][b] = (v4d){0.0, 0.0, 0.0, 0.0};
      accQ[a][b] = (v4d){0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll 2
  for (int kq = 0; kq < kLuW / 4; ++kq) {
    const int kk = 4 * kq + (lane >> 4);
    double a[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) a[r] = As[kk][32 * wave + 16 * r + (lane & 15)];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const double br = Br[kk][16 * cb + (lane & 15)];
      const double bi = Bi[kk][16 * cb + (lane & 15)];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        accP[r][cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], br, accP[r][cb], 0, 0, 0);
        accQ[r][cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], bi, accQ[r][cb], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int r2 = 0; r2 < 2; ++r2)
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const i64 col = c0 + 16 * cb + (lane & 15);
      const v4d p = accP[r2][cb], q = accQ[r2][cb];
      double po[4], qo[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        po[r] = __shfl_xor(p[r], 16, 64);
        qo[r] = __shfl_xor(q[r], 16, 64);
      }
      if (col >= ncols) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool odd = (g & 1) != 0;
        const i64 mrow = row_at(r2, h);
        if (mrow >= mr) continue;
        // even g: (p, q) are the real row's, (po, qo) the imaginary row's
        const double pre = odd ? po[2 + h] : p[h], pim = odd ? p[2 + h] : po[h];
        const double qre = odd ? qo[2 + h] : q[h], qim = odd ? q[2 + h] : qo[h];
        const double2 e = ev[r2][cb][h];
        T[mrow + col * ldt] = make_double2(e.x - (pre - qim), e.y - (qre + pim));
      }
    }
}

// U x = y for one right-hand side per workgroup, written to X: blocks of 32
// rows from the bottom.  One wave solves the block's triangle (rows in
// registers, the triangle staged in LDS with the reciprocals of its
// diagonal), then every thread updates the rows above with the 32 solved
// values.  The right-hand side sits in LDS when LDSB.  Bound by one CU's
// reads of U from L2: 0.64 ms at n = 1976 for up to 256 right-hand sides, each
// on its own CU (one column after the other, forward and back, took 3.4 ms each).
constexpr int kBackT = 512;
template <bool LDSB>
__global__ __launch_bounds__(kBackT) void k_lu_back(i64 n, i64 ld, const double2* __restrict__ A,
                                                  double2* __restrict__ Y, i64 ldy, double2* __restrict__ X, i64 ldx) {
  extern __shared__ double2 sb[];
  __shared__ double2 xs[32], dinv[32];
  __shared__ double2 tri[32][33];  // [row][column]
  double2* yg = Y + (i64)blockIdx.x * ldy;
  double2* b = LDSB ? sb : yg;
  double2* xg = X + (i64)blockIdx.x * ldx;
  const int tid = threadIdx.x, lane = tid & 63;
  if (LDSB)
    for (i64 i = tid; i < n; i += kBackT) sb[i] = yg[i];
  for (i64 k1 = n; k1 > 0;) {
    const i64 k0 = (k1 - 1) / 32 * 32;
    const int w = (int)(k1 - k0);
#pragma unroll
    for (int t = tid; t < 1024; t += kBackT) {
      const int r = t & 31, c = t >> 5;
      if (r < w && c < w && r <= c) {
        const double2 u = A[k0 + r + (k0 + c) * ld];
        tri[r][c] = u;
        if (r == c) dinv[r] = crecip(u);
      }
    }
    // the columns of the first rows above, loaded while the triangle is solved
    double2 e[32];
    const i64 i0 = tid;
#pragma unroll
    for (int j = 0; j < 32; ++j) e[j] = (i0 < k0 && j < w) ? A[i0 + (k0 + j) * ld] : make_double2(0.0, 0.0);
    __syncthreads();
    if (tid < 64) {
      double2 v = lane < w ? b[k0 + lane] : make_double2(0.0, 0.0);
      for (int j = w - 1; j >= 0; --j) {
        const double2 xj = cmul2(make_double2(rl_f64(v.x, j), rl_f64(v.y, j)), dinv[j]);
        if (lane == j) v = xj;
        if (lane < j) v = cfms(v, tri[lane][j], xj);
      }
      if (lane < 32) xs[lane] = lane < w ? v : make_double2(0.0, 0.0);
      if (lane < w) xg[k0 + lane] = v;
    }
    __syncthreads();
    if (i0 < k0) {
      double2 v = b[i0];
#pragma unroll
      for (int j = 0; j < 32; ++j) v = cfms(v, e[j], xs[j]);
      b[i0] = v;
    }
    for (i64 i = i0 + kBackT; i < k0; i += kBackT) {
      double2 v = b[i];
#pragma unroll 16
      for (int j = 0; j < w; ++j) v = cfms(v, A[i + (k0 + j) * ld], xs[j]);
      b[i] = v;
    }
    k1 = k0;
    __syncthreads();
  }
}

inline unsigned nblocks(i64 n, int t) { return (unsigned)((n + t - 1) / t); }

// The panel kernel by the rows it has: up to RPT W = 32 values a thread (128 of
// the 256 registers 512 threads have; 1024 threads spilled), so the sub-panel
// narrows beyond 2048 rows; 16 columns a sub-panel were slower than 8 (62
// against 54 us a panel of 256 rows).  Beyond 4096 rows the memory-resident
// panel (0.8 ms) is as fast as two columns a sub-panel would be.
void launch_panel(i64 n, i64 ld, int k0, int w, double2* a, int* ipiv, int* status, hipStream_t s) {
  const i64 m = n - k0;
  if (m <= 256)
    k_lu_panel<256, 1, 8><<<1, 256, 0, s>>>(n, ld, k0, w, a, ipiv, status);
  else if (m <= 512)
    k_lu_panel<256, 2, 8><<<1, 256, 0, s>>>(n, ld, k0, w, a, ipiv, status);
  else if (m <= 1024)
    k_lu_panel<512, 2, 8><<<1, 512, 0, s>>>(n, ld, k0, w, a, ipiv, status);
  else if (m <= 2048)
    k_lu_panel<512, 4, 8><<<1, 512, 0, s>>>(n, ld, k0, w, a, ipiv, status);
  else if (m <= 4096)
    k_lu_panel<512, 8, 4><<<1, 512, 0, s>>>(n, ld, k0, w, a, ipiv, status);
  else
    k_lu_panel_mem<<<1, 1024, 0, s>>>(n, ld, k0, w, a, ipiv, status);
}

void launch_update(i64 mr, i64 ncols, const double2* L, i64 ld, const double2* U, i64 ldu, double2* T, i64 ldt,
                   hipStream_t s) {
  if (mr <= 0 || ncols <= 0) return;
  dim3 g(nblocks(mr, LU_T), nblocks(ncols, LU_T));
  DM_REQUIRE(g.y <= 65535, DM_ERR_ARGUMENT, "dense LU: too many columns for one launch");
  k_lu_update<<<g, 256, 0, s>>>(mr, ncols, L, ld, U, ldu, T, ldt);
}

constexpr i64 kLuBackLds = 8192;  // right-hand side in LDS up to this many rows (128 KB)

}  // namespace

namespace dml {

void lu_factor(i64 n, i64 ld, double* A, i64 nrhs, int* ipiv, int* status, hipStream_t s) {
  DM_REQUIRE(n >= 1 && n < (1LL << 31) && ld >= n && nrhs >= 0, DM_ERR_ARGUMENT, "dense LU: bad dimensions");
  double2* a = reinterpret_cast<double2*>(A);
  const i64 nc = n + nrhs;
  for (i64 k0 = 0; k0 < n; k0 += kLuW) {
    const int w = (int)std::min<i64>(kLuW, n - k0);
    launch_panel(n, ld, (int)k0, w, a, ipiv, status, s);
    if (nc > w)
      k_lu_top<<<nblocks(nc, 64), 256, 0, s>>>(ld, (int)k0, w, a, ipiv, a, ld, nc, k0 + w, 1, 1);
    // a partial panel is the last one: nothing below it
    launch_update(n - k0 - w, nc - k0 - w, a + (k0 + w) + k0 * ld, ld, a + k0 + (k0 + w) * ld, ld,
                  a + (k0 + w) + (k0 + w) * ld, ld, s);
  }
  HIP_OK(hipGetLastError());
}

void lu_forward(i64 n, i64 ld, const double* A, const int* ipiv, double* B, i64 ldb, i64 nrhs, hipStream_t s) {
  if (nrhs <= 0) return;
  const double2* a = reinterpret_cast<const double2*>(A);
  double2* b = reinterpret_cast<double2*>(B);
  // the stored L has every later exchange applied, so all exchanges come first
  for (int pass = 0; pass < 2; ++pass)
    for (i64 k0 = 0; k0 < n; k0 += kLuW) {
      const int w = (int)std::min<i64>(kLuW, n - k0);
      k_lu_top<<<nblocks(nrhs, 64), 256, 0, s>>>(ld, (int)k0, w, a, ipiv, b, ldb, nrhs, pass ? 0 : nrhs, 0, pass ? 0 : 1);
      if (pass) launch_update(n - k0 - w, nrhs, a + (k0 + w) + k0 * ld, ld, b + k0, ldb, b + k0 + w, ldb, s);
    }
  HIP_OK(hipGetLastError());
}

void lu_back(i64 n, i64 ld, const double* A, double* Y, i64 ldy, double* X, i64 ldx, i64 nrhs, hipStream_t s) {
  if (nrhs <= 0) return;
  const double2* a = reinterpret_cast<const double2*>(A);
  double2 *y = reinterpret_cast<double2*>(Y), *x = reinterpret_cast<double2*>(X);
  if (n <= kLuBackLds) {
    const size_t smem = (size_t)n * sizeof(double2);
    HIP_OK(hipFuncSetAttribute((const void*)k_lu_back<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    k_lu_back<true><<<(unsigned)nrhs, kBackT, smem, s>>>(n, ld, a, y, ldy, x, ldx);
  } else {
    k_lu_back<false><<<(unsigned)nrhs, kBackT, 0, s>>>(n, ld, a, y, ldy, x, ldx);
  }
  HIP_OK(hipGetLastError());
}

}  // namespace dml
