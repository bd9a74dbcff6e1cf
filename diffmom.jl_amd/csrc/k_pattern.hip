// k_pattern.hip — the near-field pattern of the sparse approximate inverse on
// the device: J_j = the (at most maxJ nearest) bases with centre distance <=
// cutJ from basis j, I_j = the bases within 1.6 x the radius J_j covers (at most
// 512 nearest), equal distances in the order of the internal index, and the CSR
// form of the J lists.  The distances are formed exactly as
// dmh::spai_pattern_host forms them (no contraction), so both give the same
// lists.
//
// One wave per column: the internal order's blocks of 64 bases are compact
// patches, so their bounding boxes select the candidates (every lane tests a
// block, the chosen blocks' 64 bases are tested together, and the candidates
// stay in index order); the nearest maxJ (and 512) are the candidates up to a
// distance found bit by bit (first_k), which needs no sort.  Bound by the waves'
// serial steps.  A plate of 4720 bases with a cutoff of one wavelength: the host
// form (hash grid, sort per column, one thread) takes 140 ms, this 0.25 ms
// (0.14 of it k_pat_cols; counting every candidate's rank against the others, c^2
// comparisons, it was 1.1).
#include <hip/hip_runtime.h>

#include "dm_common.h"

namespace {

constexpr int kBlk = 64;
constexpr int kCap = 1024;   // candidates a wave holds
constexpr int kMaxI = 512;   // rows of a column's least-squares problem
constexpr int kWaves = 4;    // columns per workgroup

__device__ inline double dist3(const double* __restrict__ c, i64 a, double x, double y, double z) {
#pragma clang fp contract(off)
  const double dx = c[3 * a] - x, dy = c[3 * a + 1] - y, dz = c[3 * a + 2] - z;
  return sqrt(dx * dx + dy * dy + dz * dz);
}

// distance of a point to a box, not above the computed distance to any centre
// in it (every operation is monotone)
__device__ inline double box_dist(const double* __restrict__ b, double x, double y, double z) {
#pragma clang fp contract(off)
  const double dx = fmax(fmax(b[0] - x, x - b[3]), 0.0), dy = fmax(fmax(b[1] - y, y - b[4]), 0.0),
               dz = fmax(fmax(b[2] - z, z - b[5]), 0.0);
  return sqrt(dx * dx + dy * dy + dz * dz);
}

// what the host reads back
struct PatInfo {
  i64 nnzJ, nnzI, capped;
  int maxJ, fail;
};

__global__ __launch_bounds__(kBlk) void k_pat_boxes(i64 n, const double* __restrict__ c, double* __restrict__ box) {
  const i64 i = blockIdx.x * (i64)kBlk + threadIdx.x;
  double lo[3], hi[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    lo[k] = i < n ? c[3 * i + k] : INFINITY;
    hi[k] = i < n ? c[3 * i + k] : -INFINITY;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo[k] = fmin(lo[k], __shfl_xor(lo[k], o, 64));
      hi[k] = fmax(hi[k], __shfl_xor(hi[k], o, 64));
    }
  }
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      box[6 * (i64)blockIdx.x + k] = lo[k];
      box[6 * (i64)blockIdx.x + 3 + k] = hi[k];
    }
}

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Which of a wave's cnt distances (lane, lane + 64, ... in v; infinite past cnt)
// are among the first k by (distance, position): bit q of sel.  The k-th smallest
// distance is built bit by bit from the top (distances are not negative, so they
// order as integers), each bit by a count of the smaller ones; among equal ones
// the first positions are taken.
__device__ inline void first_k(const double (&v)[kCap / 64], int cnt, int k, unsigned long long below, unsigned& sel) {
  sel = ~0u;
  if (cnt <= k) return;
  unsigned long long t = 0;
  int less = 0;
  for (int bit = 62; bit >= 0; --bit) {
    const unsigned long long trial = t | 1ull << bit;
    int c = 0;
#pragma unroll
    for (int q = 0; q < kCap / 64; ++q)
      if (q * 64 < cnt) c += __popcll(__ballot((unsigned long long)__double_as_longlong(v[q]) < trial));
    if (c < k) {
      t = trial;
      less = c;
    }
  }
  sel = 0;
  int eq = k - less;  // equal ones still to be taken
#pragma unroll
  for (int q = 0; q < kCap / 64; ++q) {
    if (q * 64 >= cnt) continue;
    const unsigned long long b = (unsigned long long)__double_as_longlong(v[q]);
    const unsigned long long same = __ballot(b == t);
    if (b < t || (b == t && (int)__popcll(same & below) < eq)) sel |= 1u << q;
    eq -= (int)__popcll(same);
  }
}

// Lists of column j at tJ + j maxJ and tI + j kMaxI, their lengths and the
// radius.  The search radius R starts at `cell` and grows by `cell` until both
// lists are certain to be complete; a patch with more than kCap bases within R
// is searched again with radii between (fail = 1 if none serves: the host
// form is used instead).
__global__ __launch_bounds__(64 * kWaves) void k_pat_cols(i64 n, i64 nblk, const double* __restrict__ c,
                                                          const double* __restrict__ box, double cutJ, double cell,
                                                          int maxJ, int* __restrict__ tJ, int* __restrict__ tI,
                                                          int* __restrict__ nJo, int* __restrict__ nIo,
                                                          double* __restrict__ rJo, PatInfo* info) {
  __shared__ double ds[kWaves][kCap];
  __shared__ int ms[kWaves][kCap];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const i64 j = blockIdx.x * (i64)kWaves + wave;
  if (j >= n) return;
  double* d = ds[wave];
  int* m = ms[wave];
  const double x = c[3 * j], y = c[3 * j + 1], z = c[3 * j + 2];
  const unsigned long long below = (1ull << lane) - 1;
  double R = cell, lo = 0.0, hi = INFINITY;
  int w = 1;
  for (int iter = 0; iter < 64; ++iter) {
    int cnt = 0;
    for (i64 b0 = 0; b0 < nblk && cnt <= kCap; b0 += 64) {
      const i64 b = b0 + lane;
      unsigned long long sel = __ballot(b < nblk && box_dist(box + 6 * (b < nblk ? b : 0), x, y, z) <= R);
      while (sel && cnt <= kCap) {
        const i64 i = (b0 + __ffsll(sel) - 1) * kBlk + lane;
        sel &= sel - 1;
        const double dd = i < n ? dist3(c, i, x, y, z) : INFINITY;
        const bool in = dd <= R;
        const unsigned long long bal = __ballot(in);
        const int at = cnt + __popcll(bal & below);
        if (in && at < kCap) {
          d[at] = dd;
          m[at] = (int)i;
        }
        cnt += __popcll(bal);
      }
    }
    wave_sync();
    if (cnt > kCap) {
      hi = R;
      R = 0.5 * (lo + hi);
      continue;
    }
    // candidates lane, lane + 64, ... (list order is index order)
    double dv[kCap / 64];
#pragma unroll
    for (int q = 0; q < kCap / 64; ++q)
      dv[q] = q * 64 < cnt && lane + 64 * q < cnt ? d[lane + 64 * q] : INFINITY;
    unsigned selJ, selI;  // bit q: among the first maxJ (kMaxI) by (distance, index)
    first_k(dv, cnt, maxJ, below, selJ);
    first_k(dv, cnt, kMaxI, below, selI);
    int nJ = 0;
    bool self = false, next = false;
    double rJ = 0.0;
#pragma unroll
    for (int q = 0; q < kCap / 64; ++q) {
      if (q * 64 >= cnt) continue;
      const bool near = dv[q] <= cutJ && lane + 64 * q < cnt, in = near && (selJ >> q & 1);
      nJ += __popcll(__ballot(in));
      self = self || (in && m[lane + 64 * q] == (int)j);
      next = next || (near && !in);  // past the first maxJ
      if (in) rJ = fmax(rJ, dv[q]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) rJ = fmax(rJ, __shfl_xor(rJ, o, 64));
    const bool all = cnt == n, shrunk = hi < INFINITY;
    const double rI = fmax(1.6 * rJ, 1e-300);
    const bool j_done = (nJ >= maxJ && (!shrunk || cnt > maxJ)) || cutJ <= R || all;
    const bool i_done = rI <= R || all || (shrunk && cnt >= kMaxI);
    if (!(j_done && i_done)) {
      lo = R;
      if (shrunk)
        R = 0.5 * (lo + hi);
      else
        R = ++w * cell;
      wave_sync();
      continue;
    }
    if (!__any(self)) break;  // more than maxJ bases at the same place
    int nI = 0, at = 0;
#pragma unroll
    for (int q = 0; q < kCap / 64; ++q) {
      if (q * 64 >= cnt) continue;
      const bool ok = lane + 64 * q < cnt;
      const int mm = m[ok ? lane + 64 * q : 0];
      const bool inJ = ok && (selJ >> q & 1) && dv[q] <= cutJ, inI = ok && (selI >> q & 1) && dv[q] <= rI;
      const unsigned long long bJ = __ballot(inJ), bI = __ballot(inI);
      if (inJ) tJ[j * maxJ + at + __popcll(bJ & below)] = mm;
      if (inI) tI[j * kMaxI + nI + __popcll(bI & below)] = mm;
      at += __popcll(bJ);
      nI += __popcll(bI);
    }
    const bool capped = nJ >= maxJ && __any(next);
    if (lane == 0) {
      nJo[j] = nJ;
      nIo[j] = nI;
      rJo[j] = rJ;
      if (capped) atomicAdd((unsigned long long*)&info->capped, 1ull);
    }
    return;
  }
  if (lane == 0) {
    nJo[j] = nIo[j] = 0;
    rJo[j] = 0.0;
    info->fail = 1;
  }
}

// exclusive prefix sums of cnt into ptr (n + 1 values), one workgroup;
// total and maximum, where given, to the host's record
__global__ __launch_bounds__(1024) void k_pat_scan(i64 n, const int* __restrict__ cnt, int* __restrict__ ptr,
                                                   i64* total, int* most) {
  __shared__ i64 part[16];
  __shared__ int mx[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const i64 per = (n + 1023) / 1024, i0 = per * tid, i1 = min(n, i0 + per);
  i64 s = 0;
  int m = 0;
  for (i64 i = i0; i < i1; ++i) {
    s += cnt[i];
    m = max(m, cnt[i]);
  }
  i64 inc = s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const i64 v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
  if (lane == 63) part[wave] = inc;
  if (lane == 0) mx[wave] = m;
  __syncthreads();
  i64 base = 0;
  for (int q = 0; q < wave; ++q) base += part[q];
  i64 at = base + inc - s;
  for (i64 i = i0; i < i1; ++i) {
    ptr[i] = (int)at;
    at += cnt[i];
  }
  if (tid == 1023) {
    ptr[n] = (int)(base + inc);
    if (total) *total = base + inc;
    if (most) {
      for (int q = 0; q < 16; ++q) m = max(m, mx[q]);
      *most = m;
    }
  }
}

// the lists of column blockIdx.x in their places, and the row counts of M
__global__ __launch_bounds__(256) void k_pat_pack(i64 n, int maxJ, const int* __restrict__ tJ,
                                                  const int* __restrict__ tI, const int* __restrict__ jptr,
                                                  const int* __restrict__ iptr, int* __restrict__ jidx,
                                                  int* __restrict__ iidx, int* __restrict__ rows) {
  const i64 j = blockIdx.x * (i64)4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (j >= n) return;
  const int j0 = jptr[j], nJ = jptr[j + 1] - j0, i0 = iptr[j], nI = iptr[j + 1] - i0;
  for (int a = lane; a < nJ; a += 64) {
    const int r = tJ[j * maxJ + a];
    jidx[j0 + a] = r;
    atomicAdd(rows + r, 1);
  }
  for (int a = lane; a < nI; a += 64) iidx[i0 + a] = tI[j * kMaxI + a];
}

// largest radius of the columns of every block of 64
__global__ __launch_bounds__(kBlk) void k_pat_reach(i64 n, const double* __restrict__ rJ, double* __restrict__ reach) {
  const i64 i = blockIdx.x * (i64)kBlk + threadIdx.x;
  double r = i < n ? rJ[i] : 0.0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) r = fmax(r, __shfl_xor(r, o, 64));
  if (threadIdx.x == 0) reach[blockIdx.x] = r;
}

// Row r of M: the columns whose list holds r, in index order (a column within
// its own radius of r is looked up in its sorted list), and each entry's
// place among the columns' entries.
__global__ __launch_bounds__(256) void k_pat_rows(i64 n, i64 nblk, const double* __restrict__ c,
                                                  const double* __restrict__ box, const double* __restrict__ reach,
                                                  const double* __restrict__ rJ, const int* __restrict__ jptr,
                                                  const int* __restrict__ jidx, const int* __restrict__ rowptr,
                                                  int* __restrict__ colidx, int* __restrict__ map, PatInfo* info) {
  const i64 r = blockIdx.x * (i64)4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= n) return;
  const double x = c[3 * r], y = c[3 * r + 1], z = c[3 * r + 2];
  const unsigned long long below = (1ull << lane) - 1;
  int at = rowptr[r];
  const int end = rowptr[r + 1];
  for (i64 b0 = 0; b0 < nblk; b0 += 64) {
    const i64 b = b0 + lane;
    unsigned long long sel = __ballot(b < nblk && box_dist(box + 6 * (b < nblk ? b : 0), x, y, z) <= reach[b < nblk ? b : 0]);
    while (sel) {
      const i64 j = (b0 + __ffsll(sel) - 1) * kBlk + lane;
      sel &= sel - 1;
      int p = -1;
      if (j < n && dist3(c, j, x, y, z) <= rJ[j]) {
        int l = jptr[j], h = jptr[j + 1];
        while (l < h) {
          const int mid = (l + h) >> 1;
          if (jidx[mid] < (int)r)
            l = mid + 1;
          else
            h = mid;
        }
        if (l < jptr[j + 1] && jidx[l] == (int)r) p = l;
      }
      const unsigned long long bal = __ballot(p >= 0);
      const int q = at + __popcll(bal & below);
      if (p >= 0 && q < end) {
        colidx[q] = (int)j;
        map[q] = p;
      }
      at += __popcll(bal);
    }
  }
  if (lane == 0 && at != end) info->fail = 1;
}

}  // namespace

namespace dmp {

bool spai_pattern_device(i64 n, const double* centres, double mean_len, double cutJ, int maxJ, SpaiPattern& P,
                         hipStream_t s) {
  if (n >= (1LL << 31) / kMaxI) return false;  // 32-bit list positions
  const i64 nblk = (n + kBlk - 1) / kBlk;
  const double reach0 = std::sqrt((double)maxJ / 3.0) * mean_len;  // ~ radius of maxJ nearest
  const double cell = 1.6 * std::max(std::min(cutJ, reach0), 1e-300);
  DBuf<double> c, box, rJ, reach;
  DBuf<int> tJ, tI, nJ, nI, rows;
  DBuf<PatInfo> info;
  c.upload(centres, 3 * n, s);
  box.alloc(6 * nblk);
  reach.alloc(nblk);
  rJ.alloc(n);
  tJ.alloc((size_t)n * maxJ);
  tI.alloc((size_t)n * kMaxI);
  nJ.alloc(n);
  nI.alloc(n);
  rows.alloc(n);
  info.alloc(1);
  P.d_jptr.alloc(n + 1);
  P.d_iptr.alloc(n + 1);
  P.d_rowptr.alloc(n + 1);
  HIP_OK(hipMemsetAsync(info.p, 0, sizeof(PatInfo), s));
  HIP_OK(hipMemsetAsync(rows.p, 0, sizeof(int) * n, s));
  k_pat_boxes<<<(unsigned)nblk, kBlk, 0, s>>>(n, c.p, box.p);
  k_pat_cols<<<(unsigned)((n + kWaves - 1) / kWaves), 64 * kWaves, 0, s>>>(n, nblk, c.p, box.p, cutJ, cell, maxJ, tJ.p,
                                                                          tI.p, nJ.p, nI.p, rJ.p, info.p);
  k_pat_scan<<<1, 1024, 0, s>>>(n, nJ.p, P.d_jptr.p, &info.p->nnzJ, &info.p->maxJ);
  k_pat_scan<<<1, 1024, 0, s>>>(n, nI.p, P.d_iptr.p, &info.p->nnzI, nullptr);
  HIP_OK(hipGetLastError());
  PatInfo h;
  std::vector<double> rh(n);
  HIP_OK(hipMemcpyAsync(&h, info.p, sizeof(h), hipMemcpyDeviceToHost, s));
  HIP_OK(hipMemcpyAsync(rh.data(), rJ.p, sizeof(double) * n, hipMemcpyDeviceToHost, s));
  HIP_OK(hipStreamSynchronize(s));
  if (h.fail || h.nnzJ >= (1LL << 31) || h.nnzI >= (1LL << 31)) return false;
  P.nnz = h.nnzJ;
  P.max_cols = h.maxJ;
  P.capped = h.capped;
  double rsum = 0;
  for (double v : rh) rsum += v;
  P.mean_radius = rsum / (double)n;
  P.d_jidx.alloc(h.nnzJ);
  P.d_iidx.alloc(h.nnzI);
  P.d_colidx.alloc(h.nnzJ);
  P.d_map.alloc(h.nnzJ);
  const unsigned g = (unsigned)((n + 3) / 4);
  k_pat_pack<<<g, 256, 0, s>>>(n, maxJ, tJ.p, tI.p, P.d_jptr.p, P.d_iptr.p, P.d_jidx.p, P.d_iidx.p, rows.p);
  k_pat_scan<<<1, 1024, 0, s>>>(n, rows.p, P.d_rowptr.p, nullptr, nullptr);
  k_pat_reach<<<(unsigned)nblk, kBlk, 0, s>>>(n, rJ.p, reach.p);
  k_pat_rows<<<g, 256, 0, s>>>(n, nblk, c.p, box.p, reach.p, rJ.p, P.d_jptr.p, P.d_jidx.p, P.d_rowptr.p, P.d_colidx.p,
                               P.d_map.p, info.p);
  HIP_OK(hipGetLastError());
  HIP_OK(hipMemcpyAsync(&h, info.p, sizeof(h), hipMemcpyDeviceToHost, s));
  HIP_OK(hipStreamSynchronize(s));
  return h.fail == 0;
}

}  // namespace dmp
