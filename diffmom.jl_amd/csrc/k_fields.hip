// k_fields.hip — plane-wave right-hand sides and radiation vectors.
//
// With f = sigma * len/(2A) * (r - v_e) on each half of a basis (sigma already
// folded with the mesh/RWG area ratio in hsig), the reference's per-point
// terms reduce to
//   v_n   = -len_n sum_halves hsig sum_q w_q (r_q - v_e) . E_inc(r_q)
//           (assemble_plane_wave, src/assembly/Excitation.jl:2829-2896;
//            E_inc = pol E0 exp(-i k.r), src/assembly/Excitation.jl:1517-1547)
//   g_n(r^) = (i k eta0/4pi) len_n sum_halves hsig sum_q w_q
//             r^ x (r^ x (r_q - v_e)) exp(+i k r^.r_q) / |r^|^2
//           (radiation_vectors, src/postprocessing/FarField.jl:425-574)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "dm_common.h"
#include "k_linalg.h"

namespace {

struct PwArgs {
  i64 n;
  int nq, M;
  const int* tp;
  const int* tm;
  const int* ep;
  const int* em;
  const double* len;
  const double* hsig;
  const double* rq;
  const double* vtx;
  const double* kvec;  // 3*M
  const double* pol;   // 3*M
  const double* E0;    // M
  const int* out_idx;
  double w[7];
};

__global__ __launch_bounds__(256) void k_planewave(PwArgs a, double2* __restrict__ V, i64 ldv) {
  i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx >= a.n * a.M) return;
  i64 i = idx % a.n;
  int m = (int)(idx / a.n);
  const double* kv = a.kvec + 3 * m;
  const double* pl = a.pol + 3 * m;
  double E0 = a.E0[m];
  double accr = 0, acci = 0;
  for (int side = 0; side < 2; ++side) {
    i64 t = side ? a.tm[i] : a.tp[i];
    int e = side ? a.em[i] : a.ep[i];
    double s = a.hsig[3 * t + e];
    const double* v = a.vtx + 9 * t + 3 * e;
    double hr = 0, hi = 0;
    for (int q = 0; q < a.nq; ++q) {
      const double* r = a.rq + (t * a.nq + q) * 3;
      double arg = kv[0] * r[0] + kv[1] * r[1] + kv[2] * r[2];
      double sn, cs;
      sincos(arg, &sn, &cs);
      double fe = (r[0] - v[0]) * pl[0] + (r[1] - v[1]) * pl[1] + (r[2] - v[2]) * pl[2];
      double c = a.w[q] * fe * E0;
      hr += c * cs;
      hi -= c * sn;
    }
    accr += s * hr;
    acci += s * hi;
  }
  double l = a.len[i];
  V[(a.out_idx ? (i64)a.out_idx[i] : i) + (i64)m * ldv] = make_double2(-l * accr, -l * acci);
}

struct RadArgs {
  i64 n, nomega;
  int nq;
  const int* tp;
  const int* tm;
  const int* ep;
  const int* em;
  const int* ext;
  const double* len;
  const double* hsig;
  const double* rq;
  const double* vtx;
  const double* rhat;
  double k, eta0;
  double w[7];
};

__global__ __launch_bounds__(256) void k_radiation(RadArgs a, double2* __restrict__ G) {
  i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx >= a.n * a.nomega) return;
  i64 i = idx / a.nomega;
  i64 qd = idx % a.nomega;
  double rh[3] = {a.rhat[3 * qd], a.rhat[3 * qd + 1], a.rhat[3 * qd + 2]};
  double rn2 = rh[0] * rh[0] + rh[1] * rh[1] + rh[2] * rh[2];
  double tr[3] = {0, 0, 0}, ti[3] = {0, 0, 0};
  for (int side = 0; side < 2; ++side) {
    i64 t = side ? a.tm[i] : a.tp[i];
    int e = side ? a.em[i] : a.ep[i];
    double s = a.hsig[3 * t + e];
    const double* v = a.vtx + 9 * t + 3 * e;
    for (int q = 0; q < a.nq; ++q) {
      const double* r = a.rq + (t * a.nq + q) * 3;
      double sn, cs;
      sincos(a.k * (rh[0] * r[0] + rh[1] * r[1] + rh[2] * r[2]), &sn, &cs);
      double f[3] = {r[0] - v[0], r[1] - v[1], r[2] - v[2]};
      // r^ x (r^ x f) = r^ (r^.f) - f |r^|^2
      double rf = rh[0] * f[0] + rh[1] * f[1] + rh[2] * f[2];
      double c = s * a.w[q] / rn2;
      for (int j = 0; j < 3; ++j) {
        double b = (rh[j] * rf - f[j] * rn2) * c;
        tr[j] += b * cs;
        ti[j] += b * sn;
      }
    }
  }
  // prefactor i k eta0 / (4 pi) * len
  double pf = a.k * a.eta0 * 0.07957747154594767 * a.len[i];
  i64 col = a.ext[i];
  i64 rows = 3 * a.nomega;
  for (int j = 0; j < 3; ++j) G[3 * qd + j + col * rows] = make_double2(-pf * ti[j], pf * tr[j]);
}

// ------------------------------------------------------------ far fields
// E = G I without the radial component: g_n is transverse, so with u, v an
// orthonormal pair perpendicular to r^ only u . g and v . g are formed and
// multiplied (two rows a direction instead of three), and E = u (u.E) + v (v.E).
__device__ inline void transverse_pair(const double* r, double* u, double* v) {
  const double rn = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
  const double h[3] = {r[0] / rn, r[1] / rn, r[2] / rn};
  const double a[3] = {fabs(h[0]), fabs(h[1]), fabs(h[2])};
  const int k = a[0] <= a[1] && a[0] <= a[2] ? 0 : a[1] <= a[2] ? 1 : 2;  // e_k: the axis farthest from r^
  const double e[3] = {k == 0 ? 1.0 : 0.0, k == 1 ? 1.0 : 0.0, k == 2 ? 1.0 : 0.0};
  u[0] = e[1] * h[2] - e[2] * h[1];
  u[1] = e[2] * h[0] - e[0] * h[2];
  u[2] = e[0] * h[1] - e[1] * h[0];
  const double un = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
  for (int c = 0; c < 3; ++c) u[c] /= un;
  v[0] = h[1] * u[2] - h[2] * u[1];
  v[1] = h[2] * u[0] - h[0] * u[2];
  v[2] = h[0] * u[1] - h[1] * u[0];
}

struct FfArgs {
  i64 n, nt, nomega;
  int nq, TB;
  const int* blk_off;
  const int* blk_tri;
  const int* hrwg;
  const double* hsig;
  const int* tp;
  const int* ext;
  const double* len;
  const double* rq;
  const double* vtx;
  const double* rhat;
  double k, pf;  // pf = k eta0 / (4 pi)
  double w[7];
};

// Rows (u.g, v.g) of DIRS directions for one block of bases.  The block's
// triangles' phases are formed once in LDS and serve every half-basis on them
// (a block of 64 bases has 128 halves on ~53 triangles), which is where the
// time goes (FP64 sincos).  7680 bases x 2592 directions: 0.36 ms (every basis
// forming its six phases and three components: 0.53).  G: 2 nomega x n, caller
// basis order.
template <int DIRS>
__global__ __launch_bounds__(256) void k_rad_uv(FfArgs a, double2* __restrict__ G) {
  // phases [triangle of the block x nq][DIRS], then the halves' weighted
  // vectors [basis][side x nq][3]
  extern __shared__ double2 ph[];
  __shared__ double rh[DIRS][3], uu[DIRS][3], vv[DIRS][3];
  __shared__ int loc[64][2];
  const int tid = threadIdx.x, b = blockIdx.x, nq = a.nq;
  const i64 d0 = blockIdx.y * (i64)DIRS, base = (i64)b * a.TB;
  const int nb = (int)min((i64)a.TB, a.n - base);
  const int t0 = a.blk_off[b], nt = a.blk_off[b + 1] - t0;
  if (tid < DIRS) {
    const i64 d = min(d0 + tid, a.nomega - 1);
    double r[3], u[3], v[3];
    for (int c = 0; c < 3; ++c) r[c] = a.rhat[3 * d + c];
    transverse_pair(r, u, v);
    for (int c = 0; c < 3; ++c) {
      rh[tid][c] = r[c];
      uu[tid][c] = u[c];
      vv[tid][c] = v[c];
    }
  }
  double* fc = reinterpret_cast<double*>(ph + (size_t)nt * nq * DIRS);
  // the two halves of every basis of the block: local triangle, vectors
  for (int e = tid; e < 3 * nt; e += 256) {
    const int t = a.blk_tri[t0 + e / 3], slot = a.hrwg[3 * t + e % 3] - (int)base;
    if (slot >= 0 && slot < nb) {
      const int side = a.tp[base + slot] == t ? 0 : 1;
      loc[slot][side] = e / 3;
      const double sg = a.hsig[3 * t + e % 3];
      const double* vx = a.vtx + 9 * (i64)t + 3 * (e % 3);
      for (int q = 0; q < nq; ++q) {
        const double* r = a.rq + ((i64)t * nq + q) * 3;
        double* f = fc + ((slot * 2 + side) * nq + q) * 3;
        for (int c = 0; c < 3; ++c) f[c] = sg * a.w[q] * (r[c] - vx[c]);
      }
    }
  }
  __syncthreads();  // rh
  for (int e = tid; e < nt * nq * DIRS; e += 256) {
    const int d = e % DIRS, p = e / DIRS;
    const double* r = a.rq + ((i64)a.blk_tri[t0 + p / nq] * nq + p % nq) * 3;
    double sn, cs;
    sincos(a.k * (rh[d][0] * r[0] + rh[d][1] * r[1] + rh[d][2] * r[2]), &sn, &cs);
    ph[e] = make_double2(cs, sn);
  }
  __syncthreads();
  for (int e = tid; e < nb * DIRS; e += 256) {
    const int d = e % DIRS, s = e / DIRS;
    if (d0 + d >= a.nomega) continue;
    double ur = 0, ui = 0, vr = 0, vi = 0;
    const double u0 = uu[d][0], u1 = uu[d][1], u2 = uu[d][2], v0 = vv[d][0], v1 = vv[d][1], v2 = vv[d][2];
    for (int side = 0; side < 2; ++side) {
      const double2* x = ph + (size_t)loc[s][side] * nq * DIRS + d;
      const double* f = fc + (s * 2 + side) * nq * 3;
      for (int q = 0; q < nq; ++q) {
        const double fu = f[3 * q] * u0 + f[3 * q + 1] * u1 + f[3 * q + 2] * u2;
        const double fv = f[3 * q] * v0 + f[3 * q + 1] * v1 + f[3 * q + 2] * v2;
        const double2 e = x[q * DIRS];
        ur += fu * e.x;
        ui += fu * e.y;
        vr += fv * e.x;
        vi += fv * e.y;
      }
    }
    // r^ x (r^ x f) / |r^|^2 = -(f - r^ (r^.f) / |r^|^2); prefactor i k eta0 / (4 pi) len
    const double pf = -a.pf * a.len[base + s];
    double2* g = G + (i64)a.ext[base + s] * (2 * a.nomega) + 2 * (d0 + d);
    g[0] = make_double2(-pf * ui, pf * ur);
    g[1] = make_double2(-pf * vi, pf * vr);
  }
}

// E (3 nomega rows) from the nk partial sums of (u.E, v.E): part[c][col][2 nomega]
__global__ __launch_bounds__(256) void k_ff_join(i64 nomega, int R, int nk, const double* __restrict__ rhat,
                                                 const double2* __restrict__ part, double2* __restrict__ E, i64 lde) {
  const i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx >= nomega * R) return;
  const i64 d = idx % nomega, col = idx / nomega;
  double2 a = make_double2(0.0, 0.0), b = a;
  for (int c = 0; c < nk; ++c) {
    const double2* p = part + ((i64)c * R + col) * (2 * nomega) + 2 * d;
    a.x += p[0].x;
    a.y += p[0].y;
    b.x += p[1].x;
    b.y += p[1].y;
  }
  double u[3], v[3];
  transverse_pair(rhat + 3 * d, u, v);
  for (int c = 0; c < 3; ++c)
    E[3 * d + c + col * lde] = make_double2(u[c] * a.x + v[c] * b.x, u[c] * a.y + v[c] * b.y);
}

// Few currents (up to eight): G is never formed; forming and multiplying it costs
// the same for 1 and for 64 currents (0.77 ms at 7680 bases x 2592 directions).
// F[p][r] = the currents' (unnormalised) vector at quadrature point p of every
// triangle, 3 complex, times its weight;
// E(r^) = -i k eta0 / (4 pi) (1 - r^ r^) sum_p F[p] exp(i k r^.r_p).
constexpr int FF_R = dmf::kFfCurrents;  // currents per pass
constexpr int FF_ROW = 6 * FF_R;  // doubles per point: [current][x, y, z][re, im]
__global__ __launch_bounds__(256) void k_ff_points(FfArgs a, const double2* __restrict__ I, i64 ldi, int R,
                                                   double* __restrict__ F) {
  const i64 p = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (p >= a.nt * a.nq) return;
  const i64 t = p / a.nq;
  double f[FF_ROW];
#pragma unroll
  for (int i = 0; i < FF_ROW; ++i) f[i] = 0.0;
  for (int e = 0; e < 3; ++e) {
    const int s = a.hrwg[3 * t + e];
    if (s < 0) continue;
    const double c = a.hsig[3 * t + e] * a.w[p % a.nq] * a.len[s];
#pragma unroll
    for (int r = 0; r < FF_R; ++r) {
      const double2 x = I[a.ext[s] + min(r, R - 1) * ldi];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double d = c * (a.rq[3 * p + k] - a.vtx[9 * t + 3 * e + k]);
        f[6 * r + 2 * k] += d * x.x;
        f[6 * r + 2 * k + 1] += d * x.y;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < FF_ROW; ++i) F[p * FF_ROW + i] = f[i];
}

// One direction per thread, the points [blockIdx.y per, ...) in sequence (their
// data is uniform over the wave); part[chunk][current][u, v interleaved] as
// k_ff_join reads it.  Bound by FP64 sincos.
__global__ __launch_bounds__(64) void k_ff_direct(FfArgs a, i64 per, int R, const double* __restrict__ F,
                                                  double2* __restrict__ part) {
  const i64 d = blockIdx.x * (i64)64 + threadIdx.x;
  const i64 dc = min(d, a.nomega - 1);
  const i64 p0 = blockIdx.y * per, p1 = min(p0 + per, a.nt * a.nq);
  const double r[3] = {a.rhat[3 * dc], a.rhat[3 * dc + 1], a.rhat[3 * dc + 2]};
  double acc[FF_ROW];
#pragma unroll
  for (int i = 0; i < FF_ROW; ++i) acc[i] = 0.0;
  for (i64 p = p0; p < p1; ++p) {
    const double* q = a.rq + 3 * p;
    const double* f = F + p * FF_ROW;
    double sn, cs;
    sincos(a.k * (r[0] * q[0] + r[1] * q[1] + r[2] * q[2]), &sn, &cs);
#pragma unroll
    for (int i = 0; i < FF_ROW; i += 2) {
      acc[i] += f[i] * cs - f[i + 1] * sn;
      acc[i + 1] += f[i] * sn + f[i + 1] * cs;
    }
  }
  if (d >= a.nomega) return;
  double u[3], v[3];
  transverse_pair(r, u, v);
#pragma unroll
  for (int c = 0; c < FF_R; ++c) {
    if (c >= R) break;
    const double* s = acc + 6 * c;
    double2* o = part + ((i64)blockIdx.y * R + c) * (2 * a.nomega) + 2 * d;
    // times -i pf
    const double ur = u[0] * s[0] + u[1] * s[2] + u[2] * s[4], ui = u[0] * s[1] + u[1] * s[3] + u[2] * s[5];
    const double vr = v[0] * s[0] + v[1] * s[2] + v[2] * s[4], vi = v[0] * s[1] + v[1] * s[3] + v[2] * s[5];
    o[0] = make_double2(a.pf * ui, -a.pf * ur);
    o[1] = make_double2(a.pf * vi, -a.pf * vr);
  }
}

FfArgs ff_args(const dm_rwg& r, const TriTables& t, const double* rhat, i64 nomega, double k, double eta0) {
  FfArgs a;
  a.n = r.n;
  a.nt = r.mesh->nt;
  a.nomega = nomega;
  a.nq = t.nq;
  a.TB = r.TB;
  a.blk_off = r.d_blk_off.p;
  a.blk_tri = r.d_blk_tri.p;
  a.hrwg = r.d_hrwg.p;
  a.hsig = r.d_hsig.p;
  a.tp = r.d_tplus_i.p;
  a.ext = r.d_ext.p;
  a.len = r.d_len.p;
  a.rq = t.rq.p;
  a.vtx = t.vtx.p;
  a.rhat = rhat;
  a.k = k;
  a.pf = k * eta0 * 0.07957747154594767;
  double xi[14], w[7];
  dmh::quad_rule(t.quad_order, xi, w);
  for (int i = 0; i < 7; ++i) a.w[i] = i < t.nq ? w[i] : 0.0;
  return a;
}

template <int DIRS>
void launch_rad_uv(const FfArgs& a, int nblk, size_t smem, double* G, hipStream_t s) {
  HIP_OK(hipFuncSetAttribute((const void*)k_rad_uv<DIRS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
  const i64 rows = (a.nomega + DIRS - 1) / DIRS;
  DM_REQUIRE(rows <= 65535, DM_ERR_ARGUMENT, "too many directions for one launch");
  k_rad_uv<DIRS><<<dim3((unsigned)nblk, (unsigned)rows), 256, smem, s>>>(a, reinterpret_cast<double2*>(G));
}

}  // namespace

namespace dmf {

// The lines between the routes, whole calls in us, full / transverse / direct
// (n x directions):
//   4 currents   96 x 648 125 / 132 / 146, 280 x 648 159 / 164 / 152,
//                408 x 32 163 / 169 / 145, 1160 x 648 - / 182 / 175,
//                2640 x 468 535 / 195 / 205, 4720 x 162 - / 191 / 233,
//                7701 x 468 1343 / 315 / 288, 7701 x 2592 - / 971 / 418
//   8 currents   96 x 32 175 / 183 / 263, 736 x 576 306 / 253 / 323,
//                1160 x 648 - / 263 / 354, 7701 x 1200 1577 / 636 / 636,
//                4720 x 2160 1159 / 646 / 595, 7701 x 2592 - / 1093 / 848
//   16 currents  176 x 648 358 / 363 / -, 736 x 432 446 / 394 / -,
//                7701 x 2592 - / 1322 / 1618
// Directly, a pass of four currents costs the phases of all points, in waves of 64
// directions that walk 1/256 of the points each: it pays for one pass unless many
// points meet few directions, for two only where the phases dominate.  Up to 512
// bases the product is a single part and the third row costs less than the join.
FfRoute farfield_route(i64 n, i64 nomega, i64 ncur) {
  const double pairs = (double)n * (double)nomega;
  if (ncur <= FF_R && n >= 256 && (n <= 1200 || (nomega >= 256 && pairs >= 1.5e6))) return FfRoute::direct;
  if (ncur <= 2 * FF_R && nomega >= 1024 && pairs >= 1e7) return FfRoute::direct;
  return n < 512 ? FfRoute::full : FfRoute::transverse;
}

// Chunks of points: enough one-wave workgroups to fill the chip (4096), at
// least 32 points each.
static i64 direct_chunks(i64 np, i64 nomega) {
  const i64 gd = (nomega + 63) / 64;
  return std::max<i64>(1, std::min<i64>(std::min<i64>(256, (np + 31) / 32), 4096 / gd));
}

size_t farfield_direct_ws(const dm_rwg& r, const TriTables& t, i64 nomega) {
  const i64 np = r.mesh->nt * t.nq;
  return (size_t)np * FF_ROW + (size_t)direct_chunks(np, nomega) * FF_R * 4 * nomega;
}

// E (3 nomega x R, lde) of R <= FF_R currents (caller order, ldi); ws:
// farfield_direct_ws doubles.
void farfield_few(const dm_rwg& r, const TriTables& t, const double* rhat, i64 nomega, double k, double eta0,
                  const double* I, i64 ldi, int R, double* E, i64 lde, double* ws, hipStream_t s) {
  const FfArgs a = ff_args(r, t, rhat, nomega, k, eta0);
  const i64 np = a.nt * a.nq;
  double* F = ws;
  double2* part = reinterpret_cast<double2*>(ws + np * FF_ROW);
  const unsigned gd = (unsigned)((nomega + 63) / 64);
  const i64 want = direct_chunks(np, nomega), per = (np + want - 1) / want;
  const int nk = (int)((np + per - 1) / per);
  k_ff_points<<<(unsigned)((np + 255) / 256), 256, 0, s>>>(a, reinterpret_cast<const double2*>(I), ldi, R, F);
  k_ff_direct<<<dim3(gd, (unsigned)nk), 64, 0, s>>>(a, per, R, F, part);
  k_ff_join<<<(unsigned)((nomega * R + 255) / 256), 256, 0, s>>>(nomega, R, nk, rhat, part,
                                                                 reinterpret_cast<double2*>(E), lde);
  HIP_OK(hipGetLastError());
}

void radiation_uv(const dm_rwg& r, const TriTables& t, const double* rhat, i64 nomega, double k, double eta0,
                  double* G, hipStream_t s) {
  const FfArgs a = ff_args(r, t, rhat, nomega, k, eta0);
  // 16 directions per workgroup while the block's phases fit in half of a CU's
  // LDS (nq = 3: always), 8 beyond
  const size_t row = (size_t)r.max_blk_tris * t.nq * sizeof(double2);
  const size_t vec = (size_t)r.TB * 2 * t.nq * 3 * sizeof(double);
  if (16 * row + vec <= 76 * 1024)
    launch_rad_uv<16>(a, r.nblk, 16 * row + vec, G, s);
  else
    launch_rad_uv<8>(a, r.nblk, 8 * row + vec, G, s);
  HIP_OK(hipGetLastError());
}

void farfield_join(i64 nomega, int R, int nk, const double* rhat, const double* part, double* E, i64 lde,
                   hipStream_t s) {
  k_ff_join<<<(unsigned)((nomega * R + 255) / 256), 256, 0, s>>>(nomega, R, nk, rhat,
                                                                 reinterpret_cast<const double2*>(part),
                                                                 reinterpret_cast<double2*>(E), lde);
  HIP_OK(hipGetLastError());
}

void planewave(const dm_rwg& r, const TriTables& t, const double* kvec, const double* pol, const double* E0, int M,
               const int* out_idx, double* V, i64 ldv, hipStream_t s) {
  PwArgs a;
  a.n = r.n;
  a.nq = t.nq;
  a.M = M;
  a.tp = r.d_tplus_i.p;
  a.tm = r.d_tminus_i.p;
  a.ep = r.d_eplus_i.p;
  a.em = r.d_eminus_i.p;
  a.len = r.d_len.p;
  a.hsig = r.d_hsig.p;
  a.rq = t.rq.p;
  a.vtx = t.vtx.p;
  a.kvec = kvec;
  a.pol = pol;
  a.E0 = E0;
  a.out_idx = out_idx;
  double xi[14], w[7];
  dmh::quad_rule(t.quad_order, xi, w);
  for (int i = 0; i < 7; ++i) a.w[i] = i < t.nq ? w[i] : 0.0;
  i64 total = r.n * M;
  k_planewave<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(a, reinterpret_cast<double2*>(V), ldv);
  HIP_OK(hipGetLastError());
}

void radiation_vectors(const dm_rwg& r, const TriTables& t, const double* rhat, i64 nomega, double k, double eta0,
                       double* G, hipStream_t s) {
  RadArgs a;
  a.n = r.n;
  a.nomega = nomega;
  a.nq = t.nq;
  a.tp = r.d_tplus_i.p;
  a.tm = r.d_tminus_i.p;
  a.ep = r.d_eplus_i.p;
  a.em = r.d_eminus_i.p;
  a.ext = r.d_ext.p;
  a.len = r.d_len.p;
  a.hsig = r.d_hsig.p;
  a.rq = t.rq.p;
  a.vtx = t.vtx.p;
  a.rhat = rhat;
  a.k = k;
  a.eta0 = eta0;
  double xi[14], w[7];
  dmh::quad_rule(t.quad_order, xi, w);
  for (int i = 0; i < 7; ++i) a.w[i] = i < t.nq ? w[i] : 0.0;
  i64 total = r.n * nomega;
  k_radiation<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(a, reinterpret_cast<double2*>(G));
  HIP_OK(hipGetLastError());
}

}  // namespace dmf
