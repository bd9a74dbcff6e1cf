// k_mpnn.hip — forward, backward and Adam kernels of the learned
// preconditioner's message-passing network (layout and equations in k_mpnn.h).
//
// Training products with the samples' matrices A = Z S are small (n up to a
// few thousand): 16 rows per workgroup for A y, four rows per wave for A^H q.
//
// Layers run 64 nodes per workgroup: the layer's two 64 x 64 weight matrices
// (bfloat16 in memory, widened to FP32 in LDS), the nodes' hidden states and
// their aggregated neighbour messages are staged in LDS; each of the 256
// threads produces four outputs of four nodes.  Weight
// gradients are sums of per-node outer products, reduced per workgroup into
// FP32 partials and across workgroups in FP64 (fixed order).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "k_mpnn.h"

namespace {

using dmn::DEG;
using dmn::FIN;
using dmn::H;

constexpr int NT = 64;       // nodes per workgroup
constexpr int HP = H + 1;    // padded LDS row
constexpr int OUTER_G = 256; // workgroups of the outer-product kernels

__device__ inline float bf(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ inline uint16_t to_bf(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ inline double bsum(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
  return t;
}

// one workgroup per sample: c from r, then tau = rms |c z| and den
__global__ __launch_bounds__(256) void k_stats(const int64_t* __restrict__ ptr, int64_t node0,
                                               const double2* __restrict__ z, const double2* __restrict__ r,
                                               double* __restrict__ cden) {
  __shared__ double red[4];
  const int s = blockIdx.x;
  const int64_t a = ptr[s] - node0, b = ptr[s + 1] - node0;
  double r2 = 0, qr = 0, qi = 0, z2 = 0;
  for (int64_t i = a + threadIdx.x; i < b; i += 256) {
    const double2 v = r[i];
    const double m2 = v.x * v.x + v.y * v.y, m = sqrt(m2);
    r2 += m2;
    qr += v.x * m;
    qi += v.y * m;
    const double2 w = z[i];
    z2 += w.x * w.x + w.y * w.y;
  }
  r2 = bsum(r2, red);
  qr = bsum(qr, red);
  qi = bsum(qi, red);
  z2 = bsum(z2, red);
  if (threadIdx.x == 0) {
    double cr = 0, ci = 0;
    const double rho = b > a ? sqrt(r2 / (double)(b - a)) : 0.0;
    if (rho > 0) {
      const double qa = sqrt(qr * qr + qi * qi);
      if (qa > 0) {
        cr = qr / (qa * rho);
        ci = -qi / (qa * rho);
      } else {
        cr = 1.0 / rho;
      }
    }
    const double c2 = cr * cr + ci * ci;
    cden[4 * s] = cr;
    cden[4 * s + 1] = ci;
    cden[4 * s + 2] = c2 * r2;
    cden[4 * s + 3] = b > a ? sqrt(c2 * z2 / (double)(b - a)) : 0.0;
  }
}

__global__ void k_features(i64 n, const int* __restrict__ smp, int s0, const double* __restrict__ cden,
                           const double2* __restrict__ z, const double2* __restrict__ r, const float2* __restrict__ geom,
                           float* __restrict__ u) {
  i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int s = smp[i] - s0;
  const double cr = cden[4 * s], ci = cden[4 * s + 1], tau = cden[4 * s + 3];
  const double it = tau > 0 ? 1.0 / tau : 0.0;
  const double2 zv = z[i], rv = r[i];
  float* ui = u + i * FIN;
  ui[0] = (float)((cr * zv.x - ci * zv.y) * it);
  ui[1] = (float)((cr * zv.y + ci * zv.x) * it);
  ui[2] = (float)(cr * rv.x - ci * rv.y);
  ui[3] = (float)(cr * rv.y + ci * rv.x);
  const float2 g = geom[i];
  ui[4] = g.x;
  ui[5] = g.y;
}

__global__ void k_encode(i64 n, const float* __restrict__ u, const uint16_t* __restrict__ we, float* __restrict__ h) {
  i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx >= n * H) return;
  i64 i = idx / H;
  int o = (int)(idx % H);
  float acc = 0.f;
#pragma unroll
  for (int k = 0; k < FIN; ++k) acc += bf(we[o * FIN + k]) * u[i * FIN + k];
  h[idx] = acc;
}

// The two 64 x 64 matrices of a layer, widened to FP32, transposed to
// [input][output] rows of TP floats (16-byte reads of four outputs).
constexpr int TP = H + 4;
__device__ inline void stage_weights(const uint16_t* __restrict__ prm, float (*ws)[TP], float (*wn)[TP], bool transpose) {
  for (int e = threadIdx.x; e < H * H; e += 256) {
    const int o = e / H, k = e % H;
    const float a = bf(prm[e]), b = bf(prm[H * H + e]);
    if (transpose) {
      ws[k][o] = a;
      wn[k][o] = b;
    } else {
      ws[o][k] = a;
      wn[o][k] = b;
    }
  }
}

// h_out = h + tanh(W_s h + W_n m + b), m_i = dinv_i sum_q sgn_iq h_{nbr_iq}.
// Each thread forms 4 nodes x 4 outputs from 16-byte LDS reads (four of the
// weights' outputs, one value of each node: 10 reads for 32 FMAs), so the FMAs
// and not the LDS pipe bound it: 30 us for 46 000 nodes (a node x 16 outputs
// per thread read LDS once per FMA, and the missing neighbours' branches kept
// the loads from overlapping: 50 us).
__global__ __launch_bounds__(256) void k_layer(i64 n, i64 gnode0, const int* __restrict__ nbr,
                                               const float* __restrict__ sgn, const float* __restrict__ dinv,
                                               const float* __restrict__ hin, const uint16_t* __restrict__ prm,
                                               float* __restrict__ hout, float* __restrict__ tcache,
                                               float* __restrict__ mcache) {
  __shared__ __align__(16) float Ws[H][TP], Wn[H][TP];
  __shared__ float bs[H];
  __shared__ float hs[NT][HP], ms[NT][HP];
  const int tid = threadIdx.x;
  const i64 i0 = (i64)blockIdx.x * NT;
  stage_weights(prm, Ws, Wn, true);
  if (tid < H) bs[tid] = bf(prm[2 * H * H + tid]);
#pragma unroll 4
  for (int e = tid; e < NT * H; e += 256) {
    const int nd = e / H, k = e % H;
    const i64 gi = min(i0 + nd, n - 1);
    const float hv = hin[gi * H + k];
    float mv = 0.f;
    // every neighbour is read (a missing one as the node itself, weight 0)
#pragma unroll
    for (int q = 0; q < DEG; ++q) {
      const int j = nbr[gi * DEG + q];
      const float w = j >= 0 ? sgn[gi * DEG + q] : 0.f;
      mv += w * hin[(j >= 0 ? (i64)j - gnode0 : gi) * H + k];
    }
    hs[nd][k] = hv;
    ms[nd][k] = mv * dinv[gi];
  }
  __syncthreads();
  const int n0 = (tid >> 4) * 4, o0 = (tid & 15) * 4;
  float acc[4][4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[r][j] = bs[o0 + j];
#pragma unroll 4
  for (int k = 0; k < H; ++k) {
    const float4 w = *reinterpret_cast<const float4*>(&Ws[k][o0]), v = *reinterpret_cast<const float4*>(&Wn[k][o0]);
    const float wj[4] = {w.x, w.y, w.z, w.w}, vj[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float hk = hs[n0 + r][k], mk = ms[n0 + r][k];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[r][j] += wj[j] * hk + vj[j] * mk;
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const i64 gi = i0 + n0 + r;
    if (gi >= n) continue;
    float t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j] = tanhf(acc[r][j]);
    *reinterpret_cast<float4*>(hout + gi * H + o0) = make_float4(
        hs[n0 + r][o0] + t[0], hs[n0 + r][o0 + 1] + t[1], hs[n0 + r][o0 + 2] + t[2], hs[n0 + r][o0 + 3] + t[3]);
    if (tcache) *reinterpret_cast<float4*>(tcache + gi * H + o0) = make_float4(t[0], t[1], t[2], t[3]);
    if (mcache)
      *reinterpret_cast<float4*>(mcache + gi * H + o0) =
          make_float4(ms[n0 + r][o0], ms[n0 + r][o0 + 1], ms[n0 + r][o0 + 2], ms[n0 + r][o0 + 3]);
  }
}

__global__ void k_decode(i64 n, const float* __restrict__ h, const uint16_t* __restrict__ wd, float* __restrict__ y) {
  i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (i >= n) return;
  float a = 0.f, b = 0.f;
  for (int k = 0; k < H; ++k) {
    float hv = h[i * H + k];
    a += bf(wd[k]) * hv;
    b += bf(wd[H + k]) * hv;
  }
  y[2 * i] = a;
  y[2 * i + 1] = b;
}

__global__ __launch_bounds__(1024) void k_sum(i64 n, const double* __restrict__ v, double* __restrict__ out) {
  __shared__ double red[16];
  double s = 0;
  for (i64 i = threadIdx.x; i < n; i += 1024) s += v[i];
  s = bsum(s, red);
  if (threadIdx.x == 0) out[0] = s;
}

// gh = W_d^T gy
__global__ void k_decode_back(i64 n, const float2* __restrict__ gy, const uint16_t* __restrict__ wd,
                              float* __restrict__ gh) {
  i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx >= n * H) return;
  i64 i = idx / H;
  int k = (int)(idx % H);
  float2 g = gy[i];
  gh[idx] = bf(wd[k]) * g.x + bf(wd[H + k]) * g.y;
}

// ga = gh (1 - t^2); gh_out = gh + W_s^T ga; gm = dinv W_n^T ga (tiles as in
// k_layer)
__global__ __launch_bounds__(256) void k_layer_back(i64 n, const float* __restrict__ gh, const float* __restrict__ t,
                                                    const float* __restrict__ dinv, const uint16_t* __restrict__ prm,
                                                    float* __restrict__ gh_out, float* __restrict__ gm) {
  __shared__ __align__(16) float Ws[H][TP], Wn[H][TP];
  __shared__ float gas[NT][HP];
  const int tid = threadIdx.x;
  const i64 i0 = (i64)blockIdx.x * NT;
  stage_weights(prm, Ws, Wn, false);
#pragma unroll 4
  for (int e = tid; e < NT * H; e += 256) {
    const int nd = e / H, o = e % H;
    const i64 at = min(i0 + nd, n - 1) * H + o;
    const float tt = t[at];
    gas[nd][o] = gh[at] * (1.f - tt * tt);
  }
  __syncthreads();
  const int n0 = (tid >> 4) * 4, k0 = (tid & 15) * 4;
  float as[4][4], an[4][4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int j = 0; j < 4; ++j) as[r][j] = an[r][j] = 0.f;
#pragma unroll 4
  for (int o = 0; o < H; ++o) {
    const float4 w = *reinterpret_cast<const float4*>(&Ws[o][k0]), v = *reinterpret_cast<const float4*>(&Wn[o][k0]);
    const float wj[4] = {w.x, w.y, w.z, w.w}, vj[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float g = gas[n0 + r][o];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        as[r][j] += wj[j] * g;
        an[r][j] += vj[j] * g;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const i64 gi = i0 + n0 + r;
    if (gi >= n) continue;
    const float di = dinv[gi];
    const float4 g = *reinterpret_cast<const float4*>(gh + gi * H + k0);
    *reinterpret_cast<float4*>(gh_out + gi * H + k0) =
        make_float4(g.x + as[r][0], g.y + as[r][1], g.z + as[r][2], g.w + as[r][3]);
    *reinterpret_cast<float4*>(gm + gi * H + k0) =
        make_float4(an[r][0] * di, an[r][1] * di, an[r][2] * di, an[r][3] * di);
  }
}

// gh_out_j += sum_q sgn_jq gm_{nbr_jq}  (adjoint of the aggregation; the graph is symmetric)
__global__ void k_scatter(i64 n, i64 gnode0, const int* __restrict__ nbr, const float* __restrict__ sgn,
                          const float* __restrict__ gm, float* __restrict__ gh_out) {
  i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx >= n * H) return;
  i64 i = idx / H;
  int k = (int)(idx % H);
  float acc = 0.f;
#pragma unroll
  for (int q = 0; q < DEG; ++q) {
    int j = nbr[i * DEG + q];
    if (j >= 0) acc += sgn[i * DEG + q] * gm[(i64)(j - gnode0) * H + k];
  }
  gh_out[idx] += acc;
}

// part[b][a * KB + c] = sum over this workgroup's nodes of A[i][a] B[i][c]
template <int LA, int KB>
__global__ __launch_bounds__(256) void k_outer(i64 n, const float* __restrict__ A, const float* __restrict__ B,
                                               float* __restrict__ part) {
  constexpr int KB1 = KB + 1;  // padded rows
  constexpr int O = LA * KB;
  constexpr int PER = (O + 255) / 256;
  __shared__ float As[NT * LA];
  __shared__ float Bs[NT * KB1];
  const int tid = threadIdx.x;
  float acc[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) acc[j] = 0.f;
  const i64 ntile = (n + NT - 1) / NT;
  for (i64 tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const i64 i0 = tile * NT;
    __syncthreads();
    for (int e = tid; e < NT * LA; e += 256) {
      int nd = e / LA, a = e % LA;
      i64 gi = i0 + nd;
      As[nd * LA + a] = gi < n ? A[gi * LA + a] : 0.f;
    }
    for (int e = tid; e < NT * KB; e += 256) {
      int nd = e / KB, c = e % KB;
      i64 gi = i0 + nd;
      Bs[nd * KB1 + c] = gi < n ? B[gi * KB + c] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int o = tid + 256 * j;
      if (o < O) {
        const int a = o / KB, c = o % KB;
        float s = 0.f;
        for (int nd = 0; nd < NT; ++nd) s += As[nd * LA + a] * Bs[nd * KB1 + c];
        acc[j] += s;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int o = tid + 256 * j;
    if (o < O) part[(i64)blockIdx.x * O + o] = acc[j];
  }
}

// The H x H form for up to two right factors that share the left one (the
// layer's inputs and its messages): 4 x 4 sums per thread and factor from
// 16-byte LDS reads; the bias sums ride with the first factor.  Reading one
// value of each factor per FMA, and the left factor once per right factor,
// took 2 x 22 us for 46 000 nodes; this takes 11 us.
__global__ __launch_bounds__(256) void k_outer_pair(i64 n, const float* __restrict__ A, const float* __restrict__ T,
                                                    const float* __restrict__ B0, const float* __restrict__ B1,
                                                    float* __restrict__ part) {
  constexpr int O = H * (H + 1);
  __shared__ __align__(16) float As[NT][TP], Bs[2][NT][TP];
  const int tid = threadIdx.x;
  const int a0 = (tid >> 4) * 4, c0 = (tid & 15) * 4;
  float acc[2][4][4], bias = 0.f;
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[f][i][j] = 0.f;
  const i64 ntile = (n + NT - 1) / NT;
  for (i64 tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const i64 i0 = tile * NT;
    __syncthreads();
#pragma unroll 4
    for (int e = tid; e < NT * H / 4; e += 256) {
      const int nd = e / (H / 4), c = e % (H / 4) * 4;
      const i64 at = min(i0 + nd, n - 1) * H + c;
      float4 a = *reinterpret_cast<const float4*>(A + at);
      const float4 t = *reinterpret_cast<const float4*>(T + at);
      a = make_float4(a.x * (1.f - t.x * t.x), a.y * (1.f - t.y * t.y), a.z * (1.f - t.z * t.z),
                      a.w * (1.f - t.w * t.w));
      if (i0 + nd >= n) a = make_float4(0.f, 0.f, 0.f, 0.f);
      *reinterpret_cast<float4*>(&As[nd][c]) = a;
      *reinterpret_cast<float4*>(&Bs[0][nd][c]) = *reinterpret_cast<const float4*>(B0 + at);
      *reinterpret_cast<float4*>(&Bs[1][nd][c]) = *reinterpret_cast<const float4*>(B1 + at);
    }
    __syncthreads();
    float s[2][4][4];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) s[f][i][j] = 0.f;
#pragma unroll 2
    for (int nd = 0; nd < NT; ++nd) {
      const float4 a = *reinterpret_cast<const float4*>(&As[nd][a0]);
      const float ai[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const float4 b = *reinterpret_cast<const float4*>(&Bs[f][nd][c0]);
        const float bj[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) s[f][i][j] += ai[i] * bj[j];
      }
    }
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[f][i][j] += s[f][i][j];
    if (tid < H) {
      float sb = 0.f;
      for (int nd = 0; nd < NT; ++nd) sb += As[nd][tid];
      bias += sb;
    }
  }
  // factor f's partials of workgroup b at (f gridDim.x + b) O
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    float* p = part + ((i64)f * gridDim.x + blockIdx.x) * O;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) p[(a0 + i) * (H + 1) + c0 + j] = acc[f][i][j];
    if (f == 0 && tid < H) p[tid * (H + 1) + H] = bias;
  }
}

// grad[woff + a * KB + c] (c < KB), grad[boff + a] (c == KB, bias) from G
// partials of LA rows of KB1 values (KB, or KB + 1 with a bias column): the four
// waves of a workgroup take the partials b = wave mod 4 of 64 sums, then their
// FP64 sums are added in order.
__global__ __launch_bounds__(256) void k_outer_reduce(int G, int LA, int KB, int KB1, int bias,
                                                      const float* __restrict__ part, float* __restrict__ grad,
                                                      int woff, int boff) {
  __shared__ double red[4][64];
  const int O = LA * KB1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int o = blockIdx.x * 64 + lane;
  double s = 0;
#pragma unroll 8
  for (int b = wave; b < G; b += 4) s += part[(i64)b * O + min(o, O - 1)];
  red[wave][lane] = s;
  __syncthreads();
  if (wave != 0 || o >= O) return;
  const int a = o / KB1, c = o % KB1;
  if (c == KB && !bias) return;
  s = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
  if (c < KB)
    grad[woff + a * KB + c] = (float)s;
  else
    grad[boff + a] = (float)s;
}

__global__ void k_adam(int np, float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, float b1t, float b2t, float lr, uint16_t* __restrict__ bf16) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  float gi = g[i];
  float mi = b1 * m[i] + (1.f - b1) * gi;
  float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  float mh = mi / (1.f - b1t), vh = vi / (1.f - b2t);
  float pi = p[i] - lr * mh / (sqrtf(vh) + eps);
  p[i] = pi;
  bf16[i] = to_bf(pi);
}

__global__ void k_to_bf16(int np, const float* __restrict__ p, uint16_t* __restrict__ bf16) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < np) bf16[i] = to_bf(p[i]);
}

// d = (y0 + i y1) / c = (y0 + i y1) conj(c) / |c|^2
__global__ void k_correction(i64 n, const float2* __restrict__ y, const double* __restrict__ cden,
                             double2* __restrict__ d) {
  i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double cr = cden[0], ci = cden[1];
  const double c2 = cr * cr + ci * ci;
  if (!(c2 > 0)) {
    d[i] = make_double2(0.0, 0.0);
    return;
  }
  const float2 yv = y[i];
  d[i] = make_double2(((double)yv.x * cr + (double)yv.y * ci) / c2, ((double)yv.y * cr - (double)yv.x * ci) / c2);
}

__global__ void k_identity(i64 n, double2* __restrict__ out) {
  const i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx < n * n) out[idx] = make_double2(idx % n == idx / n ? 1.0 : 0.0, 0.0);
}

__global__ void k_add(i64 n, const double2* __restrict__ a, const double2* __restrict__ b, double2* __restrict__ out) {
  i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (i < n) out[i] = make_double2(a[i].x + b[i].x, a[i].y + b[i].y);
}

// out[:, c] = A x[:, c] for c < k, FP64 sums: 16 rows per workgroup, its 16
// waves and the four 16-lane groups of a wave over the columns j of A (64 at a
// time, 128 contiguous bytes of A per group), the 64 partial sums of a row
// added in a fixed order.  Bound by FP64 issue and L2 latency: 25 us for n =
// 1278, k = 6 (a row per thread left all but five CUs idle: 1.13 ms).
constexpr int AC_ROWS = 16, AC_WAVES = 16;
template <int KMAX, class TX>
__global__ __launch_bounds__(64 * AC_WAVES) void k_acols(i64 n, int k, const float2* __restrict__ A,
                                                         const TX* __restrict__ x, double2* __restrict__ out) {
  __shared__ double2 part[AC_WAVES][KMAX][AC_ROWS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane & (AC_ROWS - 1);
  const i64 i0 = blockIdx.x * (i64)AC_ROWS, i = min(i0 + row, n - 1);
  double ar[KMAX], ai[KMAX];
#pragma unroll
  for (int c = 0; c < KMAX; ++c) ar[c] = ai[c] = 0.0;
#pragma unroll 2
  for (i64 j = 4 * wave + lane / AC_ROWS; j < n; j += 4 * AC_WAVES) {
    const float2 af = A[i + j * n];
    const double zr = af.x, zi = af.y;
    TX xv[KMAX];
#pragma unroll
    for (int c = 0; c < KMAX; ++c) xv[c] = x[j + min(c, k - 1) * n];  // clamped: no load behind a branch
#pragma unroll
    for (int c = 0; c < KMAX; ++c) {
      const double xr = xv[c].x, xi = xv[c].y;
      ar[c] += zr * xr - zi * xi;
      ai[c] += zr * xi + zi * xr;
    }
  }
#pragma unroll
  for (int c = 0; c < KMAX; ++c) {
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
      ar[c] += __shfl_xor(ar[c], o, 64);
      ai[c] += __shfl_xor(ai[c], o, 64);
    }
    if (lane < AC_ROWS) part[wave][c][row] = make_double2(ar[c], ai[c]);
  }
  __syncthreads();
  if (threadIdx.x < KMAX * AC_ROWS) {
    const int c = threadIdx.x / AC_ROWS, q = threadIdx.x % AC_ROWS;
    double sr = 0, si = 0;
#pragma unroll
    for (int w = 0; w < AC_WAVES; ++w) {
      sr += part[w][c][q].x;
      si += part[w][c][q].y;
    }
    if (c < k && i0 + q < n) out[i0 + q + c * n] = make_double2(sr, si);
  }
}

// out[:, c] = A^H x[:, c] for c < k, FP64 lane sums: four output rows (columns
// of A, read contiguously by the lanes) per wave, which share the reads of x;
// the wave's 2 x 4 KMAX = 64 sums are reduced by one transposing butterfly
// (each step halves the values a lane holds), lane l ends with sum l.
template <int KMAX>
__global__ __launch_bounds__(256) void k_acols_adj(i64 n, int k, const float2* __restrict__ A,
                                                   const float2* __restrict__ x, double2* __restrict__ out) {
  constexpr int AR = 4;
  static_assert(2 * AR * KMAX == 64, "one sum per lane");
  const i64 i0 = (blockIdx.x * (i64)4 + (threadIdx.x >> 6)) * AR;
  const int lane = threadIdx.x & 63;
  if (i0 >= n) return;
  double v[64];  // [row][c][re, im]
#pragma unroll
  for (int q = 0; q < 64; ++q) v[q] = 0.0;
  for (i64 j = lane; j < n; j += 64) {
    float2 af[AR], xv[KMAX];
#pragma unroll
    for (int r = 0; r < AR; ++r) af[r] = A[j + min(i0 + r, n - 1) * n];
#pragma unroll
    for (int c = 0; c < KMAX; ++c) xv[c] = x[j + min(c, k - 1) * n];
#pragma unroll
    for (int r = 0; r < AR; ++r) {
      const double zr = af[r].x, zi = -(double)af[r].y;
#pragma unroll
      for (int c = 0; c < KMAX; ++c) {
        v[2 * (r * KMAX + c)] += zr * xv[c].x - zi * xv[c].y;
        v[2 * (r * KMAX + c) + 1] += zr * xv[c].y + zi * xv[c].x;
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const bool hi = (lane & o) != 0;
#pragma unroll
    for (int q = 0; q < o; ++q) {
      const double send = hi ? v[q] : v[q + o], keep = hi ? v[q + o] : v[q];
      v[q] = keep + __shfl_xor(send, o, 64);
    }
  }
  const double im = __shfl_xor(v[0], 1, 64);
  const int r = lane / (2 * KMAX), c = lane % (2 * KMAX) / 2;
  if ((lane & 1) == 0 && c < k && i0 + r < n) out[i0 + r + c * n] = make_double2(v[0], im);
}

__global__ void k_gather_c64(i64 n, const double2* __restrict__ a, const int* __restrict__ iofe,
                             float2* __restrict__ out) {
  const i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx >= n * n) return;
  const i64 r = idx % n, c = idx / n;
  const double2 v = a[(i64)iofe[r] + (i64)iofe[c] * n];
  out[idx] = make_float2((float)v.x, (float)v.y);
}

// p = r - Ar
__global__ void k_res_rhs(i64 nk, const double2* __restrict__ r, const double2* __restrict__ ar,
                          double2* __restrict__ p) {
  const i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (i >= nk) return;
  p[i] = make_double2(r[i].x - ar[i].x, r[i].y - ar[i].y);
}

// q = Ay - c p, parts = |q|^2 / (den ns)
__global__ void k_res_q(i64 n, int k, const double2* __restrict__ zy, const double2* __restrict__ p,
                        const double* __restrict__ cden, int ns, float2* __restrict__ q, double* __restrict__ parts) {
  const i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx >= n * k) return;
  const int c = (int)(idx / n);
  const double cr = cden[4 * c], ci = cden[4 * c + 1], den = cden[4 * c + 2];
  const double2 pv = p[idx], v = zy[idx];
  const double qr = v.x - (cr * pv.x - ci * pv.y), qi = v.y - (cr * pv.y + ci * pv.x);
  q[idx] = make_float2((float)qr, (float)qi);
  parts[idx] = den > 0 ? (qr * qr + qi * qi) / den / ns : 0.0;
}

// gy = 2 A^H q / (den ns)
__global__ void k_res_gy(i64 n, int k, const double2* __restrict__ g, const double* __restrict__ cden, int ns,
                         float2* __restrict__ gy) {
  const i64 idx = blockIdx.x * (i64)blockDim.x + threadIdx.x;
  if (idx >= n * k) return;
  const double den = cden[4 * (idx / n) + 2];
  const double f = den > 0 ? 2.0 / den / ns : 0.0;
  gy[idx] = make_float2((float)(f * g[idx].x), (float)(f * g[idx].y));
}

unsigned nb256(i64 n) { return (unsigned)((n + 255) / 256); }

constexpr int ZC_K = 8;  // columns per pass of the small products

template <class TX>
void acols(i64 n, int k, const float* A, const TX* x, double* out, hipStream_t s) {
  for (int c0 = 0; c0 < k; c0 += ZC_K) {
    const int kk = std::min(ZC_K, k - c0);
    k_acols<ZC_K, TX><<<(unsigned)((n + AC_ROWS - 1) / AC_ROWS), 64 * AC_WAVES, 0, s>>>(n, kk, reinterpret_cast<const float2*>(A), x + (i64)c0 * n,
                                               reinterpret_cast<double2*>(out) + (i64)c0 * n);
  }
}

void acols_adj(i64 n, int k, const float* A, const float2* x, double* out, hipStream_t s) {
  for (int c0 = 0; c0 < k; c0 += ZC_K) {
    const int kk = std::min(ZC_K, k - c0);
    k_acols_adj<ZC_K><<<(unsigned)((n + 15) / 16), 256, 0, s>>>(n, kk, reinterpret_cast<const float2*>(A),
                                                              x + (i64)c0 * n,
                                                              reinterpret_cast<double2*>(out) + (i64)c0 * n);
  }
}

template <int LA, int KB>
void outer(i64 n, const float* A, const float* B, float* part, float* grad, int woff, hipStream_t s) {
  const int G = (int)std::min<i64>(OUTER_G, std::max<i64>(1, (n + NT - 1) / NT));
  k_outer<LA, KB><<<G, 256, 0, s>>>(n, A, B, part);
  k_outer_reduce<<<(LA * KB + 63) / 64, 256, 0, s>>>(G, LA, KB, KB, 0, part, grad, woff, 0);
}

// weight and bias gradients of one layer: left factor gh (1 - t^2), right
// factors the layer's inputs hin and messages ml
void outer_layer(i64 n, const float* gh, const float* t, const float* hin, const float* ml, float* part, float* grad,
                 int ws, int bo, int wn, hipStream_t s) {
  const int G = (int)std::min<i64>(OUTER_G, std::max<i64>(1, (n + NT - 1) / NT));
  constexpr int O = H * (H + 1);
  k_outer_pair<<<G, 256, 0, s>>>(n, gh, t, hin, ml, part);
  k_outer_reduce<<<(O + 63) / 64, 256, 0, s>>>(G, H, H, H + 1, 1, part, grad, ws, bo);
  k_outer_reduce<<<(O + 63) / 64, 256, 0, s>>>(G, H, H, H + 1, 0, part + (size_t)G * O, grad, wn, 0);
}

}  // namespace

namespace dmn {

void stats(int ns, const int64_t* ptr, int64_t node0, const double* z, const double* r, double* cden, hipStream_t s) {
  if (ns <= 0) return;
  k_stats<<<ns, 256, 0, s>>>(ptr, node0, reinterpret_cast<const double2*>(z), reinterpret_cast<const double2*>(r),
                             cden);
  HIP_OK(hipGetLastError());
}

void features(i64 n, const int* smp, int s0, const double* cden, const double* z, const double* r, const float* geom,
              float* u, hipStream_t s) {
  k_features<<<nb256(n), 256, 0, s>>>(n, smp, s0, cden, reinterpret_cast<const double2*>(z),
                                      reinterpret_cast<const double2*>(r), reinterpret_cast<const float2*>(geom), u);
  HIP_OK(hipGetLastError());
}

void forward(const Graph& g, i64 gnode0, const uint16_t* prm, const Cache& c, float* hbuf, hipStream_t s) {
  const i64 n = g.n;
  // training keeps every layer's input in c.h; inference ping-pongs between
  // c.h (layers 0, 2, 4) and hbuf (layers 1, 3)
  auto hl = [&](int l) -> float* {
    if (c.t) return c.h + (i64)l * n * H;
    return (l & 1) ? hbuf : c.h;
  };
  k_encode<<<nb256(n * H), 256, 0, s>>>(n, c.u, prm + OFF_WE, hl(0));
  const unsigned gl = (unsigned)((n + NT - 1) / NT);
  for (int l = 0; l < L; ++l) {
    k_layer<<<gl, 256, 0, s>>>(n, gnode0, g.nbr, g.sgn, g.dinv, hl(l), prm + off_ws(l), hl(l + 1),
                               c.t ? c.t + (i64)l * n * H : nullptr, c.m ? c.m + (i64)l * n * H : nullptr);
  }
  k_decode<<<nb256(n), 256, 0, s>>>(n, hl(L), prm + OFF_WD, c.y);
  HIP_OK(hipGetLastError());
}

void sum(i64 n, const double* parts, double* out, hipStream_t s) {
  k_sum<<<1, 1024, 0, s>>>(n, parts, out);
  HIP_OK(hipGetLastError());
}

size_t backward_floats(i64 n) { return (size_t)3 * n * H; }
size_t outer_floats() { return (size_t)2 * OUTER_G * H * (H + 1); }

void backward(const Graph& g, i64 gnode0, const uint16_t* prm, const Cache& c, const float* gy, float* grad,
              float* work, float* part, hipStream_t s) {
  const i64 n = g.n;
  float* gh = work;
  float* gh2 = work + n * H;
  float* gm = work + 2 * n * H;
  outer<2, H>(n, gy, c.h + (i64)L * n * H, part, grad, OFF_WD, s);
  k_decode_back<<<nb256(n * H), 256, 0, s>>>(n, reinterpret_cast<const float2*>(gy), prm + OFF_WD, gh);
  const unsigned gl = (unsigned)((n + NT - 1) / NT);
  for (int l = L - 1; l >= 0; --l) {
    const float* hin = c.h + (i64)l * n * H;
    const float* tl = c.t + (i64)l * n * H;
    const float* ml = c.m + (i64)l * n * H;
    outer_layer(n, gh, tl, hin, ml, part, grad, off_ws(l), off_b(l), off_wn(l), s);
    k_layer_back<<<gl, 256, 0, s>>>(n, gh, tl, g.dinv, prm + off_ws(l), gh2, gm);
    k_scatter<<<nb256(n * H), 256, 0, s>>>(n, gnode0, g.nbr, g.sgn, gm, gh2);
    std::swap(gh, gh2);
  }
  outer<H, FIN>(n, gh, c.u, part, grad, OFF_WE, s);
  HIP_OK(hipGetLastError());
}

void adam(float* p, const float* grad, float* m, float* v, int step, float lr, uint16_t* bf16, hipStream_t s) {
  const float b1t = powf(0.9f, (float)step), b2t = powf(0.999f, (float)step);
  k_adam<<<(NPARAM + 255) / 256, 256, 0, s>>>(NPARAM, p, grad, m, v, b1t, b2t, lr, bf16);
  HIP_OK(hipGetLastError());
}

void to_bf16(const float* p, uint16_t* bf16, hipStream_t s) {
  k_to_bf16<<<(NPARAM + 255) / 256, 256, 0, s>>>(NPARAM, p, bf16);
  HIP_OK(hipGetLastError());
}

void gather_c64(i64 n, const double* a_int, const int* iofe, float* out, hipStream_t s) {
  k_gather_c64<<<nb256(n * n), 256, 0, s>>>(n, reinterpret_cast<const double2*>(a_int), iofe,
                                            reinterpret_cast<float2*>(out));
  HIP_OK(hipGetLastError());
}

void res_rhs(i64 n, int k, const float* A, const double* r, double* p, hipStream_t s) {
  // A r into p, then p = r - p
  acols(n, k, A, reinterpret_cast<const double2*>(r), p, s);
  k_res_rhs<<<nb256(n * k), 256, 0, s>>>(n * k, reinterpret_cast<const double2*>(r),
                                         reinterpret_cast<const double2*>(p), reinterpret_cast<double2*>(p));
  HIP_OK(hipGetLastError());
}

void res_loss(i64 n, int k, const float* A, const float* y, const double* p, const double* cden, int ns, float* q,
              double* parts, float* gy, double* work, hipStream_t s) {
  acols(n, k, A, reinterpret_cast<const float2*>(y), work, s);
  k_res_q<<<nb256(n * k), 256, 0, s>>>(n, k, reinterpret_cast<const double2*>(work),
                                       reinterpret_cast<const double2*>(p), cden, ns, reinterpret_cast<float2*>(q),
                                       parts);
  if (gy) {
    acols_adj(n, k, A, reinterpret_cast<const float2*>(q), work, s);
    k_res_gy<<<nb256(n * k), 256, 0, s>>>(n, k, reinterpret_cast<const double2*>(work), cden, ns,
                                          reinterpret_cast<float2*>(gy));
  }
  HIP_OK(hipGetLastError());
}

void correction(i64 n, const float* y, const double* cden, double* d, hipStream_t s) {
  k_correction<<<nb256(n), 256, 0, s>>>(n, reinterpret_cast<const float2*>(y), cden, reinterpret_cast<double2*>(d));
  HIP_OK(hipGetLastError());
}

void identity(i64 n, double* out, hipStream_t s) {
  k_identity<<<nb256(n * n), 256, 0, s>>>(n, reinterpret_cast<double2*>(out));
  HIP_OK(hipGetLastError());
}

void add(i64 n, const double* a, const double* b, double* out, hipStream_t s) {
  k_add<<<nb256(n), 256, 0, s>>>(n, reinterpret_cast<const double2*>(a), reinterpret_cast<const double2*>(b),
                                 reinterpret_cast<double2*>(out));
  HIP_OK(hipGetLastError());
}

}  // namespace dmn
