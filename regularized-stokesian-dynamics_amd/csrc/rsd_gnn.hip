// rsd_gnn.hip -- the learned preconditioner of the iterative resistance route:
// the pair bases it weights, the graph network's forward and backward passes,
// its loss and Adam.  The model and the correction it builds are described in
// rsd_gnn.h.
//
//   kblocks_kernel     K's 11x11 blocks on the lubrication structure: a
//                      particle's rows of R_lub times M on the FP64 matrix
//                      cores, a wave per 16 columns
//   pair_basis_kernel  the inverse of each pair's 22x22 block by Gauss-Jordan
//                      (FP64), half a wave per pair, a lane per row
//   gnn_layer_fwd      one workgroup per particle, a lane per hidden unit, four
//                      waves of four edges each
//   gnn_bwd            the layers backwards, one workgroup per particle; the
//                      contributions a particle receives as a neighbour are
//                      gathered through the reverse slots (no atomics: the
//                      gradients are reproducible)
//   gnn_wgrad          the gradients of all weights from sums per particle,
//                      split over chunks of particles, summed in a fixed order
#include <hip/hip_runtime.h>

#include <cmath>
#include <random>
#include <vector>

#include "rsd_gnn.h"
#include "rsd_step.h"

namespace rsd {

namespace {

__device__ __forceinline__ int gdof(int N, int g, int c) {
  return c < 3 ? 3 * g + c : (c < 6 ? 3 * N + 3 * g + (c - 3) : 6 * N + 5 * g + (c - 6));
}

// ------------------------------------------------------------ pair bases
// Rows r < 6 of K's block (g, d): delta_gd + sum_e R_lub(g, e) M(e, d) over
// e = g and its neighbours; rows r >= 6: M's.  For all of a particle's slots
// that is one product, (6 x 11(nn+1)) times (11(nn+1) x 11(nn+1)), whose right
// factor is gathered from M.  It is bound by that gather (25 neighbours: 600 KB
// a particle in pieces of 24 and 40 bytes): each element is loaded once, by the
// lane that feeds it to the matrix core, kAhead loads a lane in flight.  The
// workgroup per slot whose threads walked the neighbours one after the other
// loaded each element six times: 227 -> 92 us at N = 256 (17 neighbours a
// particle), 5.6 TB/s of the 128-byte lines touched.
constexpr int kKbChunk = 24 * 11;  // rows of M per LDS pass
typedef double v4d __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void kblocks_kernel(LubBsr<double> L, const double* __restrict__ M, int ld,
                                                      double* __restrict__ kb) {
  constexpr int kAhead = 6;
  static_assert(kKbChunk % (4 * kAhead) == 0, "whole groups of steps");
  __shared__ double As[kKbChunk * 6];
  __shared__ int row[kKbChunk];
  const int g = blockIdx.x, t = threadIdx.x, N = L.N, nn = L.nnb[g], K = 11 * (nn + 1);
  const int lane = t & 63, wave = t >> 6;
  if ((int)blockIdx.y * 64 >= K) return;
  const int* cols = L.col + (size_t)g * L.cap;
  const int c0 = (blockIdx.y * 4 + wave) * 16 + (lane & 15);  // this lane's column
  const int cc = min(c0, K - 1), slot = cc / 11, c = cc - 11 * slot;
  const int d = slot == 0 ? g : cols[slot - 1];
  const double* Mc = M + (size_t)gdof(N, d, c) * ld;
  v4d acc = {0.0, 0.0, 0.0, 0.0};
  const int kr = lane >> 4, ar = lane & 15;
  for (int k0 = 0; k0 < K; k0 += kKbChunk) {
    __syncthreads();
    for (int k = t; k < kKbChunk; k += 256) {
      const int kk = min(k0 + k, K - 1), sl = kk / 11;
      row[k] = gdof(N, sl == 0 ? g : cols[sl - 1], kk - 11 * sl);
    }
    for (int u = t; u < kKbChunk * 6; u += 256) {
      const int k = u / 6, r = u - 6 * k, kk = k0 + k, sl = kk / 11;
      As[u] = kk >= K ? 0.0
              : sl == 0 ? L.self[121 * (size_t)g + r + 11 * kk]
                        : L.blk[121 * ((size_t)g * L.cap + sl - 1) + r + 11 * (kk - 11 * sl)];
    }
    __syncthreads();
    const int kn = min(K - k0, kKbChunk);
    for (int k = 0; k < kn; k += 4 * kAhead) {
      double b[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) b[u] = Mc[row[k + 4 * u + kr]];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const double a = ar < 6 ? As[(k + 4 * u + kr) * 6 + ar] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b[u], acc, 0, 0, 0);
      }
    }
  }
  if (c0 >= K) return;
  // lane (kr, ar): rows kr and 4 + kr (kr < 2) of the product; M's rows 6 ..
  double* out = kb + ((size_t)g * (L.cap + 1) + slot) * 121 + 11 * c;
  out[kr] = acc[0] + (slot == 0 && kr == c ? 1.0 : 0.0);
  if (kr < 2) out[4 + kr] = acc[1] + (slot == 0 && 4 + kr == c ? 1.0 : 0.0);
  out[6 + kr] = Mc[gdof(N, g, 6 + kr)];
  if (kr == 0) out[10] = Mc[gdof(N, g, 10)];
}

__global__ void rev_kernel(LubBsr<double> L, int* __restrict__ rev) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long long)L.N * L.cap) return;
  const int g = (int)(e / L.cap), q = (int)(e % L.cap);
  if (q >= L.nnb[g]) return;
  const int d = L.col[e];
  int found = -1;
  for (int k = 0; k < L.nnb[d]; ++k)
    if (L.col[(size_t)d * L.cap + k] == g) {
      found = k;
      break;
    }
  rev[e] = found;
}

// inv([K_gg K_gd; K_dg K_dd]) by Gauss-Jordan with partial pivoting; the
// slot's A - D_g and B out.
// 22 dependent steps of little work: what bounds it is the latency of a step,
// so the pairs are many to a compute unit and no step has a barrier.  Half a
// wave holds a pair, lane i its row i in registers; the inverse grows in place
// (step k's slot takes the column of the step's pivot row p_k), rows stay where
// they are (the row of step k is row k of the inverse), and the pivot row goes
// to the other lanes through LDS.  The pivot is the largest entry to 15 bits
// (the key's low bits hold the lane).  The steps are a loop (a row turns by one
// column a step): unrolled they are 32 KB of code.  N = 256: 149 us with a
// workgroup per pair and seven barriers a step, 41 so (50 unrolled).
constexpr int kPbPairs = 8;  // pairs per workgroup
// LDS written by some lanes of a wave, then read by others of the same wave
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
template <int CTRL>
__device__ __forceinline__ unsigned dpp_max(unsigned v) {
  const unsigned o = (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, true);
  return o > v ? o : v;
}
__global__ __launch_bounds__(32 * kPbPairs) void pair_basis_kernel(LubBsr<double> L, const double* __restrict__ kb,
                                                                   const int* __restrict__ rev,
                                                                   const double* __restrict__ dinv,
                                                                   double* __restrict__ pa, double* __restrict__ pb) {
  constexpr int n = 22;
  __shared__ double prow[kPbPairs][24];
  __shared__ double X[kPbPairs][11][n + 1];
  const int half = threadIdx.x >> 5, i = threadIdx.x & 31, cap = L.cap;
  const int g = blockIdx.x, q = blockIdx.y * kPbPairs + half;
  if (q >= L.nnb[g]) return;  // (no barriers below)
  const size_t e = (size_t)g * cap + q;
  const int d = L.col[e], rq = rev[e], cp = cap + 1;
  double a[n];
  {
    const int bi = i / 11, r = i - 11 * bi;
    const double* b0 = bi == 0 ? kb + (size_t)g * cp * 121 + r : kb + ((size_t)d * cp + 1 + max(rq, 0)) * 121 + r;
    const double* b1 = bi == 0 ? kb + ((size_t)g * cp + 1 + q) * 121 + r : kb + (size_t)d * cp * 121 + r;
#pragma unroll
    for (int j = 0; j < 11; ++j) {
      a[j] = i < n && (bi == 0 || rq >= 0) ? b0[11 * j] : 0.0;
      a[11 + j] = i < n ? b1[11 * j] : 0.0;
    }
  }
  int mine = i < n ? -1 : n;  // the step whose pivot this lane's row is
  int pk = 0;                 // lane k: the row of step k
#pragma unroll 1
  for (int k = 0; k < n; ++k) {  // (columns turn with the steps: column k is in a[0])
    const unsigned hi = (unsigned)__double2hiint(a[0]) & 0x7fffffffu;
    unsigned key = mine < 0 ? ((hi & ~31u) | (31u - i)) + 32u : 0u;  // (+32: above a used row's, also where all are 0)
    key = dpp_max<0x128>(key);  // row_ror 8, 4, 2, 1: the largest of 16 lanes
    key = dpp_max<0x124>(key);
    key = dpp_max<0x122>(key);
    key = dpp_max<0x121>(key);
    const unsigned other = (unsigned)__builtin_amdgcn_ds_swizzle((int)key, 0x401f);  // lane ^ 16
    key = other > key ? other : key;
    const int p = 31 - (int)(key & 31u);
    if (i == k) pk = p;
    const double f = a[0];
    if (i == p) {
      const double inv = 1.0 / f;
#pragma unroll
      for (int j = 1; j < n; ++j) a[j - 1] = a[j] * inv;
      a[n - 1] = inv;
#pragma unroll
      for (int j = 0; j < n; ++j) prow[half][j] = a[j];
      mine = k;
    }
    wave_lds_sync();
    if (i != p) {
#pragma unroll
      for (int j = 1; j < n; ++j) a[j - 1] = fma(-f, prow[half][j - 1], a[j]);
      a[n - 1] = -f * prow[half][n - 1];
    }
    wave_lds_sync();
  }
#pragma unroll
  for (int k = 0; k < n; ++k) {
    const int p = __shfl(pk, k, 32);
    if (mine < 11) X[half][mine][p] = a[k];
  }
  wave_lds_sync();
  for (int t = i; t < 121; t += 32) {
    const int r = t % 11, j = t / 11;
    pa[e * 121 + t] = X[half][r][j] - dinv[(size_t)g * 121 + t];
    pb[e * 121 + t] = X[half][r][11 + j];
  }
}

__global__ void features_kernel(LubBsr<double> L, const double* __restrict__ dist, const double* __restrict__ radii,
                                float* __restrict__ feat, float* __restrict__ xn) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long long)L.N * L.cap) return;
  const int g = (int)(e / L.cap), q = (int)(e % L.cap);
  if (q == 0) {
    xn[2 * g] = (float)radii[g];
    xn[2 * g + 1] = (float)L.nnb[g] / 16.0f;
  }
  if (q >= L.nnb[g]) return;
  const int d = L.col[e];
  const double ag = radii[g], ad = radii[d], abar = 0.5 * (ag + ad);
  const double h = (dist[e] - ag - ad) / abar;
  feat[4 * e] = (float)h;
  feat[4 * e + 1] = (float)(0.25 * log(fmax(h, 0.0) + 1e-3));
  feat[4 * e + 2] = (float)ag;
  feat[4 * e + 3] = (float)ad;
}

// -------------------------------------------------------------- forward
__global__ void gnn_input_kernel(int N, const float* __restrict__ P, const float* __restrict__ xn,
                                 float* __restrict__ H0) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= N * kGnnH) return;
  const int g = id / kGnnH, i = id % kGnnH;
  const float* W = P + kGnnOffW0;
  const float pre = P[kGnnOffB0 + i] + W[2 * i] * xn[2 * g] + W[2 * i + 1] * xn[2 * g + 1];
  H0[id] = fmaxf(pre, 0.0f);
}

// One layer forward for one particle: lane i of each wave forms hidden unit i,
// the four waves take four edges each at a time.  What the edges share is done
// once: the part of the pre-activation that h_g gives (64 of 132 terms) and a
// term's read of the weight; per term and edge what is left is a multiply-add
// and a quarter of a broadcast LDS read: 97 us with one wave a particle, 15 so
// (N = 256; 19 with the weights in registers, which spills).  Sums run in the order be,
// h_g, h_d, f, and the edges' in slot order, whatever the split.
constexpr int kFwdEdges = 4;  // edges per wave and pass
__global__ __launch_bounds__(256, 2) void gnn_layer_fwd_kernel(LubBsr<double> L, const float* __restrict__ P, int l,
                                                            const float* __restrict__ feat,
                                                            const float* __restrict__ Hl, float* __restrict__ Hn,
                                                            float* __restrict__ U, float* __restrict__ AGG,
                                                            float* __restrict__ V) {
  constexpr int kIn = kGnnH + kGnnF;  // the edge inputs that differ between edges
  __shared__ float We[kGnnH][kGnnEdgeIn + 1], Wn[kGnnH][kGnnNodeIn + 1];
  __shared__ float4 in[4][kFwdEdges][kIn / 4];
  __shared__ float act[4 * kFwdEdges][kGnnH], nin[kGnnNodeIn];
  const int g = blockIdx.x, t = threadIdx.x, i = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int cap = L.cap, nn = L.nnb[g];
  const int* cols = L.col + (size_t)g * cap;
  const float4* pwe = (const float4*)(P + gnn_off_we(l));
  const float4* pwn = (const float4*)(P + gnn_off_wn(l));
  static_assert(gnn_off_we(0) % 4 == 0 && gnn_off_wn(0) % 4 == 0 && kGnnLayerSize % 4 == 0, "float4 weights");
  for (int k = t; k < kGnnH * kGnnEdgeIn / 4; k += 256) {
    const float4 x = pwe[k];
    float* y = &We[k / (kGnnEdgeIn / 4)][4 * (k % (kGnnEdgeIn / 4))];
    y[0] = x.x, y[1] = x.y, y[2] = x.z, y[3] = x.w;
  }
  for (int k = t; k < kGnnH * kGnnNodeIn / 4; k += 256) {
    const float4 x = pwn[k];
    float* y = &Wn[k / (kGnnNodeIn / 4)][4 * (k % (kGnnNodeIn / 4))];
    y[0] = x.x, y[1] = x.y, y[2] = x.z, y[3] = x.w;
  }
  const float hg = Hl[(size_t)g * kGnnH + i];
  if (w == 0) nin[i] = hg;
  float v0 = P[gnn_off_be(l) + i], u = P[gnn_off_bn(l) + i], agg = 0.0f;
  __syncthreads();
#pragma unroll 8
  for (int j = 0; j < kGnnH; ++j) {
    v0 = fmaf(We[i][j], nin[j], v0);
    u = fmaf(Wn[i][j], nin[j], u);
  }
  for (int q0 = 0; q0 < nn; q0 += 4 * kFwdEdges) {
    const int qw = q0 + kFwdEdges * w;
    if (qw < nn) {
#pragma unroll
      for (int x = 0; x < kFwdEdges; ++x) {
        const int q = min(qw + x, nn - 1);
        float* dst = (float*)in[w][x];
        dst[i] = Hl[(size_t)cols[q] * kGnnH + i];
        if (i < kGnnF) dst[kGnnH + i] = feat[4 * ((size_t)g * cap + q) + i];
      }
    }
    __syncthreads();
    if (qw < nn) {
      float v[kFwdEdges];
#pragma unroll
      for (int x = 0; x < kFwdEdges; ++x) v[x] = v0;
#pragma unroll 4
      for (int j = 0; j < kIn / 4; ++j) {
        const float* we = &We[i][kGnnH + 4 * j];
        const float w0 = we[0], w1 = we[1], w2 = we[2], w3 = we[3];
#pragma unroll
        for (int x = 0; x < kFwdEdges; ++x) {
          const float4 y = in[w][x][j];
          v[x] = fmaf(w0, y.x, v[x]);
          v[x] = fmaf(w1, y.y, v[x]);
          v[x] = fmaf(w2, y.z, v[x]);
          v[x] = fmaf(w3, y.w, v[x]);
        }
      }
#pragma unroll
      for (int x = 0; x < kFwdEdges; ++x) {
        if (qw + x < nn) V[((size_t)g * cap + qw + x) * kGnnH + i] = v[x];
        act[kFwdEdges * w + x][i] = fmaxf(v[x], 0.0f);
      }
    }
    __syncthreads();
    const int n = min(nn - q0, 4 * kFwdEdges);
    for (int x = 0; x < n; ++x) agg += act[x][i];  // each wave its own copy
  }
  agg = nn > 0 ? agg / (float)nn : 0.0f;
  if (w == 0) {
    AGG[(size_t)g * kGnnH + i] = agg;
    nin[kGnnH + i] = agg;
  }
  __syncthreads();
  if (w != 0) return;
#pragma unroll 8
  for (int j = kGnnH; j < kGnnNodeIn; ++j) u = fmaf(Wn[i][j], nin[j], u);
  U[(size_t)g * kGnnH + i] = u;
  Hn[(size_t)g * kGnnH + i] = hg + fmaxf(u, 0.0f);
}

__device__ __forceinline__ double sigmoid(float o) { return 1.0 / (1.0 + exp(-(double)o)); }

// The pair weights' logits of one particle, a thread per slot, and its
// correction blocks, a thread per entry.
__global__ __launch_bounds__(128) void gnn_out_kernel(LubBsr<double> L, const float* __restrict__ P,
                                                      const float* __restrict__ feat, const float* __restrict__ H3,
                                                      const double* __restrict__ pa, const double* __restrict__ pb,
                                                      float* __restrict__ OUT, double* __restrict__ corr) {
  __shared__ float Wo[kGnnEdgeIn], hg[kGnnH];
  __shared__ double ws[128];
  const int g = blockIdx.x, t = threadIdx.x, cap = L.cap, nn = L.nnb[g];
  for (int k = t; k < kGnnEdgeIn; k += 128) Wo[k] = P[kGnnOffWo + k];
  if (t < kGnnH) hg[t] = H3[(size_t)g * kGnnH + t];
  __syncthreads();
  double self = 0.0;
  for (int q0 = 0; q0 < nn; q0 += 128) {
    if (q0 + t < nn) {
      const size_t e = (size_t)g * cap + q0 + t;
      const float4* hd = (const float4*)(H3 + (size_t)L.col[e] * kGnnH);
      float4 x[kGnnH / 4];
#pragma unroll
      for (int j = 0; j < kGnnH / 4; ++j) x[j] = hd[j];
      const float4 f = ((const float4*)feat)[e];
      float o = P[kGnnOffBo];
      for (int j = 0; j < kGnnH; ++j) o = fmaf(Wo[j], hg[j], o);
#pragma unroll
      for (int j = 0; j < kGnnH / 4; ++j) {
        o = fmaf(Wo[kGnnH + 4 * j], x[j].x, o);
        o = fmaf(Wo[kGnnH + 4 * j + 1], x[j].y, o);
        o = fmaf(Wo[kGnnH + 4 * j + 2], x[j].z, o);
        o = fmaf(Wo[kGnnH + 4 * j + 3], x[j].w, o);
      }
      o = fmaf(Wo[2 * kGnnH], f.x, o);
      o = fmaf(Wo[2 * kGnnH + 1], f.y, o);
      o = fmaf(Wo[2 * kGnnH + 2], f.z, o);
      o = fmaf(Wo[2 * kGnnH + 3], f.w, o);
      OUT[e] = o;
      ws[t] = sigmoid(o);
    }
    __syncthreads();
    if (t < 121) {
      const size_t e0 = (size_t)g * cap + q0;
      const int n = min(nn - q0, 128);
#pragma unroll 8
      for (int x = 0; x < n; ++x) {
        const double w = ws[x];
        self = fma(w, pa[(e0 + x) * 121 + t], self);
        corr[((size_t)g * (cap + 1) + 1 + q0 + x) * 121 + t] = w * pb[(e0 + x) * 121 + t];
      }
    }
    __syncthreads();
  }
  if (t < 121) corr[(size_t)g * (cap + 1) * 121 + t] = self;
}

// ------------------------------------------------------------- the loss
// All vectors in one launch each, vector blockIdx.y at stride ld: one after the
// other the loss's products and vector kernels took 330 us for four vectors at
// N = 256, and 100 so.
// r -= z; t = r's rows < 6N, zero below
__global__ void loss_residual_kernel(int n, int n6, size_t ld, const double* __restrict__ z, double* __restrict__ r,
                                     double* __restrict__ t) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t at = blockIdx.y * ld + i;
  const double v = r[at] - z[blockIdx.y * (size_t)n + i];
  r[at] = v;
  t[at] = i < n6 ? v : 0.0;
}
// y += r's rows >= 6N
__global__ void add_q_kernel(int n, int n6, size_t ld, const double* __restrict__ r, double* __restrict__ y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n6 && i < n) y[blockIdx.y * ld + i] += r[blockIdx.y * ld + i];
}
// g += t
__global__ void add_kernel(int n, size_t ld, const double* __restrict__ t, double* __restrict__ g) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) g[blockIdx.y * (size_t)n + i] += t[blockIdx.y * ld + i];
}
// acc[0] = sum |r|^2, acc[1] = sum |z|^2 (one workgroup, fixed-order tree)
__global__ __launch_bounds__(1024) void sumsq2_kernel(int n, int nz, size_t ld, const double* __restrict__ r,
                                                      const double* __restrict__ z, double* __restrict__ acc) {
  __shared__ double s1[1024], s2[1024];
  double a = 0.0, b = 0.0;
  for (int k = 0; k < nz; ++k)
    for (int i = threadIdx.x; i < n; i += 1024) {
      const double rv = r[k * ld + i], zv = z[k * (size_t)n + i];
      a = fma(rv, rv, a);
      b = fma(zv, zv, b);
    }
  s1[threadIdx.x] = a;
  s2[threadIdx.x] = b;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      s1[threadIdx.x] += s1[threadIdx.x + w];
      s2[threadIdx.x] += s2[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    acc[0] = s1[0];
    acc[1] = s2[0];
  }
}

// dL/do per slot (o the pair weight's logit): scale w (1 - w) sum_z G_g^T
// ((A - D) z_g + B z_d).  A wave per slot, two of the 11 x 11 products G_r z_c
// per lane; the sum over z of those with z_g is the same for all slots.
__global__ __launch_bounds__(256) void gnn_dout_kernel(LubBsr<double> L, const double* __restrict__ pa,
                                                       const double* __restrict__ pb, const double* __restrict__ G,
                                                       const double* __restrict__ Z, int nz,
                                                       const double* __restrict__ acc, int log_loss,
                                                       const float* __restrict__ OUT, float* __restrict__ dOUT) {
  const int g = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6, cap = L.cap, nn = L.nnb[g], N = L.N;
  const size_t n = 11 * (size_t)N;
  // d(|r|^2 / |z|^2) = 2 r . dr / |z|^2; of the log, divided by |r|^2 / |z|^2 too
  const double scale = log_loss ? 2.0 / acc[0] : 2.0 / acc[1];
  const int t1 = min(64 + lane, 120);  // (lanes 57 .. 63: no second entry)
  const int r0 = gdof(N, g, lane % 11), r1 = gdof(N, g, t1 % 11), c0 = lane / 11, c1 = t1 / 11;
  const bool two = 64 + lane < 121;
  double y0 = 0.0, y1 = 0.0;
  {
    const int z0 = gdof(N, g, c0), z1 = gdof(N, g, c1);
    for (int z = 0; z < nz; ++z) {
      y0 = fma(G[z * n + r0], Z[z * n + z0], y0);
      y1 = fma(G[z * n + r1], Z[z * n + z1], y1);
    }
  }
  for (int q = w; q < nn; q += 4) {
    const size_t e = (size_t)g * cap + q;
    const int d = L.col[e];
    const int z0 = gdof(N, d, c0), z1 = gdof(N, d, c1);
    double x0 = 0.0, x1 = 0.0;
    for (int z = 0; z < nz; ++z) {
      x0 = fma(G[z * n + r0], Z[z * n + z0], x0);
      x1 = fma(G[z * n + r1], Z[z * n + z1], x1);
    }
    double sum = fma(pa[e * 121 + lane], y0, pb[e * 121 + lane] * x0);
    if (two) sum += fma(pa[e * 121 + t1], y1, pb[e * 121 + t1] * x1);
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_down(sum, o);
    if (lane == 0) {
      const double s = sigmoid(OUT[e]);
      dOUT[e] = (float)(scale * sum * s * (1.0 - s));
    }
  }
}

// ------------------------------------------------------------- backward
// The mean over the edges passes one and the same gradient dm = dagg to all of
// a particle's messages, so dV_e = dagg where V_e > 0: every sum over edges is
// a count (own slots) or a gather (slots where the particle is the neighbour)
// per hidden unit, and each weight matrix is applied once per particle, not
// once per edge.  Kept per layer and particle for the weight gradients:
//   S1 = sum over own slots of dV, S2 = the same over the slots where it is the
//   neighbour, F = sum over own slots of dV f, DU = dU
// (the output layer's: o1, o2, of[4] in DO).
//
// One launch per l = 3 .. 0: dH_l is completed (l = 3: from the output layer;
// else dHp + We_d^T S2 of layer l), then layer l - 1's own-slot part gives S1,
// F, dU and dHp = dH_l + Wn_h^T dU + We_g^T S1; l = 0 ends at the input layer.
// Four waves of 64 units: sums over slots by slot modulo 4, products with
// W^T by 16 rows each (coalesced rows of W, nothing staged).  N = 256: 9 us a
// launch; a product per edge took 107 a layer.  Against 64 bits the gradients'
// error fell by 2 to 8 (counts are exact where the same number was added up).
__device__ __forceinline__ float wave_sum4(float (&red)[4][kGnnH], float x, int w, int i) {
  __syncthreads();
  red[w][i] = x;
  __syncthreads();
  return (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
}
// sum_k W[k][i] x[k] over this wave's 16 rows k
__device__ __forceinline__ float rows16(const float* __restrict__ W, int stride, const float* x, int w, int i) {
  float r = 0.0f;
#pragma unroll
  for (int k = 0; k < 16; ++k) r = fmaf(W[(size_t)(16 * w + k) * stride + i], x[16 * w + k], r);
  return r;
}
struct GnnBwd {
  const float *H, *U, *V, *feat;  // all layers'
  const float* dOUT;
  const int* rev;
  float *S1, *S2, *F, *DU;        // 3 x N x 64 each (F: x 4)
  float *DO, *dagg, *dHp, *dpre0; // 6 N; 2 x N x 64 (by layer's parity); N x 64; N x 64
};
__global__ __launch_bounds__(256) void gnn_bwd_kernel(LubBsr<double> L, const float* __restrict__ P, int l, GnnBwd b) {
  __shared__ float red[4][kGnnH], xs[kGnnH];
  const int g = blockIdx.x, t = threadIdx.x, i = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int N = L.N, cap = L.cap, nn = L.nnb[g];
  const size_t e0 = (size_t)g * cap, gi = (size_t)g * kGnnH + i, NH = (size_t)N * kGnnH;
  float dh;
  if (l == kGnnLayers) {
    float x = 0.0f;  // lane 0: sum dOUT, 1: over the reverse slots, 2 .. 5: dOUT f
    if (i < 6)
      for (int q = w; q < nn; q += 4) {
        const float o = b.dOUT[e0 + q];
        if (i == 0) x += o;
        else if (i == 1) x += b.rev[e0 + q] >= 0 ? b.dOUT[(size_t)L.col[e0 + q] * cap + b.rev[e0 + q]] : 0.0f;
        else x = fmaf(o, b.feat[4 * (e0 + q) + i - 2], x);
      }
    x = wave_sum4(red, x, w, i);
    if (w == 0 && i < 6) b.DO[6 * (size_t)g + i] = x;
    if (w == 0) xs[i] = x;
    __syncthreads();
    dh = fmaf(P[kGnnOffWo + i], xs[0], P[kGnnOffWo + kGnnH + i] * xs[1]);
  } else {
    const float* V = b.V + l * NH * cap;
    const float* da = b.dagg + (l & 1) * NH;
    float s2 = 0.0f;
#pragma unroll 4
    for (int q = w; q < nn; q += 4) {
      const int d = L.col[e0 + q], rq = b.rev[e0 + q];
      if (rq >= 0) {
        const float v = V[((size_t)d * cap + rq) * kGnnH + i], x = da[(size_t)d * kGnnH + i];
        s2 += v > 0.0f ? x : 0.0f;
      }
    }
    s2 = wave_sum4(red, s2, w, i);
    if (w == 0) {
      b.S2[l * NH + gi] = s2;
      xs[i] = s2;
    }
    __syncthreads();
    dh = b.dHp[gi] + wave_sum4(red, rows16(P + gnn_off_we(l) + kGnnH, kGnnEdgeIn, xs, w, i), w, i);
  }
  if (l == 0) {
    if (w == 0) b.dpre0[gi] = b.H[gi] > 0.0f ? dh : 0.0f;
    return;
  }
  const int m = l - 1;
  const float* V = b.V + m * NH * cap;
  const float du = b.U[m * NH + gi] > 0.0f ? dh : 0.0f;
  float cnt = 0.0f, f0 = 0.0f, f1 = 0.0f, f2 = 0.0f, f3 = 0.0f;
#pragma unroll 4
  for (int q = w; q < nn; q += 4) {
    const float4 f = ((const float4*)b.feat)[e0 + q];
    if (V[(e0 + q) * kGnnH + i] > 0.0f) {
      cnt += 1.0f;
      f0 += f.x, f1 += f.y, f2 += f.z, f3 += f.w;
    }
  }
  cnt = wave_sum4(red, cnt, w, i);  // (its first barrier: xs above has been read)
  if (w == 0) xs[i] = du;
  f0 = wave_sum4(red, f0, w, i);    // (its barriers: xs is written)
  f1 = wave_sum4(red, f1, w, i);
  f2 = wave_sum4(red, f2, w, i);
  f3 = wave_sum4(red, f3, w, i);
  const float* Wn = P + gnn_off_wn(m);
  dh += wave_sum4(red, rows16(Wn, kGnnNodeIn, xs, w, i), w, i);
  float dagg = wave_sum4(red, rows16(Wn + kGnnH, kGnnNodeIn, xs, w, i), w, i);
  dagg = nn > 0 ? dagg / (float)nn : 0.0f;
  const float s1 = cnt > 0.0f ? cnt * dagg : 0.0f;
  if (w == 0) {  // (the barriers of the sum above: xs has been read)
    xs[i] = s1;
    b.DU[m * NH + gi] = du;
    b.dagg[(m & 1) * NH + gi] = dagg;
    b.S1[m * NH + gi] = s1;
    const bool any = cnt > 0.0f;
    ((float4*)b.F)[m * NH + gi] = make_float4(any ? f0 * dagg : 0.0f, any ? f1 * dagg : 0.0f, any ? f2 * dagg : 0.0f,
                                              any ? f3 * dagg : 0.0f);
  }
  __syncthreads();
  dh += wave_sum4(red, rows16(P + gnn_off_we(m), kGnnEdgeIn, xs, w, i), w, i);
  if (w == 0) b.dHp[gi] = dh;
}

// The gradients of all weights, partial sums over a chunk of particles: layer
// y < 3: dWe = [S1^T h | S2^T h | sum F], dbe = sum S1, dWn = [dU^T h | dU^T s],
// dbn = sum dU, four 64 x 64 products in 4 x 4 tiles per thread; y = 3: the
// output and the input layer.  (Per edge instead of per particle these are
// nnb times the work: that kernel took 113 us a layer at N = 256.)
constexpr int kGradStage = 8;                             // particles per LDS pass
constexpr int kGradParts = 64;                            // chunks at most ...
constexpr int kPartStride = (kGnnParams + 3) / 4 * 4;
__host__ __device__ inline int grad_chunk(int N) {        // ... of 8 particles at least
  const int c = (N + kGradParts - 1) / kGradParts;
  return c < 8 ? 8 : c;
}
__device__ __forceinline__ void outer4(float (&acc)[4][4], const float4 a, const float4 b) {
  const float x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[r][c] = fmaf(x[r], y[c], acc[r][c]);
}
__global__ __launch_bounds__(256) void gnn_wgrad_kernel(int N, int chunk, GnnBwd b, const float* __restrict__ AGG,
                                                        const float* __restrict__ xn, float* __restrict__ part) {
  const int t = threadIdx.x, y = blockIdx.y;
  const int g0 = blockIdx.x * chunk, g1 = min(N, g0 + chunk);
  const size_t NH = (size_t)N * kGnnH;
  float* out = part + (size_t)blockIdx.x * kPartStride;
  if (y == kGnnLayers) {
    const float* H3 = b.H + kGnnLayers * NH;
    if (t <= 2 * kGnnH + kGnnF) {  // Wo, bo
      float acc = 0.0f;
      for (int g = g0; g < g1; ++g) {
        const float* o = b.DO + 6 * (size_t)g;
        if (t < kGnnH) acc = fmaf(o[0], H3[(size_t)g * kGnnH + t], acc);
        else if (t < 2 * kGnnH) acc = fmaf(o[1], H3[(size_t)g * kGnnH + t - kGnnH], acc);
        else acc += t < kGnnEdgeIn ? o[2 + t - 2 * kGnnH] : o[0];
      }
      out[kGnnOffWo + t] = acc;
    }
    if (t < 3 * kGnnH) {  // W0 (row-major 64 x 2), b0
      float acc = 0.0f;
      for (int g = g0; g < g1; ++g)
        acc = t < 2 * kGnnH ? fmaf(b.dpre0[(size_t)g * kGnnH + t / 2], xn[2 * g + (t & 1)], acc)
                            : acc + b.dpre0[(size_t)g * kGnnH + t - 2 * kGnnH];
      out[kGnnOffW0 + t] = acc;
    }
    return;
  }
  __shared__ float4 s1[kGradStage][16], s2[kGradStage][16], du[kGradStage][16], h[kGradStage][16], ag[kGradStage][16];
  const int to = t >> 4, tj = t & 15;
  float e1[4][4] = {}, e2[4][4] = {}, n1[4][4] = {}, n2[4][4] = {}, bias = 0.0f, fs = 0.0f;
  for (int g = g0; g < g1; g += kGradStage) {
    __syncthreads();
    for (int k = t; k < kGradStage * 16; k += 256) {
      const int gg = g + k / 16;
      const size_t at = (y * NH + (size_t)gg * kGnnH) / 4 + k % 16;
      const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      s1[k / 16][k % 16] = gg < g1 ? ((const float4*)b.S1)[at] : z;
      s2[k / 16][k % 16] = gg < g1 ? ((const float4*)b.S2)[at] : z;
      du[k / 16][k % 16] = gg < g1 ? ((const float4*)b.DU)[at] : z;
      h[k / 16][k % 16] = gg < g1 ? ((const float4*)b.H)[at] : z;
      ag[k / 16][k % 16] = gg < g1 ? ((const float4*)AGG)[at] : z;
    }
    __syncthreads();
    const int n = min(g1 - g, kGradStage);
    for (int k = 0; k < n; ++k) {
      const float4 hj = h[k][tj], d4 = du[k][to];
      outer4(e1, s1[k][to], hj);
      outer4(e2, s2[k][to], hj);
      outer4(n1, d4, hj);
      outer4(n2, d4, ag[k][tj]);
      fs += b.F[(y * NH + (size_t)(g + k) * kGnnH) * 4 + t];
      if (t < kGnnH) bias += ((const float*)s1[k])[t];
      else if (t < 2 * kGnnH) bias += ((const float*)du[k])[t - kGnnH];
    }
  }
  float* we = out + gnn_off_we(y);
  float* wn = out + gnn_off_wn(y);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int o = 4 * to + r;
    *(float4*)(we + o * kGnnEdgeIn + 4 * tj) = make_float4(e1[r][0], e1[r][1], e1[r][2], e1[r][3]);
    *(float4*)(we + o * kGnnEdgeIn + kGnnH + 4 * tj) = make_float4(e2[r][0], e2[r][1], e2[r][2], e2[r][3]);
    *(float4*)(wn + o * kGnnNodeIn + 4 * tj) = make_float4(n1[r][0], n1[r][1], n1[r][2], n1[r][3]);
    *(float4*)(wn + o * kGnnNodeIn + kGnnH + 4 * tj) = make_float4(n2[r][0], n2[r][1], n2[r][2], n2[r][3]);
  }
  we[(t >> 2) * kGnnEdgeIn + 2 * kGnnH + (t & 3)] = fs;
  if (t < kGnnH) out[gnn_off_be(y) + t] = bias;
  else if (t < 2 * kGnnH) out[gnn_off_bn(y) + t - kGnnH] = bias;
}

__global__ __launch_bounds__(256) void wgrad_sum_kernel(int parts, const float* __restrict__ part,
                                                        float* __restrict__ grad) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= kGnnParams) return;
  float acc = 0.0f;
#pragma unroll 16
  for (int c = 0; c < parts; ++c) acc += part[(size_t)c * kPartStride + id];
  grad[id] = acc;
}

__global__ void adam_kernel(int n, float* __restrict__ p, float* __restrict__ m, float* __restrict__ v,
                            const float* __restrict__ g, float lr, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = 0.9f * m[i] + 0.1f * gi, vi = 0.999f * v[i] + 0.001f * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
}

}  // namespace

// ------------------------------------------------------------------ host
int gnn_model_init(GnnModel& g, unsigned long long seed) {
  std::vector<float> h(kGnnParams, 0.0f);
  std::mt19937_64 rng(seed);
  std::normal_distribution<float> nd(0.0f, 1.0f);
  auto fill = [&](int off, int rows, int cols, float gain) {
    const float sd = gain * std::sqrt(2.0f / (float)cols);
    for (int k = 0; k < rows * cols; ++k) h[off + k] = sd * nd(rng);
  };
  fill(kGnnOffW0, kGnnH, 2, 1.0f);
  for (int l = 0; l < kGnnLayers; ++l) {
    fill(gnn_off_we(l), kGnnH, kGnnEdgeIn, 1.0f);
    fill(gnn_off_wn(l), kGnnH, kGnnNodeIn, 0.5f);
  }
  // Wo, bo zero: the untrained model weights every pair 1/2
  RSD_HIP(hipGetDevice(&g.dev));
  if (!g.p) RSD_HIP(hipMalloc(&g.p, kGnnParams * sizeof(float)));
  if (!g.m) RSD_HIP(hipMalloc(&g.m, kGnnParams * sizeof(float)));
  if (!g.v) RSD_HIP(hipMalloc(&g.v, kGnnParams * sizeof(float)));
  RSD_HIP(hipMemcpy(g.p, h.data(), kGnnParams * sizeof(float), hipMemcpyHostToDevice));
  RSD_HIP(hipMemset(g.m, 0, kGnnParams * sizeof(float)));
  RSD_HIP(hipMemset(g.v, 0, kGnnParams * sizeof(float)));
  g.t = 0;
  return RSD_OK;
}

void gnn_model_release(GnnModel& g) {
  for (void* p : {(void*)g.p, (void*)g.m, (void*)g.v})
    if (p) (void)hipFree(p);
  g = GnnModel{};
}

int gnn_work_reserve(GnnWork& w, int N, int cap, int nz) {
  if (w.N == N && w.cap == cap && w.nz >= nz) return RSD_OK;
  gnn_work_release(w);
  const size_t S = (size_t)N * cap, n = 11 * (size_t)N;
  const size_t nparts = (size_t)((N + grad_chunk(N) - 1) / grad_chunk(N)) * kPartStride;
  RSD_HIP(hipMalloc(&w.kb, (size_t)N * (cap + 1) * 121 * sizeof(double)));
  RSD_HIP(hipMalloc(&w.pa, S * 121 * sizeof(double)));
  RSD_HIP(hipMalloc(&w.pb, S * 121 * sizeof(double)));
  RSD_HIP(hipMalloc(&w.dist, S * sizeof(double)));
  RSD_HIP(hipMalloc(&w.rev, S * sizeof(int)));
  RSD_HIP(hipMalloc(&w.feat, S * kGnnF * sizeof(float)));
  RSD_HIP(hipMalloc(&w.xn, 2 * (size_t)N * sizeof(float)));
  RSD_HIP(hipMalloc(&w.H, 4 * (size_t)N * kGnnH * sizeof(float)));
  RSD_HIP(hipMalloc(&w.U, 3 * (size_t)N * kGnnH * sizeof(float)));
  RSD_HIP(hipMalloc(&w.AGG, 3 * (size_t)N * kGnnH * sizeof(float)));
  RSD_HIP(hipMalloc(&w.V, 3 * S * kGnnH * sizeof(float)));
  RSD_HIP(hipMalloc(&w.OUT, S * sizeof(float)));
  RSD_HIP(hipMalloc(&w.dOUT, S * sizeof(float)));
  RSD_HIP(hipMalloc(&w.bwd, (25 * kGnnH + 8) * (size_t)N * sizeof(float)));
  RSD_HIP(hipMalloc(&w.grad, kGnnParams * sizeof(float)));
  RSD_HIP(hipMalloc(&w.gpart, nparts * sizeof(float)));
  RSD_HIP(hipMalloc(&w.zv, (size_t)nz * n * sizeof(double)));
  RSD_HIP(hipMalloc(&w.gv, (size_t)nz * n * sizeof(double)));
  RSD_HIP(hipMalloc(&w.wv, 4 * (size_t)nz * (n + 1) * sizeof(double)));
  RSD_HIP(hipMalloc(&w.red, 2 * sizeof(double)));
  RSD_HIP(hipHostMalloc(&w.hred, 2 * sizeof(double)));
  w.N = N;
  w.cap = cap;
  w.nz = nz;
  return RSD_OK;
}

void gnn_work_release(GnnWork& w) {
  for (void* p : {(void*)w.kb, (void*)w.pa, (void*)w.pb, (void*)w.dist, (void*)w.rev, (void*)w.feat, (void*)w.xn,
                  (void*)w.H, (void*)w.U, (void*)w.AGG, (void*)w.V, (void*)w.OUT, (void*)w.dOUT, (void*)w.bwd,
                  (void*)w.grad, (void*)w.gpart, (void*)w.zv, (void*)w.gv, (void*)w.wv,
                  (void*)w.red})
    if (p) (void)hipFree(p);
  if (w.hred) (void)hipHostFree(w.hred);
  w = GnnWork{};
}

int gnn_prepare(GnnWork& w, const LubBsr<double>& L, const double* M, int ld, const double* radii, const double* dinv,
                hipStream_t s) {
  if (L.N != w.N || L.cap != w.cap) {
    set_error("gnn_prepare: buffers reserved for another size");
    return RSD_ERR_ARG;
  }
  const long long S = (long long)L.N * L.cap;
  hipLaunchKernelGGL(kblocks_kernel, dim3(L.N, (11 * (L.cap + 1) + 63) / 64), dim3(256), 0, s, L, M, ld, w.kb);
  hipLaunchKernelGGL(rev_kernel, dim3((unsigned)((S + 255) / 256)), dim3(256), 0, s, L, w.rev);
  hipLaunchKernelGGL(pair_basis_kernel, dim3(L.N, (L.cap + kPbPairs - 1) / kPbPairs), dim3(32 * kPbPairs), 0, s, L, (const double*)w.kb,
                     (const int*)w.rev, dinv, w.pa, w.pb);
  hipLaunchKernelGGL(features_kernel, dim3((unsigned)((S + 255) / 256)), dim3(256), 0, s, L, (const double*)w.dist,
                     radii, w.feat, w.xn);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

int gnn_forward(GnnWork& w, const float* params, const LubBsr<double>& L, double* corr, hipStream_t s) {
  const int N = L.N;
  const size_t NH = (size_t)N * kGnnH, SH = (size_t)N * L.cap * kGnnH;
  hipLaunchKernelGGL(gnn_input_kernel, dim3((unsigned)((NH + 255) / 256)), dim3(256), 0, s, N, params,
                     (const float*)w.xn, w.H);
  for (int l = 0; l < kGnnLayers; ++l)
    hipLaunchKernelGGL(gnn_layer_fwd_kernel, dim3(N), dim3(256), 0, s, L, params, l, (const float*)w.feat,
                       (const float*)(w.H + l * NH), w.H + (l + 1) * NH, w.U + l * NH, w.AGG + l * NH,
                       w.V + l * SH);
  hipLaunchKernelGGL(gnn_out_kernel, dim3(N), dim3(128), 0, s, L, params, (const float*)w.feat,
                     (const float*)(w.H + kGnnLayers * NH), (const double*)w.pa, (const double*)w.pb, w.OUT, corr);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

int gnn_loss_grad(GnnWork& w, const float* params, const LubBsr<double>& L, const double* M, int ld,
                  const double* dinv, const double* corr, int nz, unsigned long long seed, unsigned long long draw,
                  bool grad, bool log_loss, double* loss, hipStream_t s) {
  const int N = L.N, n = 11 * N, n6 = 6 * N;
  if (nz < 1 || nz > w.nz) {
    set_error("gnn_loss_grad: nz outside the reserved buffers");
    return RSD_ERR_ARG;
  }
  const dim3 blk(256), grd((n + 255) / 256, nz);
  // nz vectors of each, an even number of elements apart
  const size_t nv = ((size_t)n + 1) & ~(size_t)1;
  double* y = w.wv;
  double* mw = y + w.nz * nv;
  double* r = mw + w.nz * nv;
  double* t = r + w.nz * nv;
  for (int z = 0; z < nz; ++z)
    RSD_TRY(launch_brown_normal(n, seed, draw * 4096ull + (unsigned long long)z, w.zv + (size_t)z * n, s));
  // r = K P z - z
  RSD_TRY(block_apply_many(N, dinv, corr, L, w.zv, n, y, nv, nz, s));
  RSD_TRY(apply_k_many(L, M, ld, y, r, mw, nv, nz, s));
  hipLaunchKernelGGL(loss_residual_kernel, grd, blk, 0, s, n, n6, nv, (const double*)w.zv, r, t);
  hipLaunchKernelGGL(sumsq2_kernel, dim3(1), dim3(1024), 0, s, n, nz, nv, (const double*)r, (const double*)w.zv, w.red);
  if (grad) {
    // G = K^T r = r_P + M (R_lub r_P + r_Q)
    RSD_TRY(bsr_apply_many(L, t, y, nv, nz, s));
    hipLaunchKernelGGL(add_q_kernel, grd, blk, 0, s, n, n6, nv, (const double*)r, y);
    RSD_TRY(dense_gemv_many(M, ld, n, y, nv, w.gv, n, nz, s));
    hipLaunchKernelGGL(add_kernel, grd, blk, 0, s, n, nv, (const double*)t, w.gv);
  }
  RSD_HIP(hipGetLastError());
  if (grad) {
    const size_t NH = (size_t)N * kGnnH;
    const int chunk = grad_chunk(N), parts = (N + chunk - 1) / chunk;
    hipLaunchKernelGGL(gnn_dout_kernel, dim3(N), dim3(256), 0, s, L, (const double*)w.pa, (const double*)w.pb,
                       (const double*)w.gv, (const double*)w.zv, nz, (const double*)w.red, log_loss ? 1 : 0,
                       (const float*)w.OUT, w.dOUT);
    GnnBwd b{w.H, w.U, w.V, w.feat, w.dOUT, w.rev};
    b.F = w.bwd;  // (first: read as float4)
    b.S1 = b.F + 12 * NH;
    b.S2 = b.S1 + 3 * NH;
    b.DU = b.S2 + 3 * NH;
    b.dagg = b.DU + 3 * NH;
    b.dHp = b.dagg + 2 * NH;
    b.dpre0 = b.dHp + NH;
    b.DO = b.dpre0 + NH;
    for (int l = kGnnLayers; l >= 0; --l) hipLaunchKernelGGL(gnn_bwd_kernel, dim3(N), blk, 0, s, L, params, l, b);
    hipLaunchKernelGGL(gnn_wgrad_kernel, dim3(parts, kGnnLayers + 1), blk, 0, s, N, chunk, b, (const float*)w.AGG,
                       (const float*)w.xn, w.gpart);
    hipLaunchKernelGGL(wgrad_sum_kernel, dim3((kGnnParams + 255) / 256), blk, 0, s, parts, (const float*)w.gpart,
                       w.grad);
    RSD_HIP(hipGetLastError());
  }
  RSD_HIP(hipMemcpyAsync(w.hred, w.red, 2 * sizeof(double), hipMemcpyDeviceToHost, s));
  RSD_HIP(hipStreamSynchronize(s));
  *loss = w.hred[0] / w.hred[1];
  return RSD_OK;
}

int gnn_adam(GnnModel& g, const float* grad, float lr, hipStream_t s) {
  ++g.t;
  const float c1 = 1.0f - std::pow(0.9f, (float)g.t), c2 = 1.0f - std::pow(0.999f, (float)g.t);
  hipLaunchKernelGGL(adam_kernel, dim3((kGnnParams + 255) / 256), dim3(256), 0, s, kGnnParams, g.p, g.m, g.v, grad,
                     lr, c1, c2);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

}  // namespace rsd
