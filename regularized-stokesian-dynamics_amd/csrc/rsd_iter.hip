// rsd_iter.hip -- the iterative resistance solve: flexible GMRES on
//   K x = [F; -EIN],  K = [ (I + R_lub M)_P ; M_Q ],
// the mobility form the reference's hydro_SD_FTS (stepper.f90:476-546) hands
// to GMRES (gmres_mod_gmres.f90:23-61) instead of inverting M.
//
//   dense_gemv     y = M x for the symmetric M: a workgroup multiplies a few
//                  whole columns by x (HBM-bound: one pass over M)
//   bsr_apply      R_lub w from the 11x11 neighbour blocks, a wave a particle;
//   k_rows_kernel  K's rows from M x, with the partial dots of Gram-Schmidt
//   block_jacobi   K's 11x11 diagonal blocks, formed from the lubrication
//                  blocks and M, inverted by Gauss-Jordan with partial pivoting
//   gmres_solve    FP64 right-preconditioned flexible GMRES with classical
//                  Gram-Schmidt applied twice; the Hessenberg's Givens
//                  rotations on the host (one wait per iteration).  The mixed
//                  preconditioner is a fixed number of FP32 GMRES iterations
//                  on FP32 copies of M and R_lub, entirely on the device (its
//                  small least-squares problem solved by one wave), so the
//                  bulk of the matrix traffic moves half the bytes.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "rsd_iter.h"
#include "rsd_prof.h"

namespace rsd {

constexpr int kGemvCols = 8;  // columns a workgroup of the dense product

// particle g's local dof c (T 0-2, R 3-5, Q 6-10) in the field-major vector
__device__ __forceinline__ int dof(int N, int g, int c) {
  return c < 3 ? 3 * g + c : (c < 6 ? 3 * N + 3 * g + (c - 3) : 6 * N + 5 * g + (c - 6));
}

// 16-byte loads: 4 floats or 2 doubles
template <typename T>
struct Vec16;
template <>
struct Vec16<float> {
  using type = float4;
  static constexpr int n = 4;
};
template <>
struct Vec16<double> {
  using type = double2;
  static constexpr int n = 2;
};
__device__ __forceinline__ float vec_dot(const float4& a, const float4& b, float acc) {
  return fmaf(a.w, b.w, fmaf(a.z, b.z, fmaf(a.y, b.y, fmaf(a.x, b.x, acc))));
}
__device__ __forceinline__ double vec_dot(const double2& a, const double2& b, double acc) {
  return fma(a.y, b.y, fma(a.x, b.x, acc));
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// y = M x for a symmetric M: y_c is column c times x, so that a workgroup's
// kGemvCols columns are read along their contiguous length, each x vector
// serves all of them from a register, and no partial sums cross workgroups.
// Bound by the read of M (VEC: 16-byte loads, kGemvCols of them in flight a
// lane; M and x 16-byte aligned, ld a multiple of the vector).  The row
// products of column chunks that this replaced needed a second pass over 88
// partial vectors: 41 us for the FP32 M of N = 512 and 67 us for the FP64 one,
// against 20 us (6.3 TB/s) and 43 us (5.9 TB/s) here.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void sym_gemv_kernel(const T* __restrict__ M, size_t ld, int n,
                                                       const T* __restrict__ x, T* __restrict__ y) {
  constexpr int V = VEC ? Vec16<T>::n : 1, C = kGemvCols;
  __shared__ T red[4][C];
  const int c0 = blockIdx.x * C, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // columns past the last one repeat it
  const T* col[C];
#pragma unroll
  for (int c = 0; c < C; ++c) col[c] = M + (size_t)min(c0 + c, n - 1) * ld;
  T acc[C];
#pragma unroll
  for (int c = 0; c < C; ++c) acc[c] = 0;
  const int nv = n / V * V;
  for (int r = threadIdx.x * V; r < nv; r += 256 * V) {
    if (VEC) {
      using VT = typename Vec16<T>::type;
      const VT xv = *reinterpret_cast<const VT*>(x + r);
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c] = vec_dot(*reinterpret_cast<const VT*>(col[c] + r), xv, acc[c]);
    } else {
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c] = fma(col[c][r], x[r], acc[c]);
    }
  }
  if (nv + (int)threadIdx.x < n) {  // the rows past the last whole vector
    const int r = nv + threadIdx.x;
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = fma(col[c][r], x[r], acc[c]);
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const T v = wave_sum(acc[c]);
    if (lane == 0) red[wave][c] = v;
  }
  __syncthreads();
  const int c = threadIdx.x;
  if (c < C && c0 + c < n) y[c0 + c] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
}

// The same for NZ vectors (strides ldx, ldy) with one read of M, each vector's
// sums in the same order.  N = 256, four vectors: 52 us one by one, 20 so.
template <int NZ>
__global__ __launch_bounds__(256) void sym_gemv_many_kernel(const double* __restrict__ M, size_t ld, int n,
                                                            const double* __restrict__ x, size_t ldx,
                                                            double* __restrict__ y, size_t ldy) {
  constexpr int C = kGemvCols;
  __shared__ double red[4][C * NZ];
  const int c0 = blockIdx.x * C, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double* col[C];
#pragma unroll
  for (int c = 0; c < C; ++c) col[c] = M + (size_t)min(c0 + c, n - 1) * ld;
  double acc[C][NZ];
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int z = 0; z < NZ; ++z) acc[c][z] = 0.0;
  const int nv = n / 2 * 2;
  for (int r = threadIdx.x * 2; r < nv; r += 512) {
    double2 m[C];
#pragma unroll
    for (int c = 0; c < C; ++c) m[c] = *reinterpret_cast<const double2*>(col[c] + r);
#pragma unroll
    for (int z = 0; z < NZ; ++z) {
      const double2 xv = *reinterpret_cast<const double2*>(x + z * ldx + r);
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c][z] = vec_dot(m[c], xv, acc[c][z]);
    }
  }
  if (nv + (int)threadIdx.x < n) {
    const int r = nv + threadIdx.x;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int z = 0; z < NZ; ++z) acc[c][z] = fma(col[c][r], x[z * ldx + r], acc[c][z]);
  }
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int z = 0; z < NZ; ++z) {
      const double v = wave_sum(acc[c][z]);
      if (lane == 0) red[wave][c + C * z] = v;
    }
  __syncthreads();
  const int t = threadIdx.x, c = t % C, z = t / C;
  if (z < NZ && c0 + c < n) y[z * ldy + c0 + c] = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
}

int dense_gemv_many(const double* M, int ld, int n, const double* x, size_t ldx, double* y, size_t ldy, int nz,
                    hipStream_t s) {
  if (ld % 2 || ldx % 2 || ((reinterpret_cast<uintptr_t>(M) | reinterpret_cast<uintptr_t>(x)) & 15)) {
    for (int z = 0; z < nz; ++z) RSD_TRY(dense_gemv<double>(M, ld, n, x + z * ldx, y + z * ldy, s));
    return RSD_OK;
  }
  const double nn = (double)n * n;
  for (int z = 0; z < nz; z += 4) {
    const int k = std::min(4, nz - z);
    auto kern = k == 4 ? sym_gemv_many_kernel<4>
                       : k == 3 ? sym_gemv_many_kernel<3> : k == 2 ? sym_gemv_many_kernel<2> : sym_gemv_many_kernel<1>;
    hipEvent_t pe = prof_begin(kProfGemvSplit64, 2.0 * nn * k, 8.0 * (nn + 2.0 * n * k), s);
    hipLaunchKernelGGL(kern, dim3((n + kGemvCols - 1) / kGemvCols), dim3(256), 0, s, M, (size_t)ld, n, x + z * ldx, ldx,
                       y + z * ldy, ldy);
    prof_end(pe, s);
  }
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

template <typename T>
int dense_gemv(const T* M, int ld, int n, const T* x, T* y, hipStream_t s) {
  constexpr int V = Vec16<T>::n;
  // algorithmic work: 2 n^2 flops; bytes: M once, x, y
  const double nn = (double)n * n, by = sizeof(T) * (nn + 2.0 * n);
  const bool vec = ld % V == 0 && ((reinterpret_cast<uintptr_t>(M) | reinterpret_cast<uintptr_t>(x)) & 15) == 0;
  hipEvent_t pe = prof_begin(sizeof(T) == 8 ? kProfGemvSplit64 : kProfGemvSplit32, 2.0 * nn, by, s);
  hipLaunchKernelGGL((vec ? sym_gemv_kernel<T, true> : sym_gemv_kernel<T, false>),
                     dim3((n + kGemvCols - 1) / kGemvCols), dim3(256), 0, s, M, (size_t)ld, n, x, y);
  prof_end(pe, s);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// The neighbour-block products: a wave per particle g, four particles a
// workgroup.  Lane l takes the (slot, column) pairs l, l+64, ... of g's block
// row (slot 0 the self block, 1+q neighbour q), so that each lane reads whole
// 11-entry columns of the 11x11 blocks; the eleven row sums are then reduced
// across the wave.  The neighbours' indices are read once, a lane each, with
// the count, and handed round by shuffles.
constexpr int kGroup = 4;  // particles a workgroup

struct NeighbourCols {
  int lo, hi;  // neighbours lane, 64 + lane
};
__device__ __forceinline__ NeighbourCols neighbour_cols(const int* col, int cap, int g, int lane) {
  const int* c = col + (size_t)g * cap;
  return {lane < cap ? c[lane] : 0, 64 + lane < cap ? c[64 + lane] : 0};
}
static_assert(kIterMaxNeighbours == 2 * 64, "two neighbours a lane");
// neighbour q (every lane of the wave active)
__device__ __forceinline__ int neighbour(const NeighbourCols& nc, int q) {
  const int a = __shfl(nc.lo, q & 63, 64), b = __shfl(nc.hi, q & 63, 64);
  return q < 64 ? a : b;
}

// the rows of R_lub w of particle g (the first nrows), on every lane
template <typename T>
__device__ __forceinline__ void bsr_rows(const LubBsr<T>& L, int g, int lane, const T* __restrict__ w, int nrows,
                                         T (&acc)[11]) {
  const int N = L.N, nn = L.nnb[g];
  const NeighbourCols nc = neighbour_cols(L.col, L.cap, g, lane);
#pragma unroll
  for (int r = 0; r < 11; ++r) acc[r] = 0;
  for (int it0 = 0; it0 < 11 * (nn + 1); it0 += 64) {
    const int it = it0 + lane, slot = it / 11, c = it % 11;
    const int dq = neighbour(nc, max(slot - 1, 0));
    if (it < 11 * (nn + 1)) {
      const int d = slot == 0 ? g : dq;
      const T* b = slot == 0 ? L.self + 121 * (size_t)g : L.blk + 121 * ((size_t)g * L.cap + slot - 1);
      const T x = w[dof(N, d, c)];
#pragma unroll
      for (int r = 0; r < 11; ++r)
        if (r < nrows) acc[r] = fma(b[r + 11 * c], x, acc[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < 11; ++r)
    if (r < nrows) acc[r] = wave_sum(acc[r]);
}

// lw rows of particle g: self block and neighbour blocks times the
// neighbours' dofs (rows < 6 only when nrows is 6)
template <typename T>
__global__ __launch_bounds__(64 * kGroup) void bsr_apply_kernel(LubBsr<T> L, const T* __restrict__ w,
                                                                T* __restrict__ lw, int nrows, size_t ldv) {
  w += blockIdx.y * ldv;  // vector blockIdx.y
  lw += blockIdx.y * ldv;
  const int g = blockIdx.x * kGroup + (threadIdx.x >> 6), lane = threadIdx.x & 63, N = L.N;
  if (g >= N) return;
  T acc[11];
  bsr_rows(L, g, lane, w, nrows, acc);
#pragma unroll
  for (int r = 0; r < 11; ++r)
    if (lane == r && r < nrows) lw[dof(N, g, r)] = acc[r];
}

template <typename T>
int bsr_apply(const LubBsr<T>& L, const T* w, T* lw, bool p_rows_only, hipStream_t s) {
  const int nrows = p_rows_only ? 6 : 11;
  hipLaunchKernelGGL(bsr_apply_kernel<T>, dim3((L.N + kGroup - 1) / kGroup), dim3(64 * kGroup), 0, s, L, w, lw, nrows,
                     (size_t)0);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}
int bsr_apply_many(const LubBsr<double>& L, const double* w, double* lw, size_t ldv, int nz, hipStream_t s) {
  hipLaunchKernelGGL(bsr_apply_kernel<double>, dim3((L.N + kGroup - 1) / kGroup, nz), dim3(64 * kGroup), 0, s, L, w, lw,
                     11, ldv);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// K's rows from w = M x: y_P = x_P + (R_lub w)_P, y_Q = w_Q.  With k > 0 also
// the workgroup's share of V_j . y for the k vectors V_j (stride ldv), to
// part[j * gridDim.x + blockIdx.x]; with k = 0 for gridDim.y vectors x, w, y
// (stride ldv).
template <typename T>
__global__ __launch_bounds__(64 * kGroup) void k_rows_kernel(LubBsr<T> L, const T* __restrict__ x,
                                                             const T* __restrict__ w, T* __restrict__ y, int k,
                                                             const T* __restrict__ V, size_t ldv,
                                                             double* __restrict__ part) {
  __shared__ T ys[11 * kGroup];
  if (k == 0) {  // vector blockIdx.y of several
    x += blockIdx.y * ldv;
    w += blockIdx.y * ldv;
    y += blockIdx.y * ldv;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, N = L.N;
  const int g0 = blockIdx.x * kGroup, g = g0 + wave;
  if (g < N) {
    T acc[11];
    bsr_rows(L, g, lane, w, 6, acc);
    T v = 0;
#pragma unroll
    for (int r = 0; r < 6; ++r)
      if (lane == r) v = acc[r];
    if (lane < 11) {
      const int i = dof(N, g, lane);
      v = lane < 6 ? x[i] + v : w[i];
      y[i] = v;
      ys[11 * wave + lane] = v;
    }
  }
  if (k == 0) return;
  __syncthreads();
  const int rows = 11 * min(kGroup, N - g0);
  const int i = lane < rows ? dof(N, g0 + lane / 11, lane % 11) : 0;
  for (int j = wave; j < k; j += kGroup) {
    const double d = lane < rows ? (double)V[(size_t)j * ldv + i] * (double)ys[lane] : 0.0;
    const double sum = wave_sum(d);
    if (lane == 0) part[(size_t)j * gridDim.x + blockIdx.x] = sum;
  }
}

// workgroups of k_rows_kernel, the row length of its partial sums
static int k_rows_groups(int N) { return (N + kGroup - 1) / kGroup; }

template <typename T>
static int apply_k_dots(const LubBsr<T>& L, const T* M, int ld, const T* x, T* y, T* w, int k, const T* V, size_t ldv,
                        double* part, hipStream_t s) {
  RSD_TRY(dense_gemv(M, ld, 11 * L.N, x, w, s));
  hipLaunchKernelGGL(k_rows_kernel<T>, dim3(k_rows_groups(L.N)), dim3(64 * kGroup), 0, s, L, x, (const T*)w, y, k, V,
                     ldv, part);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

template <typename T>
int apply_k(const LubBsr<T>& L, const T* M, int ld, const T* x, T* y, T* wbuf, hipStream_t s) {
  return apply_k_dots<T>(L, M, ld, x, y, wbuf, 0, nullptr, 0, nullptr, s);
}

int apply_k_many(const LubBsr<double>& L, const double* M, int ld, const double* x, double* y, double* wbuf, size_t ldv,
                 int nz, hipStream_t s) {
  RSD_TRY(dense_gemv_many(M, ld, 11 * L.N, x, ldv, wbuf, ldv, nz, s));
  hipLaunchKernelGGL(k_rows_kernel<double>, dim3(k_rows_groups(L.N), nz), dim3(64 * kGroup), 0, s, L, x,
                     (const double*)wbuf, y, 0, (const double*)nullptr, ldv, (double*)nullptr);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// ----------------------------------------------------------- block Jacobi
__global__ __launch_bounds__(128) void block_jacobi_kernel(LubBsr<double> L, const double* __restrict__ M, int ld,
                                                           double* __restrict__ dinv) {
  __shared__ double A[11][12], X[11][12];
  __shared__ int piv;
  const int g = blockIdx.x, t = threadIdx.x, N = L.N;
  if (t < 121) {
    const int r = t % 11, c = t / 11;
    double v;
    if (r < 6) {
      v = (r == c) ? 1.0 : 0.0;
      // sum over the blocks of row g of R_lub (self and neighbours) of R(g,d)[r,:] M(d,g)[:,c]
      const double* b = L.self + 121 * (size_t)g;
      const int cg = dof(N, g, c);
      for (int k = 0; k < 11; ++k) v = fma(b[r + 11 * k], M[(size_t)dof(N, g, k) + (size_t)cg * ld], v);
      for (int q = 0; q < L.nnb[g]; ++q) {
        const int d = L.col[(size_t)g * L.cap + q];
        const double* bk = L.blk + 121 * ((size_t)g * L.cap + q);
        for (int k = 0; k < 11; ++k) v = fma(bk[r + 11 * k], M[(size_t)dof(N, d, k) + (size_t)cg * ld], v);
      }
    } else {
      v = M[(size_t)dof(N, g, r) + (size_t)dof(N, g, c) * ld];
    }
    A[r][c] = v;
    X[r][c] = (r == c) ? 1.0 : 0.0;
  }
  __syncthreads();
  // Gauss-Jordan with partial pivoting: A -> I, X -> inv(A)
  for (int k = 0; k < 11; ++k) {
    if (t == 0) {
      int p = k;
      double best = fabs(A[k][k]);
      for (int i = k + 1; i < 11; ++i)
        if (fabs(A[i][k]) > best) {
          best = fabs(A[i][k]);
          p = i;
        }
      piv = p;
    }
    __syncthreads();
    if (piv != k && t < 11) {
      double a = A[k][t], b = A[piv][t];
      A[k][t] = b;
      A[piv][t] = a;
      a = X[k][t];
      b = X[piv][t];
      X[k][t] = b;
      X[piv][t] = a;
    }
    __syncthreads();
    const double inv = 1.0 / A[k][k];
    __syncthreads();
    if (t < 11) {
      A[k][t] *= inv;
      X[k][t] *= inv;
    }
    __syncthreads();
    double fa = 0.0, fx = 0.0, f = 0.0;
    int r = 0, c = 0;
    if (t < 121) {
      r = t % 11;
      c = t / 11;
      f = A[r][k];
      fa = A[k][c];
      fx = X[k][c];
    }
    __syncthreads();
    if (t < 121 && r != k) {
      A[r][c] -= f * fa;
      X[r][c] -= f * fx;
    }
    __syncthreads();
  }
  if (t < 121) dinv[121 * (size_t)g + (t % 11) + 11 * (t / 11)] = X[t % 11][t / 11];
}

int block_jacobi_build(const LubBsr<double>& L, const double* M, int ld, double* dinv, hipStream_t s) {
  hipLaunchKernelGGL(block_jacobi_kernel, dim3(L.N), dim3(128), 0, s, L, M, ld, dinv);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// The squared norm left in partial sums by the vector kernels, by one wave
__device__ __forceinline__ double sum_partials(const double* __restrict__ part, int np, int lane) {
  double a = 0.0;
  for (int p = lane; p < np; p += 64) a += part[p];
  return wave_sum(a);
}

// z_g = dinv_g v_g + (corr_gg v_g + sum_d corr_gd v_d when a correction is
// given), for v scaled to unit norm when its squared norm's partial sums are
// given (np > 0); the norm and its reciprocal then go to norm[0] and inv[0].
// A wave per particle, as bsr_rows.
template <typename T>
__global__ __launch_bounds__(64 * kGroup) void block_apply_kernel(int N, const T* __restrict__ dinv,
                                                                  const double* __restrict__ corr, LubBsr<double> Lc,
                                                                  const T* __restrict__ v, T* __restrict__ z, int np,
                                                                  const double* __restrict__ partn,
                                                                  T* __restrict__ norm, double* __restrict__ inv,
                                                                  size_t ldv, size_t ldz) {
  v += blockIdx.y * ldv;  // vector blockIdx.y
  z += blockIdx.y * ldz;
  const int g = blockIdx.x * kGroup + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (g >= N) return;
  const int nn = corr ? Lc.nnb[g] : 0;
  NeighbourCols nc{0, 0};
  if (corr) nc = neighbour_cols(Lc.col, Lc.cap, g, lane);
  T sc = 1;
  if (np > 0) {
    const double nrm = sqrt(sum_partials(partn, np, lane)), r = nrm > 0.0 ? 1.0 / nrm : 0.0;
    sc = (T)r;
    if (g == 0 && lane == 0) {
      norm[0] = (T)nrm;
      inv[0] = r;
    }
  }
  const size_t base = (size_t)g * (Lc.cap + 1);
  T acc[11];
#pragma unroll
  for (int r = 0; r < 11; ++r) acc[r] = 0;
  // items 0..10: dinv's columns; 11..: the correction's (slot, column) pairs
  // (slot 0 its self block, 1+q neighbour q), only when there is a correction
  const int items = corr ? 11 * (nn + 2) : 11;
  for (int it0 = 0; it0 < items; it0 += 64) {
    const int it = it0 + lane, slot = it / 11 - 1, c = it % 11;
    const int dq = neighbour(nc, max(slot - 1, 0));
    if (it < 11) {
      const T x = sc * v[dof(N, g, it)];
      const T* b = dinv + 121 * (size_t)g;
#pragma unroll
      for (int r = 0; r < 11; ++r) acc[r] = fma(b[r + 11 * it], x, acc[r]);
    } else if (it < items) {
      const int d = slot == 0 ? g : dq;
      const double* b = corr + 121 * (base + slot);
      const double x = (double)(sc * v[dof(N, d, c)]);
#pragma unroll
      for (int r = 0; r < 11; ++r) acc[r] += (T)(b[r + 11 * c] * x);
    }
  }
  T out = 0;
#pragma unroll
  for (int r = 0; r < 11; ++r) {
    const T s = wave_sum(acc[r]);
    if (lane == r) out = s;
  }
  if (lane < 11) z[dof(N, g, lane)] = out;
}

template <typename T>
static int block_apply_scaled(int N, const T* dinv, const double* corr, const LubBsr<double>* Lcorr, const T* v, T* z,
                              int np, const double* partn, T* norm, double* inv, hipStream_t s) {
  LubBsr<double> Lc{};
  if (corr && Lcorr) Lc = *Lcorr;
  hipLaunchKernelGGL(block_apply_kernel<T>, dim3((N + kGroup - 1) / kGroup), dim3(64 * kGroup), 0, s, N, dinv,
                     (corr && Lcorr) ? corr : nullptr, Lc, v, z, np, partn, norm, inv, (size_t)0, (size_t)0);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}
int block_apply_many(int N, const double* dinv, const double* corr, const LubBsr<double>& Lcorr, const double* v,
                     size_t ldv, double* z, size_t ldz, int nz, hipStream_t s) {
  hipLaunchKernelGGL(block_apply_kernel<double>, dim3((N + kGroup - 1) / kGroup, nz), dim3(64 * kGroup), 0, s, N, dinv,
                     corr, Lcorr, v, z, 0, (const double*)nullptr, (double*)nullptr, (double*)nullptr, ldv, ldz);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

template <typename T>
int block_apply(int N, const T* dinv, const double* corr, const LubBsr<double>* Lcorr, const T* v, T* z,
                hipStream_t s) {
  return block_apply_scaled<T>(N, dinv, corr, Lcorr, v, z, 0, nullptr, nullptr, nullptr, s);
}

// ------------------------------------------------------------ vector kernels
// h[0] = v . v (one workgroup, fixed-order tree in LDS)
__global__ __launch_bounds__(256) void squared_norm_kernel(int n, const double* __restrict__ v, double* __restrict__ h) {
  __shared__ double red[256];
  double a = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) a = fma(v[i], v[i], a);
  red[threadIdx.x] = a;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) h[0] = red[0];
}

// The two passes of classical Gram-Schmidt of w against V_0..V_{k-1} (unit
// vectors inv[j] V_j; k <= kKrylov), a thread a row, kVecRows rows a
// workgroup.  Each workgroup first adds up the np partial sums of every V_j . w
// (part, rows of np), then w -= sum_j h_j inv[j] V_j with h_j = inv[j] V_j . w.
// SECOND = false: h goes to h1 and the partial sums of the next pass's dots to
// part2 (rows of gridDim.x).  SECOND: h1 + h goes to H and the squared norm's
// partial sums to partn.
// The sums over partials and over rows each go for all k vectors at once (8
// lanes a vector; a wave transposes while it reduces): one vector after
// another, the two passes took 9.0 and 5.3 us at N = 512, now 8.1 and 4.7.
constexpr int kKrylov = 32, kVecRows = 256;
static_assert(8 * kKrylov == kVecRows, "eight lanes a Krylov vector");

// v[0..31] of a wave's lanes -> the sum over the lanes of v[lane >> 1]
__device__ __forceinline__ double wave_sum32(double (&v)[32], int lane) {
#pragma unroll
  for (int half = 16, bit = 32; half >= 1; half >>= 1, bit >>= 1) {
    const bool up = lane & bit;
#pragma unroll
    for (int q = 0; q < half; ++q) {
      const double keep = up ? v[q + half] : v[q], send = up ? v[q] : v[q + half];
      v[q] = keep + __shfl_xor(send, bit, 64);
    }
  }
  return v[0] + __shfl_xor(v[0], 1, 64);
}

template <typename T, bool SECOND>
__global__ __launch_bounds__(kVecRows) void ortho_kernel(const T* __restrict__ V, size_t ldv, int n, int k,
                                                         const double* __restrict__ inv, T* __restrict__ w,
                                                         const double* __restrict__ part, int np,
                                                         double* __restrict__ h1, double* __restrict__ part2,
                                                         T* __restrict__ H, double* __restrict__ partn) {
  __shared__ double hs[kKrylov], red[kKrylov][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = blockIdx.x * kVecRows + tid;
  T v[kKrylov];
#pragma unroll
  for (int j = 0; j < kKrylov; ++j) v[j] = (j < k && i < n) ? V[(size_t)j * ldv + i] : (T)0;
  T a = i < n ? w[i] : (T)0;
  {
    const int j = tid >> 3;
    double h = 0.0;
    if (j < k) {
      const double* pj = part + (size_t)j * np;
#pragma unroll 16
      for (int p = tid & 7; p < np; p += 8) h += pj[p];
    }
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) h += __shfl_xor(h, off, 64);
    if (j < k && (tid & 7) == 0) {
      h *= inv[j];
      hs[j] = inv[j] * h;
      if (blockIdx.x == 0) {
        if (SECOND) H[j] = (T)(h1[j] + h);
        else h1[j] = h;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kKrylov; ++j)
    if (j < k) a -= v[j] * (T)hs[j];
  if (i < n) w[i] = a;
  if (SECOND) {
    const double s = wave_sum((double)a * (double)a);
    if (lane == 0) red[0][wave] = s;
    __syncthreads();
    if (tid == 0) partn[blockIdx.x] = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
  } else {
    double d[kKrylov];
#pragma unroll
    for (int j = 0; j < kKrylov; ++j) d[j] = (double)v[j] * (double)a;  // v is 0 past the k vectors and n rows
    const double s = wave_sum32(d, lane);
    if ((lane & 1) == 0) red[lane >> 1][wave] = s;
    __syncthreads();
    if (tid < k) part2[(size_t)tid * gridDim.x + blockIdx.x] = (red[tid][0] + red[tid][1]) + (red[tid][2] + red[tid][3]);
  }
}
static int vec_groups(int n) { return (n + kVecRows - 1) / kVecRows; }

// The device arrays of the two passes: part1 (k_rows_kernel's sums), part2,
// h1, and inv, the reciprocal norms of the Krylov vectors
struct OrthoWork {
  double *part1, *part2, *h1, *inv;
};
template <typename T>
static int orthogonalise(const T* V, size_t ldv, int n, int k, const OrthoWork& o, T* w, T* H, double* partn,
                         hipStream_t s) {
  const dim3 grd(vec_groups(n)), blk(kVecRows);
  hipLaunchKernelGGL((ortho_kernel<T, false>), grd, blk, 0, s, V, ldv, n, k, (const double*)o.inv, w,
                     (const double*)o.part1, k_rows_groups(n / 11), o.h1, o.part2, (T*)nullptr, (double*)nullptr);
  hipLaunchKernelGGL((ortho_kernel<T, true>), grd, blk, 0, s, V, ldv, n, k, (const double*)o.inv, w,
                     (const double*)o.part2, vec_groups(n), o.h1, (double*)nullptr, H, partn);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// y = (float) x, and the partial sums of the squared norm of y
__global__ __launch_bounds__(kVecRows) void krylov_start_kernel(int n, const double* __restrict__ x,
                                                                float* __restrict__ y, double* __restrict__ partn) {
  __shared__ double red[4];
  const int i = blockIdx.x * kVecRows + threadIdx.x, lane = threadIdx.x & 63;
  const float v = i < n ? (float)x[i] : 0.0f;
  if (i < n) y[i] = v;
  const double s = wave_sum((double)v * (double)v);
  if (lane == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) partn[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// x scaled to unit norm in place, from the partial sums of its squared norm
__global__ __launch_bounds__(kVecRows) void unit_norm_kernel(int n, double* __restrict__ x, int np,
                                                             const double* __restrict__ partn) {
  const double nrm = sqrt(sum_partials(partn, np, threadIdx.x & 63)), r = nrm > 0.0 ? 1.0 / nrm : 0.0;
  const int i = blockIdx.x * kVecRows + threadIdx.x;
  if (i < n) x[i] *= r;
}

// x += Z y (k columns)
__global__ void add_zy_kernel(const double* __restrict__ Z, size_t ldz, int n, int k, const double* __restrict__ y,
                              double* __restrict__ x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double a = x[i];
  for (int j = 0; j < k; ++j) a += Z[(size_t)j * ldz + i] * y[j];
  x[i] = a;
}

// y = x / *den
__global__ void scale_kernel(int n, const double* __restrict__ x, double* __restrict__ y,
                             const double* __restrict__ den) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i] * (1.0 / *den);
}

// r = b - y
__global__ void residual_kernel(int n, const double* __restrict__ b, const double* __restrict__ y,
                                double* __restrict__ r) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) r[i] = b[i] - y[i];
}

__global__ void f64_to_f32_kernel(const double* __restrict__ x, float* __restrict__ y, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    y[i] = (float)x[i];
}
__global__ void matrix_to_f32_kernel(const double* __restrict__ A, int lda, float* __restrict__ B, int ldb, int m,
                                     int n) {
  const int c = blockIdx.y;
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < m; r += gridDim.x * blockDim.x)
    B[(size_t)r + (size_t)c * ldb] = (float)A[(size_t)r + (size_t)c * lda];
}

int to_f32(const double* x, float* y, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(f64_to_f32_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 4096)), dim3(256), 0, s, x,
                     y, n);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}
int matrix_to_f32(const double* A, int lda, float* B, int ldb, int m, int n, hipStream_t s) {
  hipLaunchKernelGGL(matrix_to_f32_kernel, dim3((m + 255) / 256, n), dim3(256), 0, s, A, lda, B, ldb, m, n);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// ------------------------------------------------ the FP32 inner GMRES (device only)
// Least squares of the (k+1) x k Hessenberg H (column j at H + j*ldh; its last
// subdiagonal entry is the norm whose partial sums are in partn) with
// right-hand side beta e1 by Givens rotations, in FP64, then z = Z y.  k <= 31.
// Every workgroup solves the small problem for itself: column c in lane c of
// one wave, a rotation applied to all columns at once.
__global__ __launch_bounds__(kVecRows) void inner_result_kernel(const float* __restrict__ H, int ldh, int k,
                                                                const float* __restrict__ beta,
                                                                const double* __restrict__ partn, int np,
                                                                const float* __restrict__ Z, size_t ldz, int n,
                                                                double* __restrict__ z) {
  __shared__ double R[kKrylov + 1][kKrylov + 1];
  __shared__ float ys[kKrylov];
  const int lane = threadIdx.x & 63, i = blockIdx.x * kVecRows + threadIdx.x;
  float zv[kKrylov];
#pragma unroll
  for (int j = 0; j < kKrylov; ++j) zv[j] = (j < k && i < n) ? Z[(size_t)j * ldz + i] : 0.0f;
  for (int e = threadIdx.x; e < (k + 1) * k; e += kVecRows) {
    const int r = e % (k + 1), c = e / (k + 1);
    R[r][c] = r <= c + 1 && r + c < 2 * k - 1 ? (double)H[(size_t)c * ldh + r] : 0.0;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const double last = sqrt(sum_partials(partn, np, lane));
    if (lane == 0) R[k][k - 1] = (double)(float)last;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const int c = min(lane, k - 1);
    double g = lane == 0 ? (double)beta[0] : 0.0;  // the right-hand side's entry `lane`
    for (int j = 0; j < k; ++j) {
      const double a = R[j][j], b = R[j + 1][j], rr = sqrt(a * a + b * b);
      const double cs = rr > 0.0 ? a / rr : 1.0, sn = rr > 0.0 ? b / rr : 0.0;
      const double u = R[j][c], v = R[j + 1][c];
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (lane == j) {
        R[j][j] = rr;
        R[j + 1][j] = 0.0;
      } else if (lane > j && lane < k) {
        R[j][lane] = cs * u + sn * v;
        R[j + 1][lane] = -sn * u + cs * v;
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      const double t = __shfl(g, j, 64);
      if (lane == j) g = cs * t;
      if (lane == j + 1) g = -sn * t;
    }
    // back substitution, y_r in lane r: the solved unknown leaves all rows above it
    for (int r = k - 1; r >= 0; --r) {
      const double d = R[r][r], yr = d != 0.0 ? __shfl(g, r, 64) / d : 0.0;
      if (lane < r) g -= R[lane][r] * yr;
      if (lane == 0) ys[r] = (float)yr;
    }
  }
  __syncthreads();
  float a = 0.0f;
#pragma unroll
  for (int j = 0; j < kKrylov; ++j)
    if (j < k) a += zv[j] * ys[j];
  if (i < n) z[i] = (double)a;
}

constexpr int kInnerMax = 31;
static_assert(kInnerMax < kKrylov, "the Gram-Schmidt passes hold every Krylov vector");

// the stride of Krylov vectors: whole 16-byte vectors
static size_t vec_ld(int n) { return ((size_t)n + 3) & ~(size_t)3; }

// z = approximately inv(K) v: `its` right-preconditioned FP32 GMRES
// iterations on K32 (block-Jacobi dinv32 inside), from zero.  Five launches an
// iteration, each leaving the partial sums that the next one adds up itself:
// the preconditioner (of the Krylov vector scaled to unit norm), the product
// with M, K's rows with the first Gram-Schmidt pass's dots, and the two passes.
// An inner iteration of N = 512 takes 60 us, the product with M 20 of them (110
// in fourteen launches before).
static int inner_solve(IterWork& w, const GmresSetup& g, const double* v, double* z, hipStream_t s) {
  const int n = w.n, N = n / 11, its = std::max(1, std::min(g.inner_iters, kInnerMax));
  const size_t ld = vec_ld(n);
  float* V = w.V32;                          // its+1 vectors, not scaled (inv: their reciprocal norms)
  float* Zs = w.V32 + (size_t)(kInnerMax + 1) * ld;  // its preconditioned vectors
  float* H = w.h32;                          // (kInnerMax+1) x kInnerMax Hessenberg, then beta
  float* beta = w.h32 + (kInnerMax + 1) * kInnerMax;
  const OrthoWork o{w.part1, w.part2, w.h1, w.inv};
  const dim3 blk(kVecRows), grd(vec_groups(n));
  const bool learned = g.precond == kIterMixedLearned;
  hipLaunchKernelGGL(krylov_start_kernel, grd, blk, 0, s, n, v, V, w.partn);
  for (int j = 0; j < its; ++j) {
    float* Vj = V + (size_t)j * ld;
    float* Zj = Zs + (size_t)j * ld;
    float* wv = V + (size_t)(j + 1) * ld;
    float* hj = H + (size_t)j * (kInnerMax + 1);
    float* norm = j == 0 ? beta : H + (size_t)(j - 1) * (kInnerMax + 1) + j;
    RSD_TRY(block_apply_scaled<float>(N, w.dinv32, learned ? w.corr : nullptr, learned ? g.Lcorr : nullptr, Vj, Zj,
                                      vec_groups(n), w.partn, norm, w.inv + j, s));
    RSD_TRY(apply_k_dots<float>(*g.L32, g.M32, g.ld32, Zj, wv, w.w32, j + 1, V, ld, w.part1, s));
    RSD_TRY(orthogonalise<float>(V, ld, n, j + 1, o, wv, hj, w.partn, s));
  }
  hipLaunchKernelGGL(inner_result_kernel, grd, blk, 0, s, (const float*)H, kInnerMax + 1, its, (const float*)beta,
                     (const double*)w.partn, vec_groups(n), (const float*)Zs, ld, n, z);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

__global__ void copy_kernel(int n, const double* __restrict__ x, double* __restrict__ y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i];
}

// inner_solve on the fixed buffers w.vin -> w.zout, captured once into a HIP
// graph and replayed: its five launches an iteration cost the host one graph
// launch.  Everything it reads is fixed by the key (the matrices, the
// preconditioner's blocks, the iteration count), and it records no memset.
static int inner_solve_graph(IterWork& w, const GmresSetup& g, const double* v, double* z, hipStream_t s) {
  const int n = w.n;
  const void* key[8] = {g.M32, g.L32->blk, g.L32->self, g.L32->nnb, w.dinv32, w.corr,
                        g.Lcorr ? (const void*)g.Lcorr->nnb : nullptr, w.V32};
  const int key_i[4] = {n, std::max(1, std::min(g.inner_iters, kInnerMax)), g.precond, g.ld32};
  bool same = w.inner_exec != nullptr;
  for (int k = 0; k < 8 && same; ++k) same = key[k] == w.inner_key[k];
  for (int k = 0; k < 4 && same; ++k) same = key_i[k] == w.inner_key_i[k];
  if (!same) {
    if (w.inner_exec) (void)hipGraphExecDestroy(w.inner_exec);
    if (w.inner_graph) (void)hipGraphDestroy(w.inner_graph);
    w.inner_exec = nullptr;
    w.inner_graph = nullptr;
    RSD_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    const int rc = inner_solve(w, g, w.vin, w.zout, s);
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(s, &graph);
    if (rc != RSD_OK) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc;
    }
    RSD_HIP(e);
    w.inner_graph = graph;
    RSD_HIP(hipGraphInstantiate(&w.inner_exec, graph, nullptr, nullptr, 0));
    for (int k = 0; k < 8; ++k) w.inner_key[k] = key[k];
    for (int k = 0; k < 4; ++k) w.inner_key_i[k] = key_i[k];
  }
  const dim3 blk(256), grd((n + 255) / 256);
  hipLaunchKernelGGL(copy_kernel, grd, blk, 0, s, n, v, w.vin);
  // one replay streams the FP32 M through the gemv once per inner iteration
  const double its = key_i[1], mb = (double)g.ld32 * n * sizeof(float);
  hipEvent_t pe = prof_begin(kProfInnerGraph, its * 2.0 * (double)n * n, its * mb, s);
  RSD_HIP(hipGraphLaunch(w.inner_exec, s));
  prof_end(pe, s);
  hipLaunchKernelGGL(copy_kernel, grd, blk, 0, s, n, (const double*)w.zout, z);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// ------------------------------------------------------- the FP64 outer FGMRES
int iter_reserve(IterWork& w, int n11, int m, int N, int bsr_cap) {
  if (m > kInnerMax) m = kInnerMax;
  if ((size_t)n11 <= w.cap_n && w.m == m) {
    w.n = n11;
    return RSD_OK;
  }
  iter_release(w);
  const size_t n = vec_ld(n11), groups = (size_t)vec_groups(n11);
  RSD_HIP(hipMalloc(&w.V, (size_t)(m + 1) * n * sizeof(double)));
  RSD_HIP(hipMalloc(&w.Z, (size_t)m * n * sizeof(double)));
  RSD_HIP(hipMalloc(&w.w, 4 * n * sizeof(double)));
  RSD_HIP(hipHostMalloc(&w.hh, (kKrylov + groups) * sizeof(double)));
  // the short vectors, in one allocation; the outer iteration's Hessenberg
  // column and norm partials are side by side, as the host reads them
  const size_t np1 = (size_t)kKrylov * k_rows_groups(N), np2 = (size_t)kKrylov * groups;
  RSD_HIP(hipMalloc(&w.h, (2 * (size_t)(m + 2) + kKrylov + groups + np1 + np2 + groups + 3 * kKrylov) * sizeof(double)));
  w.hcol = w.h + 2 * (m + 2);
  w.part1 = w.hcol + kKrylov + groups;
  w.part2 = w.part1 + np1;
  w.partn = w.part2 + np2;
  w.h1 = w.partn + groups;
  w.inv = w.h1 + kKrylov;
  w.ones = w.inv + kKrylov;
  const std::vector<double> ones(kKrylov, 1.0);
  RSD_HIP(hipMemcpy(w.ones, ones.data(), kKrylov * sizeof(double), hipMemcpyHostToDevice));
  RSD_HIP(hipMalloc(&w.V32, (size_t)(2 * kInnerMax + 1) * n * sizeof(float)));
  RSD_HIP(hipMalloc(&w.w32, n * sizeof(float)));
  RSD_HIP(hipMalloc(&w.h32, ((kInnerMax + 1) * kInnerMax + 1) * sizeof(float)));
  RSD_HIP(hipMalloc(&w.dinv, 121 * (size_t)N * sizeof(double)));
  RSD_HIP(hipMalloc(&w.dinv32, 121 * (size_t)N * sizeof(float)));
  RSD_HIP(hipMalloc(&w.corr, 121 * (size_t)N * (bsr_cap + 1) * sizeof(double)));
  RSD_HIP(hipMalloc(&w.vin, n * sizeof(double)));
  RSD_HIP(hipMalloc(&w.zout, n * sizeof(double)));
  w.cap_n = n11;
  w.n = n11;
  w.m = m;
  return RSD_OK;
}

void iter_release(IterWork& w) {
  if (w.inner_exec) (void)hipGraphExecDestroy(w.inner_exec);
  if (w.inner_graph) (void)hipGraphDestroy(w.inner_graph);
  for (void* p : {(void*)w.V, (void*)w.Z, (void*)w.w, (void*)w.h, (void*)w.V32, (void*)w.w32, (void*)w.h32,
                  (void*)w.dinv, (void*)w.dinv32, (void*)w.corr, (void*)w.vin, (void*)w.zout})
    if (p) (void)hipFree(p);
  if (w.hh) (void)hipHostFree(w.hh);
  w = IterWork{};
}

static int precondition(IterWork& w, const GmresSetup& g, const double* v, double* z, hipStream_t s) {
  const int n = w.n, N = n / 11;
  switch (g.precond) {
    case kIterNone:
      RSD_HIP(hipMemcpyAsync(z, v, n * sizeof(double), hipMemcpyDeviceToDevice, s));
      return RSD_OK;
    case kIterBlockJacobi:
      return block_apply<double>(N, w.dinv, nullptr, nullptr, v, z, s);
    case kIterLearned:
      return block_apply<double>(N, w.dinv, w.corr, g.Lcorr, v, z, s);
    case kIterMixed:
    case kIterMixedLearned:
      return g.graphs ? inner_solve_graph(w, g, v, z, s) : inner_solve(w, g, v, z, s);
  }
  set_error("gmres: unknown preconditioner");
  return RSD_ERR_ARG;
}

int gmres_solve(IterWork& w, const GmresSetup& g, const double* b, double* x, double tol, int max_iter,
                GmresResult* res, hipStream_t s) {
  const int n = w.n, m = w.m;
  const size_t ld = vec_ld(n);
  double* r = w.w;             // residual / work
  double* y = w.w + ld;        // K x
  double* kw = w.w + 2 * ld;   // M x
  const dim3 blk(256), grd((n + 255) / 256);
  auto kx = [&](const double* in, double* out) { return apply_k<double>(*g.L, g.M, g.ld, in, out, kw, s); };
  auto norm = [&](const double* v, double* out) -> int {
    hipLaunchKernelGGL(squared_norm_kernel, dim3(1), blk, 0, s, n, v, out);
    RSD_HIP(hipGetLastError());
    return RSD_OK;
  };
  // ||b||
  RSD_TRY(norm(b, w.h));
  RSD_HIP(hipMemcpyAsync(w.hh, w.h, sizeof(double), hipMemcpyDeviceToHost, s));
  RSD_HIP(hipStreamSynchronize(s));
  const double bnorm = std::sqrt(w.hh[0]);
  *res = GmresResult{};
  if (!(bnorm > 0.0)) {
    RSD_HIP(hipMemsetAsync(x, 0, n * sizeof(double), s));
    res->converged = true;
    return RSD_OK;
  }
  int it = 0;
  double prev_beta = 0.0;
  std::vector<double> H((size_t)(m + 1) * m), cs(m), sn(m), gg(m + 1), yy(m);
  while (true) {
    RSD_TRY(kx(x, y));
    hipLaunchKernelGGL(residual_kernel, grd, blk, 0, s, n, b, (const double*)y, r);
    RSD_TRY(norm(r, w.h));
    RSD_HIP(hipMemcpyAsync(w.hh, w.h, sizeof(double), hipMemcpyDeviceToHost, s));
    RSD_HIP(hipStreamSynchronize(s));
    const double beta = std::sqrt(w.hh[0]);
    res->relres = beta / bnorm;
    if (beta <= tol * bnorm) {
      res->converged = true;
      break;
    }
    if (!std::isfinite(beta) || it >= max_iter) break;
    // near the tolerance, a cycle that did not halve the true residual has
    // met FP64's floor for this system (the rounding of R_lub (M x), whose
    // entries grow as 1/gap): within 100 tol that is the answer, else give up
    // rather than spin to max_iter
    if (prev_beta > 0.0 && beta > 0.5 * prev_beta && beta < 1e3 * tol * bnorm) {
      res->converged = beta <= 1e2 * tol * bnorm;
      res->at_floor = res->converged;
      break;
    }
    prev_beta = beta;
    // V0 = r / beta
    double* hb = w.h + (m + 2);
    w.hh[1] = beta;
    RSD_HIP(hipMemcpyAsync(hb, w.hh + 1, sizeof(double), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(scale_kernel, grd, blk, 0, s, n, (const double*)r, w.V, (const double*)hb);
    std::fill(gg.begin(), gg.end(), 0.0);
    gg[0] = beta;
    int k = 0;
    bool done = false;
    for (; k < m && it < max_iter; ++k, ++it) {
      double* Vk = w.V + (size_t)k * ld;
      double* Zk = w.Z + (size_t)k * ld;
      double* wv = w.V + (size_t)(k + 1) * ld;
      RSD_TRY(precondition(w, g, Vk, Zk, s));
      // K Z_k, orthogonalised twice; its Hessenberg column and norm partials to the host
      double* partn = w.hcol + kKrylov;
      const OrthoWork o{w.part1, w.part2, w.h1, w.ones};
      RSD_TRY(apply_k_dots<double>(*g.L, g.M, g.ld, Zk, wv, kw, k + 1, w.V, ld, w.part1, s));
      RSD_TRY(orthogonalise<double>(w.V, ld, n, k + 1, o, wv, w.hcol, partn, s));
      RSD_HIP(hipMemcpyAsync(w.hh, w.hcol, (kKrylov + (size_t)vec_groups(n)) * sizeof(double), hipMemcpyDeviceToHost,
                             s));
      hipLaunchKernelGGL(unit_norm_kernel, dim3(vec_groups(n)), dim3(kVecRows), 0, s, n, wv, vec_groups(n),
                         (const double*)partn);
      RSD_HIP(hipGetLastError());
      RSD_HIP(hipStreamSynchronize(s));
      double* hc = &H[(size_t)k * (m + 1)];
      for (int i = 0; i <= k; ++i) hc[i] = w.hh[i];
      double hn2 = 0.0;
      for (int p = 0; p < vec_groups(n); ++p) hn2 += w.hh[kKrylov + p];
      hc[k + 1] = std::sqrt(hn2);
      for (int i = 0; i < k; ++i) {
        const double a = hc[i], bb = hc[i + 1];
        hc[i] = cs[i] * a + sn[i] * bb;
        hc[i + 1] = -sn[i] * a + cs[i] * bb;
      }
      const double a = hc[k], bb = hc[k + 1], rr = std::sqrt(a * a + bb * bb);
      cs[k] = rr > 0.0 ? a / rr : 1.0;
      sn[k] = rr > 0.0 ? bb / rr : 0.0;
      hc[k] = rr;
      hc[k + 1] = 0.0;
      gg[k + 1] = -sn[k] * gg[k];
      gg[k] = cs[k] * gg[k];
      if (!std::isfinite(gg[k + 1])) {
        done = true;
        ++k;
        ++it;
        break;
      }
      if (std::fabs(gg[k + 1]) <= 0.5 * tol * bnorm) {  // the estimate; the true residual decides below
        ++k;
        ++it;
        done = true;
        break;
      }
    }
    // x += Z y, y from the triangular system
    for (int i = k - 1; i >= 0; --i) {
      double acc = gg[i];
      for (int c = i + 1; c < k; ++c) acc -= H[(size_t)c * (m + 1) + i] * yy[c];
      yy[i] = H[(size_t)i * (m + 1) + i] != 0.0 ? acc / H[(size_t)i * (m + 1) + i] : 0.0;
    }
    if (k > 0) {
      RSD_HIP(hipMemcpyAsync(w.h, yy.data(), k * sizeof(double), hipMemcpyHostToDevice, s));
      hipLaunchKernelGGL(add_zy_kernel, grd, blk, 0, s, (const double*)w.Z, ld, n, k, (const double*)w.h, x);
      RSD_HIP(hipGetLastError());
      RSD_HIP(hipStreamSynchronize(s));  // w.h is reused as the next step's scratch
    }
    (void)done;
  }
  res->iterations = it;
  return RSD_OK;
}

template int dense_gemv<double>(const double*, int, int, const double*, double*, hipStream_t);
template int dense_gemv<float>(const float*, int, int, const float*, float*, hipStream_t);
template int apply_k<double>(const LubBsr<double>&, const double*, int, const double*, double*, double*, hipStream_t);
template int bsr_apply<double>(const LubBsr<double>&, const double*, double*, bool, hipStream_t);
template int block_apply<double>(int, const double*, const double*, const LubBsr<double>*, const double*, double*,
                                 hipStream_t);

}  // namespace rsd
