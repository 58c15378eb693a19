// rsd_dense.hip -- FP64 dense linear algebra for the grand-resistance solve.
//
// Replaces MATREV (matrices.f90:4-34: DPOTRF('U') + DPOTRI('U') + mirror)
// with a dataflow tile Cholesky in one launch, and a recursive triangular
// inverse and a triangular X^T X product on one batched 64x64-tile GEMM, all
// on the CDNA4 FP64 matrix cores (v_mfma_f64_16x16x4_f64).
//
// Layout: column-major, order padded to a multiple of 64 with an identity
// block so no kernel needs edge handling.  The symmetric input is read from
// its lower triangle; the reference reads the upper one, and the callers
// build the lower triangle as the mirror of the reference's upper triangle.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "rsd_dag.h"
#include "rsd_internal.h"
#include "rsd_prof.h"

namespace rsd {

typedef double v4d __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ GEMM
// One workgroup = one 64x64 output tile, 4 waves in a 2x2 arrangement, each
// wave a 32x32 sub-tile = 2x2 MFMA 16x16 blocks.  The inner dimension goes
// through LDS in chunks of 32, NS = 2 or 3 chunks in flight: a chunk is
// staged by direct 16-byte global->LDS loads (8 per wave), issued NS-1 chunks
// ahead of the products that read it.  NS = 3 (96 KB of LDS, one workgroup
// per CU) hides more latency; NS = 2 (64 KB, two per CU) wins once a launch
// has tiles enough for two rounds of workgroups.
//
// MFMA f64 16x16x4 operand layout (lane l, 0..63):
//   A: A[l%16][l/16]     B: B[l/16][l%16]     D: D[(l/16)+4*v][l%16], v=0..3
constexpr int LDSP = 64 + 2;  // padded LDS row (doubles)
constexpr int GKC = 32;              // inner dimension per staged chunk
constexpr int GCH = 64 * GKC;        // doubles per operand chunk
constexpr int GLD = 8;               // direct loads per wave per chunk (both operands)
constexpr int kWaitVm0 = 0x0f70;     // s_waitcnt vmcnt(0): expcnt and lgkmcnt left at their maxima
constexpr int kCpolSc1 = 16;         // cache policy of a direct-to-LDS load: sc1 (agent scope, coherent)
// s_waitcnt vmcnt(n), n < 64, expcnt and lgkmcnt left at their maxima
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0f70; }

// Up to kInlineDesc descriptors travel in the kernel arguments (no copy on
// the stream); larger batches use a device array.
constexpr int kInlineDesc = 20;
struct GemmArgs {
  GemmDesc d[kInlineDesc];
  const GemmDesc* ext;
  int nd, flags;
};

// Staged operand chunks, two layouts (r = the output row or column index,
// k = the inner index within the chunk, 0..31):
//  r-contiguous (op(X)(r, k) = X[r + k ld]: A, or B transposed): element
//    (r, k) at k*64 + (r ^ 16 (k & 1));
//  k-contiguous (op(X)(r, k) = X[k + r ld]: A transposed, or B): element
//    (r, k) at r*32 + 2 ((k/2) ^ (r & 15)) + (k & 1).
// The swaps put the 16 rows (or the 4 inner indices) that one MFMA operand
// read touches on different LDS banks.
template <bool KCONT>
__device__ __forceinline__ int gemm_staged(int r, int k) {
  return KCONT ? r * 32 + 2 * ((k >> 1) ^ (r & 15)) + (k & 1) : k * 64 + (r ^ ((k & 1) << 4));
}

// 64 x 32 chunk of op(X) at (r0, k0), 4 direct loads per wave
template <bool KCONT>
__device__ __forceinline__ void gemm_stage(const double* __restrict__ X, size_t ld, int r0, int k0,
                                           double* __restrict__ dst) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int q = wave * 4 + u;  // 16 loads of 1 KB: 2 columns (r-contiguous) or 4 rows (k-contiguous)
    const double* src;
    if (KCONT) {
      const int r = 4 * q + (lane >> 4), p = (lane & 15) ^ (r & 15);
      src = X + (size_t)(k0 + 2 * p) + (size_t)(r0 + r) * ld;
    } else {
      const int k = 2 * q + (lane >> 5), p = (lane & 31) ^ ((k & 1) << 3);
      src = X + (size_t)(r0 + 2 * p) + (size_t)(k0 + k) * ld;
    }
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)(dst + q * 128), 16, 0, 0);
  }
}

// one chunk's products (cur), the loads of a later chunk (into nxt, when
// pre) in flight meanwhile; cur and nxt are distinct restrict pointers so
// that the compiler lets the reads of cur pass the loads into nxt
template <bool TA, bool TB>
__device__ __forceinline__ void gemm_chunk(v4d (&acc)[2][2], const GemmDesc& D, int m0, int n0, int kload, bool pre,
                                           const double* __restrict__ cur, double* __restrict__ nxt) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  if (pre) {
    gemm_stage<TA>(D.A, (size_t)D.lda, m0, kload, nxt);
    gemm_stage<!TB>(D.B, (size_t)D.ldb, n0, kload, nxt + GCH);
  }
  const double* cb = cur + GCH;
#pragma unroll
  for (int kk = 0; kk < GKC; kk += 4) {
    const int kr = kk + (lane >> 4), m = lane & 15;
    const double a0 = cur[gemm_staged<TA>(wm + m, kr)];
    const double a1 = cur[gemm_staged<TA>(wm + 16 + m, kr)];
    const double b0 = cb[gemm_staged<!TB>(wn + m, kr)];
    const double b1 = cb[gemm_staged<!TB>(wn + 16 + m, kr)];
    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
  }
}

// LDS reads done and every wave here: a barrier without the fence of
// __syncthreads, which would also wait for the chunks still in flight
__device__ __forceinline__ void gemm_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <bool TA, bool TB, int NS>
__global__ __launch_bounds__(256) void gemm64_kernel(GemmArgs args) {
  static_assert(NS == 2 || NS == 3, "two or three chunks in flight");
  const GemmDesc* __restrict__ descs = (args.nd <= kInlineDesc) ? args.d : args.ext;
  const int ndesc = args.nd, flags = args.flags;
  // NS staged chunks of op(A) and op(B); the output tile reuses the space
  __shared__ __attribute__((aligned(16))) double smem[NS * 2 * GCH];
  double(*Cs)[LDSP] = reinterpret_cast<double(*)[LDSP]>(smem);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int t = blockIdx.x;
  int d = 0;
  while (d + 1 < ndesc && descs[d + 1].tile_base <= t) ++d;
  const GemmDesc D = descs[d];
  const int local = t - D.tile_base;
  int ti, tj;
  if (flags & kLowerC) {
    ti = (int)((sqrt(8.0 * local + 1.0) - 1.0) * 0.5);
    while ((ti + 1) * (ti + 2) / 2 <= local) ++ti;
    while (ti * (ti + 1) / 2 > local) --ti;
    tj = local - ti * (ti + 1) / 2;
  } else if (flags & kKhiRow) {
    // longest inner ranges first (they end after the row): rows from the bottom
    ti = D.mt - 1 - local / D.nt;
    tj = local % D.nt;
  } else {
    ti = local % D.mt;
    tj = local / D.mt;
  }
  // the tile is the workgroup's: keep its indices (and the chunk loop) scalar
  ti = __builtin_amdgcn_readfirstlane(ti);
  tj = __builtin_amdgcn_readfirstlane(tj);
  int klo = 0, khi = D.kt;
  if (flags & kKloRow) klo = max(klo, ti);
  if (flags & kKloCol) klo = max(klo, tj);
  if (flags & kKhiRow) khi = min(khi, ti + 1);

  const int m0 = ti * 64, n0 = tj * 64;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  v4d acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = (v4d){0.0, 0.0, 0.0, 0.0};

  const int k_begin = __builtin_amdgcn_readfirstlane(klo * 64);
  const int nch = __builtin_amdgcn_readfirstlane(khi > klo ? (khi - klo) * (64 / GKC) : 0);
  if (nch > 0) {
#pragma unroll
    for (int c = 0; c < NS - 1; ++c)
      if (c < nch) {
        gemm_stage<TA>(D.A, (size_t)D.lda, m0, k_begin + c * GKC, smem + c * 2 * GCH);
        gemm_stage<!TB>(D.B, (size_t)D.ldb, n0, k_begin + c * GKC, smem + (c * 2 + 1) * GCH);
      }
    for (int c = 0; c < nch; ++c) {
      // chunk c is in (each wave waits for its own loads; the barrier for
      // everyone's), and chunk c-1's buffer is free for chunk c+NS-1
      const int later = min(NS - 2, nch - 1 - c);  // chunks issued after c
      if (NS == 3 && later == 1)
        __builtin_amdgcn_s_waitcnt(wait_vm(GLD));
      else
        __builtin_amdgcn_s_waitcnt(kWaitVm0);
      gemm_barrier();
      const int cn = c + NS - 1;
      gemm_chunk<TA, TB>(acc, D, m0, n0, k_begin + cn * GKC, cn < nch, smem + (c % NS) * 2 * GCH,
                         smem + (cn % NS) * 2 * GCH);
    }
    gemm_barrier();
  }
  // stage the tile through LDS for column-contiguous stores
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        int r = wm + bm * 16 + (lane >> 4) + 4 * v;
        int c = wn + bn * 16 + (lane & 15);
        Cs[c][r] = acc[bm][bn][v];
      }
  __syncthreads();
  double* __restrict__ Cg = D.C;
  for (int idx = tid; idx < 4096; idx += 256) {
    int r = idx & 63, c = idx >> 6;
    size_t off = (size_t)(m0 + r) + (size_t)(n0 + c) * D.ldc;
    double v = D.alpha * Cs[c][r];
    if (D.beta != 0.0) v += D.beta * Cg[off];
    Cg[off] = v;
  }
}

// inner-dimension tiles actually multiplied, summed over the output tiles
static double desc_ktiles(const GemmDesc& g, int flags) {
  double tot = 0.0;
  const int ntile = (flags & kLowerC) ? g.mt : g.nt;
  for (int ti = 0; ti < g.mt; ++ti)
    for (int tj = 0; tj < ntile; ++tj) {
      if ((flags & kLowerC) && tj > ti) continue;
      int klo = 0, khi = g.kt;
      if (flags & kKloRow) klo = std::max(klo, ti);
      if (flags & kKloCol) klo = std::max(klo, tj);
      if (flags & kKhiRow) khi = std::min(khi, ti + 1);
      if (khi > klo) tot += khi - klo;
    }
  return tot;
}

static int desc_tiles(const GemmDesc& g, int flags) {
  if (flags & kLowerC) return g.mt * (g.mt + 1) / 2;
  return g.mt * g.nt;
}

int gemm_batched(DenseWork& w, const std::vector<GemmDesc>& in, bool ta, bool tb, int flags, hipStream_t s) {
  if (in.empty()) return RSD_OK;
  std::vector<GemmDesc> descs;
  descs.reserve(in.size());
  int total = 0;
  for (GemmDesc g : in) {
    if (g.mt <= 0 || g.nt <= 0) continue;
    g.tile_base = total;
    total += desc_tiles(g, flags);
    descs.push_back(g);
  }
  if (descs.empty()) return RSD_OK;
  GemmArgs args{};
  args.nd = (int)descs.size();
  args.flags = flags;
  if (descs.size() <= (size_t)kInlineDesc) {
    for (size_t i = 0; i < descs.size(); ++i) args.d[i] = descs[i];
  } else {
    if (descs.size() > w.desc_cap) {
      set_error("gemm_batched: descriptor buffer too small");
      return RSD_ERR_CAPACITY;
    }
    RSD_HIP(hipMemcpyAsync(w.d_desc, descs.data(), descs.size() * sizeof(GemmDesc), hipMemcpyHostToDevice, s));
    args.ext = w.d_desc;
  }
  dim3 grid(total), block(256);
  hipEvent_t pe = nullptr;
  if (prof_on()) {
    double kt = 0.0;
    for (const GemmDesc& g : descs) kt += desc_ktiles(g, flags);
    pe = prof_begin(kProfGemm, kt * 2.0 * 64.0 * 64.0 * 64.0, 0.0, s);
  }
  const bool two = total >= 1024;  // two rounds of workgroups at two per CU
  void (*kern)(GemmArgs);
  if (!ta && !tb)
    kern = two ? gemm64_kernel<false, false, 2> : gemm64_kernel<false, false, 3>;
  else if (!ta && tb)
    kern = two ? gemm64_kernel<false, true, 2> : gemm64_kernel<false, true, 3>;
  else if (ta && !tb)
    kern = two ? gemm64_kernel<true, false, 2> : gemm64_kernel<true, false, 3>;
  else
    kern = two ? gemm64_kernel<true, true, 2> : gemm64_kernel<true, true, 3>;
  hipLaunchKernelGGL(kern, grid, block, 0, s, args);
  prof_end(pe, s);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// The thread index through an empty asm: address arithmetic derived from it
// is redone at each call instead of being hoisted out of the persistent
// Cholesky's ticket loop and held in registers (spilled) across the tasks.
__device__ __forceinline__ int opaque_tid() {
  int t = threadIdx.x;
  __asm__ volatile("" : "+v"(t));
  return t;
}

// Hand-offs between workgroups of one launch (the dataflow Cholesky and the
// triangular solves) write through: the producer stores
// the data with agent-scope relaxed atomic stores, which write through the
// L2 to the device's coherence point; each wave waits for its own stores to
// complete (wt_stores_done) before the workgroup barrier that precedes the
// flag store (wt_publish, relaxed).  The consumer polls the flag and then
// reads the data with agent-scope loads, which do not return stale L2 or L1
// copies.  Neither side needs an agent-scope release or acquire fence, which
// writes back or invalidates the whole XCD's L2: under
// load they made each hand-off 1-2 us slower and made the other tiles on
// the XCD re-read their operands.
__device__ __forceinline__ void wt_store(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double wt_load(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void wt_stores_done() { __builtin_amdgcn_s_waitcnt(kWaitVm0); }
__device__ __forceinline__ void wt_publish(int* flag, int gen) {
  __hip_atomic_store(flag, gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// after a flag was seen: keeps the compiler from moving the data loads above
// the poll (the hardware issues them after the polled value is in)
__device__ __forceinline__ void wt_seen() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront"); }

// A 64x64 tile of the factorization (published by another workgroup; column-
// major, leading dimension ld) into LDS by direct 16-byte loads at agent scope,
// past any stale cached copy, 1 KB (two columns) per wave instruction: a wave's
// u-th load (of 8) moves columns 16 wave + 2u and 16 wave + 2u + 1; at: the
// lane's offset into the tile (stage_at), the same for every u.  Column c of
// the staged tile holds row m at c*64 + (m ^ 16 (c & 1)): the swap of 16-row
// halves on odd columns puts the two columns an MFMA operand read touches on
// different LDS banks.
__device__ __forceinline__ unsigned stage_at(int ld) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
  return (unsigned)((16 * wave + (lane >> 5)) * ld + 2 * ((lane & 31) ^ ((lane >> 5) << 3)));
}
__device__ __forceinline__ void stage_load(const double* p, int ld, unsigned at, int u, double* dst) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p + (size_t)(2 * u) * ld + at),
                                   (__attribute__((address_space(3))) void*)(dst + (wave * 8 + u) * 128), 16, 0,
                                   kCpolSc1);
}
__device__ __forceinline__ void stage_tile(const double* src, int ld, double* dst) {
  const unsigned at = stage_at(ld);
#pragma unroll
  for (int u = 0; u < 8; ++u) stage_load(src, ld, at, u, dst);
}

// element (m, c) of a staged tile
__device__ __forceinline__ int staged(int m, int c) { return c * 64 + (m ^ ((c & 1) << 4)); }

// ------------------------------------------------------------- FP32 GEMM
// The CG preconditioner's products (triangular inverse and Gram product of an
// FP32 copy of the factor): gemm64_kernel's organisation with
// v_mfma_f32_16x16x4f32 (twice the FP64 MFMA rate) and 4-byte elements.
// Operand lanes as the FP64 instruction; output D[4*(l/16)+v][l%16].
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int FCH = 64 * GKC;  // floats per operand chunk

// Staged FP32 chunks (r = output row or column index, k = inner index within
// the chunk, 0..31), 16-byte units swapped so that the 64 lanes of an MFMA
// operand read touch 64 distinct banks:
//  r-contiguous: element (r, k) at k*64 + (r ^ 16 (k & 3));
//  k-contiguous: element (r, k) at r*32 + 4 ((k/4) ^ ((r/2) & 7)) + (k & 3).
template <bool KCONT>
__device__ __forceinline__ int gemm32_staged(int r, int k) {
  return KCONT ? r * 32 + 4 * ((k >> 2) ^ ((r >> 1) & 7)) + (k & 3) : k * 64 + (r ^ ((k & 3) << 4));
}

// 64 x 32 chunk of op(X) at (r0, k0), 2 direct 16-byte loads per wave
template <bool KCONT>
__device__ __forceinline__ void gemm32_stage(const float* __restrict__ X, size_t ld, int r0, int k0,
                                             float* __restrict__ dst) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int q = wave * 2 + u;  // 8 loads of 1 KB: 4 columns (r-contiguous) or 8 rows (k-contiguous)
    const float* src;
    if (KCONT) {
      const int r = 8 * q + (lane >> 3), p = (lane & 7) ^ ((r >> 1) & 7);
      src = X + (size_t)(k0 + 4 * p) + (size_t)(r0 + r) * ld;
    } else {
      const int k = 4 * q + (lane >> 4), p = (lane & 15) ^ ((k & 3) << 2);
      src = X + (size_t)(r0 + 4 * p) + (size_t)(k0 + k) * ld;
    }
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)(dst + q * 256), 16, 0, 0);
  }
}

struct Gemm32Desc {
  const float* A;
  const float* B;
  float* C;
  int lda, ldb, ldc;
  int mt, nt, kt;  // C is (mt*64) x (nt*64), inner dimension kt*64
  float alpha, beta;
  int tile_base;
};
struct Gemm32Args {
  Gemm32Desc d[kInlineDesc];
  const Gemm32Desc* ext;
  int nd, flags;
};

template <bool TA, bool TB>
__device__ __forceinline__ void gemm32_chunk(v4f (&acc)[2][2], const Gemm32Desc& D, int m0, int n0, int kload,
                                             bool pre, const float* __restrict__ cur, float* __restrict__ nxt) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  if (pre) {
    gemm32_stage<TA>(D.A, (size_t)D.lda, m0, kload, nxt);
    gemm32_stage<!TB>(D.B, (size_t)D.ldb, n0, kload, nxt + FCH);
  }
  const float* cb = cur + FCH;
#pragma unroll
  for (int kk = 0; kk < GKC; kk += 4) {
    const int kr = kk + (lane >> 4), m = lane & 15;
    const float a0 = cur[gemm32_staged<TA>(wm + m, kr)];
    const float a1 = cur[gemm32_staged<TA>(wm + 16 + m, kr)];
    const float b0 = cb[gemm32_staged<!TB>(wn + m, kr)];
    const float b1 = cb[gemm32_staged<!TB>(wn + 16 + m, kr)];
    acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1, acc[1][1], 0, 0, 0);
  }
}

// three chunks in flight (48 KB of LDS)
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void gemm32_kernel(Gemm32Args args) {
  const Gemm32Desc* __restrict__ descs = (args.nd <= kInlineDesc) ? args.d : args.ext;
  const int ndesc = args.nd, flags = args.flags;
  __shared__ __attribute__((aligned(16))) float smem[3 * 2 * FCH];
  float(*Cs)[65] = reinterpret_cast<float(*)[65]>(smem);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t = blockIdx.x;
  int d = 0;
  while (d + 1 < ndesc && descs[d + 1].tile_base <= t) ++d;
  const Gemm32Desc D = descs[d];
  const int local = t - D.tile_base;
  int ti, tj;
  if (flags & kLowerC) {
    ti = (int)((sqrt(8.0 * local + 1.0) - 1.0) * 0.5);
    while ((ti + 1) * (ti + 2) / 2 <= local) ++ti;
    while (ti * (ti + 1) / 2 > local) --ti;
    tj = local - ti * (ti + 1) / 2;
  } else if (flags & kKhiRow) {
    ti = D.mt - 1 - local / D.nt;  // longest inner ranges first
    tj = local % D.nt;
  } else {
    ti = local % D.mt;
    tj = local / D.mt;
  }
  ti = __builtin_amdgcn_readfirstlane(ti);
  tj = __builtin_amdgcn_readfirstlane(tj);
  int klo = 0, khi = D.kt;
  if (flags & kKloRow) klo = max(klo, ti);
  if (flags & kKloCol) klo = max(klo, tj);
  if (flags & kKhiRow) khi = min(khi, ti + 1);
  const int m0 = ti * 64, n0 = tj * 64;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  v4f acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  const int k_begin = __builtin_amdgcn_readfirstlane(klo * 64);
  const int nch = __builtin_amdgcn_readfirstlane(khi > klo ? (khi - klo) * (64 / GKC) : 0);
  if (nch > 0) {
    for (int c = 0; c < 2 && c < nch; ++c) {
      gemm32_stage<TA>(D.A, (size_t)D.lda, m0, k_begin + c * GKC, smem + c * 2 * FCH);
      gemm32_stage<!TB>(D.B, (size_t)D.ldb, n0, k_begin + c * GKC, smem + (c * 2 + 1) * FCH);
    }
    for (int c = 0; c < nch; ++c) {
      if (c + 1 < nch)
        __builtin_amdgcn_s_waitcnt(wait_vm(4));  // chunk c+1's 4 loads per wave may fly on
      else
        __builtin_amdgcn_s_waitcnt(kWaitVm0);
      gemm_barrier();
      const int cn = c + 2;
      gemm32_chunk<TA, TB>(acc, D, m0, n0, k_begin + cn * GKC, cn < nch, smem + (c % 3) * 2 * FCH,
                           smem + (cn % 3) * 2 * FCH);
    }
    gemm_barrier();
  }
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v) Cs[wn + bn * 16 + (lane & 15)][wm + bm * 16 + 4 * (lane >> 4) + v] = acc[bm][bn][v];
  __syncthreads();
  float* __restrict__ Cg = D.C;
  for (int idx = tid; idx < 4096; idx += 256) {
    const int r = idx & 63, c = idx >> 6;
    const size_t off = (size_t)(m0 + r) + (size_t)(n0 + c) * D.ldc;
    float v = D.alpha * Cs[c][r];
    if (D.beta != 0.f) v += D.beta * Cg[off];
    Cg[off] = v;
  }
}

static int gemm32_batched(DenseWork& w, const std::vector<Gemm32Desc>& in, bool ta, int flags, hipStream_t s) {
  std::vector<Gemm32Desc> descs;
  int total = 0;
  for (Gemm32Desc g : in) {
    if (g.mt <= 0 || g.nt <= 0) continue;
    if ((g.lda & 3) || (g.ldb & 3) || (reinterpret_cast<uintptr_t>(g.A) & 15) ||
        (reinterpret_cast<uintptr_t>(g.B) & 15)) {
      set_error("gemm32: operands must be 16-byte aligned with leading dimensions a multiple of 4");
      return RSD_ERR_ARG;
    }
    g.tile_base = total;
    total += (flags & kLowerC) ? g.mt * (g.mt + 1) / 2 : g.mt * g.nt;
    descs.push_back(g);
  }
  if (descs.empty()) return RSD_OK;
  Gemm32Args args{};
  args.nd = (int)descs.size();
  args.flags = flags;
  if (descs.size() <= (size_t)kInlineDesc) {
    for (size_t i = 0; i < descs.size(); ++i) args.d[i] = descs[i];
  } else {
    if (descs.size() > w.desc_cap) {
      set_error("gemm32: descriptor buffer too small");
      return RSD_ERR_CAPACITY;
    }
    static_assert(sizeof(Gemm32Desc) <= sizeof(GemmDesc), "FP32 descriptors fit the descriptor buffer");
    RSD_HIP(hipMemcpyAsync(w.d_desc, descs.data(), descs.size() * sizeof(Gemm32Desc), hipMemcpyHostToDevice, s));
    args.ext = reinterpret_cast<const Gemm32Desc*>(w.d_desc);
  }
  hipEvent_t pe = nullptr;
  if (prof_on()) {  // timed with the FP64 GEMMs' family; inner tiles as desc_ktiles counts them
    double kt = 0.0;
    for (const Gemm32Desc& g : descs) {
      const int ntile = (flags & kLowerC) ? g.mt : g.nt;
      for (int ti = 0; ti < g.mt; ++ti)
        for (int tj = 0; tj < ntile; ++tj) {
          if ((flags & kLowerC) && tj > ti) continue;
          int klo = 0, khi = g.kt;
          if (flags & kKloRow) klo = std::max(klo, ti);
          if (flags & kKloCol) klo = std::max(klo, tj);
          if (flags & kKhiRow) khi = std::min(khi, ti + 1);
          if (khi > klo) kt += khi - klo;
        }
    }
    pe = prof_begin(kProfGemm, kt * 2.0 * 64.0 * 64.0 * 64.0, 0.0, s);
  }
  if (ta)
    hipLaunchKernelGGL((gemm32_kernel<true, false>), dim3(total), dim3(256), 0, s, args);
  else
    hipLaunchKernelGGL((gemm32_kernel<false, false>), dim3(total), dim3(256), 0, s, args);
  prof_end(pe, s);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// ------------------------------------------------ 64x64 diagonal factor
// 1/sqrt(d) to full FP64 accuracy for the pivots, instead of an IEEE sqrt
// and a divide on the serial pivot chain: the hardware estimate y0
// (v_rsq_f64, relative error 5e-8 measured on gfx950) and one third-order
// correction y = y0 (1 + e/2 + 3e^2/8), e = 1 - d y0^2, whose error is
// O(e^3): within 2 ulp (max 2.2e-16 over 2^20 inputs spanning 2^-56..2^56).
__device__ __forceinline__ double rsqrt_nr(double d) {
  const double y0 = __builtin_amdgcn_rsq(d);
  const double e = fma(-d * y0, y0, 1.0);
  return fma(y0 * e, fma(0.375, e, 0.5), y0);
}

// lane N of each row of 16 lanes to the whole row
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
  return __builtin_amdgcn_update_dpp(v, v, 0x150 + N, 0xf, 0xf, true);
}

// D += P(16x16) * Q(16x16) on the matrix cores: P points at the block's first
// element in a row-major LDS array with row stride PS, Q is in registers in the
// layout of a result (lane: rows (lane>>4)+4v of column lane&15), which is also
// that of the right operand's k-steps v and, for Q^T, of the left operand's: a
// product's result feeds the next one without a trip through LDS.
template <int PS>
__device__ __forceinline__ v4d mm16(const double* P, const v4d& q, v4d acc, int lane) {
  double a[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) a[kb] = P[(lane & 15) * PS + 4 * kb + (lane >> 4)];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kb], q[kb], acc, 0, 0, 0);
  return acc;
}

struct DiagSmem {
  double P[4][64][18];   // the factor by 16-column panels, rows below the panel's diagonal block
  double Xs[64][65];     // its inverse, lower 16x16 blocks
  double R[64][65];      // the tile; then U, the previous panel's rank-16 term: [column - 16][row], rows of 66
  double T[64][66];      // the next column's tile (j+1,j) of the factor, transposed
  int bad;
  int ready;             // 1 + the last column whose partial tiles are known to be published
  int stored;            // waves whose part of an inverse is stored, over all columns
};

// columns Q2 .. 15 less a pivot's term
template <int Q2>
__device__ __forceinline__ void panel_terms(double (&dg)[16], double (&a)[16], double vd, double va) {
  if constexpr (Q2 < 16) {
    const double m = row_bcast<Q2>(vd);
    dg[Q2] = fma(-vd, m, dg[Q2]);
    a[Q2] = fma(-va, m, a[Q2]);
    panel_terms<Q2 + 1>(dg, a, vd, va);
  }
}
// Pivots Q .. 15 of a 16x16 block and its share of the rows below.  Each of the
// four rows of 16 lanes holds the block, lane i its row i in dg, so that every
// multiplier is a broadcast within 16 lanes (one instruction); a is one more
// row per lane, solved along.  A bit of `ok` per positive pivot.
template <int Q>
__device__ __forceinline__ void panel_pivots(double (&dg)[16], double (&a)[16], unsigned& ok) {
  const double d = row_bcast<Q>(dg[Q]);
  const double y = rsqrt_nr(d);
  ok |= ((unsigned)__ballot(d > 0.0) & 1u) << Q;
  const double vd = dg[Q] * y, va = a[Q] * y;
  dg[Q] = vd;
  a[Q] = va;
  panel_terms<Q + 1>(dg, a, vd, va);
  if constexpr (Q + 1 < 16) panel_pivots<Q + 1>(dg, a, ok);
}

// 16x16 blocks in MFMA layout (lane holds rows (lane>>4)+4v of column lane&15)
template <int DS>
__device__ __forceinline__ v4d blk_load(const double* src, int lane) {
  v4d t;
#pragma unroll
  for (int v = 0; v < 4; ++v) t[v] = src[((lane >> 4) + 4 * v) * DS + (lane & 15)];
  return t;
}
template <int DS>
__device__ __forceinline__ void blk_store(double* dst, v4d t, double sign, int lane) {
#pragma unroll
  for (int v = 0; v < 4; ++v) dst[((lane >> 4) + 4 * v) * DS + (lane & 15)] = sign * t[v];
}
// orders a wave's LDS writes before its later reads of other lanes' elements
__device__ __forceinline__ void wave_lds_order() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// Cholesky of one 64x64 diagonal tile held in registers by 256 threads, and
// its triangular inverse: thread (w, l) has row l, columns 16w..16w+15 in
// a[], and row 16w + l%16 of the same columns in dg[].  The tile is done in
// four 16-column panels, panel b by wave b alone: the pivot chain runs on its
// diagonal block, which each row of 16 lanes holds for itself (panel_pivots),
// and lane l's row of the panel follows it.  The lanes of the diagonal block's
// own rows solve the identity's rows instead, which gives X_bb^T = L_bb^-T
// with the panel.  A pivot is bound by its chain, broadcast, reciprocal square
// root, scale, next column's term, with the other columns' terms between.
// The finished panel goes to LDS; after a barrier, its rank-16 term for all
// the columns to its right is formed by MFMA 16x16x16 products (the lower
// blocks only, spread over the waves) and handed over through LDS after a
// second barrier.
// The inverse's other blocks: wave m < 3 has column m, X_im = -X_ii sum_{k=m}^{i-1}
// L_ik X_km, the sums and blocks in registers; a sum grows by one product per
// panel while the wave has no panel of its own, and after the last one only
// the products with X_33 are left.
// A 64x64 tile and its inverse take 21k clocks so (a panel's 16 pivots 2.4k); with
// the multipliers read from lanes and LDS, X_bb by substitutions of their own and
// two levels of products after the last panel they took 34.5k.
// On return sm.P holds L's panels, sm.Xs the lower blocks of X, sm.bad the
// LAPACK-style INFO of the first non-positive pivot (k0 + j + 1) or 0x7fffffff,
// a[] this wave's columns of L in the rows below the diagonal block and dg[]
// the block's own rows; a barrier has to follow.
// idle(b) runs while panel b is factored on the waves that do not own it, last()
// on all when the panels are done, before the last products.
template <class Idle, class Last>
__device__ __forceinline__ void diag_factor64(double (&a)[16], double (&dg)[16], DiagSmem& sm, int k0, Idle&& idle,
                                              Last&& last) {
  const int w = __builtin_amdgcn_readfirstlane(opaque_tid() >> 6);
  if (threadIdx.x == 0) sm.bad = 0x7fffffff;
  const v4d z = {0.0, 0.0, 0.0, 0.0};
  double(*U)[66] = reinterpret_cast<double(*)[66]>(&sm.R[0][0]);
  v4d xt[4] = {z, z, z, z};  // the sums for X_im, i > m = w
#pragma unroll 1
  for (int b = 0; b < 4; ++b) {
    const int l = opaque_tid() & 63;  // (LDS addresses not kept over the panels: there are too many)
    if (b > 0) {
      // U = the previous panel's rank-16 term for the columns to its right:
      // block (rb, cb) = Pp[16rb.., :] Pp[16cb.., :]^T for rb >= cb >= b (the
      // blocks above the diagonal are not needed), by MFMA, spread over the
      // waves; every wave then subtracts its own columns' blocks
      double(*Pp)[18] = sm.P[b - 1];
      for (int n = w; n < (4 - b) * (5 - b) / 2; n += 4) {
        // block n, by columns
        int cb = b, k = n;
        while (k >= 4 - cb) k -= 4 - cb++;
        const int rb = cb + k;
        const int r = l & 15, kq = l >> 4;
        v4d u = z;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
          u = __builtin_amdgcn_mfma_f64_16x16x4f64(Pp[16 * rb + r][4 * kb + kq], Pp[16 * cb + r][4 * kb + kq], u, 0,
                                                   0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v) U[16 * (cb - 1) + r][16 * rb + kq + 4 * v] = u[v];
      }
      __syncthreads();
      if (w >= b) {
        // (rows above the column block are above the diagonal: a is not read there)
        const double *ud = &U[16 * (w - 1)][16 * w + (l & 15)], *ua = &U[16 * (w - 1)][l];
        double td[16], ta[16];  // (all read, then subtracted: left to itself the compiler waits for each pair)
#pragma unroll
        for (int q = 0; q < 16; ++q) td[q] = ud[66 * q], ta[q] = ua[66 * q];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 16; ++q) dg[q] -= td[q], a[q] -= ta[q];
      }
    }
    if (w == b) {
      const int g = l >> 4, i = l & 15;
      unsigned ok = 0;
      if (g == b) {
#pragma unroll
        for (int q = 0; q < 16; ++q) a[q] = (q == i) ? 1.0 : 0.0;
      }
      panel_pivots<0>(dg, a, ok);
      if (g == b) {
        // a is row i of X_bb^T, dg row i of L_bb
#pragma unroll
        for (int q = 0; q < 16; ++q) sm.Xs[16 * b + q][l] = a[q];
      }
      // (nothing reads the rows of the diagonal block or above it)
#pragma unroll
      for (int q = 0; q < 16; ++q) sm.P[b][l][q] = a[q];
      if (ok != 0xffffu && l == 0) atomicMin(&sm.bad, k0 + 16 * b + __builtin_ctz(~ok) + 1);
    } else {
      if (w < b && w < 3) {
        // X_{b-1,w}, and its products for the sums of the rows below
        const int k = b - 1;
        v4d x;
        if (k == w) {
          x = blk_load<65>(&sm.Xs[16 * w][16 * w], l);
        } else {
          const v4d t = k == 1 ? xt[1] : xt[2];
          x = -mm16<65>(&sm.Xs[16 * k][16 * k], t, z, l);
          blk_store<65>(&sm.Xs[16 * k][16 * w], x, 1.0, l);
        }
#pragma unroll
        for (int i = 1; i < 4; ++i)
          if (i >= b) xt[i] = mm16<18>(&sm.P[k][16 * i][0], x, xt[i], l);
      }
      idle(b);
    }
    __syncthreads();
  }
  // the inverse's last row of blocks
  last();
  if (w < 3) {
    const int l = opaque_tid() & 63;
    blk_store<65>(&sm.Xs[48][16 * w], mm16<65>(&sm.Xs[48][48], xt[3], z, l), -1.0, l);
  }
}

// the factor (this wave's columns in a and dg, as diag_factor64 leaves them)
// into the matrix, from its element (k0, k0) at A
__device__ __forceinline__ void diag_store_factor(const double (&a)[16], const double (&dg)[16],
                                                  double* __restrict__ A, size_t ld) {
  const int tid = opaque_tid(), w = tid >> 6, l = tid & 63, g = l >> 4, i = l & 15;
#pragma unroll
  for (int q = 0; q < 16; ++q)
    A[(size_t)l + (size_t)(16 * w + q) * ld] = g > w ? a[q] : (g == w && q <= i) ? dg[q] : 0.0;
}
// rows 16 rb .. of the inverse, columns 4n .. 4n+3 (column-major, zero upper
// blocks; written through)
__device__ __forceinline__ void diag_store_inverse(const DiagSmem& sm, double* __restrict__ dinv, int rb, int n, int lane) {
  const int r = 16 * rb + (lane & 15), c = 4 * n + (lane >> 4);
  wt_store(dinv + r + (size_t)c * 64, n < 4 * rb + 4 ? sm.Xs[r][c] : 0.0);
}

__global__ void set_int_kernel(int* p, int v) { *p = v; }

int dense_info_reset(DenseWork& w, hipStream_t s) {
  hipLaunchKernelGGL(set_int_kernel, dim3(1), dim3(1), 0, s, w.d_info, 0x7fffffff);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// ------------------------------------------- tile hand-off (shared by the
// dataflow Cholesky and the triangular solves)

// Spin (relaxed, agent scope) until *flag holds gen; a wait that runs out
// sets the error word and returns (the result is then garbage, never a hang).
// Once the error word is set every later wait returns at once, so a failed
// launch drains in one time-out rather than one per dependency.  The limit is
// wall-clock time, read from the GPU's constant 100 MHz counter: 20 s for any
// one wait, whatever the launch's size or what else shares the GPU.
constexpr unsigned long long kWaitTicks = 20ull * 100000000ull;

// rec (may be null): the first wait to time out records [1, who, what, the
// flag's value], for the host's error message.
__device__ __forceinline__ void wait_flag(const int* flag, int gen, int* err, int* rec = nullptr, int who = 0,
                                          int what = 0) {
  int it = 0;
  unsigned long long t0 = 0;
  while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != gen) {
    if ((++it & 1023) == 0) {
      if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
      const unsigned long long now = __builtin_amdgcn_s_memrealtime();
      if (t0 == 0) {
        t0 = now;
      } else if (now - t0 > kWaitTicks) {
        if (rec && atomicCAS(&rec[0], 0, 1) == 0) {
          rec[1] = who;
          rec[2] = what;
          rec[3] = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        atomicOr(err, 1);
        break;
      }
    }
    __builtin_amdgcn_s_sleep(1);
  }
}


// --------------------------------------------- dataflow (tile) Cholesky
// Left-looking Cholesky of an n x n matrix (n = 64 nt) in one launch.
//
// Ticket 0 is the walker: one workgroup that runs the serial chain down the
// diagonal by itself.  For column j it takes the partial sum of tile (j,j)
// (all updates but the last), subtracts the last update L_{j,j-1} L_{j,j-1}^T
// from the tile it computed one column earlier and still has in LDS,
// factors the tile (diag_factor64, which also forms the 64x64 inverse),
// publishes the inverse, and turns the partial sum of tile (j+1,j) into
// L_{j+1,j} by forward substitution with the factor's 16x16 blocks.  No
// hand-off between workgroups sits on the diagonal chain.
//
// Tickets 1.. are the lower tiles (i,j), one workgroup each: first the
// early tiles (c,c), (c+1,c), (c+2,c) of columns 0..kAhead-1, then for each
// column j the early tiles of column j + kAhead followed by column j's other
// tiles (rows j+3..).  The early tiles thus start kAhead columns before the
// walker needs them and take their terms as they are published, instead of
// running a long accumulation at the end: (c,c) and (c+1,c) are the walker's
// partial sums, and (c+2,c) feeds the last term of partial tile (c+2,c+1),
// which the walker needs one column later.  A task keeps its tile in MFMA
// accumulators and subtracts
// L_ik L_jk^T for every earlier column k as soon as tiles (i,k) and (j,k)
// are published.  Tiles (j,j) and (j+1,j) stop there and publish their
// partial sums for the walker (the diagonal one without the k = j-1 term);
// every other tile waits for the walker's diagonal inverse and solves
// L_ij = A_ij L_jj^-T as a product with it.
//
// Hand-off: the producer writes its tile through to the device's coherence
// point (wt_store), every wave waits for its stores, and after a barrier
// one thread stores the launch's generation into the tile's flag; the
// consumer spins on the flag and reads the tile with agent-scope loads (no
// cache-wide fence on either side).  The walker waits only for the two
// partial tiles of the column it is on.  Other tiles wait only for lower
// tickets or for the walker; early tiles wait for other tiles, some of
// higher tickets, but at any time only the early tiles within kAhead columns of
// the walker's can be waiting, so the other tiles have workgroups to run on as
// long as kDagBeside of them are resident beside the walker.  Every wait is
// bounded.
constexpr int kDagStage = 2 * 8192;  // two staged terms of two 64x64 tiles
constexpr int kDiagDoubles = (sizeof(DiagSmem) + 15) / 16 * 2;  // the walker's share, 16-byte aligned
constexpr int kDagSmemDoubles = kDiagDoubles > kDagStage ? kDiagDoubles : kDagStage;
static_assert(kDagStage <= kDagSmemDoubles && 2 * 64 * 66 <= kDagSmemDoubles, "staging fits the shared buffer");

struct DagArgs {
  double* A;
  int ld, nt;
  double* dinv;  // nt inverted 64x64 diagonal factors, column-major
  double* part;  // 2 nt partial tiles (part_at): (j,j) at 2j, (j+1,j), transposed, at 2j+1;
                 // then (with X) the transposed diagonal blocks of X, ns tiles
  int* sync;     // [0] ticket, [1] error word, [2, 2+nt*nt) tile flags, then 2 nt partial
                 // flags, then (with X) ns*ns flags of X's tiles
  int gen;
  int nfac;      // the factorization's tickets after the walker's
  int* info;
  int* rec;      // the first timed-out wait: [1, ticket, flag index, flag value]
  // optional: X = inv(L_S) of the trailing block L_S (tiles s0..nt-1, ns = nt - s0
  // of them) into X (leading dimension ldx), formed in the same launch; s0 < 0: none
  int s0;
  double* X;
  int ldx;
};

// a 64x64 tile (column-major, leading dimension ld) <-> MFMA accumulator
// layout; Published: a tile written by another workgroup of the launch
// (agent-scope loads)
template <bool Published = false>
__device__ __forceinline__ void tile_load(v4d (&acc)[2][2], const double* src, size_t ld) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const double* e = src + (size_t)(wm + 16 * bm + (lane >> 4) + 4 * v) + (size_t)(wn + 16 * bn + (lane & 15)) * ld;
        acc[bm][bn][v] = Published ? wt_load(e) : *e;
      }
}

// The columns of a solved tile in registers: waves 0, 1 have the 16-column
// blocks 0 and 3, waves 2, 3 the blocks 1 and 2 (elsewhere 0, 1 and 2, 3).
template <bool SOLVED>
__device__ __forceinline__ int tile_col(int wave, int bn) {
  return 16 * (SOLVED ? (bn ? 3 - (wave >> 1) : wave >> 1) : 2 * (wave >> 1) + bn);
}
// the transpose of a 64x64 tile into accumulator layout
__device__ __forceinline__ void tile_load_t(v4d (&acc)[2][2], const double* src, size_t ld) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        acc[bm][bn][v] = src[(size_t)(wn + 16 * bn + (lane & 15)) + (size_t)(wm + 16 * bm + (lane >> 4) + 4 * v) * ld];
}
// The walker's partial tiles are kept as it loads them: 16x16 block (rb, cb) in
// MFMA layout, register v of the lanes in lane order at part_at(rb, cb, v), so
// that a store or load is 512 bytes in a row (as a matrix, 16 pieces of 32: the
// stores of a tile then took 2.3 us, on the chain).
__device__ __forceinline__ int part_at(int rb, int cb, int v) { return ((4 * rb + cb) * 4 + v) * 64; }
__device__ __forceinline__ void part_store(const v4d (&acc)[2][2], double* dst) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        wt_store(dst + part_at(2 * (wave & 1) + bm, 2 * (wave >> 1) + bn, v) + lane, acc[bm][bn][v]);
}

template <bool SOLVED>
__device__ __forceinline__ void tile_store_direct(const v4d (&acc)[2][2], double* dst, size_t ld) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 32;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        wt_store(dst + (size_t)(wm + 16 * bm + (lane >> 4) + 4 * v) + (size_t)(tile_col<SOLVED>(wave, bn) + (lane & 15)) * ld,
                 acc[bm][bn][v]);
}

// the transpose of a tile held in accumulator layout, written through
template <bool SOLVED>
__device__ __forceinline__ void tile_store_direct_t(const v4d (&acc)[2][2], double* dst, size_t ld) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 32;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        wt_store(dst + (size_t)(tile_col<SOLVED>(wave, bn) + (lane & 15)) + (size_t)(wm + 16 * bm + (lane >> 4) + 4 * v) * ld,
                 acc[bm][bn][v]);
}

__device__ __forceinline__ void tile_negate(v4d (&acc)[2][2]) {
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn) acc[bm][bn] = -acc[bm][bn];
}

// The MFMA operands of eight 4-deep steps of a staged pair (T1 at the buffer,
// T2 4096 doubles on), and their products.  Half h of a term is steps 8h..8h+7.
struct HalfOps {
  double a0[8], a1[8], b0[8], b1[8];
};
// where this lane's operands of an even step (T1's two row blocks, T2's) lie
// in a buffer; odd steps' columns have the same parity, so one offset serves
// all steps: step st is 256 st doubles on
struct HalfAt {
  int a0, a1, b0, b1;
};
__device__ __forceinline__ HalfAt half_at() {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32, m = lane & 15, kq = lane >> 4;
  return {staged(wm + m, kq), staged(wm + 16 + m, kq), 4096 + staged(wn + m, kq), 4096 + staged(wn + 16 + m, kq)};
}
__device__ __forceinline__ void half_read(HalfOps& o, const HalfAt& at, int u, int h, const double* buf) {
  const double* b = buf + 256 * (8 * h + u);
  o.a0[u] = b[at.a0];
  o.a1[u] = b[at.a1];
  o.b0[u] = b[at.b0];
  o.b1[u] = b[at.b1];
}
__device__ __forceinline__ void half_mfma(v4d (&nacc)[2][2], const HalfOps& o, int u) {
  nacc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a0[u], o.b0[u], nacc[0][0], 0, 0, 0);
  nacc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a0[u], o.b1[u], nacc[0][1], 0, 0, 0);
  nacc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a1[u], o.b0[u], nacc[1][0], 0, 0, 0);
  nacc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a1[u], o.b1[u], nacc[1][1], 0, 0, 0);
}
// the tiles of one term
struct TermSrc {
  const double *p1, *p2;
  int ld1, ld2;
};
// one half's products.  Between each step's MFMAs go one step's reads of the
// next half's operands (half hnext of the term at rd) and, with ST, two loads
// of a later term's tiles t1, t2 into wr: bunched in front, either would leave
// the matrix cores idle behind them (the fence keeps them where they are).
// The restrict pointers tell the compiler that the reads of rd may pass the
// loads into wr.
template <bool ST>
__device__ __forceinline__ void half_product(v4d (&nacc)[2][2], const HalfOps& use, HalfOps& next, const HalfAt& at,
                                             int hnext, const double* __restrict__ rd, const double* __restrict__ t1,
                                             int ld1, const double* __restrict__ t2, int ld2,
                                             double* __restrict__ wr) {
  unsigned at1 = 0, at2 = 0;
  if (ST) {
    at1 = stage_at(ld1);
    at2 = stage_at(ld2);
  }
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    half_read(next, at, u, hnext, rd);
    if (ST) {
      stage_load(t1, ld1, at1, u, wr);
      stage_load(t2, ld2, at2, u, wr + 4096);
    }
    half_mfma(nacc, use, u);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The terms of a task's accumulation, kbeg <= k < kend (wave-uniform): T1_k and
// T2_k are the 64x64 tiles 64 k columns after p1 and p2 (leading dimensions ld1,
// ld2; T1 of the first term is at first1, ldf), and their flags lie at
// f1 + k fs1 and f2 + k fs2.
struct Terms {
  int kbeg, kend;
  const double *first1, *p1, *p2;
  int ldf, ld1, ld2;
  int f1, fs1, f2, fs2;
};

// acc -= sum_{kbeg <= k < kend} T1_k T2_k^T, each term once both of its tiles
// are published.
//
// Terms go through two LDS buffers of 2 x 64 x 64 doubles.  A term is two
// halves of eight 4-deep steps, whose operands are read from LDS one half
// ahead of their MFMAs, so that with one wave on each SIMD the matrix cores
// wait neither for LDS nor for the term's one barrier.  That barrier is in
// the middle of the term: by then every wave has read the whole term, so its
// buffer takes the loads of the term after next, and the next term's loads,
// issued one term ago, have landed.
// Which terms are published is found 64 at a time, one lane per term (a
// scan of one flag pair at a time costs about a microsecond of memory
// latency per term), and the next scan's loads are in flight during a half.
// N = 997 (11N = 10967, one factorisation of each order): 16.3 -> 13.6 ms; N = 4096: 981 -> 811 ms; N = 512:
// 3.22 -> 3.03 ms.  From N ~ 550 on the tile reads bound it, 64 KB a term, L2 misses at
// 5.2 TB/s: 2.4 of an 11N launch's 2.4 ms at N = 576 (1.7 of 1.8 at 512, 0.8 of 1.15 at 400).
__device__ __forceinline__ void pair_accumulate(v4d (&acc)[2][2], const Terms& T, const int* flags, int gen, int* err,
                                                double* smem, int* rec, int who) {
  const int kbeg = T.kbeg, kend = T.kend;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int* kready_x = reinterpret_cast<int*>(smem + kDagSmemDoubles) + 1;  // the scans' result by the term's parity;
                                                                       // [2] the blocking wait's
  if (kend <= kbeg) return;
  int kready = kbeg;  // every term before it is known to be published
  auto load = [&](int f) { return __hip_atomic_load(&flags[f], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  // the first unpublished term from k on, of those that lane l's answer ok covers (term k + l)
  auto first_not = [&](int k, bool ok) {
    const unsigned long long no = ~__ballot(ok);
    return k + (no ? __builtin_ctzll(no) : 64);
  };
  // waits for term k; takes the later ones that are already published too
  auto ready = [&](int k) {
    if (wave == 0) {
      bool ok = false;
      if (k + lane < kend) {
        const int v1 = load(T.f1 + (k + lane) * T.fs1), v2 = load(T.f2 + (k + lane) * T.fs2);
        ok = v1 == gen && v2 == gen;
      }
      int kk = first_not(k, ok);
      if (kk == k) {
        const int f1 = T.f1 + k * T.fs1, f2 = T.f2 + k * T.fs2;
        if (lane == 0) {
          wait_flag(&flags[f1], gen, err, rec, who, f1);
          wait_flag(&flags[f2], gen, err, rec, who, f2);
        }
        kk = k + 1;
      }
      if (lane == 0) kready_x[2] = kk;
    }
    __syncthreads();
    kready = __builtin_amdgcn_readfirstlane(kready_x[2]);
    wt_seen();
  };
  auto term = [&](int k) {
    const bool first = k == kbeg;
    return TermSrc{first ? T.first1 : T.p1 + (size_t)(64 * k) * T.ld1, T.p2 + (size_t)(64 * k) * T.ld2,
                   first ? T.ldf : T.ld1, T.ld2};
  };
  auto buffer = [&](int k) { return smem + ((k - kbeg) & 1) * 8192; };
  const HalfAt at = half_at();
  HalfOps P, Q;
  int issued;  // terms before it are staged or on their way
  // waits for term k, stages it and reads its first half
  auto restart = [&](int k) {
    ready(k);
    const TermSrc t = term(k);
    stage_tile(t.p1, t.ld1, buffer(k));
    stage_tile(t.p2, t.ld2, buffer(k) + 4096);
    issued = k + 1;
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    gemm_barrier();
#pragma unroll
    for (int u = 0; u < 8; ++u) half_read(P, at, u, 0, buffer(k));
  };
  // a half's products with the loads of the next term not yet issued, when it is published
  auto half = [&](const HalfOps& use, HalfOps& next, int hnext, const double* rd, double* wr) {
    if (issued < kready) {
      const TermSrc t = term(issued);
      half_product<true>(acc, use, next, at, hnext, rd, t.p1, t.ld1, t.p2, t.ld2, wr);
      ++issued;
    } else {
      half_product<false>(acc, use, next, at, hnext, rd, nullptr, 0, nullptr, 0, wr);
    }
  };
  tile_negate(acc);  // the terms add to the negated tile (exact: negation commutes with rounding)
  restart(kbeg);
  for (int k = kbeg; k < kend; ++k) {
    // the known published terms run out: the next scan's loads
    const bool scan = kready < kend && kready <= k + 2;
    int v1 = gen, v2 = gen;
    if (scan) {
      const int kk = min(kready + lane, kend - 1);
      v1 = load(T.f1 + kk * T.fs1);
      v2 = load(T.f2 + kk * T.fs2);
    }
    // (term k+1's loads go out here only after a restart; else they are a half older)
    if (issued == k + 1) half(P, Q, 1, buffer(k), buffer(k + 1));
    else half_product<false>(acc, P, Q, at, 1, buffer(k), nullptr, 0, nullptr, 0, buffer(k + 1));
    if (k + 1 == kend) {
#pragma unroll
      for (int u = 0; u < 8; ++u) half_mfma(acc, Q, u);
      break;
    }
    __builtin_amdgcn_s_waitcnt(kWaitVm0);  // this wave's share of term k+1 has landed
    if (scan) {
      asm volatile("" : "+v"(v1), "+v"(v2));  // (compared here, not where they were loaded)
      const int kk = first_not(kready, kready + lane < kend && v1 == gen && v2 == gen);
      if (threadIdx.x == 0) kready_x[k & 1] = kk;
    }
    gemm_barrier();
    if (scan) {
      kready = __builtin_amdgcn_readfirstlane(kready_x[k & 1]);
      wt_seen();
    }
    if (issued <= k + 1) {
#pragma unroll
      for (int u = 0; u < 8; ++u) half_mfma(acc, Q, u);
      restart(k + 1);
    } else {
      half(Q, P, 0, buffer(k + 1), buffer(k));
    }
  }
  tile_negate(acc);
  __syncthreads();  // the staging buffers are free again
}

// ------------------------------------------------ macro tasks (large matrices)
// A macro task is two block rows by two block columns of the factor, a 128x128
// tile, accumulated as one: each wave keeps a 64x64 tile of it.  A 64-deep term
// of four tiles then moves 128 KB into LDS where four single tiles move 256 KB,
// and from N ~ 550 on those reads (L2 misses, 5.2 TB/s) are what bounds the
// single-tile tasks.  A term is two 32-column halves through two LDS buffers;
// an 8-step half keeps the matrix cores busy for 8192 cycles, its one barrier
// is before its last step, and each step's operands are read during the step
// before it.  Both factorisations of a step: N = 4096 815 -> 617 ms (57 TF/s),
// N = 2048 99 -> 83 ms.
struct MacroOps {
  double a[4], b[4];
};
// a lane's operands of step 0 in a buffer (T1's 128 rows x 32 columns, then T2's, laid out as stage_macro does)
struct MacroAt {
  int a[4], b[4];
};
__device__ __forceinline__ MacroAt macro_at() {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, kq = lane >> 4, swap = (kq & 1) << 4;
  MacroAt at;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    at.a[q] = kq * 128 + ((64 * (wave & 1) + 16 * q + m) ^ swap);
    at.b[q] = 4096 + kq * 128 + ((64 * (wave >> 1) + 16 * q + m) ^ swap);
  }
  return at;
}
// a quarter of the reads, and of a step's products (its 16 MFMAs by rows)
__device__ __forceinline__ void macro_read(MacroOps& o, const MacroAt& at, int u, int q, const double* buf) {
  const double* b = buf + 512 * u;
  o.a[q] = b[at.a[q]];
  o.b[q] = b[at.b[q]];
}
__device__ __forceinline__ void macro_mfma(v4d (&nacc)[4][4], const MacroOps& o, int bm) {
#pragma unroll
  for (int bn = 0; bn < 4; ++bn)
    nacc[bm][bn] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[bm], o.b[bn], nacc[bm][bn], 0, 0, 0);
}
// this wave's q-th (of 8) direct load of a 128x32 chunk: column 8 wave + q, its
// 16-row blocks swapped in pairs on odd columns (as staged())
__device__ __forceinline__ void macro_load(const double* p, int ld, int lane, int q, double* dst) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = 8 * wave + q;
  const unsigned at = 2 * (lane ^ ((q & 1) << 3));
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p + (size_t)c * ld + at),
                                   (__attribute__((address_space(3))) void*)(dst + c * 128), 16, 0, kCpolSc1);
}
// steps 0..6 of the half at rd (its step 0 in P; step 7 is left in Q), with the
// loads of the next half into wr (ST): two reads and, in the first four steps,
// one load between every four MFMAs.  (All 16 loads in front of the half's
// products, the matrix cores idle until they are issued: N = 4096's step took
// 993 ms so, 934 with eight in each of two steps, 924 with four in each of four.)
template <bool ST>
__device__ __forceinline__ void macro_half(v4d (&nacc)[4][4], MacroOps& P, MacroOps& Q, const MacroAt& at,
                                           const double* __restrict__ rd, const double* __restrict__ t1,
                                           const double* __restrict__ t2, int ld, double* __restrict__ wr) {
  const int lane = ST ? opaque_tid() & 63 : 0;
#pragma unroll
  for (int u = 0; u < 7; ++u)
#pragma unroll
    for (int bm = 0; bm < 4; ++bm) {
      macro_read(u & 1 ? P : Q, at, u + 1, bm, rd);
      if (ST && u < 4) macro_load(bm & 1 ? t2 : t1, ld, lane, 2 * u + (bm >> 1), bm & 1 ? wr + 4096 : wr);
      macro_mfma(nacc, u & 1 ? Q : P, bm);
      __builtin_amdgcn_sched_barrier(0);
    }
}

// nacc += sum_{k < kend} T1_k T2_k^T, T1_k the 128 rows at p1 + 64 k ld (block
// rows i0, i0 + 1 of the factor), T2_k those at p2 (block rows j0, j0 + 1); each
// term once its four tiles are published
__device__ __forceinline__ void macro_accumulate(v4d (&nacc)[4][4], int kend, const double* p1, const double* p2, int ld,
                                                 int nt, int i0, int j0, const int* flags, int gen, int* err,
                                                 double* smem, int* rec, int who) {
  if (kend <= 0) return;
  const int lane = opaque_tid() & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int* kready_x = reinterpret_cast<int*>(smem + kDagSmemDoubles) + 1;
  int kready = 0;
  auto load = [&](int f) { return __hip_atomic_load(&flags[f], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  auto first_not = [&](int k, bool ok) {
    const unsigned long long no = ~__ballot(ok);
    return k + (no ? __builtin_ctzll(no) : 64);
  };
  auto ready = [&](int k) {
    if (wave == 0) {
      bool ok = false;
      if (k + lane < kend) {
        const int c = nt * (k + lane);
        const int v1 = load(i0 + c), v2 = load(i0 + 1 + c), v3 = load(j0 + c), v4 = load(j0 + 1 + c);
        ok = v1 == gen && v2 == gen && v3 == gen && v4 == gen;
      }
      int kk = first_not(k, ok);
      if (kk == k) {
        if (lane == 0) {
          const int c = nt * k;
          for (int f : {i0 + c, i0 + 1 + c, j0 + c, j0 + 1 + c}) wait_flag(&flags[f], gen, err, rec, who, f);
        }
        kk = k + 1;
      }
      if (lane == 0) kready_x[2] = kk;
    }
    __syncthreads();
    kready = __builtin_amdgcn_readfirstlane(kready_x[2]);
    wt_seen();
  };
  auto buffer = [&](int h) { return smem + (h & 1) * 8192; };
  const MacroAt at = macro_at();
  MacroOps P, Q;
  int issued;  // halves before it are staged or on their way
  auto restart = [&](int h) {
    ready(h >> 1);
    const size_t col = (size_t)(32 * h) * ld;
    const int ln = opaque_tid() & 63;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      macro_load(p1 + col, ld, ln, q, buffer(h));
      macro_load(p2 + col, ld, ln, q, buffer(h) + 4096);
    }
    issued = h + 1;
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    gemm_barrier();
#pragma unroll
    for (int q = 0; q < 4; ++q) macro_read(P, at, 0, q, buffer(h));
  };
  auto last_step = [&] {
#pragma unroll
    for (int q = 0; q < 4; ++q) macro_mfma(nacc, Q, q);
  };
  restart(0);
  const int halves = 2 * kend;
  for (int h = 0; h < halves; ++h) {
    const bool scan = kready < kend && kready <= (h >> 1) + 2;
    int v1 = gen, v2 = gen, v3 = gen, v4 = gen;
    if (scan) {
      const int c = nt * min(kready + lane, kend - 1);
      v1 = load(i0 + c);
      v2 = load(i0 + 1 + c);
      v3 = load(j0 + c);
      v4 = load(j0 + 1 + c);
    }
    if (issued == h + 1 && h + 1 < halves && (h + 1) >> 1 < kready) {
      const size_t col = (size_t)(32 * (h + 1)) * ld;
      macro_half<true>(nacc, P, Q, at, buffer(h), p1 + col, p2 + col, ld, buffer(h + 1));
      issued = h + 2;
    } else {
      macro_half<false>(nacc, P, Q, at, buffer(h), nullptr, nullptr, 0, buffer(h + 1));
    }
    if (h + 1 == halves) {
      last_step();
      break;
    }
    __builtin_amdgcn_s_waitcnt(kWaitVm0);  // this wave's share of half h+1 has landed
    if (scan) {
      asm volatile("" : "+v"(v1), "+v"(v2), "+v"(v3), "+v"(v4));  // (compared here, not where they were loaded)
      const int kk = first_not(kready, kready + lane < kend && v1 == gen && v2 == gen && v3 == gen && v4 == gen);
      if (threadIdx.x == 0) kready_x[h & 1] = kk;
    }
    gemm_barrier();
    if (scan) {
      kready = __builtin_amdgcn_readfirstlane(kready_x[h & 1]);
      wt_seen();
    }
    if (issued <= h + 1) {
      last_step();
      restart(h + 1);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        macro_read(P, at, 0, q, buffer(h + 1));
        macro_mfma(nacc, Q, q);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  __syncthreads();  // the staging buffers are free again
}

// LDS of a macro task's end: a 128x64 block by columns (Cs[kk][m], m < 128),
// then a staged 64x64 tile.  A wave owns rows 32 wave..32 wave + 31 of the block.
constexpr int kMacroLd = 130;
static_assert(64 * kMacroLd + 4096 <= kDagSmemDoubles, "a macro task's end fits the shared buffer");
// acc += C T^T for this wave's 32 rows of the block in Cs and the staged tile T
__device__ __forceinline__ void macro_rows_product(v4d (&acc)[2][4], const double* Cs, const double* T) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6, m = lane & 15;
#pragma unroll
  for (int st = 0; st < 16; ++st) {
    const int kr = 4 * st + (lane >> 4);
    const double a0 = Cs[kr * kMacroLd + 32 * wave + m], a1 = Cs[kr * kMacroLd + 32 * wave + 16 + m];
#pragma unroll
    for (int bn = 0; bn < 4; ++bn) {
      const double b = T[staged(16 * bn + m, kr)];
      acc[0][bn] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b, acc[0][bn], 0, 0, 0);
      acc[1][bn] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b, acc[1][bn], 0, 0, 0);
    }
  }
}
// this wave's rows of the block, accumulator layout <-> Cs; sign: of what is written
__device__ __forceinline__ void macro_rows_put(const v4d (&x)[2][4], double* Cs, double sign) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 4; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        Cs[(16 * bn + (lane & 15)) * kMacroLd + 32 * wave + 16 * bm + (lane >> 4) + 4 * v] = sign * x[bm][bn][v];
  wave_lds_order();
}
// this wave's rows of the block in Cs out to dst (written through), 256-byte column pieces
__device__ __forceinline__ void macro_rows_store(const double* Cs, double* dst, size_t ld) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int it = 0; it < 16; ++it) {
    const int c = 4 * it + (lane >> 4), r = 32 * wave + 2 * (lane & 15);
    const double2 x = *reinterpret_cast<const double2*>(&Cs[c * kMacroLd + r]);
    wt_store(dst + (size_t)r + (size_t)c * ld, x.x);
    wt_store(dst + (size_t)r + 1 + (size_t)c * ld, x.y);
  }
}

// The macro task (I, J): block rows 2I, 2I + 1 of block columns 2J, 2J + 1
__device__ __forceinline__ void macro_task(const DagArgs& g, int I, int J, int t, double* __restrict__ smem) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6, nt = g.nt, ld = g.ld;
  const int i0 = 2 * I, j0 = 2 * J;
  int* err = g.sync + 1;
  int* flags = g.sync + 2;
  double* tile = g.A + 64 * i0 + (size_t)(64 * j0) * ld;
  double* Cs = smem;
  double* Dj = smem + 64 * kMacroLd;
  v4d d1[2][4];  // this wave's rows of the second block column, negated
  {
    const int wm = 64 * (wave & 1), wn = 64 * (wave >> 1);
    v4d acc[4][4];  // negated: the terms add to it
#pragma unroll
    for (int bm = 0; bm < 4; ++bm)
#pragma unroll
      for (int bn = 0; bn < 4; ++bn)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc[bm][bn][v] = -tile[(size_t)(wm + 16 * bm + (lane >> 4) + 4 * v) +
                                 (size_t)(wn + 16 * bn + (lane & 15)) * ld];
    macro_accumulate(acc, j0, g.A + 64 * i0, g.A + 64 * j0, ld, nt, i0, j0, flags, g.gen, err, smem, g.rec, t);
    // the two block columns through Cs, from a 64x64 tile a wave to 32 rows a wave
    auto put = [&](double sign) {
#pragma unroll
      for (int bm = 0; bm < 4; ++bm)
#pragma unroll
        for (int bn = 0; bn < 4; ++bn)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            Cs[(16 * bn + (lane & 15)) * kMacroLd + wm + 16 * bm + (lane >> 4) + 4 * v] = sign * acc[bm][bn][v];
    };
    if (wave >> 1) put(1.0);
    __syncthreads();
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
      for (int bn = 0; bn < 4; ++bn)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          d1[bm][bn][v] = Cs[(16 * bn + (lane & 15)) * kMacroLd + 32 * wave + 16 * bm + (lane >> 4) + 4 * v];
    __syncthreads();
    if (!(wave >> 1)) put(-1.0);
  }
  // a published tile into Dj, once its flag is up (and every wave is past its
  // use of Dj and, the first time, has written Cs)
  auto fetch = [&](int f, const double* src, int sld) {
    if (tid == 0) wait_flag(&flags[f], g.gen, err, g.rec, t, f);
    __syncthreads();
    wt_seen();
    stage_tile(src, sld, Dj);
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
  };
  auto publish = [&](int j) {
    wt_stores_done();
    __syncthreads();
    if (tid == 0) {
      wt_publish(&flags[i0 + nt * j], g.gen);
      wt_publish(&flags[i0 + 1 + nt * j], g.gen);
    }
  };
  v4d out[2][4];
  auto clear = [&] {
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
      for (int bn = 0; bn < 4; ++bn) out[bm][bn] = (v4d){0.0, 0.0, 0.0, 0.0};
  };
  // L of the first block column
  fetch(j0 + nt * j0, g.dinv + (size_t)j0 * 4096, 64);
  clear();
  macro_rows_product(out, Cs, Dj);
  wave_lds_order();
  macro_rows_put(out, Cs, 1.0);
  macro_rows_store(Cs, tile, ld);
  publish(j0);
  // its term of the second, and L of that
  fetch(j0 + 1 + nt * j0, g.A + 64 * (j0 + 1) + (size_t)(64 * j0) * ld, ld);
  macro_rows_product(d1, Cs, Dj);
  wave_lds_order();
  macro_rows_put(d1, Cs, -1.0);
  fetch(j0 + 1 + nt * (j0 + 1), g.dinv + (size_t)(j0 + 1) * 4096, 64);
  clear();
  macro_rows_product(out, Cs, Dj);
  wave_lds_order();
  macro_rows_put(out, Cs, 1.0);
  macro_rows_store(Cs, tile + (size_t)64 * ld, ld);
  publish(j0 + 1);
}

// Column blocks C0 < C1 of out = C Dinv^T for this wave's 32 rows: Dinv^T is zero
// below its block diagonal, so block c takes the k-steps 0 .. 4c+3 only, 40
// products a wave instead of 64.
template <int C0, int C1>
__device__ __forceinline__ void trsm_product(v4d (&out)[2][2], const double (*Cs)[66], const double* Dj, int wm, int lane) {
  constexpr int S0 = 4 * (C0 + 1), S1 = 4 * (C1 + 1);
  double a0[S1], a1[S1], b0[S0], b1[S1];  // every step's operands read ahead of the MFMAs
#pragma unroll
  for (int st = 0; st < S1; ++st) {
    const int kr = 4 * st + (lane >> 4);
    a0[st] = Cs[kr][wm + (lane & 15)];
    a1[st] = Cs[kr][wm + 16 + (lane & 15)];
    if (st < S0) b0[st < S0 ? st : 0] = Dj[staged(16 * C0 + (lane & 15), kr)];
    b1[st] = Dj[staged(16 * C1 + (lane & 15), kr)];
  }
#pragma unroll
  for (int st = 0; st < S1; ++st) {
    if (st < S0) {
      out[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[st], b0[st < S0 ? st : 0], out[0][0], 0, 0, 0);
      out[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[st], b0[st < S0 ? st : 0], out[1][0], 0, 0, 0);
    }
    out[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[st], b1[st], out[0][1], 0, 0, 0);
    out[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[st], b1[st], out[1][1], 0, 0, 0);
  }
}
// out = acc Dinv^T, Dinv a column-major lower triangular 64x64 tile in global memory (out's columns: tile_col<true>)
__device__ __forceinline__ void tile_trsm(const v4d (&acc)[2][2], const double* __restrict__ Dg, double* smem,
                                          v4d (&out)[2][2]) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  // Cs[kk][m] = acc(m, kk); Dinv staged, so that element (n, kk) = Dinv^T(kk, n)
  double(*Cs)[66] = reinterpret_cast<double(*)[66]>(smem);
  double* Dj = smem + 64 * 66;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v) Cs[wn + 16 * bn + (lane & 15)][wm + 16 * bm + (lane >> 4) + 4 * v] = acc[bm][bn][v];
  stage_tile(Dg, 64, Dj);
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
  __syncthreads();
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn) out[bm][bn] = (v4d){0.0, 0.0, 0.0, 0.0};
  if (wave >> 1) trsm_product<1, 2>(out, Cs, Dj, wm, lane);
  else trsm_product<0, 3>(out, Cs, Dj, wm, lane);
  __syncthreads();
}

// tile store through LDS, so each column is written contiguously; written
// through, every wave's stores complete at the closing barrier
__device__ __forceinline__ void tile_store(const v4d (&out)[2][2], double* dst, int ld, double* smem) {
  const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 32;
  double(*Cs)[66] = reinterpret_cast<double(*)[66]>(smem);
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int v = 0; v < 4; ++v) Cs[tile_col<true>(wave, bn) + (lane & 15)][wm + 16 * bm + (lane >> 4) + 4 * v] = out[bm][bn][v];
  __syncthreads();
  for (int idx = tid; idx < 4096; idx += 256) {
    const int r = idx & 63, c = idx >> 6;
    wt_store(dst + (size_t)r + (size_t)c * ld, Cs[c][r]);
  }
  wt_stores_done();
  __syncthreads();
}

// The walker's tile (j+1,j+1) by 16x16 blocks on and below the diagonal, three
// on waves 0 and 3 and two on waves 1 and 2, in MFMA layout: waves 0 and 3 have
// (B+1,B), (B+1,B+1), (B,B) with B = 0, 2; waves 1 and 2 (R,0), (R,1) with R = 2, 3.
struct DiagBlocks {
  v4d b[3];
};
__device__ __forceinline__ bool diag_three(int wave) { return wave == 0 || wave == 3; }
__device__ __forceinline__ int diag_block_row(int wave, int n) { return diag_three(wave) ? (wave & 2) + (n < 2) : 1 + wave; }
__device__ __forceinline__ int diag_block_col(int wave, int n) { return diag_three(wave) ? (wave & 2) + (n == 1) : n; }
__device__ __forceinline__ int diag_block_count(int wave) { return diag_three(wave) ? 3 : 2; }
__device__ __forceinline__ void diag_blocks_load(DiagBlocks& t, const double* src) {
  const int tid = opaque_tid(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
  for (int n = 0; n < 3; ++n)
    if (n < diag_block_count(wave)) {
      const double* e = src + part_at(diag_block_row(wave, n), diag_block_col(wave, n), 0) + lane;
#pragma unroll
      for (int v = 0; v < 4; ++v) t.b[n][v] = wt_load(e + 64 * v);
    }
}

// t -= X X^T for X = L_{j+1,j} (transposed in T).  halfway() runs after half of
// the products, store(0) .. store(15) between the others (a store is issued while
// the matrix core is busy; one behind the other the sixteen take as long as the
// products).
template <class Store, class Halfway>
__device__ __forceinline__ void column_syrk(DiagBlocks& t, const DiagSmem& sm, Store&& store, Halfway&& halfway) {
  const int tid = opaque_tid(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
  for (int n = 0; n < 3; ++n) t.b[n] = -t.b[n];  // adds the products to the negated blocks (exact)
  const bool three = diag_three(wave);
  const double* k0 = &sm.T[lane >> 4][lane & 15];
  const int oq = 16 * diag_block_row(wave, 0), op = 16 * diag_block_col(wave, 0), oy1 = 16 * diag_block_col(wave, 1);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    double x[8], y[8], y1[8];
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const double* k = k0 + 4 * 66 * (8 * h + st);
      x[st] = k[oq], y[st] = k[op], y1[st] = k[oy1];
    }
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      t.b[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[st], y[st], t.b[0], 0, 0, 0);
      t.b[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[st], y1[st], t.b[1], 0, 0, 0);
      if (three) t.b[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[st], y[st], t.b[2], 0, 0, 0);
      if (h == 1) {
        __builtin_amdgcn_sched_barrier(0);
        store(2 * st);
        store(2 * st + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (h == 0) {
      __builtin_amdgcn_sched_barrier(0);
      halfway();
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int n = 0; n < 3; ++n) t.b[n] = -t.b[n];
}

// The walker's L_{j+1,j} = P L_jj^-T for this wave's rows 16w.., transposed and in
// registers (S: P^T, then L^T): column block c's L_c^T = X_cc S_c^T, then S_c' -=
// L_c L_c'c^T for c' > c, with the operands read ahead and the independent
// products interleaved.
__device__ __forceinline__ void rows_solve(v4d (&S)[4], const DiagSmem& sm, int lane) {
  const int r = lane & 15, kq = lane >> 4;
  double xa[4][4], la[4][4][4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      xa[c][kb] = sm.Xs[16 * c + r][16 * c + 4 * kb + kq];
#pragma unroll
      for (int e = c + 1; e < 4; ++e) la[c][e][kb] = sm.P[c][16 * e + r][4 * kb + kq];
    }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    v4d x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) x = __builtin_amdgcn_mfma_f64_16x16x4f64(xa[c][kb], S[c][kb], x, 0, 0, 0);
    S[c] = x;
    const v4d n = -x;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int e = c + 1; e < 4; ++e) S[e] = __builtin_amdgcn_mfma_f64_16x16x4f64(la[c][e][kb], n[kb], S[e], 0, 0, 0);
  }
}

// The walker (ticket 0; see above).  A column's chain: the tile into rows, four
// panels, L_{j+1,j} and X_33's products, L_{j+1,j} L_{j+1,j}^T.  What is not on it
// is done by the waves that a panel leaves idle.  N = 200: a column takes 14.6 us,
// 8.3 for the panels, 3.2 for L_{j+1,j}, 3.1 for the last update and the stores
// (20.4 before: 14 for the panels and the whole inverse, and then its stores, the
// product with it and the update one after the other).  About as long, 10 us from
// the inverse's publication, takes the next column's partial tile, two hand-offs
// away; doing its last term where the tile before it is solved, one hand-off
// away, needs that workgroup to wait for L_{j+1,j} too and came later (16 us).
// Little is kept in registers over the panels: with the partial tiles loaded and
// L_{j+1,j} begun during them, the copies between the two register files cost
// more (16.9 us) than what they hid.
__device__ __forceinline__ void dag_walker(const DagArgs& g, double* __restrict__ smem) {
  const int nt = g.nt, ld = g.ld;
  double* __restrict__ A = g.A;
  int* err = g.sync + 1;
  int* flags = g.sync + 2;
  int* pflags = g.sync + 2 + nt * nt;
  int* rec = g.rec;  // the first timed-out wait
  // the partial sum of the current diagonal tile, already including the
  // last update (the previous column's L_{j,j-1} L_{j,j-1}^T)
  DiagBlocks acc = {};
  DiagSmem& sm = *reinterpret_cast<DiagSmem*>(smem);
  if (threadIdx.x == 0) {
    sm.ready = 0;
    sm.stored = 0;
    wait_flag(&pflags[0], g.gen, err, rec, 0, nt * nt);
  }
  __syncthreads();
  wt_seen();
  diag_blocks_load(acc, g.part);
  for (int j = 0; j < nt; ++j) {
    const int tid = opaque_tid(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
    for (int n = 0; n < 3; ++n)
      if (n < diag_block_count(wave)) {
        const int r0 = 16 * diag_block_row(wave, n), c0 = 16 * diag_block_col(wave, n);
        blk_store<65>(&sm.R[r0][c0], acc.b[n], 1.0, lane);
      }
    wt_stores_done();  // the previous column's
    __syncthreads();
    double a[16], dg[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      a[q] = sm.R[lane][16 * wave + q];
      dg[q] = sm.R[16 * wave + (lane & 15)][16 * wave + q];
    }
    __builtin_amdgcn_sched_barrier(0);
    // the previous column's L_{j,j-1}: every wave's stores are behind the barrier
    if (j > 0 && tid == 192) wt_publish(&flags[j + nt * (j - 1)], g.gen);
    const double* sub_src = g.part + (size_t)(2 * j + 1) * 4096;
    const double* acc_src = g.part + (size_t)(2 * (j + 1)) * 4096;
    double* dinv = g.dinv + (size_t)j * 4096;
    double* Ljj = A + 64 * j + (size_t)(64 * j) * ld;
    const bool more = j + 1 < nt;
    auto idle = [&](int b) {
      const int lane = opaque_tid() & 63;
      // column j+1's partial tiles: a wave without a panel asks whether both are
      // published, near the end, and tells the others through LDS
      if (more && wave == (b == 3 ? 0 : 3) && b >= 2 && __builtin_amdgcn_readfirstlane(sm.ready) != j + 1) {
        const int there =
            __hip_atomic_load(&pflags[2 * j + 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g.gen &&
            __hip_atomic_load(&pflags[2 * (j + 1)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g.gen;
        if (there && lane == 0) sm.ready = j + 1;
      }
      // what the column has finished leaves while there is time: the factor's
      // columns by the panel's wave, the inverse's rows
      if (b == wave + 1) diag_store_factor(a, dg, Ljj, ld);
      if (b == 3)
        for (int n = wave; n < 32; n += 3) diag_store_inverse(sm, dinv, n >> 4, n & 15, lane);
    };
    v4d S[4];
    auto last = [&] {
      const int lane = opaque_tid() & 63;
      if (more) {
        if (lane == 0 && sm.ready != j + 1) {
          wait_flag(&pflags[2 * j + 1], g.gen, err, rec, 0, nt * nt + 2 * j + 1);
          wait_flag(&pflags[2 * (j + 1)], g.gen, err, rec, 0, nt * nt + 2 * (j + 1));
        }
        wt_seen();
        // (j+1,j) into S, this wave's rows, transposed; (j+1,j+1) into acc
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int v = 0; v < 4; ++v) S[c][v] = wt_load(sub_src + part_at(c, wave, v) + lane);
        diag_blocks_load(acc, acc_src);
      }
#pragma unroll
      for (int n = 0; n < 4; ++n) diag_store_inverse(sm, dinv, 2, 4 * wave + n, lane);
    };
    diag_factor64(a, dg, sm, 64 * j, idle, last);
    if (more) {
      const int lane = opaque_tid() & 63;
      rows_solve(S, sm, lane);
#pragma unroll
      for (int c = 0; c < 4; ++c) blk_store<66>(&sm.T[16 * c][16 * wave], S[c], 1.0, lane);
    }
    __syncthreads();
    if (tid == 0 && sm.bad != 0x7fffffff) atomicMin(g.info, sm.bad);
#pragma unroll
    for (int n = 0; n < 4; ++n) diag_store_inverse(sm, dinv, 3, 4 * wave + n, lane);
    // the inverse is published by the last wave whose stores are complete
    auto stored = [&] {
      if (lane == 0 && atomicAdd(&sm.stored, 1) == 4 * j + 3) wt_publish(&flags[j + nt * j], g.gen);
    };
    if (!more) {
      if (wave == 3) diag_store_factor(a, dg, Ljj, ld);
      wt_stores_done();
      stored();
      break;
    }
    // L_{j+1,j} out (complete at the next column's start)
    double* e0 = Ljj + 64 + 16 * wave + (lane & 15) + (size_t)(lane >> 4) * ld;
    column_syrk(acc, sm, [&](int q) { wt_store(e0 + (size_t)(16 * (q >> 2) + 4 * (q & 3)) * ld, S[q >> 2][q & 3]); }, [&] {
      wt_stores_done();
      stored();
      if (wave == 3) diag_store_factor(a, dg, Ljj, ld);
    });
    // L_{j+1,j} is published at the start of the next column
  }
}

// One tile task of the dataflow Cholesky, t >= 1 (see above).  Returns when the
// task is done.
template <bool MACRO>
__device__ __forceinline__ void dag_task(const DagArgs& g, int t, double* __restrict__ smem) {
  const int tid = threadIdx.x;
  const int nt = g.nt, ld = g.ld;
  double* __restrict__ A = g.A;
  int* err = g.sync + 1;
  int* flags = g.sync + 2;
  int* pflags = g.sync + 2 + nt * nt;
  int* rec = g.rec;  // the first timed-out wait
  v4d acc[2][2];

  // A tile task: the tile (i,j) of the factor, or (past the factorization's
  // tickets) the tile (xi,xj) of X = inv(L_S), I = s0 + xi (see potrf_lower_x)
  const int xf = nt * nt + 2 * nt;  // X's flags, after the partial flags
  const int s0 = g.s0, ns = nt - s0;
  double* X = g.X;
  const int ldx = g.ldx;
  const bool is_x = t > g.nfac;
  int i, j;  // the tile; of X: (xi, xj)
  Terms T;
  if (is_x) {
    const int r = t - g.nfac - 1;
    double* xdT = g.part + (size_t)2 * nt * 4096;   // X_jj^T = Dinv^T of the diagonal blocks
    if (r < ns) {
      // diagonal block j: X_jj = Dinv_J into X (read by the LL^T product after
      // the launch) and its transpose (the first term's operand of block
      // column j)
      const int jj = r, J = s0 + jj;
      if (tid == 0) wait_flag(&flags[J + nt * J], g.gen, err, rec, t, J + nt * J);
      __syncthreads();
      wt_seen();
      tile_load<true>(acc, g.dinv + (size_t)J * 4096, 64);
      tile_store_direct<false>(acc, X + 64 * jj + (size_t)(64 * jj) * ldx, ldx);
      tile_store_direct_t<false>(acc, xdT + (size_t)jj * 4096, 64);
      wt_stores_done();
      __syncthreads();
      if (tid == 0) wt_publish(&flags[xf + jj + ns * jj], g.gen);
      return;
    }
    // tile (xi, xj), xi > xj, in row order: X_ij = -Dinv_I sum_{k=j}^{i-1} L_Ik X_kj
    // (I = s0 + i).  The sum is accumulated transposed, acc = -sum X_kj^T L_Ik^T,
    // from X_kj^T (kept in X's upper block (j,k); X_jj^T in xdT), so that the
    // solve with Dinv_I is tile_trsm's product: X_ij^T = acc Dinv_I^T.
#include "rsd_dag_x.inc"
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
      for (int bn = 0; bn < 2; ++bn) acc[bm][bn] = (v4d){0.0, 0.0, 0.0, 0.0};
    const int I = s0 + i;
    T = Terms{j, i, xdT + (size_t)j * 4096, X + 64 * j, A + 64 * I + (size_t)(64 * s0) * ld,
              64, ldx, ld, xf + ns * j, 1, I + nt * s0, nt};
  } else {
#define MACRO_TASK(I, J)               \
  {                                    \
    macro_task(g, I, J, t, smem);      \
    return;                            \
  }
#include "rsd_dag_tile.inc"
#undef MACRO_TASK
    // (the walker takes the tile (j+1,j) transposed)
    const bool tr = i == j + 1;
    const double* src = A + 64 * i + (size_t)(64 * j) * ld;
    if (tr) tile_load_t(acc, src, ld);
    else tile_load(acc, src, ld);
    // partial sums for the walker: (j,j) without its last term, (j+1,j) complete
    const int r1 = tr ? j : i, r2 = tr ? i : j;
    T = Terms{0, i == j ? max(j - 1, 0) : j, A + 64 * r1, A + 64 * r1, A + 64 * r2, ld, ld, ld, r1, nt, r2, nt};
  }
  pair_accumulate(acc, T, flags, g.gen, err, smem, rec, t);
  if (!is_x && i - j <= 1) {
    part_store(acc, g.part + (size_t)(2 * j + (i - j)) * 4096);
    wt_stores_done();
    __syncthreads();
    if (tid == 0) wt_publish(&pflags[2 * j + (i - j)], g.gen);
    return;
  }
  // the solve with the walker's diagonal inverse: of column j, or of X's row
  const int D = is_x ? s0 + i : j;
  if (tid == 0) wait_flag(&flags[D + nt * D], g.gen, err, rec, t, D + nt * D);
  __syncthreads();
  wt_seen();
  v4d out[2][2];
  tile_trsm(acc, g.dinv + (size_t)D * 4096, smem, out);
  if (is_x) {
    // X_ij^T into the upper block (j,i) for the later tiles of block column j;
    // X_ij into the lower block (i,j)
    tile_store_direct<true>(out, X + 64 * j + (size_t)(64 * i) * ldx, ldx);
    tile_store_direct_t<true>(out, X + 64 * i + (size_t)(64 * j) * ldx, ldx);
    wt_stores_done();
    __syncthreads();
    if (tid == 0) wt_publish(&flags[xf + i + ns * j], g.gen);
  } else {
    tile_store(out, A + 64 * i + (size_t)(64 * j) * ld, ld, smem);
    if (tid == 0) wt_publish(&flags[i + nt * j], g.gen);
  }
}

// The launch is persistent: dag_workgroups() workgroups, at most one per CU (the
// tile staging fills the LDS), each taking tickets in turn until they run out.
// A task waits only for tasks of lower tickets, for the walker, or (the early
// tiles) for tiles of higher tickets; every ticket taken is held by a running
// workgroup, and a workgroup takes the next ticket as soon as it is free, so
// with kDagBeside workgroups beside the walker's the tasks waited for always
// run.  (With one workgroup per task, the hardware assigns the workgroups to the
// XCDs in advance: when the only XCD with workgroups left to start is full of
// waiting ones, the lowest untaken ticket never starts.)
template <bool MACRO>
__global__ __launch_bounds__(256) void potrf_dag_kernel(DagArgs g) {
  // one LDS variable: with several, the compiler's record of which pointers
  // are distinct is lost, and LDS reads wait for every load into LDS before
  // them (half_product)
  __shared__ __attribute__((aligned(16))) double smem[kDagSmemDoubles + 2];
  int& t_s = *reinterpret_cast<int*>(smem + kDagSmemDoubles);  // then the three words of pair_accumulate
  const int ns = g.s0 >= 0 ? g.nt - g.s0 : 0;
  const int total = g.nfac + ns * (ns + 1) / 2;  // the last ticket
  auto take = [&] {
    if (threadIdx.x == 0) {
      const int t = atomicAdd(&g.sync[0], 1);
      t_s = t;
      // each workgroup ends with one take past the last ticket: the last of
      // those clears the counter for the next launch
      if (t == total + (int)gridDim.x)
        __hip_atomic_store(&g.sync[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(t_s);
    __syncthreads();
    return t;
  };
  int t = take();
  // the walker outside the loop over tile tasks, so that what the compiler
  // hoists out of either takes no registers from the other
  if (t == 0) {
    dag_walker(g, smem);
    __syncthreads();
    t = take();
  }
  for (; t <= total; t = take()) {
    dag_task<MACRO>(g, t, smem);
    __syncthreads();
  }
}

static int dag_cus() {
  static int n = 0;
  if (n == 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
      n = cus;
    else
      n = 256;
  }
  return n;
}

__global__ void dag_wait_reset_kernel(int* err, int* rec) {
  if (threadIdx.x == 0) *err = 0;
  if (threadIdx.x < 4) rec[threadIdx.x] = 0;
}

static int dag_reserve(DenseWork& w, int nt, hipStream_t s) {
  // The ticket and the error word have fixed places; the flags hold the
  // generation of the launch that set them, so launches of another order
  // (whose flags sit elsewhere) need no clearing in between.  Room for X's
  // flags and transposed diagonal blocks (up to nt of each side) is always
  // kept.
  const size_t need = 2 + (size_t)nt * nt + 2 * (size_t)nt + (size_t)nt * nt;
  if (need > w.dag_cap) {
    if (w.d_dag) RSD_HIP(hipFree(w.d_dag));
    RSD_HIP(hipMalloc(&w.d_dag, need * sizeof(int)));
    RSD_HIP(hipMemsetAsync(w.d_dag, 0, need * sizeof(int), s));
    if (!w.d_rec) {
      RSD_HIP(hipMalloc(&w.d_rec, 4 * sizeof(int)));
      RSD_HIP(hipMemsetAsync(w.d_rec, 0, 4 * sizeof(int), s));
    }
    w.dag_cap = need;
    w.dag_gen = 0;
  }
  const size_t need_part = 3 * (size_t)nt * 4096;
  if (need_part > w.part_cap) {
    if (w.d_part) RSD_HIP(hipFree(w.d_part));
    RSD_HIP(hipMalloc(&w.d_part, need_part * sizeof(double)));
    w.part_cap = need_part;
  }
  return RSD_OK;
}

int potrf_lower(DenseWork& w, double* A, int n, int ld, hipStream_t s) {
  return potrf_lower_x(w, A, n, ld, -1, nullptr, 0, s);
}

int potrf_lower_x(DenseWork& w, double* A, int n, int ld, int s0, double* X, int ldx, hipStream_t s) {
  const int nt = n / 64;
  if (nt < 1) return RSD_OK;
  if ((ld & 1) || (reinterpret_cast<uintptr_t>(A) & 15)) {
    // the tile loads move 16-byte pairs of rows
    set_error("potrf_lower: the matrix must be 16-byte aligned with an even leading dimension");
    return RSD_ERR_ARG;
  }
  if (X && (s0 < 0 || s0 >= nt || (ldx & 1) || ldx < 64 * (nt - s0) || (reinterpret_cast<uintptr_t>(X) & 15))) {
    set_error("potrf_lower_x: X needs 0 <= s0 < n/64, 16-byte alignment and an even ldx >= n - 64 s0");
    return RSD_ERR_ARG;
  }
  if (!X) s0 = -1;
  const int rc = dag_reserve(w, nt, s);
  if (rc) return rc;
  if (++w.dag_gen == 0x7fffffff) w.dag_gen = 1;
  const bool macro = nt >= kMacroTiles;
  const int nfac = dag_tickets(nt, macro);
  DagArgs g{A, ld, nt, w.dinv, w.d_part, w.d_dag, w.dag_gen, nfac, w.d_info, w.d_rec, s0, X, ldx};
  const int ns = s0 >= 0 ? nt - s0 : 0;
  // algorithmic flops: n^3/3 for the factor, plus m^3/3 for the triangular inverse of its trailing
  // m = 64 ns rows when X is asked for
  const double nd = (double)n, md = 64.0 * ns;
  hipEvent_t pe = prof_begin(kProfPotrfDiag, (nd * nd * nd + md * md * md) / 3.0, 0.0, s);
  hipLaunchKernelGGL((macro ? potrf_dag_kernel<true> : potrf_dag_kernel<false>),
                     dim3(dag_workgroups(nt, 1 + nfac + ns * (ns + 1) / 2, dag_cus())), dim3(256), 0, s, g);
  prof_end(pe, s);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// ------------------------------------------- triangular solves (potrs)
// (L L^T) X = B for up to two right-hand sides, one persistent launch per
// direction.  Workgroup t takes block row k by an atomic ticket (forward:
// k = t, backward: k = nb-1-t), accumulates L_kj y_j for the blocks j it
// depends on as soon as each is published, applies the 64x64 diagonal
// inverse and publishes its own block: the 64 values written through, then
// (once every wave's stores are done) a store of the solve's generation into
// the block's flag; readers take published blocks with agent-scope loads.
// A workgroup only ever waits for blocks of lower tickets, which running
// workgroups hold, so the
// solve finishes whatever the residency; every wait is bounded and a wait
// that runs out sets the error word instead of hanging.
// Forward: y_k = Dinv_k (b_k - sum_{j<k} L_kj y_j).  Lane = row of block k,
// wave wv takes columns 16wv..16wv+15 of every L_kj; each wave waits for
// block j on its own (no workgroup barrier in the loop) after issuing the
// loads of L_kj, so the loads overlap the wait.
template <int NR>
__global__ __launch_bounds__(256) void potrs_fwd_kernel(const double* __restrict__ L, int ld,
                                                        const double* __restrict__ dinv, double* X, int ldx, int nb,
                                                        int* sync, int gen) {
  __shared__ int k_s;
  __shared__ double yv[NR][64];
  __shared__ double red[NR][4][64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int* err = sync + 2;
  int* flags = sync + 3;
  if (tid == 0) {
    const int t = atomicAdd(&sync[0], 1);
    k_s = t;
    // every workgroup has its ticket: the last one clears the counter for the next launch
    if (t == nb - 1) __hip_atomic_store(&sync[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  const int k = k_s;
  const size_t row = (size_t)64 * k + lane;
  // Dinv_k and b_k depend on no other workgroup (only this one writes block
  // row k of X): load them now, off the chain of waits below
  const double* D = dinv + (size_t)k * 4096;
  double dv[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) dv[c] = D[lane + 64 * (16 * wv + c)];
  const double bk = wv < NR ? X[(size_t)wv * ldx + row] : 0.0;
  double acc[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) acc[r] = 0.0;
  for (int j = 0; j < k; ++j) {
    const double* Lb = L + row + (size_t)(64 * j + 16 * wv) * ld;
    double lv[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) lv[c] = Lb[(size_t)c * ld];
    if (lane == 0) wait_flag(&flags[j], gen, err);
    __builtin_amdgcn_wave_barrier();
    wt_seen();
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const double* yj = X + (size_t)r * ldx + (size_t)64 * j + 16 * wv;
#pragma unroll
      for (int c = 0; c < 16; ++c) acc[r] += lv[c] * wt_load(yj + c);
    }
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) red[r][wv][lane] = acc[r];
  __syncthreads();
  // t = b_k - sum; y_k = Dinv_k t
  if (wv < NR) yv[wv][lane] = bk - ((red[wv][0][lane] + red[wv][1][lane]) + (red[wv][2][lane] + red[wv][3][lane]));
  __syncthreads();
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    double t = 0.0;
#pragma unroll
    for (int c = 0; c < 16; ++c) t += dv[c] * yv[r][16 * wv + c];
    acc[r] = t;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < NR; ++r) red[r][wv][lane] = acc[r];
  __syncthreads();
  if (wv < NR)
    wt_store(X + (size_t)wv * ldx + row, (red[wv][0][lane] + red[wv][1][lane]) + (red[wv][2][lane] + red[wv][3][lane]));
  wt_stores_done();
  __syncthreads();
  if (tid == 0) wt_publish(&flags[k], gen);
}

// Sum over the 64 lanes of a wave of p[c], c < 16 (this lane's shares of
// 16 column sums): the set is halved across lane bits 32, 16, 8, 4 (each lane
// keeps half and adds its partner's half), then added across bits 2 and 1.
// Lanes with (lane & 3) == 0 end with the sum of column lane >> 2 in p[0].
template <int CNT, int BIT>
__device__ __forceinline__ void colsum_halve(double (&p)[16], int lane) {
  const bool upper = (lane & BIT) != 0;
#pragma unroll
  for (int m = 0; m < CNT; ++m) {
    const double send = upper ? p[m] : p[m + CNT];
    const double keep = upper ? p[m + CNT] : p[m];
    p[m] = keep + __shfl_xor(send, BIT, 64);
  }
}
__device__ __forceinline__ void wave_colsum16(double (&p)[16], int lane) {
  colsum_halve<8, 32>(p, lane);
  colsum_halve<4, 16>(p, lane);
  colsum_halve<2, 8>(p, lane);
  colsum_halve<1, 4>(p, lane);
  p[0] += __shfl_xor(p[0], 2, 64);
  p[0] += __shfl_xor(p[0], 1, 64);
}

// Backward: x_k = Dinv_k^T (y_k - sum_{j>k} L_jk^T x_j).  Lanes run down the
// rows of each L_jk block (coalesced) and keep per-column partial sums,
// summed over the wave's lanes once, at the end (wave_colsum16).  Waits as
// in the forward pass.
template <int NR>
__global__ __launch_bounds__(256) void potrs_bwd_kernel(const double* __restrict__ L, int ld,
                                                        const double* __restrict__ dinv, double* X, int ldx, int nb,
                                                        int* sync, int gen) {
  __shared__ int k_s;
  __shared__ double xv[NR][64];
  __shared__ double cs[NR][64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int* err = sync + 2;
  int* flags = sync + 3 + nb;
  if (tid == 0) {
    const int t = atomicAdd(&sync[1], 1);
    k_s = nb - 1 - t;
    if (t == nb - 1) __hip_atomic_store(&sync[1], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  const int k = k_s;
  // Dinv_k and y_k depend on no other workgroup: load them now, off the chain
  const double* D = dinv + (size_t)k * 4096;
  double dv[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) dv[c] = D[lane + 64 * (16 * wv + c)];
  const double yk = wv < NR ? X[(size_t)wv * ldx + (size_t)64 * k + lane] : 0.0;
  double p[NR][16];
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int c = 0; c < 16; ++c) p[r][c] = 0.0;
  for (int j = nb - 1; j > k; --j) {
    const double* Lb = L + (size_t)64 * j + lane + (size_t)(64 * k + 16 * wv) * ld;
    double lv[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) lv[c] = Lb[(size_t)c * ld];
    if (lane == 0) wait_flag(&flags[j], gen, err);
    __builtin_amdgcn_wave_barrier();
    wt_seen();
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const double xr = wt_load(X + (size_t)r * ldx + (size_t)64 * j + lane);
#pragma unroll
      for (int c = 0; c < 16; ++c) p[r][c] += lv[c] * xr;
    }
  }
  // t = y_k - column sums (columns 16 wv + c of the wave)
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    wave_colsum16(p[r], lane);
    if ((lane & 3) == 0) cs[r][16 * wv + (lane >> 2)] = p[r][0];
  }
  __syncthreads();
  if (wv < NR) xv[wv][lane] = yk - cs[wv][lane];
  __syncthreads();
  // x_k = Dinv_k^T t: the same column sums, of Dinv_k's columns times t
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const double t = xv[r][lane];
#pragma unroll
    for (int c = 0; c < 16; ++c) p[r][c] = dv[c] * t;
    wave_colsum16(p[r], lane);
    if ((lane & 3) == 0) wt_store(X + (size_t)r * ldx + (size_t)64 * k + 16 * wv + (lane >> 2), p[r][0]);
  }
  wt_stores_done();
  __syncthreads();
  if (tid == 0) wt_publish(&flags[k], gen);
}

// [0] forward ticket, [1] backward ticket, [2] error word, then the forward
// and the backward flags (nb each, holding the generation that set them).
// The tickets are cleared by each launch's last workgroup.
static int sync_reserve(DenseWork& w, int nb, hipStream_t s) {
  const size_t need = 3 + 2 * (size_t)nb;
  if (need > w.sync_cap) {
    if (w.d_sync) RSD_HIP(hipFree(w.d_sync));
    RSD_HIP(hipMalloc(&w.d_sync, need * sizeof(int)));
    RSD_HIP(hipMemsetAsync(w.d_sync, 0, need * sizeof(int), s));
    w.sync_cap = need;
    w.gen = 0;
  }
  return RSD_OK;
}

int potrs_lower(DenseWork& w, const double* A, int n, int ld, double* X, int ldx, int nrhs, hipStream_t s) {
  if (n % 64 || nrhs < 1 || nrhs > 2) {
    set_error("potrs_lower: n must be a multiple of 64 and nrhs 1 or 2");
    return RSD_ERR_ARG;
  }
  const int nb = n / 64;
  const int rc = sync_reserve(w, nb, s);
  if (rc) return rc;
  // flags hold the generation that set them; a new generation needs no clearing
  if (++w.gen == 0x7fffffff) w.gen = 1;
  hipEvent_t pe = prof_begin(kProfTrsv, 2.0 * n * n * nrhs / 2.0, 8.0 * n * n / 2.0, s);
  if (nrhs == 1)
    hipLaunchKernelGGL(potrs_fwd_kernel<1>, dim3(nb), dim3(256), 0, s, A, ld, (const double*)w.dinv, X, ldx, nb,
                       w.d_sync, w.gen);
  else
    hipLaunchKernelGGL(potrs_fwd_kernel<2>, dim3(nb), dim3(256), 0, s, A, ld, (const double*)w.dinv, X, ldx, nb,
                       w.d_sync, w.gen);
  prof_end(pe, s);
  pe = prof_begin(kProfTrsv, 2.0 * n * n * nrhs / 2.0, 8.0 * n * n / 2.0, s);
  if (nrhs == 1)
    hipLaunchKernelGGL(potrs_bwd_kernel<1>, dim3(nb), dim3(256), 0, s, A, ld, (const double*)w.dinv, X, ldx, nb,
                       w.d_sync, w.gen);
  else
    hipLaunchKernelGGL(potrs_bwd_kernel<2>, dim3(nb), dim3(256), 0, s, A, ld, (const double*)w.dinv, X, ldx, nb,
                       w.d_sync, w.gen);
  prof_end(pe, s);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

int trsv_lower(DenseWork& w, const double* L, int n, int ld, const double* dinv, double* x, bool trans,
               hipStream_t s) {
  if (n % 64) {
    set_error("trsv_lower: n must be a multiple of 64");
    return RSD_ERR_ARG;
  }
  const int nb = n / 64;
  const int rc = sync_reserve(w, nb, s);
  if (rc) return rc;
  if (++w.gen == 0x7fffffff) w.gen = 1;
  hipEvent_t pe = prof_begin(kProfTrsv, (double)n * n, 8.0 * n * n / 2.0, s);
  if (trans)
    hipLaunchKernelGGL(potrs_bwd_kernel<1>, dim3(nb), dim3(256), 0, s, L, ld, dinv, x, n, nb, w.d_sync, w.gen);
  else
    hipLaunchKernelGGL(potrs_fwd_kernel<1>, dim3(nb), dim3(256), 0, s, L, ld, dinv, x, n, nb, w.d_sync, w.gen);
  prof_end(pe, s);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// G' = [C B^T; B A] (lower triangle) from G = [A B; B^T C]: C (n5 x n5) padded to
// n5p with identity, then A (n6 x n6) padded to n6p; B below C
// The padding of the reordered grand mobility [C B^T; B A] (order n5p + n6p):
// rows and columns n5..n5p-1 (C's) and n5p+n6..n5p+n6p-1 (A's) become the
// identity's.  One thread per (padding index, column).
__global__ void grand_padding_kernel(double* __restrict__ Gp, int ld, int n5, int n5p, int n6, int n6p) {
  const int np = n5p + n6p, pc = n5p - n5;
  const int k = blockIdx.y;  // the k-th padding index
  const int p = k < pc ? n5 + k : n5p + n6 + (k - pc);
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < np; c += gridDim.x * blockDim.x) {
    const double v = c == p ? 1.0 : 0.0;
    Gp[(size_t)p + (size_t)c * ld] = v;
    Gp[(size_t)c + (size_t)p * ld] = v;
  }
}

int grand_padding(double* Gp, int ld, int n5, int n5p, int n6, int n6p, hipStream_t s) {
  const int npad = (n5p - n5) + (n6p - n6);
  if (npad == 0) return RSD_OK;
  hipLaunchKernelGGL(grand_padding_kernel, dim3((n5p + n6p + 255) / 256, npad), dim3(256), 0, s, Gp, ld, n5, n5p, n6,
                     n6p);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

const int* dense_solve_error_word(const DenseWork& w) { return w.d_sync ? w.d_sync + 2 : nullptr; }
const int* dense_factor_error_word(const DenseWork& w) { return w.d_dag ? w.d_dag + 1 : nullptr; }

int dense_factor_wait_record(const DenseWork& w, int rec[4]) {
  for (int k = 0; k < 4; ++k) rec[k] = 0;
  if (!w.d_rec) return RSD_OK;
  RSD_HIP(hipMemcpy(rec, w.d_rec, 4 * sizeof(int), hipMemcpyDeviceToHost));
  return RSD_OK;
}

int dense_wait_reset(DenseWork& w, hipStream_t s) {
  if (!w.d_dag || !w.d_rec) return RSD_OK;
  hipLaunchKernelGGL(dag_wait_reset_kernel, dim3(1), dim3(64), 0, s, w.d_dag + 1, w.d_rec);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

int dense_sync_error(DenseWork& w, hipStream_t s, int* err) {
  int e[2] = {0, 0};
  if (w.d_sync) RSD_HIP(hipMemcpyAsync(&e[0], w.d_sync + 2, sizeof(int), hipMemcpyDeviceToHost, s));
  if (w.d_dag) RSD_HIP(hipMemcpyAsync(&e[1], w.d_dag + 1, sizeof(int), hipMemcpyDeviceToHost, s));
  RSD_HIP(hipStreamSynchronize(s));
  *err = e[0] | e[1];
  return RSD_OK;
}

// copy the stored diagonal inverses onto the diagonal tiles
__global__ __launch_bounds__(256) void put_dinv_kernel(double* A, int ld, const double* dinv) {
  const int k = blockIdx.x;
  for (int idx = threadIdx.x; idx < 4096; idx += 256) {
    int r = idx & 63, c = idx >> 6;
    A[(size_t)(64 * k + r) + (size_t)(64 * k + c) * ld] = dinv[(size_t)k * 4096 + r + (size_t)c * 64];
  }
}

// Recursive blocked inverse of a lower-triangular matrix:
//   inv([L11 0; L21 L22]) = [X11 0; -X22 L21 X11  X22]
// The leaves are the 64x64 inverses potrf_lower left in dinv; every level
// of the recursion is one batched launch for T = L21 X11 and one for
// X21 = -X22 T.
namespace {
struct Node {
  int a, m, b;  // tile range [a,b) split at m
};
void build_levels(int a, int b, int depth, std::vector<std::vector<Node>>& lv) {
  if (b - a <= 1) return;
  int m = a + (b - a + 1) / 2;
  if ((int)lv.size() <= depth) lv.resize(depth + 1);
  lv[depth].push_back({a, m, b});
  build_levels(a, m, depth + 1, lv);
  build_levels(m, b, depth + 1, lv);
}
}  // namespace

int trtri_lower(DenseWork& w, double* A, int n, int ld, hipStream_t s, const double* dinv) {
  const int nt = n / 64;
  hipLaunchKernelGGL(put_dinv_kernel, dim3(nt), dim3(256), 0, s, A, ld, dinv ? dinv : (const double*)w.dinv);
  std::vector<std::vector<Node>> lv;
  build_levels(0, nt, 0, lv);
  double* T = w.tmp;  // same shape as A (leading dim n); node blocks never overlap
  for (int d = (int)lv.size() - 1; d >= 0; --d) {
    std::vector<GemmDesc> g1, g2;
    for (const Node& nd : lv[d]) {
      GemmDesc g{};
      // T[m:b, a:m] = L21 * X11   (X11 lower: inner index starts at the column tile)
      g.A = A + (size_t)(64 * nd.m) + (size_t)(64 * nd.a) * ld;
      g.B = A + (size_t)(64 * nd.a) + (size_t)(64 * nd.a) * ld;
      g.C = T + (size_t)(64 * nd.m) + (size_t)(64 * nd.a) * n;
      g.lda = ld;
      g.ldb = ld;
      g.ldc = n;
      g.mt = nd.b - nd.m;
      g.nt = nd.m - nd.a;
      g.kt = nd.m - nd.a;
      g.alpha = 1.0;
      g.beta = 0.0;
      g1.push_back(g);
      GemmDesc h{};
      // X21 = -X22 * T   (X22 lower: inner index ends at the row tile)
      h.A = A + (size_t)(64 * nd.m) + (size_t)(64 * nd.m) * ld;
      h.B = T + (size_t)(64 * nd.m) + (size_t)(64 * nd.a) * n;
      h.C = A + (size_t)(64 * nd.m) + (size_t)(64 * nd.a) * ld;
      h.lda = ld;
      h.ldb = n;
      h.ldc = ld;
      h.mt = nd.b - nd.m;
      h.nt = nd.m - nd.a;
      h.kt = nd.b - nd.m;
      h.alpha = -1.0;
      h.beta = 0.0;
      g2.push_back(h);
    }
    int rc = gemm_batched(w, g1, false, false, kKloCol, s);
    if (rc) return rc;
    rc = gemm_batched(w, g2, false, false, kKhiRow, s);
    if (rc) return rc;
  }
  return RSD_OK;
}

int lauum_lower(DenseWork& w, const double* X, int ldx, double* C, int ldc, int n, hipStream_t s) {
  const int nt = n / 64;
  GemmDesc g{};
  g.A = X;
  g.B = X;
  g.C = C;
  g.lda = ldx;
  g.ldb = ldx;
  g.ldc = ldc;
  g.mt = g.nt = g.kt = nt;
  g.alpha = 1.0;
  g.beta = 0.0;
  // C_ij = sum_{k >= i} X_ki^T X_kj   (i >= j)
  return gemm_batched(w, {g}, true, false, kLowerC | kKloRow, s);
}

// FP32 copies for the CG preconditioner: the lower triangle of an FP64 factor
// (diagonal tiles excepted: they get the FP32 diagonal-tile inverses)
__global__ void lower_to_f32_kernel(const double* __restrict__ L, int ldl, float* __restrict__ F, int ldf, int n) {
  const int r = blockIdx.x * 64 + (threadIdx.x & 63), c = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (r < n && c < n && (r >> 6) > (c >> 6)) F[(size_t)r + (size_t)c * ldf] = (float)L[(size_t)r + (size_t)c * ldl];
}

__global__ __launch_bounds__(256) void put_dinv32_kernel(float* A, int ld, const double* dinv) {
  const int k = blockIdx.x;
  for (int idx = threadIdx.x; idx < 4096; idx += 256) {
    const int r = idx & 63, c = idx >> 6;
    A[(size_t)(64 * k + r) + (size_t)(64 * k + c) * ld] = (float)dinv[(size_t)k * 4096 + r + (size_t)c * 64];
  }
}

int factor_to_f32(DenseWork& w, const double* L, int n, int ld, float* F, int ldf, hipStream_t s) {
  hipLaunchKernelGGL(lower_to_f32_kernel, dim3((n + 63) / 64, (n + 3) / 4), dim3(256), 0, s, L, ld, F, ldf, n);
  hipLaunchKernelGGL(put_dinv32_kernel, dim3(n / 64), dim3(256), 0, s, F, ldf, (const double*)w.dinv);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// trtri_lower's recursion in FP32, on a matrix whose diagonal tiles already
// hold their inverses (factor_to_f32); T is n x n FP32 scratch
int trtri_lower32(DenseWork& w, float* A, int n, int ld, float* T, hipStream_t s) {
  const int nt = n / 64;
  std::vector<std::vector<Node>> lv;
  build_levels(0, nt, 0, lv);
  for (int d = (int)lv.size() - 1; d >= 0; --d) {
    std::vector<Gemm32Desc> g1, g2;
    for (const Node& nd : lv[d]) {
      Gemm32Desc g{};
      g.A = A + (size_t)(64 * nd.m) + (size_t)(64 * nd.a) * ld;
      g.B = A + (size_t)(64 * nd.a) + (size_t)(64 * nd.a) * ld;
      g.C = T + (size_t)(64 * nd.m) + (size_t)(64 * nd.a) * n;
      g.lda = ld;
      g.ldb = ld;
      g.ldc = n;
      g.mt = nd.b - nd.m;
      g.nt = nd.m - nd.a;
      g.kt = nd.m - nd.a;
      g.alpha = 1.f;
      g.beta = 0.f;
      g1.push_back(g);
      Gemm32Desc h{};
      h.A = A + (size_t)(64 * nd.m) + (size_t)(64 * nd.m) * ld;
      h.B = T + (size_t)(64 * nd.m) + (size_t)(64 * nd.a) * n;
      h.C = A + (size_t)(64 * nd.m) + (size_t)(64 * nd.a) * ld;
      h.lda = ld;
      h.ldb = n;
      h.ldc = ld;
      h.mt = nd.b - nd.m;
      h.nt = nd.m - nd.a;
      h.kt = nd.b - nd.m;
      h.alpha = -1.f;
      h.beta = 0.f;
      g2.push_back(h);
    }
    RSD_TRY(gemm32_batched(w, g1, false, kKloCol, s));
    RSD_TRY(gemm32_batched(w, g2, false, kKhiRow, s));
  }
  return RSD_OK;
}

// the upper triangle of an n x n FP32 matrix from its lower one, through LDS
// so that both sides are read and written column-contiguously
__global__ __launch_bounds__(256) void sym_fill_upper_f32_kernel(float* P, int n) {
  const int R = blockIdx.x, C = blockIdx.y;  // destination block of 32 x 32
  if (R >= C) return;
  __shared__ float t[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int j = ty; j < 32; j += 8) t[j][tx] = P[(size_t)(C * 32 + tx) + (size_t)(R * 32 + j) * n];
  __syncthreads();
  for (int j = ty; j < 32; j += 8) P[(size_t)(R * 32 + tx) + (size_t)(C * 32 + j) * n] = t[tx][j];
}

int sym_fill_upper_f32(float* P, int n, hipStream_t s) {
  hipLaunchKernelGGL(sym_fill_upper_f32_kernel, dim3(n / 32, n / 32), dim3(256), 0, s, P, n);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// C = X^T X (lower tiles), X lower-triangular FP32
int lauum_lower32(DenseWork& w, const float* X, int ldx, float* C, int ldc, int n, hipStream_t s) {
  const int nt = n / 64;
  Gemm32Desc g{};
  g.A = X;
  g.B = X;
  g.C = C;
  g.lda = ldx;
  g.ldb = ldx;
  g.ldc = ldc;
  g.mt = g.nt = g.kt = nt;
  g.alpha = 1.f;
  g.beta = 0.f;
  return gemm32_batched(w, {g}, true, kLowerC | kKloRow, s);
}

__global__ void symmetrize_kernel(double* A, int n, int ld) {
  const int c = blockIdx.y * 16 + threadIdx.y;
  const int r = blockIdx.x * 16 + threadIdx.x;
  if (r < n && c < n && r < c) A[(size_t)r + (size_t)c * ld] = A[(size_t)c + (size_t)r * ld];
}

int symmetrize_from_lower(double* A, int n, int ld, hipStream_t s) {
  dim3 b(16, 16), g((n + 15) / 16, (n + 15) / 16);
  hipLaunchKernelGGL(symmetrize_kernel, g, b, 0, s, A, n, ld);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

__global__ void zero_upper_kernel(double* A, int n, int ld) {
  const int c = blockIdx.y * 16 + threadIdx.y;
  const int r = blockIdx.x * 16 + threadIdx.x;
  if (r < n && c < n && r < c) A[(size_t)r + (size_t)c * ld] = 0.0;
}

int zero_strict_upper(double* A, int n, int ld, hipStream_t s) {
  dim3 b(16, 16), g((n + 15) / 16, (n + 15) / 16);
  hipLaunchKernelGGL(zero_upper_kernel, g, b, 0, s, A, n, ld);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

__global__ void load_sym_upper_kernel(const double* src, int n, int lds, double* A, int np, int ld) {
  const int c = blockIdx.y * 16 + threadIdx.y;
  const int r = blockIdx.x * 16 + threadIdx.x;
  if (r >= np || c >= np) return;
  double v;
  if (r < n && c < n)
    v = (r <= c) ? src[(size_t)r + (size_t)c * lds] : src[(size_t)c + (size_t)r * lds];
  else
    v = (r == c) ? 1.0 : 0.0;
  A[(size_t)r + (size_t)c * ld] = v;
}

int load_sym_from_upper(const double* src, int n, int ldsrc, double* A, int np, int ld, hipStream_t s) {
  dim3 b(16, 16), g((np + 15) / 16, (np + 15) / 16);
  hipLaunchKernelGGL(load_sym_upper_kernel, g, b, 0, s, src, n, ldsrc, A, np, ld);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

__global__ void identity_pad_kernel(double* A, int n, int np, int ld) {
  const int c = blockIdx.y * 16 + threadIdx.y;
  const int r = blockIdx.x * 16 + threadIdx.x;
  if (r >= np || c >= np) return;
  if (r < n && c < n) return;
  A[(size_t)r + (size_t)c * ld] = (r == c) ? 1.0 : 0.0;
}

int set_identity_padding(double* A, int n, int np, int ld, hipStream_t s) {
  if (np == n) return RSD_OK;
  dim3 b(16, 16), g((np + 15) / 16, (np + 15) / 16);
  hipLaunchKernelGGL(identity_pad_kernel, g, b, 0, s, A, n, np, ld);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

__global__ void copy_block_kernel(const double* src, int lds, double* dst, int ldd, int m, int n) {
  const int c = blockIdx.y;
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < m; r += gridDim.x * blockDim.x)
    if (c < n) dst[(size_t)r + (size_t)c * ldd] = src[(size_t)r + (size_t)c * lds];
}

int copy_block(const double* src, int lds, double* dst, int ldd, int m, int n, hipStream_t s) {
  if (m <= 0 || n <= 0) return RSD_OK;
  dim3 g(std::max(1, std::min(64, (m + 255) / 256)), n), b(256);
  hipLaunchKernelGGL(copy_block_kernel, g, b, 0, s, src, lds, dst, ldd, m, n);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

__global__ void matrix_axpy_kernel(double alpha, const double* X, int ldx, double* Y, int ldy, int m, int n) {
  const int c = blockIdx.y;
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < m; r += gridDim.x * blockDim.x)
    if (c < n) Y[(size_t)r + (size_t)c * ldy] += alpha * X[(size_t)r + (size_t)c * ldx];
}

int matrix_axpy(double alpha, const double* X, int ldx, double* Y, int ldy, int m, int n, hipStream_t s) {
  if (m <= 0 || n <= 0) return RSD_OK;
  dim3 g(std::max(1, std::min(64, (m + 255) / 256)), n), b(256);
  hipLaunchKernelGGL(matrix_axpy_kernel, g, b, 0, s, alpha, X, ldx, Y, ldy, m, n);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

__global__ void vector_sum_kernel(const double* __restrict__ a, const double* __restrict__ b, double* __restrict__ y,
                                  int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = a[i] + b[i];
}

int vector_sum(const double* a, const double* b, double* y, int n, hipStream_t s) {
  if (n <= 0) return RSD_OK;
  hipLaunchKernelGGL(vector_sum_kernel, dim3((n + 255) / 256), dim3(256), 0, s, a, b, y, n);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

int spd_inverse(DenseWork& w, double* A, double* Ainv, int np, int ld, hipStream_t s) {
  int rc = potrf_lower(w, A, np, ld, s);
  if (rc) return rc;
  rc = trtri_lower(w, A, np, ld, s);
  if (rc) return rc;
  rc = lauum_lower(w, A, ld, Ainv, ld, np, s);
  if (rc) return rc;
  return symmetrize_from_lower(Ainv, np, ld, s);
}

// ------------------------------------------------------------------ GEMV
// y = alpha*A x + beta*y: 64-row x column-chunk workgroups write partial sums
// (4 waves stride the chunk's columns, lanes run down contiguous rows), then
// a second pass adds the chunks in a fixed order (deterministic).
__global__ __launch_bounds__(256) void gemv_n_part_kernel(const double* __restrict__ A, int lda, int m, int n,
                                                          const double* __restrict__ x, int cchunk,
                                                          double* __restrict__ part) {
  __shared__ double red[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int r = blockIdx.x * 64 + lane;
  const int c0 = blockIdx.y * cchunk, c1 = min(n, c0 + cchunk);
  double acc = 0.0;
  if (r < m)
    for (int c = c0 + wv; c < c1; c += 4) acc += A[(size_t)r + (size_t)c * lda] * x[c];
  red[wv][lane] = acc;
  __syncthreads();
  if (wv == 0 && r < m) part[(size_t)blockIdx.y * m + r] = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

// 64 rows per workgroup: wave w sums chunks w, w+4, ... in order, then the
// four wave sums combine in a fixed order (bitwise repeatable)
__global__ __launch_bounds__(256) void gemv_n_reduce_kernel(int m, int nchunk, const double* __restrict__ part,
                                                            double alpha, double beta, double* __restrict__ y) {
  __shared__ double red[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int r = blockIdx.x * 64 + lane;
  double acc = 0.0;
  if (r < m) {
#pragma unroll 4
    for (int c = wv; c < nchunk; c += 4) acc += part[(size_t)c * m + r];
  }
  red[wv][lane] = acc;
  __syncthreads();
  if (wv == 0 && r < m) {
    const double tot = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
    y[r] = alpha * tot + (beta != 0.0 ? beta * y[r] : 0.0);
  }
}

// y = alpha*A^T x + beta*y : one wavefront per output (column), lanes down the column
__global__ __launch_bounds__(256) void gemv_t_kernel(const double* __restrict__ A, int lda, int m, int n, double alpha,
                                                     const double* __restrict__ x, double beta, double* y) {
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (c >= n) return;
  double acc = 0.0;
  for (int r = lane; r < m; r += 64) acc += A[(size_t)r + (size_t)c * lda] * x[r];
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if (lane == 0) y[c] = alpha * acc + (beta != 0.0 ? beta * y[c] : 0.0);
}

int gemv(DenseWork& w, const double* A, int lda, int m, int n, bool trans, double alpha, const double* x, double beta,
         double* y, hipStream_t s) {
  if (m <= 0 || n <= 0) return RSD_OK;
  hipEvent_t pe = prof_begin(kProfGemv, 2.0 * m * n, 8.0 * m * n, s);
  if (!trans) {
    const int nchunk = std::max(1, std::min(64, (n + 63) / 64));
    const int cchunk = (n + nchunk - 1) / nchunk;
    const size_t need = (size_t)m * nchunk;
    if (need > w.gv_cap) {
      if (w.gv_part) RSD_HIP(hipFree(w.gv_part));
      w.gv_part = nullptr;
      RSD_HIP(hipMalloc(&w.gv_part, need * sizeof(double)));
      w.gv_cap = need;
    }
    hipLaunchKernelGGL(gemv_n_part_kernel, dim3((m + 63) / 64, nchunk), dim3(256), 0, s, A, lda, m, n, x, cchunk,
                       w.gv_part);
    hipLaunchKernelGGL(gemv_n_reduce_kernel, dim3((m + 63) / 64), dim3(256), 0, s, m, nchunk,
                       (const double*)w.gv_part, alpha, beta, y);
  } else {
    hipLaunchKernelGGL(gemv_t_kernel, dim3((n + 3) / 4), dim3(256), 0, s, A, lda, m, n, alpha, x, beta, y);
  }
  prof_end(pe, s);
  RSD_HIP(hipGetLastError());
  return RSD_OK;
}

// ------------------------------------------------------------------ scratch
int dense_reserve(DenseWork& w, int n, hipStream_t s) {
  (void)s;
  size_t nt = (size_t)(n / 64);
  size_t need_dinv = std::max<size_t>(nt, 1) * 4096;
  if (need_dinv > w.dinv_cap) {
    if (w.dinv) RSD_HIP(hipFree(w.dinv));
    RSD_HIP(hipMalloc(&w.dinv, need_dinv * sizeof(double)));
    w.dinv_cap = need_dinv;
  }
  size_t need_tmp = (size_t)n * (size_t)n;
  if (need_tmp > w.tmp_cap) {
    if (w.tmp) RSD_HIP(hipFree(w.tmp));
    RSD_HIP(hipMalloc(&w.tmp, need_tmp * sizeof(double)));
    w.tmp_cap = need_tmp;
  }
  if (!w.d_desc) {
    w.desc_cap = 64 * 1024;
    RSD_HIP(hipMalloc(&w.d_desc, w.desc_cap * sizeof(GemmDesc)));
  }
  if (!w.d_info) RSD_HIP(hipMalloc(&w.d_info, sizeof(int)));
  return RSD_OK;
}

void dense_release(DenseWork& w) {
  if (w.dinv) (void)hipFree(w.dinv);
  if (w.tmp) (void)hipFree(w.tmp);
  if (w.d_desc) (void)hipFree(w.d_desc);
  if (w.d_info) (void)hipFree(w.d_info);
  if (w.gv_part) (void)hipFree(w.gv_part);
  if (w.d_sync) (void)hipFree(w.d_sync);
  if (w.d_dag) (void)hipFree(w.d_dag);
  if (w.d_rec) (void)hipFree(w.d_rec);
  if (w.d_part) (void)hipFree(w.d_part);
  w = DenseWork{};
}

}  // namespace rsd
