// Vector kernels of the two Krylov solvers (sddc_krylov.hip: one system, host
// least squares; sddc_newton_batch.hip: B systems in lockstep), float64.
//
// An Arnoldi step orthogonalises w against the basis twice.  On a 20-60 vector
// basis of 4-60 thousand entries every kernel is bound by its launch and by one
// chain of loads, so a pass is two launches: the dot products, split over
// vectors and entries at once, and the update, whose workgroups each sum the
// partial products themselves (from L2) instead of waiting for a reduction
// launch.  Measured at 64 modes, 24 radial points (n = 4416): dots, reduction and
// update 11.6 + 20.5 + 5.1 us a pass before (a workgroup walked all vectors, a
// thread summed 240 partial products), see k_project for now.
//
// All sums have a fixed order that depends on the vector length alone.  flags
// (may be null): per instance b of kFlags ints; the kernels skip an instance whose flag
// `gate` is 0 (gate < 0: none).
#pragma once
#include <hip/hip_runtime.h>

#include "sddc_internal.h"

namespace sddc {
namespace krylov {

constexpr int kThreads = 256;
constexpr int kFlags = 8;
constexpr int kChunk = 1024;    // entries of a partial dot product
constexpr int kUpdate = 256;    // entries of an update workgroup, of a partial norm
constexpr int kVectors = 8;     // basis vectors of a dots workgroup
constexpr int kAhead = 16;      // basis vectors an update loads before it needs them

inline int chunks(int n) { return (n + kChunk - 1) / kChunk; }
inline int updates(int n) { return (n + kUpdate - 1) / kUpdate; }

struct Gate {
  const int* flags;
  int gate;
  __device__ __forceinline__ bool skips(int b) const {
    return flags && gate >= 0 && !flags[(size_t)b * kFlags + gate];
  }
};

// Basis vector i of instance b: at + i*ld + b*n; null: the vector x itself.
struct Basis {
  const double* at;
  size_t ld;
};

// Sum over the workgroup's threads, in every thread; tmp: one per wavefront.
__device__ __forceinline__ double block_sum(double v, double* tmp) {
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
  if ((threadIdx.x & 63) == 0) tmp[threadIdx.x >> 6] = v;
  __syncthreads();
  return (tmp[0] + tmp[1]) + (tmp[2] + tmp[3]);
}

// partial[(b*pstride + i)*gridDim.x + chunk] = V_i[b] . (x[b] - sub[b]) over a
// chunk, i < nv; V null: (x - sub) . (x - sub).  sub may be null.
// Grid: (chunks, ceil(nv / kVectors), B).
template <bool SELF, bool SUB>   // V is null; sub is not
__global__ __launch_bounds__(kThreads) void k_dots(Basis V, const double* __restrict__ x,
                                                   const double* __restrict__ sub, int n, int nv,
                                                   int pstride, double* __restrict__ partial,
                                                   Gate gate) {
  constexpr int E = kChunk / kThreads;
  __shared__ double red[kVectors][kThreads / 64];
  const int b = blockIdx.z, i0 = blockIdx.y * kVectors;
  if (gate.skips(b)) return;
  const size_t o = (size_t)b * n;
  const int e0 = blockIdx.x * kChunk + threadIdx.x;
  // every load before the first use: a launch is one memory latency
  double xv[E], sv[E], a[SELF ? 1 : kVectors][E], s[kVectors];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int e = e0 + u * kThreads < n ? e0 + u * kThreads : 0;
    xv[u] = x[o + e];
    sv[u] = SUB ? sub[o + e] : 0.0;
    if (!SELF)
#pragma unroll
      for (int q = 0; q < kVectors; ++q)
        a[SELF ? 0 : q][u] = V.at[(i0 + q < nv ? i0 + q : nv - 1) * V.ld + o + e];
  }
#pragma unroll
  for (int u = 0; u < E; ++u) xv[u] = e0 + u * kThreads < n ? xv[u] - sv[u] : 0.0;
#pragma unroll
  for (int q = 0; q < (SELF ? 1 : kVectors); ++q) {
    s[q] = 0.0;
#pragma unroll
    for (int u = 0; u < E; ++u)
      if (e0 + u * kThreads < n) s[q] = fma(SELF ? xv[u] : a[SELF ? 0 : q][u], xv[u], s[q]);
  }
  // sums over the wavefront: halves exchange vectors first, so that each lane ends
  // with one (vector lane / 8) and 10 exchanges do instead of 48
  const int lane = threadIdx.x & 63;
  if (!SELF) {
#pragma unroll
    for (int m = 32, k = kVectors / 2; k > 0; m >>= 1, k >>= 1)
#pragma unroll
      for (int q = 0; q < k; ++q) {
        const bool up = lane & m;
        const double keep = up ? s[q + k] : s[q], give = up ? s[q] : s[q + k];
        s[q] = keep + __shfl_xor(give, m);
      }
  }
#pragma unroll
  for (int m = SELF ? 32 : 4; m > 0; m >>= 1) s[0] += __shfl_xor(s[0], m);
  if ((lane & 7) == 0) red[lane >> 3][threadIdx.x >> 6] = s[0];
  __syncthreads();
  const int q = threadIdx.x;
  if (q < (SELF ? 1 : kVectors) && i0 + q < nv)
    partial[((size_t)b * pstride + i0 + q) * gridDim.x + blockIdx.x] =
        (red[q][0] + red[q][1]) + (red[q][2] + red[q][3]);
}

// out[b*ostride + i] = sum of vector i's partial products.  Grid: (nv, B), 64 threads.
static __global__ __launch_bounds__(64) void k_total(const double* __restrict__ partial, int pstride,
                                              int nchunk, double* __restrict__ out, int ostride,
                                              Gate gate) {
  const int b = blockIdx.y, i = blockIdx.x;
  if (gate.skips(b)) return;
  const double* p = partial + ((size_t)b * pstride + i) * nchunk;
  double s = 0.0;
  for (int c = threadIdx.x; c < nchunk; c += 64) s += p[c];
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m);
  if (threadIdx.x == 0) out[(size_t)b * ostride + i] = s;
}

// w = (w - sub) - sum_{i < nv} h_i V_i with h_i the sums of the partial products,
// which go to hout[b*hstride + i]; norm (may be null): the updates' partial sums of
// w . w, npart[b*gridDim.x + update]; -1 first for a skipped instance.
// Grid: (updates, B); LDS: nv doubles.  At n = 4416: dots 5.8-6.8 us for 8-40 vectors, update 5.4 us.
static __global__ __launch_bounds__(kThreads) void k_project(double* __restrict__ w, Basis V,
                                                      const double* __restrict__ sub, int n,
                                                      int nv, const double* __restrict__ partial,
                                                      int pstride, int nchunk,
                                                      double* __restrict__ hout, int hstride,
                                                      double* __restrict__ npart, Gate gate) {
  constexpr int LANES = 16;
  static_assert(kUpdate == kThreads, "one entry per thread");
  extern __shared__ double h[];
  __shared__ double tmp[kThreads / 64];
  const int b = blockIdx.y;
  if (gate.skips(b)) {
    if (npart && blockIdx.x == 0 && threadIdx.x == 0) npart[(size_t)b * gridDim.x] = -1.0;
    return;
  }
  const size_t o = (size_t)b * n;
  const int e = blockIdx.x * kUpdate + threadIdx.x, ec = e < n ? e : 0;
  const double* v = V.at + o + ec;
  double a[kAhead];
#pragma unroll
  for (int i = 0; i < kAhead; ++i) a[i] = v[(i < nv ? i : nv - 1) * V.ld];
  double y = w[o + ec];
  if (sub) y -= sub[o + ec];
  const int lane = threadIdx.x % LANES;
  for (int i = threadIdx.x / LANES; i < nv; i += kThreads / LANES) {
    const double* p = partial + ((size_t)b * pstride + i) * nchunk;
    double t = 0.0;
    for (int c = lane; c < nchunk; c += LANES) t += p[c];
#pragma unroll
    for (int m = LANES / 2; m > 0; m >>= 1) t += __shfl_xor(t, m);
    if (lane == 0) {
      h[i] = t;
      if (blockIdx.x == 0) hout[(size_t)b * hstride + i] = t;
    }
  }
  lds_barrier();
  double s = 0.0;
  for (int i0 = 0; i0 < nv; i0 += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (i0 + i < nv) s = fma(h[i0 + i], a[i], s);
    if (i0 + kAhead >= nv) break;
#pragma unroll
    for (int i = 0; i < kAhead; ++i) a[i] = v[(i0 + kAhead + i < nv ? i0 + kAhead + i : nv - 1) * V.ld];
  }
  y -= s;
  if (e < n) w[o + e] = y;
  if (!npart) return;
  const double q = block_sum(e < n ? y * y : 0.0, tmp);
  if (threadIdx.x == 0) npart[(size_t)b * gridDim.x + blockIdx.x] = q;
}

// ||w||^2 of instance b from its partial sums, in every thread.
__device__ __forceinline__ double norm_total(const double* npart, int nupd, double* tmp) {
  double s = 0.0;
  for (int c = threadIdx.x; c < nupd; c += kThreads) s += npart[c];
  return block_sum(s, tmp);
}

// w *= 1 / ||w|| over one update (nothing for a zero w).
__device__ __forceinline__ void scale_update(double* w, int n, double norm) {
  const double inv = norm > 0.0 ? 1.0 / norm : 1.0;
#pragma unroll
  for (int u = 0; u < kUpdate / kThreads; ++u) {
    const int e = blockIdx.x * kUpdate + threadIdx.x + u * kThreads;
    if (e < n) w[e] *= inv;
  }
}

// out[b*ostride + i] = V_i . (x - sub), i < nv, summed (a launch more than k_project).
inline int launch_dots(Basis V, const double* x, const double* sub, int n, int nv, int pstride,
                       double* partial, int B, Gate gate, hipStream_t s) {
  const dim3 grid(chunks(n), (nv + kVectors - 1) / kVectors, B);
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, s, V, x, sub, n, nv, pstride, partial, gate);
  };
  if (V.at)
    sub ? run(k_dots<false, true>) : run(k_dots<false, false>);
  else
    sub ? run(k_dots<true, true>) : run(k_dots<true, false>);
  return hip_check(hipGetLastError(), "k_dots");
}

inline int launch_total(const double* partial, int pstride, int n, int nv, double* out,
                        int ostride, int B, Gate gate, hipStream_t s) {
  hipLaunchKernelGGL(k_total, dim3(nv, B), dim3(64), 0, s, partial, pstride, chunks(n), out,
                     ostride, gate);
  return hip_check(hipGetLastError(), "k_total");
}

inline int launch_project(double* w, Basis V, const double* sub, int n, int nv,
                          const double* partial, int pstride, double* hout, int hstride,
                          double* npart, int B, Gate gate, hipStream_t s) {
  hipLaunchKernelGGL(k_project, dim3(updates(n), B), dim3(kThreads), nv * sizeof(double), s, w, V,
                     sub, n, nv, partial, pstride, chunks(n), hout, hstride, npart, gate);
  return hip_check(hipGetLastError(), "k_project");
}

}  // namespace krylov
}  // namespace sddc
