// Small matrix products on the float64 matrix cores, shared by the solves.
//
// Every product is (matrix) x (vectors of four instances) with
// v_mfma_f64_4x4x4: one instruction is four independent 4x4x4 blocks, used as
// 16 rows of the operator times four instances over four columns.  Lane l
//   supplies the operator entry  row 16w + l%16, column group l/16,
//   supplies the vector entry    instance l%4,   column group l/16,
//   receives the result          row 16w + l%16, instance l/16,
// so a wavefront owns 16 radial rows of four instances, one result per lane.
// Matrices are stored in that order ("fragments"): element (r, c) of an
// NRP x NC matrix sits at
//   ((w*(NC/8) + q)*64 + l)*2 + h,  r = 16w + l%16,  c = 8q + 2(l/16) + h,
// so one 16-byte load per lane (1 KiB of consecutive memory per wavefront)
// feeds two instructions.  The vectors come from LDS as [instance][entry]; a
// lane reads its two entries of a q with one 16-byte read.  Two accumulators
// per product (even and odd h) halve the length of the dependent chain (an
// instruction issues every 17-20 cycles and its result is ready after 44,
// measured).
#pragma once
#include "sddc_internal.h"

namespace sddc {

template <int NRS>
struct CShape {
  static constexpr int NRP = ((NRS + 15) / 16) * 16;
  static constexpr int WR = NRP / 16;     // wavefronts per workgroup
  static constexpr int NQ = NRS / 8;      // 16-byte loads per lane of an NRP x NRS block
  static constexpr int BLK = NRP * NRS;   // doubles per NRP x NRS block
  // LDS stride of an instance's vector: an odd multiple of 8 doubles, so the
  // four instances of a read fall in different banks
  static constexpr int XS = (NRS / 8) % 2 ? NRS : NRS + 8;
};

template <int NQ>
__device__ __forceinline__ void load_blk(double2 (&a)[NQ], const double* p) {
#pragma unroll
  for (int q = 0; q < NQ; ++q) a[q] = *reinterpret_cast<const double2*>(p + q * 128);
}

// The lane's entries of the vectors of instance group g: xs is [4 NG][stride].
template <int NQ, int NG>
__device__ __forceinline__ void load_vec(double2 (&x)[NG][NQ], const double* xs, int stride,
                                         int lane) {
  const double* p = xs + (lane & 3) * stride + 2 * (lane >> 4);
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      x[g][q] = *reinterpret_cast<const double2*>(p + 4 * g * stride + 8 * q);
}

__device__ __forceinline__ void pin_schedule() { __builtin_amdgcn_sched_barrier(0); }

// y[g] = (m x)[row of the lane][instance of the lane], every group.
template <int NQ, int NG>
__device__ __forceinline__ void product(double (&y)[NG], const double2 (&m)[NQ],
                                        const double2 (&x)[NG][NQ]) {
  double c0[NG], c1[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) c0[g] = c1[g] = 0.0;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      c0[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(x[g][q].x, m[q].x, c0[g], 0, 0, 0);
      c1[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(x[g][q].y, m[q].y, c1[g], 0, 0, 0);
    }
  }
#pragma unroll
  for (int g = 0; g < NG; ++g) y[g] = c0[g] + c1[g];
}

// A wave-uniform pointer plus a lane's byte offset: the compiler can then
// address with a scalar base and one 32-bit vector offset, so a loop that
// moves the base from row to row spends no vector instructions on addresses.
__device__ __forceinline__ const double* lane_at(const double* base, unsigned byte_off) {
  return reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + byte_off);
}
__device__ __forceinline__ double* lane_at(double* base, unsigned byte_off) {
  return reinterpret_cast<double*>(reinterpret_cast<char*>(base) + byte_off);
}

// A loop-invariant lane offset made opaque to loop-invariant code motion:
// otherwise the compiler adds it to each uniform base once, outside the
// loop, as a 64-bit vector address that every row then advances with vector
// adds.  No instruction is emitted.
__device__ __forceinline__ unsigned opaque(unsigned v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Fragment order of an nrows x ncols row-major matrix (leading dimension lda)
// in an NRP x NC tile (zero padded).
void pack_frag(const double* A, int nrows, int ncols, int lda, int NRP, int NC, double* out);

}  // namespace sddc
