// Chains: the back substitutions of the implicit solves row by row, float64.
//   A4_BSub_TSTEP_V2   (Matrix_Operators.py:1115-1194)  field 0 (psi)
//   NAB2_BSub_TSTEP_V2 (Matrix_Operators.py:1033-1086)  fields 1 (T), 2 (S)
//
// Each field has two independent chains (the two row parities).  A chain is a
// linear recurrence over its rows, high to low: a state vector (NAB2: the
// running sum b, nr values; A4: the running sums f_e and bf_e, 2 nr values)
// is updated after every row, and the row's solution is Linv_row applied to
// g_row plus terms in the state.
//
// The products run on the float64 matrix cores, four instances at a time
// (sddc_frag.h): the running state, the right-hand side and the result of a
// (row, instance) all live in one lane, and the operator entries in registers
// serve the NG groups of four instances of a workgroup.  The vectors are
// exchanged through LDS.  Rows r >= nr are padding: their matrix rows and
// columns are zero, their values stay finite, never reach a real row through
// the zero columns, and are not stored.  Instances past the batch read the
// last real instance and are not stored.  Operator data of the next KD rows is
// loaded into registers ahead of use.
#pragma once
#include "sddc_frag.h"

namespace sddc {

constexpr int kFeedPad = 16;   // spare blocks past the last row that a block feed may read

struct ChainArgs {
  const double* G;          // right-hand sides, field f of instance b at b*gstride+goff[f]
  double* X;                // solutions, b*xstride + xoff[f]
  double* P;                // psi suffix sums [B][N] or null
  const double* Lq[3];      // block inverses per field, block index jj = K-1-row
  const double* D2q;        // D2 of the A4 solve (one block, all modes)
  const double* vecs;
  long long gstride, xstride;
  long long goff[3], xoff[3];
  int K, nr, B, symmetric, fields_mask;
  double dtf[3];            // Pr*dt, dt, Tau*dt
};

// The lane's place in a workgroup that holds the instances [4 NG group, ...):
// its radial row and its places in the LDS vectors.
template <int NRS, int NG>
struct Lanes {
  int lane, r, rr;         // rr: r clamped to the real rows
  unsigned lo;             // byte offset of the lane's operator entries
  bool put;                // r has a place in the LDS vectors
  int wp[NG];              // LDS position of (instance of the lane, r); past the arrays if none
  bool st[NG];             // (row, instance) is a real one
  __device__ __forceinline__ Lanes(const ChainArgs& a, int group, int wave, int stride) {
    lane = threadIdx.x & 63;
    r = 16 * wave + (lane & 15);
    rr = r < a.nr ? r : a.nr - 1;
    put = r < NRS;
    // lanes past the last column group of rows (NRS is a multiple of 8) read
    // the entries of the row eight above: the same cache lines, so the padding
    // of the last tile is not streamed; their results are never used
    lo = 16u * (unsigned)(put ? lane : lane - 8);
    const int t0 = lane >> 4, b0 = 4 * NG * group;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const int t = 4 * i + t0;
      st[i] = r < a.nr && b0 + t < a.B;
      wp[i] = put ? t * stride + r : 4 * NG * stride + lane;
    }
  }
};

// Wavefronts 0 .. WR-1 run the chain, one more (the carrier) moves the data of
// its rows: a row is a serial chain of an LDS write, a barrier, LDS reads,
// dependent matrix instructions and the update, and a right-hand-side load or a
// solution store in it (64 lanes over four instances) costs 25-45 ns of issue
// each, measured, beside the wait for the oldest of them that the in-order
// memory counter adds to every wait for operator data.  The carrier loads the
// right-hand sides some rows ahead into registers, puts row k + 3 into a ring
// of four LDS slots while row k runs, and stores the results the chain left in
// LDS.  With three chain wavefronts (N_r = 40) it takes the CU's idle SIMD.
// LDS of one workgroup, in doubles (XB: an [instance][entry] array and 64
// places for lanes with no entry):
//   [0, 2 XB)        exchange buffers
//   [2 XB, 6 XB)     ring of right-hand sides, row q of the chain in slot q % 4
//   [6 XB, 8 XB)     solutions, row q in slot q % 2
template <int NRS, int NG>
struct LdsMap {
  static constexpr int XB = 4 * NG * CShape<NRS>::XS + 64;
  static constexpr int G = 2 * XB, F = 6 * XB, SIZE = 8 * XB;
};

// The operator blocks of the rows to come: a uniform pointer that moves by
// one row per fetch.  Past the chain's last row it runs on (the block arrays
// end in kFeedPad spare blocks) into values that are not used.
template <int NRS>
struct BlockFeed {
  using S = CShape<NRS>;
  const double* l;
  unsigned lo;
  __device__ __forceinline__ BlockFeed(const double* blocks, int w, unsigned lane_off, int K,
                                       int row)
      : l(blocks + (size_t)(K - 1 - row) * S::BLK + w * S::NQ * 128), lo(lane_off) {}
  __device__ __forceinline__ void next(double2 (&blk)[S::NQ]) {
    load_blk<S::NQ>(blk, lane_at(l, opaque(lo)));
    l += 2 * S::BLK;
  }
};

// The carrier of n rows from row0 down.  A4: also stores P_row = f_e, found in
// exchange buffer 0.  Barriers: one after the prologue, one (A4: two) per row,
// one at the end, as in the chains.
template <int NRS, int NG, bool A4>
__device__ __forceinline__ void carry(const ChainArgs& a, int field, int group, int row0, int n,
                                      double* xs) {
  using M = LdsMap<NRS, NG>;
  constexpr int XS = CShape<NRS>::XS;
  constexpr int NI = (4 * NG * NRS + 63) / 64;   // (instance, entry) pairs per lane, at most
  constexpr int R = 6;                           // rows in registers
  const int lane = threadIdx.x & 63, nr = a.nr, b0 = 4 * NG * group;
  const size_t N = (size_t)a.K * nr;
  const double* gb = a.G + (size_t)b0 * a.gstride + a.goff[field];
  double* xb = a.X + (size_t)b0 * a.xstride + a.xoff[field];
  double* pb = (A4 && a.P) ? a.P + (size_t)b0 * N : nullptr;
  unsigned go[NI], xo[NI], po[NI];
  int lp[NI];
  bool st[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int e = lane + 64 * i, t = e / nr, r = e - t * nr;
    const bool in = t < 4 * NG;
    const int tc = !in ? 0 : (b0 + t < a.B ? t : a.B - 1 - b0);
    go[i] = 8u * (unsigned)(tc * a.gstride + r);
    xo[i] = 8u * (unsigned)(tc * a.xstride + r);
    po[i] = 8u * (unsigned)(tc * (long long)N + r);
    lp[i] = in ? t * XS + r : 4 * NG * XS + lane;
    st[i] = in && b0 + t < a.B;
  }
  // entries nr .. NRS-1 of the ring stay zero (they meet zero operator columns)
  for (int e = lane; e < 4 * M::XB; e += 64) xs[M::G + e] = 0.0;
  auto load = [&](int q, double (&v)[NI]) {
    const int j = row0 - 2 * q;   // past the chain: row 0 or 1 again
    const double* g = gb + (size_t)(j >= 0 ? j : j & 1) * nr;
#pragma unroll
    for (int i = 0; i < NI; ++i) v[i] = *lane_at(g, opaque(go[i]));
  };
  double v[R][NI], first[3][NI];
#pragma unroll
  for (int d = 0; d < 3; ++d) load(d, first[d]);
#pragma unroll
  for (int d = 0; d < R; ++d) load(3 + d, v[d]);
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int i = 0; i < NI; ++i) xs[M::G + d * M::XB + lp[i]] = first[d][i];
  lds_barrier();
  int q = 0;   // the row of the chain
  auto row = [&](int d) {
    lds_barrier();
    double f[NI], pv[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      f[i] = xs[M::F + ((q + 1) & 1) * M::XB + lp[i]];   // row q - 1
      if (A4) pv[i] = xs[lp[i]];
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) xs[M::G + ((q + 3) & 3) * M::XB + lp[i]] = v[d][i];
    load(q + 3 + R, v[d]);
    if (q > 0) {
      double* x = xb + (size_t)(row0 - 2 * q + 2) * nr;
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (st[i]) *lane_at(x, opaque(xo[i])) = f[i];
    }
    if (A4 && pb) {
      double* p = pb + (size_t)(row0 - 2 * q) * nr;
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (st[i]) *lane_at(p, opaque(po[i])) = pv[i];
    }
    if (A4) lds_barrier();
    ++q;
  };
  while (q + R <= n) {
#pragma unroll
    for (int d = 0; d < R; ++d) row(d);
  }
#pragma unroll
  for (int d = 0; d < R - 1; ++d)
    if (q < n) row(d);
  lds_barrier();
  double* x = xb + (size_t)(row0 - 2 * (n - 1)) * nr;
#pragma unroll
  for (int i = 0; i < NI; ++i)
    if (st[i]) *lane_at(x, xo[i]) = xs[M::F + ((n - 1) & 1) * M::XB + lp[i]];
}

template <int NRS, int NG, int KD>
__device__ __forceinline__ void chain_nab2(const ChainArgs& a, int field, int group, int wave,
                                           int row0, int n, double* xs) {
  using S = CShape<NRS>;
  using M = LdsMap<NRS, NG>;
  const Lanes<NRS, NG> ln(a, group, wave, S::XS);
  const double dtf = a.dtf[field];
  double2 blk[KD][S::NQ];
  BlockFeed<NRS> feed(a.Lq[field], wave, ln.lo, a.K, row0);
#pragma unroll
  for (int d = 0; d < KD; ++d) feed.next(blk[d]);
  drain_loads();
  double b[NG];
  lds_barrier();
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    b[g] = 0.0;
    xs[ln.wp[g]] = xs[M::G + ln.wp[g]];
  }
  int q = 0;
  auto row = [&](int d) {
    // NAB2 (Matrix_Operators.py:1061-1083): f_j = Linv (g_j - c_j b),
    // c_0 = 1/2; then b += 2 dt j f_j for row j-2.
    const int j = row0 - 2 * q;
    lds_barrier();
    double2 xv[NG][S::NQ];
    double gn[NG], f[NG];
    load_vec<S::NQ, NG>(xv, xs + (q & 1) * M::XB, S::XS, ln.lane);
#pragma unroll
    for (int g = 0; g < NG; ++g) gn[g] = xs[M::G + ((q + 1) & 3) * M::XB + ln.wp[g]];
    const double alpha = 2.0 * dtf * j;
    const double cn = (j == 2) ? 0.5 : 1.0;   // c of the next row
    product<S::NQ, NG>(f, blk[d], xv);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      b[g] = b[g] + alpha * f[g];
      xs[((q + 1) & 1) * M::XB + ln.wp[g]] = gn[g] - cn * b[g];
      xs[M::F + (q & 1) * M::XB + ln.wp[g]] = f[g];
    }
    pin_schedule();
    feed.next(blk[d]);
    ++q;
  };
  while (q + KD <= n) {
#pragma unroll
    for (int d = 0; d < KD; ++d) row(d);
  }
#pragma unroll
  for (int d = 0; d < KD - 1; ++d)
    if (q < n) row(d);
  lds_barrier();
}

// A4 (Matrix_Operators.py:1141-1164), dt = Pr dt, j = row + 1:
// b = dt bjt (L1 f_e + IR4 bf_e) - bjt IR2 f_e with L1 = D2 + bj IR4;
// f = Linv (g + b); bf_e += bj f + bjt f_e; f_e += f.  f_e is also the
// same-parity suffix sum P of the row.
// D2 f_e needs an exchange of its own: f_e is exchanged, D2 f_e is
// formed with D2 (the same block for every mode) held in registers, then the
// right-hand side is exchanged, and a row streams one block.  Carrying D2 f_e
// as a state instead (from (D2 Linv) times the same vector: one exchange, two
// blocks per row) was slower, 117 against 102 us for 64 instances at
// N_fm = 512, N_r = 40: a CU draws about 58 GB/s of operator data from beyond
// its L2, which two blocks per row use up.
// fe and bfe: the state above row0 (zero at the top).
template <int NRS, int NG, int KD>
__device__ __forceinline__ void chain_a4(const ChainArgs& a, int group, int wave, int row0, int n,
                                         double (&fe)[NG], double (&bfe)[NG], double* xs) {
  using S = CShape<NRS>;
  using M = LdsMap<NRS, NG>;
  const Lanes<NRS, NG> ln(a, group, wave, S::XS);
  const double dta = a.dtf[0];
  const double ir4 = a.vecs[V_IR4A4 * S::NRP + ln.rr];
  const double ir2 = a.vecs[V_IR2A4 * S::NRP + ln.rr];
  double2 d2[S::NQ];
  load_blk<S::NQ>(d2, lane_at(a.D2q + wave * S::NQ * 128, ln.lo));
  double2 blk[KD][S::NQ];
  BlockFeed<NRS> feed(a.Lq[0], wave, ln.lo, a.K, row0);
#pragma unroll
  for (int d = 0; d < KD; ++d) feed.next(blk[d]);
  drain_loads();
#pragma unroll
  for (int g = 0; g < NG; ++g) xs[ln.wp[g]] = fe[g];
  lds_barrier();
  int q = 0;
  auto row = [&](int d) {
    const double jp = (double)(row0 - 2 * q + 1);
    const double bj = -jp * (jp + 1.0), bjt = -2.0 * jp;
    const double c1 = dta * bjt, c4 = c1 * ir4, c2 = bjt * ir2;
    // buffer 0 carries f_e, buffer 1 the right-hand side; the barrier after
    // buffer 1 is written orders every read of buffer 0 before its next write
    lds_barrier();
    double2 xv[NG][S::NQ];
    double pre[NG], t[NG], f[NG];
    load_vec<S::NQ, NG>(xv, xs, S::XS, ln.lane);
#pragma unroll
    for (int g = 0; g < NG; ++g)
      pre[g] = xs[M::G + (q & 3) * M::XB + ln.wp[g]] +
               (c4 * (bj * fe[g] + bfe[g]) - c2 * fe[g]);
    product<S::NQ, NG>(t, d2, xv);
#pragma unroll
    for (int g = 0; g < NG; ++g) xs[M::XB + ln.wp[g]] = c1 * t[g] + pre[g];
    lds_barrier();
    load_vec<S::NQ, NG>(xv, xs + M::XB, S::XS, ln.lane);
#pragma unroll
    for (int g = 0; g < NG; ++g) bfe[g] = bfe[g] + bjt * fe[g];
    product<S::NQ, NG>(f, blk[d], xv);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      fe[g] = fe[g] + f[g];
      xs[ln.wp[g]] = fe[g];
      xs[M::F + (q & 1) * M::XB + ln.wp[g]] = f[g];
      bfe[g] = bfe[g] + bj * f[g];
    }
    pin_schedule();
    feed.next(blk[d]);
    ++q;
  };
  while (q + KD <= n) {
#pragma unroll
    for (int d = 0; d < KD; ++d) row(d);
  }
#pragma unroll
  for (int d = 0; d < KD - 1; ++d)
    if (q < n) row(d);
  lds_barrier();
}

// Eq_SYM keeps odd psi rows and even T/S rows (Matrix_Operators.py:1054,1166).
__device__ __forceinline__ bool parity_is_zero(int symmetric, int field, int parity) {
  return symmetric && (field == 0 ? parity == 0 : parity == 1);
}

struct Plan;
// The solves of c in the theta eigenbasis.
int launch_theta_solve(const Plan& p, const ChainArgs& c, hipStream_t s);

}  // namespace sddc
