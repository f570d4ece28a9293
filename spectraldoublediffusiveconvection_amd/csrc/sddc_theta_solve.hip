// The implicit solves without their chains: the three solves of the step in
// the eigenbasis of the theta operator.
//
// The matrices the solves invert are polynomials in one theta operator L that
// couples the rows of one parity, with radial matrices as coefficients:
//   A4    A2 + IR2 L - h (D4 + D2 L + IR4 L^2)  on sine rows
//         (Matrix_Operators.py:1089-1194; L f = bj f_j + bjt sum_{k>j} f_k),
//   NAB2  r^2 - h (r^2 Lap + L)                 on cosine rows
//         (Matrix_Operators.py:1014-1086).
// L is upper triangular with the distinct eigenvalues -j(j+1), so
// L = V Lambda W with V unit upper triangular and W = V^-1 (the expansions of
// Legendre functions in sines and cosines; condition number 5-22 for 64-512
// modes with normalised columns), and in the variables W f every mode solves
// with its own pre-inverted block:
//   f = V blockdiag(Linv_j) W g.
// The K/2-row recurrence becomes two triangular products and K independent
// blocks, in three launches:
//   k_theta_forward  W g;
//   k_theta_blocks   the modes' blocks;
//   k_theta_back     V of the result, and for psi the suffix sums P, whose
//                    rows are those of V summed over the rows above.
// It takes more arithmetic than the chains (n = K/2: about n nr against 2 nr^2
// multiply-adds per row and field), all of it parallel: the form of small and
// medium batches, whose chains wait for latency.
//
// Accuracy.  The given A4 blocks are inverses to a few digits less than float64
// (their condition number is up to 1e9 at low modes), and chain and eigenbasis
// carry that differently.  For a right-hand side with all modes, at N_fm = 512,
// N_r = 40, dt = 5e-3, both are 4.7e-13 from the exact solution of the
// discretised operators and 2.6e-13 from each other; T and S differ by 2e-15.
// Most of that comes from the lowest modes, so the lowest psi rows
// are solved by the chain, entered with the state of the rows above, which is
// linear in their eigenbasis solution: with 32 of the 512 rows left to the
// chain the difference is 2.4e-14; at N_fm = 64, N_r = 20 it is
// 2e-14 with none.  The plan measures it with a seeded right-hand side of all
// modes and takes the fewest rows (in steps of four per parity) that meet
// kStepTol.  That is no bound for every right-hand side: one confined to a few
// rows above the chain's shows the blocks' own error, 1e-14 to 1.5e-13 from the
// chain at 128/30 and up to 1.5e-12 at 300/48 (single rows and bands of 4 to 64,
// dt = 5e-3, 12 low rows).  Against the exact solution the worst such case is the
// chain's own (chain and this form: 4.7e-13 both at 128/30, 7.7e-12 both at 300/48,
// 1.1e-12 both at 512/40; single rows between 0.5 and 4.7 times the chain's).  The
// back substitution entry point (sddc_bsub), whose result is defined by the blocks
// it is given, therefore takes the chains in every plan.  The low rows run in the
// last launch beside the back products.
//
// V, W: 16-row tiles in the fragment order of sddc_frag.h, for 16x16x4 matrix
// instructions with 16 modes as rows and 16 radial points as columns.  A
// workgroup takes one tile of one chain of one instance; its wavefronts split
// the tile's columns into kRanges runs.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <vector>

#include "sddc_chain.h"

namespace sddc {

typedef double v4d_th __attribute__((ext_vector_type(4)));

constexpr int kThetaModes = 16;    // modes per tile
constexpr int kEntryModes = 4;     // modes per partial sum of the entry state
constexpr int kThetaMats = 10;     // W, V: (sine, cosine) x (even, odd rows); U: sine
// Largest relative difference to the chains, measured with one right-hand side of
// all modes (see the head of this file): psi, which takes low rows until it is met,
// and T and S, which keep the chains where it is not.
constexpr double kStepTol = 2.5e-14, kHeatTol = 5e-15;

struct ThetaArgs {
  ChainArgs c;
  double* GH;             // W g: [3][2][n modes][B][RP]
  double* H;              // blocks' results [B][3][2][n][nr]
  double* EN;             // partial entry states [B][2][tiles * 4][2][NRP]
  const double* W[2][2];  // [0 sine, 1 cosine][row parity]
  const double* V[2][2];
  const double* U[2];     // suffix sums of the rows of V (sine)
  const double* entry[2]; // per parity: row 16 low - 1 of U, the same times -j(j+1)
  long long N;
  int n, nq, tiles, rp;   // rp: nr rounded up to even (16-byte loads)
  int low;                // psi rows per parity left to the chain
};

constexpr int kRanges = 4;         // runs of a tile's columns

// Column groups of the matrices, and run i of a tile (the entries left of its
// diagonal are zero).  All are even, in pairs of groups.
__host__ __device__ inline int theta_nq(int tiles) { return 2 * tiles; }
__device__ __forceinline__ int run_begin(int tile, int nq, int i) {
  const int q0 = 2 * tile;
  return q0 + (nq - q0) / 2 * i / kRanges * 2;
}

// Column groups qa .. qb of one tile times the rows of one chain in memory: row b
// at in + b*stride, columns 16w + lane % 16 of every w at off[w].  An operand of
// the tile serves all WR column groups.
template <int WR>
__device__ __forceinline__ void run_product(v4d_th (&acc)[WR], const double* tile,
                                            const double* in, int stride,
                                            const unsigned (&off)[WR], int qa, int qb, int n,
                                            int lane) {
  struct Stage {
    double2 av[2];
    double b[2][2][WR];
  } s[2];
  const int kk = 2 * (lane >> 4);
  auto load = [&](Stage& d, int q) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      d.av[i] = *reinterpret_cast<const double2*>(lane_at(tile, 1024u * (q + i) + 16u * lane));
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // rows past n meet zero columns of the tile: any row of the chain will do
        const int c = 8 * (q + i) + kk + h;
        const unsigned row = 8u * (unsigned)((c < n ? c : n - 1) * stride);
#pragma unroll
        for (int w = 0; w < WR; ++w) d.b[i][h][w] = *lane_at(in, row + off[w]);
      }
    }
  };
  auto multiply = [&](const Stage& d) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int w = 0; w < WR; ++w)
          acc[w] = __builtin_amdgcn_mfma_f64_16x16x4f64(h ? d.av[i].y : d.av[i].x, d.b[i][h][w],
                                                        acc[w], 0, 0, 0);
  };
  if (qa >= qb) return;
  load(s[0], qa);
  for (int q = qa; q < qb; q += 4) {
    if (q + 2 < qb) load(s[1], q + 2);
    multiply(s[0]);
    if (q + 2 >= qb) break;
    if (q + 4 < qb) load(s[0], q + 4);
    multiply(s[1]);
  }
}

// Wavefronts of a workgroup of the triangular products: a run each; the chains
// in k_theta_back need WR and a carrier.
template <int WR>
constexpr int theta_waves() { return WR < kRanges ? kRanges : WR + 1; }

// Wavefronts per SIMD that the registers of the products must allow.
template <int NRS>
constexpr int theta_occupancy() { return NRS <= 40 ? 4 : 2; }

// One tile by kRanges wavefronts, a run each; put(mode, column, value) of the
// sums, from LDS.
template <int WR, typename F>
__device__ __forceinline__ void split_tile(double* xs, const double* mat, const double* in,
                                           int stride, int tile, int nq, int n, int nr, int wave,
                                           int lane, F put) {
  constexpr int PS = 16 * WR, THREADS = 64 * theta_waves<WR>();
  if (wave < kRanges) {
    unsigned off[WR];
    v4d_th acc[WR];
#pragma unroll
    for (int w = 0; w < WR; ++w) {
      const int r = 16 * w + (lane & 15);
      off[w] = 8u * (r < nr ? r : nr - 1);
      acc[w] = (v4d_th){0.0, 0.0, 0.0, 0.0};
    }
    run_product<WR>(acc, mat + (size_t)tile * nq * 128, in, stride, off, run_begin(tile, nq, wave),
                    run_begin(tile, nq, wave + 1), n, lane);
#pragma unroll
    for (int w = 0; w < WR; ++w)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        xs[(wave * kThetaModes + (lane >> 4) + 4 * v) * PS + 16 * w + (lane & 15)] = acc[w][v];
  }
  lds_barrier();
  for (int e = threadIdx.x; e < kThetaModes * PS; e += THREADS) {
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < kRanges; ++i) sum += xs[i * kThetaModes * PS + e];
    put(tile * kThetaModes + e / PS, e % PS, sum);
  }
}

// (pair, tile) of workgroup i: the workgroups of a pair (a chain of one
// instance), which read the same rows, follow each other on one XCD (workgroup i
// runs on XCD i % 8), the longest first.
__device__ __forceinline__ int2 theta_item(int i, int tiles) {
  const int k = i / 8;
  return make_int2(k / tiles * 8 + i % 8, k % tiles);
}

// (field, parity) of type i among the fields of mask.
__device__ __forceinline__ int theta_field(int i, int mask) {
  int f = 0;
  for (int q = i >> 1; f < 3; ++f)
    if ((mask >> f) & 1) {
      if (q == 0) break;
      --q;
    }
  return f;
}

// W g: one tile of one chain of one instance.
template <int NRS>
__global__ __launch_bounds__(64 * theta_waves<CShape<NRS>::WR>(), theta_occupancy<NRS>()) void
k_theta_forward(ThetaArgs a, int pairs) {
  constexpr int WR = CShape<NRS>::WR;
  __shared__ double xs[kRanges * kThetaModes * 16 * WR];
  const int2 item = theta_item(blockIdx.x, a.tiles);
  if (item.x >= pairs) return;
  const int type = item.x / a.c.B, b = item.x % a.c.B, tile = item.y;
  const int field = theta_field(type, a.c.fields_mask), parity = type & 1, nr = a.c.nr;
  if (parity_is_zero(a.c.symmetric, field, parity)) return;
  if (field == 0 && (tile + 1) * kThetaModes <= a.low) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  double* out = a.GH + ((size_t)(2 * field + parity) * a.n * a.c.B + b) * a.rp;
  split_tile<WR>(xs, a.W[field > 0][parity],
                 a.c.G + (size_t)b * a.c.gstride + a.c.goff[field] + parity * nr, 2 * nr, tile,
                 a.nq, a.n, nr, wave, lane, [&](int m, int r, double v) {
                   if (m < a.n && r < a.rp) out[(size_t)m * a.c.B * a.rp + r] = r < nr ? v : 0.0;
                 });
}

// Sets of WR wavefronts in a workgroup of k_theta_blocks.
template <int WR>
constexpr int theta_sets() { return WR < 4 ? 4 : 2; }

// The blocks of four consecutive modes of one (field, parity), one mode per set
// of WR wavefronts (two at WR = 4), and 4 NG instances; psi: also their part of
// the low rows' entry state.  The workgroups of one mode group, which read the
// same operator blocks, follow each other on one XCD (workgroup i runs on XCD
// i % 8).
template <int NRS, int NG>
__global__ __launch_bounds__(64 * CShape<NRS>::WR * theta_sets<CShape<NRS>::WR>()) void
k_theta_blocks(ThetaArgs a, int types, int groups) {
  using S = CShape<NRS>;
  constexpr int SETS = theta_sets<S::WR>(), PM = kEntryModes / SETS;
  __shared__ double ys[kEntryModes * 4 * NG * S::NRP];
  const int quads = (a.n + kEntryModes - 1) / kEntryModes;
  const int k = blockIdx.x / 8, mg = k / groups * 8 + blockIdx.x % 8;
  if (mg >= types * quads) return;
  const int type = mg / quads, quad = mg % quads;
  const int field = theta_field(type, a.c.fields_mask), parity = type & 1, nr = a.c.nr;
  if (parity_is_zero(a.c.symmetric, field, parity)) return;
  if (field == 0 && quad * kEntryModes < a.low / kThetaModes * kThetaModes) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int w = wave % S::WR, set = wave / S::WR, t0 = lane >> 4;
  const int b0 = k % groups * 4 * NG, r = 16 * w + (lane & 15), rr = r < nr ? r : nr - 1;
  const unsigned lo = 16u * (unsigned)(r < NRS ? lane : lane - 8);
  double2 blk[PM][S::NQ];
#pragma unroll
  for (int d = 0; d < PM; ++d) {
    const int m = quad * kEntryModes + set * PM + d, j = parity + 2 * (m < a.n ? m : a.n - 1);
    load_blk<S::NQ>(blk[d], lane_at(a.c.Lq[field] + (size_t)(a.c.K - 1 - j) * S::BLK +
                                        w * S::NQ * 128, lo));
  }
  const bool entry = field == 0 && a.low > 0;
#pragma unroll
  for (int d = 0; d < PM; ++d) {
    const int mq = set * PM + d, m = quad * kEntryModes + mq, mc = m < a.n ? m : a.n - 1;
    const double* gh = a.GH + ((size_t)(2 * field + parity) * a.n + mc) * a.c.B * a.rp;
    double2 xv[NG][S::NQ];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int b = b0 + 4 * g + (lane & 3), bc = b < a.c.B ? b : a.c.B - 1;
#pragma unroll
      for (int q = 0; q < S::NQ; ++q) {
        // entries past nr (the padding to rp is zero; beyond it, entry 0) meet
        // zero operator columns
        const int c = 8 * q + 2 * t0;
        xv[g][q] = *reinterpret_cast<const double2*>(gh + (size_t)bc * a.rp + (c < a.rp ? c : 0));
      }
    }
    double y[NG];
    product<S::NQ, NG>(y, blk[d], xv);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int b = b0 + 4 * g + t0;
      if (m < a.n && b < a.c.B && r < nr)
        a.H[((((size_t)b * 3 + field) * 2 + parity) * a.n + m) * nr + r] = y[g];
      if (entry) ys[(mq * 4 * NG + 4 * g + t0) * S::NRP + r] = y[g];
    }
  }
  if (!entry) return;
  lds_barrier();
  const double* eu = a.entry[parity];
  for (int g = set; g < NG; g += SETS) {
    const int b = b0 + 4 * g + t0;
    double sf = 0.0, sb = 0.0;
#pragma unroll
    for (int d = 0; d < kEntryModes; ++d) {
      const int m = quad * kEntryModes + d;
      const double y = ys[(d * 4 * NG + 4 * g + t0) * S::NRP + r];
      sf = fma(m < a.n ? eu[m] : 0.0, y, sf);
      sb = fma(m < a.n ? eu[a.n + m] : 0.0, y, sb);
    }
    if (b < a.c.B && r < nr) {
      double* e = a.EN + (((size_t)b * 2 + parity) * a.tiles * 4 + quad) * 2 * S::NRP;
      e[rr] = sf;
      e[S::NRP + rr] = sb;
    }
  }
}

// The first workgroups: the chain of the low psi rows of one parity and four
// instances.  The others: one tile of V of one chain of one instance, or of the
// suffix sums of psi (the types behind the fields').
template <int NRS, int KD>
__global__ __launch_bounds__(64 * theta_waves<CShape<NRS>::WR>(), theta_occupancy<NRS>()) void
k_theta_back(ThetaArgs a, int chains, int types) {
  using S = CShape<NRS>;
  constexpr int SUMS = kRanges * kThetaModes * S::WR * 16, LDS = LdsMap<NRS, 1>::SIZE;
  __shared__ __align__(16) double xs[LDS > SUMS ? LDS : SUMS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nr = a.c.nr, t0 = lane >> 4;
  if ((int)blockIdx.x < chains) {
    const int parity = blockIdx.x & 1, group = blockIdx.x >> 1;
    const int n = a.low, row0 = parity + 2 * (n - 1);
    const int r = 16 * wave + (lane & 15), rr = r < nr ? r : nr - 1;
    if (parity_is_zero(a.c.symmetric, 0, parity)) {
      for (int q = 0; q < n && wave < S::WR; ++q) {
        const int b = 4 * group + t0;
        const size_t o = (size_t)(row0 - 2 * q) * nr + r;
        if (r >= nr || b >= a.c.B) continue;
        a.c.X[(size_t)b * a.c.xstride + a.c.xoff[0] + o] = 0.0;
        if (a.c.P) a.c.P[(size_t)b * a.N + o] = 0.0;
      }
      return;
    }
    if (wave == S::WR) {
      carry<NRS, 1, true>(a.c, 0, group, row0, n, xs);
      return;
    }
    if (wave > S::WR) {   // no work: the chain's barriers only
      for (int i = 0; i < 2 * n + 2; ++i) lds_barrier();
      return;
    }
    // the entry state: the lanes of a radial point take every fourth of the
    // quads' partial sums, kEntryBurst of two instances in flight
    constexpr int kEntryBurst = 6;
    const int quads = (a.n + kEntryModes - 1) / kEntryModes;
    double sf[4] = {0.0, 0.0, 0.0, 0.0}, sb[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i0 = 0; i0 < 4; i0 += 2) {
      if (4 * group + i0 >= a.c.B) break;
      for (int q = a.low / kEntryModes + t0; q < quads; q += 4 * kEntryBurst) {
        double f[2][kEntryBurst], g[2][kEntryBurst];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int b = 4 * group + i0 + i < a.c.B ? 4 * group + i0 + i : a.c.B - 1;
          const double* e = a.EN + ((size_t)b * 2 + parity) * a.tiles * 4 * 2 * S::NRP + rr;
#pragma unroll
          for (int u = 0; u < kEntryBurst; ++u) {
            const size_t o = (size_t)(q + 4 * u < quads ? q + 4 * u : q) * 2 * S::NRP;
            f[i][u] = e[o];
            g[i][u] = e[o + S::NRP];
          }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int u = 0; u < kEntryBurst; ++u)
            if (q + 4 * u < quads) {
              sf[i0 + i] += f[i][u];
              sb[i0 + i] += g[i][u];
            }
      }
    }
    double fe[1] = {0.0}, bfe[1] = {0.0};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sf[i] += __shfl_xor(sf[i], 16);
      sf[i] += __shfl_xor(sf[i], 32);
      sb[i] += __shfl_xor(sb[i], 16);
      sb[i] += __shfl_xor(sb[i], 32);
      if (t0 == i && 4 * group + i < a.c.B && r < nr) {
        fe[0] = sf[i];
        bfe[0] = sb[i];
      }
    }
    chain_a4<NRS, 1, KD>(a.c, group, wave, row0, n, fe, bfe, xs);
    return;
  }
  const int2 item = theta_item(blockIdx.x - (chains + 7) / 8 * 8, a.tiles);
  if ((int)blockIdx.x < (chains + 7) / 8 * 8 || item.x >= types * a.c.B) return;
  const int type = item.x / a.c.B, b = item.x % a.c.B, tile = item.y;
  const int nfields = types / 2 - (a.c.P != nullptr ? 1 : 0);
  const bool sums = type / 2 >= nfields;   // P
  const int field = sums ? 0 : theta_field(type, a.c.fields_mask), parity = type & 1;
  if (field == 0 && (tile + 1) * kThetaModes <= a.low) return;
  double* x = (sums ? a.c.P + (size_t)b * a.N : a.c.X + (size_t)b * a.c.xstride + a.c.xoff[field]) +
              parity * nr;
  auto put = [&](int m, int r, double v) {
    if (r < nr && m < a.n && (field > 0 || m >= a.low)) x[(size_t)2 * m * nr + r] = v;
  };
  if (parity_is_zero(a.c.symmetric, field, parity)) {
    for (int e = threadIdx.x; e < kThetaModes * S::WR * 16; e += blockDim.x)
      put(tile * kThetaModes + e / (16 * S::WR), e % (16 * S::WR), 0.0);
    return;
  }
  split_tile<S::WR>(xs, sums ? a.U[parity] : a.V[field > 0][parity],
                    a.H + (((size_t)b * 3 + field) * 2 + parity) * a.n * nr, nr, tile, a.nq, a.n,
                    nr, wave, lane, put);
}

template <int NRS>
static int launch_theta_t(const ThetaArgs& a, hipStream_t s) {
  using S = CShape<NRS>;
  const int mask = a.c.fields_mask, B = a.c.B;
  const int types = 2 * ((mask & 1) + ((mask >> 1) & 1) + ((mask >> 2) & 1));
  const dim3 threads(64 * theta_waves<S::WR>());
  auto grid = [&](int pairs) { return (pairs + 7) / 8 * 8 * a.tiles; };
  hipLaunchKernelGGL((k_theta_forward<NRS>), dim3(grid(types * B)), threads, 0, s, a, types * B);
  if (int rc = hip_check(hipGetLastError(), "k_theta_forward")) return rc;
  const int quads = (a.n + kEntryModes - 1) / kEntryModes, rows = (types * quads + 7) / 8 * 8;
  auto blocks = [&](auto kernel, int ng) {
    const int groups = (B + 4 * ng - 1) / (4 * ng);
    hipLaunchKernelGGL(kernel, dim3(rows * groups), dim3(64 * S::WR * theta_sets<S::WR>()), 0, s, a,
                       types, groups);
    return hip_check(hipGetLastError(), "k_theta_blocks");
  };
  if (int rc = B <= 4 ? blocks(k_theta_blocks<NRS, 1>, 1) : blocks(k_theta_blocks<NRS, 2>, 2))
    return rc;
  const int btypes = types + (a.c.P ? 2 : 0);
  const int chains = (a.low > 0 && (mask & 1)) ? 2 * ((B + 3) / 4) : 0;
  hipLaunchKernelGGL((k_theta_back<NRS, 2>), dim3((chains + 7) / 8 * 8 + grid(btypes * B)),
                     threads, 0, s, a, chains, btypes);
  return hip_check(hipGetLastError(), "k_theta_back");
}

static int theta_tiles(int K) { return (K / 2 + kThetaModes - 1) / kThetaModes; }

// The workspaces of the solves, for B instances: arrays that are dead by then.
// W g is at most 24 bytes a mode and radial point (28 in the slabs), the
// blocks' results as large as the linear part; the partial entry states have to
// fit the products (16 bytes in mixed precision), which tiny sizes do not.
static bool theta_fits(int K, int nr, int NRP) {
  return nr >= 8 && (size_t)theta_tiles(K) * 4 * 2 * 2 * NRP * 8 <= (size_t)16 * K * nr;
}

int launch_theta_solve(const Plan& p, const ChainArgs& c, hipStream_t s) {
  ThetaArgs a;
  a.c = c;
  a.GH = static_cast<double*>(p.slabs);
  a.H = p.L;
  a.rp = p.nr + (p.nr & 1);
  a.EN = static_cast<double*>(p.F);
  a.n = p.K / 2;
  a.tiles = theta_tiles(p.K);
  a.nq = theta_nq(a.tiles);
  a.low = p.theta_low;
  a.N = (long long)p.K * p.nr;
  const size_t sz = (size_t)a.tiles * a.nq * 128;
  for (int basis = 0; basis < 2; ++basis)
    for (int par = 0; par < 2; ++par) {
      a.W[basis][par] = p.theta + (size_t)(2 * basis + par) * sz;
      a.V[basis][par] = p.theta + (size_t)(4 + 2 * basis + par) * sz;
    }
  for (int par = 0; par < 2; ++par) {
    a.U[par] = p.theta + (size_t)(8 + par) * sz;
    a.entry[par] = p.theta + kThetaMats * sz + (size_t)par * 2 * a.n;
  }
  switch (p.NRS) {
    case 8: return launch_theta_t<8>(a, s);
    case 16: return launch_theta_t<16>(a, s);
    case 24: return launch_theta_t<24>(a, s);
    case 32: return launch_theta_t<32>(a, s);
    case 40: return launch_theta_t<40>(a, s);
    case 48: return launch_theta_t<48>(a, s);
    case 56: return launch_theta_t<56>(a, s);
    case 64: return launch_theta_t<64>(a, s);
    default: return fail(SDDC_ERR_UNSUPPORTED, "unsupported radial size");
  }
}

// ---------------------------------------------------------------------------
// Host side (once per plan).
// ---------------------------------------------------------------------------
// V (unit upper triangular, columns eigenvectors of L) and W = V^-1 (rows left
// eigenvectors) of the rows of one parity, in extended precision.  The
// off-diagonal entries of a row of L are -2 u_a v_b: sine rows u = j + 1,
// v = 1; cosine rows u = c_j (1/2 for row 0, else 1), v = j.
static void theta_basis(int n, int parity, bool cosine, std::vector<double>& V,
                        std::vector<double>& W) {
  std::vector<long double> lam(n), u(n), v(n);
  for (int a = 0; a < n; ++a) {
    const long double j = parity + 2 * a;
    lam[a] = cosine ? -j * (j + 1) : -(j + 1) * (j + 2);
    u[a] = cosine ? (j == 0 ? 0.5L : 1.0L) : j + 1;
    v[a] = cosine ? j : 1.0L;
  }
  V.assign((size_t)n * n, 0.0);
  W.assign((size_t)n * n, 0.0);
  for (int c = 0; c < n; ++c) {   // column c of V, upwards
    V[(size_t)c * n + c] = 1.0;
    long double sum = v[c];
    for (int a = c - 1; a >= 0; --a) {
      const long double x = -2.0L * u[a] * sum / (lam[c] - lam[a]);
      V[(size_t)a * n + c] = (double)x;
      sum += v[a] * x;
    }
  }
  for (int a = 0; a < n; ++a) {   // row a of W, to the right
    W[(size_t)a * n + a] = 1.0;
    long double sum = u[a];
    for (int b = a + 1; b < n; ++b) {
      const long double x = -2.0L * v[b] * sum / (lam[a] - lam[b]);
      W[(size_t)a * n + b] = (double)x;
      sum += u[b] * x;
    }
  }
}

// One seeded right-hand side through the chains and the eigenbasis, on the
// host.  False when the operator set's blocks are not those of the operators
// above (the set may hold any matrices; the chains define the result then).
// Else the number of low psi rows per parity that meets kStepTol.  fields:
// those solved with blocks (the modal NAB2 solve leaves psi).
static bool theta_probe(const sddc_operators* o, int K, int nr, int fields, const double dtf[3],
                        const std::vector<double> (&V)[2][2],
                        const std::vector<double> (&W)[2][2], int& low) {
  const int n = K / 2;
  const size_t NN = (size_t)nr * nr;
  const double* inv[3] = {o->Linv_A4, o->Linv_T, o->Linv_S};
  std::vector<double> g((size_t)n * nr), f(g), h(g), t(g), x(nr);
  unsigned seed = 12345u;
  for (double& e : g) {
    seed = seed * 1664525u + 1013904223u;
    e = (double)(seed >> 8) / 8388608.0 - 1.0;
  }
  auto apply = [&](const double* M, const double* in, double* out) {
    for (int i = 0; i < nr; ++i) {
      double s = 0.0;
      for (int c = 0; c < nr; ++c) s += M[(size_t)i * nr + c] * in[c];
      out[i] = s;
    }
  };
  auto tri = [&](const std::vector<double>& M, const std::vector<double>& in,
                 std::vector<double>& out) {
    for (int a = 0; a < n; ++a) {
      double* y = out.data() + (size_t)a * nr;
      for (int i = 0; i < nr; ++i) y[i] = 0.0;
      for (int b = a; b < n; ++b) {
        const double m = M[(size_t)a * n + b];
        const double* q = in.data() + (size_t)b * nr;
        for (int i = 0; i < nr; ++i) y[i] += m * q[i];
      }
    }
  };
  // the chain of rows top .. 0 of one parity into out, the rows above given
  // (Matrix_Operators.py:1061-1083, 1141-1164)
  auto chain = [&](int fld, int par, int top, std::vector<double>& out) {
    std::vector<double> s1(nr, 0.0), s2(nr, 0.0);
    for (int a = n - 1; a >= 0; --a) {
      const int row = par + 2 * a;
      const double* L = inv[fld] + (size_t)(K - 1 - row) * NN;
      const double* ga = g.data() + (size_t)a * nr;
      double* fa = out.data() + (size_t)a * nr;
      if (fld == 0) {
        const double jp = row + 1.0, bj = -jp * (jp + 1.0), bjt = -2.0 * jp;
        if (a < top) {
          apply(o->D2_A4, s1.data(), x.data());
          for (int i = 0; i < nr; ++i) {
            const double i4 = o->IR4_A4[i], i2 = o->IR2_A4[i];
            x[i] = ga[i] + dtf[0] * bjt * (x[i] + bj * i4 * s1[i] + i4 * s2[i]) - bjt * i2 * s1[i];
          }
          apply(L, x.data(), fa);
        }
        for (int i = 0; i < nr; ++i) {
          s2[i] += bj * fa[i] + bjt * s1[i];
          s1[i] += fa[i];
        }
      } else {
        const double c = row == 0 ? 0.5 : 1.0;
        for (int i = 0; i < nr; ++i) x[i] = ga[i] - c * s1[i];
        apply(L, x.data(), fa);
        for (int i = 0; i < nr; ++i) s1[i] += 2.0 * dtf[fld] * row * fa[i];
      }
    }
  };
  auto diff = [&](const std::vector<double>& u, const std::vector<double>& v) {
    double d2 = 0.0, f2 = 0.0;
    for (size_t e = 0; e < v.size(); ++e) {
      d2 += (u[e] - v[e]) * (u[e] - v[e]);
      f2 += v[e] * v[e];
    }
    return f2 > 0.0 ? std::sqrt(d2 / f2) : (d2 == 0.0 ? 0.0 : INFINITY);
  };
  low = 0;
  for (int fld = 0; fld < fields; ++fld)
    for (int par = 0; par < 2; ++par) {
      chain(fld, par, n, f);
      tri(W[fld > 0][par], g, t);
      for (int a = 0; a < n; ++a)
        apply(inv[fld] + (size_t)(K - 1 - par - 2 * a) * NN, t.data() + (size_t)a * nr,
              h.data() + (size_t)a * nr);
      tri(V[fld > 0][par], h, t);
      if (!(diff(t, f) <= 1e-10)) return false;   // NaN counts as a mismatch
      if (fld > 0) {
        if (diff(t, f) > kHeatTol) return false;
        continue;
      }
      for (; low < n; low = std::min(n, low + kEntryModes)) {
        h = t;
        chain(0, par, low, h);
        if (diff(h, f) <= kStepTol) break;
      }
    }
  return true;
}

int build_theta(Plan& p, const sddc_operators* ops) {
  if (!theta_fits(p.K, p.nr, p.NRP)) return SDDC_OK;
  const int n = p.K / 2, tiles = theta_tiles(p.K), nq = theta_nq(tiles);
  const size_t sz = (size_t)tiles * nq * 128;
  std::vector<double> V[2][2], W[2][2], U((size_t)n * n);
  for (int basis = 0; basis < 2; ++basis)
    for (int par = 0; par < 2; ++par) theta_basis(n, par, basis == 1, V[basis][par], W[basis][par]);
  const double dtf[3] = {p.Pr * p.dt, p.dt, p.Tau * p.dt};
  if (!theta_probe(ops, p.K, p.nr, p.nab2_modal ? 1 : 3, dtf, V, W, p.theta_low)) return SDDC_OK;   // the chains solve
  std::vector<double> all(kThetaMats * sz + 4 * (size_t)n, 0.0);
  for (int basis = 0; basis < 2; ++basis)
    for (int par = 0; par < 2; ++par) {
      pack_frag(W[basis][par].data(), n, n, n, 16 * tiles, 8 * nq,
                all.data() + (size_t)(2 * basis + par) * sz);
      pack_frag(V[basis][par].data(), n, n, n, 16 * tiles, 8 * nq,
                all.data() + (size_t)(4 + 2 * basis + par) * sz);
    }
  for (int par = 0; par < 2; ++par) {
    // P_a = sum over the rows b > a of f; the state above row 16 low - 1 is
    // f_e = P of that row and bf_e = the same sum of L f = V Lambda f^
    for (int c = 0; c < n; ++c) {
      long double s = 0.0L;
      for (int a = n - 1; a >= 0; --a) {
        U[(size_t)a * n + c] = (double)s;
        s += V[0][par][(size_t)a * n + c];
      }
    }
    pack_frag(U.data(), n, n, n, 16 * tiles, 8 * nq, all.data() + (size_t)(8 + par) * sz);
    const int top = p.theta_low - 1;
    if (top < 0) continue;
    double* e = all.data() + kThetaMats * sz + (size_t)par * 2 * n;
    for (int c = top + 1; c < n; ++c) {   // zero for the chain's own rows
      const double j = par + 2 * c;
      e[c] = U[(size_t)top * n + c];
      e[n + c] = -(j + 1) * (j + 2) * e[c];
    }
  }
  SDDC_HIP(hipMalloc(&p.theta, all.size() * sizeof(double)));
  SDDC_HIP(hipMemcpy(p.theta, all.data(), all.size() * sizeof(double), hipMemcpyHostToDevice));
  return SDDC_OK;
}

}  // namespace sddc
