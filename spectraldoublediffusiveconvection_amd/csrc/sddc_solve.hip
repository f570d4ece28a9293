// The implicit solves of the step, float64 always: launches and host side.
//   A4_BSub_TSTEP_V2   (Matrix_Operators.py:1115-1194)  field 0 (psi)
//   NAB2_BSub_TSTEP_V2 (Matrix_Operators.py:1033-1086)  fields 1 (T), 2 (S)
// Two forms, chosen per plan (chain_segment): the chains of sddc_chain.h over
// all rows, for batches whose many chains fill the device, and the theta
// eigenbasis of sddc_theta_solve.hip for smaller ones.
#include <cstdlib>
#include <vector>

#include "sddc_chain.h"

namespace sddc {

// Work items of a k_chain launch, which is one dimensional and holds only live
// items: per (field, chain) type, za (A4) or zn (T and S) instance groups;
// types in order, then groups.  Workgroups go to the eight XCDs round-robin
// (workgroup w to XCD w % 8), so the list is cut into eight runs of consecutive
// items and run c is given to the workgroups of XCD c: each XCD's L2 then
// streams the operator blocks of one or two types.  In (type, group) grid order
// four XCDs fetched every type's blocks (the solve read 1.7x its bytes).
struct ChainItem {
  int field, chain, group;   // field -1: padding past the list
};

__host__ __device__ inline int chain_item_count(int mask, int za, int zn) {
  return 2 * (((mask & 1) ? za : 0) + ((mask & 2) ? zn : 0) + ((mask & 4) ? zn : 0));
}

__host__ __device__ inline int chain_grid(int mask, int za, int zn) {
  return (chain_item_count(mask, za, zn) + 7) / 8 * 8;
}

__device__ __forceinline__ ChainItem chain_item(int w, int mask, int za, int zn) {
  int i = (w % 8) * (chain_grid(mask, za, zn) / 8) + w / 8;
  ChainItem it{-1, 0, 0};
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    if (!((mask >> f) & 1)) continue;
    const int z = f == 0 ? za : zn;
    if (it.field < 0 && i < 2 * z) it = ChainItem{f, i / z, i % z};
    i -= 2 * z;
  }
  return it;
}

template <int NRS, int NG>
__device__ __forceinline__ void zero_chain(const ChainArgs& a, int field, int group, int wave,
                                           int row0, int n) {
  const int lane = threadIdx.x & 63, r = 16 * wave + (lane & 15);
  for (int t = lane >> 4; t < 4 * NG; t += 4) {
    const int b = 4 * NG * group + t;
    if (r >= a.nr || b >= a.B) continue;
    for (int q = 0; q < n; ++q) {
      const size_t o = (size_t)(row0 - 2 * q) * a.nr + r;
      a.X[(size_t)b * a.xstride + a.xoff[field] + o] = 0.0;
      if (field == 0 && a.P) a.P[(size_t)b * a.K * a.nr + o] = 0.0;
    }
  }
}

// NGA and NGN: groups of four instances per A4 and per T/S workgroup.
template <int NRS, int NGA, int NGN, int KD>
__global__ __launch_bounds__(64 * CShape<NRS>::WR + 64) void k_chain(ChainArgs a) {
  constexpr int NGX = NGA > NGN ? NGA : NGN;
  __shared__ __align__(16) double xs[LdsMap<NRS, NGX>::SIZE];
  const ChainItem it = chain_item(blockIdx.x, a.fields_mask, (a.B + 4 * NGA - 1) / (4 * NGA),
                                  (a.B + 4 * NGN - 1) / (4 * NGN));
  const int field = it.field;
  if (field < 0) return;
  const int row0 = a.K - 1 - it.chain, n = row0 / 2 + 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool carrier = wave == CShape<NRS>::WR;
  if (parity_is_zero(a.symmetric, field, row0 & 1)) {
    if (carrier) return;
    if (field == 0)
      zero_chain<NRS, NGA>(a, field, it.group, wave, row0, n);
    else
      zero_chain<NRS, NGN>(a, field, it.group, wave, row0, n);
  } else if (field == 0) {
    if (carrier) {
      carry<NRS, NGA, true>(a, field, it.group, row0, n, xs);
    } else {
      double fe[NGA], bfe[NGA];
#pragma unroll
      for (int g = 0; g < NGA; ++g) fe[g] = bfe[g] = 0.0;
      chain_a4<NRS, NGA, KD>(a, it.group, wave, row0, n, fe, bfe, xs);
    }
  } else {
    if (carrier)
      carry<NRS, NGN, false>(a, field, it.group, row0, n, xs);
    else
      chain_nab2<NRS, NGN, KD>(a, field, it.group, wave, row0, n, xs);
  }
}

// ---------------------------------------------------------------------------
// NAB2 solves in the eigenbasis (Plan::nab2_modal).  The block of row j is
// Linv_j = (P + h j(j+1) I)^-1 with P = V diag(lam) V^-1, so in the variables
// gt = V^-1 g, ft = V^-1 f, bt = V^-1 b the chain of NAB2_BSub_TSTEP_V2
// (Matrix_Operators.py:1061-1083)
//   f_j = Linv_j (g_j - c_j b),  then b += 2 h j f_j for row j - 2
// is nr independent scalar recurrences (c_j = 1/2 at j = 0, else 1):
//   ft_j = (gt_j - c_j bt) q_j,  q_j = 1 / (lam + h j (j+1)),
//   bt  <- bt + 2 h j ft_j = (lam + h j (j-1)) q_j bt + 2 h j q_j gt_j.
// One workgroup per (instance, field, chain) takes the chain in chunks of 64
// consecutive rows from the top.  Per chunk: the rows go to LDS (the next
// chunk's rows are loaded meanwhile); gt = g V^-T as four 16-row tiles times
// the wavefront's 16-column tile of V^-T on f64 MFMA (16x16x4: A = rows from
// LDS, B = V^-1 entries held in registers for the whole chain); the
// recurrences run on wavefront 0, one component per lane, carrying bt from
// chunk to chunk in registers; f = ft V^T the same way; the rows go back to
// memory.
// ---------------------------------------------------------------------------
struct ModalArgs {
  const double* G;
  double* X;
  long long gstride, xstride;
  long long goff[3], xoff[3];
  int K, nr, symmetric, field0;
  double h[3];
};

typedef double v4d_m __attribute__((ext_vector_type(4)));

// out[row][16w + l%16] = sum_e buf[row][e] M[16w + l%16][e] for the 64 rows
// of the chunk (lane l, register v of tile t: row 16t + l/16 + 4v), with
// bm[s] = M[16w + l%16][4s + l/16].  All reads of buf happen here; the
// caller writes the results after a barrier.
template <int NRS, int PITCH>
__device__ __forceinline__ void modal_tiles(const double* buf, const double (&bm)[NRS / 4],
                                            int lane, v4d_m (&acc)[4]) {
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = (v4d_m){0.0, 0.0, 0.0, 0.0};
  const double* arow = buf + (lane & 15) * PITCH + (lane >> 4);
#pragma unroll
  for (int s = 0; s < NRS / 4; ++s)
#pragma unroll
    for (int t = 0; t < 4; ++t)
      acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(arow[16 * t * PITCH + 4 * s], bm[s], acc[t],
                                                    0, 0, 0);
}

template <int NRS, int PITCH>
__device__ __forceinline__ void modal_store(double* buf, const v4d_m (&acc)[4], int col, int lane) {
  if (col >= NRS) return;   // columns past NRS do not exist in buf (and are zero)
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) buf[(16 * t + (lane >> 4) + 4 * v) * PITCH + col] = acc[t][v];
}

template <int NRS, int WR>
__global__ __launch_bounds__(64 * WR) void k_nab2_modal(ModalArgs a, const double* __restrict__ m1,
                                                        const double* __restrict__ m2) {
  constexpr int CH = 64;                  // rows per chunk
  constexpr int PITCH = NRS + 1;          // odd: column accesses spread over the banks
  constexpr int RPW = (CH + WR - 1) / WR; // rows of a chunk each wavefront loads
  __shared__ double buf[CH * PITCH];
  const int field = a.field0 + (int)(blockIdx.x >> 1), chain = blockIdx.x & 1;
  const int K = a.K, nr = a.nr;
  const int start = K - 1 - chain, n = start / 2 + 1;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const double* __restrict__ g = a.G + (size_t)blockIdx.y * a.gstride + a.goff[field];
  double* __restrict__ x = a.X + (size_t)blockIdx.y * a.xstride + a.xoff[field];
  if (a.symmetric && chain == 0) {   // Eq_SYM: odd T/S rows are zero (Matrix_Operators.py:1054)
    for (int i = w; i < n; i += WR)
      if (lane < nr) x[(size_t)(start - 2 * i) * nr + lane] = 0.0;
    return;
  }
  const double* __restrict__ md = field == 1 ? m1 : m2;
  const double h = a.h[field];
  const double lamk = md[lane < NRS ? lane : 0];
  // B operands of this wavefront's column tile: V^-1 [NRS][NRS] and V [nr][NRS]
  const int col = 16 * w + (lane & 15);
  double bvi[NRS / 4], bv[NRS / 4];
#pragma unroll
  for (int s = 0; s < NRS / 4; ++s) {
    const int e = 4 * s + (lane >> 4);
    bvi[s] = col < NRS ? md[NRS + (size_t)nr * NRS + (size_t)col * NRS + e] : 0.0;
    bv[s] = col < nr ? md[NRS + (size_t)col * NRS + e] : 0.0;
  }
  double pre[RPW];
  auto fetch = [&](int c0) {
#pragma unroll
    for (int u = 0; u < RPW; ++u) {
      const int i = w + WR * u;
      const bool ok = i < CH && c0 + i < n && lane < nr;
      pre[u] = ok ? g[(size_t)(start - 2 * (c0 + i)) * nr + lane] : 0.0;
    }
  };
  fetch(0);
  double bt = 0.0;
  v4d_m acc[4];
  for (int c0 = 0; c0 < n; c0 += CH) {
    const int cn = n - c0 < CH ? n - c0 : CH;
#pragma unroll
    for (int u = 0; u < RPW; ++u) {   // padding rows and columns are zero
      const int i = w + WR * u;
      if (i < CH && lane < NRS) buf[i * PITCH + lane] = pre[u];
    }
    __syncthreads();
    if (c0 + CH < n) fetch(c0 + CH);
    modal_tiles<NRS, PITCH>(buf, bvi, lane, acc);
    __syncthreads();
    modal_store<NRS, PITCH>(buf, acc, col, lane);
    __syncthreads();
    if (w == 0 && lane < nr) {
      // eight rows at a time: their inputs and q are ready before the
      // recurrence reaches them (rows past the chunk are zero and skipped)
      for (int i0 = 0; i0 < cn; i0 += 8) {
        double gt[8], q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int j = start - 2 * (c0 + i0 + u);
          gt[u] = buf[(i0 + u) * PITCH + lane];
          q[u] = 1.0 / (lamk + (h * j) * (j + 1));
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (i0 + u < cn) {
            const int j = start - 2 * (c0 + i0 + u);
            const double hj = h * j;
            const double cj = j == 0 ? 0.5 : 1.0;
            buf[(i0 + u) * PITCH + lane] = (gt[u] - cj * bt) * q[u];
            bt = fma((lamk + hj * (j - 1)) * q[u], bt, (2.0 * hj * q[u]) * gt[u]);
          }
        }
      }
    }
    __syncthreads();
    modal_tiles<NRS, PITCH>(buf, bv, lane, acc);
    __syncthreads();
    modal_store<NRS, PITCH>(buf, acc, col, lane);
    __syncthreads();
    for (int i = w; i < cn; i += WR)
      if (lane < nr) x[(size_t)(start - 2 * (c0 + i)) * nr + lane] = buf[i * PITCH + lane];
    __syncthreads();
  }
}

template <int NRS>
static int launch_modal_t(const ModalArgs& a, int nf, int B, const Plan& p, hipStream_t s) {
  using S = CShape<NRS>;
  const dim3 grid(2 * nf, B), block(64 * S::WR);
  hipLaunchKernelGGL((k_nab2_modal<NRS, S::WR>), grid, block, 0, s, a, p.nab2_modes[1],
                     p.nab2_modes[2]);
  return hip_check(hipGetLastError(), "k_nab2_modal");
}

static int dispatch_modal(const ModalArgs& a, int nf, int B, const Plan& p, hipStream_t s) {
  switch (p.NRS) {
    case 8: return launch_modal_t<8>(a, nf, B, p, s);
    case 16: return launch_modal_t<16>(a, nf, B, p, s);
    case 24: return launch_modal_t<24>(a, nf, B, p, s);
    case 32: return launch_modal_t<32>(a, nf, B, p, s);
    case 40: return launch_modal_t<40>(a, nf, B, p, s);
    case 48: return launch_modal_t<48>(a, nf, B, p, s);
    case 56: return launch_modal_t<56>(a, nf, B, p, s);
    case 64: return launch_modal_t<64>(a, nf, B, p, s);
    default: return fail(SDDC_ERR_UNSUPPORTED, "unsupported radial size");
  }
}

template <int NRS, int NGA, int NGN, int KD>
static int launch_chain_t(const ChainArgs& a, hipStream_t s) {
  const dim3 grid(chain_grid(a.fields_mask, (a.B + 4 * NGA - 1) / (4 * NGA),
                             (a.B + 4 * NGN - 1) / (4 * NGN))),
      block(64 * CShape<NRS>::WR + 64);
  hipLaunchKernelGGL((k_chain<NRS, NGA, NGN, KD>), grid, block, 0, s, a);
  return hip_check(hipGetLastError(), "k_chain");
}

template <int NRS>
static int dispatch_width(const ChainArgs& a, int width, hipStream_t s) {
  switch (width) {
    case 1:
    case 2:
    case 4:
    case 5: return launch_chain_t<NRS, 1, 1, 4>(a, s);
    case 6:
    case 10: return launch_chain_t<NRS, 1, 1, 6>(a, s);
    case 3:
    case 7: return launch_chain_t<NRS, 1, 2, 4>(a, s);
    case 9: return launch_chain_t<NRS, 1, 2, 6>(a, s);
    case 8: return launch_chain_t<NRS, 2, 2, 4>(a, s);
    case 16: return launch_chain_t<NRS, 2, 4, 4>(a, s);
    default: return fail(SDDC_ERR_INVALID, "unsupported instances per workgroup");
  }
}

static int dispatch_chain(const ChainArgs& a, int nrs, int width, hipStream_t s) {
  switch (nrs) {
    case 8: return dispatch_width<8>(a, width, s);
    case 16: return dispatch_width<16>(a, width, s);
    case 24: return dispatch_width<24>(a, width, s);
    case 32: return dispatch_width<32>(a, width, s);
    case 40: return dispatch_width<40>(a, width, s);
    case 48: return dispatch_width<48>(a, width, s);
    case 56: return dispatch_width<56>(a, width, s);
    case 64: return dispatch_width<64>(a, width, s);
    default: return fail(SDDC_ERR_UNSUPPORTED, "unsupported radial size");
  }
}

// step: a step's solves, in the plan's form; else (sddc_bsub) the chains, which
// agree with the sequential recurrence to rounding for every right-hand side.
int launch_solve_ex(const Plan& p, int B, const double* G, long long gstride,
                    const long long goff[3], double* X, long long xstride,
                    const long long xoff[3], double* Pout, int fields_mask, bool step, hipStream_t s) {
  if (B <= 0) return SDDC_OK;
  ChainArgs a;
  a.G = G;
  a.X = X;
  a.P = Pout;
  for (int f = 0; f < 3; ++f) {
    a.Lq[f] = p.chain_L[f];
    a.goff[f] = goff[f];
    a.xoff[f] = xoff[f];
  }
  a.D2q = p.chain_D2;
  a.vecs = p.vecs;
  a.gstride = gstride;
  a.xstride = xstride;
  a.K = p.K;
  a.nr = p.nr;
  a.B = B;
  a.symmetric = p.symmetric;
  a.fields_mask = fields_mask;
  a.dtf[0] = p.Pr * p.dt;
  a.dtf[1] = p.dt;
  a.dtf[2] = p.Tau * p.dt;   // NAB2 of S uses Tau*dt (Main.py:281)
  if (p.nab2_modal && (fields_mask & 6)) {
    ModalArgs m;
    m.G = G;
    m.X = X;
    m.gstride = gstride;
    m.xstride = xstride;
    for (int f = 0; f < 3; ++f) {
      m.goff[f] = goff[f];
      m.xoff[f] = xoff[f];
      m.h[f] = a.dtf[f];
    }
    m.K = p.K;
    m.nr = p.nr;
    m.symmetric = p.symmetric;
    m.field0 = (fields_mask & 2) ? 1 : 2;
    const int nf = ((fields_mask >> 1) & 1) + ((fields_mask >> 2) & 1);
    if (int rc = dispatch_modal(m, nf, B, p, s)) return rc;
    a.fields_mask = fields_mask & 1;
    if (!a.fields_mask) return SDDC_OK;
  }
  if (p.theta && step) return launch_theta_solve(p, a, s);
  const int width = p.tune_solve_nbi > 0 ? p.tune_solve_nbi : (B >= 64 ? 3 : 1);
  return dispatch_chain(a, p.NRS, width, s);
}

int launch_solve(const Plan& p, int B, const double* G, double* Xout, double* Pout,
                 int fields_mask, int /*mask_out*/, hipStream_t s) {
  const long long N = (long long)p.K * p.nr;
  const long long off[3] = {0, N, 2 * N};
  return launch_solve_ex(p, B, G, 3 * N, off, Xout, 3 * N, off, Pout, fields_mask, true, s);
}

// ---------------------------------------------------------------------------
// Host side (once per plan).
// ---------------------------------------------------------------------------
void pack_frag(const double* A, int nrows, int ncols, int lda, int NRP, int NC,
                      double* out) {
  const int NQ = NC / 8;
  for (int w = 0; w < NRP / 16; ++w)
    for (int q = 0; q < NQ; ++q)
      for (int l = 0; l < 64; ++l)
        for (int h = 0; h < 2; ++h) {
          const int r = 16 * w + (l & 15), c = 8 * q + 2 * (l >> 4) + h;
          out[((size_t)(w * NQ + q) * 64 + l) * 2 + h] =
              (r < nrows && c < ncols) ? A[(size_t)r * lda + c] : 0.0;
        }
}

// The form of a plan's solves: n, the rows of a chain, or less for the
// eigenbasis of the theta operator (sddc_theta_solve.hip), where the value itself
// stands for nothing else.  Solve of a step on
// MI355X, chains against eigenbasis (timed from the host, where three launches
// cost about 16 us at least and one 8):
//   N_fm/N_r  64/20   B = 1, 16        12.4, 12.7   17.6, 16.9 us
//   90/25     B = 1, 16                16.5, 16.7   17.8, 18.4   (a step 37.7 -> 35.5)
//   128/30    B = 1, 16, 64            23.6, 24, 25        17.7, 18.2, 28.8
//   256/30    B = 1, 16, 64            43.6, 43.9, 45      18.6, 23.6, 44.3
//   512/40    B = 1, 16, 64            112, 113, 115       23, 49, 137
// The chains take as long for 1 instance as for 64, and a plan may be called with
// fewer instances than it has room for, so the line of 96 trades one for the other:
// full batches of 65 to 96 would be faster with the chains (a float64 step, chains
// and eigenbasis, 65 and 96 instances: 128/30 64, 68 and 72, 80 us, 300/48 267, 284
// and 362, 402, 512/40 298, 320 and 386, 459), single instances slower (512/40 solve
// 112 and 23).  Up to 80 modes
// the chains are as fast, and agree with the sequential recurrence to rounding.
// SDDC_CHAIN_SEGMENT overrides.  Fixed per plan, so that the bits of a result do
// not depend on the batch it was computed in.
static int default_segment(int n, int max_batch) {
  if (const char* env = std::getenv("SDDC_CHAIN_SEGMENT")) {
    const int m = std::atoi(env);
    if (m > 0) return m;
  }
  return n <= 40 || max_batch > 96 ? n : 8;
}

template <typename T>
static int upload_vec(T** dst, const std::vector<T>& v) {
  SDDC_HIP(hipMalloc(dst, v.size() * sizeof(T)));
  SDDC_HIP(hipMemcpy(*dst, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return SDDC_OK;
}

int build_chain(Plan& p, const sddc_operators* ops, int max_batch, int segment) {
  const int K = p.K, nr = p.nr, NRS = p.NRS, NRP = p.NRP;
  const size_t BLK = (size_t)NRP * NRS, NN = (size_t)nr * nr;
  const int n = K / 2;   // rows per chain (K is even)
  p.chain_segment = segment > 0 ? segment : default_segment(n, max_batch);
  if (p.chain_segment > n) p.chain_segment = n;
  const double* inv[3] = {ops->Linv_A4, ops->Linv_T, ops->Linv_S};
  const int nfb = p.nab2_modal ? 1 : 3;   // fields solved with per-mode blocks
  std::vector<double> buf((size_t)(K + kFeedPad) * BLK, 0.0);
  for (int f = 0; f < nfb; ++f) {
    for (int jj = 0; jj < K; ++jj)
      pack_frag(inv[f] + jj * NN, nr, nr, nr, NRP, NRS, buf.data() + jj * BLK);
    if (int rc = upload_vec(&p.chain_L[f], buf)) return rc;
  }
  if (p.nab2_modal) {   // lam | V | V^-1, rows padded to NRS
    const double* md[3] = {nullptr, ops->modes_T, ops->modes_S};
    for (int f = 1; f < 3; ++f) {
      std::vector<double> m((size_t)NRS + (size_t)nr * NRS + (size_t)NRS * NRS, 0.0);
      for (int k = 0; k < NRS; ++k) m[k] = k < nr ? md[f][k] : 1.0;
      for (int r = 0; r < nr; ++r)
        for (int k = 0; k < nr; ++k) {
          m[NRS + (size_t)r * NRS + k] = md[f][nr + (size_t)r * nr + k];
          m[NRS + (size_t)nr * NRS + (size_t)r * NRS + k] = md[f][nr + NN + (size_t)r * nr + k];
        }
      if (int rc = upload_vec(&p.nab2_modes[f], m)) return rc;
    }
  }
  {
    std::vector<double> d2b((size_t)BLK);
    pack_frag(ops->D2_A4, nr, nr, nr, NRP, NRS, d2b.data());
    if (int rc = upload_vec(&p.chain_D2, d2b)) return rc;
  }
  return SDDC_OK;
}

void free_chain(Plan& p) {
  if (p.theta) (void)hipFree(p.theta);
  p.theta = nullptr;
  for (int f = 0; f < 3; ++f) {
    if (p.chain_L[f]) (void)hipFree(p.chain_L[f]);
    p.chain_L[f] = nullptr;
  }
  if (p.chain_D2) (void)hipFree(p.chain_D2);
  p.chain_D2 = nullptr;
  for (int f = 0; f < 3; ++f) {
    if (p.nab2_modes[f]) (void)hipFree(p.nab2_modes[f]);
    p.nab2_modes[f] = nullptr;
  }
}

}  // namespace sddc
