// Kernels of the overintegrated Navier-Stokes operator (ns_operator with a
// quadrature tag).
#pragma once
#include <type_traits>

#include "mgdg_kernels.h"

namespace mgdg {

// ns_grad_quad_kernel: grad_cv_operator / grad_t_operator on the points.
// The conserved state and T at the volume points and at both sides' face
// points (T from the EOS there; mixtures: Newton from the interpolated
// nodal T), the central face value (boundaries: the exterior state), then,
// per (field, element) column, the DIM reference-direction volume
// contractions and the NF face contractions on the matrix cores, combined
// per lane with -rx and n into the nodal gradient [NS][DIM][N] (NS = F + 1,
// T last).
//
// ns_div_quad_kernel: F_I - F_V at the volume points (the nodal gradients
// interpolated there) and F_I* - F_V* at the face points: the central viscous
// flux of both sides' states and interpolated gradient traces (boundary
// points: the exterior state with the interior gradients, which for a dummy
// boundary -- exterior state = interior state -- is the one-sided flux), then
// the contraction of euler_quad_kernel.
//
// A workgroup owns epb elements.  LDS: s_n the nodal values, node by node
// [epb][NP + NF NFP][ST] -- the element's nodes, then the neighbours' values at
// its face nodes (interior faces); columns q, T (mixtures), and from column G0
// the gradients (divergence) without the energy's, which no flux takes -- then
// the point values: s_g [cols][gs], s_f [cols][fs], row strides 4 mod 32
// doubles for the matrix cores' operand reads, and the results s_o.
//
// The points are dealt to the waves 64 at a time, volume points first, so that
// the waves' shares differ by at most one such task.  In 3-D the interpolations
// to them are matrix products of the nodal columns with the points' weights.
// Read by every lane instead, a node's columns are 16-byte LDS broadcasts of
// two columns each: at the matrix cores' rate, one wave's keep LDS busy for as
// long as its products take, and the four SIMDs share it.  Ideal gas, p = 3,
// 82,944 elements, 64 volume and 48 face points: divergence 2194 -> 1317 us;
// mixture, p = 2, 24,576 elements: 1057 -> 1000 us.  2-D faces have p + 1
// points, which would leave most of a tile empty, and the ideal gas's gradient
// has 5 columns (p = 1, 6,000 to 384,000 elements: the products take 4 % longer;
// p = 3, 4 alike): there the lanes keep reading the columns, several nodes per
// step, the next step's weights and face nodes already on their way.  ST is 2
// mod 4 doubles, which spreads the node-by-node writes over the LDS banks.
template <int DIM, int P, int NSP, int MIX, bool GRAD>
struct QuadNs {
  using E = Elem<DIM, P>;
  // interpolation on the matrix cores
  static constexpr bool MM = DIM == 3 && (GRAD || NSP > 0);
  static constexpr int NFLD = 2 + DIM + NSP, NS = NFLD + 1, NSD = NS * DIM;
  static constexpr int NQC = NFLD + (MIX != 0 ? 1 : 0);
  static constexpr int NG = NSD - DIM;   // the viscous flux takes no energy gradient
  static constexpr int G0 = MM ? NQC : (NQC + 1) / 2 * 2;
  static constexpr int NCOL = GRAD ? G0 + NG : NQC;
  static constexpr int NC4 = (NCOL + 3) / 4 * 4;
  // columns interpolated together before the point's state is formed
  static constexpr int NC1 = NC4 > 20 ? 16 : NC4;
  static constexpr int ST = (NCOL + 1) / 4 * 4 + 2;
  // columns past NCOL up to NC4 (never used) are the next row's, or, behind the
  // last row, these
  static constexpr int PAD = MM ? 4 : 0;
  static constexpr int ROWS = E::NP + E::NFN;
  static_assert(ST >= NCOL && ST % 4 == 2 && (!MM || NC4 - ST <= PAD), "LDS row stride");
  static_assert(NQC <= NC1 || !MM, "the state's columns");
};

// The contraction's K range is cut over ks waves per tile while that keeps
// more of the workgroup's four waves busy.
__host__ __device__ constexpr int quad_ksplit(int ntile) {
  return ntile >= 3 ? 1 : (ntile == 2 ? 2 : 4);
}
__host__ __device__ constexpr int quad_tiles(int np, int ncol) {
  return ((np + 15) / 16) * ((ncol + 15) / 16);
}

// LDS doubles of a workgroup of epb elements.
template <int DIM, int P, int NSP, int MIX>
constexpr size_t quad_div_lds(int gs, int fs, int epb) {
  using C = QuadNs<DIM, P, NSP, MIX, true>;
  using E = Elem<DIM, P>;
  const size_t nodes = size_t(epb) * C::ROWS * C::ST + C::PAD;
  const size_t parts = size_t(quad_ksplit(quad_tiles(E::NP, C::NFLD * epb))) * C::NFLD * epb *
                       E::NP;
  // (the results go over the nodal values)
  return (nodes > parts ? nodes : parts) + size_t(C::NFLD) * epb * (gs + fs);
}
template <int DIM, int P, int NSP, int MIX>
constexpr size_t quad_grad_lds(int gs, int fs, int epb) {
  using C = QuadNs<DIM, P, NSP, MIX, false>;
  using E = Elem<DIM, P>;
  const size_t nodes = size_t(epb) * C::ROWS * C::ST + C::PAD;
  const size_t out = size_t(C::NSD) * epb * E::NP;
  return (nodes > out ? nodes : out) + size_t(C::NS) * epb * (gs + fs);
}

// Nodal values of the workgroup's elements and their neighbours' at the face
// nodes; a thread per node, its loads in flight together.
template <int DIM, int P, int NSP, int MIX, bool GRAD>
__device__ __forceinline__ void quad_load_nodes(const KArgs& a, const QuadArgs& qa,
                                                int64_t e0, int ne, double* s_n) {
  using C = QuadNs<DIM, P, NSP, MIX, GRAD>;
  using E = Elem<DIM, P>;
  constexpr int NP = E::NP, NFN = E::NFN;
  const int64_t N = a.nnodes;
  for (int t = threadIdx.x; t < ne * C::ROWS; t += kBlock) {
    const bool own = t < ne * NP;
    const int u = own ? t : t - ne * NP;
    const int le = u / (own ? NP : NFN);
    const int r = u - le * (own ? NP : NFN);
    int64_t g = e0 * NP + u;
    if (!own) g = a.vmap_p[e0 * NFN + u];
    if (g < 0) continue;   // boundary face node: not read
    double* row = s_n + (le * C::ROWS + (own ? r : NP + r)) * C::ST;
    double v[C::NCOL];
#pragma unroll
    for (int f = 0; f < C::NFLD; ++f) v[f] = a.q[f * N + g];
    if constexpr (MIX != 0) v[C::NFLD] = qa.temp[g];
    if constexpr (GRAD) {
#pragma unroll
      for (int k = 0; k < C::NG; ++k) v[C::G0 + k] = a.grad[(k < DIM ? k : k + DIM) * N + g];
    }
#pragma unroll
    for (int f = 0; f < C::NQC; ++f) row[f] = v[f];
    if constexpr (GRAD) {
#pragma unroll
      for (int k = 0; k < C::NG; ++k) row[C::G0 + k] = v[C::G0 + k];
    }
  }
}

// out[c] = sum_j w[j ws] rows[off(j) + c] (c < NC, j < N), a few nodes per
// step: the next step's weights are on their way while this one's columns are
// read from LDS.  The loop stays rolled: unrolled, the compiler starts the
// LDS reads of all nodes at once and spills up to 5 KB per lane.
template <int NC, int N, typename Off>
__device__ __forceinline__ void quad_interp(const double* w, int ws, const double* rows,
                                            Off off, double* out) {
  // nodes per step: at least two steps, and for many columns few nodes
  constexpr int CH = NC > 24 ? (N % 2 == 0 && N > 2 ? 2 : 1)
                             : (N % 5 == 0 && N > 5 ? 5
                                : N % 3 == 0 && N > 3 ? 3
                                : N % 2 == 0 && N > 2 ? 2 : 1);
  static_assert(N % CH == 0 && CH < N, "nodes per step");
#pragma unroll
  for (int c = 0; c < NC; ++c) out[c] = 0.0;
  double wn[CH];
  int on[CH];
#pragma unroll
  for (int u = 0; u < CH; ++u) {
    wn[u] = w[u * ws];
    on[u] = off(u);
  }
#pragma unroll 1
  for (int j = 0; j < N; j += CH) {
    double wv[CH];
    int ov[CH];
    const int jn = j + CH < N ? j + CH : 0;
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      wv[u] = wn[u];
      ov[u] = on[u];
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      wn[u] = w[(jn + u) * ws];
      on[u] = off(jn + u);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u)
#pragma unroll
      for (int c = 0; c < NC; ++c) out[c] += wv[u] * rows[ov[u] + c];
  }
}

// {{{ interpolation on the matrix cores
//
// A wave interpolates 4 tiles of 16 points: D[column][point] +=
// A[column][node] B[node][point], 16 columns to a v_mfma_f64_16x16x4 and 4 to
// each v_mfma_f64_4x4x4 (four blocks: 4 columns x 16 points), which have the
// same operand and result lanes: lane (kk, li) = (lane / 16, lane % 16) holds
// B of node kk and point li, A of node kk and column li (li % 4), and gets
// columns 4 g + kk of point li.  Transposing the 4 x 4 (tile, kk) squares over
// registers and rows of 16 lanes then gives every lane all columns of the one
// point (lane / 16, li).

// r[t] in lane row k -> r[k] in lane row t
__device__ __forceinline__ void quad_transpose(double* r) {
  unsigned v[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t) __builtin_memcpy(v[t], &r[t], 8);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const auto x = __builtin_amdgcn_permlane32_swap(v[t][h], v[t + 2][h], false, false);
      v[t][h] = x[0];
      v[t + 2][h] = x[1];
    }
#pragma unroll
    for (int t = 0; t < 4; t += 2) {
      const auto x = __builtin_amdgcn_permlane16_swap(v[t][h], v[t + 1][h], false, false);
      v[t][h] = x[0];
      v[t + 1][h] = x[1];
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) __builtin_memcpy(&r[t], v[t], 8);
}

// A wave's accumulators: NC columns (a multiple of 4) of 4 tiles.
template <int NC>
struct QuadAcc {
  static constexpr int NB = NC / 16, NQ = NC % 16 / 4;
  doublex4 b[4][NB > 0 ? NB : 1];
  double q[4][NQ > 0 ? NQ : 1];

  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int i = 0; i < NB; ++i) b[t][i] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int i = 0; i < NQ; ++i) q[t][i] = 0.0;
    }
  }
  // one step of 4 nodes of tile t: this lane's node row and its weight
  __device__ __forceinline__ void step(int t, const double* row, double w) {
    const int li = threadIdx.x & 15;
#pragma unroll
    for (int i = 0; i < NB; ++i)
      b[t][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(row[16 * i + li], w, b[t][i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < NQ; ++i)
      q[t][i] = __builtin_amdgcn_mfma_f64_4x4x4f64(row[16 * NB + 4 * i + (li & 3)], w,
                                                   q[t][i], 0, 0, 0);
  }
  __device__ __forceinline__ void points(double* out) {
#pragma unroll
    for (int i = 0; i < NC / 4; ++i) {
#pragma unroll
      for (int t = 0; t < 4; ++t) out[4 * i + t] = i < 4 * NB ? b[t][i / 4][i % 4] : q[t][i - 4 * NB];
      quad_transpose(out + 4 * i);
    }
  }
};

// The 4 tiles of a wave, and this lane's point among them.  Tiles beyond the
// last and points beyond a tile's n repeat the last one (valid = false).
template <int DIM, int P>
struct QuadTiles {
  using E = Elem<DIM, P>;
  bool valid;
  int le, fc, m;   // this lane's point
  int m0;          // its tile's first point

  QuadTiles() = default;
  __device__ __forceinline__ QuadTiles(bool face, int task, int ne, int n) {
    const int lane = threadIdx.x & 63;
    const int per = (n + 15) / 16, nt = ne * per * (face ? E::NF : 1);
    const int u = task * 4 + (lane >> 4), t = u < nt ? u : nt - 1;
    const int r = t / per;
    m0 = (t - r * per) * 16;
    le = face ? r / E::NF : r;
    fc = face ? r - le * E::NF : 0;
    const int k = m0 + (lane & 15);
    valid = u < nt && k < n;
    m = k < n ? k : n - 1;
  }
  // this lane's point column of tile t's weights (n points to a node)
  __device__ __forceinline__ int column(int t, int n) const {
    const int k = __builtin_amdgcn_readlane(m0, 16 * t) + int(threadIdx.x & 15);
    return k < n ? k : n - 1;
  }
};

// Columns [C0, C0 + NC) at volume points; s_n: node rows of stride ST,
// rows node rows to an element.
template <int DIM, int P, int C0, int NC, int ST, int ROWS>
__device__ __forceinline__ void quad_mm_volume(const double* interp, int nq,
                                               const QuadTiles<DIM, P>& tl, const double* s_n,
                                               double* out) {
  constexpr int NP = Elem<DIM, P>::NP, NK = (NP + 3) / 4;
  const int kk = (threadIdx.x >> 4) & 3;
  int col[4], row[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    col[t] = tl.column(t, nq);
    row[t] = __builtin_amdgcn_readlane(tl.le, 16 * t) * ROWS * ST + C0;
  }
  QuadAcc<NC> acc;
  acc.zero();
  double wn[4];
  auto weights = [&](int s) {
    const int k = 4 * s + kk;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const double w = interp[(k < NP ? k : NP - 1) * nq + col[t]];
      wn[t] = k < NP ? w : 0.0;
    }
  };
  weights(0);
#pragma unroll 1
  for (int s = 0; s < NK; ++s) {
    double w[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) w[t] = wn[t];
    weights(s + 1 < NK ? s + 1 : 0);
    const int k = 4 * s + kk < NP ? 4 * s + kk : NP - 1;
#pragma unroll
    for (int t = 0; t < 4; ++t) acc.step(t, s_n + row[t] + k * ST, w[t]);
  }
  acc.points(out);
}

// Face points: the weights and both sides' node rows, shared by the two sides'
// (and all columns') interpolations.
template <int DIM, int P, int ST, int ROWS>
struct QuadFaceTiles {
  using E = Elem<DIM, P>;
  static constexpr int NFP = E::NFP, NK = (NFP + 3) / 4;
  double w[NK][4];
  int own[NK][4], ext[4];

  QuadFaceTiles() = default;
  // v0: the face's first exterior map entry of this lane's point (boundary
  // faces, v0 < 0: the exterior rows are the own ones)
  __device__ __forceinline__ QuadFaceTiles(const double* finterp, int nfq,
                                           const QuadTiles<DIM, P>& tl, const int* s_fm,
                                           int32_t v0) {
    const int kk = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int fc = __builtin_amdgcn_readlane(tl.fc, 16 * t);
      const int base = __builtin_amdgcn_readlane(tl.le, 16 * t) * ROWS * ST;
      const int col = tl.column(t, nfq);
      const bool in = int(__builtin_amdgcn_readlane(v0, 16 * t)) >= 0;
      ext[t] = in ? base + (E::NP + fc * NFP) * ST : -1;
#pragma unroll
      for (int s = 0; s < NK; ++s) {
        const int k = 4 * s + kk, kc = fc * NFP + (k < NFP ? k : NFP - 1);
        const double x = finterp[kc * nfq + col];
        w[s][t] = k < NFP ? x : 0.0;
        own[s][t] = base + s_fm[kc];
      }
    }
  }
  template <int C0, int NC, bool EXT>
  __device__ __forceinline__ void interp(const double* s_n, double* out) const {
    const int kk = (threadIdx.x >> 4) & 3;
    QuadAcc<NC> acc;
    acc.zero();
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const int k = 4 * s + kk < NFP ? 4 * s + kk : NFP - 1;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int row = EXT && ext[t] >= 0 ? ext[t] + k * ST : own[s][t];
        acc.step(t, s_n + C0 + row, w[s][t]);
      }
    }
    acc.points(out);
  }
};

// }}}

// The gradients [NS][DIM] from the columns, which hold all but the energy's.
template <int DIM, int NG>
__device__ __forceinline__ void quad_gradients(const double* g, double* out) {
#pragma unroll
  for (int k = 0; k < DIM; ++k) out[DIM + k] = 0.0;   // not read
#pragma unroll
  for (int k = 0; k < NG; ++k) out[k < DIM ? k : k + DIM] = g[k];
}

// Temperature at a point with interpolated state q and seed.
template <int DIM>
__device__ __forceinline__ double ideal_temperature(const double* q, const GasDev& g) {
  const double irho = 1.0 / q[0];
  double mm = 0.0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) mm += q[2 + d] * q[2 + d];
  return ((g.gamma - 1.0) / g.gas_const) * (q[1] - 0.5 * mm * irho) * irho;
}

template <int DIM, int NSP, int MIX>
__device__ __forceinline__ double quad_point_temperature(const double* q, double seed,
                                                         const GasDev& g, int niter) {
  if constexpr (MIX != 0)
    return point_temperature<DIM, NSP>(q, seed, niter);
  else
    return ideal_temperature<DIM>(q, g);
}

// The waves' tasks: volume points 64 at a time (3-D: four tiles of 16 points
// of one element each), then face points; the first wave rotates with the
// block, so that two workgroups on a CU do not both give their surplus task to
// the same SIMD.
template <bool MM>
__host__ __device__ __forceinline__ int quad_task_count(int groups, int n) {
  return MM ? (groups * ((n + 15) / 16) + 3) / 4 : (groups * n + 63) / 64;
}
__device__ __forceinline__ int quad_first_task() {
  return (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + (blockIdx.x >> 3)) & (kWaves - 1);
}
// The lane's point of a task; without tiles 64 consecutive points, at most one
// past the last.
template <int DIM, int P, bool MM>
__device__ __forceinline__ QuadTiles<DIM, P> quad_point(bool face, int task, int ne, int n) {
  if constexpr (MM) {
    return QuadTiles<DIM, P>(face, task, ne, n);
  } else {
    QuadTiles<DIM, P> tl;
    const int nf = face ? Elem<DIM, P>::NF : 1;
    const int t = task * 64 + int(threadIdx.x & 63);
    const int r = t / n;
    tl.valid = t < ne * nf * n;
    tl.m = t - r * n;
    tl.le = r / nf;
    tl.fc = r - tl.le * nf;
    tl.m0 = 0;
    return tl;
  }
}

template <int DIM, int P, int NSP, int MIX>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(2))) void ns_grad_quad_kernel(KArgs a, QuadArgs qa) {
  using E = Elem<DIM, P>;
  using C = QuadNs<DIM, P, NSP, MIX, false>;
  constexpr int NP = E::NP, NFP = E::NFP, NF = E::NF, ST = C::ST;
  constexpr int NFLD = C::NFLD, NS = C::NS, NQC = C::NQC;
  extern __shared__ __align__(16) double lds16[];
  const int nq = qa.nq, nfq = qa.nfq, epb = qa.epb, nfq_all = NF * qa.nfq;
  const int gs = qa.gs, fs = qa.fs;
  double* s_u = lds16;                    // [NS*epb][gs]
  double* s_s = s_u + NS * epb * gs;      // [NS*epb][fs]
  double* s_n = s_s + NS * epb * fs;
  double* s_o = s_n;                      // [NS*DIM][epb][NP]
  __shared__ int s_fm[E::NFN];            // LDS row offsets of the face nodes
  auto node = [](int j) { return j * ST; };
  const int64_t e0 = int64_t(blockIdx.x) * epb;
  const int ne = a.K - e0 < epb ? int(a.K - e0) : epb;
  const int64_t N = a.nnodes;
  // 1: nodal values
  for (int t = threadIdx.x; t < E::NFN; t += kBlock) s_fm[t] = a.fmask[t] * ST;
  quad_load_nodes<DIM, P, NSP, MIX, false>(a, qa, e0, ne, s_n);
  __syncthreads();
  // 2: state and temperature at the volume points; at the face points the
  // gradient flux value (central inside, the exterior value on boundaries)
  // times the face Jacobian ratio
  const int nvt = quad_task_count<C::MM>(ne, nq);
  const int ntask = nvt + quad_task_count<C::MM>(ne * NF, nfq);
  for (int task = quad_first_task(); task < ntask; task += kWaves) {
    const bool face = task >= nvt;
    const auto tl = quad_point<DIM, P, C::MM>(face, face ? task - nvt : task, ne, face ? nfq : nq);
    if (!C::MM && !tl.valid) continue;
    const int le = tl.le, m = tl.m;
    const double* rows = s_n + le * C::ROWS * ST;
    if (!face) {
      double u[C::NC4];
      if constexpr (C::MM)
        quad_mm_volume<DIM, P, 0, C::NC4, ST, C::ROWS>(qa.interp, nq, tl, s_n, u);
      else
        quad_interp<NQC, NP>(qa.interp + m, nq, rows, node, u);
      const double tq = quad_point_temperature<DIM, NSP, MIX>(u, MIX ? u[NQC - 1] : 0.0,
                                                              a.gas, qa.niter);
      if (!tl.valid) continue;
#pragma unroll
      for (int f = 0; f < NFLD; ++f) s_u[(f * epb + le) * gs + m] = u[f];
      s_u[(NFLD * epb + le) * gs + m] = tq;
    } else {
      const int fc = tl.fc, rem = fc * nfq + m;
      const int64_t e = e0 + le;
      const int32_t v0 = a.vmap_p[(e * NF + fc) * NFP];
      const double sc = a.fscale[e * NF + fc];
      double um[C::NC4], up[C::NC4];
      if constexpr (C::MM) {
        const QuadFaceTiles<DIM, P, ST, C::ROWS> ft(qa.finterp, nfq, tl, s_fm, v0);
        ft.template interp<0, C::NC4, false>(s_n, um);
        ft.template interp<0, C::NC4, true>(s_n, up);
      } else {
        const double* w = qa.finterp + fc * NFP * nfq + m;
        if (v0 >= 0) {
          quad_interp<NQC, NFP>(w, nfq, rows, [&](int j) { return s_fm[fc * NFP + j]; }, um);
          quad_interp<NQC, NFP>(w, nfq, rows + (NP + fc * NFP) * ST, node, up);
        }
      }
      if (!tl.valid) continue;
      double tp;
      if (v0 >= 0) {
        const double tm = quad_point_temperature<DIM, NSP, MIX>(
            um, MIX ? um[NQC - 1] : 0.0, a.gas, qa.niter);
        tp = quad_point_temperature<DIM, NSP, MIX>(up, MIX ? up[NQC - 1] : 0.0, a.gas,
                                                   qa.niter);
#pragma unroll
        for (int f = 0; f < NFLD; ++f)
          s_s[(f * epb + le) * fs + rem] = sc * ((um[f] + up[f]) / 2);
        s_s[(NFLD * epb + le) * fs + rem] = sc * ((tm + tp) / 2);
      } else {
        const int64_t bq = (-int64_t(v0) - 1) / NFP * nfq + m;
#pragma unroll
        for (int f = 0; f < NFLD; ++f) up[f] = qa.qbq[f * qa.nbq + bq];
        if constexpr (MIX != 0)
          tp = qa.tbq[bq];
        else
          tp = ideal_temperature<DIM>(up, a.gas);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) s_s[(f * epb + le) * fs + rem] = sc * up[f];
        s_s[(NFLD * epb + le) * fs + rem] = sc * tp;
      }
    }
  }
  __syncthreads();
  // 3: per column j = f * epb + le: D_r = Wq_r u (r < DIM) and L_c = Lq_c
  // (fscale u*) (c < NF) on the matrix cores (operand layout as in
  // euler_quad_kernel: each lane's accumulators hold its own column j), then
  // grad_d = sum_r -rx[r][d] D_r + sum_c n_c[d] L_c with the element's
  // factors read per lane.
  {
    constexpr int RT = (NP + 15) / 16;
    const int ncol = NS * epb;
    const int ntile = RT * ((ncol + 15) / 16);
    const int li = threadIdx.x & 15, kk = (threadIdx.x >> 4) & 3;
    for (int tile = threadIdx.x >> 6; tile < ntile; tile += blockDim.x >> 6) {
      const int rt = tile % RT, ct = tile / RT;
      const int row = rt * 16 + li;
      const int j = ct * 16 + li;
      const int lej = j % epb;
      const bool cok = j < ncol && lej < ne;
      const int jc = j < ncol ? j : 0;
      const int r0 = row < NP ? row : 0;
      const int64_t ej = e0 + (cok ? lej : 0);
      doublex4 g[DIM];
#pragma unroll
      for (int d = 0; d < DIM; ++d) g[d] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int r = 0; r < DIM; ++r) {
        doublex4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = acc0;
        quad_mfma_panel<NP>(qa.wdiff + r * nq * NP + r0, s_u + jc * gs, nq, kk, acc0, acc1);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
          const double c = -a.rx[ej * DIM * DIM + r * DIM + d];
          g[d] += c * (acc0 + acc1);
        }
      }
#pragma unroll
      for (int fc = 0; fc < NF; ++fc) {
        doublex4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = acc0;
        quad_mfma_panel<NP>(qa.lift + fc * nfq * NP + r0, s_s + jc * fs + fc * nfq, nfq, kk,
                            acc0, acc1);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
          const double c = a.normals[(ej * NF + fc) * DIM + d];
          g[d] += c * (acc0 + acc1);
        }
      }
      if (cok) {
        const int f = j / epb;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int i = rt * 16 + 4 * q4 + kk;
          if (i < NP) {
#pragma unroll
            for (int d = 0; d < DIM; ++d)
              s_o[((f * DIM + d) * epb + lej) * NP + i] = g[d][q4];
          }
        }
      }
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < C::NSD * ne * NP; t += blockDim.x) {
    const int k = t / (ne * NP);
    const int r = t - k * ne * NP;
    a.out[k * N + e0 * NP + r] = s_o[k * epb * NP + r];
  }
}

// Waves per SIMD that the divergence's registers are planned for.  Two spill 100
// to 280 VGPRs with species, one none; which is faster as measured, MI355X,
// mixture, two -> one: 2-D p = 1..4, 4,608 triangles 28, 48, 53, 77 -> 33, 53,
// 58, 96 us; 3-D p = 1, 131,712 tets 2.71 -> 2.35 ms, p = 2 5.54 -> 5.74 ms,
// p = 3, 10,368 0.79 -> 0.73 ms, p = 4 (one workgroup fills a CU's LDS) 2.56 ->
// 1.62 ms.
constexpr int quad_div_waves(int dim, int p, int nsp) {
  return dim == 3 && p != 2 && nsp > 0 ? 1 : 2;
}

template <int DIM, int P, int NSP, int MIX>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(quad_div_waves(DIM, P, NSP)))) void ns_div_quad_kernel(KArgs a, QuadArgs qa) {
  using E = Elem<DIM, P>;
  using C = QuadNs<DIM, P, NSP, MIX, true>;
  constexpr int NP = E::NP, NFP = E::NFP, NF = E::NF, ST = C::ST;
  constexpr int NFLD = C::NFLD, NSD = C::NSD, NQC = C::NQC, G0 = C::G0;
  constexpr int NC4 = C::NC4, NC1 = C::NC1;
  extern __shared__ __align__(16) double lds16[];
  const int nq = qa.nq, nfq = qa.nfq, epb = qa.epb, nfq_all = NF * qa.nfq;
  const int gs = qa.gs, fs = qa.fs;
  double* s_g = lds16;                      // [F*epb][gs]
  double* s_f = s_g + NFLD * epb * gs;      // [F*epb][fs]
  double* s_n = s_f + NFLD * epb * fs;
  double* s_o = s_n;                        // [ks][F*epb][NP]
  __shared__ int s_fm[E::NFN];              // LDS row offsets of the face nodes
  auto node = [](int j) { return j * ST; };
  const int64_t e0 = int64_t(blockIdx.x) * epb;
  const int ne = a.K - e0 < epb ? int(a.K - e0) : epb;
  const int64_t N = a.nnodes;
  // 1: nodal values
  for (int t = threadIdx.x; t < E::NFN; t += kBlock) s_fm[t] = a.fmask[t] * ST;
  quad_load_nodes<DIM, P, NSP, MIX, true>(a, qa, e0, ne, s_n);
  __syncthreads();
  // 2: F_I - F_V at the volume points, in reference directions, and
  // F_I* - F_V* at the face points
  const int nvt = quad_task_count<C::MM>(ne, nq);
  const int ntask = nvt + quad_task_count<C::MM>(ne * NF, nfq);
  for (int task = quad_first_task(); task < ntask; task += kWaves) {
    const bool face = task >= nvt;
    const auto tl = quad_point<DIM, P, C::MM>(face, face ? task - nvt : task, ne, face ? nfq : nq);
    if (!C::MM && !tl.valid) continue;
    const int le = tl.le, m = tl.m;
    const double* rows = s_n + le * C::ROWS * ST;
    // a point's columns: state, Newton seed, gradients
    double col[C::NC4];
    if (!face) {
      const double* w = qa.interp + m;
      Node<DIM, NSP> s;
      if constexpr (C::MM)
        quad_mm_volume<DIM, P, 0, NC1, ST, C::ROWS>(qa.interp, nq, tl, s_n, col);
      else
        quad_interp<NQC, NP>(w, nq, rows, node, col);
      double tq = 0.0;
      if constexpr (MIX != 0) tq = point_temperature<DIM, NSP>(col, col[NQC - 1], qa.niter);
#pragma unroll
      for (int f = 0; f < NFLD; ++f) s.q[f] = col[f];
      node_state<DIM, NSP, MIX>(s, a.gas, tq);
      if constexpr (!C::MM)
        quad_interp<C::NG, NP>(w, nq, rows + G0, node, col + G0);
      else if constexpr (NC4 > NC1)
        quad_mm_volume<DIM, P, NC1, NC4 - NC1, ST, C::ROWS>(qa.interp, nq, tl, s_n, col + NC1);
      double gacc[NSD], F[NFLD][DIM];
      quad_gradients<DIM, C::NG>(col + G0, gacc);
      viscous_flux<DIM, NSP, MIX>(s, reinterpret_cast<const double(*)[DIM]>(gacc),
                                  gacc + NFLD * DIM, F);
      if (a.inviscid_on) {
        double FI[NFLD][DIM];
        inviscid_flux<DIM, NSP>(s, FI);
#pragma unroll
        for (int f = 0; f < NFLD; ++f)
#pragma unroll
          for (int d = 0; d < DIM; ++d) F[f][d] = FI[f][d] - F[f][d];
      } else {
#pragma unroll
        for (int f = 0; f < NFLD; ++f)
#pragma unroll
          for (int d = 0; d < DIM; ++d) F[f][d] = -F[f][d];
      }
      if (!tl.valid) continue;
      const double* rx = a.rx + (e0 + le) * DIM * DIM;
#pragma unroll
      for (int f = 0; f < NFLD; ++f)
#pragma unroll
        for (int r = 0; r < DIM; ++r) {
          double g = 0.0;
#pragma unroll
          for (int d = 0; d < DIM; ++d) g += rx[r * DIM + d] * F[f][d];
          s_g[(f * epb + le) * gs + r * nq + m] = g;
        }
    } else {
      const int fc = tl.fc, rem = fc * nfq + m;
      const int64_t e = e0 + le;
      const int32_t v0 = a.vmap_p[(e * NF + fc) * NFP];
      double n[DIM];
#pragma unroll
      for (int d = 0; d < DIM; ++d) n[d] = a.normals[(e * NF + fc) * DIM + d];
      const double* w = qa.finterp + fc * NFP * nfq + m;
      const int ext0 = (NP + fc * NFP) * ST;
      auto own = [&](int j) { return s_fm[fc * NFP + j]; };
      using Tiles = QuadFaceTiles<DIM, P, ST, C::ROWS>;
      std::conditional_t<C::MM, Tiles, int> ft;
      if constexpr (C::MM) ft = Tiles(qa.finterp, nfq, tl, s_fm, v0);
      Node<DIM, NSP> sm, sp;
      double fstar[NFLD], fv[NFLD], gacc[NSD];
      // the own side's state and viscous flux first, then the other side's, so
      // that one gradient set is live
      {
        double tm = 0.0;
        if constexpr (C::MM)
          ft.template interp<0, NC1, false>(s_n, col);
        else
          quad_interp<NQC, NFP>(w, nfq, rows, own, col);
        if constexpr (MIX != 0) tm = point_temperature<DIM, NSP>(col, col[NQC - 1], qa.niter);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) sm.q[f] = col[f];
        node_state<DIM, NSP, MIX>(sm, a.gas, tm);
        if constexpr (!C::MM)
          quad_interp<C::NG, NFP>(w, nfq, rows + G0, own, col + G0);
        else if constexpr (NC4 > NC1)
          ft.template interp<NC1, NC4 - NC1, false>(s_n, col + NC1);
        quad_gradients<DIM, C::NG>(col + G0, gacc);
        viscous_flux_n<DIM, NSP, MIX>(sm, reinterpret_cast<const double(*)[DIM]>(gacc),
                                      gacc + NFLD * DIM, n, fv);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) fstar[f] = -0.5 * fv[f];
      }
      // (boundary faces: the other side's gradient trace is the own one)
      double tp = 0.0;
      if constexpr (C::MM)
        ft.template interp<0, NC1, true>(s_n, col);
      if (v0 >= 0) {
        if constexpr (!C::MM) quad_interp<NQC, NFP>(w, nfq, rows + ext0, node, col);
        if constexpr (MIX != 0) tp = point_temperature<DIM, NSP>(col, col[NQC - 1], qa.niter);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) sp.q[f] = col[f];
      } else {
        const int64_t bq = (-int64_t(v0) - 1) / NFP * nfq + m;
#pragma unroll
        for (int f = 0; f < NFLD; ++f) sp.q[f] = qa.qbq[f * qa.nbq + bq];
        if constexpr (MIX != 0) tp = qa.tbq[bq];
      }
      node_state<DIM, NSP, MIX>(sp, a.gas, tp);
      if (a.inviscid_on) {
        inviscid_numflux<DIM, NSP>(sm, sp, n, a.flux_kind, fv);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) fstar[f] += fv[f];
      }
      if constexpr (!C::MM)
        quad_interp<C::NG, NFP>(
            w, nfq, rows + G0, [&](int j) { return v0 >= 0 ? ext0 + j * ST : own(j); },
            col + G0);
      else if constexpr (NC4 > NC1)
        ft.template interp<NC1, NC4 - NC1, true>(s_n, col + NC1);
      quad_gradients<DIM, C::NG>(col + G0, gacc);
      viscous_flux_n<DIM, NSP, MIX>(sp, reinterpret_cast<const double(*)[DIM]>(gacc),
                                    gacc + NFLD * DIM, n, fv);
#pragma unroll
      for (int f = 0; f < NFLD; ++f) fstar[f] -= 0.5 * fv[f];
      if (!tl.valid) continue;
      const double sc = a.fscale[e * NF + fc];
#pragma unroll
      for (int f = 0; f < NFLD; ++f) s_f[(f * epb + le) * fs + rem] = -sc * fstar[f];
    }
  }
  __syncthreads();
  // 3: the contraction of euler_quad_kernel, its K range cut into ks pieces:
  // the volume points' and the face points' 16-point steps dealt in turn
  constexpr int RT = (NP + 15) / 16;
  const int ncol = NFLD * epb;
  const int ntile = RT * ((ncol + 15) / 16);
  const int ks = quad_ksplit(ntile);
  {
    const int li = threadIdx.x & 15, kk = (threadIdx.x >> 4) & 3;
    for (int job = threadIdx.x >> 6; job < ntile * ks; job += blockDim.x >> 6) {
      const int tile = job / ks, piece = job - tile * ks;
      const int rt = tile % RT, ct = tile / RT;
      const int row = rt * 16 + li;
      const int j = ct * 16 + li;
      const int lej = j % epb;
      const bool rok = row < NP, cok = j < ncol && lej < ne;
      doublex4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = acc0;
      const int jc = j < ncol ? j : 0;
      const int r0 = rok ? row : 0;
      const int v0 = DIM * nq * piece / ks, v1 = DIM * nq * (piece + 1) / ks;
      const int f0 = nfq_all * piece / ks, f1 = nfq_all * (piece + 1) / ks;
      quad_mfma_panel<NP>(qa.wdiff + v0 * NP + r0, s_g + jc * gs + v0, v1 - v0, kk, acc0, acc1);
      quad_mfma_panel<NP>(qa.lift + f0 * NP + r0, s_f + jc * fs + f0, f1 - f0, kk, acc0, acc1);
      if (cok) {
        double* o = s_o + piece * ncol * NP;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int i = rt * 16 + 4 * q4 + kk;
          if (i < NP) o[j * NP + i] = acc0[q4] + acc1[q4];
        }
      }
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < NFLD * ne * NP; t += blockDim.x) {
    const int f = t / (ne * NP);
    const int r = t - f * ne * NP;
    double v = s_o[f * epb * NP + r];
    for (int p = 1; p < ks; ++p) v += s_o[(p * ncol + f * epb) * NP + r];
    a.out[f * N + e0 * NP + r] = v;
  }
}

}  // namespace mgdg
