// Kernels of the overintegrated Navier-Stokes operator (ns_operator with a
// quadrature tag).
#pragma once
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
// its face nodes (interior faces); columns q, T (mixtures), and from the even
// column G0 the gradients (divergence) -- then the point values: s_g
// [cols][gs], s_f [cols][fs], row strides 4 mod 32 doubles for the matrix
// cores' operand reads, and the results s_o.
//
// The points are dealt to the waves 64 at a time, volume points first, so that
// the waves' shares differ by at most one such task.  Interpolations read a
// node's columns with 16-byte LDS broadcasts, several nodes per step, the
// next step's weights and face nodes already on their way.  (Node by node
// each waited for its weight, then for the face node's index, then for LDS,
// and one wave could hold three tasks while another held one: 73,000 of a
// workgroup's 102,000 cycles at p = 3, ideal gas.)  ST is
// 2 mod 4 doubles, which spreads the node-by-node writes over the LDS banks.
template <int DIM, int P, int NSP, int MIX, bool GRAD>
struct QuadNs {
  using E = Elem<DIM, P>;
  static constexpr int NFLD = 2 + DIM + NSP, NS = NFLD + 1, NSD = NS * DIM;
  static constexpr int NQC = NFLD + (MIX != 0 ? 1 : 0);
  static constexpr int G0 = (NQC + 1) / 2 * 2;
  static constexpr int NCOL = GRAD ? G0 + NSD : NQC;
  static constexpr int ST = (NCOL + 1) / 4 * 4 + 2;
  static constexpr int ROWS = E::NP + E::NFN;
  static_assert(ST >= NCOL && ST % 4 == 2, "LDS row stride");
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
  const size_t nodes = size_t(epb) * C::ROWS * C::ST;
  const size_t parts = size_t(quad_ksplit(quad_tiles(E::NP, C::NFLD * epb))) * C::NFLD * epb *
                       E::NP;
  // (the results go over the nodal values)
  return (nodes > parts ? nodes : parts) + size_t(C::NFLD) * epb * (gs + fs);
}
template <int DIM, int P, int NSP, int MIX>
constexpr size_t quad_grad_lds(int gs, int fs, int epb) {
  using C = QuadNs<DIM, P, NSP, MIX, false>;
  using E = Elem<DIM, P>;
  const size_t nodes = size_t(epb) * C::ROWS * C::ST;
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
      for (int k = 0; k < C::NSD; ++k) v[C::G0 + k] = a.grad[k * N + g];
    }
#pragma unroll
    for (int f = 0; f < C::NQC; ++f) row[f] = v[f];
    if constexpr (GRAD) {
#pragma unroll
      for (int k = 0; k < C::NSD; ++k) row[C::G0 + k] = v[C::G0 + k];
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

// The waves' tasks: volume points 64 at a time, then face points; the first
// wave rotates with the block, so that two workgroups on a CU do not both
// give their surplus task to the same SIMD.
struct QuadTask {
  bool face;
  int t;   // point index among the workgroup's volume / face points, or -1
};
__device__ __forceinline__ int quad_task_count(int nvol, int nface) {
  return (nvol + 63) / 64 + (nface + 63) / 64;
}
__device__ __forceinline__ QuadTask quad_task(int task, int nvol, int nface) {
  const int nv = (nvol + 63) / 64;
  QuadTask k;
  k.face = task >= nv;
  k.t = (k.face ? task - nv : task) * 64 + int(threadIdx.x & 63);
  if (k.t >= (k.face ? nface : nvol)) k.t = -1;
  return k;
}
__device__ __forceinline__ int quad_first_task() {
  return ((threadIdx.x >> 6) + (blockIdx.x >> 3)) & (kWaves - 1);
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
  const int ntask = quad_task_count(ne * nq, ne * nfq_all);
  for (int task = quad_first_task(); task < ntask; task += kWaves) {
    const QuadTask tk = quad_task(task, ne * nq, ne * nfq_all);
    if (tk.t < 0) continue;
    if (!tk.face) {
      const int le = tk.t / nq;
      const int m = tk.t - le * nq;
      double u[NQC];
      quad_interp<NQC, NP>(qa.interp + m, nq, s_n + le * C::ROWS * ST, node, u);
      const double tq = quad_point_temperature<DIM, NSP, MIX>(u, MIX ? u[NQC - 1] : 0.0,
                                                              a.gas, qa.niter);
#pragma unroll
      for (int f = 0; f < NFLD; ++f) s_u[(f * epb + le) * gs + m] = u[f];
      s_u[(NFLD * epb + le) * gs + m] = tq;
    } else {
      const int le = tk.t / nfq_all;
      const int rem = tk.t - le * nfq_all;
      const int fc = rem / nfq;
      const int m = rem - fc * nfq;
      const int64_t e = e0 + le;
      const int32_t v0 = a.vmap_p[(e * NF + fc) * NFP];
      const double sc = a.fscale[e * NF + fc];
      double um[NQC], up[NQC];
      const double* w = qa.finterp + fc * NFP * nfq + m;
      const double* rows = s_n + le * C::ROWS * ST;
      auto own = [&](int j) { return s_fm[fc * NFP + j]; };
      double tp;
      if (v0 >= 0) {
        quad_interp<NQC, NFP>(w, nfq, rows, own, um);
        const double tm = quad_point_temperature<DIM, NSP, MIX>(
            um, MIX ? um[NQC - 1] : 0.0, a.gas, qa.niter);
        quad_interp<NQC, NFP>(w, nfq, rows + (NP + fc * NFP) * ST, node, up);
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

template <int DIM, int P, int NSP, int MIX>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(2))) void ns_div_quad_kernel(KArgs a, QuadArgs qa) {
  using E = Elem<DIM, P>;
  using C = QuadNs<DIM, P, NSP, MIX, true>;
  constexpr int NP = E::NP, NFP = E::NFP, NF = E::NF, ST = C::ST;
  constexpr int NFLD = C::NFLD, NSD = C::NSD, NQC = C::NQC, G0 = C::G0;
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
  const int ntask = quad_task_count(ne * nq, ne * nfq_all);
  for (int task = quad_first_task(); task < ntask; task += kWaves) {
    const QuadTask tk = quad_task(task, ne * nq, ne * nfq_all);
    if (tk.t < 0) continue;
    if (!tk.face) {
      const int le = tk.t / nq;
      const int m = tk.t - le * nq;
      const double* rows = s_n + le * C::ROWS * ST;
      const double* w = qa.interp + m;
      Node<DIM, NSP> s;
      {
        double u[NQC];
        quad_interp<NQC, NP>(w, nq, rows, node, u);
        double tq = 0.0;
        if constexpr (MIX != 0) tq = point_temperature<DIM, NSP>(u, u[NQC - 1], qa.niter);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) s.q[f] = u[f];
        node_state<DIM, NSP, MIX>(s, a.gas, tq);
      }
      double gacc[NSD], F[NFLD][DIM];
      quad_interp<NSD, NP>(w, nq, rows + G0, node, gacc);
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
      const int le = tk.t / nfq_all;
      const int rem = tk.t - le * nfq_all;
      const int fc = rem / nfq;
      const int m = rem - fc * nfq;
      const int64_t e = e0 + le;
      const int32_t v0 = a.vmap_p[(e * NF + fc) * NFP];
      const double* rows = s_n + le * C::ROWS * ST;
      double n[DIM];
#pragma unroll
      for (int d = 0; d < DIM; ++d) n[d] = a.normals[(e * NF + fc) * DIM + d];
      const double* w = qa.finterp + fc * NFP * nfq + m;
      const int ext0 = (NP + fc * NFP) * ST;
      auto own = [&](int j) { return s_fm[fc * NFP + j]; };
      Node<DIM, NSP> sm, sp;
      double fstar[NFLD], fv[NFLD];
      // the own side's state and viscous flux first, then the other side's, so
      // that one gradient set is live
      {
        double u[NQC], tm = 0.0, gacc[NSD];
        quad_interp<NQC, NFP>(w, nfq, rows, own, u);
        if constexpr (MIX != 0) tm = point_temperature<DIM, NSP>(u, u[NQC - 1], qa.niter);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) sm.q[f] = u[f];
        node_state<DIM, NSP, MIX>(sm, a.gas, tm);
        quad_interp<NSD, NFP>(w, nfq, rows + G0, own, gacc);
        viscous_flux_n<DIM, NSP, MIX>(sm, reinterpret_cast<const double(*)[DIM]>(gacc),
                                      gacc + NFLD * DIM, n, fv);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) fstar[f] = -0.5 * fv[f];
      }
      double tp = 0.0;
      if (v0 >= 0) {
        double u[NQC];
        quad_interp<NQC, NFP>(w, nfq, rows + ext0, node, u);
        if constexpr (MIX != 0) tp = point_temperature<DIM, NSP>(u, u[NQC - 1], qa.niter);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) sp.q[f] = u[f];
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
      {
        // the other side's gradient trace: the neighbour's (interior faces)
        // or this element's own (boundary faces)
        double gacc[NSD];
        quad_interp<NSD, NFP>(
            w, nfq, rows + G0, [&](int j) { return v0 >= 0 ? ext0 + j * ST : own(j); }, gacc);
        viscous_flux_n<DIM, NSP, MIX>(sp, reinterpret_cast<const double(*)[DIM]>(gacc),
                                      gacc + NFLD * DIM, n, fv);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) fstar[f] -= 0.5 * fv[f];
      }
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
