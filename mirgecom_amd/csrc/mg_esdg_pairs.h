// Entropy-stable (flux-differencing) Euler kernels of 3-D elements with a
// quadrature of (Q+1)^3 volume and 12 (Q+1)^2 face points: the default one (Q = p)
// and, without a mixture, Q = 3 at every order.  Each two-point flux is evaluated
// once, for both of its rows; other rules and 2-D take the row-by-row kernels
// (mgdg_kernels.h).
//
// Measured on an MI355X (kernel with the projection, row by row -- ideal gas
// p = 3: an earlier paired kernel -- -> this layout): ideal gas p = 3, 82,944 tets
// 6.33 -> 4.39 ms; uiuc_7sp mixture p = 2, 24,576 tets 4.37 -> 1.14 ms (the
// row-by-row kernel evaluates 6,561 fluxes per element, this one 3,267); p = 1,
// 15,288 tets 0.92 -> 0.28 ms; p = 3, 6,000 tets 3.08 -> 1.15 ms.  The ideal gas is
// bound by FP64 VALU issue (busy 70 % of the cycles with two waves per SIMD; LDS
// 32 %), half of it in the pair loop, the rest in the states and the contraction;
// the mixture at p = 2 by LDS (70 % busy) and VALU (51 %).
#pragma once
#include <cstddef>
#include <type_traits>

#include "mgdg_kernels.h"

namespace mgdg {

// {{{ the pair loop
//
// (Q_h - Q_h^T) is skew and F_S symmetric, so a pair of points adds its flux
// to one row and the negative to the other.  The rows fall into groups of nq:
// the volume rows and G = 12/(p+1) blocks of face rows.  A group takes nq
// lanes of a wave (GPW groups per wave).  In step t lane l meets the volume
// point (l + t) mod nq -- a face row for t = 0..nq-1, a volume row for
// t = 1..nq/2 (the last, for even nq, meets its own pair from both ends and
// each lane adds its own row) -- adds the flux to its own row and to a
// vector that moves one lane down per step, so that lane l always holds the
// partner row (l + t) mod nq; the face-face block is zero.
//
// An element has four slots, spread over the workgroup's 4 GPW lane groups:
// NB of them share the face blocks (RT = G/NB rows per lane, all meeting the
// same volume point, which is then read from LDS once and moved once per step
// for RT fluxes) and each block's steps are cut into NC = 4/NB pieces; the
// volume rows' steps are cut into four.  Every slot so has the same work.
// RT as large as the registers hold: of two waves per SIMD where two
// workgroups share a CU's LDS (the ideal gas, and 12 fields at p = 2: for the
// mixture two rows per lane spilled in the loop there and took 5 % longer
// than one; three waves per SIMD for the ideal gas spilled and
// took 7.5 ms.  The sums stay in registers until all of the
// workgroup's pairs are done and then go over the points' LDS: four pieces
// of the volume rows, NC of the face rows, added before the last phase.
template <int Q, bool MIX>
struct EsdgPairs {
  static constexpr int NQ = (Q + 1) * (Q + 1) * (Q + 1);
  static constexpr int NFQ = 3 * (Q + 1) * (Q + 1);
  static constexpr int NFT = 4 * NFQ;
  static constexpr int NH = NQ + NFT;
  static constexpr int G = NFT / NQ;
  static constexpr int GPW = 64 / NQ;
  static constexpr int EPB = GPW;            // elements per workgroup
  static constexpr int SPAN = GPW > 4 ? 256 / GPW : 64;   // a wave's lanes to an element
  static constexpr int NB = Q == 3 ? 1 : (Q == 2 && MIX) ? 4 : 2;
  static constexpr int RT = G / NB;
  static constexpr int NC = 4 / NB;
  static constexpr int NACC = 4 * NQ + NC * NFT;   // row sums per field
  // doubles between two elements' points past the points themselves: at p = 2
  // a wave's two lane groups then read as one run of points (LDS banks)
  static constexpr int PAD = Q == 2 ? 24 : 0;
  template <class Pt>
  static constexpr int POINTS = EPB * (int(sizeof(Pt)) / 8 * NH + PAD);
  template <class Pt>
  static __device__ __forceinline__ Pt* points(Pt* s_pt, int le) {
    using D = std::conditional_t<std::is_const_v<Pt>, const double, double>;
    return reinterpret_cast<Pt*>(reinterpret_cast<D*>(s_pt) +
                                 le * (int(sizeof(Pt)) / 8 * NH + PAD));
  }
  // lane group and element of a thread (lanes past GPW * NQ repeat the first
  // group's first lane and store nothing)
  static __device__ __forceinline__ int group() {
    const int wl = threadIdx.x & 63;
    return wl < GPW * NQ ? wl / NQ : 0;
  }
  static __device__ __forceinline__ int element() {
    return ((threadIdx.x >> 6) * GPW + group()) >> 2;
  }
  static_assert(G * NQ == NFT && RT * NB == G && kWaves == 4, "row groups");
};

template <int Q, bool MIX, class Flux>
__device__ __forceinline__ void esdg_pair_rows(const KArgs& a, const EsdgArgs& ea,
                                               const Flux& flux,
                                               const typename Flux::Point* s_pt,
                                               const double* s_log, int s_off,
                                               const double* s_fs,
                                               double* s_acc, int64_t e0, int ne) {
  using C = EsdgPairs<Q, MIX>;
  constexpr int DIM = 3, NF = DIM + 1, NFLD = Flux::NFLD, NSP = Flux::NSP, NV = 2 + DIM;
  constexpr int NQ = C::NQ, NFT = C::NFT, RT = C::RT, NC = C::NC;
  using Pt = typename Flux::Point;
  const int wl = threadIdx.x & 63;
  const bool lane_on = wl < C::GPW * NQ;
  const int sub = C::group();
  const int l = lane_on ? wl - sub * NQ : 0;
  const int base = sub * NQ;
  const int le = C::element(), sq = ((threadIdx.x >> 6) * C::GPW + sub) & 3;
  const int64_t e = le < ne ? e0 + le : e0;
  const Pt* pt = C::points(s_pt, le);
  const double* lg = Flux::LOGS == 2 ? s_log + le * C::NH * 2
                                     : reinterpret_cast<const double*>(pt) + s_off;
  const int next = base + (l + 1 == NQ ? 0 : l + 1);

  // face rows: block b = blk + r holds rows b NQ + l.  The row's own half of
  // the mean velocity and mass fractions and its face's constant normal are
  // taken out of the sums: acc holds sum m, sum energy, sum m u_j / 2,
  // sum m Y_j / 2, and prs the sum of the pressures.
  const int blk = (sq % C::NB) * RT, chunk = sq / C::NB;
  const int t0 = chunk * NQ / NC, t1 = (chunk + 1) * NQ / NC;
  double acc[RT][NFLD], mv[NFLD];
#pragma unroll
  for (int f = 0; f < NFLD; ++f) {
    mv[f] = 0.0;
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][f] = 0.0;
  }
  {
    Pt pm[RT];
    double nrm[RT][DIM], un0[RT], prs[RT], en[RT];
    const double* ed = ea.ext_diag + blk * NQ + l;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int m = (blk + r) * NQ + l;
      const int fc = m / C::NFQ;
      pm[r] = pt[NQ + m];
      const double bsc = a.fscale[e * NF + fc] * ea.wf[m - fc * C::NFQ];
      un0[r] = 0.0;
      prs[r] = 0.0;
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        nrm[r][d] = bsc * a.normals[(e * NF + fc) * DIM + d];
        un0[r] += nrm[r][d] * pm[r].uh[d];
      }
      en[r] = ed[t0 * NFT + r * NQ];
    }
    int j = l + t0 < NQ ? l + t0 : l + t0 - NQ;
    for (int t = t0; t < t1; ++t) {
      double ev[RT];
#pragma unroll
      for (int r = 0; r < RT; ++r) ev[r] = en[r];
      const int tn = t + 1 < t1 ? t + 1 : t0;   // the next step's entries
#pragma unroll
      for (int r = 0; r < RT; ++r) en[r] = ed[tn * NFT + r * NQ];
      const Pt pj = pt[j];
      LnPair ln[RT];
#pragma unroll
      for (int r = 0; r < RT; ++r) flux.begin(pm[r], pj, ln[r]);
      ln_means<Flux::SHORT, C::SPAN>(ln, [&](int r, double& e1, double& e2) {
        const double* lm = lg + Flux::LOGS * (NQ + (blk + r) * NQ + l);
        const double* lj = lg + Flux::LOGS * j;
        e1 = lj[0] - lm[0];
        e2 = lj[Flux::LOG2] - lm[Flux::LOG2];
      });
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        double rho, eng, prm, un = un0[r];
        flux.finish(pm[r], pj, ln[r], rho, eng, prm);
#pragma unroll
        for (int d = 0; d < DIM; ++d) un = fma(nrm[r][d], pj.uh[d], un);
        const double m = rho * (ev[r] * un), pe = prm * ev[r];
        const double en_flux = fma(eng, m, pe * un);
        acc[r][0] += m;
        acc[r][1] += en_flux;
        prs[r] += pe;
        mv[0] += m;
        mv[1] += en_flux;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
          acc[r][2 + d] = fma(m, pj.uh[d], acc[r][2 + d]);
          mv[2 + d] = fma(m, pm[r].uh[d], fma(nrm[r][d], pe, mv[2 + d]));
        }
        if constexpr (NSP > 0) {
#pragma unroll
          for (int k = 0; k < NSP; ++k) {
            acc[r][NV + k] = fma(m, pj.yh[k], acc[r][NV + k]);
            mv[NV + k] = fma(m, pm[r].yh[k], mv[NV + k]);
          }
        }
      }
#pragma unroll
      for (int f = 0; f < NFLD; ++f) mv[f] = __shfl(mv[f], next, 64);
      j = j + 1 == NQ ? 0 : j + 1;
    }
    // face rows take the negative sums
#pragma unroll
    for (int r = 0; r < RT; ++r) {
#pragma unroll
      for (int d = 0; d < DIM; ++d)
        acc[r][2 + d] = -fma(acc[r][0], pm[r].uh[d], fma(nrm[r][d], prs[r], acc[r][2 + d]));
      if constexpr (NSP > 0)
#pragma unroll
        for (int k = 0; k < NSP; ++k)
          acc[r][NV + k] = -fma(acc[r][0], pm[r].yh[k], acc[r][NV + k]);
      acc[r][0] = -acc[r][0];
      acc[r][1] = -acc[r][1];
    }
  }
  // the moving rows back home: lane l held row (l + t1) mod NQ
  double vol[NFLD];
  {
    const int h = l - t1;
    const int from = base + (h < 0 ? h + NQ : h);
#pragma unroll
    for (int f = 0; f < NFLD; ++f) {
      vol[f] = __shfl(mv[f], from, 64);
      mv[f] = 0.0;
    }
  }

  // volume rows (mv collects with the opposite sign)
  {
    constexpr int H = NQ / 2;
    const int u0 = 1 + sq * H / 4, u1 = 1 + (sq + 1) * H / 4;
    const Pt ph = pt[l];
    double rx[DIM * DIM];
#pragma unroll
    for (int k = 0; k < DIM * DIM; ++k) rx[k] = a.rx[e * DIM * DIM + k];
    int j = l + u0 < NQ ? l + u0 : l + u0 - NQ;
    for (int t = u0; t < u1; ++t) {
      double sd[DIM];
#pragma unroll
      for (int d = 0; d < DIM; ++d) sd[d] = 0.0;
#pragma unroll
      for (int r = 0; r < DIM; ++r) {
        const double sr = ea.skew_diag[(r * NQ + t) * NQ + l];
#pragma unroll
        for (int d = 0; d < DIM; ++d) sd[d] += rx[r * DIM + d] * sr;
      }
      const Pt pj = pt[j];
      double rho, eng, prm, un = 0.0;
      LnPair ln[1];
      flux.begin(ph, pj, ln[0]);
      ln_means<Flux::SHORT, C::SPAN>(ln, [&](int, double& e1, double& e2) {
        e1 = lg[Flux::LOGS * j] - lg[Flux::LOGS * l];
        e2 = lg[Flux::LOGS * j + Flux::LOG2] - lg[Flux::LOGS * l + Flux::LOG2];
      });
      flux.finish(ph, pj, ln[0], rho, eng, prm);
#pragma unroll
      for (int d = 0; d < DIM; ++d) un = fma(sd[d], ph.uh[d] + pj.uh[d], un);
      const double m = rho * un;
      const double en_flux = fma(eng, m, prm * un);
      // (t = nq/2: both lanes of a pair add their own row)
      const double mo = 2 * t == NQ ? 0.0 : m;
      vol[0] += m;
      vol[1] += en_flux;
      mv[0] += mo;
      mv[1] += 2 * t == NQ ? 0.0 : en_flux;
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        const double sp = sd[d] * prm;
        vol[2 + d] += fma(m, pj.uh[d], sp);
        mv[2 + d] += fma(mo, ph.uh[d], 2 * t == NQ ? 0.0 : sp);
      }
      if constexpr (NSP > 0) {
#pragma unroll
        for (int k = 0; k < NSP; ++k) {
          vol[NV + k] = fma(m, pj.yh[k], vol[NV + k]);
          mv[NV + k] = fma(mo, ph.yh[k], mv[NV + k]);
        }
      }
#pragma unroll
      for (int f = 0; f < NFLD; ++f) mv[f] = __shfl(mv[f], next, 64);
      j = j + 1 == NQ ? 0 : j + 1;
    }
    const int h = l - u1;
    const int from = base + (h < 0 ? h + NQ : h);
#pragma unroll
    for (int f = 0; f < NFLD; ++f) vol[f] -= __shfl(mv[f], from, 64);
    // the row's own halves, with its mass sum
#pragma unroll
    for (int d = 0; d < DIM; ++d) vol[2 + d] = fma(vol[0], ph.uh[d], vol[2 + d]);
    if constexpr (NSP > 0) {
#pragma unroll
      for (int k = 0; k < NSP; ++k) vol[NV + k] = fma(vol[0], ph.yh[k], vol[NV + k]);
    }
  }
  const bool on = lane_on && le < ne;
  if (on && chunk == 0) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int f = 0; f < NFLD; ++f)
        acc[r][f] += s_fs[(f * C::EPB + le) * NFT + (blk + r) * NQ + l];
  }
  __syncthreads();
  if (on) {
#pragma unroll
    for (int f = 0; f < NFLD; ++f) {
      double* row = s_acc + (f * C::EPB + le) * C::NACC;
      row[sq * NQ + l] = vol[f];
#pragma unroll
      for (int r = 0; r < RT; ++r)
        row[4 * NQ + chunk * NFT + (blk + r) * NQ + l] = acc[r][f];
    }
  }
  __syncthreads();
}

// dQ/dt = -M^-1 V_h^T acc: the pieces of every row added in place; then a
// lane holds one node and NFLD/FS fields of one element and takes every SPL-th
// part of the rows, so that each operator entry it reads serves those fields
// and its reads are all in flight together (lanes over outputs, a quarter of
// the rows per wave, waited on the operator eight reads at a time); s_part
// holds the SPL partial results.
template <int P, int Q, bool MIX, int NFLD>
struct EsdgApply {
  using C = EsdgPairs<Q, MIX>;
  static constexpr int NP = Elem<3, P>::NP;
  static constexpr int FS = NFLD > 6 ? 2 : 1;
  static constexpr int FL = (NFLD + FS - 1) / FS;
  static constexpr int GRP = NP * FS;                      // lanes of one split
  static constexpr int SPL = kBlock / GRP / C::EPB;        // splits per element
  static constexpr int RPL = (C::NH + SPL - 1) / SPL;      // rows per lane
  static constexpr int PART = SPL * C::EPB * NFLD * NP;    // doubles of s_part
  static_assert(FL * FS == NFLD && SPL >= 1, "fields per lane");
};

template <int P, int Q, bool MIX, int NFLD>
__device__ __forceinline__ void esdg_pair_apply(const KArgs& a, const EsdgArgs& ea,
                                                double* s_acc, double* s_part, int64_t e0,
                                                int ne) {
  using C = EsdgPairs<Q, MIX>;
  using A = EsdgApply<P, Q, MIX, NFLD>;
  constexpr int NP = A::NP, NQ = C::NQ, NFT = C::NFT, NH = C::NH;
  constexpr int FS = A::FS, FL = A::FL, SPL = A::SPL, RPL = A::RPL;
  const int split = threadIdx.x / A::GRP;
  const int le = split / SPL, sp = split - le * SPL;
  const int lane = threadIdx.x - split * A::GRP;
  const int fs = lane / NP, i = lane - fs * NP;
  const bool on = le < C::EPB;
  const int r0 = sp * RPL;
  double w[RPL];
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    // (rows past the last one: the last row's sums times zero)
    const bool in = on && r0 + k < NH;
    const double x = ea.apply[(in ? r0 + k : 0) * NP + i];
    w[k] = in ? x : 0.0;
  }
  for (int t = threadIdx.x; t < NFLD * C::EPB * NH; t += kBlock) {
    const int fl = t / NH;
    const int h = t - fl * NH;
    double* sa = s_acc + fl * C::NACC;
    if (h < NQ) {
      sa[h] = (sa[h] + sa[NQ + h]) + (sa[2 * NQ + h] + sa[3 * NQ + h]);
    } else {
      double* sf = sa + 4 * NQ + (h - NQ);
      double v = sf[0];
#pragma unroll
      for (int c = 1; c < C::NC; ++c) v += sf[c * NFT];
      sf[0] = v;
    }
  }
  __syncthreads();
  if (on) {
    double o[FL];
#pragma unroll
    for (int f = 0; f < FL; ++f) o[f] = 0.0;
    const double* sa = s_acc + (fs * FL * C::EPB + le) * C::NACC;
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int h = r0 + k < NH ? r0 + k : NH - 1;
      const double* row = sa + (h < NQ ? h : h + 3 * NQ);
#pragma unroll
      for (int f = 0; f < FL; ++f) o[f] += w[k] * row[f * C::EPB * C::NACC];
    }
#pragma unroll
    for (int f = 0; f < FL; ++f)
      s_part[((sp * NFLD + fs * FL + f) * C::EPB + le) * NP + i] = o[f];
  }
  __syncthreads();
  const int64_t N = a.nnodes;
  constexpr int NOUT = NFLD * C::EPB * NP;
  for (int o = threadIdx.x; o < NOUT; o += kBlock) {
    const int f = o / (C::EPB * NP);
    const int r = o - f * C::EPB * NP;
    double v = s_part[o];
#pragma unroll
    for (int k = 1; k < SPL; ++k) v += s_part[k * NOUT + o];
    if (r < ne * NP) a.out[f * N + e0 * NP + r] = -v;
  }
}

// Waves per SIMD to plan the registers for: two where two workgroups fit a CU's
// LDS, all registers for one otherwise (12 fields at Q = 1 and 3: with the
// registers of two they spilled up to 330; mixture p = 1, 24,576 tets 723 -> 413
// us, p = 3, 6,000 tets 2541 -> 1143; passive species p = 1 374 -> 250, p = 3
// 1502 -> 855).
constexpr int esdg_waves(size_t lds) { return lds <= 80 * 1024 ? 2 : 1; }

// }}}

// {{{ states at the hybridized points
//
// The projected entropy variables are held in LDS node by node, relative to
// the element's first node (the interpolations reproduce constants), the
// neighbours' face-node values alike: [EPB][NP + NF NFP][STRIDE], STRIDE
// even for 16-byte reads, and the first node's own values [EPB][STRIDE].
// With w = -v_1 (= rho/p), k = sum v_d^2 / (2 w) the state follows without
// powers:  ln rho = v_0 + k - (gamma + ln w) / (gamma - 1),  u_d = v_d / w,
// p = rho / w  (entropy_to_cons, gas_model.py:1063-1100, in logarithms): one
// log and one exp per point instead of two pows and an exp, taken relative to
// the first node so that nothing is lost to the size of the exponents.  The
// interior states took 24,000 cycles per workgroup with the powers, 16,000 so.

template <int P, int Q, int STRIDE>
struct EsdgNodes {
  using E = Elem<3, P>;
  using C = EsdgPairs<Q, false>;
  static constexpr int ROWS = E::NP + E::NFN + 1;
  static constexpr int SIZE = C::EPB * ROWS * STRIDE;
};

// Element le's nodal values: rows 0..NP-1 own nodes, then the face nodes'
// exterior values, then the reference (first node).
template <int P, int Q, int STRIDE>
__device__ __forceinline__ double* esdg_node_row(double* s_n, int le, int row) {
  return s_n + (le * EsdgNodes<P, Q, STRIDE>::ROWS + row) * STRIDE;
}

// Fill them (fields of ev; extra(row, g) adds columns of its own for node g).
template <int P, int Q, int NFLD, int STRIDE, typename Extra>
__device__ __forceinline__ void esdg_load_nodes(const KArgs& a, const EsdgArgs& ea,
                                                double* s_n, int64_t e0, int ne,
                                                Extra extra) {
  using E = Elem<3, P>;
  constexpr int NP = E::NP, NFN = E::NFN, ROWS = EsdgNodes<P, Q, STRIDE>::ROWS;
  const int64_t N = a.nnodes;
  for (int t = threadIdx.x; t < ne * ROWS; t += kBlock) {
    const int le = t / ROWS;
    const int r = t - le * ROWS;
    const int64_t g0 = (e0 + le) * NP;
    int64_t g = g0;
    if (r < NP) g = g0 + r;
    else if (r < NP + NFN) g = a.vmap_p[(e0 + le) * NFN + r - NP];
    if (g < 0) continue;   // boundary face node: not read
    double* row = esdg_node_row<P, Q, STRIDE>(s_n, le, r);
    const bool first = r == NP + NFN;
#pragma unroll
    for (int f = 0; f < NFLD; ++f) {
      const double v = ea.ev[f * N + g], v0 = ea.ev[f * N + g0];
      row[f] = first ? v0 : v - v0;
    }
    extra(row, g);
  }
}

// sum_i w[i ws] row_i[c] over n rows (LDS, STRIDE apart) for all columns.
template <int STRIDE, int NCOL, int NMAX>
__device__ __forceinline__ void esdg_interp(const double* w, int ws, const double* rows,
                                            int n, double* out) {
  double wi[NMAX];
#pragma unroll
  for (int i = 0; i < NMAX; ++i) wi[i] = w[(i < n ? i : 0) * ws];
#pragma unroll
  for (int c = 0; c < NCOL; ++c) out[c] = 0.0;
#pragma unroll
  for (int i = 0; i < NMAX; ++i) {
    if (i < n) {
#pragma unroll
      for (int c = 0; c < NCOL; ++c) out[c] += wi[i] * rows[i * STRIDE + c];
    }
  }
}

// }}}

// {{{ ideal gas

template <int P, int Q, int NSP>
struct EsdgPairCfg {
  using C = EsdgPairs<Q, false>;
  static constexpr int NFLD = 5 + NSP;
  static constexpr int STRIDE = (NFLD + 1) / 2 * 2;
  static constexpr int NODES = EsdgNodes<P, Q, STRIDE>::SIZE;
  static constexpr int PART = EsdgApply<P, Q, false, NFLD>::PART;
  static constexpr int POINTS = C::template POINTS<EcPair<3, NSP>> +
                                C::EPB * (2 * C::NH + NFLD * C::NFT);
  static constexpr int ACC = C::EPB * NFLD * C::NACC;
  // the sums go over the points and face fluxes, the partial results over
  // the nodal values
  static constexpr size_t LDS =
      sizeof(double) * ((POINTS > ACC ? POINTS : ACC) + (NODES > PART ? NODES : PART));
  static_assert(LDS <= 160 * 1024, "LDS per workgroup");
};

// The state of entropy variables ref + d: d relative to the reference node
// whose 1/w0, rho0 and k0 are given; logarithms relative to its own.
template <int NSP>
__device__ __forceinline__ void ec_state(const double* ref, const double* d, double gamma,
                                         EcPrim<3, NSP>& s) {
  const double igm1 = 1.0 / (gamma - 1.0);
  const double w0 = -ref[1], w = w0 - d[1];
  const double iw0 = rcp_nr(w0), iw = rcp_nr(w);
  double u2 = 0.0, v20 = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const double u = (ref[2 + i] + d[2 + i]) * iw;
    s.uh[i] = 0.5 * u;
    u2 += u * u;
    v20 += ref[2 + i] * ref[2 + i];
  }
  // k - k0 = w |u|^2 / 2 - sum ref_d^2 / (2 w0)
  const double l = log(w * iw0);
  const double x = d[0] + (0.5 * w * u2 - 0.5 * v20 * iw0) - l * igm1;
  s.lbeta = l;
  s.lrho = x;
  s.beta = 0.5 * w;
  s.kh = 0.25 * u2;
  s.rho = ref[0] * exp(x);
  s.p = s.rho * iw;
  s.c = sqrt(u2) + sqrt(gamma * iw);
  if constexpr (NSP > 0)
#pragma unroll
    for (int k = 0; k < NSP; ++k) s.yh[k] = 0.5 * (gamma - 1.0) * (ref[5 + k] + d[5 + k]);
}

// Entropy-stable face flux at an interior face point, times `sc`.
template <int NSP>
__device__ __forceinline__ void ec_face_flux(const EcPrim<3, NSP>& m, const EcPrim<3, NSP>& p,
                                             const double* n, double gamma, int dissipation,
                                             double sc, double* out) {
  double rho, eng, prm, un = 0.0;
  const EcPaired<3, NSP> flux(gamma);
  const EcPair<3, NSP> pm(m), pp(p);
  LnPair ln[1];
  flux.begin(pm, pp, ln[0]);
  // (the long series: the wave's other points belong to other elements)
  ln_means<false, 64>(ln, [&](int, double& e1, double& e2) {
    e1 = p.lrho - m.lrho;
    e2 = p.lbeta - m.lbeta;
  });
  flux.finish(pm, pp, ln[0], rho, eng, prm);
#pragma unroll
  for (int i = 0; i < 3; ++i) un += n[i] * (m.uh[i] + p.uh[i]);
  const double mass = rho * un;
  const double al = dissipation ? 0.5 * fmax(m.c, p.c) : 0.0;
  const double igm1 = 1.0 / (gamma - 1.0);
  const double em = m.p * igm1 + 2.0 * m.rho * m.kh, ep = p.p * igm1 + 2.0 * p.rho * p.kh;
  out[0] = sc * (mass - al * (p.rho - m.rho));
  out[1] = sc * (mass * eng + prm * un - al * (ep - em));
#pragma unroll
  for (int i = 0; i < 3; ++i)
    out[2 + i] = sc * (mass * (m.uh[i] + p.uh[i]) + n[i] * prm -
                       al * (2.0 * (p.rho * p.uh[i] - m.rho * m.uh[i])));
  if constexpr (NSP > 0)
#pragma unroll
    for (int k = 0; k < NSP; ++k)
      out[5 + k] = sc * (mass * (m.yh[k] + p.yh[k]) -
                         al * (2.0 * (p.rho * p.yh[k] - m.rho * m.yh[k])));
}

// ... at a boundary face point (quadrature point mm of face fc of element e):
// the interpolated interior state, through the entropy variables and back as
// the reference's projection does, and the condition's exterior state.
template <int P, int Q, int NSP>
__device__ __forceinline__ void ec_boundary_flux(const KArgs& a, const EsdgArgs& ea, int64_t e,
                                                 int fc, int mm, int32_t v0, const double* n,
                                                 double gamma, double sc, double* out) {
  using E = Elem<3, P>;
  using C = EsdgPairs<Q, false>;
  constexpr int NFLD = 5 + NSP;
  double ui[NFLD], vi[NFLD], qm[NFLD], qp[NFLD];
#pragma unroll
  for (int f = 0; f < NFLD; ++f) ui[f] = 0.0;
#pragma unroll 1
  for (int j = 0; j < E::NFP; ++j) {
    const double wj = ea.finterp[(fc * E::NFP + j) * C::NFQ + mm];
    const int64_t g = e * E::NP + a.fmask[fc * E::NFP + j];
#pragma unroll
    for (int f = 0; f < NFLD; ++f) ui[f] += wj * a.q[f * a.nnodes + g];
  }
  cons_to_entropy<3, NSP>(ui, gamma, vi);
  entropy_to_cons<3, NSP>(vi, gamma, qm);
  const int64_t bq = (-int64_t(v0) - 1) / E::NFP * C::NFQ + mm;
#pragma unroll
  for (int f = 0; f < NFLD; ++f) qp[f] = ea.qbq[f * ea.nbq + bq];
  EcPrim<3, NSP> pm, pp;
  ec_prim<3, NSP>(qm, gamma, pm);
  ec_prim<3, NSP>(qp, gamma, pp);
  double fs[NFLD];
#pragma unroll
  for (int f = 0; f < NFLD; ++f) fs[f] = 0.0;
  ec_flux_dot<3, NSP>(pm, pp, n, gamma, fs);
  const double al = ea.dissipation ? 0.5 * fmax(pm.c, pp.c) : 0.0;
#pragma unroll
  for (int f = 0; f < NFLD; ++f) out[f] = sc * (fs[f] - al * (qp[f] - qm[f]));
}

template <int P, int Q, int NSP>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(esdg_waves(EsdgPairCfg<P, Q, NSP>::LDS)))) void
esdg_pair_kernel(KArgs a, EsdgArgs ea) {
  using E = Elem<3, P>;
  using C = EsdgPairs<Q, false>;
  using Cfg = EsdgPairCfg<P, Q, NSP>;
  constexpr int NFLD = Cfg::NFLD, ST = Cfg::STRIDE, NH = C::NH, NFT = C::NFT;
  using Pt = EcPair<3, NSP>;
  extern __shared__ __align__(16) double lds16[];
  Pt* s_pt = reinterpret_cast<Pt*>(lds16);                            // [EPB][NH]
  double* s_log = lds16 + C::template POINTS<Pt>;                     // [EPB][NH][2]
  double* s_fs = s_log + 2 * C::EPB * NH;                             // [F][EPB][NFT]
  double* s_n = lds16 + (Cfg::POINTS > Cfg::ACC ? Cfg::POINTS : Cfg::ACC);
  const int64_t e0 = int64_t(blockIdx.x) * C::EPB;
  const int ne = a.K - e0 < C::EPB ? int(a.K - e0) : C::EPB;
  const double gamma = a.gas.gamma;
  // 1: projected entropy variables of the own and the neighbours' nodes
  esdg_load_nodes<P, Q, NFLD, ST>(a, ea, s_n, e0, ne, [](double*, int64_t) {});
  __syncthreads();
  if (int(threadIdx.x) < ne) {
    // the reference's v_0 becomes its density
    double* r = esdg_node_row<P, Q, ST>(s_n, threadIdx.x, E::NP + E::NFN);
    const double w0 = -r[1];
    const double v2 = r[2] * r[2] + r[3] * r[3] + r[4] * r[4];
    r[0] = exp(r[0] + 0.5 * v2 / w0 - (gamma + log(w0)) / (gamma - 1.0));
  }
  __syncthreads();
  // 2: the state at the hybridized points (face points first); at face
  // points also the neighbour's and the face flux times fscale * w
  for (int t = threadIdx.x; t < ne * NH; t += kBlock) {
    const bool face = t < ne * NFT;
    const int u = face ? t : t - ne * NFT;
    const int le = u / (face ? NFT : C::NQ);
    const int m = u - le * (face ? NFT : C::NQ);
    const int h = face ? C::NQ + m : m;
    const double* ref = esdg_node_row<P, Q, ST>(s_n, le, E::NP + E::NFN);
    double d[NFLD];
    EcPrim<3, NSP> s;
    esdg_interp<ST, NFLD, E::NP>(ea.vh + h, NH, esdg_node_row<P, Q, ST>(s_n, le, 0), E::NP, d);
    ec_state<NSP>(ref, d, gamma, s);
    C::points(s_pt, le)[h] = s;
    s_log[2 * (le * NH + h)] = s.lrho;
    s_log[2 * (le * NH + h) + 1] = s.lbeta;
    if (!face) continue;
    const int fc = m / C::NFQ;
    const int mm = m - fc * C::NFQ;
    const int64_t e = e0 + le;
    const int32_t v0 = a.vmap_p[(e * 4 + fc) * E::NFP];
    double n[3], fs[NFLD];
#pragma unroll
    for (int i = 0; i < 3; ++i) n[i] = a.normals[(e * 4 + fc) * 3 + i];
    const double sc = a.fscale[e * 4 + fc] * ea.wf[mm];
    if (v0 >= 0) {
      EcPrim<3, NSP> p;
      esdg_interp<ST, NFLD, E::NFP>(ea.finterp + fc * E::NFP * C::NFQ + mm, C::NFQ,
                                    esdg_node_row<P, Q, ST>(s_n, le, E::NP + fc * E::NFP),
                                    E::NFP, d);
      ec_state<NSP>(ref, d, gamma, p);
      ec_face_flux<NSP>(s, p, n, gamma, ea.dissipation, sc, fs);
    } else {
      ec_boundary_flux<P, Q, NSP>(a, ea, e, fc, mm, v0, n, gamma, sc, fs);
    }
#pragma unroll
    for (int f = 0; f < NFLD; ++f) s_fs[(f * C::EPB + le) * NFT + m] = fs[f];
  }
  __syncthreads();
  // 3: rows of (Q_h - Q_h^T) o F_S, plus the face flux on face rows
  esdg_pair_rows<Q, false>(a, ea, EcPaired<3, NSP>(gamma), s_pt, s_log, 0, s_fs, lds16, e0, ne);
  // 4: dQ/dt = -M^-1 V_h^T acc
  esdg_pair_apply<P, Q, false, NFLD>(a, ea, lds16, s_n, e0, ne);
}

// }}}

// {{{ uiuc_7sp mixture (Renac's flux; the phases of esdg_mix_kernel)

template <int P>
struct EsdgMixCfg {
  using C = EsdgPairs<P, true>;
  static constexpr int NFLD = 5 + MIX_NSP;
  static constexpr int STRIDE = NFLD + 2;   // + T, gamma(cv, T)
  static constexpr int NODES = EsdgNodes<P, P, STRIDE>::SIZE;
  static constexpr int PART = EsdgApply<P, P, true, NFLD>::PART;
  static constexpr int POINTS =
      C::template POINTS<RnPoint<3>> + C::EPB * NFLD * C::NFT;
  static constexpr int ACC = C::EPB * NFLD * C::NACC;
  static constexpr int BODY = POINTS > ACC ? POINTS : ACC;
  static constexpr size_t LDS =
      sizeof(double) * (BODY + (NODES > PART ? NODES : PART)) + sizeof(int) * 8;
  static_assert(STRIDE % 2 == 0 && C::EPB <= 8 && LDS <= 160 * 1024, "LDS per workgroup");
};

// State of a mixture point in the form the pair loop reads.
struct RnState {
  RnPoint<3> pt;
  double rho, c, energy;
};

// The state of entropy variables ref + d with ratio gh, T by Newton from
// `seed`: internal energy 1 / ((gh - 1) w).
__device__ __forceinline__ void rn_state(const double* ref, const double* d, double gh,
                                         double seed, int niter, RnState& s) {
  const double w = -(ref[1] + d[1]);
  const double iw = 1.0 / w, gm1 = gh - 1.0, igm1 = 1.0 / gm1;
  double u2 = 0.0, u[3], y[MIX_NSP];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    u[i] = (ref[2 + i] + d[2 + i]) * iw;
    u2 += u[i] * u[i];
  }
#pragma unroll
  for (int k = 0; k < MIX_NSP; ++k) y[k] = gm1 * (ref[5 + k] + d[5 + k]);
  s.pt.lrho[0] = (d[0] + ref[0]) + (0.5 * w * u2 - (gh + log(w)) * igm1);
  const double rho = exp(s.pt.lrho[0]);
  double cvp[5], r;
  const double t = mix_temperature_poly(iw * igm1, seed, y, niter, cvp, r);
  const double cv = horner5(cvp, t);
  s.pt.rhoh = 0.5 * rho;
  s.pt.t = 0.5 * t;
  s.pt.th = 1.0 / t;
  s.pt.pth = 0.5 * rho * r;
  s.rho = rho;
#pragma unroll
  for (int i = 0; i < 3; ++i) s.pt.uh[i] = 0.5 * u[i];
#pragma unroll
  for (int k = 0; k < MIX_NSP; ++k) s.pt.yh[k] = 0.5 * y[k];
#pragma unroll
  for (int i = 0; i < 5; ++i) s.pt.cv[i] = 0.5 * cvp[i];
  s.pt.lth = -log(t);
  s.c = sqrt(u2) + sqrt((1.0 + r / cv) * r * t);
  s.energy = rho * (iw * igm1 + 0.5 * u2);
}

// Boundary face point: the entropy-stable projected interior state and the
// condition's exterior state, times sc.
template <int P>
__device__ __forceinline__ void rn_boundary_flux(const KArgs& a, const EsdgArgs& ea, int64_t e,
                                                 int fc, int mm, int32_t v0, const double* n,
                                                 double sc, double* out) {
  using E = Elem<3, P>;
  using C = EsdgPairs<P, true>;
  constexpr int NFLD = 5 + MIX_NSP;
  double ui[NFLD];
#pragma unroll
  for (int f = 0; f < NFLD; ++f) ui[f] = 0.0;
  double seed = 0.0;
#pragma unroll 1
  for (int j = 0; j < E::NFP; ++j) {
    const double wj = ea.finterp[(fc * E::NFP + j) * C::NFQ + mm];
    const int64_t g = e * E::NP + a.fmask[fc * E::NFP + j];
#pragma unroll
    for (int f = 0; f < NFLD; ++f) ui[f] += wj * a.q[f * a.nnodes + g];
    seed += wj * a.temp[g];
  }
  Node<3, MIX_NSP> sm, sp;
  es_projected_state<3>(ui, seed, a.gas, ea.niter, sm);
  const int64_t bq = (-int64_t(v0) - 1) / E::NFP * C::NFQ + mm;
#pragma unroll
  for (int f = 0; f < NFLD; ++f) sp.q[f] = ea.qbq[f * ea.nbq + bq];
  node_state<3, MIX_NSP, 1, false>(sp, a.gas, ea.tbq[bq]);
  RnPrim<3> pm, pp;
  rn_prim<3>(sm, pm);
  rn_prim<3>(sp, pp);
  double fs[NFLD];
#pragma unroll
  for (int f = 0; f < NFLD; ++f) fs[f] = 0.0;
  rn_flux_dot<3>(pm, pp, n, fs);
  const double al = ea.dissipation ? 0.5 * fmax(pm.c, pp.c) : 0.0;
#pragma unroll
  for (int f = 0; f < NFLD; ++f) out[f] = sc * (fs[f] - al * (sp.q[f] - sm.q[f]));
}

template <int P>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(esdg_waves(EsdgMixCfg<P>::LDS)))) void
esdg_mix_pair_kernel(KArgs a, EsdgArgs ea) {
  using E = Elem<3, P>;
  using C = EsdgPairs<P, true>;
  using Cfg = EsdgMixCfg<P>;
  constexpr int NFLD = Cfg::NFLD, ST = Cfg::STRIDE, NH = C::NH, NFT = C::NFT, NQ = C::NQ;
  constexpr int IT = NFLD, IG = NFLD + 1;   // columns of T and gamma
  using Pt = RnPoint<3>;
  extern __shared__ __align__(16) double lds16[];
  Pt* s_pt = reinterpret_cast<Pt*>(lds16);                            // [EPB][NH]
  double* s_fs = lds16 + C::template POINTS<Pt>;                      // [F][EPB][NFT]
  double* s_n = lds16 + Cfg::BODY;
  // NASA7 ranges that hold all of an element's points (bit 0 low, 1 high)
  int* s_rng = reinterpret_cast<int*>(
      s_n + (Cfg::NODES > Cfg::PART ? Cfg::NODES : Cfg::PART));       // [EPB]
  const int64_t e0 = int64_t(blockIdx.x) * C::EPB;
  const int ne = a.K - e0 < C::EPB ? int(a.K - e0) : C::EPB;
  // 1: projected entropy variables and T of the own and the neighbours'
  // nodes, gamma(cv, T) of the own
  esdg_load_nodes<P, P, NFLD, ST>(a, ea, s_n, e0, ne, [&](double* row, int64_t g) {
    row[IT] = a.temp[g];
  });
  if (int(threadIdx.x) < C::EPB) s_rng[threadIdx.x] = 3;
  for (int t = threadIdx.x; t < ne * E::NP; t += kBlock) {
    const int64_t g = e0 * E::NP + t;
    const double irho = 1.0 / a.q[g], tn = a.temp[g];
    double y[MIX_NSP], cvp[5], r;
#pragma unroll
    for (int k = 0; k < MIX_NSP; ++k) y[k] = a.q[(5 + k) * a.nnodes + g] * irho;
    mix_temperature_poly(0.0, tn, y, 0, cvp, r);
    esdg_node_row<P, P, ST>(s_n, t / E::NP, t % E::NP)[IG] = 1.0 + r / horner5(cvp, tn);
  }
  __syncthreads();
  double tmid_lo, tmid_hi;
  nasa7_tmid_range(tmid_lo, tmid_hi);
  // 2: the state at the hybridized points, face points first, and for a face
  // point the neighbour's and the face flux times fscale * w.  A pass takes
  // 256 points in two evaluations: the second is the neighbour's state on
  // lanes with a face point, and on the others a volume point that the
  // passes over the face points leave over.
  constexpr int PASSES = (C::EPB * NFT + kBlock - 1) / kBlock;
  const int total = ne * NH, nface = ne * NFT;
#pragma unroll 1
  for (int pass = 0; pass < PASSES; ++pass) {
    const int it = pass * kBlock + int(threadIdx.x);
    const bool face = it < nface;
    RnState own;
    double gh = 0.0;
    int le = 0, m = 0;
#pragma unroll 1
    for (int ev = 0; ev < 2; ++ev) {
      const bool nbr = ev == 1 && face;
      // what this lane evaluates: a hybridized point, the neighbour's state
      // at its face point, or nothing
      int item = it;
      if (ev == 1 && !face)
        item = pass == PASSES - 1 ? PASSES * kBlock + (it - nface) : total;
      if (item >= total || (ev == 1 && !face && it >= total)) continue;
      if (!nbr) {
        const int u = item < nface ? item : item - nface;
        le = u / (item < nface ? NFT : NQ);
        m = u - le * (item < nface ? NFT : NQ);
      }
      const int h = (nbr || item < nface) ? NQ + m : m;
      const int fc = m / C::NFQ, mm = m - fc * C::NFQ;
      const int64_t e = e0 + le;
      const int32_t v0 = nbr ? a.vmap_p[(e * 4 + fc) * E::NFP] : 0;
      double n[3], fs[NFLD], sc = 0.0;
      if (nbr) {
#pragma unroll
        for (int i = 0; i < 3; ++i) n[i] = a.normals[(e * 4 + fc) * 3 + i];
        sc = a.fscale[e * 4 + fc] * ea.wf[mm];
      }
      if (v0 >= 0) {
        const double* ref = esdg_node_row<P, P, ST>(s_n, le, E::NP + E::NFN);
        double d[NFLD + 2];
        const double* w = nbr ? ea.finterp + fc * E::NFP * C::NFQ + mm : ea.vh + h;
        esdg_interp<ST, NFLD + 2, E::NP>(
            w, nbr ? C::NFQ : NH,
            esdg_node_row<P, P, ST>(s_n, le, nbr ? E::NP + fc * E::NFP : 0),
            nbr ? E::NFP : E::NP, d);
        if (!nbr) gh = d[IG];   // the neighbour's state takes this side's gamma
        RnState s;
        rn_state(ref, d, gh, d[IT], ea.niter, s);
        if (!nbr) {
          C::points(s_pt, le)[h] = s.pt;
          const int bits = (2.0 * s.pt.t < tmid_lo * (1.0 - 1e-9) ? 1 : 0) |
                           (2.0 * s.pt.t > tmid_hi * (1.0 + 1e-9) ? 2 : 0);
          if (bits != 3) atomicAnd(s_rng + le, bits);
          own = s;
        } else {
          double rho, eng, prm, un = 0.0;
          const RnPaired<3, false> flux(false);
          LnPair ln[1];
          flux.begin(own.pt, s.pt, ln[0]);
          ln_means<false, 64>(ln, [&](int, double& e1, double& e2) {
            e1 = s.pt.lrho[0] - own.pt.lrho[0];
            e2 = s.pt.lth - own.pt.lth;
          });
          flux.finish(own.pt, s.pt, ln[0], rho, eng, prm);
#pragma unroll
          for (int i = 0; i < 3; ++i) un += n[i] * (own.pt.uh[i] + s.pt.uh[i]);
          const double mass = rho * un;
          const double al = ea.dissipation ? 0.5 * fmax(own.c, s.c) : 0.0;
          fs[0] = mass - al * (s.rho - own.rho);
          fs[1] = mass * eng + prm * un - al * (s.energy - own.energy);
#pragma unroll
          for (int i = 0; i < 3; ++i)
            fs[2 + i] = mass * (own.pt.uh[i] + s.pt.uh[i]) + n[i] * prm -
                        al * (2.0 * (s.rho * s.pt.uh[i] - own.rho * own.pt.uh[i]));
#pragma unroll
          for (int k = 0; k < MIX_NSP; ++k)
            fs[5 + k] = mass * (own.pt.yh[k] + s.pt.yh[k]) -
                        al * (2.0 * (s.rho * s.pt.yh[k] - own.rho * own.pt.yh[k]));
#pragma unroll
          for (int f = 0; f < NFLD; ++f)
            s_fs[(f * C::EPB + le) * NFT + m] = sc * fs[f];
        }
      } else {
        rn_boundary_flux<P>(a, ea, e, fc, mm, v0, n, sc, fs);
#pragma unroll
        for (int f = 0; f < NFLD; ++f) s_fs[(f * C::EPB + le) * NFT + m] = fs[f];
      }
    }
  }
  __syncthreads();
  // 3: rows of (Q_h - Q_h^T) o F_S, plus the face flux on face rows: the loop
  // without the sums over species where every element of the workgroup keeps
  // to one NASA7 range
  bool poly = true;
  for (int le = 0; le < ne; ++le) poly = poly && s_rng[le] != 0;
  const bool own_poly = s_rng[C::element()] != 0;
  constexpr int LOG0 = offsetof(Pt, lrho) / sizeof(double);
  static_assert(sizeof(Pt) == 22 * 8 && offsetof(Pt, lth) == 8 * (LOG0 + 8), "point layout");
  if (poly)
    esdg_pair_rows<P, true>(a, ea, RnPaired<3, true>(true), s_pt, nullptr, LOG0, s_fs, lds16, e0,
                            ne);
  else
    esdg_pair_rows<P, true>(a, ea, RnPaired<3, false>(own_poly), s_pt, nullptr, LOG0, s_fs, lds16,
                            e0, ne);
  // 4: dQ/dt = -M^-1 V_h^T acc
  esdg_pair_apply<P, P, true, NFLD>(a, ea, lds16, s_n, e0, ne);
}

// }}}

}  // namespace mgdg
