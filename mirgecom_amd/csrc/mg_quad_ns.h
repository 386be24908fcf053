// Shared host code of the overintegrated Navier-Stokes entry points
// (mg_quad_ns.hip, mg_quad_ns_div.hip).
#pragma once
#include <algorithm>
#include <string>

#include "mg_quad_ns_kernels.h"
#include "mgdg_host.h"

namespace {

mg_status quad_ns_check(const mg_mesh* mesh, const mg_gas* gas, const mg_quad* quad,
                        const double* q, const double* temperature,
                        const double* q_bnd_quad, const double* t_bnd_quad, int32_t niter,
                        const double* out) {
  mg_status s = check_mesh(mesh);
  if (s) return s;
  if ((s = check_gas(gas, true))) return s;
  const bool mix = gas->eos_kind == 1;
  if (mix && (s = ensure_mech())) return s;
  if (gas->nspecies != 0 && gas->nspecies != 7)
    return fail(MG_ERR_UNSUPPORTED, "nspecies must be 0 or 7");
  if (mix && (!temperature || niter < 0 || (mesh->nbnd_nodes > 0 && !t_bnd_quad)))
    return fail(MG_ERR_ARG, "mixture needs temperature (and t_bnd_quad), niter >= 0");
  if (!quad || !quad->interp || !quad->weak_diff || !quad->face_interp || !quad->lift ||
      quad->nq < 1 || quad->nfq < 1)
    return fail(MG_ERR_ARG, "mg_quad incomplete");
  if (!q || !out) return fail(MG_ERR_ARG, "q/output NULL");
  if (mesh->nbnd_nodes > 0 && !q_bnd_quad)
    return fail(MG_ERR_ARG, "boundary exterior state missing");
  if (mesh->nbnd_nodes % mesh->nfp) return fail(MG_ERR_ARG, "nbnd_nodes % nfp");
  return MG_OK;
}

// LDS row strides = 4 mod 32 doubles (bank spread of the matrix-core reads)
int bank_stride(int n) { return n + ((4 - n % 32) + 32) % 32; }

// Elements per workgroup: at most 16, as many as leave room for two workgroups
// on a CU (80 KiB each); at least one, which may take up to 128 KiB.
constexpr size_t kQuadBudget = 128 * 1024;

template <typename Lds>
int quad_epb(Lds lds, const mgdg::QuadArgs& qa) {
  int epb = 1;
  while (epb < 16 && sizeof(double) * lds(qa.gs, qa.fs, epb + 1) <= 80 * 1024) ++epb;
  return epb;
}

// ... of those, the number with the fewest rounds(epb) of the four waves per
// element (tasks of points, and twice the contraction's tiles, one of whose rounds
// takes about as long as two of points), the largest on a tie.  Gradients, MI355X,
// the largest number -> this: ideal gas, tets, p = 1, 131,712 392 -> 335 us (14 ->
// 10 elements: 84 columns are six tiles of 16 and two rounds, 60 four and one),
// p = 4, 10,368 400 -> 334 us (3 -> 2), p = 2, 10,368 63 -> 55 us (8 -> 7), p = 3
// unchanged (5); mixture, 4,608 triangles, p = 4 44 -> 34 us.
template <typename Rounds>
int quad_epb_rounds(int most, Rounds rounds) {
  int epb = 1;
  for (int n = 2; n <= most; ++n)
    if (rounds(n) * epb <= rounds(epb) * n) epb = n;
  return epb;
}

template <typename Kern, typename Lds>
mg_status quad_launch(Kern kern, Lds lds, int epb, const char* name, const mgdg::KArgs& a,
                      mgdg::QuadArgs& qa, hipStream_t st) {
  const size_t bytes = sizeof(double) * lds(qa.gs, qa.fs, epb);
  if (bytes > kQuadBudget) return fail(MG_ERR_UNSUPPORTED, "quadrature too large for LDS");
  qa.epb = epb;
  mg_status s = set_lds(kern, kQuadBudget);
  if (s) return s;
  hipLaunchKernelGGL(kern, dim3(unsigned((a.K + epb - 1) / epb)), dim3(mgdg::kBlock), bytes, st,
                     a, qa);
  return check_launch(name);
}

void quad_args(mgdg::QuadArgs& qa, const mg_mesh* mesh, const mg_quad* quad,
               const double* temperature, const double* q_bnd_quad,
               const double* t_bnd_quad, int32_t niter) {
  qa.nq = quad->nq;
  qa.nfq = quad->nfq;
  qa.interp = quad->interp;
  qa.wdiff = quad->weak_diff;
  qa.finterp = quad->face_interp;
  qa.lift = quad->lift;
  qa.qbq = q_bnd_quad;
  qa.nbq = mesh->nbnd_nodes / mesh->nfp * quad->nfq;
  qa.temp = temperature;
  qa.tbq = t_bnd_quad;
  qa.niter = niter;
}

}  // namespace

#define MG_NSQ_CASES(X)                                                              \
  X(2, 1, 0, 0) X(2, 2, 0, 0) X(2, 3, 0, 0) X(2, 4, 0, 0)                           \
  X(3, 1, 0, 0) X(3, 2, 0, 0) X(3, 3, 0, 0) X(3, 4, 0, 0)                           \
  X(2, 1, 7, 0) X(2, 2, 7, 0) X(2, 3, 7, 0) X(2, 4, 7, 0)                           \
  X(3, 1, 7, 0) X(3, 2, 7, 0) X(3, 3, 7, 0) X(3, 4, 7, 0)                           \
  X(2, 1, 7, 1) X(2, 2, 7, 1) X(2, 3, 7, 1) X(2, 4, 7, 1)                           \
  X(3, 1, 7, 1) X(3, 2, 7, 1) X(3, 3, 7, 1) X(3, 4, 7, 1)                           \
  X(2, 1, 7, 2) X(2, 2, 7, 2) X(2, 3, 7, 2) X(2, 4, 7, 2)                           \
  X(3, 1, 7, 2) X(3, 2, 7, 2) X(3, 3, 7, 2) X(3, 4, 7, 2)

