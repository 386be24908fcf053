// Overintegrated Navier-Stokes RHS (include/mgdg.h): mg_ns_rhs_quad.
#include "mg_quad_ns.h"

extern "C" {

mg_status mg_ns_rhs_quad(const mg_mesh* mesh, const mg_gas* gas, const mg_quad* quad,
                         const double* q, const double* temperature, const double* grad,
                         const double* q_bnd_quad, const double* t_bnd_quad, int32_t niter,
                         int32_t flux_kind, int32_t inviscid_on, double* rhs,
                         void* stream) {
  mg_status s = quad_ns_check(mesh, gas, quad, q, temperature, q_bnd_quad, t_bnd_quad,
                              niter, rhs);
  if (s) return s;
  if (!grad) return fail(MG_ERR_ARG, "grad NULL");
  if (flux_kind < 0 || flux_kind > 2) return fail(MG_ERR_ARG, "flux_kind");
  const int var = gas_variant(gas);
  const int gs = bank_stride(mesh->dim * quad->nq);
  const int fs = bank_stride(mesh->nfaces * quad->nfq);
  mgdg::KArgs a = make_args(mesh, gas);
  a.q = q;
  a.grad = grad;
  a.out = rhs;
  a.flux_kind = flux_kind;
  a.inviscid_on = inviscid_on ? 1 : 0;
  mgdg::QuadArgs qa{};
  quad_args(qa, mesh, quad, temperature, q_bnd_quad, t_bnd_quad, niter);
  qa.gs = gs;
  qa.fs = fs;
  hipStream_t st = static_cast<hipStream_t>(stream);
#define MG_DCASE(D, P, NS, MX)                                                      \
  if (mesh->dim == D && mesh->order == P && gas->nspecies == NS && var == MX) {     \
    constexpr auto lds = mgdg::quad_div_lds<D, P, NS, MX>;                          \
    return quad_launch(mgdg::ns_div_quad_kernel<D, P, NS, MX>, lds,                 \
                       quad_epb(lds, qa), "ns_div_quad_kernel", a, qa, st);         \
  }
  MG_NSQ_CASES(MG_DCASE)
#undef MG_DCASE
  return fail(MG_ERR_UNSUPPORTED, "dim/order/gas");
}

}  // extern "C"
