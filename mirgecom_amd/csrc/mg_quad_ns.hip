// Overintegrated Navier-Stokes gradients (include/mgdg.h):
// mg_ns_gradient_quad.
#include "mg_quad_ns.h"

extern "C" {

mg_status mg_ns_gradient_quad(const mg_mesh* mesh, const mg_gas* gas, const mg_quad* quad,
                              const double* q, const double* temperature,
                              const double* q_bnd_quad, const double* t_bnd_quad,
                              int32_t niter, double* grad, void* stream) {
  mg_status s = quad_ns_check(mesh, gas, quad, q, temperature, q_bnd_quad, t_bnd_quad,
                              niter, grad);
  if (s) return s;
  const int var = gas_variant(gas);
  const int gs = bank_stride(quad->nq);
  const int fs = bank_stride(mesh->nfaces * quad->nfq);
  mgdg::KArgs a = make_args(mesh, gas);
  a.q = q;
  a.out = grad;
  mgdg::QuadArgs qa{};
  quad_args(qa, mesh, quad, temperature, q_bnd_quad, t_bnd_quad, niter);
  qa.gs = gs;
  qa.fs = fs;
  hipStream_t st = static_cast<hipStream_t>(stream);
#define MG_GCASE(D, P, NS, MX)                                                      \
  if (mesh->dim == D && mesh->order == P && gas->nspecies == NS && var == MX) {     \
    constexpr auto lds = mgdg::quad_grad_lds<D, P, NS, MX>;                         \
    auto rounds = [&](int epb) {                                                    \
      using C = mgdg::QuadNs<D, P, NS, MX, false>;                                  \
      const int tasks = mgdg::quad_task_count<C::MM>(epb, qa.nq) +                  \
                        mgdg::quad_task_count<C::MM>((D + 1) * epb, qa.nfq);        \
      const int tiles = mgdg::quad_tiles(mgdg::Elem<D, P>::NP, (3 + D + NS) * epb);  \
      return (tasks + 3) / 4 + 2 * ((tiles + 3) / 4);                               \
    };                                                                              \
    return quad_launch(mgdg::ns_grad_quad_kernel<D, P, NS, MX>, lds,                \
                       quad_epb_rounds(quad_epb(lds, qa), rounds),                  \
                       "ns_grad_quad_kernel", a, qa, st);                           \
  }
  MG_NSQ_CASES(MG_GCASE)
#undef MG_GCASE
  return fail(MG_ERR_UNSUPPORTED, "dim/order/gas");
}

}  // extern "C"
