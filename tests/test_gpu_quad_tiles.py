"""The overintegrated Navier-Stokes kernels' 3-D interpolation on the matrix
cores (mirgecom_amd/csrc/mg_quad_ns_kernels.h) against the oracle
(oracle/overintegration.py) where its tiles of 16 points and steps of 4 nodes
have remainders: rules of 8 to 125 volume and 12 to 75 face points at every
order, element counts that leave the last workgroup partly empty (6 elements of
a single cell, 36, 48), interior next to dummy-boundary faces in one wave.

Tolerance 1e-11 relative per field, as for the operator at the default rules
(tests/test_gpu_ns_quad.py).  At p = 3 and 4 it is the oracle's: its monomial
Lagrange basis makes the reference-element weak gradient differ from the
product's by 5.8e-13 and 1.06e-11 in the infinity norm (4.7e-14 at p = 2), which
up to 3 reference directions with metric factors 2 / 0.25 on the finest of these
grids carry into gradients of about 0.6 of fields of size 1: at most 40 times
that, 2.4e-11 and 4.3e-10 (seen: 1.1e-11 and 1.1e-10).
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests.cases import (  # noqa: E402
    Problem, mixture_state, rel_err, smooth_perturbed_state)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,degree", [(1, 2), (1, 5), (2, 3), (2, 4), (2, 7),
                                          (3, 4), (3, 8), (4, 6), (4, 8)])
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 2, 1), (4, 1, 2)])
def test_remainders(order, degree, n):
    from mirgecom_amd.boundary import DummyBoundary
    from mirgecom_amd.discretization import create_discretization_collection
    from mirgecom_amd.dof_desc import DISCR_TAG_QUAD
    from mirgecom_amd.eos import IdealSingleGas
    from mirgecom_amd.fluid import ConservedVars
    from mirgecom_amd.gas_model import GasModel, make_fluid_state
    from mirgecom_amd.navierstokes import ns_operator
    from mirgecom_amd.transport import SimpleTransport
    from oracle import operators as oop, physics as ph
    from oracle.overintegration import ns_operator_quad
    pb = Problem(3, order, n, 0.0, (1.0, 0.8, 0.9), (False,) * 3)
    dcoll = create_discretization_collection(pb.mesh, order, quadrature_order=degree)
    q = smooth_perturbed_state(pb.x, seed=order + degree, amp=0.1)
    kw = {"viscosity": 0.05, "thermal_conductivity": 0.07, "bulk_viscosity": 0.01}
    gm = GasModel(eos=IdealSingleGas(gas_const=1.0), transport=SimpleTransport(**kw))
    ogm = ph.GasModel(ph.IdealSingleGas(gas_const=1.0), ph.SimpleTransport(**kw))
    print(f"quad tiles p={order} degree={degree} n={n}", flush=True)
    dev = torch.as_tensor(np.ascontiguousarray(q), dtype=torch.float64, device="cuda")
    st = make_fluid_state(ConservedVars(3, dev), gm)
    rhs, gcv, gt = ns_operator(dcoll, gm, st, {"all": DummyBoundary()},
                               quadrature_tag=DISCR_TAG_QUAD, return_gradients=True)
    ref, rgcv, rgt = ns_operator_quad(pb.odisc, pb.box, q, ogm,
                                      {"all": oop.DummyBoundary()}, degree=degree,
                                      return_gradients=True)
    tol = {3: 2.4e-11, 4: 4.3e-10}.get(order, 1e-11)
    err = rel_err(rhs.q.cpu().numpy(), ref)
    eg = rel_err(gcv.q.cpu().numpy().reshape(-1, *ref.shape[1:]),
                 rgcv.reshape(-1, *ref.shape[1:]))
    et = rel_err(gt.cpu().numpy(), rgt)
    print("errors", err.max(), eg.max(), et.max())
    for e in (err, eg, et):
        assert (e < tol).all()


@pytest.mark.parametrize("gas", ["species", "mixture"])
@pytest.mark.parametrize("dim,order", [(2, 1), (2, 2), (2, 3), (2, 4),
                                       (3, 1), (3, 3), (3, 4)])
def test_columns(dim, order, gas):
    """Passive species and the mixture: 11 to 52 columns, in 3-D in two
    groups.  The mixture's pressure varies by a tenth of itself over the box, so
    the basis's error enters its right-hand side ten times larger."""
    from mirgecom_amd.boundary import DummyBoundary
    from mirgecom_amd.dof_desc import DISCR_TAG_QUAD
    from mirgecom_amd.eos import IdealSingleGas, PyrometheusMixture
    from mirgecom_amd.fluid import ConservedVars
    from mirgecom_amd.gas_model import GasModel, make_fluid_state
    from mirgecom_amd.navierstokes import ns_operator
    from mirgecom_amd.transport import SimpleTransport
    from oracle import operators as oop, physics as ph, thermochem as tc
    from oracle.overintegration import ns_operator_quad
    pb = Problem(dim, order, (3, 2, 1)[:dim], 0.0, (1.0, 0.8, 0.9)[:dim],
                 (False,) * dim)
    kw = {"species_diffusivity": np.linspace(0.01, 0.07, 7)}
    t = None
    if gas == "mixture":
        q, t = mixture_state(pb.x, seed=order)
        kw["species_diffusivity"] = kw["species_diffusivity"] * 1e-3
        kw.update(viscosity=2e-5, thermal_conductivity=0.05)
        eos, oeos = PyrometheusMixture(), tc.PyrometheusMixture()
    else:
        q = smooth_perturbed_state(pb.x, seed=order, nspecies=7, amp=0.1)
        kw.update(viscosity=0.05, thermal_conductivity=0.07, bulk_viscosity=0.01)
        eos, oeos = IdealSingleGas(gas_const=1.0), ph.IdealSingleGas(gas_const=1.0)
    gm = GasModel(eos=eos, transport=SimpleTransport(**kw))
    ogm = ph.GasModel(oeos, ph.SimpleTransport(**kw))
    print(f"quad columns dim={dim} p={order} {gas}", flush=True)

    def dev(a):
        return None if a is None else torch.as_tensor(
            np.ascontiguousarray(a), dtype=torch.float64, device="cuda")
    st = make_fluid_state(ConservedVars(dim, dev(q)), gm, temperature_seed=dev(t))
    rhs, gcv, gt = ns_operator(pb.dcoll, gm, st, {"all": DummyBoundary()},
                               quadrature_tag=DISCR_TAG_QUAD, return_gradients=True)
    okw = {} if t is None else {"temperature": st.temperature.cpu().numpy()}
    ref, rgcv, rgt = ns_operator_quad(pb.odisc, pb.box, q, ogm,
                                      {"all": oop.DummyBoundary()},
                                      return_gradients=True, **okw)
    tol = {3: 2.4e-11, 4: 4.3e-10}.get(order, 1e-11)
    for name, got, want in (
            ("rhs", rhs.q.cpu().numpy(), ref),
            ("grad cv", gcv.q.cpu().numpy().reshape(-1, *ref.shape[1:]),
             rgcv.reshape(-1, *ref.shape[1:])),
            ("grad t", gt.cpu().numpy(), rgt)):
        e = rel_err(got, want)
        print(name, e.max())
        assert (e < tol * (10 if gas == "mixture" and name == "rhs" else 1)).all(), name
