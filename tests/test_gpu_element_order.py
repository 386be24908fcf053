"""An element's result does not depend on which elements share its wave or
workgroup: the temperatures and the overintegrated and entropy-stable
right-hand sides of a mesh and of the same mesh with its elements in another
order are bit-equal, element by element, and so are two calls with another
state's call between them.  An odd number of elements (one removed from a box,
its faces left as boundaries) leaves lanes of the last workgroup without an
element.  The states vary by a percent inside most elements (the limit of the
logarithmic means' short series), with a steep bump; mixtures cross the NASA7
switch at 1000 K inside elements, between elements of one workgroup and nowhere
near others."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore")]


def bump_state(x, gas):
    """Conserved variables (and a mixture's temperature) on nodes ``x``."""
    from mirgecom_amd import mechanisms as mech
    from oracle import thermochem as tc
    dim = x.shape[0]
    r2 = sum((xd - 0.4)**2 for xd in x)
    bump = np.exp(-20.0 * r2)
    wave = np.cos(3 * x[0] + 2 * x[1])
    vel = [1.0 + 0.1 * wave, 0.5 + 0.2 * bump, 0.2 * wave][:dim]
    if gas == "mixture":
        t = 900.0 - 650.0 * bump + 3.0 * wave
        y = np.stack([a * (1 + 0.1 * wave) for a in
                      (0.1, 0.2, 2e-4, 2e-4, 2e-4, 1e-4)])
        y = np.concatenate([y, 1.0 - y.sum(0, keepdims=True)])
        rho = tc.density(mech.ONE_ATM * (1 + 0.01 * wave), t, y)
        energy = rho * (tc.mixture_energy_mass(t, y) + 0.5 * sum(v * v for v in vel))
        return np.stack([rho, energy] + [rho * v for v in vel]
                        + [rho * yk for yk in y]), t * (1 + 2e-3 * wave)
    rho = 1.0 + 2.0 * bump + 0.02 * wave
    energy = (1.0 + bump + 0.02 * wave) / 0.4 + 0.5 * rho * sum(v * v for v in vel)
    rows = [rho, energy] + [rho * v for v in vel]
    if gas == "species":
        rows += [rho * (0.1 + 0.01 * k * wave) for k in range(7)]
    return np.stack(rows), None


def _meshes(monkeypatch, dim, order, degree):
    """A box without one element, and the same with its elements shuffled."""
    from dataclasses import replace

    from mirgecom_amd import discretization as disc
    monkeypatch.setattr(disc, "_boundary_tag", lambda mesh, centroid: "+1")
    box = disc.generate_box_mesh(dim, 0.0, 1.0, (9, 8) if dim == 2 else (4, 3, 3))
    keep = np.arange(1, box.nelements)
    perm = np.random.default_rng(7).permutation(keep.size)
    return perm, [disc.create_discretization_collection(
        replace(box, elements=box.elements[keep[p]]), order, quadrature_order=degree)
        for p in (np.arange(keep.size), perm)]


@pytest.mark.parametrize("degree", [-1, 7])
@pytest.mark.parametrize("gas", ["ideal", "species", "mixture"])
@pytest.mark.parametrize("dim,order", [(2, 1), (2, 3), (3, 1), (3, 2), (3, 3)])
@pytest.mark.parametrize("path", ["temperature", "esdg", "ns_quad"])
def test_order_of_elements(monkeypatch, path, dim, order, gas, degree):
    from mirgecom_amd.boundary import DummyBoundary
    from mirgecom_amd.dof_desc import DISCR_TAG_QUAD
    from mirgecom_amd.eos import IdealSingleGas, PyrometheusMixture
    from mirgecom_amd.euler import euler_operator
    from mirgecom_amd.fluid import ConservedVars
    from mirgecom_amd.gas_model import GasModel, make_fluid_state
    from mirgecom_amd.navierstokes import ns_operator
    from mirgecom_amd.transport import SimpleTransport
    if path == "temperature" and (degree > 0 or gas != "mixture"):
        pytest.skip("mixtures' temperatures, nodal")
    if path == "esdg" and degree > 0 and order == 3 and dim == 3:
        pytest.skip("too many points for LDS")
    print(f"element order: {path} {dim}-D p={order} {gas} degree={degree}", flush=True)
    gm = GasModel(
        eos=PyrometheusMixture() if gas == "mixture" else IdealSingleGas(gas_const=1.0),
        transport=SimpleTransport(viscosity=1e-3, thermal_conductivity=2e-3,
                                  species_diffusivity=None if gas == "ideal"
                                  else (1e-3,) * 7))
    bnd = {"all": DummyBoundary()}
    perm, dcolls = _meshes(monkeypatch, dim, order, degree)

    def rhs(dcoll, scale=1.0):
        q, t = bump_state(dcoll.host_nodes, gas)
        q[1] *= scale
        st = make_fluid_state(
            ConservedVars(dim, torch.as_tensor(q, device="cuda")), gm,
            temperature_seed=None if t is None else torch.as_tensor(t, device="cuda"))
        if path == "temperature":
            return st.temperature[None].cpu()
        if path == "ns_quad":
            out = ns_operator(dcoll, gm, st, bnd, quadrature_tag=DISCR_TAG_QUAD)
        else:
            out = euler_operator(dcoll, st, gm, bnd, use_esdg=True,
                                 quadrature_tag=DISCR_TAG_QUAD)
        return out.q.cpu()

    ref = rhs(dcolls[0])
    assert torch.isfinite(ref).all()
    moved = rhs(dcolls[1])
    different = (moved != ref[:, torch.as_tensor(perm)]).any(2).any(0)
    print("elements that differ:", int(different.sum()), "of", perm.size)
    assert not different.any()
    rhs(dcolls[0], 1.3)
    assert torch.equal(rhs(dcolls[0]), ref)
