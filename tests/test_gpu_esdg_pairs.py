"""The paired entropy-stable kernels (3-D, the default quadrature and the
64-point rules: each two-point flux once, for both rows) against the row-by-row
kernels, which run when ``mg_esdg`` carries no diagonal layouts: p = 1..3 on
element counts that leave the last workgroup ragged, both gases, smooth and far
states -- densities up to a factor of four apart inside an element (the
logarithmic means' long series and logarithms), projected temperatures across
the NASA7 switch (elements without one range for all points, beside others with
one) -- and dummy boundaries.

Both orders of summation agree to the states' own rounding: fluxes p/rho ~ 1
(ideal) or ~1e5 J/m^3 (mixture) enter a difference of ~1e2 terms with
round-off 1e-16 each, and cancel by up to 1e2 in a field's right-hand side:
1e-12 to 1e-11."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mirgecom_amd.discretization import create_discretization_collection  # noqa: E402
from tests.cases import Problem, mixture_state, rel_err, smooth_perturbed_state  # noqa: E402
from tests.test_gpu_element_order import bump_state  # noqa: E402

pytestmark = pytest.mark.gpu


def _both(pb, q, t, bnd):
    from mirgecom_amd.device import get_device_discretization
    from mirgecom_amd.dof_desc import DISCR_TAG_QUAD
    from mirgecom_amd.eos import IdealSingleGas, PyrometheusMixture
    from mirgecom_amd.euler import euler_operator
    from mirgecom_amd.fluid import ConservedVars
    from mirgecom_amd.gas_model import GasModel, make_fluid_state
    gm = GasModel(eos=IdealSingleGas(gamma=1.4, gas_const=1.0) if t is None
                  else PyrometheusMixture())

    def dev(a):
        return torch.as_tensor(np.ascontiguousarray(a), device="cuda")
    st = make_fluid_state(ConservedVars(3, dev(q)), gm,
                          temperature_seed=None if t is None else dev(t))
    ops = get_device_discretization(pb.dcoll).esdg_ops()

    def run():
        return euler_operator(pb.dcoll, st, gm, bnd, use_esdg=True,
                              quadrature_tag=DISCR_TAG_QUAD).q.cpu().numpy()
    paired = run()
    diag = ops.skew_diag, ops.ext_diag
    ops.skew_diag = ops.ext_diag = None
    try:
        rows = run()
    finally:
        ops.skew_diag, ops.ext_diag = diag
    return paired, rows


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("order,degree", [(1, 2), (2, 4), (3, 6), (1, 6), (2, 6), (2, 7)])
@pytest.mark.parametrize("gas,far", [("ideal", False), ("ideal", True),
                                     ("species", True), ("mixture", False),
                                     ("mixture", True), ("switch", True)])
def test_paired_matches_rows(order, degree, gas, far):
    if degree > 2 * order and gas in ("mixture", "switch"):
        pytest.skip("mixtures: the default rule only")
    print(f"paired esdg p={order} degree={degree} {gas} far={far}", flush=True)
    box = 1.0 if gas == "switch" else (2.0, 2.1, 1.9)
    pb = Problem(3, order, (3, 5, 3), 0.0, box, (True,) * 3)
    t = None
    if gas == "switch":
        # the entropy-stable projection's temperatures lie several hundred
        # kelvin above the state's (no formation energy in p / (gamma - 1))
        from oracle import esdg, physics as ph, thermochem as tc
        q, t = bump_state(pb.x, "mixture")
        tp = esdg._es_projected_state(q, t, ph.GasModel(tc.PyrometheusMixture(5)),
                                      3).temperature
        cross = (tp.min(1) < 950.0) & (tp.max(1) > 1050.0)
        assert cross.any() and (tp.min(1) > 1050.0).any()
    elif gas == "mixture":
        q, t = mixture_state(pb.x, 5, t_mean=1100.0 if far else 1700.0,
                             t_amp=600.0 if far else 200.0)
    else:
        q = smooth_perturbed_state(pb.x, 5, amp=0.6 if far else 0.05,
                                   nspecies=7 if gas == "species" else 0)
    if degree > 2 * order:
        pb.dcoll = create_discretization_collection(pb.mesh, order,
                                                    quadrature_order=degree)
    paired, rows = _both(pb, q, t, {})
    assert np.isfinite(rows).all()
    assert (paired != rows).any()   # two kernels
    err = rel_err(paired, rows)
    print("err", err)
    assert err.max() < 1e-11


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("gas", ["ideal", "mixture"])
def test_paired_matches_rows_on_boundaries(gas):
    from mirgecom_amd.boundary import DummyBoundary
    pb = Problem(3, 2, (3, 1, 1), 0.0, 1.0, (False,) * 3)
    t = None
    if gas == "mixture":
        q, t = mixture_state(pb.x, 6)
    else:
        q = smooth_perturbed_state(pb.x, 6, amp=0.2)
    paired, rows = _both(pb, q, t, {"all": DummyBoundary()})
    err = rel_err(paired, rows)
    print("err", err)
    assert err.max() < 1e-11
