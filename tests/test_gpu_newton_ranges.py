"""The mixture temperature's Newton solve where its route through the NASA7
ranges changes: waves whose nodes all lie in one range (the species summed
into that range's polynomials once), waves across the switch, and updates that
move a wave from one to the other -- against the oracle's fixed-iteration
solve.  An update divides an energy difference by c_v: the round-off of the
energy (terms of ~1e7 J/kg, formation enthalpies included, eps 1e-16) over
c_v ~ 1e3 J/kg/K is 1e-12 K, 1e-15 of T; 1e-13 as for the other solves."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests.cases import mixture_state  # noqa: E402

pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


@pytest.mark.parametrize("niter", [0, 1, 2, 5])
@pytest.mark.parametrize("t_mean,t_amp,seed", [
    (1000.0, 400.0, 1.05),    # waves across the switch
    (700.0, 100.0, 1.6),      # all start above it and fall below
    (1500.0, 100.0, 0.6),     # all start below it and rise above
    (500.0, 100.0, 1.0), (2000.0, 300.0, 0.95)])
def test_newton_across_ranges(niter, t_mean, t_amp, seed):
    from mirgecom_amd.eos import PyrometheusMixture
    from mirgecom_amd.fluid import ConservedVars
    from oracle import thermochem as tc
    print(f"newton ranges niter={niter} T={t_mean}+-{t_amp} seed {seed} T", flush=True)
    x = np.random.default_rng(3).uniform(0, 2 * np.pi, size=(3, 1000 + 37))
    q, t = mixture_state(x, 11, t_mean=t_mean, t_amp=t_amp)
    got = PyrometheusMixture(temperature_niter=niter).temperature(
        ConservedVars(3, _dev(q)), _dev(seed * t)).cpu().numpy()
    ref = tc.PyrometheusMixture(niter).temperature(q, 3, seed * t)
    err = np.abs(got - ref).max() / np.abs(ref).max()
    print("err", err)
    assert err < 1e-13


def test_species_with_different_switch_temperatures():
    """A mechanism whose species switch ranges at temperatures of their own:
    nodes between them take each species' own range in every update."""
    from mirgecom_amd import _lib
    from mirgecom_amd import mechanisms as mech
    from mirgecom_amd.eos import PyrometheusMixture
    from mirgecom_amd.fluid import ConservedVars
    lo, hi = mech.nasa7_tables()
    tmid = 1000.0 + 60.0 * np.arange(-3, 4)
    inv_wt = 1.0 / mech.molecular_weights()

    def e_cv(t, y):
        a = np.where((t > tmid[:, None])[..., None], hi[:, None], lo[:, None])
        cp = sum(a[..., i] * t**i for i in range(5))
        h = sum(a[..., i] * t**i / (i + 1) for i in range(5)) + a[..., 5] / t
        w = mech.GAS_CONSTANT * inv_wt[:, None] * y
        return t * (w * (h - 1)).sum(0), (w * (cp - 1)).sum(0)

    rng = np.random.default_rng(5)
    n = 1000 + 37
    t = rng.uniform(700.0, 1300.0, n)
    y = rng.uniform(0.05, 1.0, (7, n))
    y /= y.sum(0)
    rho = rng.uniform(0.1, 0.5, n)
    q = np.concatenate([[rho, rho * e_cv(t, y)[0]], np.zeros((3, n)), rho * y])
    seed = t * rng.uniform(0.95, 1.05, n)
    packed = mech.packed_mechanism()
    own = packed.copy()
    own[98:105] = tmid
    _lib.ensure_mechanism()

    def load(arr):
        _lib.check(_lib.load().mg_load_mechanism(
            arr.ctypes.data_as(_lib.ctypes.POINTER(_lib.ctypes.c_double)), arr.size))
    load(own)
    try:
        for niter in (1, 3):
            got = PyrometheusMixture(temperature_niter=niter).temperature(
                ConservedVars(3, _dev(q)), _dev(seed)).cpu().numpy()
            ref = seed
            for _ in range(niter):
                e, cv = e_cv(ref, y)
                ref = ref + (q[1] / rho - e) / cv
            assert np.abs(got - ref).max() / ref.max() < 1e-13
    finally:
        load(packed)
