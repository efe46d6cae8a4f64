"""Rounding of the FP64 path.  Each bar follows from the roundings that the
arithmetic needs, or is the error of the reference's own sums evaluated in
FP64; nothing here is a measured margin."""
import numpy as np
import pytest

from pyocfd import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ma", [0.5, 2.0, 5.0])
def test_stages_keep_the_conserved_state(ma):
    """With dt = 0 the three stages return the state: stage 2 exactly (a
    quarter of f is exact and its sum is one fused operation), stage 3 to
    2^-54 + 2/3 2^-53 of the value (1/3 and 2/3 in FP64 sum to 1 - 2^-54, one
    product rounds) before the last rounding: at most one ulp.  f formed again from the
    primitives between the stages is two or three ulps off in the energy.
    Faces are left out: there f is formed from the primitives (OCFD_bc)."""
    case = cases.wavy_box(40, 32, 24, ma=ma, scheme="UP7")
    case.cfg.dt = 0.0
    g = case.load(capi.Solver(case.cfg))
    f0 = g.get_state()
    g.step(1)
    f1 = g.get_state()
    inner = np.s_[:, 1:-1, 1:-1, 1:-1]
    assert (np.abs(f1 - f0)[inner] <= np.spacing(np.abs(f0))[inner]).all()
    g.close()


@pytest.mark.parametrize("ma", [0.1, 0.3])
def test_initial_energy(ma):
    """d (|u|^2 / 2 + cv T) at low Mach, where cv T is nearly all of it: one
    fused sum and one product, 2^-53 each, and three roundings of the square
    in the kinetic share.  A product cv T rounded by itself would add a third 2^-53."""
    case = cases.wavy_box(40, 32, 24, ma=ma)
    g = case.load(capi.Solver(case.cfg))
    E = g.get_state()[4]
    g.close()
    d, u, v, w, T = (a.astype(np.longdouble) for a in case.prims)
    gamma = case.cfg.gamma
    cv = np.longdouble(1.0 / (gamma * (gamma - 1.0) * ma * ma))
    kin = d * (u * u + v * v + w * w) / 2
    exact = kin + d * cv * T
    assert (np.abs(E - exact) <= (2 * exact + 3 * kin) * 2.0 ** -53).all()
