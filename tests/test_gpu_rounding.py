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


def split(prims, A, ma, gamma, real):
    """f+ and f- of the reference's split (src/OCFD_split.cu:92-142), its sums
    as they stand, in the type real; the constants are the FP64 ones."""
    d, u, v, w, T = (a.astype(real) for a in prims)
    A = [a.astype(real) for a in A]
    c = np.sqrt(T) * real(1.0 / ma)
    ss = np.sqrt(A[0] * A[0] + A[1] * A[1] + A[2] * A[2])
    n = [a / ss for a in A]
    E1 = A[0] * u + A[1] * v + A[2] * w
    E = (E1, E1 - c * ss, E1 + c * ss)
    lo, hi = ([x + s * c * m for x, m in zip((u, v, w), n)] for s in (-1, 1))
    klo, khi = ((q[0] * q[0] + q[1] * q[1] + q[2] * q[2]) * real(0.5) for q in (lo, hi))
    vv = real(gamma - 1.0) * (u * u + v * v + w * w)
    c1, W2 = real(2.0 * (gamma - 1.0)), real((3.0 - gamma) / (2.0 * (gamma - 1.0))) * c * c
    out = []
    for s in (1, -1):
        l1, l2, l3 = ((e + s * np.abs(e)) * real(0.5) for e in E)
        f = [c1 * l1 + l2 + l3]
        f += [c1 * l1 * x + l2 * m + l3 * p for x, m, p in zip((u, v, w), lo, hi)]
        f += [l1 * vv + l2 * klo + l3 * khi + W2 * (l2 + l3)]
        out.append(np.stack(f) * (d * real(1.0 / (2.0 * gamma))))
    return out


def nnd2_rhs(case, jac, real):
    """Inviscid right-hand side of a periodic box with NND2, whose few
    operations leave the split's rounding visible."""
    def minmod(a, b):
        return np.where(a * b > 0, np.where(np.abs(a) < np.abs(b), a, b), 0 * a)

    du = 0
    for q, n in enumerate((case.cfg.nx, case.cfg.ny, case.cfg.nz)):
        ax, h = -1 - q, real(1.0 / (n - 1.0))
        fp, fm = split(case.prims, jac[3 + 3 * q:6 + 3 * q], case.cfg.ama, case.cfg.gamma, real)
        ahead = np.roll(fp, -1, ax)
        hp = fp + real(0.5) * minmod(ahead - fp, fp - np.roll(fp, 1, ax))
        a1, a2 = np.roll(fm, -1, ax), np.roll(fm, -2, ax)
        hm = a1 - real(0.5) * minmod(a2 - a1, a1 - fm)
        for x in (hp, hm):
            du = du - (x - np.roll(x, 1, ax)) / h
    return du * jac[12].astype(real)


def test_split_rounds_no_more_than_the_references_sums():
    """Right-hand side of a Mach 0.3 flow, where the waves' parts of a flux
    cancel most: in each component the rms distance from 80-bit arithmetic, over
    three seeds, is no larger than that of the reference's sums in plain FP64."""
    gpu, plain = np.zeros(5), np.zeros(5)
    for seed in (2, 5, 7):
        case = cases.wavy_box(40, 36, 32, ma=0.3, re=1e30, seed=seed, scheme="NND2")
        g = case.load(capi.Solver(case.cfg))
        jac = g.get_metrics()
        g.rhs(1)
        du = g.get_du()
        g.close()
        exact = nnd2_rhs(case, jac, np.longdouble)
        for tot, a in ((gpu, du), (plain, nnd2_rhs(case, jac, np.float64))):
            tot += (((a - exact).astype(np.float64)) ** 2).sum(axis=(1, 2, 3))
    print("[rounding] rms of the GPU over plain FP64, by component:", np.sqrt(gpu / plain))
    assert (gpu <= plain).all()
