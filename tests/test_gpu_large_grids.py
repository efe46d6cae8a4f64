"""The kernels of grids above 500,000 points that only some schemes and options
reach, against the CPU oracle: each scheme's tile sweeps (x and y, then z), the
fused stage with one du on both paths, the learned sensor in the x sweep, and an
x sweep of two row segments per wave by itself.  Bars: 1e-12 of each component's
largest value in FP64 (test_gpu_parity.py); mixed 1e-4 at 20 nodes times the
number of nodes over 20 for the right-hand side (test_gpu_tile_sweeps.py) and
1e-6 relative L2 for the state (test_gpu_mixed.py)."""
import numpy as np
import pytest

import oracle as O
from pyocfd import capi, cases

pytestmark = pytest.mark.gpu

SIZE = (97, 71, 75)


def close(a, b, bar=1e-12):
    for v in range(5):
        assert np.abs(a[v] - b[v]).max() <= bar * np.abs(b[v]).max(), v


def pair(case, prec):
    ref = case.load(O.Oracle(case.cfg))
    cfg = capi.OcfdConfig.from_buffer_copy(case.cfg)
    cfg.precision = prec
    return ref, case.load(capi.Solver(cfg))


@pytest.mark.parametrize("scheme", ["WENO7_SYMBO", "WENO7_SYMBO_LIM", "NND2", "OMP6_HR", "OMP6_LD", "OMP6_CD8"])
def test_right_hand_side_and_step_of_each_scheme(scheme):
    case = cases.wavy_box(*SIZE, scheme=scheme, periodic=(0, 0, 1))
    for q in range(4):
        case.cfg.dif_bound[q] = 1
    case.cfg.non_ref[1] = case.cfg.non_ref[2] = 1
    ref, g = pair(case, capi.PREC_FP64)
    g.rhs(1)
    ref.rhs(1)
    close(g.get_du(), ref.get_du())
    g.step(1)
    ref.step(1)
    close(g.get_state(), ref.get_state())
    close(g.get_du(), ref.get_du())
    g.close()


@pytest.mark.parametrize("scheme,periodic", [("WENO5", (0, 0, 1)), ("WENO7_SYMBO", (1, 1, 1)), ("NND2", (1, 1, 1))])
def test_mixed_right_hand_side_and_steps(scheme, periodic):
    case = cases.wavy_box(*SIZE, scheme=scheme, periodic=periodic)
    for q in range(6):
        case.cfg.dif_bound[q] = 0 if periodic[q // 2] else 1
    ref, g = pair(case, capi.PREC_MIXED)
    g.rhs(1)
    ref.rhs(1)
    close(g.get_du(), ref.get_du(), 1e-4 * max(SIZE) / 20)
    g.step(2)
    ref.step(2)
    a, b = g.get_state(), ref.get_state()
    for v in range(5):
        assert np.linalg.norm(a[v] - b[v]) <= 1e-6 * np.linalg.norm(b[v]), v
    g.close()


@pytest.mark.parametrize("scheme,vis,periodic", [("UP7", "CD8", (1, 1, 1)), ("WENO7", "CD6", (0, 1, 0))])
def test_steps_with_one_du(scheme, vis, periodic):
    case = cases.wavy_box(*SIZE, scheme=scheme, scheme_vis=vis, periodic=periodic)
    for q in range(6):
        case.cfg.dif_bound[q] = 0 if periodic[q // 2] else 1
    ref, g = pair(case, capi.PREC_FP64)
    g.step(2)
    ref.step(2)
    close(g.get_state(), ref.get_state())
    close(g.get_flow()[0], ref.get_flow()[0])
    close(g.get_du(), ref.get_du())
    g.close()


def test_x_sweep_of_two_segments_by_itself():
    # hybrid_auto in FP64 keeps x and y apart here; 64 nodes are 3 x 24
    case = cases.wavy_box(64, 150, 160, scheme="SCHEME_HYBRIDAUTO", periodic=(0, 1, 0))
    for q in (0, 1, 4, 5):
        case.cfg.dif_bound[q] = 1
    case.cfg.hy_dp_intv[0], case.cfg.hy_dp_intv[1] = 0.005, 0.02
    ref, g = pair(case, capi.PREC_FP64)
    g.rhs(1)
    ref.rhs(1)
    close(g.get_du(), ref.get_du())
    g.close()


@pytest.mark.parametrize("size", [SIZE, (129, 113, 104)])
def test_learned_sensor_in_the_x_sweep(size):
    """Beside x and y in one launch and apart: the same state as with the
    sensor in its own pass."""
    case = cases.wavy_box(*size, scheme="SCHEME_HYBRIDAUTO", amp=0.02)
    params = np.load(capi.SENSOR_PARAMS)
    a, b = (case.load(capi.Solver(case.cfg)) for _ in range(2))
    for s, fused in ((a, True), (b, False)):
        s.set_sensor(params, 0.2, 0.8)
        s.set_sensor_fused(fused)
        s.rhs(1)
    close(a.get_du(), b.get_du())
    for x, y in zip(a.get_flags(), b.get_flags()):
        assert np.array_equal(x, y)
    a.step(2)
    b.step(2)
    close(a.get_state(), b.get_state())
    a.close()
    b.close()
