"""The three sweeps in one launch (grids up to 500,000 points) and one after
the other (above): right-hand side and state against the CPU oracle at the
sizes where the tilings can go wrong: rows of one and of two segments per wave
(24 and 56 nodes), remainders of the y/z tiles, closures, and grids on either
side of the limit.  Bar: 1e-12 of each component's largest value, as in
test_gpu_parity.py."""
import numpy as np
import pytest

import oracle as O
from pyocfd import capi, cases

pytestmark = pytest.mark.gpu


def close(a, b):
    for v in range(5):
        assert np.abs(a[v] - b[v]).max() <= 1e-12 * np.abs(b[v]).max(), v


# x: one segment exactly, one over, two of 24, 24 over; y/z: 14 exactly, one over
@pytest.mark.parametrize("size", [(24, 14, 14), (25, 15, 8), (48, 28, 15), (56, 13, 29), (57, 9, 16), (112, 12, 9),
                                  (79, 80, 79), (80, 80, 79)])
@pytest.mark.parametrize("scheme", ["WENO7", "SCHEME_HYBRIDAUTO"])
def test_sweep_forms_match_oracle(size, scheme):
    case = cases.wavy_box(*size, scheme=scheme, periodic=(0, 1, 0))
    for q in (0, 1, 4, 5):
        case.cfg.dif_bound[q] = 1
    case.cfg.non_ref[1] = case.cfg.non_ref[5] = 1
    case.cfg.hy_dp_intv[0], case.cfg.hy_dp_intv[1] = 0.005, 0.02
    ref = case.load(O.Oracle(case.cfg))
    g = case.load(capi.Solver(case.cfg))
    g.rhs(1)
    ref.rhs(1)
    close(g.get_du(), ref.get_du())
    g.step(1)
    ref.step(1)
    close(g.get_state(), ref.get_state())
    close(g.get_du(), ref.get_du())
    g.close()


def test_learned_sensor_on_a_small_grid():
    """With the learned sensor in the x sweep the first stage's sweeps run one
    after the other, the later ones in one launch: the same state as with the
    sensor in its own pass, and the last right-hand side after every step."""
    case = cases.wavy_box(30, 16, 15, scheme="SCHEME_HYBRIDAUTO", amp=0.08)
    params = np.load(capi.SENSOR_PARAMS)
    a, b = (case.load(capi.Solver(case.cfg)) for _ in range(2))
    for s, fused in ((a, True), (b, False)):
        s.set_sensor(params, 0.2, 0.8)
        s.set_sensor_fused(fused)
    for _ in range(2):
        a.rhs(1)
        b.rhs(1)
        close(a.get_du(), b.get_du())
        a.step(2)
        b.step(2)
        close(a.get_state(), b.get_state())
        close(a.get_du(), b.get_du())
