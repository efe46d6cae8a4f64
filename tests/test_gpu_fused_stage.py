"""The RK stage fused with the viscous divergence, at tile edges (32 x 8
columns) and remainders, over the periodic and closed directions whose
neighbours it reads wrapped and whose ghost layers it writes: state, primitives
and the last right-hand side after a few steps against the CPU oracle.  Bars
as in test_gpu_parity.py (1e-12 of each component's largest value) and
test_gpu_mixed.py (state to 1e-6 relative L2, right-hand side to 1e-4)."""
import numpy as np
import pytest

import oracle as O
from pyocfd import capi, cases

pytestmark = pytest.mark.gpu


def closed_box(size, periodic, vis, scheme="WENO7"):
    case = cases.wavy_box(*size, scheme=scheme, scheme_vis=vis, periodic=periodic)
    for q in range(3):
        if not periodic[q]:
            case.cfg.dif_bound[2 * q] = case.cfg.dif_bound[2 * q + 1] = 1
    return case


# 8: ghost copies to both sides from one tile; 31/33: a partial tile's wrapped
# neighbours; scheme hybrid_auto: the sensor reads the ghosts of the stage before
@pytest.mark.parametrize("size,periodic,vis,scheme", [
    ((8, 8, 8), (1, 1, 1), "CD6", "WENO7"),
    ((33, 9, 12), (1, 1, 1), "CD8", "UP7"),
    ((31, 17, 8), (0, 1, 1), "CD8", "WENO7"),
    ((32, 8, 40), (1, 0, 1), "CD6", "WENO7"),
    ((65, 23, 11), (1, 1, 0), "CD8", "UP7"),
    ((20, 16, 37), (1, 1, 1), "CD6", "SCHEME_HYBRIDAUTO"),
    ((35, 12, 10), (0, 0, 0), "CD8", "WENO5"),
])
def test_steps_and_last_rhs(size, periodic, vis, scheme):
    case = closed_box(size, periodic, vis, scheme)
    ref = case.load(O.Oracle(case.cfg))
    g = case.load(capi.Solver(case.cfg))
    g.step(3)
    ref.step(3)

    def close(a, b):
        for v in range(len(b)):
            assert np.abs(a[v] - b[v]).max() <= 1e-12 * np.abs(b[v]).max(), v

    close(g.get_state(), ref.get_state())
    close(g.get_flow()[0], ref.get_flow()[0])
    du = g.get_du()
    close(du, ref.get_du())
    assert np.array_equal(du, g.get_du())  # asking does not change it
    g.step(1)                              # nor the next step
    ref.step(1)
    close(g.get_state(), ref.get_state())

    cfg = capi.OcfdConfig.from_buffer_copy(case.cfg)
    cfg.precision = capi.PREC_MIXED
    m = case.load(capi.Solver(cfg))
    m.step(4)
    a, b = m.get_state(), ref.get_state()
    for v in range(5):
        assert np.linalg.norm(a[v] - b[v]) <= 1e-6 * np.linalg.norm(b[v]), v
    a, b = m.get_du(), ref.get_du()
    for v in range(5):
        assert np.abs(a[v] - b[v]).max() <= 1e-4 * np.abs(b[v]).max(), v
    assert np.array_equal(a, m.get_du())
