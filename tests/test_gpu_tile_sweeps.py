"""The x and y sweeps of larger grids in one launch, tile by tile: right-hand
side against the CPU oracle with whole and ragged tiles (16 x 14 in FP64, 16 x
15 mixed) and closures, and hybrid_auto on either side of the limits between
which x and y run apart.  Bars: 1e-12 of each component's largest value in
FP64 (test_gpu_parity.py); mixed 1e-4 at 20 nodes (test_gpu_mixed.py) times the
number of nodes over 20, since the FP32 rounding of a face value is divided by
the spacing."""
import numpy as np
import pytest

import oracle as O
from pyocfd import capi, cases

pytestmark = pytest.mark.gpu


# above 500,000 points: one over a tile in x, y and z; whole tiles; hybrid apart
@pytest.mark.parametrize("size,scheme,mixed", [
    ((97, 71, 75), "UP7", False), ((96, 70, 77), "WENO5", False), ((97, 71, 75), "SCHEME_HYBRIDAUTO", False),
    ((129, 113, 104), "SCHEME_HYBRIDAUTO", False), ((97, 76, 74), "WENO7", True), ((96, 75, 75), "UP7", True)])
def test_x_and_y_in_one_launch(size, scheme, mixed):
    case = cases.wavy_box(*size, scheme=scheme, periodic=(0, 0, 1))
    for q in range(4):
        case.cfg.dif_bound[q] = 1
    case.cfg.non_ref[1] = case.cfg.non_ref[2] = 1
    case.cfg.hy_dp_intv[0], case.cfg.hy_dp_intv[1] = 0.005, 0.02
    ref = case.load(O.Oracle(case.cfg))
    cfg = capi.OcfdConfig.from_buffer_copy(case.cfg)
    cfg.precision = capi.PREC_MIXED if mixed else capi.PREC_FP64
    g = case.load(capi.Solver(cfg))
    g.rhs(1)
    ref.rhs(1)
    a, b = g.get_du(), ref.get_du()
    bar = 1e-4 * max(size) / 20 if mixed else 1e-12
    for v in range(5):
        assert np.abs(a[v] - b[v]).max() <= bar * np.abs(b[v]).max(), v
    g.close()
