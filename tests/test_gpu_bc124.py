"""IBC 124 and the face refresh in one launch, on grids whose planes lie as
close as they may (8 nodes) and on ragged ones, free-stream and tabulated upper
face, isothermal and adiabatic wall: state against the CPU oracle, 1e-12 of each
component's largest value over the steps (test_gpu_parity.py)."""
import numpy as np
import pytest

import oracle as O
from pyocfd import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(8, 8, 8), (33, 9, 8), (16, 17, 11)])
@pytest.mark.parametrize("kw", [{}, {"mzmax": 3, "tw": -1.0, "upper": 1, "withleading": 1}], ids=["free", "upper-adiabatic"])
def test_planes_in_one_launch(size, kw):
    case = cases.liftbody(*size, nsteps=3, **kw)
    ref = case.load(O.Oracle(case.cfg))
    g = case.load(capi.Solver(case.cfg))
    g.step(3)
    ref.step(3)
    a, b = g.get_state(), ref.get_state()
    for v in range(5):
        assert np.abs(a[v] - b[v]).max() <= 1e-12 * np.abs(b[v]).max(), v
    g.close()
