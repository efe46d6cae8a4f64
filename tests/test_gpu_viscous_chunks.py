"""The z chunks of the viscous kernels follow the grid (one plane per block on
the smallest, the fixed chunk on the largest): the right-hand side at sizes on
either side of the rule, remainders included, against the CPU oracle.  Bar:
1e-12 of each component's largest value, as in test_gpu_parity.py."""
import numpy as np
import pytest

import oracle as O
from pyocfd import capi, cases

pytestmark = pytest.mark.gpu


# one plane a block, two, a chunk with a remainder, the largest chunk short of
# the fixed one; few columns and many
@pytest.mark.parametrize("size", [(8, 8, 8), (40, 24, 33), (33, 17, 70), (260, 136, 19), (352, 184, 9)])
@pytest.mark.parametrize("vis", ["CD6", "CD8"])
def test_rhs_over_chunk_sizes(size, vis):
    case = cases.wavy_box(*size, scheme="UP7", scheme_vis=vis)
    ref = case.load(O.Oracle(case.cfg))
    g = case.load(capi.Solver(case.cfg))
    g.rhs(1)
    ref.rhs(1)
    a, b = g.get_du(), ref.get_du()
    for v in range(5):
        assert np.abs(a[v] - b[v]).max() <= 1e-12 * np.abs(b[v]).max(), v
