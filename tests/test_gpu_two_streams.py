"""Steps above 500,000 points, where the viscous gradients run on a second
stream beside the sweeps (x and y in one launch, then z) and the fused stage
joins them: replayed from a captured graph, launched one by one, and on one
stream (OCFD_SERIAL=1 at ocfd_create).  The launches are the same and their
order fixes every value, so the states are equal bit for bit after each call of a
sequence that mixes replays (4 and 6 steps), single steps and downloads."""
import numpy as np
import pytest

from pyocfd import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme,prec,periodic", [
    ("WENO7", capi.PREC_FP64, (1, 1, 1)), ("WENO7", capi.PREC_MIXED, (1, 1, 1)),
    ("SCHEME_HYBRIDAUTO", capi.PREC_FP64, (0, 1, 1)), ("UP7", capi.PREC_MIXED, (1, 0, 0))])
def test_replayed_overlapped_and_serial_steps_are_equal(scheme, prec, periodic, monkeypatch):
    case = cases.wavy_box(97, 71, 75, scheme=scheme, periodic=periodic, precision=prec)
    for q in range(6):
        case.cfg.dif_bound[q] = 0 if periodic[q // 2] else 1
    sols = []
    for graph, serial in (("1", "0"), ("0", "0"), ("0", "1")):
        monkeypatch.setenv("OCFD_GRAPH", graph)
        monkeypatch.setenv("OCFD_SERIAL", serial)
        sols.append(case.load(capi.Solver(case.cfg)))
    for n in (4, 1, 6):
        for s in sols:
            s.step(n)
        ref, (prims, istep, tt), du = sols[0].get_state(), sols[0].get_flow(), sols[0].get_du()
        for s in sols[1:]:
            f, i, t = s.get_flow()
            assert (i, t) == (istep, tt)
            assert np.array_equal(s.get_state(), ref)
            assert all(np.array_equal(x, y) for x, y in zip(f, prims))
            assert np.array_equal(s.get_du(), du)
    for s in sols:
        s.close()
