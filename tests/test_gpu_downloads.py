"""Downloads in one piece and in several: the values a context returns equal
the ones loaded into it, at sizes below and above the direct and the piecewise
limits (1 MiB and 16 MiB of packed values) and with fields left out."""
import ctypes as C

import numpy as np
import pytest

from pyocfd import capi, cases

pytestmark = pytest.mark.gpu


# 5 FP64 fields: 0.02 MiB; just above 1 MiB; 16.0 MiB +- a row; 2 pieces and a
# remainder; more pieces than slots
@pytest.mark.parametrize("size", [(8, 9, 8), (35, 29, 27), (64, 64, 102), (64, 64, 103), (131, 99, 80), (160, 130, 110)])
@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_MIXED])
def test_flow_comes_back_as_loaded(size, prec):
    nx, ny, nz = size
    rng = np.random.default_rng(1)
    # exactly representable in FP32, so the mixed path returns them unchanged
    prims = [1.0 + rng.integers(0, 1 << 16, (nz, ny, nx)) / float(1 << 20) for _ in range(5)]
    cfg = cases.wavy_box(8, 8, 8).cfg
    cfg.nx, cfg.ny, cfg.nz, cfg.precision = nx, ny, nz, prec
    s = capi.Solver(cfg)
    s.load_flow(*prims, istep=3, tt=0.5)
    got, istep, tt = s.get_flow()
    assert (istep, tt) == (3, 0.5)
    for a, b in zip(got, prims):
        assert np.array_equal(a, b)
    # only u and T
    dp = C.POINTER(C.c_double)
    fn = C.cast(s.lib.ocfd_get_flow, C.c_void_p).value
    get = C.CFUNCTYPE(C.c_int, C.c_void_p, dp, dp, dp, dp, dp, C.POINTER(C.c_int), dp)(fn)
    u, T = np.zeros((nz, ny, nx)), np.zeros((nz, ny, nx))
    as_p = lambda a: a.ctypes.data_as(dp)  # noqa: E731
    assert get(s.h, None, as_p(u), None, None, as_p(T), None, None) == 0
    assert np.array_equal(u, prims[1]) and np.array_equal(T, prims[4])
    s.close()


@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_MIXED])
def test_a_stepping_run_holds_no_viscous_right_hand_side(prec):
    """The four fields of the viscous part of the right-hand side are
    allocated by the first call that wants them in memory, not by a run that
    only steps."""
    case = cases.wavy_box(160, 128, 64, scheme="UP7", precision=prec)
    s = case.load(capi.Solver(case.cfg))
    hip = C.CDLL("libamdhip64.so")

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    s.step(2)  # with what the runtime allocates for the streams
    before = free()
    assert np.isfinite(s.get_du()).all()
    fields = 4 * case.npoints * (8 if prec == capi.PREC_FP64 else 4)
    assert fields <= before - free() <= 2 * fields
    s.close()


@pytest.mark.parametrize("size,scheme,prec", [
    ((8, 9, 8), "UP7", capi.PREC_FP64), ((20, 16, 12), "WENO7", capi.PREC_MIXED),
    ((65, 41, 33), "WENO5", capi.PREC_FP64), ((97, 71, 75), "UP7", capi.PREC_MIXED)])
def test_right_hand_side_in_one_download(size, scheme, prec):
    """The parts of the right-hand side are added on the GPU and fetched at
    once, after ocfd_rhs and after a step, in one launch beside the divergence
    that a step leaves out."""
    case = cases.wavy_box(*size, scheme=scheme, precision=prec)
    s = case.load(capi.Solver(case.cfg))
    s.rhs(1)
    a = s.get_du()
    s.profile(True)
    s.step(1)
    s.profile_reset()
    b = s.get_du()
    assert np.array_equal(b, s.get_du())
    s.step(1)
    launches = s.profile_entries()
    s.profile(False)
    assert launches["pack"][0] == 2 and launches["visc_div"][0] == 1
    # the step moved the state by 1e-3 of it or less, and du with it
    for v in range(5):
        assert np.linalg.norm(a[v] - b[v]) <= 0.1 * np.linalg.norm(a[v])
    s.close()


# padded fields of 32 and 126 KiB, fetched as they are, and of 133 KiB, packed
@pytest.mark.parametrize("size,packed", [((8, 8, 8), 0), ((23, 20, 10), 0), ((24, 20, 11), 1)])
def test_single_small_field_without_a_launch(size, packed):
    """A single small FP64 field comes over without a launch of its own, with
    the same values as with others."""
    case = cases.wavy_box(*size, scheme="UP7")
    s = case.load(capi.Solver(case.cfg))
    s.step(2)
    p = s.get_pressure()
    d, _, _, _, T = s.get_flow()[0]
    c = case.cfg
    assert np.abs(p - d * T / (c.gamma * c.ama ** 2)).max() <= 4 * 2.0 ** -52 * p.max()
    s.profile(True)
    s.profile_reset()
    s.get_pressure()
    s.step(1)
    assert s.profile_entries().get("pack", (0, 0.0))[0] == packed
    s.close()
