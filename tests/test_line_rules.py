"""When the x sweep of a step without sources runs on line tables: rows that vary
along x, and rows of more than 512 cells, which the class-map kernel sweeps
faster from some number on.  Sources' steps stay on the tables."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from heatsim2_amd import _lib
from hs2_cases import cases, to_package_args

pytestmark = pytest.mark.gpu

TOL = 1e-10  # max |T_gpu - T_ref| / peak temperature rise, as every parity test


def _body(shape, planes, distinct=False, seed=0):
    """One material; thin z faces on `planes`, in the middle half of every row or
    at random (each row another one); a stepped source on the top layer."""
    rng = np.random.default_rng(seed)
    nz, ny, nx = shape
    m, bz, by, bx, v = cases._zero(nz, ny, nx)
    cases._outer(bz, by, bx, 1)
    for k in planes:
        if distinct:
            bz[k][rng.random((ny, nx)) < 0.3] = 2
        else:
            bz[k, :, nx // 4:3 * nx // 4] = 2
    v[0] = 1
    dt = 2e-3
    return dict(shape=shape, d=(4e-4, 5e-4, 6e-4), dt=dt, t0=0.0, nsteps=4,
                materials=[(0, 5.0, 5.0, 5.0, 1550.0, 1200.0, 0)],
                boundaries=[(cases.BND_CONDUCTING, 0.0), (cases.BND_INSULATING, 0.0),
                            (cases.BND_THIN, 800.0)],
                volumetric=[(0,), (2, 0.0, 1.5 * dt, 2e7)], maps=(m, bz, by, bx, v),
                T0=293.0 + rng.random(shape))


def _state(P):
    a = ctypes.c_int()
    _lib.check("hs2_plan_get_option", _lib.load().hs2_plan_get_option(
        P.plan, _lib.HS2_OPT_LINE_TABLES, ctypes.byref(a)))
    info = (ctypes.c_int * 14)()
    _lib.check("hs2_plan_info", _lib.load().hs2_plan_info(P.plan, info))
    return a.value & 1, info[12], info[13] > 0  # x on tables; y from x; source-free x on classes


# shape, thin planes, all rows different; x on tables, on classes without sources
RULES = [((8, 64, 1024), (3,), False, 1, True),      # 512 rows, a quarter vary
         ((8, 48, 1024), (3,), False, 1, False),     # 384 rows
         ((8, 64, 1024), (), False, 1, False),       # none vary
         ((64, 24, 256), range(2, 62, 6), True, 1, True),    # 480 rows of 12 KB each
         ((64, 24, 256), range(2, 62, 6), False, 1, False),  # the same rows alike
         ((12, 20, 256), (3, 7), True, 1, False),    # 80 of 240 rows: a third
         ((12, 20, 256), (3, 7, 10), False, 1, False),       # half, but no whole tiles
         ((24, 20, 256), (3, 7, 10, 15), True, 1, False),    # whole tiles, a third
         ((24, 20, 256), (3, 7, 10, 15, 19), False, 1, True),
         ((10, 24, 250), (3, 7), True, 1, False),    # no whole lines: tables
         ((10, 24, 600), (4,), False, 1, False),     # a fifth vary
         ((10, 24, 600), (3, 7), False, 0, False)]   # two fifths


@pytest.mark.parametrize("shape,planes,distinct,tables,classes", RULES,
                         ids=["%dx%dx%d-%d%s" % (r[0] + (len(r[1]), "d" if r[2] else "")) for r in RULES])
def test_rows(shape, planes, distinct, tables, classes):
    """The route, and steps with a source and without against the oracle, one by
    one and in one call (the same bits)."""
    import heatsim2_amd as hs
    case = _body(shape, planes, distinct, sum(shape))
    args = to_package_args(hs, case)
    P, S = hs.setup(*args["setup"])
    x, ry, on_classes = _state(P)
    assert (x, on_classes) == (tables, classes)
    assert ry == 1 or not tables
    ref = oracle.run_ref(case)
    rise = max(np.abs(np.array(ref) - case["T0"]).max(), 1e-300)
    T = torch.from_numpy(case["T0"]).cuda()
    for n in range(case["nsteps"]):
        T = hs.run_adi_steps(P, S, n * case["dt"], case["dt"], T, args["vmap"], args["volumetric"])
        assert np.abs(T.cpu().numpy() - ref[n]).max() / rise < TOL, n
    R, _ = hs.run_adi_steps_many(P, 0.0, case["dt"], case["nsteps"],
                                 torch.from_numpy(case["T0"]).cuda(), args["vmap"],
                                 args["volumetric"])
    assert torch.equal(R, T)


def test_many_long_rows():
    """Rows of 1024 cells, 21000 of them: source-free steps on the classes."""
    import heatsim2_amd as hs
    case = _body((21, 1000, 1024), ())
    P, _ = hs.setup(*to_package_args(hs, case)["setup"])
    assert _state(P) == (1, 1, True)
