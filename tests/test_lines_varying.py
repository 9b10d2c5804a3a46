"""Line tables where lines are not all alike: rows that vary along x in some of
the planes, columns of two kinds side by side that are put into groups, and the
sweeps that keep T* for a gradient; against the oracle and per-voxel plans."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from heatsim2_amd import _lib, adjoint
from hs2_cases import cases, to_package_args

pytestmark = pytest.mark.gpu

TOL = 1e-10  # max |T_gpu - T_ref| / peak temperature rise, as every parity test


def _body(shape, dt, seed):
    """Steel over a laminate, a stepped source on the layers 0 and 4 in stripes."""
    nz, ny, nx = shape
    m, bz, by, bx, v = cases._zero(nz, ny, nx)
    cases._outer(bz, by, bx, 1)
    m[nz // 2:] = 1
    v[0] = 1
    v[min(4, nz - 1), :, ::3] = 2
    return dict(shape=shape, d=(4e-4, 5e-4, 6e-4), dt=dt, t0=0.0, nsteps=4,
                materials=[(0, 50.0, 50.0, 50.0, 7850.0, 470.0, 0),
                           (0, 5.0, 5.0, 5.0, 1550.0, 1200.0, 0)],
                boundaries=[(cases.BND_CONDUCTING, 0.0), (cases.BND_INSULATING, 0.0),
                            (cases.BND_THIN, 800.0)],
                volumetric=[(0,), (1, 0.0, 1e4 / 4e-4), (2, 0.0, 2.5 * dt, 2e7)],
                maps=(m, bz, by, bx, v), T0=293.0 + np.random.default_rng(seed).random(shape))


def _axes(P):
    a = ctypes.c_int()
    _lib.check("hs2_plan_get_option", _lib.load().hs2_plan_get_option(
        P.plan, _lib.HS2_OPT_LINE_TABLES, ctypes.byref(a)))
    return a.value


def _steps(case, bit):
    """Step by step and in one call on the tables, which the axis has."""
    import heatsim2_amd as hs
    args = to_package_args(hs, case)
    P, S = hs.setup(*args["setup"])
    assert _axes(P) & bit, "no line tables"
    info = (ctypes.c_int * 14)()
    _lib.check("hs2_plan_info", _lib.load().hs2_plan_info(P.plan, info))
    assert bit != 1 or info[13] == 0, "source-free steps are not on them"
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


# rows of 16 lanes x 1..4 cells, 32 x 3..4, 64 x 3..6, 128 x 4, 256 x 3..4
ROWS = [7, 16, 17, 33, 49, 64, 65, 97, 128, 129, 193, 255, 256, 257, 321, 384, 385, 511, 512, 513,
        768, 769, 1023, 1024]


@pytest.mark.parametrize("dt", [1e-3, 5e-2], ids=["weak", "strong"])
@pytest.mark.parametrize("nx", ROWS)
def test_rows_that_vary(nx, dt):
    """Ten planes, two of them with a thin face on parts of their rows (another
    part in each second row), one kind of line."""
    case = _body((10, 5, nx), dt, nx)
    bz = case["maps"][1]
    bz[4, :, nx // 4:3 * nx // 4] = 2
    bz[4, ::2, nx // 2:] = 2
    _steps(case, 1)


@pytest.mark.parametrize("dt", [1e-3, 5e-2], ids=["weak", "strong"])
@pytest.mark.parametrize("L", [5, 20, 32, 33, 50, 64, 65, 80, 200, 255, 256, 300, 512])
@pytest.mark.parametrize("axis", [0, 1], ids=["z", "y"])
def test_columns_of_two_kinds(axis, L, dt):
    """Every other column has a thin face: sixteen of a kind come from a window of
    neighbours (a last one of fewer columns among them)."""
    other = 30 if L <= 128 else 9
    shape = (L, other, 37) if axis == 0 else (other, L, 37)
    case = _body(shape, dt, L + axis)
    if axis == 0:
        case["maps"][1][L // 3, :, ::2] = 2
    else:
        case["maps"][2][:, L // 3, ::2] = 2
    _steps(case, 4 if axis == 0 else 2)


@pytest.mark.parametrize("shape", [(10, 6, 40), (9, 12, 150), (10, 4, 300), (10, 4, 400),
                                   (10, 3, 600), (8, 64, 256)],
                         ids=lambda s: "x".join(map(str, s)))
def test_gradient_on_line_tables(shape):
    """hs2_grad_forward and _backward on class maps, whose recomputation keeps T*
    (the x sweep without y's right-hand side) and takes source fields: history and
    gradients against a per-voxel plan of the same coefficients."""
    import heatsim2_amd as hs
    L = _lib.load()
    steps, every = 7, 3
    case = _body(shape, 2e-3, sum(shape))
    case["maps"][1][4, :, shape[2] // 3:] = 2
    P, _ = hs.setup(*to_package_args(hs, case)["setup"])
    assert _axes(P) & 1
    up = lambda a: torch.from_numpy(a).cuda()
    new = lambda *s: torch.empty(s, dtype=torch.float64, device="cuda")
    f = [new(*shape) for _ in range(5)]
    s = _lib.stream_handle()
    _lib.check("hs2_plan_expand", L.hs2_plan_expand(P.plan, *[_lib.ptr(t) for t in f], s))
    gp = adjoint.GradPlan(shape, case["d"], case["dt"])
    gp.set_coefficients([f[0], f[1].to(torch.uint8)] + f[2:])
    rng = np.random.default_rng(1)
    src = up(1e8 * rng.random((2,) + shape))
    when = (ctypes.c_int32 * 2)(1, 4)
    G = up(rng.random((steps,) + shape[1:]))
    out = []
    for plan in (P.plan, gp.plan):
        T = up(case["T0"])
        ckpt, hist = new(3, *shape), new(steps, *shape[1:])
        _lib.check("hs2_grad_forward", L.hs2_grad_forward(
            plan, _lib.ptr(T), steps, every, _lib.ptr(ckpt), _lib.ptr(src), when, 2,
            _lib.ptr(hist), s))
        work = new(L.hs2_grad_work_doubles(plan, every))
        g = [new(*shape) for _ in range(5)] + [new(2, *shape)]
        _lib.check("hs2_grad_backward", L.hs2_grad_backward(
            plan, steps, every, _lib.ptr(ckpt), _lib.ptr(src), when, 2, _lib.ptr(G),
            *[_lib.ptr(t) for t in g[:4]], _lib.ptr(g[5]), _lib.ptr(g[4]), _lib.ptr(work),
            work.numel(), s))
        torch.cuda.synchronize()
        out.append([T, hist] + g)
    # fields of about 300 and gradients of differences of them: round-off of the
    # fields against the rise, as in the step tests
    for a, b in zip(*out):
        assert float((a - b).abs().max()) <= TOL * float(b.abs().max())
