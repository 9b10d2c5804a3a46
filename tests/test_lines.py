"""Line tables (HS2_OPT_LINE_TABLES): the sweeps that read factors computed
once per distinct line, against the oracle and against the class-map kernels,
at the edges of their lane and segment shapes."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from heatsim2_amd import _lib
from hs2_cases import cases, to_package_args

pytestmark = pytest.mark.gpu

TOL = 1e-10  # max |T_gpu - T_ref| / peak temperature rise, as every parity test

# rows: 16 lanes x 1..4 cells, 32 x 3..4, 64 x 3..6, 128 x 4, 256 x 3..4;
# columns: segments of 4, 8 and 16 cells, one to 32 of them, whole and cut
SHAPES = [(1, 1, 1), (2, 3, 16), (5, 7, 17), (9, 4, 49), (3, 33, 64), (33, 2, 65), (4, 5, 97),
          (6, 32, 128), (64, 3, 129), (2, 65, 193), (7, 6, 256), (3, 4, 257), (2, 9, 321),
          (4, 3, 385), (3, 5, 512), (2, 3, 513), (2, 2, 769), (2, 3, 1024), (40, 24, 40),
          (256, 3, 5), (3, 300, 18), (512, 2, 3), (2, 512, 19), (17, 129, 21)]


def _case(shape, seed, dt):
    """Two materials in layers, a block of a third and a FIXED corner, thin z,
    y and x faces in patches, a flash and a stepped source: few distinct
    lines, several of them side by side, rows that vary along x."""
    rng = np.random.default_rng(seed)
    nz, ny, nx = shape
    m, bz, by, bx, v = cases._zero(nz, ny, nx)
    cases._outer(bz, by, bx, 1)
    m[nz // 2:] = 1
    m[nz // 3:nz // 3 + 2, ny // 2:, :nx // 3] = 2
    if nx * ny > 16:
        m[-1, :max(1, ny // 4), :max(1, nx // 5)] = 3
    if nz > 1:
        bz[nz // 2, :(ny + 1) // 2, nx // 3:2 * nx // 3 + 1] = 2
    if ny > 2:
        by[:nz // 2 + 1, ny // 2, nx // 4:] = 2
    if nx > 2:
        bx[nz // 2:, :, nx // 2] = 2
    v[0] = 1
    v[nz // 2, :, ::2] = 2
    materials = [(0, 50.0, 50.0, 50.0, 7850.0, 470.0, 0), (0, 0.4, 0.4, 0.4, 1200.0, 1300.0, 0),
                 (0, 5.0, 5.0, 5.0, 1550.0, 1200.0, 0), (1, 0, 0, 0, 0, 0, 0)]
    boundaries = [(cases.BND_CONDUCTING, 0.0), (cases.BND_INSULATING, 0.0),
                  (cases.BND_THIN, 800.0)]
    d = (4e-4, 5e-4, 6e-4)
    volumetric = [(0,), (1, 0.0, 1e4 / d[0]), (2, 0.0, 2.5 * dt, 2e7)]
    T0 = 293.0 + rng.random(shape)
    T0[m == 3] = 290.0
    return dict(shape=shape, d=d, dt=dt, t0=0.0, nsteps=5, materials=materials,
                boundaries=boundaries, volumetric=volumetric, maps=(m, bz, by, bx, v), T0=T0)


def _layers(shape, seed, dt):
    """The same without what varies along x: every axis has line tables."""
    case = _case(shape, seed, dt)
    m, bz, by, bx, v = case["maps"]
    nz, ny, nx = shape
    m[:] = 0
    m[nz // 2:] = 1
    case["T0"] = 293.0 + np.random.default_rng(seed).random(shape)
    for f in (bz, by, bx):
        f[:] = 0
    cases._outer(bz, by, bx, 1)
    if nz > 1:
        bz[nz // 2] = 2
    if ny > 2:
        by[:, ny // 2] = 2
    return case


def _axes(P):
    a = ctypes.c_int()
    _lib.check("hs2_plan_get_option", _lib.load().hs2_plan_get_option(
        P.plan, _lib.HS2_OPT_LINE_TABLES, ctypes.byref(a)))
    return a.value


@pytest.mark.parametrize("dt", [1e-3, 5e-2], ids=["weak", "strong"])
@pytest.mark.parametrize("body", [_case, _layers], ids=["patches", "layers"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_line_tables_match_oracle_and_class_kernels(shape, body, dt):
    """Steps with both sources, with one and with none, weakly coupled lines
    (a few scan steps, neighbouring segments) and strongly coupled ones (all
    of them)."""
    import heatsim2_amd as hs
    case = body(shape, 3 + sum(shape), dt)
    args = to_package_args(hs, case)
    P, S = hs.setup(*args["setup"])
    on = _axes(P)
    assert body is _case or on == 7
    ref = oracle.run_ref(case)
    rise = max(np.abs(np.array(ref) - case["T0"]).max(), 1e-300)
    L = _lib.load()
    got = {}
    for tables in (1, 0):
        _lib.check("hs2_plan_set_option",
                   L.hs2_plan_set_option(P.plan, _lib.HS2_OPT_LINE_TABLES, tables))
        assert _axes(P) == (on if tables else 0)
        T = torch.from_numpy(case["T0"]).cuda()
        for n in range(case["nsteps"]):
            T = hs.run_adi_steps(P, S, n * dt, dt, T, args["vmap"], args["volumetric"])
            assert np.abs(T.cpu().numpy() - ref[n]).max() / rise < TOL, (tables, n)
        got[tables] = T
    assert float((got[1] - got[0]).abs().max()) / rise < TOL
    # a run in one call, in place, with the readout: the same steps
    _lib.check("hs2_plan_set_option",
               L.hs2_plan_set_option(P.plan, _lib.HS2_OPT_LINE_TABLES, 1))
    T, hist = hs.run_adi_steps_many(P, 0.0, dt, case["nsteps"], torch.from_numpy(case["T0"]).cuda(),
                                    args["vmap"], args["volumetric"], surface_history=shape[0] > 1)
    assert torch.equal(T, got[1])
    if hist is not None:
        assert torch.equal(hist[-1], hs.surface_temperature.insulating_z_min_surface_temperature(
            T, case["d"][0]))


def test_line_tables_need_few_lines():
    """Maps with a distinct line almost everywhere keep the class-map kernels,
    and shapes asked for are the class-map kernels'."""
    import heatsim2_amd as hs
    from heatsim2_amd import autotune
    shape = (48, 64, 96)
    case = _case(shape, 1, 1e-3)
    case["maps"][0][:] = np.random.default_rng(2).integers(0, 3, size=shape).astype(np.uint8)
    P, _ = hs.setup(*to_package_args(hs, case)["setup"])
    assert _axes(P) == 0
    P, _ = hs.setup(*to_package_args(hs, _layers(shape, 1, 1e-3))["setup"])
    assert _axes(P) == 7
    info = _lib.plan_info(P.plan)
    autotune._apply(_lib.load(), P.plan, {
        "x": (info["x_cpl"], info["x_lanes"], info["x_lines"], info["x_lines_y"]),
        "y": (info["y_seg"], info["y_lines"]), "z": (info["z_seg"], info["z_lines"])})
    assert _axes(P) == 0
