"""The general sweep kernels on per-voxel coefficients: what the fixed shapes
for short axes leave to them (rows of more than 256 cells, columns of more than
512, fields of 4 GiB)."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from heatsim2_amd import _lib, autotune
from hs2_cases import oracle_coef
from test_dense import _plan, _problem
from test_gpu_parity import _curved_case, _every_launch_shape

pytestmark = pytest.mark.gpu

SHAPES = [(5, 6, 257), (4, 5, 300), (8, 4, 512), (3, 4, 513), (2, 3, 1000), (4, 2, 1024),
          (513, 2, 5), (600, 3, 17), (1024, 2, 9), (2, 520, 6), (2, 1000, 33), (2, 1024, 8)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_every_launch_shape_per_side(shape):
    """Curved bodies: every launch shape of the long axis against the oracle, with
    sources and without."""
    import heatsim2_amd as hs
    case = _curved_case(shape, seed=5 + sum(shape))
    case["nsteps"] = 6
    _every_launch_shape(hs, case)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_every_launch_shape_symmetric(shape):
    """The same on coefficients with one conductance per face, strongly coupled,
    with a source field in the first step."""
    p = _problem(shape, 1)
    gp = _plan(p)
    L = _lib.load()
    rows = oracle_coef(p["M"], p["w"], *p["g"])
    ref = [oracle.fast_step(rows, p["T0"], p["S"])]
    ref.append(oracle.fast_step(rows, ref[0], None))
    info = _lib.plan_info(gp.plan)
    base = {"x": (info["x_cpl"], info["x_lanes"], info["x_lines"], info["x_lines_y"]),
            "y": (info["y_seg"], info["y_lines"]), "z": (info["z_seg"], info["z_lines"])}
    S = torch.from_numpy(p["S"]).cuda()
    for axis, cands in (("x", autotune.x_candidates(shape[2])),
                        ("y", autotune.strided_candidates(shape[1])),
                        ("z", autotune.strided_candidates(shape[0]))):
        for cand in cands:
            autotune._apply(L, gp.plan, dict(base, **{axis: cand}))
            T = torch.from_numpy(p["T0"]).cuda()
            for n in range(2):
                _lib.check("hs2_step", L.hs2_step(gp.plan, _lib.ptr(T), _lib.ptr(T), None, None,
                                                  0, _lib.ptr(S) if n == 0 else None, None,
                                                  _lib.stream_handle()))
                assert np.abs(T.cpu().numpy() - ref[n]).max() <= 1e-12 * np.abs(ref[n]).max(), \
                    (axis, cand, n)


@pytest.mark.parametrize("asym", [False, True], ids=["symmetric", "per side"])
@pytest.mark.parametrize("shape", [(512, 1024, 1024), (1024, 512, 1024)],
                         ids=lambda s: "x".join(map(str, s)))
def test_short_segments_on_fields_of_4_gib(shape, asym):
    """Columns of 512 cells in fields of 4 GiB run in segments of 8 cells by 8
    lines, which hs2_plan_set_config accepts there, as in the default ones of 16
    (the same equations, each solve to a few 1e-15)."""
    L = _lib.load()
    grid = _lib.GridDesc(*shape, 1e-3, 1e-3, 1e-3, 1e-2)
    plan = ctypes.c_void_p()
    _lib.check("hs2_plan_create", L.hs2_plan_create(ctypes.byref(grid), ctypes.byref(plan)))
    gen = torch.Generator("cuda").manual_seed(sum(shape) + asym)

    def field():
        return torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen)

    try:
        M = field().add_(1.0)
        w = torch.ones(shape, dtype=torch.uint8, device="cuda")
        minus, plus = [], []
        for a in range(3):
            g = field().mul_(0.5)
            g.select(a, 0).zero_()
            minus.append(g)
            if asym:
                g = field().mul_(0.5)
                g.select(a, shape[a] - 1).zero_()
                plus.append(g)
        if asym:
            _lib.check("hs2_plan_set_dense_asym", L.hs2_plan_set_dense_asym(
                plan, _lib.ptr(M), _lib.ptr(w), *[_lib.ptr(g) for g in minus + plus]))
        else:
            _lib.check("hs2_plan_set_dense", L.hs2_plan_set_dense(
                plan, _lib.ptr(M), _lib.ptr(w), *[_lib.ptr(g) for g in minus]))
        info = _lib.plan_info(plan)
        T0 = field()
        out = []
        for seg, lines in ((None, None), (8, 8)):
            y = (info["y_seg"], info["y_lines"])
            z = (info["z_seg"], info["z_lines"])
            if seg and shape[1] == 512:
                y = (seg, lines)
            if seg and shape[0] == 512:
                z = (seg, lines)
            _lib.check("hs2_plan_set_config", L.hs2_plan_set_config(
                plan, info["x_cpl"], info["x_lanes"], info["x_lines"], info["x_lines_y"], *y, *z))
            T = T0.clone()
            _lib.check("hs2_step", L.hs2_step(plan, _lib.ptr(T), _lib.ptr(T), None, None, 0, None,
                                              None, _lib.stream_handle()))
            out.append(T)
        torch.cuda.synchronize()
        # away from the initial field, and to round-off of each other
        assert float(T0.sub_(out[0]).abs_().max()) > 1e-3
        assert float(out[0].sub_(out[1]).abs_().max()) <= 1e-13
    finally:
        L.hs2_plan_destroy(plan)
