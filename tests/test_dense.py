"""Sweeps and adjoint solves on per-voxel coefficients at the edges of their
lane and segment shapes: steps against the oracle, the adjoint against two
identities of the step.

The step is linear in T without sources, so J = <G, history> of a run from T0
equals <dJ/dT0, T0>; and it does not change when M and every conductance are
scaled together, so sum(M dJ/dM) + sum(g dJ/dg) = 0 (steps without sources).
Each line solve has a relative error of a few 1e-15; six steps of three
solves, forwards and backwards, stay below 1e-12 of the sums' magnitudes."""

import ctypes

import numpy as np
import pytest
import torch

import oracle
from heatsim2_amd import _lib, adjoint, batch
from hs2_cases import oracle_coef

pytestmark = pytest.mark.gpu

# rows: 16 lanes x 2..4 cells, 32 x 3..4, 64 x 3..4, then the per-cell kernels;
# columns: segments of 4, 8 and 16 cells, one to 32 of them, whole and cut
SHAPES = [(2, 1, 1), (2, 3, 2), (3, 2, 15), (4, 5, 32), (5, 4, 33), (9, 7, 48), (8, 9, 49),
          (32, 6, 64), (33, 5, 65), (6, 33, 96), (5, 32, 97), (64, 3, 128), (3, 65, 129),
          (2, 128, 192), (129, 2, 193), (6, 7, 256), (3, 130, 255), (4, 5, 257), (2, 3, 511),
          (512, 2, 3), (513, 2, 3), (2, 512, 5), (2, 513, 4), (17, 40, 51)]
STEPS, EVERY = 6, 4


def _problem(shape, strong):
    """Coefficients that vary from cell to cell, some faces without
    conductance, some FIXED cells."""
    rng = np.random.default_rng(sum(shape) + 7 * strong)
    M = 1.0 + rng.random(shape)
    w = (rng.random(shape) > 0.1).astype(np.uint8)
    g = [(50.0 if strong else 0.5) * rng.random(shape) * (rng.random(shape) > 0.1)
         for _ in range(3)]
    g[0][0] = 0.0
    g[1][:, 0] = 0.0
    g[2][:, :, 0] = 0.0
    for a in range(3):  # no conductance between two FIXED cells
        f = np.roll(w, 1, a) | w
        g[a] *= f
    return dict(M=M, w=w, g=g, T0=rng.random(shape), S=rng.random(shape),
                G=rng.random((STEPS,) + shape[1:]) - 0.5)


def _plan(p):
    gp = adjoint.GradPlan(p["M"].shape, (1e-3, 1e-3, 1e-3), 1e-2)
    up = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (p["M"], p["w"], *p["g"])]
    gp.set_coefficients(up)
    return gp


@pytest.mark.parametrize("strong", [0, 1], ids=["weak", "strong"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_dense_steps_match_oracle_and_adjoint_identities(shape, strong):
    p = _problem(shape, strong)
    gp = _plan(p)
    L = _lib.load()
    rows = oracle_coef(p["M"], p["w"], *p["g"])
    T = torch.from_numpy(p["T0"]).cuda()
    S = torch.from_numpy(p["S"]).cuda()
    ref = p["T0"]
    for n in range(3):  # with a source, without, and into another array
        out = torch.empty_like(T) if n == 2 else T
        _lib.check("hs2_step", L.hs2_step(gp.plan, _lib.ptr(T), _lib.ptr(out), None, None, 0,
                                          _lib.ptr(S) if n == 0 else None, None,
                                          _lib.stream_handle()))
        T = out
        ref = oracle.fast_step(rows, ref, p["S"] if n == 0 else None)
        assert np.abs(T.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max(), n

    T = torch.from_numpy(p["T0"]).cuda()
    G = torch.from_numpy(p["G"]).cuda()
    ckpt = torch.empty(((STEPS + EVERY - 1) // EVERY,) + shape, dtype=torch.float64, device="cuda")
    hist = torch.empty_like(G)
    s = _lib.stream_handle()
    _lib.check("hs2_grad_forward", L.hs2_grad_forward(
        gp.plan, _lib.ptr(T), STEPS, EVERY, _lib.ptr(ckpt), None, None, 0, _lib.ptr(hist), s))
    work = torch.empty(L.hs2_grad_work_doubles(gp.plan, EVERY), dtype=torch.float64, device="cuda")
    out = [torch.empty(shape, dtype=torch.float64, device="cuda") for _ in range(5)]
    _lib.check("hs2_grad_backward", L.hs2_grad_backward(
        gp.plan, STEPS, EVERY, _lib.ptr(ckpt), None, None, 0, _lib.ptr(G),
        *[_lib.ptr(t) for t in out[:4]], None, _lib.ptr(out[4]), _lib.ptr(work), work.numel(), s))
    torch.cuda.synchronize()
    # the history is the readout of the oracle's run
    ref = p["T0"]
    for t in range(STEPS):
        ref = oracle.fast_step(rows, ref, None)
        want = ref[0] - 5.0 / 16.0 * (ref[1] - ref[0])
        assert np.abs(hist[t].cpu().numpy() - want).max() <= 1e-12 * max(1.0, np.abs(ref).max()), t
    gM, gz, gy, gx, gT0 = (t.cpu().numpy() for t in out)
    assert all(np.isfinite(a).all() for a in (gM, gz, gy, gx, gT0))
    h = hist.cpu().numpy()
    size = np.abs(p["G"] * h).sum() + np.abs(gT0 * p["T0"]).sum()
    assert abs((p["G"] * h).sum() - (gT0 * p["T0"]).sum()) <= 1e-12 * size
    terms = [p["M"] * gM] + [a * b for a, b in zip(p["g"], (gz, gy, gx))]
    assert abs(sum(t.sum() for t in terms)) <= 1e-12 * sum(np.abs(t).sum() for t in terms)


@pytest.mark.parametrize("every", [1, 3, 9])
def test_gradients_do_not_depend_on_the_workspace(every):
    """A second stream and sensitivities added four steps at a time, without the
    one, and without both (the smaller workspaces), with sources in neighbouring
    steps: the same bits."""
    shape, steps, at = (9, 21, 35), 11, (0, 4, 5, 7)
    p = _problem(shape, 0)
    gp = _plan(p)
    L = _lib.load()
    n, s = int(np.prod(shape)), _lib.stream_handle()
    rng = np.random.default_rng(every)
    src = torch.from_numpy(rng.random((len(at),) + shape)).cuda()
    G = torch.from_numpy(rng.random((steps,) + shape[1:])).cuda()
    when = (ctypes.c_int32 * len(at))(*at)
    T = torch.from_numpy(p["T0"]).cuda()
    ckpt = torch.empty((-(-steps // every),) + shape, dtype=torch.float64, device="cuda")
    _lib.check("hs2_grad_forward", L.hs2_grad_forward(
        gp.plan, _lib.ptr(T), steps, every, _lib.ptr(ckpt), _lib.ptr(src), when, len(at), None, s))
    got = []
    for room in (L.hs2_grad_work_doubles(gp.plan, every), (3 * every + 13) * n,
                 (3 * every + 6) * n):
        work = torch.full((room,), np.nan, dtype=torch.float64, device="cuda")
        out = [torch.full(shape, np.nan, dtype=torch.float64, device="cuda") for _ in range(5)]
        out.append(torch.full_like(src, np.nan))
        _lib.check("hs2_grad_backward", L.hs2_grad_backward(
            gp.plan, steps, every, _lib.ptr(ckpt), _lib.ptr(src), when, len(at), _lib.ptr(G),
            *[_lib.ptr(t) for t in out[:4]], _lib.ptr(out[5]), _lib.ptr(out[4]), _lib.ptr(work),
            work.numel(), s))
        torch.cuda.synchronize()
        got.append(out)
    assert all(torch.isfinite(a).all() for a in got[0])
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))


EDGES = [s for s in SHAPES if max(s) <= 128] + [(2, 1, 31), (5, 127, 127), (128, 9, 34)]
# three groups of instances on two streams
GROUPS = [(128, 128, 128), (7, 9, 33), (127, 128, 120), (128, 125, 128), (40, 3, 17)]


@pytest.mark.parametrize("shapes", [EDGES, GROUPS], ids=["edges", "groups"])
def test_batches_match_single_plans(shapes):
    """Every row shape of the batched kernels and cut and whole columns in one
    batch, and a batch that is worked off in three groups; unequal step counts, a
    source in some: each instance against a plan of its own (other shapes, the
    same algebra: 1e-12 of the largest value)."""
    steps = [2 + (3 * i) % 7 for i in range(len(shapes))]
    src = [i % 3 - 1 for i in range(len(shapes))]

    def leaves(i):
        p = _problem(shapes[i], i % 2)
        up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda().requires_grad_()
        c = dict(M=up(p["M"]), w=torch.from_numpy(p["w"]).cuda(), gz=up(p["g"][0]),
                 gy=up(p["g"][1]), gx=up(p["g"][2]))
        T0 = torch.from_numpy(p["T0"]).cuda()
        S = up(p["S"])
        G = torch.from_numpy(np.random.default_rng(i).random((steps[i],) + shapes[i][1:])).cuda()
        return c, T0, S, G

    one, all_ = [], [leaves(i) for i in range(len(shapes))]
    for i in range(len(shapes)):
        c, T0, S, G = leaves(i)
        gp = adjoint.GradPlan(shapes[i], (1e-3, 1e-3, 1e-3), 1e-2)
        h = adjoint.surface_history(gp, c, T0, steps[i], ckpt_every=4,
                                    sources=[(src[i], S)] if src[i] >= 0 else [])
        (h * G).sum().backward()
        one.append((h, c, S))
    gb = batch.GradBatch(shapes, [1e-3] * len(shapes), steps, src, ckpt_every=4)
    hs_ = gb.surface_history([x[0] for x in all_], [x[1] for x in all_],
                             [x[2] if src[i] >= 0 else x[2].detach() for i, x in enumerate(all_)])
    sum((h * x[3]).sum() for h, x in zip(hs_, all_)).backward()
    for i, (h, c, S) in enumerate(one):
        pairs = [(hs_[i], h)] + [(all_[i][0][k].grad, c[k].grad) for k in ("M", "gz", "gy", "gx")]
        if src[i] >= 0:
            pairs.append((all_[i][2].grad, S.grad))
        for got, want in pairs:
            assert float((got - want).abs().max()) <= 1e-12 * float(want.abs().max()), (i, shapes[i])
