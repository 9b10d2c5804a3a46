"""The scratch of the gradients, of one plan and of a batch: what the library
asks for, what the package takes, and what it falls back to when memory is short."""
import numpy as np
import pytest
import torch

from heatsim2_amd import _lib, adjoint, batch

pytestmark = pytest.mark.gpu

SHAPE = (64, 64, 64)
N = 64 ** 3


def _problem(steps, every):
    torch.cuda.empty_cache()  # its fields in blocks of their own
    rng = np.random.default_rng(steps)
    up = lambda a: torch.from_numpy(a).cuda()
    coef = dict(M=up(1.0 + rng.random(SHAPE)).requires_grad_(),
                w=torch.ones(SHAPE, dtype=torch.uint8, device="cuda"))
    for a, name in enumerate(("gz", "gy", "gx")):
        g = 0.5 * rng.random(SHAPE)
        g[tuple(slice(None) if b != a else 0 for b in range(3))] = 0.0
        coef[name] = up(g).requires_grad_()
    gp = adjoint.GradPlan(SHAPE, (1e-3, 1e-3, 1e-3), 1e-2)
    T0 = up(rng.random(SHAPE))
    G = up(rng.random((steps,) + SHAPE[1:]))
    return gp, coef, T0, G


def _backward(gp, coef, T0, G, steps, every):
    h = adjoint.surface_history(gp, coef, T0, steps, ckpt_every=every)
    for name in ("M", "gz", "gy", "gx"):
        coef[name].grad = None
    (h * G).sum().backward()
    torch.cuda.synchronize()
    return [coef[name].grad for name in ("M", "gz", "gy", "gx")]


def test_sizes():
    """The size that is needed is (3 K + 6) n whatever the grid; the second store
    of states is asked for where there is a second segment, and not without
    limit."""
    L = _lib.load()
    gp, coef, _, _ = _problem(4, 4)
    gp.set_coefficients([coef[k] for k in ("M", "w", "gz", "gy", "gx")])
    for K in (1, 4, 50, 500):
        assert L.hs2_grad_work_doubles(gp.plan, K) == (3 * K + 6) * N
        assert L.hs2_grad_work_best(gp.plan, K, K) == (3 * K + 13) * N
        assert L.hs2_grad_work_best(gp.plan, K + 1, K) == (6 * K + 14) * N
    assert L.hs2_grad_work_best(gp.plan, 9000, 2000) == (3 * 2000 + 13) * N
    big = adjoint.GradPlan((64, 256, 256), (1e-3, 1e-3, 1e-3), 1e-2)  # above 4 million cells
    c = [torch.zeros((64, 256, 256), dtype=torch.float64, device="cuda") for _ in range(4)]
    big.set_coefficients([c[0], c[0].to(torch.uint8)] + c[1:])
    assert L.hs2_grad_work_best(big.plan, 100, 10) == (3 * 10 + 13) * 64 * 256 * 256


def test_one_segment_takes_one_store():
    """steps <= ckpt_every: 3 K + 13 fields of scratch and the five gradients."""
    steps, every = 6, 60
    gp, coef, T0, G = _problem(steps, every)
    h = adjoint.surface_history(gp, coef, T0, steps, ckpt_every=every)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    (h * G).sum().backward()
    torch.cuda.synchronize()
    fields = (torch.cuda.max_memory_allocated() - before) / (8.0 * N)
    assert fields <= 3 * every + 13 + 5 + 4, fields


@pytest.mark.parametrize("room", [6, 13])
def test_short_memory(room):
    """Memory for 3 K + 6 or 3 K + 13 fields of scratch and little more: the
    gradients come, with the bits of the larger workspace."""
    steps, every = 90, 40
    gp, coef, T0, G = _problem(steps, every)
    want = [g.cpu() for g in _backward(gp, coef, T0, G, steps, every)]
    for name in ("M", "gz", "gy", "gx"):
        coef[name].grad = None
    torch.cuda.empty_cache()  # else the next fields are put into the old workspace
    h = adjoint.surface_history(gp, coef, T0, steps, ckpt_every=every)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    # the scratch, five gradients and the history's, in the allocator's 20 MB
    # segments of small requests
    limit = torch.cuda.memory_reserved() + (3 * every + room) * 8 * N + (48 << 20)
    try:
        torch.cuda.set_per_process_memory_fraction(limit / total)
        (h * G).sum().backward()
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    got = [coef[name].grad.cpu() for name in ("M", "gz", "gy", "gx")]
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("every", [2, 6])
def test_batches_in_short_memory(every):
    """A batch whose scratch lacks the 8 fields that sensitivities four steps at a
    time take: the same bits; and one field less is refused."""
    torch.cuda.empty_cache()
    shapes, steps = [(40, 64, 64), (64, 50, 70), (33, 65, 90)], [5, 9, 14]
    rng = np.random.default_rng(every)
    up = lambda a: torch.from_numpy(a).cuda()
    coefs, T0s, Gs = [], [], []
    for shape, n in zip(shapes, steps):
        c = dict(M=up(1.0 + rng.random(shape)), w=torch.ones(shape, dtype=torch.uint8, device="cuda"))
        for a, name in enumerate(("gz", "gy", "gx")):
            c[name] = up(0.5 * rng.random(shape))
            c[name].select(a, 0).zero_()
        coefs.append(c)
        T0s.append(up(rng.random(shape)))
        Gs.append(up(rng.random((n,) + shape[1:])))

    def gradients(gb):
        leaves = [{k: v.clone().requires_grad_() if k != "w" else v for k, v in c.items()}
                  for c in coefs]
        h = gb.surface_history(leaves, T0s)
        sum((a * G).sum() for a, G in zip(h, Gs)).backward()
        torch.cuda.synchronize()
        return [c[k].grad.cpu() for c in leaves for k in ("M", "gz", "gy", "gx")]

    want = gradients(batch.GradBatch(shapes, [1e-3] * 3, steps, [-1] * 3, ckpt_every=every))
    gb = batch.GradBatch(shapes, [1e-3] * 3, steps, [-1] * 3, ckpt_every=every)
    full = gb.work_doubles
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction(
            (torch.cuda.memory_reserved() + (full - 4 * gb.N) * 8) / total)
        gb.work()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert gb.work_doubles == full - 8 * gb.N == gb._work.numel()
    got = gradients(gb)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    gb.work_doubles -= gb.N
    with pytest.raises(_lib.HS2Error):
        gradients(gb)
