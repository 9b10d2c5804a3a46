"""The autotuner's decisions, on a library of the test's own (no GPU)."""
import types

import pytest
import torch

from heatsim2_amd import _lib, autotune


class Library(object):
    """Plans are (shape, mode, line-table axes, us on tables, us of the shapes)."""

    def __init__(self):
        self.lines_on, self.timed, self.shapes = {}, [], []

    def hs2_version(self):
        return b"library"


@pytest.fixture
def library(monkeypatch, tmp_path):
    L = Library()
    monkeypatch.setenv("HS2_TUNE_CACHE", str(tmp_path / "tune.json"))
    monkeypatch.setattr(autotune, "_memo", {})
    monkeypatch.setattr(_lib, "load", lambda: L)
    monkeypatch.setattr(_lib, "plan_info", lambda plan: dict(
        mode=plan.mode, x_cpl=16, x_lanes=16, x_lines=16, x_lines_y=0, y_seg=16, y_lines=8,
        z_seg=16, z_lines=8))
    monkeypatch.setattr(_lib, "device", lambda: torch.device("cpu"))
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda: "device")
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    monkeypatch.setattr(autotune, "_line_tables", lambda lib, plan: plan.lines)

    def set_lines(lib, plan, on):
        L.lines_on[plan.name] = on

    def apply(lib, plan, cfg, strict=True):
        L.lines_on[plan.name] = False
        L.shapes.append(dict(cfg))
        if cfg.get("lines"):
            set_lines(lib, plan, True)
        return True

    def time(lib, plan, T, steps):
        L.timed.append(plan.name)
        return [plan.on if L.lines_on[plan.name] else plan.off] * 3

    monkeypatch.setattr(autotune, "_set_lines", set_lines)
    monkeypatch.setattr(autotune, "_apply", apply)
    monkeypatch.setattr(autotune, "_time", time)
    return L


def _params(name, shape=(40, 50, 60), mode=1, lines=7, on=1.0, off=2.0):
    plan = types.SimpleNamespace(name=name, mode=mode, lines=lines, on=on, off=off)
    return types.SimpleNamespace(plan=plan, shape=shape)


@pytest.mark.parametrize("fresh", [False, True], ids=["memory", "file"])
def test_line_tables_are_judged_on_each_plan(library, fresh):
    """Bodies of one shape whose tables do and do not pay: each plan gets its own
    verdict, the shapes come from the first."""
    T = torch.zeros(4, dtype=torch.float64)
    first = autotune.tune(_params("plate", on=1.0, off=2.0), T)
    assert first["lines"] is True and library.lines_on["plate"] is True
    n = len(library.timed)
    for name, on, off in (("laminate", 3.0, 2.0), ("plate 2", 1.5, 2.0)):
        if fresh:
            autotune._memo.clear()
        cfg = autotune.tune(_params(name, on=on, off=off), T)
        assert cfg["lines"] is (on < off) and library.lines_on[name] is (on < off)
        assert cfg["ms"] == [min(on, off)] * 3
        assert [cfg[a] for a in "xyz"] == [first[a] for a in "xyz"]
    assert len(library.timed) == n + 12  # three of each side, no shapes
    # a plan without tables takes the shapes as they are
    n = len(library.timed)
    autotune.tune(_params("a", lines=0), T)
    m = len(library.timed)
    assert m > n and autotune.tune(_params("b", lines=0), T)["lines"] is False
    assert len(library.timed) == m


@pytest.mark.parametrize("mode", [2, 3])
@pytest.mark.parametrize("shape,chosen", [((512, 512, 256), ""), ((512, 512, 257), "x"),
                                          ((513, 512, 256), "z"), ((40, 520, 300), "xy"),
                                          ((512, 1024, 1023), "xy"), ((512, 1024, 1024), "xyz")],
                         ids=lambda s: s if isinstance(s, str) else "x".join(map(str, s)))
def test_per_voxel_axes_with_shapes_to_choose(library, mode, shape, chosen):
    """Long axes, and y and z of any length in fields of 4 GiB and more, which the
    fixed shapes do not serve."""
    autotune.tune(_params("p", shape, mode, 0), torch.zeros(4, dtype=torch.float64))
    tried = {a: {tuple(c[a]) for c in library.shapes} for a in "xyz"}
    assert "".join(a for a in "xyz" if len(tried[a]) > 1) == chosen
