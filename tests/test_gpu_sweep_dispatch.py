"""Which sweep kernel serves which contact set (scx_get_sweep_paths)."""

import pytest

import scisim_amd as scx

import test_gpu_sweep_paths as base

pytestmark = pytest.mark.gpu

SWITCHES = ("SCX_FLOW_SWEEPS", "SCX_FLOW_BLOCKS", "SCX_FLOW_XCDS", "SCX_FORCE_PERSISTENT_BLOCKS")


def _context(monkeypatch, s, **env):
    for key in SWITCHES:
        monkeypatch.delenv(key, raising=False)
    for key, x in env.items():
        monkeypatch.setenv(key, str(x))
    ctx = scx.Context(s["dim"], s["r"].size, max_planes=8)
    ctx.set_planes(s["px"], s["pn"])
    ctx.set_bodies(s["q"], s["v"], s["r"], s["m"], inertia=s.get("inertia"))
    return ctx


def test_switches_are_read_when_a_context_is_made(monkeypatch):
    """A variable that is set later, as by another thread that makes a context of its own, leaves a
    context as it is."""
    s = base._scene("2500")
    ctx = _context(monkeypatch, s)
    try:
        monkeypatch.setenv("SCX_FLOW_BLOCKS", "1")
        monkeypatch.setenv("SCX_FLOW_XCDS", "8")
        st = ctx.step(scx.step_params(**base._params(s, "fp64", "limit")))
        print(st, ctx.sweep_paths(), flush=True)
        path, groups = ctx.sweep_paths()["fp64"]
        assert path == "flow" and 8 < groups <= 32  # one XCD's share of 128 contacts a workgroup
    finally:
        ctx.close()
