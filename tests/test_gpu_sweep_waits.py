"""A wait of the sweeps without barriers that runs out fails the call. SCX_FLOW_POLLS=1 lets a wait
for a body run out at the first look that does not find it; the kernel goes on without waiting and
ends as always.
"""

import ctypes
import threading
import time

import numpy as np
import pytest

import scisim_amd as scx

pytestmark = pytest.mark.gpu


def _grid(m, gap=-1e-4):
    """m x m circles a gap from their neighbours, at rest: 2 m (m - 1) contacts in a few colours,
    each in rows of its own, so all waves but the first wait for another's."""
    d = 0.1 + gap
    q = np.stack(np.meshgrid(np.arange(m), np.arange(m)), -1).reshape(-1, 2) * d
    return dict(q=q.ravel(), v=np.zeros(2 * m * m), r=np.full(m * m, 0.05), m=np.ones(m * m))


def _context(monkeypatch, s, polls, lds="0"):
    for key in ("SCX_FLOW_SWEEPS", "SCX_FLOW_BLOCKS", "SCX_FLOW_XCDS", "SCX_FORCE_PERSISTENT_BLOCKS"):
        monkeypatch.delenv(key, raising=False)
    monkeypatch.setenv("SCX_LDS_SWEEPS", lds)
    if polls:
        monkeypatch.setenv("SCX_FLOW_POLLS", str(polls))
    else:
        monkeypatch.delenv("SCX_FLOW_POLLS", raising=False)
    ctx = scx.Context(2, s["r"].size, max_planes=8)
    ctx.set_bodies(s["q"], s["v"], s["r"], s["m"])
    return ctx


def _params(**kw):
    return scx.step_params(**dict(dict(dt=0.01, g=[0.0, 0.0], mu=0.4, CoR=0.0, tol=1e-10, max_iters=50, eval_every=1,
                                       integrator=0, precision=scx.FP64, warm_start=scx.WARM_TRANSPORT), **kw))


def test_any_wave_reports_a_wait_that_ran_out(monkeypatch):
    """One FP32 sweep that nothing evaluates: its waves do not meet after their waits, and the first
    one, whose contacts are of the first colour, waits for nothing."""
    s = _grid(8)
    s["v"] = np.random.default_rng(1).normal(0.0, 0.1, s["v"].size)
    prm = _params(precision=scx.FP32_POLISH, max_iters=1, eval_every=5)
    ctx = _context(monkeypatch, s, None)
    try:
        st = ctx.step(prm)
        print(st, ctx.sweep_paths(), flush=True)
        assert st["sweeps_fp32"] == st["sweeps"] == 1 and ctx.sweep_paths()["fp32"] == ("flow", 1)
    finally:
        ctx.close()
    ctx = _context(monkeypatch, s, 1)
    try:
        with pytest.raises(scx.ScxError, match="ran out"):
            ctx.step(prm)
    finally:
        ctx.close()


def test_run_reports_a_wait_of_any_step(monkeypatch):
    """Overlapping circles that move apart: contacts, and waits, in the first steps only. Where a
    contact's impulse is zero the abandoned sweeps change nothing, so nothing else would tell (a
    tolerance of 0: sweeps up to the limit all the same)."""
    s = _grid(8)
    q = s["q"].reshape(-1, 2)
    s["v"] = (0.005 * (q - q.mean(0))).ravel()  # a gap 1e-4 smaller than a diameter opens in 20 steps
    ctx = _context(monkeypatch, s, None)
    try:
        contacts = [ctx.step(_params(tol=0.0))["ncontacts"] for _ in range(40)]
        print(contacts, flush=True)
        assert contacts[0] == 112 and contacts[-1] == 0
    finally:
        ctx.close()
    ctx = _context(monkeypatch, s, 1)
    try:
        with pytest.raises(scx.ScxError, match="ran out"):
            ctx.run(_params(tol=0.0), 40)
        q, v, _ = ctx.get_state()
        assert np.array_equal(q, s["q"]) and np.array_equal(v, s["v"])  # the first step's start
    finally:
        ctx.close()


@pytest.mark.parametrize("call", ["step", "run"])
@pytest.mark.parametrize("staggering", [scx.STAGGER_GEOMETRIC, scx.STAGGER_SYMPLECTIC_EULER])
def test_the_step_that_failed_leaves_its_start_state(monkeypatch, call, staggering):
    """Bodies as at the start of the step, and no impulses of it in the cache: loaded into a fresh
    context, the checkpoint goes on as a fresh scene does from the same bodies."""
    s = _grid(8)
    s["v"] = np.random.default_rng(2).normal(0.0, 0.1, s["v"].size)
    prm = _params(staggering=staggering)
    ctx = _context(monkeypatch, s, 1)
    try:
        with pytest.raises(scx.ScxError, match="ran out"):
            ctx.step(prm) if call == "step" else ctx.run(prm, 3)
        q, v, _ = ctx.get_state()
        assert np.array_equal(q, s["q"]) and np.array_equal(v, s["v"])
        with pytest.raises(scx.ScxError):  # (warm start 3 computes features, of a step that succeeds)
            ctx.samples()
        image = ctx.save_checkpoint()
        assert scx.checkpoint_info(image)["cache_entries"] == 0
    finally:
        ctx.close()
    out = []
    for loaded in (False, True):
        ctx = _context(monkeypatch, s, None)
        try:
            if loaded:
                ctx.load_checkpoint(image)
            st = ctx.step(prm)
            assert st["sweeps"] > 1 and ctx.sweep_paths()["fp64"][0] == "flow"
            out.append(ctx.get_state()[:2])
        finally:
            ctx.close()
    assert all(np.array_equal(x, y) for x, y in zip(*out))


@pytest.mark.parametrize("warm", [0.0, 0.01])
def test_the_solve_that_failed_leaves_the_impulses(monkeypatch, warm):
    """The impulses of a stand-alone solve are warm start and result; a failed one leaves them."""
    m = 8
    at = np.arange(m * m, dtype=np.int32).reshape(m, m)
    body0 = np.concatenate([at[:, :-1].ravel(), at[:-1].ravel()])
    body1 = np.concatenate([at[:, 1:].ravel(), at[1:].ravel()])
    n = np.repeat(-np.eye(2), body0.size // 2, 0)
    bases = np.stack([n, np.stack([-n[:, 1], n[:, 0]], 1)], 1).ravel()
    mass, v0, mu = np.ones(m * m), np.random.default_rng(3).normal(size=2 * m * m), np.full(body0.size, 0.4)
    cs = scx.ScxContactSet(ncontacts=body0.size, body0=scx._p(body0, scx._pi32), body1=scx._p(body1, scx._pi32),
                           bases=scx._p(bases), mu=scx._p(mu))
    for polls in (1, None):
        alpha, beta = np.full(body0.size, warm), np.full(body0.size, -0.1 * warm)
        ctx = _context(monkeypatch, _grid(m), polls)
        try:
            rc = scx.lib().scx_friction_solve(ctx.handle, m * m, scx._p(mass), None, scx._p(v0), None,
                                              ctypes.byref(cs), 1e-10, 50, 1, scx.FP64, scx._p(alpha), scx._p(beta),
                                              None, None, None, None, None, None)
            assert (rc == scx.SCX_OK) == (polls is None)
            assert ctx.sweep_paths()["fp64"][0] == "flow"
            unchanged = np.all(alpha == warm) and np.all(beta == -0.1 * warm)
            assert unchanged == (polls is not None)
        finally:
            ctx.close()


def test_a_launch_waits_for_its_workgroups(monkeypatch):
    """A solve of some seconds in one workgroup of another context leaves one CU short of LDS: sweeps
    that need all of them wait for it to end."""
    small, large = _grid(16), _grid(400)
    for s in (small, large):
        s["v"] = np.random.default_rng(4).normal(0.0, 0.1, s["v"].size)
    out, took = [], []
    for beside in (False, True):
        ctx = _context(monkeypatch, large, None)
        try:
            if beside:
                other = _context(monkeypatch, small, None, lds="1")
                done = []
                t = threading.Thread(target=lambda: done.append(
                    (other.step(_params(tol=0.0, max_iters=1500000, eval_every=1000)), time.perf_counter())))
                t.start()
                time.sleep(0.5)
            t0 = time.perf_counter()
            st = ctx.step(_params(max_iters=30))
            t1 = time.perf_counter()
            print(st, ctx.sweep_paths(), t1 - t0, flush=True)
            assert ctx.sweep_paths()["fp64"] == ("flow", 256)
            if beside:
                t.join()
                print(done, other.sweep_paths(), flush=True)
                assert other.sweep_paths()["fp64"] == ("lds", 1) and done[0][0]["sweeps"] == 1500000
                other.close()
            took.append(t1 - t0)
            out.append(ctx.get_state()[:2])
        finally:
            ctx.close()
    assert all(np.array_equal(x, y) for x, y in zip(*out))
    print("seconds", took, flush=True)
    assert took[1] > 1.0  # it did wait
