"""Which sweep kernel serves which contact set (scx_get_sweep_paths), and the kernels against each
other. The iterates of all three are the same bit for bit. At a sweep limit the one-workgroup LDS
kernel takes the velocities anew from the best impulses also where the last iterate is the best,
which the other two leave as the sweeps made them: the same impulses, velocities that round
differently.
"""

import numpy as np
import pytest

import scisim_amd as scx
from scisim_amd import scenes

import test_gpu_sweep_paths as base

pytestmark = pytest.mark.gpu

SWITCHES = ("SCX_LDS_SWEEPS", "SCX_FLOW_SWEEPS", "SCX_FLOW_BLOCKS", "SCX_FLOW_XCDS", "SCX_FORCE_PERSISTENT_BLOCKS", "SCX_FLOW_TAG")


def _context(monkeypatch, s, **env):
    for key in SWITCHES:
        monkeypatch.delenv(key, raising=False)
    for key, x in env.items():
        monkeypatch.setenv(key, str(x))
    ctx = scx.Context(s["dim"], s["r"].size, max_planes=8)
    ctx.set_planes(s["px"], s["pn"])
    ctx.set_bodies(s["q"], s["v"], s["r"], s["m"], inertia=s.get("inertia"))
    return ctx


def _run(monkeypatch, s, prm, steps, **env):
    ctx = _context(monkeypatch, s, **env)
    try:
        out, paths = [], []
        for _ in range(steps):
            st = ctx.step(scx.step_params(**prm))
            con = ctx.contacts()
            out.append((st, *ctx.get_state(), con["alpha"], con["beta"]))
            if st["ncontacts"]:
                paths.append(ctx.sweep_paths())
        return out, paths
    finally:
        ctx.close()


def _all(paths, precision, path, groups=None):
    assert paths
    for p in paths:
        for phase in ("fp32", "fp64") if precision == "fp32" else ("fp64",):
            assert p[phase][0] == path, p
            assert groups is None or p[phase][1] == groups, p


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


@pytest.mark.parametrize("kind", ["one", "60", "lattice"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("limit", ["converged", "limit", "sparse", "stagnates"])
def test_small_sets_in_all_three_kernels(monkeypatch, kind, precision, limit):
    """Sets that one workgroup's LDS holds whole, in that kernel, in the sweeps without barriers on
    one and two workgroups and in those with barriers."""
    print("case", kind, precision, limit, flush=True)
    s = base._scene(kind)
    prm = base._params(s, precision, limit)
    ref, paths = _run(monkeypatch, s, prm, 3, SCX_FORCE_PERSISTENT_BLOCKS=2)
    _all(paths, precision, "barriers", 2)
    for blocks in (1, 2):
        got, paths = _run(monkeypatch, s, prm, 3, SCX_LDS_SWEEPS=0, SCX_FLOW_BLOCKS=blocks)
        _all(paths, precision, "flow", blocks)
        base._same(ref, got)
    got, paths = _run(monkeypatch, s, prm, 3)
    _all(paths, precision, "lds", 1)
    # up to the first step that ends at the limit, whose velocities go into the next ones
    upto = next((k for k, a in enumerate(ref) if not a[0]["succeeded"]), len(ref))
    base._same(ref[:upto], got[:upto])
    if upto < len(ref):
        a, b = ref[upto], got[upto]
        for key in ("ncontacts", "ncolours", "sweeps", "sweeps_fp32", "error", "succeeded"):
            assert a[0][key] == b[0][key], key
        for x, y in zip(a[4:], b[4:]):  # impulses
            assert np.array_equal(x, y)


def _grid(m):
    """m x m circles that overlap their neighbours by a little: 2 m (m - 1) contacts."""
    q = np.stack(np.meshgrid(np.arange(m), np.arange(m)), -1).reshape(-1, 2) * 0.0999
    return dict(dim=2, q=q.ravel(), v=np.random.default_rng(m).normal(0.0, 0.1, 2 * m * m), r=np.full(m * m, 0.05),
                m=np.ones(m * m), px=np.array([[0.0, -10.0]]), pn=np.array([[0.0, 1.0]]))


@pytest.mark.parametrize("m,groups", [(160, 32), (200, 256), (1020, 256), (1030, None)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_large_sets(monkeypatch, m, groups, precision):
    """One XCD's workgroups below 65,536 contacts (50,880 here), every XCD's above (79,600), up to
    2,097,152 contacts (2,078,760); grid barriers beyond (2,119,740)."""
    print("case", m, precision, flush=True)
    s = _grid(m)
    prm = dict(base._params(s, precision, "limit"), max_iters=24, g=[0.0, 0.0])
    ref, paths = _run(monkeypatch, s, prm, 1, SCX_FLOW_SWEEPS=0)
    _all(paths, precision, "barriers")
    assert ref[0][0]["ncontacts"] >= 2 * m * (m - 1)
    got, paths = _run(monkeypatch, s, prm, 1)
    print(ref[0][0], paths, flush=True)
    _all(paths, precision, "flow" if groups else "barriers", groups)
    base._same(ref, got)


@pytest.mark.parametrize("dim,side,path,precision",
                         [(3, 10, "flow 1", "fp64"), (3, 11, "flow 29", "fp64"), (2, 38, "flow 1", "fp64"),
                          (2, 39, "flow 24", "fp64"), (3, 28, "flow 32", "fp64"), (3, 29, "barriers", "fp64"),
                          (3, 29, "barriers", "fp32"), (3, 56, "barriers", "fp64"), (3, 57, "flow 256", "fp64"),
                          (2, 190, "flow 256", "fp64")])
def test_stand_alone_solves(monkeypatch, dim, side, path, precision):
    """Contacts of bodies in no order, spheres on a cubic lattice and circles on a square one: one
    workgroup up to 2,816 contacts, one XCD up to 65,536; spheres in FP64 with grid barriers from
    there (63,504 and 70,644 here) to 524,288 (517,440 and 545,832)."""
    rng = np.random.default_rng(side)
    n = side ** dim
    at = rng.permutation(n).reshape((side,) * dim)
    a = np.concatenate([np.delete(at, -1, k).ravel() for k in range(dim)]).astype(np.int32)
    b = np.concatenate([np.delete(at, 0, k).ravel() for k in range(dim)]).astype(np.int32)
    nn = -np.eye(dim)[np.repeat(np.arange(dim), a.size // dim)]
    t1 = np.roll(nn, 1, 1) * (1.0 if dim == 3 else [[-1.0, 1.0]])
    prob = dict(m=rng.uniform(1.0, 2.0, n), v0=rng.normal(size=dim * n), body0=a, body1=b, mu=np.full(a.size, 0.4))
    if dim == 3:
        prob.update(inertia=rng.uniform(0.1, 0.2, n), omega0=rng.normal(size=3 * n), arm0=-0.5 * nn, arm1=0.5 * nn,
                    bases=np.stack([nn, t1, np.cross(nn, t1)], 1))
    else:
        prob.update(bases=np.stack([nn, t1], 1))
    out = []
    for flow in ("0", "1"):
        for key in SWITCHES:
            monkeypatch.delenv(key, raising=False)
        monkeypatch.setenv("SCX_FLOW_SWEEPS", flow)
        ctx = scx.Context(dim, n, max_planes=8)
        try:
            out.append(ctx.friction_solve(tol=1e-9, max_iters=200 if a.size < 9000 else 20, eval_every=1,
                                          precision=scx.FP64 if precision == "fp64" else scx.FP32_POLISH, **prob))
            paths = ctx.sweep_paths()
        finally:
            ctx.close()
    print(a.size, out[1]["sweeps"], paths, flush=True)
    assert ("%s %d" % paths["fp64"]).startswith(path)
    assert paths["fp32"][0] == (None if precision == "fp64" else "flow")
    for key, x in out[0].items():
        assert np.array_equal(x, out[1][key]), key


@pytest.mark.parametrize("kind", ["700", "9000"])
@pytest.mark.parametrize("short", [1, 166, 167, 300, 500])
def test_tags_start_over(monkeypatch, kind, short):
    """A launch takes its limit of 150 sweeps and 16 more tags. With fewer left, the tags start over on
    cleared slots: before the first launch, between the two phases of a step, or in a later step
    (300, 500); the steps are those of a context at its first tags."""
    print("case", kind, short, flush=True)
    s = base._scene(kind)
    prm = base._params(s, "fp32", "limit")
    ref, paths = _run(monkeypatch, s, prm, 4, SCX_LDS_SWEEPS=0)
    _all(paths, "fp32", "flow")
    got, _ = _run(monkeypatch, s, prm, 4, SCX_LDS_SWEEPS=0, SCX_FLOW_TAG=2 ** 30 - short)
    base._same(ref, got)


def _paths_at_close(monkeypatch):
    seen, close = [], scx.Context.close

    def record(self):
        seen.append(self.sweep_paths())
        close(self)

    monkeypatch.setattr(scx.Context, "close", record)
    monkeypatch.setenv("SCX_FLOW_SWEEPS", "0")
    return seen


@pytest.mark.parametrize("limit", ["converged", "sweep_limit"])
def test_compacted_ensembles_with_barriers(monkeypatch, limit):
    """The compaction belongs to the sweeps with barriers, which serve the largest ensembles."""
    import test_gpu_ensemble_compaction as t

    seen = _paths_at_close(monkeypatch)
    piles = scenes.ensemble_piles(nscenes=96, nmin=100, nmax=2000, seed=3, workers=8)
    t.test_compacted_sweeps_match_uncompacted_bit_for_bit(monkeypatch, piles, 0, limit)
    _all(seen, "fp32", "barriers")
    assert len(seen) == 2 and all(p["fp32"][1] > 1 for p in seen)


@pytest.mark.parametrize("mode", ["transport", "cold", "fp64", "fp64_limit"])
def test_skipped_evaluations_with_barriers(monkeypatch, mode):
    """The list of contacts near the maximum belongs to the sweeps with barriers."""
    import test_gpu_violator_skip as t

    seen = _paths_at_close(monkeypatch)

    class Request:
        def getfixturevalue(self, kind):
            return scenes.spheres_pile(n=8000, seed=9)

    t.test_skipped_evaluations_change_nothing(monkeypatch, Request(), "pile", 0, mode)
    _all(seen, "fp64" if mode.startswith("fp64") else "fp32", "barriers")
    assert all(p["fp64"][1] > 1 for p in seen)
