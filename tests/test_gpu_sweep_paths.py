"""The sweeps without barriers between the colours (k_gs_flow), on one workgroup and on several,
against the sweeps with grid barriers (the others switched off):
every contact is updated in its colour's turn with the same expressions, so steps are the
same bit for bit -- positions, velocities, impulses, sweep counts, residuals -- in FP64 and in
FP32 with the FP64 polish, converging, ending at a sweep limit with the best iterate, through
the FP32 stagnation test, with sparse residual checks; for contact sets around the passes of a
workgroup and the smallest and largest each path takes.
"""

import numpy as np
import pytest

import scisim_amd as scx
from scisim_amd import scenes

pytestmark = pytest.mark.gpu


def _scene(kind):
    if kind == "one":  # one sphere on the floor: a single contact, a single colour
        s = scenes.spheres_pile(n=1, base=1.0, seed=3)
    elif kind == "circles":
        s = scenes.ball2d_rsa(n=6000, seed=11)
        s["v"] = np.random.default_rng(11).normal(0.0, 2.0, s["v"].size)
    elif kind == "lattice":
        s = scenes.ball2d_lattice(m=40, side=6.25, r=0.05, vstd=0.5, seed=2)
    else:
        s = scenes.spheres_pile(n=int(kind), seed=13)
    return s


def _run(monkeypatch, s, path, prm, steps, blocks=None):
    monkeypatch.setenv("SCX_FLOW_SWEEPS", "1" if path == "flow" else "0")
    if blocks:
        monkeypatch.setenv("SCX_FLOW_BLOCKS", str(blocks))
    else:
        monkeypatch.delenv("SCX_FLOW_BLOCKS", raising=False)
    D = s["dim"]
    ctx = scx.Context(D, s["r"].size, max_planes=8)
    try:
        ctx.set_planes(s["px"], s["pn"])
        ctx.set_bodies(s["q"], s["v"], s["r"], s["m"], inertia=s.get("inertia"))
        out = []
        for _ in range(steps):
            st = ctx.step(scx.step_params(**prm))
            con = ctx.contacts()
            out.append((st, *ctx.get_state(), con["alpha"], con["beta"]))
        return out
    finally:
        ctx.close()


def _params(s, precision, limit):
    D = s["dim"]
    prm = dict(dt=0.005, g=[0.0, -9.81] if D == 2 else [0.0, -9.81, 0.0], mu=0.4, CoR=0.0,
               integrator=0 if D == 2 else 1, precision=scx.FP64 if precision == "fp64" else scx.FP32_POLISH,
               warm_start=scx.WARM_TRANSPORT)
    prm.update({"converged": dict(tol=1e-7, max_iters=3000, eval_every=1),
                "limit": dict(tol=1e-13, max_iters=150, eval_every=1),
                "sparse": dict(tol=1e-10, max_iters=310, eval_every=20),
                "stagnates": dict(tol=1e-12, max_iters=3000, eval_every=1, warm_start=scx.WARM_NONE)}[limit])
    return prm


def _same(ref, got):
    for a, b in zip(ref, got):
        print(a[0], flush=True)
        for key in ("ncontacts", "ncolours", "sweeps", "sweeps_fp32", "error", "succeeded"):
            assert a[0][key] == b[0][key], key
        for x, y in zip(a[1:], b[1:]):
            assert x is None or np.array_equal(x, y)


@pytest.mark.parametrize("kind", ["one", "circles", "lattice", "60", "700", "2500"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("limit", ["converged", "limit", "sparse", "stagnates"])
def test_one_workgroup(monkeypatch, kind, precision, limit):
    print("case", kind, precision, limit, flush=True)
    s = _scene(kind)
    prm = _params(s, precision, limit)
    _same(_run(monkeypatch, s, "", prm, 3), _run(monkeypatch, s, "flow", prm, 3, 1))


@pytest.mark.parametrize("kind,blocks", [("circles", 2), ("circles", None), ("lattice", 7), ("2500", 3), ("2500", None),
                                         ("9000", None), ("9000", 256)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("limit", ["converged", "limit", "sparse", "stagnates"])
def test_without_barriers(monkeypatch, kind, blocks, precision, limit):
    print("case", kind, blocks, precision, limit, flush=True)
    s = _scene(kind)
    prm = _params(s, precision, limit)
    _same(_run(monkeypatch, s, "", prm, 3), _run(monkeypatch, s, "flow", prm, 3, blocks))


@pytest.mark.parametrize("kind", ["circles", "2500"])
@pytest.mark.parametrize("xcds,blocks", [(1, 1), (1, 32), (2, 2), (8, 8), (8, 256)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_without_barriers_spread(monkeypatch, kind, xcds, blocks, precision):
    """The slots of bodies that one XCD holds stay in its L2, the others go through to memory."""
    print("case", kind, xcds, blocks, precision, flush=True)
    s = _scene(kind)
    prm = _params(s, precision, "converged")
    ref = _run(monkeypatch, s, "", prm, 3)
    monkeypatch.setenv("SCX_FLOW_XCDS", str(xcds))
    _same(ref, _run(monkeypatch, s, "flow", prm, 3, blocks))


@pytest.mark.parametrize("side", [7, 8, 12])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_stand_alone_solve_without_barriers(monkeypatch, side, precision):
    """Contacts in no order: 882 (one workgroup), 1,344 and 4,752 (equal shares of each colour)."""
    print("case", side, precision, flush=True)
    rng = np.random.default_rng(side)
    at = np.arange(side ** 3).reshape(side, side, side)
    a = np.concatenate([np.delete(at, -1, k).ravel() for k in range(3)])
    b = np.concatenate([np.delete(at, 0, k).ravel() for k in range(3)])
    axis = np.repeat(np.arange(3), a.size // 3)
    order = rng.permutation(a.size)
    a, b, axis = a[order], b[order], axis[order]
    nn = -np.eye(3)[axis]
    t1 = np.eye(3)[(axis + 1) % 3]
    prob = dict(m=rng.uniform(1.0, 2.0, side ** 3), inertia=rng.uniform(0.1, 0.2, side ** 3),
                v0=rng.normal(size=3 * side ** 3), omega0=rng.normal(size=3 * side ** 3), body0=a.astype(np.int32),
                body1=b.astype(np.int32), bases=np.stack([nn, t1, np.cross(nn, t1)], 1), arm0=-0.5 * nn,
                arm1=0.5 * nn, mu=np.full(a.size, 0.4))

    def run(flow):
        monkeypatch.setenv("SCX_FLOW_SWEEPS", flow)
        monkeypatch.delenv("SCX_FLOW_BLOCKS", raising=False)
        ctx = scx.Context(3, side ** 3, max_planes=8)
        try:
            return ctx.friction_solve(tol=1e-9, max_iters=400, eval_every=1,
                                      precision=scx.FP64 if precision == "fp64" else scx.FP32_POLISH, **prob)
        finally:
            ctx.close()

    ref, got = run("0"), run("1")
    print(ref["sweeps"], ref["error"], flush=True)
    for key, x in ref.items():
        assert np.array_equal(x, got[key]), key


@pytest.mark.parametrize("scenes_,blocks", [(3, None), (70, None), (70, 3), (70, 256)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("limit", ["converged", "limit", "sparse", "stagnates"])
def test_ensemble_without_barriers(monkeypatch, scenes_, blocks, precision, limit):
    """70 piles (more than two words of the frozen mask), most of which freeze on the way, and 3
    (one workgroup)."""
    print("case", scenes_, blocks, precision, limit, flush=True)
    cat, body_off, plane_off, mus, _ = scenes.ensemble_piles(nscenes=scenes_, nmin=20, nmax=200, seed=4, workers=4)
    prm = _params(cat, precision, limit)

    def run(path):
        monkeypatch.setenv("SCX_FLOW_SWEEPS", "1" if path else "0")
        monkeypatch.delenv("SCX_FLOW_BLOCKS", raising=False)
        if path and blocks:
            monkeypatch.setenv("SCX_FLOW_BLOCKS", str(blocks))
        ctx = scx.Context(3, cat["r"].size, max_planes=350)
        try:
            ctx.set_planes(cat["px"], cat["pn"])
            ctx.set_bodies(cat["q"], cat["v"], cat["r"], cat["m"], inertia=cat["inertia"])
            ctx.set_scenes(body_off, plane_off, mus)
            out = []
            for _ in range(3):
                st = ctx.step(scx.step_params(**prm))
                con = ctx.contacts()
                out.append((st, *ctx.get_state(), con["alpha"], con["beta"], *ctx.scene_stats()))
            return out
        finally:
            ctx.close()

    _same(run(False), run(True))
