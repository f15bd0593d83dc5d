"""The pair-order hint in effect, valid and stale, through every kernel that
takes it: the far units of the forward (plain, with lattice images, with the
diatomic-frame H0) and of the gradient and the adjoint (with and without the
forward's S and D), eager and in a replayed graph.  All agree with the run
without a hint: the forward's elements are the same sums (1e-12 for values up
to 1e2; with lattice images 1e-11 of the largest), the derivatives sum up to
1e4 terms in another order (1e4 u of the terms' magnitudes, which add up to at
most ten times the largest result: 1e-11 of it)."""
import numpy as np
import pytest

from tblite_amd import lib as L
from tblite_amd import synthetic

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _structures():
    """Molecules with distant pairs, d shells among them, and one without."""
    rng = np.random.default_rng(12)
    z, x = synthetic.random_molecule(20, rng)
    z2, x2 = synthetic.random_molecule(9, rng)
    far = (np.concatenate([z, z2]), np.concatenate([x, x2 + 60.0]))
    line = (np.array([17, 1, 8, 16, 6, 9, 1, 1], dtype=np.int32),
            np.array([(0.0, 0.0, 4.0 * k) for k in range(8)]) * np.array([1.0, 1.0, 4.0]))
    return [far, (z2, x2), line, synthetic.water_cluster(96, seed=3)]


def _crystals():
    mols, lats = [], []
    for n, side in ((4, 16.0), (9, 22.0)):
        z, x = synthetic.water_cluster(n, seed=n)
        mols.append((z, x))
        lats.append(([True] * 3, np.diag([side, 1.05 * side, 0.95 * side])))
    return mols, lats


def _ones(nums):
    n = len(nums)
    return [np.full((n, n), f) for f in (1.15, 0.9, 1.05)]


def _batch(kind):
    from tblite_amd.batch import Batch
    if kind == "crystals":
        mols, lats = _crystals()
        return Batch(mols, lattices=lats)
    if kind == "passes":  # more far units than a launch looks at in one pass (2048 x 4)
        b = Batch([synthetic.water_cluster(256, seed=5)])
        b.set_tiles(fwd_unit_pairs=4, grad_unit_pairs=4)
        return b
    return Batch(_structures(), diat_scale=_ones if kind == "diatomic" else None)


@pytest.mark.parametrize("kind", ["molecules", "crystals", "diatomic", "passes"])
@pytest.mark.parametrize("stale", [False, True])
def test_hint_in_effect(kind, stale):
    b = _batch(kind)
    xyz = b.tensor_xyz()
    se, dse = (t.contiguous() for t in b.selfenergy(b.ncoord(xyz)))
    rng = np.random.default_rng(3)
    t = lambda n: torch.tensor(rng.normal(size=n), device="cuda")  # noqa: E731
    adj = [t(k * b.ndense) for k in (1, 3, 6, 1)]
    P, W, vao, vdp, vqp = t(b.ndense), t(b.ndense), t(b.nao), t(3 * b.nat), t(6 * b.nat)

    def run():
        f = b.forward(xyz, se)
        out = list(f)
        if kind != "diatomic":  # no gradient of the scaled H0
            forward = [{}] if kind == "crystals" else [{}, {"S": f[0], "D": f[1]}]
            for kw in forward:
                out += b.adjoint(xyz, se, *adj, **kw)
                out += b.gradient(xyz, se, dse, P, W, vao, vdp, vqp, **kw)
        return out

    b.order_pairs(None)
    n0 = b.unit_counts()
    assert n0["fwd_far"] == n0["grad_far"] == 0
    ref = [r.clone() for r in run()]
    hint = b.xyz0.copy()
    if stale:
        hint[: 1 if kind != "passes" else b.nat // 2] += 30.0  # near pairs end up in far units
    b.order_pairs(hint, skin=0.5)
    n = b.unit_counts()
    print(f"[gpu] hint {kind} stale {stale}: {n}", flush=True)
    least = 2048 * 4 if kind == "passes" else 0
    assert n["fwd_far"] > least and n["grad_far"] > least
    for _ in range(2):
        for k, (r, g) in enumerate(zip(ref, run())):
            tol = 1e-12 if k < 4 and kind != "crystals" else 1e-11 * r.abs().max().item()
            assert torch.abs(r - g).max().item() <= tol, k


def test_replay_follows_the_geometry():
    """A captured forward and gradient, replayed with the hint valid, stale and
    valid again."""
    b = _batch("molecules")
    b.order_pairs(b.xyz0, skin=0.5)
    assert b.unit_counts()["grad_far"] > 0
    xyz = b.tensor_xyz()
    se, dse = (t.contiguous() for t in b.selfenergy(b.ncoord(xyz)))
    rng = np.random.default_rng(4)
    t = lambda n: torch.tensor(rng.normal(size=n), device="cuda")  # noqa: E731
    args = (t(b.ndense), t(b.ndense), t(b.nao), t(3 * b.nat), t(6 * b.nat))
    f = b.forward(xyz, se)
    g = b.gradient(xyz, se, dse, *args)
    print("[gpu] hint in a graph", flush=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        b.forward(xyz, se, out=f)
        b.gradient(xyz, se, dse, *args, out=g)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        b.forward(xyz, se, out=f)
        b.gradient(xyz, se, dse, *args, out=g)
    start = xyz.clone()
    for move in (0.0, 45.0, 0.0, -50.0):
        xyz.copy_(start)
        xyz[:3] += move
        for o in (*f, *g):
            o.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        got = [o.clone() for o in (*f, *g)]
        ref = [*b.forward(xyz, se), *b.gradient(xyz, se, dse, *args)]
        for k, (r, o) in enumerate(zip(ref, got)):
            assert torch.abs(r - o).max().item() <= max(1e-12, 1e-11 * r.abs().max().item()), (move, k)


def test_start_order_of_a_batch():
    """Few units: no hint until one is given; many: the starting geometry's.
    Coordinates and skin are checked in both."""
    from tblite_amd.batch import Batch
    mols = _structures()
    b = Batch(mols[:3])
    n = b.unit_counts()
    print(f"[gpu] starting order {n}", flush=True)
    assert n["fwd_far"] == n["grad_far"] == 0 and n["fwd_near"] <= 768
    b.order_pairs(b.xyz0)
    assert b.unit_counts()["fwd_far"] > 0
    big = Batch(mols + [synthetic.water_cluster(256, seed=5)])
    n = big.unit_counts()
    assert n["fwd_far"] > 0 and n["grad_far"] > 0 and n["fwd_near"] + n["fwd_far"] > 768
    for skin, bad in ((-1.0, None), (1.0, float("nan"))):
        z, x = mols[1]
        x = np.array(x)
        x[0, 0] = x[0, 0] if bad is None else bad
        with pytest.raises(L.TbxError):
            Batch([(z, x)], skin=skin)


def test_one_structure_with_one_nonzero_translation(monkeypatch):
    """The distance that decides whether a pair is distant is that of its one
    image: the clusters are 60 bohr apart and the translation brings one onto
    the other, so pairs of one cluster are distant and pairs of both are near."""
    from tblite_amd import structure
    from tblite_amd.batch import Batch
    monkeypatch.setattr(structure, "get_lattice_points",
                        lambda *a, **k: np.array([[60.0, 0.5, 0.0]]))
    z, x = synthetic.water_cluster(14, seed=8)
    z2, x2 = synthetic.random_molecule(11, np.random.default_rng(6))
    one = (np.concatenate([z, z2]), np.concatenate([x, x2 + np.array([63.0, 1.0, 2.0])]))
    b = Batch([one], lattices=[([True] * 3, np.eye(3) * 60.0)])
    xyz = b.tensor_xyz()
    se = b.selfenergy(b.ncoord(xyz))[0].contiguous()
    b.order_pairs(None)
    ref = b.forward(xyz, se)
    b.order_pairs(b.xyz0)
    print(f"[gpu] one translation: {b.unit_counts()}", flush=True)
    assert b.unit_counts()["fwd_far"] > 0 and ref[0].abs().max() > 1e-3
    out = tuple(torch.full_like(r, float("nan")) for r in ref)
    b.forward(xyz, se, out=out)
    for k, (r, g) in enumerate(zip(ref, out)):
        assert torch.isfinite(g).all(), k
        assert torch.abs(r - g).max().item() <= 1e-12, k
