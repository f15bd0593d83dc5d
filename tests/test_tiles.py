"""The tiles a batch reports are those it runs: a batch that does not fill the
device starts with smaller units, the planner checks these, they survive a
set_tiles that changes something else, and the autotuner times them too."""
import numpy as np
import pytest

from tblite_amd import synthetic

torch = pytest.importorskip("torch")

DEFAULT = dict(fwd_unit_tasks=256, fwd_unit_pairs=128, fwd_chunk=3, grad_unit_tasks=256,
               grad_unit_pairs=128, grad_chunk=1)


@pytest.mark.parametrize("hint", [False, True])
def test_planner_checks_the_units_of_a_small_batch(hint):
    from tblite_amd.batch import plan_stats
    for mols in ([synthetic.octane()], [synthetic.water_cluster(40, seed=1)],
                 [synthetic.mixed_cluster(30, seed=4), synthetic.water_cluster(3, seed=2)]):
        small, full = plan_stats(mols, hint=hint), plan_stats(mols, DEFAULT, hint=hint)
        for st in (small, full):
            assert st["bad_pairs"] == st["bad_elems"] == st["bad_units"] == 0, st
            assert st["nelem"] == st["ndense"]
        assert small["nunit_fwd"] > full["nunit_fwd"] and small["nunit_grad"] > full["nunit_grad"]
        assert small["ntask_fwd"] == full["ntask_fwd"]


@pytest.mark.gpu
def test_tiles_round_trip():
    from tblite_amd import tune
    from tblite_amd.batch import Batch
    b = Batch([synthetic.octane(), synthetic.water_cluster(12, seed=1)])
    n, t = b.unit_counts(), b.tiles()
    print(f"[gpu] tiles {t}, units {n}", flush=True)
    assert t["fwd_unit_tasks"] < 256 and t["grad_unit_tasks"] < 256
    b.set_tiles(**t)
    assert b.unit_counts() == n
    b.set_tiles(fwd_chunk=2)
    assert b.unit_counts() == n and b.tiles() == {**t, "fwd_chunk": 2}
    b.order_pairs(b.xyz0)
    b.order_pairs(None)
    assert b.unit_counts() == n
    b.set_tiles(fwd_unit_tasks=256, grad_unit_tasks=256)
    assert b.unit_counts()["fwd_near"] < n["fwd_near"]
    b.set_tiles(**t)
    xyz = b.tensor_xyz()
    se = b.selfenergy(b.ncoord(xyz))[0].contiguous()
    adj = [torch.ones(k * b.ndense, dtype=torch.float64, device="cuda") for k in (1, 3, 6, 1)]
    res = tune.tune(b, xyz, se, adj, reps=1, chunks=(1, 3))
    for key in ("fwd_unit_tasks", "grad_unit_tasks"):
        assert {r[key] for r in res["table"][:-3]} == {t[key], 192, 256}
