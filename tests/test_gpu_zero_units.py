"""Forward with a pair-order hint: the zero blocks of distant pairs go out in
runs down the columns.  Molecules whose runs are one row, a run's limit of 128
rows, one below and one above it, several runs, and none at all; the hint
valid, and stale (the far units run instead).  Every element is written,
and all agree with the forward without a hint to 1e-12 (the same sums for every
element, of values up to 1e2)."""
import numpy as np
import pytest

from tblite_amd import synthetic

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _split(za, zb):
    """Atoms of za on one line and of zb on another, 60 bohr away."""
    xyz = [(0.0, 0.0, 2.5 * k) for k in range(len(za))]
    xyz += [(60.0, 0.0, 2.5 * k) for k in range(len(zb))]
    return np.array(list(za) + list(zb), dtype=np.int32), np.array(xyz)


def _interleaved(n):
    """Neighbours in the atom order are 60 bohr apart: runs of one atom."""
    xyz = [(60.0 * (k % 2), 0.0, 2.0 * (k // 2)) for k in range(n)]
    return np.ones(n, dtype=np.int32), np.array(xyz)


def _structures():
    rows = [_split([1], [1] * n) for n in (1, 63, 64, 127, 128, 129, 257)]
    mixed = [_split([8, 17, 1], [6, 1, 53, 8]), _split([26] * 5, [1] * 131), _interleaved(65)]
    near = [(np.array([8, 1, 1], dtype=np.int32), np.array([[0, 0, 0], [0, 0, 1.8], [1.7, 0, -.5]]))]
    return rows + mixed + near + [synthetic.water_cluster(128, seed=3)]


@pytest.mark.parametrize("stale", [False, True])
def test_zero_runs(stale):
    from tblite_amd.batch import Batch
    structs = _structures()
    b = Batch(structs)
    b.set_tiles(fwd_unit_tasks=100)  # enough units for the hint to be used
    xyz = b.tensor_xyz()
    se = b.selfenergy(b.ncoord(xyz))[0]
    b.order_pairs(None)
    ref = b.forward(xyz, se)
    hint = b.xyz0.copy()
    if stale:
        hint[-1] += 30.0
    b.order_pairs(hint, skin=0.5)
    print(f"[gpu] zero runs, stale {stale}: {b.ndense} elements", flush=True)
    for _ in range(2):
        out = tuple(torch.full_like(r, float("nan")) for r in ref)
        b.forward(xyz, se, out=out)
        torch.cuda.synchronize()
        for k, (r, g) in enumerate(zip(ref, out)):
            assert torch.isfinite(g).all(), k
            assert torch.abs(r - g).max().item() <= 1e-12, k
