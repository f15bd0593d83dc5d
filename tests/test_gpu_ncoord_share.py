"""Coordination number and its derivative at the sizes where the kernels change:
one wavefront per atom or four (384 pairs an atom on average), molecules walked
directly or lattice images through the queue of 64, a cell of one atom, more
atoms in a cell than lanes.  Against the oracle, cn to 1e-12 and the gradient
and sigma to 1e-8 (absolute)."""
import numpy as np
import pytest

from oracle import oracle as O
from tblite_amd import synthetic

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _cell(nat, side, rng):
    lat = side * (np.diag([1.0, 1.1, 0.9]) + rng.normal(scale=0.03, size=(3, 3)))
    z = rng.choice([1, 6, 8, 17], size=nat).astype(np.int32)
    return (z, rng.uniform(size=(nat, 3)) @ lat), ([True, True, True], lat)


CASES = {
    "molecule_383": lambda r: [(synthetic.water_cluster(128, seed=3), None)],  # 384 atoms
    "molecules_below": lambda r: [(synthetic.water_cluster(127, seed=3), None)],
    "sparse_cells": lambda r: [_cell(1, 60.0, r), _cell(5, 45.0, r)],   # one wavefront, queue
    "dense_cells": lambda r: [_cell(1, 5.0, r), _cell(3, 7.0, r), _cell(64, 22.0, r),
                              _cell(65, 22.0, r)],
    "mixed": lambda r: [_cell(17, 12.0, r), (synthetic.random_molecule(40, r), None),
                        ((np.array([8]), np.zeros((1, 3))), None)],
}


@pytest.mark.parametrize("name", list(CASES))
def test_ncoord_split(name):
    from tblite_amd.batch import Batch
    rng = np.random.default_rng(12)
    structs, lats = zip(*CASES[name](rng))
    b = Batch(list(structs), lattices=list(lats) if any(lat for lat in lats) else None)
    print(f"[gpu] ncoord {name}: atoms {list(b.mol_nat)}", flush=True)
    cn = b.ncoord(b.tensor_xyz()).cpu().numpy()
    dEdcn = rng.normal(size=b.nat)
    grad = torch.zeros(3 * b.nat, dtype=torch.float64, device="cuda")
    sigma = torch.zeros(9 * b.nmol, dtype=torch.float64, device="cuda")
    b.ncoord_gradient(b.tensor_xyz(), torch.tensor(dEdcn, device="cuda"), grad, sigma)
    grad, sigma = grad.cpu().numpy(), sigma.cpu().numpy()
    for m, (z, x) in enumerate(structs):
        a0, a1 = int(b.atom_off[m]), int(b.atom_off[m + 1])
        ref, dr, dl = O.ncoord_dexp(b.ids[a0:a1], np.asarray(x).reshape(-1, 3),
                                    b.molecule_translations(m), b.rcov, derivatives=True)
        assert np.abs(cn[a0:a1] - ref).max() < 1e-12 * max(1.0, np.abs(ref).max()), m
        gr = np.einsum("cji,i->cj", dr, dEdcn[a0:a1])
        sr = np.einsum("abi,i->ab", dl, dEdcn[a0:a1])
        assert np.abs(grad[3 * a0: 3 * a1].reshape(-1, 3).T - gr).max() < 1e-8, m
        assert np.abs(sigma[9 * m: 9 * m + 9].reshape(3, 3, order="F") - sr).max() < 1e-8, m
