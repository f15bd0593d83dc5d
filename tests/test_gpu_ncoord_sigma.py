"""Coordination-number derivative where the atoms of a workgroup share their
sum of sigma: molecules that begin and end within a workgroup, at the launch
shapes of small molecules (four atoms a workgroup), of many atoms with many
pairs (two), and of few atoms with many (one).  Against the oracle, the gradient
and sigma to 1e-8 (absolute)."""
import numpy as np
import pytest

from oracle import oracle as O
from tblite_amd import synthetic

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

H2 = (np.array([1, 1], dtype=np.int32), np.array([[0.0, 0.0, 0.0], [0.0, 0.0, 1.4]]))
CASES = {
    "four": lambda r: [synthetic.random_molecule(n, r) for n in (2, 3, 5, 4, 9, 8, 2, 6)],
    "two_1026": lambda r: [synthetic.water_cluster(342, seed=3)],
    "two_halves": lambda r: [synthetic.water_cluster(171, seed=3),
                             synthetic.water_cluster(171, seed=4)],  # 513 atoms each
    "two_1025": lambda r: [synthetic.water_cluster(341, seed=3), H2],
    "one_939": lambda r: [synthetic.water_cluster(150, seed=3), synthetic.water_cluster(163, seed=5)],
}


@pytest.mark.parametrize("name", list(CASES))
def test_sigma_shared(name):
    from tblite_amd.batch import Batch
    rng = np.random.default_rng(12)
    mols = CASES[name](rng)
    b = Batch(mols, order_pairs=False)
    print(f"[gpu] ncoord sigma {name}: atoms {list(b.mol_nat)}", flush=True)
    dEdcn = rng.normal(size=b.nat)
    grad = torch.zeros(3 * b.nat, dtype=torch.float64, device="cuda")
    sigma = torch.zeros(9 * b.nmol, dtype=torch.float64, device="cuda")
    b.ncoord_gradient(b.tensor_xyz(), torch.tensor(dEdcn, device="cuda"), grad, sigma)
    grad, sigma = grad.cpu().numpy(), sigma.cpu().numpy()
    for m, (z, x) in enumerate(mols):
        a0, a1 = int(b.atom_off[m]), int(b.atom_off[m + 1])
        _, dr, dl = O.ncoord_dexp(b.ids[a0:a1], np.asarray(x).reshape(-1, 3),
                                  b.molecule_translations(m), b.rcov, derivatives=True)
        gr = np.einsum("cji,i->cj", dr, dEdcn[a0:a1])
        sr = np.einsum("abi,i->ab", dl, dEdcn[a0:a1])
        assert np.abs(grad[3 * a0: 3 * a1].reshape(-1, 3).T - gr).max() < 1e-8, m
        assert np.abs(sigma[9 * m: 9 * m + 9].reshape(3, 3, order="F") - sr).max() < 1e-8, m
