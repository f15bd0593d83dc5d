"""An S that is not positive definite, with the pivot that shows it in every
block of 64 rows of the batched Cholesky factorisation, at its edges and in the
first and the last row: the call names the molecule (the first, where two fail)
and the next call is not concerned.  Residuals as in any solve: 20 n u |H| cond(S)."""
import numpy as np
import pytest

from tblite_amd import lib as L

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

U = 2.0 ** -53
SIZES = [300, 41, 129]


def _pack(mats):
    return torch.tensor(np.concatenate([m.reshape(-1, order="F") for m in mats]), device="cuda")


def test_not_positive_definite():
    from tblite_amd.batch import Batch
    rng = np.random.default_rng(15)
    mols = []
    for n in SIZES:
        g = np.arange(n)
        mols.append((np.ones(n, dtype=np.int32),
                     3.0 * np.stack([g % 11, (g // 11) % 11, g // 121], axis=1)))
    b = Batch(mols, order_pairs=False)
    Hs, Ss = [], []
    for n in SIZES:
        a, q = rng.normal(size=(n, n)), rng.normal(size=(n, n)) / np.sqrt(n)
        Hs.append(0.5 * (a + a.T) / np.sqrt(n))
        Ss.append(np.eye(n) + 0.1 * (q + q.T))
    for m, rows in ((0, (0, 63, 64, 127, 130, 200, 299)), (1, (0, 40)), (2, (63, 128))):
        for r in rows:
            for value in (-1.0, 0.0, np.nan):
                bad = [s.copy() for s in Ss]
                bad[m][r, r] = value
                if m == 0:
                    bad[2][5, 5] = -2.0
                print(f"[gpu] sygvd: molecule {m} of {SIZES}, S({r}, {r}) = {value}", flush=True)
                with pytest.raises(L.TbxError, match=f"molecule {m} "):
                    b.sygvd(_pack(Hs), _pack(bad))
        C = _pack(Hs)
        e, c = b.sygvd(C, _pack(Ss)).cpu().numpy(), C.cpu().numpy()
        for k, (H, S) in enumerate(zip(Hs, Ss)):
            n = len(H)
            x = c[b.dense_off[k]: b.dense_off[k + 1]].reshape(n, n, order="F")
            tol = 20 * n * U * np.linalg.norm(H, 2) * np.linalg.cond(S)
            assert np.abs(H @ x - S @ x * e[b.ao_off[k]: b.ao_off[k + 1]]).max() <= tol, (m, k)
