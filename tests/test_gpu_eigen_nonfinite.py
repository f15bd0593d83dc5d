"""An infinity or NaN in a molecule's H: NaN for all its results and no error,
by the batched kernels and by the library route (more than 1024 orbitals, or no
room for the kernels' workspace) alike; the other molecules, and entries below
the diagonal, are not concerned.  Their residuals are bounded as in any solve:
20 n u |H| cond(S)."""
import numpy as np
import pytest

from tblite_amd import lib as L

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

U = 2.0 ** -53


def _batch(sizes):
    from tblite_amd.batch import Batch
    mols = []
    for n in sizes:
        g = np.arange(n)
        mols.append((np.ones(n, dtype=np.int32),
                     3.0 * np.stack([g % 11, (g // 11) % 11, g // 121], axis=1)))
    return Batch(mols, order_pairs=False)


def _matrices(n, rng):
    a, q = rng.normal(size=(n, n)), rng.normal(size=(n, n)) / np.sqrt(n)
    return 0.5 * (a + a.T) / np.sqrt(n), np.eye(n) + 0.1 * (q + q.T)


def _pack(mats):
    return torch.tensor(np.concatenate([m.reshape(-1, order="F") for m in mats]), device="cuda")


def _check(b, Hs, Ss, bad):
    C, S = _pack(Hs), _pack(Ss)
    e = b.sygvd(C, S).cpu().numpy()
    c = C.cpu().numpy()
    for m, (H, s) in enumerate(zip(Hs, Ss)):
        n = len(H)
        ev = e[b.ao_off[m]: b.ao_off[m + 1]]
        x = c[b.dense_off[m]: b.dense_off[m + 1]].reshape(n, n, order="F")
        if m in bad:
            assert np.isnan(ev).all() and np.isnan(x).all(), m
            continue
        full = np.triu(H) + np.triu(H, 1).T
        tol = 20 * n * U * np.linalg.norm(full, 2) * np.linalg.cond(s)
        assert np.abs(full @ x - s @ x * ev).max() <= tol, m


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("route", ["sizes", "memory"])
def test_nonfinite_h(value, route):
    rng = np.random.default_rng(9)
    sizes = [30, 1026, 70, 1030, 1] if route == "sizes" else [33, 70, 1, 5]
    b = _batch(sizes)
    pairs = [_matrices(n, rng) for n in sizes]
    Hs, Ss = [p[0] for p in pairs], [p[1] for p in pairs]
    places = {0: (3, 7), 1: (sizes[1] - 1, sizes[1] - 1), len(sizes) - 1: (0, 0)}
    for m, (r, c) in places.items():
        Hs[m][r, c] = value
    if sizes[2] > 1:
        Hs[2][sizes[2] - 1, 0] = value  # below the diagonal
    print(f"[gpu] sygvd with {value}, {route}: orbitals {sizes}", flush=True)
    ctx = L.context(0)
    if route == "memory":
        used = L.lib().tbx_context_memory_used(ctx)
        L.check(L.lib().tbx_context_set_memory_limit(ctx, used + 8 * 70 * 70 + 4096))
    try:
        _check(b, Hs, Ss, set(places))
        Ss[1][4, 4] = -1.0  # not positive definite: an error whatever H holds
        with pytest.raises(L.TbxError, match="molecule 1 "):
            b.sygvd(_pack(Hs), _pack(Ss))
    finally:
        L.check(L.lib().tbx_context_set_memory_limit(ctx, -1))
