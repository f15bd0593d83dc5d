"""The density products where occupations are exactly zero: their orbitals are
left out of the products (compacted in chunks of 256), but an infinity or NaN
in one of them still reaches P, as 0 * C does.

Tolerance: the rounding of a sum of n products, 2 n u sum_k |f_k C_ik C_jk|
(u = 2^-53)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

U = 2.0 ** -53
SIZES = [1, 2, 16, 17, 63, 64, 65, 130, 255, 256, 257, 300, 530]


@pytest.fixture(scope="module")
def batch():
    from tblite_amd.batch import Batch
    mols = []
    for n in SIZES:  # n hydrogen atoms: n orbitals
        g = np.arange(n)
        mols.append((np.ones(n, dtype=np.int32),
                     3.0 * np.stack([g % 11, (g // 11) % 11, g // 121], axis=1)))
    return Batch(mols, order_pairs=False)


def _occupations(kind, n, rng):
    f = rng.uniform(0.1, 2.0, n)
    if kind == "none":
        return np.zeros(n)
    if kind == "half":
        f[(n + 1) // 2:] = 0.0
    if kind == "alternate":
        f[1::2] = 0.0
    if kind == "last":  # only the last one occupied
        f[:-1] = 0.0
    return f


@pytest.mark.parametrize("spoil", [False, True])
@pytest.mark.parametrize("kind", ["all", "half", "alternate", "last", "none"])
def test_zero_occupations(batch, kind, spoil):
    b, rng = batch, np.random.default_rng(3)
    print(f"[gpu] density, occupations {kind}, spoiled {spoil}", flush=True)
    Cs = [rng.normal(size=(n, n)) / np.sqrt(n) for n in SIZES]
    fs = [_occupations(kind, n, rng) for n in SIZES]
    es = [rng.normal(size=n) for n in SIZES]
    if spoil:  # one element of a column in every other molecule
        for k, C in enumerate(Cs):
            n = len(C)
            if k % 2:
                C[n // 2, n - 1 - (kind == "last")] = np.nan if k % 4 == 1 else np.inf
    t = lambda v: torch.tensor(np.concatenate([x.reshape(-1, order="F") for x in v]),  # noqa: E731
                               device="cuda")
    C, f, e = t(Cs), t(fs), t(es)
    P, W = b.density_matrix(C, f).cpu().numpy(), b.wdensity(C, f, e).cpu().numpy()
    for m, n in enumerate(SIZES):
        d0 = int(b.dense_off[m])
        for got, w in ((P, fs[m]), (W, fs[m] * es[m])):
            got = got[d0: d0 + n * n].reshape(n, n, order="F")
            with np.errstate(invalid="ignore"):
                ref = (Cs[m] * w) @ Cs[m].T
                bound = 2 * n * U * (np.abs(Cs[m] * w) @ np.abs(Cs[m]).T)
            fine = np.isfinite(ref)
            assert np.array_equal(np.isnan(got), np.isnan(ref)), (n, kind)
            assert np.all(np.abs(got - ref)[fine] <= bound[fine]), (n, kind)
