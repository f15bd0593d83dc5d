"""The batched generalized eigensolver (tbx_batch_sygvd) on matrices given
directly, at the sizes where its kernels change: blocks of 64 rows, the 128
columns of the tridiagonal form held in LDS, leaves of 64 rows and their
merges, the register rows of the back-transformation, the library route above
1024 orbitals.  A molecule of k hydrogen atoms has k orbitals, so the batch
carries any sizes.

Matrices: dense with spread eigenvalues, block copies (every eigenvalue
several times), diagonal, all zero, and a chain of weakly coupled equal blocks
(clusters).  Tolerance, from the backward error of the Householder
tridiagonal form and the triangular solves: 20 n u |H| cond(S) for the
eigenvalues and residuals, 20 n u cond(S) for C^T S C = 1 (u = 2^-53)."""
import sys

import numpy as np
import pytest
import scipy.linalg

from tblite_amd import lib as L

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

U = 2.0 ** -53
SIZES = [1, 2, 3, 5, 17, 33, 63, 64, 65, 66, 100, 127, 128, 129, 130, 192, 193, 256, 257, 385,
         512, 513, 700, 769, 1024]


def _batch(sizes):
    from tblite_amd.batch import Batch
    mols = []
    for n in sizes:
        g = np.arange(n)
        mols.append((np.ones(n, dtype=np.int32),
                     3.0 * np.stack([g % 11, (g // 11) % 11, g // 121], axis=1)))
    return Batch(mols, order_pairs=False)


def _matrices(kind, n, rng):
    q = rng.normal(size=(n, n)) / np.sqrt(n)
    s = np.eye(n) + 0.2 * (q + q.T) / 2
    if kind == "dense":
        a = rng.normal(size=(n, n))
        return 0.5 * (a + a.T) / np.sqrt(n), s
    if kind == "copies":  # equal diagonal blocks
        m = max(1, n // 7)
        a = rng.normal(size=(m, m))
        blk = 0.5 * (a + a.T)
        return scipy.linalg.block_diag(*[blk[: min(m, n - k), : min(m, n - k)]
                                         for k in range(0, n, m)]), np.eye(n)
    if kind == "diagonal":
        return np.diag(np.round(rng.normal(size=n), 1)), np.eye(n)
    if kind == "zero":
        return np.zeros((n, n)), s
    t = np.diag(np.abs(np.arange(n) % 21 - 10.0))  # glued Wilkinson matrices
    off = np.where((np.arange(1, n) % 21) == 0, 1e-9, 1.0)
    return t + np.diag(off, 1) + np.diag(off, -1), np.eye(n)


def _pack(mats):
    return torch.tensor(np.concatenate([m.reshape(-1, order="F") for m in mats]), device="cuda")


def _blocks(t, b):
    h = t.cpu().numpy()
    return [h[d0:d1].reshape(n, n, order="F") for d0, d1, n in
            zip(b.dense_off[:-1], b.dense_off[1:], np.diff(b.ao_off))]


def _check(b, Hs, Ss, C, e):
    e_h = e.cpu().numpy()
    for m, (H, S, c) in enumerate(zip(Hs, Ss, _blocks(C, b))):
        n = len(H)
        ev = e_h[b.ao_off[m]: b.ao_off[m + 1]]
        cond = np.linalg.cond(S)
        norm = max(np.linalg.norm(H, 2), 1e-300)
        tol = 20 * n * U * cond
        assert np.all(np.diff(ev) >= 0.0), (m, n)
        assert np.abs(ev - scipy.linalg.eigh(H, S, eigvals_only=True)).max() <= tol * norm, (m, n)
        assert np.abs(c.T @ S @ c - np.eye(n)).max() <= tol, (m, n)
        assert np.abs(H @ c - S @ c * ev[None]).max() <= tol * norm, (m, n)


@pytest.mark.parametrize("kind", ["dense", "copies", "diagonal", "zero", "glued"])
def test_sizes(kind):
    rng = np.random.default_rng(77)
    b = _batch(SIZES)
    pairs = [_matrices(kind, n, rng) for n in SIZES]
    Hs, Ss = [p[0] for p in pairs], [p[1] for p in pairs]
    print(f"[gpu] sygvd {kind}: orbitals {SIZES}", flush=True)
    sys.stdout.flush()
    # only the upper triangles are read
    C = _pack([np.triu(h) + np.tril(np.full_like(h, 7.0), -1) for h in Hs])
    S = _pack([np.triu(s) + np.tril(np.full_like(s, 9.0), -1) for s in Ss])
    keep = S.clone()
    e = b.sygvd(C, S)
    assert torch.equal(S, keep)
    _check(b, Hs, Ss, C, e)


def test_refusals_and_library_route():
    rng = np.random.default_rng(5)
    sizes = [40, 1030, 150]
    b = _batch(sizes)
    pairs = [_matrices("dense", n, rng) for n in sizes]
    print(f"[gpu] sygvd: orbitals {sizes}, refusals", flush=True)
    Hs, Ss = [p[0] for p in pairs], [p[1] for p in pairs]
    C = _pack(Hs)
    _check(b, Hs, Ss, C, b.sygvd(C, _pack(Ss)))
    # without room for the kernels' workspace the library takes all of them
    ctx = L.context(0)
    b2 = _batch([40, 70])
    used = L.lib().tbx_context_memory_used(ctx)
    L.check(L.lib().tbx_context_set_memory_limit(ctx, used + 8 * 70 * 70 + 4096))
    try:
        C = _pack([Hs[0], Hs[2][:70, :70]])
        e = b2.sygvd(C, _pack([Ss[0], Ss[2][:70, :70]]))
    finally:
        L.check(L.lib().tbx_context_set_memory_limit(ctx, -1))
    _check(b2, [Hs[0], Hs[2][:70, :70]], [Ss[0], Ss[2][:70, :70]], C, e)
    # an S that is not positive definite names its molecule
    bad = [s.copy() for s in Ss]
    bad[2][149, 149] = -1.0
    with pytest.raises(L.TbxError, match="molecule 2"):
        b.sygvd(_pack(Hs), _pack(bad))
    # a NaN in one H stays in its molecule
    nan = [h.copy() for h in Hs]
    nan[0][3, 7] = nan[0][7, 3] = np.nan
    C = _pack(nan)
    e = b.sygvd(C, _pack(Ss)).cpu().numpy()
    assert np.isnan(e[:40]).all() and np.isfinite(e[40:]).all()
    assert np.isnan(_blocks(C, b)[0]).all()
