"""The kept self-energy tables serve training, also where they were made under
``torch.inference_mode``: on creation of a batch and after a change of its host
arrays.  No device: a batch's host side, with its tables on the CPU."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")


def _host_batch():
    from tblite_amd.batch import Batch
    rng = np.random.default_rng(7)
    b = object.__new__(Batch)
    b.sh_atom = np.repeat(np.arange(5), [1, 2, 3, 2, 1])
    b.selfenergy_sp, b.kcn_sh = rng.normal(size=9), rng.normal(size=9)
    b._se_tables = {}
    return b


@pytest.mark.parametrize("change", [False, True])
def test_tables_made_under_inference_mode(change):
    b = _host_batch()
    cn = torch.linspace(0.5, 3.0, 5, dtype=torch.float64)
    if change:
        b.selfenergy(cn)
        b.kcn_sh = 2.0 * b.kcn_sh
    with torch.inference_mode():
        assert not b.selfenergy(cn)[0].requires_grad
    cn.requires_grad_(True)
    se, dse = b.selfenergy(cn)
    (g,) = torch.autograd.grad(se.sum(), cn)
    assert torch.equal(dse, torch.as_tensor(-b.kcn_sh))
    # sums of at most three terms
    want = np.bincount(b.sh_atom, weights=-b.kcn_sh)
    assert np.abs(g.numpy() - want).max() <= 4 * 2.0 ** -53 * np.abs(b.kcn_sh).sum()
