"""Raw parameter entries after the number of states of a type has changed."""

import pytest
import torch

from micmec_amd.adjoint import CellParams, DiffField, NPS
from micmec_amd.workloads import make_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", ["corner8", "original"])
def test_entries_of_dropped_states_are_zero(model):
    """Two states, then one: the second state's entries are zeros again, not what the first
    evaluation left, and the others are those of an object that never had it."""
    system = make_system((4, 5, 3), p_b=0.5, seed=3, noise=1.0, strain=0.02)
    used, fresh = DiffField([system], model=model), DiffField([system], model=model)
    pos, rv = used.positions()
    two = used.initial_params()
    assert list(two.nstates) == [1, 2]
    one = CellParams(*two.tensors(), [1, 1], two.type_ids)
    gen = torch.Generator().manual_seed(1)
    dpos = torch.randn(pos.shape, generator=gen, dtype=torch.float64).to(pos.device)
    drv = torch.zeros_like(rv)
    weight = torch.ones(1, dtype=torch.float64, device=pos.device)
    used.set_params(two)
    first = used.adjoint(pos, rv, dpos, drv)
    assert bool((first["params"][1, NPS:2 * NPS] != 0).any())
    used.vjp(pos, rv, weight, dpos)
    for field in (used, fresh):
        field.set_params(one)
    got, want = used.adjoint(pos, rv, dpos, drv), fresh.adjoint(pos, rv, dpos, drv)
    product = used.vjp(pos, rv, weight, dpos)
    for entries in (got["params"], got["dparams"], product["params"], product["dparams"]):
        assert bool((entries[:, NPS:2 * NPS] == 0).all())
    for key in ("params", "dparams"):
        assert torch.equal(got[key], want[key])
