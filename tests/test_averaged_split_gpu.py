"""The averaged model's cell pass as one launch and, in large fields, as two side by side."""

import pytest
import torch

from micmec_amd.adjoint import DiffField
from micmec_amd.workloads import make_system

pytestmark = pytest.mark.gpu


def test_one_and_two_launches_give_the_same_bits():
    """A system of 1275 cell blocks by itself, and four of it in one field (5100, two launches)."""
    s = make_system((70, 70, 70), p_b=0.3, p_hole=0.05, seed=8, strain=0.02)
    one, four = DiffField([s], model="original"), DiffField([s] * 4, model="original")
    e, g, v = one.compute(*one.positions())
    E, G, V = four.compute(*four.positions())
    assert float(e) != 0.0 and bool((g != 0.0).any())
    for k in range(4):
        a = int(four.node_start[k])
        assert torch.equal(E[k], e[0]) and torch.equal(V[k], v[0])
        assert torch.equal(G[a:a + s.nnodes], g[:s.nnodes])
