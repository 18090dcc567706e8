"""The fused force-and-stress loss and the one-call backward pass against the same terms composed
in torch from ``micmec_energy`` (whose own derivatives are checked elsewhere)."""

import numpy as np
import pytest
import torch

from micmec_amd import units
from micmec_amd.adjoint import CellParams, DiffField, FitProblem, micmec_energy
from micmec_amd.workloads import make_system

pytestmark = pytest.mark.gpu
A = units.angstrom
# both sides round the same sums of up to 1e6 terms in other orders: 1e-16 times the square root
# of their number, times the few hundred that strains of a percent lose in differences
TOL = 1e-11


def problem_of(shapes, model):
    systems = [make_system(s, p_b=0.4, p_hole=0.05, seed=20 + i, noise=0.1 * A, strain=0.03)
               for i, s in enumerate(shapes)]
    field = DiffField(systems, model=model)
    pos, rv = field.positions()
    target = field.initial_params()
    target.cv = target.cv * 1.07
    return FitProblem(field, pos, rv, target)


def leaves_of(problem):
    p = problem.field.initial_params()
    return [t.detach().clone().requires_grad_(True)
            for t in (problem.pos, problem.rvecs) + p.tensors()], p


def close(a, b):
    scale = float(b.abs().max())
    assert float((a - b).abs().max()) <= TOL * max(scale, 1e-300)


# one small system; uneven ones with padding rows; more nodes than the loss has blocks for
@pytest.mark.parametrize("model", ["corner8", "original"])
@pytest.mark.parametrize("shapes", [[(2, 3, 2)], [(3, 4, 5), (6, 6, 7), (2, 2, 2)],
                                    [(73, 70, 75)]])
def test_fused_loss(shapes, model):
    print(shapes, model, flush=True)
    problem = problem_of(shapes, model)
    leaves, p = leaves_of(problem)
    problem.pos, problem.rvecs = leaves[:2]
    loss = problem.loss(CellParams(*leaves[2:], p.nstates, p.type_ids))
    got = torch.autograd.grad(3.0 * loss, leaves)
    other, p = leaves_of(problem)
    _, g, v = micmec_energy(problem.field, other[0], other[1],
                            CellParams(*other[2:], p.nstates, p.type_ids))
    inv = (1.0 / problem.volume)[:, None, None]
    want = ((g + problem.f_target) ** 2).mean() / problem.f_scale + \
        ((v * inv + problem.s_target) ** 2).mean() / problem.s_scale
    close(loss.detach(), want.detach())
    for a, b in zip(got, torch.autograd.grad(3.0 * want, other)):
        assert a.shape == b.shape
        close(a, b)


@pytest.mark.parametrize("needed", [[0], [1], [2], [0, 5], [3, 4]])
def test_only_what_is_needed(needed):
    """Any subset of the inputs gives the same gradients as all of them."""
    problem = problem_of([(3, 4, 3), (4, 4, 4)], "corner8")
    leaves, p = leaves_of(problem)
    gen = torch.Generator().manual_seed(2)
    wG = torch.randn(leaves[0].shape, generator=gen, dtype=torch.float64).to(leaves[0].device)

    def value(ts, fused):
        q = CellParams(*ts[2:], p.nstates, p.type_ids)
        if fused:
            problem.pos, problem.rvecs = ts[:2]
            return problem.loss(q)
        return (micmec_energy(problem.field, ts[0], ts[1], q)[1] * wG).sum()
    for fused in (True, False):
        every = torch.autograd.grad(value(leaves, fused), leaves)
        some = [t if i in needed else t.detach() for i, t in enumerate(leaves)]
        got = torch.autograd.grad(value(some, fused), [leaves[i] for i in needed])
        for i, a in zip(needed, got):
            assert torch.equal(a, every[i])


def test_double_backward_is_refused():
    problem = problem_of([(3, 3, 3)], "corner8")
    leaves, p = leaves_of(problem)
    loss = problem.loss(CellParams(*leaves[2:], p.nstates, p.type_ids))
    (g,) = torch.autograd.grad(loss, leaves[2], create_graph=True)
    with pytest.raises(RuntimeError):
        g.sum().backward()


def test_invalid_arguments():
    field = problem_of([(2, 2, 2)], "corner8").field
    from micmec_amd import _native
    n = [None]
    assert field.lib.mm_fit_loss(None, *n * 5, 1.0, 1.0, None, None) == _native.MM_ERR_ARG
    assert field.lib.mm_fit_loss(field._adj, *n * 5, 1.0, 1.0, None, None) == _native.MM_ERR_ARG
    assert field.lib.mm_adjoint_backward(field._adj, *n * 7, 1.0, *n * 7) == _native.MM_ERR_ARG
    pos, rv = field.positions()
    P = _native.ptr
    one = torch.zeros(field.nsys, dtype=torch.float64, device=pos.device)
    # the parameter gradients go together
    assert field.lib.mm_adjoint_backward(field._adj, P(pos), P(rv), P(field._node_sys32), P(one),
                                         None, None, None, 1.0, None, None, P(one), None, None,
                                         None, None) == _native.MM_ERR_ARG
    assert np.isfinite(float(one.sum()))
