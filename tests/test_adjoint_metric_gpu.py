"""The adjoint's parameter derivatives and their tangents against automatic differentiation of the
energy's definition on the CPU, for rest cells of any shape, one to four states a type, both models,
holes, open faces, and numbers of cells around the wave of 64.

Tolerance: strains of 0.2 from lengths of 20 carry a rounding of 1e-16 / 0.2 relative; a cell's
derivative sums some 10^3 products of them, a type's some 10^3 cells with random signs, and the
map to the rest cell multiplies with its condition number (below 2): 1e-11 of the largest entry
leaves a factor of 100."""

import numpy as np
import pytest
import torch

from micmec_amd import units
from micmec_amd.adjoint import DiffField
from micmec_amd.system import System
from micmec_amd.topology import build_system, build_type
from micmec_amd.workloads import CELL_MASS, cubic_elasticity, make_grid

pytestmark = pytest.mark.gpu
TOL = 1e-11
VOIGT = ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))
OFF = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1], [1, 1, 0], [1, 0, 1], [0, 1, 1],
                [1, 1, 1]])


def make(shape, states, seed, p_hole, pbc):
    rng = np.random.default_rng(seed)
    edge = 20.7 * units.angstrom

    def one():
        h = edge * (np.identity(3) + rng.uniform(-0.1, 0.1, (3, 3)))
        c = cubic_elasticity(40.0, 20.0, 10.0)
        x = rng.uniform(-1.0, 1.0, (3, 3, 3, 3)) * 4.0 * units.gigapascal
        x = 0.5 * (x + x.transpose(1, 0, 2, 3))
        x = 0.5 * (x + x.transpose(0, 1, 3, 2))
        return h, c + 0.5 * (x + x.transpose(2, 3, 0, 1))

    many = [one() for _ in range(states)]
    # a temperature at which every state of a strained cell has weight
    data = {1: build_type("A", CELL_MASS, *map(list, zip(one())), effective_temp=300.0),
            2: build_type("B", CELL_MASS, *map(list, zip(*many)),
                          free_energy=list(rng.uniform(0, 1e-3, states)), effective_temp=5.0e6)}
    grid = make_grid(shape, 0.5, p_hole, seed)
    grid.flat[0], grid.flat[1] = 1, 2
    out = build_system(data, grid, pbc=pbc)
    out["pos"] = out["pos"] + rng.normal(0.0, 0.3 * units.angstrom, out["pos"].shape)
    return System.from_dict(out)


def energy(system, model, pos, rvecs, params, nstates):
    """Sum over cells of the definition (nanocell.py, mmff.py:380-398)."""
    cv, h0, free, teff = params
    sn = torch.as_tensor(np.asarray(system.surrounding_nodes), dtype=torch.long)
    p = pos[sn]
    if len(system.domain.rvecs):
        # an edge of more than half the domain wraps
        half = torch.linalg.inv(rvecs)
        frac = (p - p[:, :1]) @ half
        want = torch.as_tensor(OFF / np.array(system.grid.shape))
        p = p + torch.round((want - frac).detach()) @ rvecs
    lo = [[int(np.flatnonzero((OFF == np.where(np.arange(3) == d, 0, o)).all(1))[0])
           for d in range(3)] for o in OFF]
    hi = [[int(np.flatnonzero((OFF == np.where(np.arange(3) == d, 1, o)).all(1))[0])
           for d in range(3)] for o in OFF]
    M = p[:, torch.tensor(hi)] - p[:, torch.tensor(lo)]
    if model == "original":
        M = M.mean(1, keepdim=True)
    types = torch.as_tensor(np.asarray(system.types))
    total = 0.0
    for t in range(cv.shape[0]):
        m = M[types == t + 1]
        es = []
        for s in range(int(nstates[t])):
            B = torch.linalg.inv(h0[t, s]) @ m
            eps = 0.5 * (B @ B.transpose(-1, -2) - torch.eye(3, dtype=torch.float64))
            e = torch.stack([eps[..., i, j] * (1.0 if i == j else 2.0) for i, j in VOIGT], -1)
            u = 0.5 * ((e @ cv[t, s]) * e).sum(-1).mean(-1)
            es.append(torch.linalg.det(h0[t, s]) * u + free[t, s])
        es = torch.stack(es, -1)
        kt = units.boltzmann * teff[t]
        total = total + (es[..., 0] if es.shape[-1] == 1
                         else -kt * torch.logsumexp(-es / kt, -1)).sum()
    return total


def close(a, b, what):
    a, b = a.detach().cpu(), b.detach().cpu()
    scale = float(b.abs().max())
    assert float((a - b).abs().max()) <= TOL * max(scale, 1e-300), (what, scale)


@pytest.mark.parametrize("model", ["corner8", "original"])
@pytest.mark.parametrize("shape,states,p_hole,pbc", [
    ((2, 2, 2), 1, 0.0, True), ((4, 4, 8), 2, 0.0, True), ((3, 5, 9), 3, 0.2, False),
    ((8, 8, 9), 4, 0.1, True)])
def test_parameter_derivatives_and_tangents(shape, states, p_hole, pbc, model):
    print("adjoint metric", shape, states, model, flush=True)
    system = make(shape, states, 7, p_hole, pbc)
    field = DiffField([system], model=model)
    pos, rv = field.positions()
    p = field.initial_params()
    gen = torch.Generator().manual_seed(5)
    dpos = torch.randn(pos.shape, generator=gen, dtype=torch.float64)
    drv = torch.randn(rv.shape, generator=gen, dtype=torch.float64) * (1.0 if pbc else 0.0)
    out = field.adjoint(pos, rv, dpos.to(pos.device), drv.to(pos.device))
    values = field.param_grads(out["params"], p)
    tangents = field.param_grads(out["dparams"], p)

    leaves = [t.detach().cpu().clone().requires_grad_(True)
              for t in (pos, rv[0], *p.tensors())]
    e = energy(system, model, leaves[0], leaves[1], leaves[2:], p.nstates)
    first = torch.autograd.grad(e, leaves, create_graph=True, allow_unused=True)
    g_pos, g_rv = first[:2]
    close(out["energy"], e.reshape(1), "energy")
    close(out["gpos"], g_pos, "gpos")
    along = (g_pos * dpos).sum()
    if pbc:
        close(out["grvecs"][0], g_rv, "grvecs")
        along = along + (g_rv * drv[0]).sum()
    second = torch.autograd.grad(along, leaves, allow_unused=True)
    close(out["dgpos"], second[0], "dgpos")
    names = ("cv", "h0", "free", "teff")
    for k, name in enumerate(names):
        for mine, ref in ((values[k], first[2 + k]), (tangents[k], second[2 + k])):
            if ref is None:
                ref = torch.zeros_like(leaves[2 + k])
            if name == "cv":  # the gradient of symmetric perturbations
                ref = 0.5 * (ref + ref.transpose(-1, -2))
                mine = mine.cpu()
            close(mine, ref, name)
