"""The cell pass in the metric of the edges: general rest cells and elasticity against the oracle,
and the same energies and virials whatever outputs a call asks for."""

import numpy as np
import pytest
import torch

from micmec_amd import units
from micmec_amd.pes import ForcePartMechanical
from micmec_amd.system import System
from micmec_amd.topology import build_system, build_type
from micmec_amd.workloads import CELL_MASS, cubic_elasticity, make_grid, make_system

from test_force_gpu import TOL, gpu_eval, oracle_eval, rel

pytestmark = pytest.mark.gpu


def skewed_system(shape, states, seed, p_hole=0.0, pbc=True):
    """Two types, of one and of `states` states: triclinic rest cells (up to 15% off the cube) and
    elasticity tensors without major symmetry (10% noise, minor symmetries kept)."""
    rng = np.random.default_rng(seed)
    edge = 20.7 * units.angstrom

    def one():
        h = edge * (np.identity(3) + rng.uniform(-0.15, 0.15, (3, 3)))
        c = cubic_elasticity(40.0, 20.0, 10.0)
        x = rng.uniform(-1.0, 1.0, (3, 3, 3, 3)) * 4.0 * units.gigapascal
        x = 0.5 * (x + x.transpose(1, 0, 2, 3))
        return h, c + 0.5 * (x + x.transpose(0, 1, 3, 2))
    many = [one() for _ in range(states)]
    data = {1: build_type("A", CELL_MASS, *map(list, zip(one())), effective_temp=300.0),
            2: build_type("B", CELL_MASS, *map(list, zip(*many)),
                          free_energy=list(rng.uniform(0, 1e-3, states)), effective_temp=300.0)}
    grid = make_grid(shape, 0.5, p_hole, seed)
    grid.flat[0], grid.flat[1] = 1, 2
    out = build_system(data, grid, pbc=pbc)
    out["pos"] = out["pos"] + rng.normal(0.0, 0.3 * units.angstrom, out["pos"].shape)
    return System.from_dict(out)


# one block; several with remainders; the longest state loop; more than 512 blocks (two instances)
@pytest.mark.parametrize("model", ["corner8", "original"])
@pytest.mark.parametrize("shape,states,p_hole,pbc", [
    ((2, 2, 3), 2, 0.0, True), ((7, 5, 11), 3, 0.2, True), ((6, 9, 65), 8, 0.0, False),
    ((51, 52, 53), 2, 0.05, True)])
def test_general_cells_against_oracle(shape, states, p_hole, pbc, model):
    print(shape, states, model, flush=True)
    s = skewed_system(shape, states, 5, p_hole, pbc)
    for got, want in zip(gpu_eval(s, model), oracle_eval(s, model)):
        assert rel(got, want) < TOL


@pytest.mark.parametrize("model", ["corner8", "original"])
@pytest.mark.parametrize("shape", [(3, 4, 5), (52, 51, 53)])
def test_same_bits_for_every_output(shape, model):
    s = skewed_system(shape, 3, 9, 0.1)
    fpm = ForcePartMechanical(s, model=model)
    kw = dict(dtype=torch.float64, device=fpm.device)
    pos = torch.tensor(np.asarray(s.pos), **kw)
    rv = torch.tensor(np.asarray(s.domain.rvecs), **kw)

    def call(want_g, want_v):
        e = torch.zeros(1, **kw)
        g = torch.zeros(pos.shape, **kw) if want_g else None
        v = torch.zeros((3, 3), **kw) if want_v else None
        fpm.compute_device(pos, rv, e, g, v)
        return e, g, v
    e, g, v = call(True, True)
    e1, _, v1 = call(False, True)
    e2, g2, _ = call(True, False)
    e3, _, _ = call(False, False)
    assert torch.equal(v, v1) and torch.equal(g, g2)
    assert torch.equal(e, e1) and torch.equal(e, e2) and torch.equal(e, e3)
    assert torch.equal(v, v.t())


def test_virial_of_small_strains():
    """A crystal of two-state cells with thermal noise only: its mean strain, and with it the virial,
    is of second order in the noise (some 1e-5), so an error that all cells share, a rounding of
    the rest metric of 1e-17 to 1e-16, would show as 1e-12 to 1e-11. The roundings of 5e-17 a cell
    average out to 5e-17 / sqrt(15000) / 1e-5 = 4e-14; ten times that is allowed."""
    s = make_system((9, 50, 34), p_b=1.0, seed=6, noise=0.05 * units.angstrom)
    assert rel(gpu_eval(s, "corner8")[2], oracle_eval(s, "corner8")[2]) < 4e-13
