"""Virials of small strains about rest cells that are no boxes, against extended precision.

The crystals have thermal noise only: their mean strain, and with it the virial, is of second order
in the noise, 3 (0.05 / 24.01)^2 = 1.3e-5 of the edges' metric and a quarter of that for the averaged
matrix. An error that all cells share does not average out of it: off-diagonal entries of the rest
metric that are rounded once, by 4e-17 (60 degrees) and 1.5e-16 (sheared) of a strain with this edge,
show as 5e-13 of the virial and more. The cells' own roundings of 1e-16 do average out, to 1e-16 /
sqrt(75600) / 1.3e-5 = 2.8e-14; six times that is allowed, four times as much for the averaged
matrix."""

import numpy as np
import pytest

from micmec_amd import units
from micmec_amd.system import System
from micmec_amd.topology import Grid, build_system, build_type
from micmec_amd.workloads import CELL_MASS, cubic_elasticity, make_grid

from test_adjoint_metric_gpu import OFF, VOIGT
from test_force_gpu import gpu_eval

pytestmark = pytest.mark.gpu
TOL = {"corner8": 1.7e-13, "original": 6.7e-13}
EDGE = 24.01 * units.angstrom
CELLS = {"60 degrees": np.array([[1.0, 0.0, 0.0], [0.5, 0.75 ** 0.5, 0.0], [0.0, 0.0, 1.0]]),
         "sheared": np.array([[1.0, 0.0, 0.0], [1.0, 1.0, 0.0], [0.3, 1.0, 1.0]])}


def crystal(h, states, shape=(18, 70, 60)):
    rest = [h * EDGE * f for f in (0.97, 1.0)[2 - states:]]  # the last is the crystal's
    data = {1: build_type("A", CELL_MASS, rest, [cubic_elasticity(30.0, 10.0, 20.0)] * states,
                          free_energy=[0.0] * states, effective_temp=300.0)}
    out = build_system(data, make_grid(shape, 0.0, 0.0, 1), pbc=True)
    # the boxes' lattice turned into that of the rest cell
    ijk = np.rint(out["pos"] / (out["rvecs"].diagonal() / shape))
    out["pos"], out["rvecs"] = ijk @ rest[-1], np.array(shape)[:, None] * rest[-1]
    rng = np.random.default_rng(3)
    out["pos"] = out["pos"] + rng.normal(0.0, 0.05 * units.angstrom, out["pos"].shape)
    return System.from_dict(out)


def inverse(h):
    """By cofactors, every operation rounded, as the parameter table has it."""
    c = np.array([[h[(i + 1) % 3, (j + 1) % 3] * h[(i + 2) % 3, (j + 2) % 3] -
                   h[(i + 1) % 3, (j + 2) % 3] * h[(i + 2) % 3, (j + 1) % 3]
                   for i in range(3)] for j in range(3)])
    det = h[0, 0] * c[0, 0] + h[0, 1] * c[1, 0] + h[0, 2] * c[2, 0]
    return c / det, det


def virial(system, model):
    """Sum of B^T sigma B over corners, the states weighted (nanocell.py, mmff.py:380-398)."""
    L = np.longdouble
    shape = np.rint(np.asarray(system.grid)).astype(int).shape
    pos, rvecs = np.asarray(system.pos).astype(L), np.asarray(system.domain.rvecs).astype(L)
    sn = np.asarray(system.surrounding_nodes)
    wrap = Grid(np.ones(shape, int)).wrap_bits()
    p = pos[sn]
    for d in range(3):
        last = ((wrap >> d) & 1).astype(L)
        p = p + (OFF[:, d].astype(L) * last[:, None])[..., None] * rvecs[d]
    corner = {tuple(o): k for k, o in enumerate(OFF)}
    M = np.stack([np.stack([p[:, corner[tuple(np.where(np.arange(3) == d, 1, o))]] -
                            p[:, corner[tuple(np.where(np.arange(3) == d, 0, o))]]
                            for d in range(3)], 1) for o in OFF], 1)
    if model == "original":
        M = M.mean(1, keepdims=True)
    cells = np.asarray(system.params["type1/cell"], float).reshape(-1, 3, 3)
    stiff = np.asarray(system.params["type1/elasticity"], float).reshape(-1, 3, 3, 3, 3)
    E, V = [], []
    for h, C in zip(cells, stiff):
        P, det = inverse(h)
        w = L(det) / M.shape[1]
        B = sum(P.astype(L)[:, k, None] * M[..., k, None, :] for k in range(3))
        eps = sum(B[..., :, None, k] * B[..., None, :, k] for k in range(3))
        eps = (eps - np.identity(3)) / 2
        cv = np.array([[C[i, j, k, l] for k, l in VOIGT] for i, j in VOIGT]).astype(L)
        e6 = np.stack([eps[..., i, j] * (1 if i == j else 2) for i, j in VOIGT], -1)
        s6 = sum(cv[:, k] * e6[..., k, None] for k in range(6))
        s = np.empty(eps.shape, L)
        for I, (i, j) in enumerate(VOIGT):
            s[..., i, j] = s[..., j, i] = s6[..., I]
        t = sum(s[..., :, k, None] * B[..., k, None, :] for k in range(3))
        E.append(w * (e6 * s6).sum((-1, -2)) / 2)
        V.append(w * sum(B[..., k, :, None] * t[..., k, None, :] for k in range(3)).sum(1))
    kt = L(units.boltzmann * 300.0)
    c = [np.exp(-(e - np.minimum.reduce(E)) / kt) for e in E]
    return sum((x / sum(c))[:, None, None] * v for x, v in zip(c, V)).sum(0)


@pytest.mark.parametrize("model", ["corner8", "original"])
@pytest.mark.parametrize("states", [1, 2])
@pytest.mark.parametrize("cell", sorted(CELLS))
def test_virial_of_small_strains(cell, states, model):
    s = crystal(CELLS[cell], states)
    want = virial(s, model)
    err = np.abs(gpu_eval(s, model)[2] - want).max() / np.abs(want).max()
    print(cell, states, model, float(err), flush=True)
    assert err < TOL[model]
