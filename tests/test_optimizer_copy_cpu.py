"""Copies of an optimiser, by copy or through pickle, search on their own degrees of freedom."""

import copy
import pickle

import numpy as np
import pytest

from micmec_amd import units
from micmec_amd.sampling import CartesianDOF, CGOptimizer
from micmec_amd.workloads import make_system

from test_trajectory_cpu import _OracleForceField


@pytest.mark.parametrize("clone", [copy.deepcopy, lambda o: pickle.loads(pickle.dumps(o))])
@pytest.mark.parametrize("before", [0, 2])
def test_clone_runs_by_itself(clone, before):
    s = make_system((3, 3, 3), p_b=0.3, seed=4, strain=0.02, noise=0.05 * units.angstrom)
    opt = CGOptimizer(CartesianDOF(_OracleForceField(s)))
    if before:
        opt.run(before)
    pos, x = np.array(s.pos), np.array(opt.minimizer.x)
    other = clone(opt)
    other.run(2)
    assert np.array_equal(s.pos, pos) and np.array_equal(opt.minimizer.x, x)
    assert np.array_equal(other.dof.mmf.system.pos.ravel(), other.minimizer.x)
    opt.run(2)
    assert np.array_equal(other.minimizer.x, opt.minimizer.x) and other.epot == opt.epot
