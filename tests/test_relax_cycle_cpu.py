"""A finished optimiser and its degrees of freedom are freed without the cycle collector, so that the
next run reuses their memory; the search outlives its optimiser."""

import gc
import weakref

from micmec_amd import units
from micmec_amd.sampling import CartesianDOF, CGOptimizer
from micmec_amd.workloads import make_system

from test_trajectory_cpu import _OracleForceField


def make():
    s = make_system((3, 3, 3), p_b=0.3, seed=4, strain=0.02, noise=0.05 * units.angstrom)
    dof = CartesianDOF(_OracleForceField(s))
    return CGOptimizer(dof), dof


def test_freed_at_once():
    opt, dof = make()
    opt.run(2)
    gone = weakref.ref(opt), weakref.ref(dof)
    gc.collect()
    gc.disable()
    try:
        del opt, dof
        assert gone[0]() is None and gone[1]() is None
    finally:
        gc.enable()


def test_search_without_its_optimiser():
    opt, dof = make()
    opt.run(1)
    search, f = opt.minimizer, opt.minimizer.f
    del opt
    assert search.propagate() and search.f < f
