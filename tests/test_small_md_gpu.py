"""Systems of at most 512 work slots and nodes step in one launch (use_graph, the default), those
of at most 512 blocks run a step's scalar phases inside its other kernels: the same bits as the
step's kernels one by one (use_graph=False), which is an identity of the arithmetic, so there
is no tolerance."""

import ctypes

import numpy as np
import pytest
import torch

from micmec_amd import _native, units
from micmec_amd.adjoint import voigt_from_tensor
from micmec_amd.pes import ForcePartMechanical, MicMecForceField
from micmec_amd.pes.mmff import parse_type_params
from micmec_amd.sampling import (LangevinBarostat, LangevinThermostat, MTKBarostat, NHCThermostat,
                                 VerletIntegrator)
from micmec_amd.workloads import make_system

pytestmark = pytest.mark.gpu
FS = units.femtosecond

# shape, probability of the two-state type, of a hole, periodic: one cell; one wave; one type and
# two types in one and two blocks with holes and open faces; the most nodes (512); one node layer
# and one slot block more than fit one workgroup; some fifty blocks
SYSTEMS = [((1, 1, 1), 0.0, 0.0, False), ((3, 3, 3), 0.5, 0.0, True), ((4, 3, 5), 0.3, 0.2, False),
           ((2, 3, 20), 1.0, 0.1, True), ((7, 7, 7), 0.5, 0.0, False), ((8, 8, 8), 0.0, 0.0, True),
           ((8, 8, 9), 0.0, 0.1, True), ((9, 9, 9), 0.5, 0.0, False), ((24, 19, 27), 0.3, 0.1, True)]


def integrator(shape, p_b, p_hole, pbc, ensemble, model, graph):
    system = make_system(shape, p_b=p_b, p_hole=p_hole, seed=31, pbc=pbc)
    mmf = MicMecForceField(system, [ForcePartMechanical(system, model=model)])
    np.random.seed(5)
    hooks = {"nve": lambda: [],
             "nvt": lambda: [NHCThermostat(temp=300.0, timecon=100 * FS)],
             "langevin": lambda: [LangevinThermostat(temp=300.0, seed=3)],
             "nph": lambda: [MTKBarostat(mmf, temp=300.0, press=units.bar)],
             "npt": lambda: [NHCThermostat(temp=300.0, timecon=100 * FS),
                             MTKBarostat(mmf, temp=300.0, press=units.bar)],
             "langevin npt": lambda: [LangevinThermostat(temp=300.0, seed=3),
                                      LangevinBarostat(mmf, temp=300.0, press=units.bar, seed=4)],
             }[ensemble]()
    return VerletIntegrator(mmf, timestep=FS, hooks=hooks, use_graph=graph)


def assert_same_bits(a, b, steps):
    for n in steps:
        a.run(n)
        b.run(n)
        torch.cuda.synchronize()
        for name in ("pos", "vel", "gpos", "S"):
            x, y = getattr(a._engine, name), getattr(b._engine, name)
            assert torch.isfinite(x).all(), (n, name)
            assert torch.equal(x, y), (n, name)


@pytest.mark.parametrize("model", ["corner8", "original"])
@pytest.mark.parametrize("ensemble", ["nve", "nvt", "langevin", "nph", "npt", "langevin npt"])
def test_one_launch_steps_have_the_bits_of_the_kernels(ensemble, model):
    for shape, p_b, p_hole, pbc in SYSTEMS:
        if not pbc and ensemble in ("nph", "npt", "langevin npt"):
            continue
        print("small", shape, ensemble, model, flush=True)
        a = integrator(shape, p_b, p_hole, pbc, ensemble, model, True)
        b = integrator(shape, p_b, p_hole, pbc, ensemble, model, False)
        assert_same_bits(a, b, (1, 2, 9, 20))


@pytest.mark.parametrize("ensemble", ["nve", "nvt", "langevin", "npt"])
@pytest.mark.parametrize("shape", [(50, 51, 50), (54, 54, 52)])
def test_merged_phases_up_to_512_blocks(shape, ensemble):
    """Just below and above the most blocks whose phases are merged into other kernels."""
    print("merged", shape, ensemble, flush=True)
    a, b = (integrator(shape, 0.3, 0.0, True, ensemble, "corner8", graph)
            for graph in (True, False))
    assert_same_bits(a, b, (2, 7))


def test_long_call_is_cut_into_launches():
    a = integrator((2, 2, 2), 0.5, 0.0, True, "npt", "corner8", True)
    b = integrator((2, 2, 2), 0.5, 0.0, True, "npt", "corner8", False)
    assert_same_bits(a, b, (2049, 4100))


@pytest.mark.parametrize("shape", [(4, 4, 3), (9, 9, 9)])
def test_new_state_counts_between_calls(shape):
    """mm_field_set_params moves blocks from the multistate to the single-state cell code: one
    launch and a graph captured anew follow it as the kernels one by one do."""
    a, b = (integrator(shape, 0.5, 0.0, True, "nve", "corner8", graph) for graph in (True, False))
    assert_same_bits(a, b, (5,))
    system = a.mmf.system
    _, ns, h0, c0, free, temp = parse_type_params(system.params, system.types)
    assert ns.max() == 2
    cv = np.array([[voigt_from_tensor(c) for c in row] for row in c0])
    arrays = [np.ascontiguousarray(x, dtype=t) for x, t in
              ((np.ones_like(ns), np.int32), (h0, np.float64), (cv, np.float64),
               (free, np.float64), (temp, np.float64))]
    for v in (a, b):
        rc = _native.lib().mm_field_set_params(
            v._engine.fpm.field._handle, *[x.ctypes.data_as(ctypes.c_void_p) for x in arrays],
            float(units.boltzmann), _native.stream_ptr())
        assert rc == 0
    assert_same_bits(a, b, (1, 7))


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("ensemble", ["nve", "langevin"])
@pytest.mark.parametrize("shape,pbc", [((3, 4, 2), True), ((9, 10, 8), False), ((20, 20, 20), True)])
def test_rows_of_steps_match_single_steps(shape, pbc, ensemble, graph):
    """Steps in one call do the second kick, the next first kick and the drift in one pass; steps
    of one call each do not: the same bits."""
    a, b = (integrator(shape, 0.3, 0.05, pbc, ensemble, "corner8", graph) for _ in range(2))
    for n in (2, 3, 11):
        a.run(n)
        for _ in range(n):
            b.propagate()
        for name in ("pos", "vel", "gpos", "S"):
            assert torch.equal(getattr(a._engine, name), getattr(b._engine, name)), (n, name)
        assert a.econs == b.econs
