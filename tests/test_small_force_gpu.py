"""One force evaluation in one launch (small fields) and the host call: against the oracle around
the limits of the one-workgroup kernel, and the same bits from host and device arrays."""

import numpy as np
import pytest
import torch

from micmec_amd.pes import ForcePartMechanical, MicMecForceField

from test_force_gpu import TOL, oracle_eval, rel
from test_metric_gpu import skewed_system

pytestmark = pytest.mark.gpu


# half a workgroup; two blocks of slots; the most nodes (open faces); just above the limit in
# slots; far above it (the inputs go through device memory)
SHAPES = [((2, 2, 3), 2, 0.0, True), ((7, 7, 7), 3, 0.0, True), ((7, 7, 7), 8, 0.2, False),
          ((8, 8, 9), 2, 0.0, True), ((21, 19, 23), 2, 0.1, True)]


@pytest.mark.parametrize("model", ["corner8", "original"])
@pytest.mark.parametrize("shape,states,p_hole,pbc", SHAPES)
def test_host_call(shape, states, p_hole, pbc, model):
    print(shape, states, model, flush=True)
    s = skewed_system(shape, states, 3, p_hole, pbc)
    fpm = ForcePartMechanical(s, model=model)
    mmf = MicMecForceField(s, [fpm])
    gpos, vtens = np.zeros(s.pos.shape), np.zeros((3, 3))
    e = mmf.compute(gpos, vtens)
    want = oracle_eval(s, model)
    for got, ref in zip((e, gpos, vtens), want):
        assert rel(got, ref) < TOL
    # the device call, each output alone, accumulation
    kw = dict(dtype=torch.float64, device=fpm.device)
    pos = torch.tensor(np.asarray(s.pos), **kw)
    rv = np.zeros((3, 3))
    rv[:len(s.domain.rvecs)] = s.domain.rvecs
    rv = torch.tensor(rv, **kw)
    ed, gd, vd = torch.zeros(1, **kw), torch.zeros(pos.shape, **kw), torch.zeros((3, 3), **kw)
    fpm.compute_device(pos, rv, ed, gd, vd)
    assert ed.item() == e
    assert np.array_equal(gd.cpu().numpy(), gpos) and np.array_equal(vd.cpu().numpy(), vtens)
    assert mmf.compute() == e
    g2 = np.zeros(gpos.shape)
    assert mmf.compute(g2) == e and np.array_equal(g2, gpos)
    fpm.compute_device(pos, rv, ed, gd, vd, accumulate=True)
    assert ed.item() == 2 * e
    assert np.array_equal(gd.cpu().numpy(), 2 * gpos) and np.array_equal(vd.cpu().numpy(), 2 * vtens)
    # moved positions and domain: nothing is kept from the call before
    mmf.update_pos(1.01 * np.asarray(s.pos))
    if pbc:
        mmf.update_rvecs(1.01 * np.asarray(s.domain.rvecs))
    g3, v3 = np.zeros(gpos.shape), np.zeros((3, 3))
    e3 = mmf.compute(g3, v3)
    for got, ref in zip((e3, g3, v3), oracle_eval(s, model)):
        assert rel(got, ref) < TOL
    assert np.array_equal(fpm._rvecs_d.cpu().numpy()[:len(s.domain.rvecs)], s.domain.rvecs)


@pytest.mark.parametrize("shape", [(3, 3, 3), (9, 9, 9)])
def test_nan_is_reported(shape):
    s = skewed_system(shape, 2, 4)
    mmf = MicMecForceField(s, [ForcePartMechanical(s)])
    bad = np.array(s.pos)
    bad[5, 1] = np.nan
    mmf.update_pos(bad)
    with pytest.raises(ValueError):
        mmf.compute(np.zeros(bad.shape), np.zeros((3, 3)))
