"""GPU: the event/walk passes at queue lengths around their claim sizes (16 to 128 requests, 64 lanes), with one and
two slot groups and several emission batches, against the lane pipeline's same packet histories."""
import numpy as np
import pytest

from skirt7_amd import skirt as S
from skirt7_amd import workloads
from skirt7_amd.capi import SG_FP64, SG_MIXED

pytestmark = pytest.mark.gpu


def _run(w, count, precision):
    w["instr"].clear()
    c = w["sim"].run_packets(0, 3, count, 1000, precision)
    frames = np.concatenate([w["instr"].frame(i).ravel() for i in range(3)])
    return frames, {k: c[k] for k in ("packets", "own_crossings", "peel_crossings", "rewalk_crossings", "scatterings",
                                      "peeloffs", "walks")}


@pytest.fixture(scope="module")
def disc():
    return workloads.disc_cartesian(grid_n=14, pixels=24, packages=1000)


@pytest.mark.parametrize("precision", [SG_FP64, SG_MIXED])
@pytest.mark.parametrize("count,groups,batch", [(1, 2, 0), (2, 2, 0), (3, 1, 0), (4, 2, 0), (16, 1, 0), (17, 2, 0),
                                                (63, 1, 0), (129, 2, 64), (700, 2, 0), (701, 1, 100), (5001, 2, 1024)])
def test_passes_equal_the_lane_pipeline(disc, count, groups, batch, precision):
    # the histories are the same, only the order of the tally additions differs: the sums of up to a few hundred
    # thousand positive FP64 terms agree to n eps < 1e-10
    try:
        S.set_pipeline(0)
        ref, cref = _run(disc, count, precision)
        S.set_pipeline(1)
        S.set_slot_groups(groups)
        S.set_emit_batch(batch)
        out, c = _run(disc, count, precision)
    finally:
        S.set_pipeline(1)
        S.set_slot_groups(2)
        S.set_emit_batch(0)
    assert c == cref
    np.testing.assert_allclose(out, ref, rtol=1e-10, atol=0)
