"""GPU: a run whose work buffers cannot be allocated is refused, and the runs after it are as before: a buffer whose
allocation failed is allocated anew, and no kernel of the refused run outlives it."""
import numpy as np
import pytest

from skirt7_amd import skirt as S
from skirt7_amd import workloads
from skirt7_amd.capi import SG_FP64, SG_MIXED

pytestmark = pytest.mark.gpu

# launch states of 2^37 packets: 3.8e12 bytes in FP32, more than any device has
TOO_MANY = 1 << 37


@pytest.mark.parametrize("precision", [SG_FP64, SG_MIXED])
@pytest.mark.parametrize("pipeline", [0, 1])
def test_runs_after_a_refused_run(pipeline, precision):
    w = workloads.disc_cartesian(grid_n=10, pixels=16, packages=1000)

    def run():
        w["instr"].clear()
        c = w["sim"].run_packets(0, 0, 1000, 1000, precision)
        return np.concatenate([w["instr"].frame(i).ravel() for i in range(3)]), c["walks"]

    try:
        S.set_pipeline(pipeline)
        S.set_slots(1024)
        ref, walks = run()
        S.set_emit_batch(TOO_MANY)
        with pytest.raises(S.FatalError):
            w["sim"].run_packets(0, 0, TOO_MANY, TOO_MANY, precision)
        S.set_emit_batch(0)
        out, again = run()
    finally:
        S.set_emit_batch(0)
        S.set_slots(0)
        S.set_pipeline(1)
    assert again == walks
    # sums of at most some ten thousand positive FP64 terms in another order
    np.testing.assert_allclose(out, ref, rtol=1e-11, atol=0)


@pytest.mark.parametrize("precision", [SG_FP64, SG_MIXED])
def test_runs_after_a_refused_batch(precision):
    """One member's buffers cannot be allocated while the shared launch of another is under way."""
    pop = workloads.fit_population(members=3, packets=(1.0e3, 3.0e3), grid_n=(6, 14), pixels=(32, 16), nsamples=2)
    ms = pop["members"]

    def run():
        for m in ms:
            m["instr"].clear()
        c = S.run_batch([m["sim"] for m in ms], [900, 2000, 3000], precision=precision)
        return np.concatenate([m["instr"].frame(0).ravel() for m in ms]), c["walks"]

    try:
        S.set_slots(1024)
        S.set_batch_alone(1000)
        ref, walks = run()
        S.set_emit_batch(TOO_MANY)
        with pytest.raises(S.FatalError):
            S.run_batch([m["sim"] for m in ms], [900, 2000, TOO_MANY], precision=precision)
        S.set_emit_batch(0)
        out, again = run()
    finally:
        S.set_emit_batch(0)
        S.set_batch_alone(3 << 16)
        S.set_slots(0)
    assert again == walks
    # sums of at most some ten thousand positive FP64 terms in another order
    np.testing.assert_allclose(out, ref, rtol=1e-11, atol=0)
