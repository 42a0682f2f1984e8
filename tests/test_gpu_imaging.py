"""The imaging of the backward pass: the receiver step of every third backward
step applies the image terms of three steps, and of whatever is pending at the
end of each rtm_backward_advance call.  Advancing in calls of any length gives
the images, sums and fields of the oracle, which images every step."""
import numpy as np
import pytest

from cases import build_case, hip_context, oracle_engine, synth_gather

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ilste,icompen,snap_every,zseg", [
    (0, 1, 0, 16), (0, 0, 0, 16), (1, 0, 7, 16), (0, 1, 7, 16),
    (0, 1, 0, 0), (1, 0, 7, 0)])
def test_images_after_calls_of_any_length(ilste, icompen, snap_every, zseg):
    """Calls of 1, 2, 3, 4 and 7 steps (pending terms of one, two and three
    steps at their ends), checkpoint pairs at every phase of the three-step
    cycle, both imaging conditions, fixed and automatic kernel choice."""
    from rtm_gpu_amd import hip
    case = build_case(name="imaging", nt=90, ilste=ilste, icompen=icompen,
                      nfdmax=6 if ilste else 4)
    n2, nt = case["cfg"]["n2"], case["cfg"]["nt"]
    seis = synth_gather(case)
    e = oracle_engine(case, snap_every=snap_every)
    e.forward_begin()
    e.forward_advance(nt)
    e.backward_begin(seis)
    ctx = hip_context(case, nshot=1, zseg=zseg, snap_every=snap_every)
    ctx.set_gathers(seis[None])
    ctx.forward_begin()
    ctx.forward_advance(nt)
    ctx.backward_begin()
    left, i = nt - 2, 0
    inner = (slice(n2, -n2), slice(n2, -n2))
    while left > 0:
        step = min(left, (1, 2, 3, 4, 7)[i % 5])
        e.backward_advance(step)
        ctx.backward_advance(step)
        left, i = left - step, i + 1
        pairs = [(2, hip.FIELD_Q), (3, hip.FIELD_I1), (4, hip.FIELD_I2)]
        if icompen:
            pairs += [(5, hip.FIELD_SU), (6, hip.FIELD_SQ)]
        for which, name in pairs:
            assert np.array_equal(ctx.field(name)[inner], e.field(which)[inner]), (left, which)
    ctx.close()
