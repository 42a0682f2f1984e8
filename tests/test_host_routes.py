"""The host code above the kernels -- which launches a call makes, on which
buffers and for which steps -- on a HIP runtime that only logs them (CPU)."""
import pytest

from fake_hip import run


@pytest.mark.parametrize("n2", [20, 8])  # 8: no float4 windows of the frame
def test_autotune_keeps_to_the_steps_of_the_pass(n2):
    """rtm_autotune on a batch for which it times two steps per launch, one, and
    whole steps: every step it launches is one of the pass, whatever nt."""
    bad = run(f"""
fake.fake_cost(b"k_two", 0.5)
bad = []
for nt in list(range(12, 150)) + [184, 366, 420, 428, 482]:
    ctx = context(nz=200, nx=600, n2={n2}, nfd=3, nt=nt, shots=41, record=1, check_every=-1)
    shots(ctx, 41)
    log()
    ctx.autotune(8)
    rows = [r for r in log() if "k" in r]
    names = {{r["kernel"] for r in rows}}
    assert {{"k_two", "k_tile", "k_interior"}} <= names, names
    last = max(r["k"] for r in rows)
    if last >= nt or min(r["k"] for r in rows) < 0 or any(r["dead"] for r in rows):
        bad.append([nt, last])
    ctx.close()
out(bad)
""")
    assert bad == []


def test_window_changed_between_the_passes():
    """A shot that moves to another shot's window after the forward pass no
    longer shares the window of its block's four: one step per launch from there."""
    got = run("""
ctx = context(check_every=-1)
ragged(ctx, 40)
for s in range(40):
    window(ctx, s, 1500.0 if s < 20 else 1600.0)
import numpy as np
ctx.set_gathers(np.zeros((40, ctx.p.n, ctx.p.nt), np.float32))
res = []
for change in (False, True):
    ctx.forward_begin()
    ctx.forward_advance(60)
    log()
    if change:
        window(ctx, 0, 1600.0)
    ctx.backward_begin()
    ctx.backward_advance(60)
    res.append(sorted({r["kernel"] for r in log() if r["kernel"] in ("k_two", "k_interior", "k_tile")}))
out(res)
""")
    assert got[0] == ["k_two"]
    assert "k_two" not in got[1]
