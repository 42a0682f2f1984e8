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


def test_lateral_factors_take_no_memory_that_nothing_reads():
    """Setting a ragged geometry allocates nothing: shots may still bring windows,
    whose factors share the plane of r1.  With one model, a plane per width is
    made when a pass needs it."""
    got = run("""
n = 12
widths = [300 + 10 * s for s in range(n)]
ctx = context(nz=120, nx=420, shots=n, check_every=-1)
b0 = ctx.device_bytes()
ragged(ctx, n, widths)
b1 = ctx.device_bytes()
for s, w in enumerate(widths):
    window(ctx, s, 1500.0 + s, w)
ctx.forward_begin(); ctx.forward_advance(60)
b2 = ctx.device_bytes()
one = context(nz=120, nx=420, shots=n, check_every=-1)
ragged(one, n, widths)
c0 = one.device_bytes()
one.forward_begin(); one.forward_advance(60)
c1 = one.device_bytes()
ragged(one, n, widths[::-1])          # the same widths: nothing new
log()
one.forward_begin(); one.forward_advance(60)
again = sum("frame_lat" in r["kernel"] for r in log())
pitch = (12 + 420 + 4 + 63) // 64 * 64  # 12 guard columns on the left with n2 = 20
out([b1 - b0, (b2 - b1) / (4 * 120 * pitch), (c1 - c0) / (4 * 120 * pitch), again, one.device_bytes() - c1])
""")
    assert got == [0, 4 * 12, 12 - 1, 0, 0]


def test_a_batch_that_finds_no_memory_leaves_the_context_usable():
    got = run("""
ctx = context(nz=120, nx=420, shots=12, check_every=-1)
shots(ctx, 12)
ctx.forward_begin(); ctx.forward_advance(60)
from rtm_gpu_amd import hip
fake.fake_limit(fake.fake_used() + 1000)
ragged(ctx, 3, [300, 310, 320])
ctx.forward_begin()
try:
    ctx.forward_advance(60)
    raised = False
except hip.RtmError as e:
    raised = "hipMalloc" in str(e)
shots(ctx, 12)
log()
ctx.forward_begin(); ctx.forward_advance(60)
rows = log()
out([raised, any(r["dead"] for r in rows), sum(r["kernel"] == "k_tile" for r in rows)])
""")
    assert got == [True, False, 58]


def test_model_set_between_the_passes():
    """A model set after the forward pass is the one the backward pass takes,
    its lateral factors included."""
    got = run("""
import numpy as np
ctx = context(nz=120, nx=420, shots=3, check_every=-1)
shots(ctx, 3)
ctx.set_gathers(np.zeros((3, ctx.p.n, ctx.p.nt), np.float32))
ctx.forward_begin(); ctx.forward_advance(60)
log()
set_model(ctx, 120, 420, 20, 3, v=1600.0)
ctx.backward_begin(); ctx.backward_advance(60)
out([r["kernel"] for r in log() if "frame_lat" in r["kernel"] or "k_tile" in r["kernel"]][:2])
""")
    assert "frame_lat" in got[0] and got[1] == "k_tile"


def test_buffers_of_two_steps_per_launch_are_held_by_batches_that_take_them():
    got = run("""
import numpy as np
fb = 4 * 41 * 440 * 640
res = []
for kind in ("two", "fixed heights", "own windows", "small"):
    ctx = context(zseg=16 if kind == "fixed heights" else 0, check_every=-1)
    b = [ctx.device_bytes()]
    n = 4 if kind == "small" else 40
    if kind == "own windows":
        ragged(ctx, n)
        for s in range(n):
            window(ctx, s, 1500.0 + s)
        b[0] += 4 * fb
    else:
        shots(ctx, n)
    log()
    ctx.forward_begin(); ctx.forward_advance(60)
    rows = log()
    res.append([round((ctx.device_bytes() - b[0]) / fb, 1), any(r["kernel"] == "k_two" for r in rows),
                any(r["dead"] for r in rows)])
    ctx.close()
out(res)
""")
    assert got == [[2.2, True, False], [0.0, False, False], [0.0, False, False], [0.0, False, False]]


@pytest.mark.parametrize("steps", [0, 1, 2, 3, 5, 6])
@pytest.mark.parametrize("backward", [False, True])
def test_required_memory_takes_the_place_of_those_buffers(steps, backward):
    """An allocation that fails beside them succeeds in their place, wherever the
    rotation has put the fields of the running pass; the pass goes on, one step per
    launch, from the two fields written last."""
    got = run(f"""
import numpy as np
backward, steps = {backward}, {steps}
kinds = dict(k_two=2, k_interior=1) if backward else dict(k_two=1, k_interior=3)  # TWO_*, EPI_*

def launches():  # of the forward or the reconstructed field
    rows = log()
    assert not any(r["dead"] for r in rows)
    return [r for r in rows if r["kernel"] in kinds and r["kind"] == kinds[r["kernel"]]]

ctx = context(nt=61, nfd=5, check_every=-1)
shots(ctx, 40)
ctx.forward_begin()
if backward:
    ctx.set_gathers(np.zeros((40, ctx.p.n, ctx.p.nt), np.float32))
    ctx.forward_advance(61)
    ctx.backward_begin()
advance = ctx.backward_advance if backward else ctx.forward_advance
log()
for n in [1] * (steps % 2) + [2] * (steps // 2):
    advance(n)
last = launches()[-1:]
held = ctx.device_bytes()
fake.fake_limit(fake.fake_used() + 1000)
ctx.set_reflectivity(np.zeros((400, 578), np.float32))
freed = held - ctx.device_bytes()
advance(3)
one = launches()
newest = [(r["ub"], r["ua"]) if r["kernel"] == "k_two" else (r["u2"], r["u1"]) for r in last]
out([freed > 2 * 4 * 41 * 440 * 640, [r["kernel"] for r in one], len({{r["u2"] for r in one}}),
     newest in ([], [(one[0]["u1"], one[0]["u0"])])])
""")
    assert got == [True, ["k_interior"] * 3, 3, True]


@pytest.mark.parametrize("nshot", [40, 12])  # two steps per launch; whole steps
def test_heights_set_after_the_autotuner_are_used(nshot):
    """The later of rtm_autotune and rtm_set_zseg / rtm_set_frame_runs decides."""
    got = run(f"""
def kernels():
    log()
    ctx.forward_begin(); ctx.forward_advance(60)
    return sorted({{r["kernel"] for r in log() if r["kernel"] in ("k_two", "k_tile", "k_interior")}})
res = []
for which in ("zseg", "runs"):
    ctx = context(check_every=-1)
    fake.fake_cost(b"k_two", 0.5)
    fake.fake_cost(b"k_tile", {9.0 if nshot == 40 else 0.5})
    shots(ctx, {nshot})
    ctx.autotune(8)
    res.append(kernels())
    if which == "zseg":
        ctx.set_zseg(14, 14, 14)
    else:
        ctx.set_frame_runs(10, 16)
    res.append(kernels())
    ctx.autotune(8)
    res.append(kernels())
    ctx.close()
out(res)
""")
    tuned = ["k_two"] if nshot == 40 else ["k_tile"]
    assert got == [tuned, ["k_interior"], tuned] * 2


def test_a_choice_of_the_autotuner_is_for_batches_like_its_own():
    """Whole steps chosen on narrow shots are not taken for a batch of the same
    count that is much larger; a batch of about the same size keeps them."""
    got = run("""
def kernels():
    log()
    ctx.forward_begin(); ctx.forward_advance(60)
    return sorted({r["kernel"] for r in log() if r["kernel"] in ("k_two", "k_tile", "k_interior")})
fake.fake_cost(b"k_tile", 0.1)
ctx = context(nx=2400, nfd=5, shots=30, check_every=-1)
res = []
for width in (900, 860, 2400, 900):
    ragged(ctx, 30, [width] * 30)
    if not res:
        ctx.autotune(8)
    res.append(kernels())
out(res)
""")
    assert got[:2] == [["k_tile"], ["k_tile"]]
    assert ["k_tile"] not in got[2:]


def test_a_longer_operator_drops_the_choice():
    got = run("""
import numpy as np
from rtm_gpu_amd import hip
def kernels():
    log()
    ctx.forward_begin(); ctx.forward_advance(60)
    return sorted({r["kernel"] for r in log() if r["kernel"] in ("k_two", "k_tile", "k_interior")})
# least-squares rows: the operator is as long as the table's longest row
nz, nx, n2, n, nt = 440, 618, 20, 578, 60
ctx = hip.Context(nz=nz, nx=nx, n2=n2, nfdmax=12, nt=nt, nt2=nt, ilste=0, icompen=1, s_l=n2,
                  s_r=nx - n2 - 1, s_z=n2, ds=1, n=n, tao2=1e-6, h2=1e-2, taoh=1e-4, taoh2=1e-8,
                  hzx2_1=1.0, max_shots=41, check_every=-1)
ctx.set_wavelet(np.zeros(nt + 1, np.float32))
z = np.full((nz, nx), 1500.0, np.float32)
def model(nfd):
    ctx.set_model(z, z * 0, np.zeros(n2 + 1), np.ones(nfd + 1), np.array([0, nfd + 1], np.int32), 1, 1500.0, 1.0)
fake.fake_cost(b"k_tile", 0.1)
model(2)
shots(ctx, 41)
ctx.autotune(8)
res = [kernels()]
model(12)
res.append(kernels())
out(res)
""")
    assert got == [["k_tile"], ["k_interior"]]


@pytest.mark.parametrize("snap_every", [0, 20, 50, 4])
def test_two_steps_are_timed_on_whole_cycles(snap_every):
    """A cycle that rtm_autotune times takes four steps each way, checkpoint or
    not: as many of the reconstruction as of the forward field, and of the
    receiver field; away from checkpoints where they leave room."""
    got = run(f"""
ctx = context(nt=150, shots=41, snap_every={snap_every}, check_every=-1)
shots(ctx, 41)
fake.fake_cost(b"k_two", 0.5)
fake.fake_cost(b"k_tile", 9.0)
log()
ctx.autotune(8)
steps = dict(fwd=0, src=0, rcv=0)
pairs = 0
for r in log():
    if r["kernel"] == "k_two":
        steps[("fwd", "fwd", "src", "rcv", "rcv")[r["kind"]]] += 2
        pairs += r["kind"] == 2
    elif r["kernel"] == "k_interior":
        name = {{0: "fwd", 3: "fwd", 1: "src", 2: "rcv", 7: "rcv"}}.get(r["kind"])
        steps[name] += 1
    elif r["kernel"] == "k_tile":
        for name in (["fwd"], ["src", "rcv"])[r["kind"]]:
            steps[name] += 1
out([steps["fwd"] - steps["src"], steps["src"] - steps["rcv"], pairs])
""")
    full = run(f"""
ctx = context(nt=150, shots=41, check_every=-1)
shots(ctx, 41)
fake.fake_cost(b"k_two", 0.5)
fake.fake_cost(b"k_tile", 9.0)
log()
ctx.autotune(8)
out(sum(r["kernel"] == "k_two" and r["kind"] == 2 for r in log()))
""")
    assert got[:2] == [0, 0]
    if snap_every != 4:  # checkpoints at steps 4, 5, 8, 9, ...: every cycle meets some
        assert got[2] == full


def test_fit_keeps_the_losses_of_a_bounded_number_of_batches():
    """Training on many small batches holds no more device memory for their
    losses than on a thousand of them."""
    got = run("""
import numpy as np
from rtm_gpu_amd import cnn
used = []
for n in (1024, 3000):
    net = cnn.Deblur([1, 4, 1], 64, 8)
    x = np.zeros((n, 1, 2, 2), np.float32)
    log()
    b = fake.fake_used()
    net.fit(x, x[:, 0], 2, 1, 1e-3)
    used.append(fake.fake_used() - b - n * (4 + 4 + 1) * 4)
    steps = sum("k_adam" in r["kernel"] for r in log())
    net.close()
    used.append(steps)
out(used)
""")
    assert got == [1024 * 256 * 8, 2048, 1024 * 256 * 8, 6000]


# Batches timed on an MI355X, ms for 60 steps each way: marching kernels, two
# steps per launch, whole steps in one launch (None: not timed or not built)
TIMED = [
    ("mig", 400, 140, 20, 8, 89, 8.3, None, 13.0), ("mig", 261, 133, 30, 7, 165, 9.1, None, 13.5),
    ("mig", 400, 270, 20, 6, 62, 7.6, None, 10.8), ("mig", 400, 140, 20, 11, 65, 7.7, None, 10.6),
    ("mig", 261, 133, 30, 5, 245, 12.3, 14.4, 16.8), ("mig", 400, 270, 20, 9, 41, 7.1, None, 9.5),
    ("mig", 400, 140, 20, 3, 107, 8.2, 7.8, 10.3), ("mig", 400, 270, 20, 4, 79, 10.4, 9.7, 12.7),
    ("mig", 400, 270, 20, 1, 37, 5.3, 3.9, 5.1), ("mig", 400, 140, 20, 12, 60, 8.0, None, 10.0),
    ("mig", 411, 1761, 30, 3, 41, 22.9, 19.2, 30.7), ("mig", 411, 1761, 30, 3, 6, 6.9, 5.5, 4.4),
    ("mig", 391, 700, 30, 3, 110, 23.8, 19.1, 32.6), ("mig", 261, 133, 30, 1, 115, 6.8, 5.5, 6.5),
    ("pairs", 400, 270, 20, 10, 83, 19.0, None, 37.1), ("pairs", 400, 270, 20, 12, 69, 16.7, None, 31.5),
    ("pairs", 400, 270, 20, 6, 139, 23.6, None, 34.4), ("pairs", 400, 270, 20, 8, 104, 20.3, None, 28.8),
    ("pairs", 391, 700, 30, 2, 18, 10.4, None, 5.5), ("pairs", 391, 700, 30, 8, 20, 16.1, None, 9.5)]


def test_a_batch_takes_the_kernel_that_was_fastest_on_it():
    picks = run(f"""
import numpy as np
out_ = []
for kind, nz, nx, n2, nfd, n in {[t[:6] for t in TIMED]}:
    ctx = context(nz=nz, nx=nx, n2=n2, nfd=nfd, nt=20, shots=n, record=1, check_every=-1)
    shots(ctx, n)
    if kind == "pairs":
        ctx.set_reflectivity(np.zeros((nz - 2 * n2, nx - 2 * n2), np.float32))
        ctx.born_begin()
    else:
        ctx.forward_begin()
    log()
    (ctx.born_advance if kind == "pairs" else ctx.forward_advance)(20)
    names = {{r["kernel"] for r in log()}}
    out_.append([i for i, k in enumerate(("k_interior", "k_two", "k_tile")) if k in names][-1])
    ctx.close()
out(out_)
""")
    slow = []
    for t, p in zip(TIMED, picks):
        ms = t[6:]
        best = min(m for m in ms if m)
        if ms[p] > 1.15 * best:
            slow.append((t, p))
    assert slow == []


@pytest.mark.parametrize("nz,nx,n2,nfd,n,ms", [
    (261, 300, 30, 4, 255, (28.1, 18.4, 31.1)), (261, 300, 30, 2, 511, (45.9, 29.6, 51.6)),
    (440, 540, 20, 3, 42, (12.6, 10.0, 11.7)), (411, 1761, 30, 2, 14, (14.7, None, 12.1))])
def test_a_rough_model_costs_the_kernels_that_gather(nz, nx, n2, nfd, n, ms):
    """Cells whose coefficient rows lie in different lines: timed as above, on
    shared windows or (None) a window per shot."""
    pick = run(f"""
import numpy as np
from rtm_gpu_amd import hip
nz, nx, n2, nfd, n, own = {nz}, {nx}, {n2}, {nfd}, {n}, {ms[1] is None}
z, x = np.mgrid[:nz, :nx].astype(np.float32)
v = (3000 + 1300 * np.sin(x / 23 + 0.7 * np.sin(z / 31)) * np.cos(z / 19 + 0.5 * np.sin(x / 41))).astype(np.float32)
m, nt = nx - 2 * n2, 20
ctx = hip.Context(nz=nz, nx=nx, n2=n2, nfdmax=nfd, nt=nt, nt2=nt, ilste=0, icompen=1, s_l=n2,
                  s_r=nx - n2 - 1, s_z=n2, ds=1, n=m, tao2=1e-6, h2=1e-2, taoh=1e-4, taoh2=1e-8,
                  hzx2_1=1.0, max_shots=n, check_every=-1)
ctx.set_model(v, v * 0, np.zeros(n2 + 1), np.ones(3001 * (nfd + 1)),
              (np.arange(3001) * (nfd + 1)).astype(np.int32), 3000, 1400.0, 1.0)
ctx.set_wavelet(np.zeros(nt + 1, np.float32))
if own:
    ragged(ctx, n)
    for s in range(n):
        ctx.set_shot_model(s, v + np.float32(0.37 * s), v * 0)
else:
    shots(ctx, n)
ctx.forward_begin()
log()
ctx.forward_advance(20)
names = {{r["kernel"] for r in log()}}
out([i for i, k in enumerate(("k_interior", "k_two", "k_tile")) if k in names][-1])
""")
    assert ms[pick] <= 1.15 * min(t for t in ms if t), pick
