"""Two time steps per launch (the kernel of large batches) against one step per
launch, bit for bit.  The marching kernels it is compared with equal the oracle
in test_gpu_parity.py (test_marching_kernels_equal_the_oracle)."""
import numpy as np
import pytest

from cases import build_case, hip_context

pytestmark = pytest.mark.gpu

# 41 shots (one past a block's four) of 440 x 618 cells: batches that take two
# steps per launch by default
SHOTS, NZ, NX, N2 = 41, 400, 578, 20


def passes(ctx, seis, calls):
    """Forward and backward pass in calls of the given lengths, with the fields
    after some of them."""
    from rtm_gpu_amd import hip
    nt, last = ctx.p.nt, ctx.nshot - 1
    ctx.set_gathers(seis)
    got = []
    ctx.forward_begin()
    for n in (*calls, nt):
        ctx.forward_advance(n)
        got += [ctx.field(w, shot=last) for w in (hip.FIELD_U, hip.FIELD_U_PREV)]
    got += [ctx.strip(s, nt // 2) for s in (0, last)]
    ctx.backward_begin()
    for n in (*calls, nt):
        ctx.backward_advance(n)
        got += [ctx.field(w, shot=last) for w in (hip.FIELD_Q, hip.FIELD_I1)]
        # the reconstructed field is the interior and the strip rings around it
        got.append(ctx.field(hip.FIELD_U, shot=last)[N2:-N2, N2:-N2])
    got += [ctx.field(w, shot=s) for s in (0, 3, last)
            for w in (hip.FIELD_I1, hip.FIELD_I2, hip.FIELD_Q)]
    if ctx.p.record:
        got.append(ctx.records())
    return got


@pytest.mark.parametrize("nfd,ilste,icompen,snap_every,strips", [
    (1, 1, 1, 0, 0), (2, 1, 0, 0, 0), (3, 1, 1, 0, 1), (4, 1, 1, 9, 0), (4, 0, 1, 0, 2),
    (5, 1, 1, 0, 0)])
def test_two_steps_per_launch(nfd, ilste, icompen, snap_every, strips):
    case = build_case(name="two", mod_nz=NZ, mod_nx=NX, n2=N2, nfdmax=nfd, nfdmin=min(2, nfd),
                      ilste=ilste, icompen=icompen, nt=44, nshot=SHOTS, depth_step=7.0, src_x1=90,
                      tao=0.0008, ds=3)
    rng = np.random.default_rng(nfd)
    seis = (0.01 * rng.standard_normal((SHOTS, case["cfg"]["n"], case["cfg"]["nt"]))).astype(np.float32)
    out = []
    for zseg in (0, 16):  # 16 rows per wave: one step per launch
        ctx = hip_context(case, nshot=SHOTS, record=1, zseg=zseg, snap_every=snap_every,
                          strip_format=strips)
        # calls of 1, 5, 2 and 7 steps: single steps between pairs, one to four
        # pending image terms at their ends
        out.append(passes(ctx, seis, (1, 5, 2, 7)))
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), i


@pytest.mark.parametrize("group", [4, 2])
def test_two_steps_with_shared_windows(group):
    """A ragged batch on two model windows of different widths, given to runs of
    four shots (a block's shots share their window) and of two (they do not, and
    the batch takes one step per launch)."""
    from rtm_gpu_amd import hip
    case = build_case(name="twowin", mod_nz=NZ, mod_nx=NX, n2=N2, nt=30, nshot=1)
    cfg, m = case["cfg"], case["model"]
    keys = ("nz", "nx", "n2", "nfdmax", "nt", "nt2", "ilste", "icompen", "s_l", "s_r", "s_z",
            "ds", "n", "tao2", "h2", "taoh", "taoh2", "hzx2_1")
    n, widths = 44, (cfg["nx"], cfg["nx"] - 37)
    geoms = []
    for s in range(n):
        nx = widths[s // group % 2]
        w = nx - 2 * N2
        geoms.append(dict(nx=nx, r_u=N2 + s, r_x=N2 + 10 * s % w, s_l=N2, s_r=N2 + w - 1, n=w, x_img=0))
    rng = np.random.default_rng(3)
    seis = (0.01 * rng.standard_normal((n, cfg["n"], cfg["nt"]))).astype(np.float32)
    out = []
    for zseg in (0, 16):
        ctx = hip.Context(**{k: cfg[k] for k in keys}, max_shots=n, zseg=zseg)
        ctx.set_model(m["v"], m["r1"], m["w"], m["c"], m["index"], m["nvel"], m["vmin"], m["dv"])
        ctx.set_wavelet(m["wav"])
        ctx.set_shot_geometry(geoms)
        for s, g in enumerate(geoms):
            v = np.ascontiguousarray(m["v"][:, :g["nx"]] if s // group % 2 == 0 else m["v"][:, -g["nx"]:])
            r1 = np.ascontiguousarray(m["r1"][:, :g["nx"]] if s // group % 2 == 0 else m["r1"][:, -g["nx"]:])
            ctx.set_shot_model(s, v, r1)
        out.append(passes(ctx, seis, (3, 8)))
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), i


def test_autotuned_batch():
    """rtm_autotune on such a batch times two steps per launch, one step and
    whole steps; the migration and its records are those of the fixed kernels.
    At 75 time samples a cycle of four steps ends at the last one."""
    case = build_case(name="two", mod_nz=NZ, mod_nx=NX, n2=N2, nfdmax=3, ilste=1, nt=75, nshot=SHOTS,
                      depth_step=7.0, src_x1=90, tao=0.0008, ds=3)
    rng = np.random.default_rng(9)
    seis = (0.01 * rng.standard_normal((SHOTS, case["cfg"]["n"], case["cfg"]["nt"]))).astype(np.float32)
    out = []
    for tuned in (True, False):
        ctx = hip_context(case, nshot=SHOTS, record=1, zseg=0 if tuned else 16)
        if tuned:
            ctx.autotune(8)
        out.append(passes(ctx, seis, (11,)))
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), i


def test_window_changed_between_the_passes():
    """Shot 0 takes the other window of the batch for the backward pass: its
    block's four shots no longer share one."""
    from rtm_gpu_amd import hip
    case = build_case(name="twochg", mod_nz=NZ, mod_nx=NX, n2=N2, nt=30, nshot=1)
    cfg, m = case["cfg"], case["model"]
    keys = ("nz", "nx", "n2", "nfdmax", "nt", "nt2", "ilste", "icompen", "s_l", "s_r", "s_z",
            "ds", "n", "tao2", "h2", "taoh", "taoh2", "hzx2_1")
    n, nt = 40, cfg["nt"]
    rng = np.random.default_rng(5)
    seis = (0.01 * rng.standard_normal((n, cfg["n"], nt))).astype(np.float32)
    v = np.ascontiguousarray(m["v"]).reshape(cfg["nz"], cfg["nx"])
    r1 = np.ascontiguousarray(m["r1"]).reshape(v.shape)
    wins = [(v, r1), (v[:, ::-1], r1[:, ::-1])]
    out = []
    for zseg in (0, 16):
        ctx = hip.Context(**{k: cfg[k] for k in keys}, max_shots=n, zseg=zseg)
        ctx.set_model(m["v"], m["r1"], m["w"], m["c"], m["index"], m["nvel"], m["vmin"], m["dv"])
        ctx.set_wavelet(m["wav"])
        ctx.set_shot_geometry([dict(nx=cfg["nx"], r_u=N2 + s, r_x=N2 + 90, s_l=cfg["s_l"], s_r=cfg["s_r"],
                                    n=cfg["n"], x_img=0) for s in range(n)])
        for s in range(n):
            ctx.set_shot_model(s, *wins[s >= 20])
        ctx.set_gathers(seis)
        ctx.forward_begin()
        ctx.forward_advance(nt)
        ctx.set_shot_model(0, *wins[1])
        ctx.backward_begin()
        ctx.backward_advance(nt)
        out.append([ctx.field(w, shot=s) for s in (0, 1, 4, 39) for w in (hip.FIELD_I1, hip.FIELD_I2, hip.FIELD_Q)])
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), i


def launches(ctx, seis, nt):
    """Interior launches of a forward and of a backward pass."""
    from rtm_gpu_amd import hip
    ctx.set_gathers(seis)
    ctx.set_timing(-1)
    ctx.forward_begin()
    ctx.forward_advance(nt)
    ctx.backward_begin()
    ctx.backward_advance(nt)
    n = [ctx.kernel_time(k)[1] for k in (hip.K_FWD_INTERIOR, hip.K_SRC_INTERIOR, hip.K_RCV_INTERIOR,
                                         hip.K_RCVI_INTERIOR, hip.K_FWD_FRAME)]
    ctx.set_timing(0)
    return n[0], n[1], n[2] + n[3], n[4]


@pytest.mark.parametrize("nfd,ilste", [(1, 1), (2, 1), (3, 1), (4, 1), (4, 0)])
def test_these_batches_take_two_steps_per_launch(nfd, ilste):
    """The batches above do what their tests compare: 42 forward steps in 21
    interior launches, and in 42 where the heights are set."""
    case = build_case(name="two", mod_nz=NZ, mod_nx=NX, n2=N2, nfdmax=nfd, nfdmin=min(2, nfd),
                      ilste=ilste, nt=44, nshot=SHOTS, depth_step=7.0, src_x1=90, tao=0.0008, ds=3)
    seis = np.zeros((SHOTS, case["cfg"]["n"], 44), np.float32)
    for zseg, want in ((0, (21, 21, 21, 42)), (16, (42, 42, 42, 42))):
        ctx = hip_context(case, nshot=SHOTS, zseg=zseg)
        assert launches(ctx, seis, 44) == want
        ctx.close()


def test_replayed_graph():
    """A batch that takes two steps per launch as a captured graph, replayed with
    eager work between the replays."""
    from rtm_gpu_amd import hip
    case = build_case(name="two", mod_nz=NZ, mod_nx=NX, n2=N2, nfdmax=3, nfdmin=2, ilste=1, nt=44,
                      nshot=SHOTS, depth_step=7.0, src_x1=90, tao=0.0008, ds=3)
    rng = np.random.default_rng(11)
    sets = [(0.01 * rng.standard_normal((SHOTS, case["cfg"]["n"], 44))).astype(np.float32) for _ in range(2)]
    fields = (hip.FIELD_U, hip.FIELD_Q, hip.FIELD_I1, hip.FIELD_I2)

    def result(ctx):
        got = [ctx.field(w, shot=s) for s in (0, SHOTS - 1) for w in fields]
        return [got[0][N2:-N2, N2:-N2], *got[1:4], got[4][N2:-N2, N2:-N2], *got[5:]]

    one = hip_context(case, nshot=SHOTS, record=1, zseg=16)
    want = []
    for d in sets:
        one.set_gathers(d)
        one.migrate()
        want.append(result(one))
    one.close()
    ctx = hip_context(case, nshot=SHOTS, record=1)
    ctx.set_graph(True)
    for i in (0, 1, 0):
        ctx.set_gathers(sets[i])
        for again in range(2):
            ctx.migrate()
            for a, b in zip(result(ctx), want[i]):
                assert np.array_equal(a, b), (i, again)
        ctx.forward_begin()     # eager work on the same buffers
        ctx.forward_advance(13)
    ctx.close()


def test_born_and_adjoint_beside_two_steps_per_launch():
    """A batch whose migration takes two steps per launch and whose Born and
    adjoint passes take one, their background frame in one launch."""
    from rtm_gpu_amd import hip
    n, nt = 103, 44
    case = build_case(name="twoborn", mod_nz=260, mod_nx=217, n2=N2, nfdmax=3, nfdmin=3, ilste=0, nt=nt,
                      nshot=n, depth_step=2.0, src_x1=90, tao=0.0008)
    rng = np.random.default_rng(12)
    refl = (0.1 * rng.standard_normal((260, 217))).astype(np.float32)
    seis = (0.01 * rng.standard_normal((n, case["cfg"]["n"], nt))).astype(np.float32)
    out = []
    for zseg in (0, 16):
        ctx = hip_context(case, nshot=n, record=1, zseg=zseg)
        assert launches(ctx, seis, nt)[0] == (21 if zseg == 0 else 42)
        ctx.set_reflectivity(refl)
        ctx.set_timing(-1)
        got = [ctx.born()]
        assert ctx.kernel_time(hip.K_BORN_FRAME)[1] == nt - 2  # not whole steps in one launch
        ctx.set_timing(0)
        got += [ctx.field(hip.FIELD_Q, shot=s) for s in (0, n - 1)]
        got.append(ctx.adjoint(seis))
        out.append(got)
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), i


def test_two_steps_per_launch_at_the_longest_half_length():
    """Half-length 5 takes two steps per launch from larger batches on."""
    n, nt = 93, 30
    case = build_case(name="two", mod_nz=NZ, mod_nx=NX, n2=N2, nfdmax=5, ilste=1, nt=nt, nshot=n,
                      depth_step=3.0, src_x1=90, tao=0.0008, ds=3)
    rng = np.random.default_rng(13)
    seis = (0.01 * rng.standard_normal((n, case["cfg"]["n"], nt))).astype(np.float32)
    out = []
    for zseg, want in ((0, (nt - 2) // 2), (16, nt - 2)):
        ctx = hip_context(case, nshot=n, record=1, zseg=zseg)
        assert launches(ctx, seis, nt)[:3] == (want,) * 3
        out.append(passes(ctx, seis, (1, 6)))
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), i
