"""The frame kernels where their shapes change: bands that pack into one wave
and bands that do not, runs longer than a wave's lanes, against the oracle; the
whole frame in one launch (large batches) against the marching frame kernel."""
import numpy as np
import pytest

from cases import build_case, hip_context, oracle_engine, synth_gather

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mod_nz,mod_nx,n2,nfdmax,ilste", [
    (30, 37, 10, 3, 1),    # both side bands in one wave
    (45, 60, 30, 5, 0),    # the widest that pack
    (37, 70, 31, 4, 1),    # one wave per side
    (20, 300, 66, 10, 1)])  # two waves per side, more bands than interior
@pytest.mark.parametrize("frame_split", [0, 1])
def test_marched_frame_equals_oracle(mod_nz, mod_nx, n2, nfdmax, ilste, frame_split):
    from rtm_gpu_amd import hip
    case = build_case(name="frame", mod_nz=mod_nz, mod_nx=mod_nx, n2=n2, nfdmax=nfdmax, ilste=ilste,
                      nt=120, tao=0.0008, src_x1=9)
    nt, inner = case["cfg"]["nt"], (slice(n2, -n2), slice(n2, -n2))
    seis = synth_gather(case)
    e = oracle_engine(case)
    ctx = hip_context(case, nshot=1, zseg=16, frame_split=frame_split)
    ctx.set_gathers(seis[None])
    e.forward_begin()
    ctx.forward_begin()
    for n in (3, nt):
        e.forward_advance(n)
        ctx.forward_advance(n)
        assert np.array_equal(ctx.field(hip.FIELD_U), e.field(0)), n
    e.backward_begin(seis)
    ctx.backward_begin()
    for n in (3, nt):
        e.backward_advance(n)
        ctx.backward_advance(n)
        assert np.array_equal(ctx.field(hip.FIELD_Q), e.field(2)), n
        assert np.array_equal(ctx.field(hip.FIELD_I1)[inner], e.field(3)[inner]), n
    ctx.close()


@pytest.mark.parametrize("nz,nx,n2,nfdmax,ilste", [
    (400, 578, 12, 3, 1),   # the narrowest frame with windows of four columns
    (370, 601, 31, 5, 1),   # one wave per side
    (300, 497, 64, 4, 0)])  # more rows than a block takes, two corner records
def test_whole_frame_launch(nz, nx, n2, nfdmax, ilste):
    from rtm_gpu_amd import hip
    shots = -(-10_000_000 // ((nz + 2 * n2) * (nx + 2 * n2)))
    shots += (2 - shots) % 4  # two of a block's four past the batch
    case = build_case(name="quad", mod_nz=nz, mod_nx=nx, n2=n2, nfdmax=nfdmax, ilste=ilste, nt=41,
                      nshot=shots, depth_step=6.0, src_x1=50, tao=0.0008)
    rng = np.random.default_rng(n2)
    seis = (0.01 * rng.standard_normal((shots, case["cfg"]["n"], 41))).astype(np.float32)
    out = []
    for zseg in (0, 16):  # 16 rows per wave: one step per launch
        ctx = hip_context(case, nshot=shots, zseg=zseg)
        ctx.set_gathers(seis)
        ctx.forward_begin()
        ctx.forward_advance(41)
        got = [ctx.field(w, shot=s) for s in (0, shots - 1) for w in (hip.FIELD_U, hip.FIELD_U_PREV)]
        got += [ctx.strip(shots - 1, k) for k in (20, 39)]
        ctx.backward_begin()
        ctx.backward_advance(41)
        got += [ctx.field(w, shot=s) for s in (0, shots - 1) for w in (hip.FIELD_Q, hip.FIELD_I1)]
        out.append(got)
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), i


@pytest.mark.parametrize("nshot,zseg,frame_split", [
    (3, 0, 0), (3, 16, 0), (3, 16, 1), (44, 0, 0)])  # whole steps by tiles, marching, two steps
def test_widths_on_one_model(nshot, zseg, frame_split):
    """Shots of several widths on the context's one model equal shots with the
    model's first columns as windows of their own."""
    from rtm_gpu_amd import hip
    nz, nx, n2 = (60, 150, 14) if nshot == 3 else (400, 578, 20)
    case = build_case(name="widths", mod_nz=nz, mod_nx=nx, n2=n2, nt=50, nshot=1, tao=0.0008)
    cfg, m = case["cfg"], case["model"]
    keys = ("nz", "nx", "n2", "nfdmax", "nt", "nt2", "ilste", "icompen", "s_l", "s_r", "s_z",
            "ds", "n", "tao2", "h2", "taoh", "taoh2", "hzx2_1")
    geoms = []
    for s in range(nshot):
        w = cfg["nx"] - 2 * n2 - 29 * (s % 3 if nshot == 3 else s // 4 % 2)
        geoms.append(dict(nx=w + 2 * n2, r_u=n2 + s % 40, r_x=n2 + 5, s_l=n2, s_r=n2 + w - 1, n=w, x_img=0))
    rng = np.random.default_rng(1)
    seis = (0.01 * rng.standard_normal((nshot, cfg["n"], cfg["nt"]))).astype(np.float32)
    v, r1 = (np.asarray(a).reshape(cfg["nz"], cfg["nx"]) for a in (m["v"], m["r1"]))
    out = []
    for windows in (False, True):
        ctx = hip.Context(max_shots=nshot, zseg=zseg, frame_split=frame_split, **{k: cfg[k] for k in keys})
        ctx.set_model(v, r1, m["w"], m["c"], m["index"], m["nvel"], m["vmin"], m["dv"])
        ctx.set_wavelet(m["wav"])
        ctx.set_shot_geometry(geoms)
        if windows:
            for s, q in enumerate(geoms):
                ctx.set_shot_model(s, np.ascontiguousarray(v[:, :q["nx"]]), np.ascontiguousarray(r1[:, :q["nx"]]))
        ctx.set_gathers(seis)
        ctx.forward_begin()
        ctx.forward_advance(cfg["nt"])
        got = [ctx.field(hip.FIELD_U, shot=s) for s in range(nshot)]
        ctx.backward_begin()
        ctx.backward_advance(cfg["nt"])
        got += [ctx.field(w, shot=s) for s in range(nshot) for w in (hip.FIELD_Q, hip.FIELD_I1)]
        out.append(got)
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), i


@pytest.mark.parametrize("nz,nx,n2,nfdmax", [
    (400, 578, 12, 3),   # the narrowest frame with windows of four columns
    (370, 601, 31, 5),   # one wave per side
    (300, 497, 64, 4)])  # more rows than a block takes, two corner records
def test_whole_frame_launch_on_a_rough_model(nz, nx, n2, nfdmax):
    """A coefficient row of its own for almost every cell: such batches take two
    steps per launch, and with them the frame in one launch."""
    from rtm_gpu_amd import hip
    shots = -(-12_000_000 // ((nz + 2 * n2) * (nx + 2 * n2)))
    shots += (2 - shots) % 4  # two of a block's four past the batch
    nt = 42
    case = build_case(name="quadr", mod_nz=nz, mod_nx=nx, n2=n2, nfdmax=nfdmax, ilste=1, nt=nt,
                      nshot=shots, depth_step=6.0, src_x1=50, tao=0.0008)
    cfg, m = case["cfg"], case["model"]
    z, x = np.mgrid[:cfg["nz"], :cfg["nx"]].astype(np.float32)
    v = (3000 + 1300 * np.sin(x / 23 + 0.7 * np.sin(z / 31)) * np.cos(z / 19 + 0.5 * np.sin(x / 41))).astype(np.float32)
    bins, row = 3000, np.asarray(m["c"], np.float32)[:nfdmax + 1]
    table = (row[None, :] * (1 + 1e-3 * np.sin(np.arange(bins)))[:, None]).astype(np.float32)
    keys = ("nz", "nx", "n2", "nfdmax", "nt", "nt2", "icompen", "s_l", "s_r", "s_z", "ds", "n",
            "tao2", "h2", "taoh", "taoh2", "hzx2_1")
    rng = np.random.default_rng(n2)
    seis = (0.01 * rng.standard_normal((shots, cfg["n"], nt))).astype(np.float32)
    out = []
    for zseg in (0, 16):  # 16 rows per wave: one step per launch
        ctx = hip.Context(**{k: cfg[k] for k in keys}, ilste=0, max_shots=shots, zseg=zseg)
        ctx.set_model(v, np.full_like(v, 0.2), m["w"], table, np.arange(bins + 1) * (nfdmax + 1), bins, 1600.0, 1.0)
        ctx.set_wavelet(m["wav"])
        ctx.set_shots(case["r_u"], case["r_x"])
        ctx.set_gathers(seis)
        ctx.set_timing(-1)
        ctx.forward_begin()
        ctx.forward_advance(nt)
        assert ctx.kernel_time(hip.K_FWD_INTERIOR)[1] == (nt - 2) // (2 if zseg == 0 else 1)
        ctx.set_timing(0)
        got = [ctx.field(w, shot=s) for s in (0, shots - 1) for w in (hip.FIELD_U, hip.FIELD_U_PREV)]
        got += [ctx.strip(shots - 1, k) for k in (2, nt // 2, nt - 1)]
        ctx.backward_begin()
        ctx.backward_advance(nt)
        got += [ctx.field(w, shot=s) for s in (0, shots - 1) for w in (hip.FIELD_Q, hip.FIELD_I1, hip.FIELD_I2)]
        out.append(got)
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.isfinite(a).all() and np.array_equal(a, b), i
