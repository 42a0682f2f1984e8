"""The work that users of rtm_gpu_amd have it do, as cases that can be timed.

A case is one whole pass through the public entry points:

  migrate   a batch of shots migrated and stacked (hip.Context.migrate,
            image_post, stack_finish): forward pass with boundary strips,
            backward pass with imaging
  model     forward modelling with receiver recording (forward_begin /
            forward_advance / records)
  aperture  a ragged batch: every shot on its own window of a large model
            (set_shot_geometry, set_shot_model), migrated and stacked
  cgls      least-squares migration of given data (lsrtm.cgls): adjoint, Born
            modelling and adjoint again
  pairs     Born data of several reflectivities and their adjoint image in one
            launch sequence, each panel on its own background (the training
            pairs of the deblurring network)
  fit       one epoch of training the deblurring network (cnn.Deblur.fit)
  grad      loss and gradient of one batch (cnn.Deblur.loss_grad)
  infer     the network applied to migrated images (cnn.Deblur.forward)

The wave-equation cases run fewer time steps than a production job (hundreds
instead of thousands), on its grids, batches, operators and options: the work
of a time step does not depend on how many there are.
"""
import math

import numpy as np
import torch

from rtm_gpu_amd import cnn, hip, host, lsrtm, synth

STRIPS = {"f32": hip.RTM_STRIP_F32, "f16": hip.RTM_STRIP_F16, "bf16": hip.RTM_STRIP_BF16}
WHITE = 1e-4  # whitening of the illumination in the image post


def _wave(kind, **kw):
    """A wave-equation case with the options it does not name at their usual
    values: adaptive LS operators, compensated imaging, FP32 strips, eager."""
    case = dict(kind=kind, mod_nz=200, mod_nx=400, shots=1, nt=400, n2=20, nfdmax=4, taylor=False,
                compensated=True, strips="f32", snap=0, graph=False, tune=False, ds=1, well=False,
                h=10.0, tao=0.001, f0=25.0)
    case.update(kw)
    return case


def listed():
    return [
        # One shot of the plain single-shot configuration (200 x 400 at 10 m,
        # eighth order, 20-point hybrid boundary, 25 Hz), as an interactive run
        # or a drop-in caller with one source per call migrates it.
        _wave("migrate", name="single_shot", nt=1000),
        # The same call on a small odd grid, captured once and replayed: the
        # latency of launches is all there is.
        _wave("migrate", name="single_graph_odd", mod_nz=101, mod_nx=157, nt=500, graph=True),
        # A handful of surface shots with a long Taylor operator, the
        # uncompensated image and every third receiver: the reference's other
        # options, on a ragged size.
        _wave("migrate", name="few_shots_taylor", mod_nz=203, mod_nx=531, shots=6, nt=300, n2=30,
              nfdmax=10, taylor=True, compensated=False, ds=3, tao=0.0008, f0=20.0),
        # The headline: reverse VSP, 128 sources down a well under the
        # 351 x 1701 faulted model, 1701 receivers, tuned once per batch.
        _wave("migrate", name="rvsp_128", mod_nz=351, mod_nx=1701, shots=128, nt=400, n2=30,
              nfdmax=10, well=True, h=12.5, f0=20.0, tune=True),
        # The same survey with memory-saving options: FP16 strips and
        # checkpoint snapshots, a sixteen-shot batch, not tuned.
        _wave("migrate", name="rvsp_16_half", mod_nz=351, mod_nx=1701, shots=16, nt=400, n2=30,
              nfdmax=4, well=True, h=12.5, f0=20.0, strips="f16", snap=100),
        # Observed data made by the engine: forward modelling with recording
        # at every eighth surface point, no strips.
        _wave("model", name="model_rvsp_32", mod_nz=351, mod_nx=1701, shots=32, nt=400, n2=30,
              nfdmax=10, well=True, ds=8, h=12.5, f0=20.0),
        # Surface shots with uneven apertures on the 4001 x 801 model, one
        # window and model per shot, tuned once.
        _wave("aperture", name="apertures_24", mod_nz=801, mod_nx=4001, shots=24, nt=250, n2=30,
              wmin=600, wmax=2400, tune=True, tao=0.0008, f0=15.0),
        # Least-squares migration of a twelve-shot surface survey: one CGLS
        # iteration from given data.
        _wave("cgls", name="cgls_12", mod_nz=200, mod_nx=400, shots=12, nt=400, n2=30, nfdmax=6,
              f0=15.0),
        # Training pairs of the network: two 1024 x 256 panels of 32 shots.
        _wave("pairs", name="pairs_2x32", mod_nz=256, mod_nx=1024, shots=32, panels=2, nt=250,
              n2=30, tune=False),
        # One epoch of the network's training on 64 x 64 patches, batch 256.
        dict(name="fit_64x64", kind="fit", n=1024, h=64, w=64, batch=256, hidden=32, layers=6),
        # The network on eight migrated images, as the evaluation calls it.
        dict(name="infer_8x256x1024", kind="infer", n=8, h=256, w=1024, hidden=32, layers=6),
        # Loss and gradient of a small odd batch with narrower layers, some
        # dilated: a training step of a network under development.
        dict(name="grad_odd", kind="grad", n=12, h=61, w=93, hidden=24, layers=4, dilated=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["migrate"] * 4 + ["model", "aperture", "cgls", "pairs", "fit", "infer", "grad"])
    if kind in ("fit", "grad"):
        case = dict(kind=kind, h=rng.randint(24, 96), w=rng.randint(24, 128),
                    hidden=rng.choice([8, 16, 24, 32, 32]), layers=rng.randint(3, 7))
        if kind == "fit":
            case["batch"] = _log_int(rng, 16, 256)
            case["n"] = case["batch"] * rng.randint(1, 3) + rng.randint(0, 7)
        else:
            case["n"] = _log_int(rng, 1, 128)
            case["dilated"] = rng.random() < 0.5
        return case
    if kind == "infer":
        return dict(kind=kind, n=_log_int(rng, 1, 8), h=rng.randint(64, 256),
                    w=rng.randint(64, 1024), hidden=rng.choice([16, 32, 32]), layers=rng.randint(3, 7))
    big = rng.random() < 0.5
    case = _wave(kind, mod_nz=rng.randint(150, 420) if big else rng.randint(100, 220),
                 mod_nx=_log_int(rng, 500, 1800) if big else _log_int(rng, 150, 500),
                 shots=_log_int(rng, 4, 64) if big else _log_int(rng, 1, 24),
                 nt=rng.randint(150, 350), n2=rng.choice([12, 20, 30, 30]),
                 nfdmax=rng.choice([4, 4, 6, 10]), ds=rng.choice([1, 1, 2, 8]),
                 f0=float(rng.choice([15, 20, 25])), well=rng.random() < 0.4)
    if kind == "aperture":
        lo = rng.randint(150, 700)
        case.update(mod_nz=rng.randint(200, 600), mod_nx=rng.randint(2600, 4001), wmin=lo,
                    wmax=rng.randint(lo + 50, 2400), shots=_log_int(rng, 3, 20), ds=1, well=False,
                    tune=rng.random() < 0.5, tao=0.0008)
    elif kind == "cgls":
        case.update(shots=_log_int(rng, 2, 16), ds=1, well=False)
        case["taylor"] = rng.random() < 0.25
    elif kind == "pairs":
        case.update(panels=rng.randint(1, 4), shots=_log_int(rng, 2, 16), ds=1, well=False)
    else:
        case["taylor"] = rng.random() < 0.25
    if kind == "migrate":
        case.update(compensated=rng.random() < 0.75, tune=big and rng.random() < 0.5,
                    strips=rng.choice(["f32", "f32", "f32", "f16", "bf16"]),
                    snap=rng.choice([0, 0, 0, 60]))
        case["graph"] = not big and rng.random() < 0.4
    if case["taylor"]:
        case.update(tao=0.0008, nfdmax=rng.choice([4, 6, 8, 10, 12]))
    return case


# ---- inputs ------------------------------------------------------------------
def _ricker(nt, tao, f0, t0):
    a = math.pi * f0 * (np.arange(nt) * tao - t0)
    return (1.0 - 2.0 * a * a) * np.exp(-a * a)


def _gathers(rng, sx, rx, nt, tao, f0, h):
    """Traces [shot][receiver][nt] of a direct arrival and three reflections
    with hyperbolic moveout, amplitudes falling with distance."""
    table = np.concatenate([np.zeros(nt), _ricker(nt, tao, f0, 1.5 / f0)]).astype(np.float32)
    window = np.lib.stride_tricks.sliding_window_view(table, nt)  # row nt - d: delayed by d
    out = np.zeros((len(sx), len(rx), nt), np.float32)
    off = np.abs(np.asarray(sx)[:, None] - np.asarray(rx)[None, :]) * h
    for e in range(4):
        t0, v = (0.01, rng.uniform(1500, 2500)) if e == 0 else (rng.uniform(0.05, 0.6) * nt * tao,
                                                                rng.uniform(2000, 4000))
        t = np.sqrt(t0 * t0 + (off / v) ** 2)
        amp = (rng.uniform(0.5, 1.5) * (0.05 if e == 0 else 0.004) /
               np.sqrt(1.0 + t / (10 * tao))).astype(np.float32)
        d = np.minimum((t / tao).astype(np.int64), nt)
        for s in range(len(sx)):
            out[s] += amp[s][:, None] * window[nt - d[s]]
    return out


def _table(case, v, d):
    """Coefficient table of the velocities v: LS per 1 m/s bin, or one Taylor row."""
    vmin, vmax, nvel = host.vrange(v, 1.0)
    if case["taylor"]:
        return dict(c=host.taylor(case["nfdmax"]), index=None, nvel=1, vmin=vmin, vmax=vmax)
    need = host.bins_needed(v, vmin, 1.0, nvel)
    _, index, c = host.design_ls(1000, case["nfdmax"], 2, nvel, case["tao"], case["h"], 1.0, 1e-5,
                                 2 * case["f0"] + 1, vmin, 1.0, need, d.hzx)
    return dict(c=c, index=index, nvel=nvel, vmin=vmin, vmax=vmax)


def _survey(case, seed):
    """Everything a job reads before it starts: geometry, models, coefficient
    table, wavelet, sources, observed data, reflectivity."""
    rng = np.random.default_rng(seed)
    n2, nz, nx, h, tao = case["n2"], case["mod_nz"], case["mod_nx"], case["h"], case["tao"]
    shots, panels = case["shots"], case.get("panels", 1)
    width = nx  # the widest grid a shot runs on
    S = dict(n2=n2, shots=shots * panels)
    if case["kind"] == "aperture":
        widths = rng.integers(case["wmin"], case["wmax"] + 1, shots)
        starts = [int(rng.integers(0, nx - w + 1)) for w in widths]
        width = int(widths.max())
    n = (width - 1) // case["ds"] + 1
    cfg = host.make_config(nfdmax=case["nfdmax"], nfdmin=2, n2=n2, f0=case["f0"],
                           fmax=2 * case["f0"] + 1, df=1.0, nthita=1000, eps=1e-5, dv=1.0,
                           ilste=int(case["taylor"]), ifv=0, whitecoe=WHITE, hz=h, tao=tao, inorm=1,
                           icompen=int(case["compensated"]), h=h, tao1=tao, mod_nz=nz, mod_nx=width,
                           nt1=case["nt"], s_l1=1, s_z1=1, n=n, ds=case["ds"], r_x1=width // 2 + 1,
                           nrec=shots, dr=1)
    d = S["d"] = host.derive(cfg)
    S.update(nz=d.nz, nx=d.nx, nt=d.nt, n=n, wav=host.wavelet_table(d.nt, tao, case["f0"]),
             w=host.blend_weights(n2))

    def pad(raw):
        return host.pad_model(raw, nz, raw.shape[0], n2, 0, tao, h)

    surface = host.source_row(h, h, n2)
    rx = np.arange(n) * case["ds"]
    if case["kind"] == "aperture":
        raw = synth.smooth(synth.grf_4001(seed=seed, mod_nz=nz, mod_nx=nx, h=h), 4.0)
        S["models"] = [pad(np.ascontiguousarray(raw[a:a + w])) for a, w in zip(starts, widths)]
        S.update(_table(case, raw, d), gw=nx)
        S["geoms"] = [dict(nx=int(w) + 2 * n2, r_u=surface, r_x=n2 + int(w) // 2, s_l=n2,
                           s_r=n2 + int(w) - 1, n=int(w), x_img=a) for a, w in zip(starts, widths)]
        S["gathers"] = np.zeros((shots, n, d.nt), np.float32)
        for s, w in enumerate(widths):
            S["gathers"][s, :w] = _gathers(rng, [w // 2], rx[:w], d.nt, tao, case["f0"], h)[0]
        return S
    if case["kind"] == "pairs":
        raws, refl = zip(*[synth.reflectors(seed * 100 + p, nz, nx, h) for p in range(panels)])
        S["refl"] = np.concatenate(refl, axis=1)
    elif nx < 300 or nz < 150:
        raws = [synth.smooth(synth.layered_5(seed, nz, nx), 2.0)]
    else:
        raws = [synth.smooth(synth.faulted_rvsp(seed, nz, nx, h), 4.0)]
    S["models"] = [pad(r) for r in raws]
    S.update(_table(case, np.concatenate([m[0].ravel() for m in S["models"]]), d), gw=nx * panels)
    if case["well"]:
        r_u = [host.source_row(min(0.5 * h * (s + 1), 0.9 * nz * h), h, n2) for s in range(shots)]
        r_x = [d.r_x] * shots
    else:
        r_u = [surface] * shots
        r_x = [int(n2 + c) for c in np.linspace(0, nx - 1, shots + 2)[1:-1].round()]
    S["geoms"] = [dict(nx=d.nx, r_u=r_u[s], r_x=r_x[s], s_l=d.s_l, s_r=d.s_r, n=n, x_img=p * nx)
                  for p in range(panels) for s in range(shots)]
    if case["kind"] in ("migrate", "cgls"):
        S["gathers"] = _gathers(rng, [x - n2 for x in r_x], rx, d.nt, tao, case["f0"], h)
    return S


def _patches(case, seed):
    """Network inputs (scaled migrated image, background velocity in [0, 1],
    depth), targets and starting parameters."""
    rng = np.random.default_rng(seed)
    n, h, w = case["n"], case["h"], case["w"]
    x = np.empty((n, 3, h, w), np.float32)
    t = rng.standard_normal((n, h, w), np.float32)
    t *= rng.random((n, h, w), np.float32) < 0.1  # thin reflectors
    x[:, 0] = 0.5 * t + 0.25 * (np.roll(t, 1, 1) + np.roll(t, -1, 1)) + \
        0.1 * rng.standard_normal((n, h, w), np.float32)
    x[:, 1] = np.linspace(0.1, 0.9, h, dtype=np.float32)[:, None]
    x[:, 1] += 0.05 * rng.standard_normal((n, 1, 1), np.float32)
    x[:, 2] = np.linspace(0.0, 1.0, h, dtype=np.float32)[:, None]
    ch = [3] + [case["hidden"]] * (case["layers"] - 1) + [1]
    p = []
    for i in range(len(ch) - 1):
        scale = math.sqrt(2.0 / (9 * ch[i])) * (0.1 if i == len(ch) - 2 else 1.0)
        p.append(rng.standard_normal(ch[i + 1] * ch[i] * 9) * scale)
        p.append(0.01 * rng.standard_normal(ch[i + 1]))
    dil = [1 << min(i, 3) if case.get("dilated") else 1 for i in range(len(ch) - 1)]
    return dict(x=x, t=t, ch=ch, dil=dil, p=np.concatenate(p).astype(np.float32))


def prepare(case, seed):
    if case["kind"] in ("fit", "grad", "infer"):
        D = _patches(case, seed)
        b = case.get("batch", case["n"])
        D["net"] = cnn.Deblur(D["ch"], b * case["h"] * case["w"], b * case["h"], dilation=D["dil"])
        D["net"].set_params(D["p"])
        return dict(case=case, **D)
    S = _survey(case, seed)
    d = S["d"]
    ctx = hip.Context(nz=d.nz, nx=d.nx, n2=S["n2"], nfdmax=case["nfdmax"], nt=d.nt, nt2=d.nt2,
                      ilste=int(case["taylor"]), icompen=int(case["compensated"]), s_l=d.s_l,
                      s_r=d.s_r, s_z=d.s_z, ds=case["ds"], n=S["n"], tao2=d.tao2, h2=d.h2,
                      taoh=d.taoh, taoh2=d.taoh2, hzx2_1=d.hzx2_1, max_shots=S["shots"],
                      strip_format=STRIPS[case["strips"]], snap_every=case["snap"],
                      record=int(case["kind"] in ("model", "cgls", "pairs")),
                      stack_nx=S["gw"], frame_split=int(case["tune"]))
    ragged = case["kind"] in ("aperture", "pairs")
    v, r1 = S["models"][0] if not ragged else [np.full((d.nz, d.nx), S["vmin"], np.float32)] * 2
    ctx.set_model(v, r1, S["w"], S["c"], S["index"], S["nvel"], S["vmin"], 1.0)
    ctx.set_wavelet(S["wav"])
    if ragged:
        ctx.set_shot_geometry(S["geoms"])
        for s in range(S["shots"]):
            m = s if case["kind"] == "aperture" else s // case["shots"]
            ctx.set_shot_model(s, *S["models"][m])
    else:
        ctx.set_shots([g["r_u"] for g in S["geoms"]], [g["r_x"] for g in S["geoms"]])
    if case["kind"] in ("migrate", "aperture"):
        ctx.set_gathers(S["gathers"])
    if case["tune"]:
        ctx.autotune(8)
    if case["graph"]:
        ctx.set_graph(True)
    state = dict(case=case, ctx=ctx, shots=S["shots"], vmax=float(S["vmax"]))
    if case["kind"] == "cgls":
        state.update(op=lsrtm.BornOperator(ctx), data=S["gathers"])
    if case["kind"] == "pairs":
        state["refl"] = S["refl"]
    return state


def run(state):
    kind = state["case"]["kind"]
    if kind == "fit":
        net, c = state["net"], state["case"]
        net.set_params(state["p"])
        loss = net.fit(state["x"], state["t"], epochs=1, batch=c["batch"], lr=1e-3, seed=5)
        return dict(loss=loss, params=net.params())
    if kind == "grad":
        loss, g = state["net"].loss_grad(state["x"], state["t"])
        return dict(loss=loss, grad=g)
    if kind == "infer":
        return state["net"].forward(state["x"])
    ctx = state["ctx"]
    if kind in ("migrate", "aperture"):
        ctx.migrate()
        ctx.image_post(state["vmax"], WHITE, want=False)
        img, illum = ctx.stack_finish(state["shots"], 1)
        return dict(image=img, illumination=illum)
    if kind == "model":
        ctx.forward_begin(save_strips=False)
        ctx.forward_advance(ctx.p.nt)
        return ctx.records()
    if kind == "cgls":
        m, hist = lsrtm.cgls(state["op"], state["data"], 1)
        return dict(model=m, misfit=[q["rr"] for q in hist])
    ctx.set_reflectivity(state["refl"])  # pairs
    ctx.born_begin()
    ctx.born_advance(ctx.p.nt)
    ctx.gathers_from_records()
    ctx.adjoint_begin()
    ctx.adjoint_advance(ctx.p.nt)
    return ctx.adjoint_gradient()


# ---- what a pass cannot do without -------------------------------------------
def work(case):
    """Time stepping: every step reads two fields and writes one (a job's
    fields are far larger than the caches; strips, gathers and images are read
    and written once per pass).  Network: inputs, targets and outputs of the
    call, and every layer's activations once per direction they are needed in;
    two flops per weight, pixel and product."""
    if case["kind"] in ("fit", "grad", "infer"):
        ch = [3] + [case["hidden"]] * (case["layers"] - 1) + [1]
        n = case["n"] // case["batch"] * case["batch"] if case["kind"] == "fit" else case["n"]
        pix = n * case["h"] * case["w"]
        mac = sum(9 * a * b for a, b in zip(ch, ch[1:]))
        if case["kind"] == "infer":
            return dict(bytes=pix * (4 * 4 + 2 * sum(2 * c for c in ch[1:-1])), flops=2 * mac * pix)
        back = 2 * mac - 9 * ch[0] * ch[1]
        return dict(bytes=pix * (4 * 4 + sum(5 * 2 * c for c in ch[1:-1])),
                    flops=2 * (mac + back) * pix)
    n2, nt = case["n2"], case["nt"]
    nz = case["mod_nz"] + 2 * n2
    nx = case["mod_nx"] + 2 * n2
    shots = case["shots"] * case.get("panels", 1)
    if case["kind"] == "aperture":
        nx = (case["wmin"] + case["wmax"]) // 2 + 2 * n2
    full = shots * nz * nx
    inner = shots * case["mod_nz"] * (nx - 2 * n2)
    point = 8 * case["nfdmax"] if case["taylor"] else 32  # the LS rows of these models have 2..4 taps
    strip = shots * 2 * case["nfdmax"] * (case["mod_nz"] + nx - 2 * n2) * \
        (4 if case["strips"] == "f32" else 2)
    data = shots * 4 * ((nx - 2 * n2 - 1) // case["ds"] + 1)
    fwd = dict(bytes=12 * full, flops=(point + 8) * full)
    if case["kind"] == "model":
        return dict(bytes=nt * (fwd["bytes"] + data), flops=nt * fwd["flops"])
    rec = dict(bytes=12 * inner, flops=(point + 8) * inner)
    if case["kind"] in ("migrate", "aperture"):
        return dict(bytes=nt * (2 * fwd["bytes"] + rec["bytes"] + 2 * strip + data) + 16 * inner,
                    flops=nt * (2 * fwd["flops"] + rec["flops"] + 6 * inner))
    born = dict(bytes=nt * (2 * fwd["bytes"] + strip + data) + 4 * inner,
                flops=nt * (2 * fwd["flops"] + 5 * inner))
    adj = dict(bytes=nt * (fwd["bytes"] + rec["bytes"] + strip + data) + 4 * inner,
               flops=nt * (fwd["flops"] + rec["flops"] + 5 * inner))
    if case["kind"] == "pairs":
        return {k: born[k] + adj[k] for k in born}
    return dict(bytes=born["bytes"] + 2 * adj["bytes"] + nt * (fwd["bytes"] + strip),
                flops=born["flops"] + 2 * adj["flops"] + nt * fwd["flops"])


# ---- 64-bit values -----------------------------------------------------------
class _Grid64:
    """The time step of one model in float64: the two-way update with per-cell
    operators and mirrored edges, and the hybrid one-way boundary with the
    reference's operands (kernel.cu:46-208)."""

    def __init__(self, S, case, v, r1, nx):
        self.dev = dev = "cuda" if torch.cuda.is_available() else "cpu"
        d, n2, nz = S["d"], S["n2"], S["nz"]
        self.nz, self.nx, self.n2, self.hzx = nz, nx, n2, float(d.hzx2_1)

        def dbl(a):
            return torch.from_numpy(np.ascontiguousarray(a)).to(dev, torch.float64)

        self.v = dbl(v)
        self.P = self.v * self.v * (float(d.tao2) * float(d.h2))
        if S["index"] is None:
            row, top, length = np.zeros((nz, nx), np.int64), np.zeros(1, int), np.array([case["nfdmax"]])
        else:
            q = ((v - np.float32(S["vmin"])) / np.float32(1.0)).astype(np.float64)
            row = np.clip((q + 0.5).astype(np.int64), 0, S["nvel"] - 1)
            top, length = S["index"][:-1], np.diff(S["index"]) - 1
        self.nfd = M = int(max(length.max(), 1))
        tab = np.zeros((len(top), M + 1))
        for i, (t, n) in enumerate(zip(top, length)):
            if n >= 0:
                tab[i, :n + 1] = S["c"][t:t + n + 1]
        taps = dbl(tab)[torch.from_numpy(row).to(dev)]
        self.c0 = (1.0 + self.hzx) * taps[..., 0]
        self.c = [taps[..., l].contiguous() for l in range(1, M + 1)]
        self.per_cell = S["index"] is not None

        def mirror(n):
            i = np.abs(np.arange(-M, n + M))
            return torch.from_numpy(np.where(i >= n, 2 * n - 2 - i, i)).to(dev)

        self.mz, self.mx = mirror(nz), mirror(nx)
        self.inner = torch.zeros(nz, nx, dtype=torch.bool, device=dev)
        self.inner[n2:nz - n2, n2:nx - n2] = True

        z, x = np.nonzero(~self.inner.cpu().numpy())
        a = np.minimum(np.minimum(z, x), np.minimum(nz - 1 - z, nx - 1 - x))
        zl, xl = z - a <= 1, x - a <= 1
        corner = (zl | (nz - 1 - a - z <= 1)) & (xl | (nx - 1 - a - x <= 1))
        top_, bot = z == a, (z != a) & (z == nz - 1 - a)
        side = ~top_ & ~bot
        left = side & (x == a)
        iz = z + np.where(top_, 1, np.where(bot, -1, 0))
        ix = x + np.where(side, np.where(left, 1, -1), 0)
        dz, dx = side.astype(int), 1 - side.astype(int)

        def at(zz, xx):
            return torch.from_numpy(np.clip(zz, 0, nz - 1) * nx + np.clip(xx, 0, nx - 1)).to(dev)

        self.cell, self.i = at(z, x), at(iz, ix)
        self.ip, self.im = at(iz + dz, ix + dx), at(iz - dz, ix - dx)
        self.sp, self.sm = at(z + dz, x + dx), at(z - dz, x - dx)
        self.cx, self.cz = at(z, x + np.where(xl, 1, -1)), at(z + np.where(zl, 1, -1), x)
        zq = np.clip(np.where(top_, z, np.where(bot, a, a + z // nx)), 0, nz - 1)
        xq = np.clip(np.where(side, z % nx, x), 0, nx - 1)
        self.corner = torch.from_numpy(corner).to(dev)
        self.tv = float(d.taoh) * self.v[z, x]
        self.tq = float(d.taoh2) * self.v[zq, xq] ** 2
        self.r1, self.w = dbl(r1)[z, x], dbl(S["w"])[np.clip(n2 - a, 0, n2)]

    def lap(self, u, transposed=False):
        M, nz, nx = self.nfd, self.nz, self.nx
        p = u[:, self.mz][:, :, self.mx]
        out = self.c0 * u

        def sh(f, a, b):
            return f[..., M + a:M + a + nz, M + b:M + b + nx]

        for l in range(1, M + 1):
            if not transposed:
                s = (sh(p, -l, 0) + sh(p, l, 0)) * self.hzx
                s += sh(p, 0, -l)
                s += sh(p, 0, l)
                out += s.mul_(self.c[l - 1])
            else:  # each tap with the coefficient of the cell it reads
                c = torch.nn.functional.pad(self.c[l - 1], (M, M, M, M))
                for a, b, k in ((-l, 0, self.hzx), (l, 0, self.hzx), (0, -l, 1.0), (0, l, 1.0)):
                    out += k * sh(c, a, b) * sh(p, a, b)
        return out

    def update(self, u1, u0, transposed=False):
        """Two-way value from u1 (newer) and u0; transposed on the interior."""
        L = self.lap(u1)
        if transposed and self.per_cell:
            L = torch.where(self.inner, self.lap(u1, True), L)
        return 2.0 * u1 - u0 + self.P * L

    def boundary(self, T, u1, u0):
        """T with its frame replaced by the blend of T and the one-way value."""
        t, a, b = (f.reshape(f.shape[0], -1) for f in (T, u1, u0))
        T0, Ti, U1, U0, U0i = t[:, self.cell], t[:, self.i], a[:, self.cell], b[:, self.cell], b[:, self.i]
        num = self.tv * (Ti - U0i + U0) - (-2.0 * U1 + U0 + Ti - 2.0 * a[:, self.i] + U0i)
        num += self.tq * (t[:, self.ip] - 2.0 * Ti + t[:, self.im] + b[:, self.sp] - 2.0 * U0 + b[:, self.sm])
        cnum = U1 + self.r1 * (t[:, self.cx] + t[:, self.cz])
        O = torch.where(self.corner, cnum / (2.0 * self.r1 + 1.0), num / (self.tv + 1.0))
        out = t.clone()
        out[:, self.cell] = (1.0 - self.w) * T0 + self.w * O
        return out.view_as(T)


class _Shots64:
    """Forward, migration, Born and adjoint passes of shots on one grid."""

    def __init__(self, S, case, geoms, v, r1):
        self.S, self.geoms = S, geoms
        self.g = _Grid64(S, case, v, r1, geoms[0]["nx"])
        dev = self.g.dev
        self.s = torch.arange(len(geoms), device=dev)
        self.ru = torch.tensor([q["r_u"] for q in geoms], device=dev)
        self.rx = torch.tensor([q["r_x"] for q in geoms], device=dev)
        q = geoms[0]
        self.cols = torch.arange(q["n"], device=dev) * case["ds"] + q["s_l"]
        self.row, self.nt, self.nt2 = S["d"].s_z, S["nt"], S["d"].nt2
        self.wav = S["wav"].astype(np.float64)

    def zero(self):
        return torch.zeros(len(self.geoms), self.g.nz, self.g.nx, dtype=torch.float64, device=self.g.dev)

    def forward(self, each, keep=True):
        """u(0 .. nt-1); each(k, u(k), u(k-1), u(k-2)) after every step."""
        u0, u1 = self.zero(), self.zero()
        u1[self.s, self.ru, self.rx] = self.wav[0] / 2.0
        hist = [u0, u1]
        each(0, u0, None, None)
        each(1, u1, u0, None)
        for k in range(2, self.nt):
            T = self.g.update(u1, u0)
            if k < self.nt2:
                T[self.s, self.ru, self.rx] += self.wav[k - 1]
            u2 = self.g.boundary(T, u1, u0)
            each(k, u2, u1, u0)
            u0, u1 = u1, u2
            if keep:
                hist.append(u2)
        return hist

    def reconstruct(self, hist):
        """Yields (k, u(k), u(k+1), u(k+2)), the interior stepped backwards."""
        f0, f1 = hist[-1], hist[-2]
        for k in range(self.nt - 3, -1, -1):
            f = self.g.update(f1, f0)
            if k < self.nt2:
                f[self.s, self.ru, self.rx] += self.wav[k + 1]
            f = torch.where(self.g.inner, f, hist[k])
            yield k, f, f1, f0
            f0, f1 = f1, f

    def migrate(self, data, compensated):
        hist = self.forward(lambda *a: None)
        b0, b1 = hist[-1], hist[-2]
        spike = self.zero()
        spike[self.s, self.ru, self.rx] = self.wav[0] / 2.0
        i2 = b1 * b1 + b0 * b0
        su, sq, i1 = (b0 + b1, spike, spike * (b0 + b1)) if compensated else (0.0, 0.0, spike * b1)
        q0, q1 = self.zero(), self.zero()
        for k, u, _, _ in self.reconstruct(hist):
            T = self.g.update(q1, q0)
            x = data[:, :, k + 1]
            T[:, self.row, self.cols] = torch.where(x != 0, x, T[:, self.row, self.cols])
            q = self.g.boundary(T, q1, q0)
            su, sq = (su + u, sq + q) if compensated else (u, q)
            i1 = i1 + sq * su
            i2 = i2 + u * u
            q0, q1 = q1, q
        return i1, i2

    def born(self, refl):
        """(records of the scattered field, background history)."""
        n2, g = self.g.n2, self.g
        m = self.zero()
        for s, q in enumerate(self.geoms):
            w = q["nx"] - 2 * n2
            m[s, n2:g.nz - n2, n2:g.nx - n2] = refl[:, q["x_img"]:q["x_img"] + w]
        rec = torch.zeros(len(self.geoms), len(self.cols), self.nt, dtype=torch.float64, device=g.dev)
        q = [self.zero(), self.zero()]

        def each(k, u2, u1, u0):
            if k < 2:
                return
            T = g.update(q[1], q[0]) + m * (u2 - 2.0 * u1 + u0)
            q[0], q[1] = q[1], g.boundary(T, q[1], q[0])
            rec[:, :, k] = q[1][:, self.row, self.cols]

        return rec, self.forward(each)

    def adjoint(self, resid, hist, grad):
        """Adds each shot's gradient to grad at its image columns."""
        g, n2 = self.g, self.g.n2
        q0, q1, G = self.zero(), self.zero(), self.zero()
        P = g.P[self.row, self.cols]

        def step(k):
            T = g.update(q1, q0, transposed=True)
            T[:, self.row, self.cols] += P * resid[:, :, k]
            return g.boundary(T, q1, q0)

        for k in (self.nt - 1, self.nt - 2):
            q0, q1 = q1, step(k)
        for k, u, u1, u2 in self.reconstruct(hist):
            G += (u2 - 2.0 * u1 + u) * q0
            q0, q1 = q1, step(k)
        G = (G / g.P)[:, n2:g.nz - n2, n2:g.nx - n2]
        for s, q in enumerate(self.geoms):
            grad[:, q["x_img"]:q["x_img"] + G.shape[2]] += G[s]


def _image64(S, case, S64, data):
    """Per-shot image post and stack (kernel.cu:935-1059) in float64."""
    n2, mnz, vmax = S["n2"], S["nz"] - 2 * S["n2"], float(S["vmax"])
    up, down = (torch.zeros(mnz, S["gw"], dtype=torch.float64, device=S64[0].g.dev) for _ in range(2))
    at = 0
    for E in S64:
        n = len(E.geoms)
        d = torch.from_numpy(data[at:at + n, :len(E.cols)]).to(E.g.dev, torch.float64)
        at += n
        cut = (slice(None), slice(n2, E.g.nz - n2), slice(n2, E.g.nx - n2))
        i1, i2 = (f[cut] for f in E.migrate(d, case["compensated"]))
        p = torch.nn.functional.pad(i1[:, None], (1, 1, 1, 1), mode="reflect")[:, 0]
        lap = p[:, 1:-1, 2:] + p[:, 1:-1, :-2] + p[:, 2:, 1:-1] + p[:, :-2, 1:-1] - 4.0 * i1
        u = -lap * E.g.v[cut[1:]] ** 2 / vmax ** 2
        w = i2 + WHITE * i2.abs().amax((1, 2), keepdim=True)
        for s, q in enumerate(E.geoms):
            up[:, q["x_img"]:q["x_img"] + u.shape[2]] += u[s]
            down[:, q["x_img"]:q["x_img"] + u.shape[2]] += w[s]
    up, down = up / S["shots"], down / S["shots"]
    bare = (up == 0) & (down == 0)
    return dict(image=torch.where(bare, up, up / torch.where(bare, torch.ones_like(down), down)),
                illumination=down)


def _conv64(a, W, dil, flip=False):
    """3x3 convolution of [n][c][h][w] as nine shifted products; flip: its
    transpose (the gradient with respect to the input)."""
    n, c, h, w = a.shape
    p = torch.nn.functional.pad(a, (dil,) * 4)
    out = 0.0
    for ky in range(3):
        for kx in range(3):
            y, x = (ky, kx) if not flip else (2 - ky, 2 - kx)
            cut = p[:, :, y * dil:y * dil + h, x * dil:x * dil + w].permute(0, 2, 3, 1).reshape(-1, c)
            out = out + cut @ (W[:, :, ky, kx] if flip else W[:, :, ky, kx].t().contiguous())
    return out.view(n, h, w, -1).permute(0, 3, 1, 2)


def _net64(p, ch, dil, x, t=None):
    """Output of the network, or (loss, gradient) against targets t."""
    layers, o = [], 0
    for a, b in zip(ch, ch[1:]):
        layers.append((p[o:o + a * b * 9].view(b, a, 3, 3), p[o + a * b * 9:o + a * b * 9 + b]))
        o += a * b * 9 + b
    act = [x]
    for i, (W, b) in enumerate(layers):
        z = _conv64(act[-1], W, dil[i]) + b[:, None, None]
        act.append(z.clamp_min(0.0) if i + 1 < len(layers) else z)
    y = act[-1][:, 0] + x[:, 0]
    if t is None:
        return y
    dz = (2.0 / y.numel() * (y - t))[:, None]
    grads = []
    for i in range(len(layers) - 1, -1, -1):
        W, d = layers[i][0], dil[i]
        n, c, h, w = act[i].shape
        pad = torch.nn.functional.pad(act[i], (d,) * 4)
        flat = dz.permute(1, 0, 2, 3).reshape(W.shape[0], -1)
        gw = torch.stack([flat @ pad[:, :, a * d:a * d + h, b * d:b * d + w].permute(0, 2, 3, 1)
                          .reshape(-1, c) for a in range(3) for b in range(3)], dim=2)
        grads = [gw.reshape(-1), flat.sum(1)] + grads
        if i:
            dz = _conv64(dz, W, d, flip=True) * (act[i] > 0)
    return ((y - t) ** 2).mean(), torch.cat(grads)


def _fit64(case, D, dev):
    """One epoch of Adam over the seeded shuffle of cnn.Deblur.fit."""
    n, b, mask = case["n"], min(case["batch"], case["n"]), (1 << 64) - 1
    order, s = list(range(n)), (5 * 6364136223846793005 + 1442695040888963407) & mask
    for i in range(n - 1, 0, -1):
        s = (s * 6364136223846793005 + 1442695040888963407) & mask
        j = (s >> 33) % (i + 1)
        order[i], order[j] = order[j], order[i]
    p = torch.from_numpy(D["p"]).to(dev, torch.float64)
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    for k in range(n // b):
        at = order[k * b:(k + 1) * b]
        x, t = (torch.from_numpy(D[q][at]).to(dev, torch.float64) for q in "xt")
        loss, g = _net64(p, D["ch"], D["dil"], x, t)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - 1e-3 * (m / (1 - 0.9 ** (k + 1))) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
        losses.append(float(loss))
    return dict(loss=np.array([np.mean(losses)]), params=p)


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] in ("fit", "grad", "infer"):
        if work(case)["flops"] > 1e13:
            return None
        D = _patches(case, seed)
        if case["kind"] == "fit":
            return _fit64(case, D, dev)
        p, x, t = (torch.from_numpy(D[q]).to(dev, torch.float64) for q in "pxt")
        if case["kind"] == "infer":
            return torch.cat([_net64(p, D["ch"], D["dil"], x[i:i + 1]) for i in range(len(x))])
        loss, g = _net64(p, D["ch"], D["dil"], x, t)
        return dict(loss=float(loss), grad=g)
    n2, steps = case["n2"], case["nt"] * {"model": 1, "migrate": 3, "aperture": 3, "pairs": 5, "cgls": 10}[case["kind"]]
    nx = case["wmax"] if case["kind"] == "aperture" else case["mod_nx"]
    shots = case["shots"] * case.get("panels", 1)
    cells = shots * (case["mod_nz"] + 2 * n2) * (nx + 2 * n2)
    grids = case["shots"] if case["kind"] == "aperture" else case.get("panels", 1)
    taps = case["nfdmax"] if case["taylor"] else 4
    seconds = steps * (grids * 0.0012 + cells * (taps + 3) * 5e-11)
    if seconds > 15 or cells * case["nt"] * 8 > 6e10:
        return None
    S = _survey(case, seed)
    per = 1 if case["kind"] == "aperture" else case["shots"]
    S64 = [_Shots64(S, case, S["geoms"][i * per:(i + 1) * per], v, r1)
           for i, (v, r1) in enumerate(S["models"])]
    if case["kind"] in ("migrate", "aperture"):
        return _image64(S, case, S64, S["gathers"])
    E = S64[0]
    if case["kind"] == "model":
        rec = torch.zeros(shots, S["n"], S["nt"], dtype=torch.float64, device=dev)

        def each(k, u, *_):
            rec[:, :, k] = u[:, E.row, E.cols]

        E.forward(each, keep=False)
        return rec
    mnz = case["mod_nz"]
    if case["kind"] == "pairs":
        grad = torch.zeros(mnz, S["gw"], dtype=torch.float64, device=dev)
        refl = torch.from_numpy(S["refl"]).to(dev, torch.float64)
        for E in S64:
            E.adjoint(*E.born(refl), grad)
        return grad
    r = torch.from_numpy(S["gathers"]).to(dev, torch.float64)
    misfit = [float((r * r).sum())]
    s = torch.zeros(mnz, S["gw"], dtype=torch.float64, device=dev)
    E.adjoint(r, E.forward(lambda *a: None), s)
    q, _ = E.born(s)
    alpha = (s * s).sum() / (q * q).sum()
    r = r - alpha * q
    return dict(model=alpha * s, misfit=misfit + [float((r * r).sum())])
