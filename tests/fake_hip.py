"""CPU tests of the host code of librtm_hip.so on tests/fake_hip.cpp, a HIP
runtime whose kernels are logged instead of run."""
import ctypes as C
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SO = os.path.join(HERE, "_build", "libfake_hip.so")


def build():
    src = os.path.join(HERE, "fake_hip.cpp")
    csrc = os.path.join(ROOT, "rtm_gpu_amd", "csrc")
    deps = [src, os.path.join(csrc, "rtm_kernels.h"), os.path.join(csrc, "rtm_plan.h")]
    if os.path.exists(SO) and all(os.path.getmtime(d) <= os.path.getmtime(SO) for d in deps):
        return
    os.makedirs(os.path.dirname(SO), exist_ok=True)
    tmp = f"{SO}.{os.getpid()}"
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I", csrc, src, "-o", tmp], check=True)
    os.replace(tmp, SO)


def run(script):
    """Runs a script in a process of its own with the names below defined and
    returns what it hands to `out`."""
    build()
    code = ("import sys; sys.path[:0] = [%r, %r]\nfrom fake_hip import *\nfake = load()\n" % (HERE, ROOT)) + script
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    return json.loads(r.stdout.strip().splitlines()[-1])


# ---- in the script's process
fake = None


def load():
    global fake
    fake = C.CDLL(SO, mode=C.RTLD_GLOBAL)  # before librtm_hip.so: its HIP symbols bind here
    fake.fake_log.restype = C.c_char_p
    fake.fake_used.restype = C.c_size_t
    fake.fake_limit.argtypes = [C.c_size_t]
    fake.fake_cost.argtypes = [C.c_char_p, C.c_double]
    return fake


def out(x):
    print(json.dumps(x))


def log():
    """The launches since the last call, as dicts."""
    rows = []
    for line in fake.fake_log().decode().splitlines():
        name, *rest = line.split(" ")
        row = dict(kernel=name, dead=rest[-1:] == ["DEAD"])
        row.update((k, int(v)) for k, v in (r.split("=") for r in rest if "=" in r))
        rows.append(row)
    fake.fake_clear()
    return rows


def context(nz=440, nx=618, n2=20, nfd=3, nt=60, shots=41, gw=None, **more):
    """A Taylor context with a constant model, its shots set."""
    import numpy as np
    from rtm_gpu_amd import hip
    n = nx - 2 * n2
    ctx = hip.Context(nz=nz, nx=nx, n2=n2, nfdmax=nfd, nt=nt, nt2=nt, ilste=1, icompen=1, s_l=n2,
                      s_r=nx - n2 - 1, s_z=n2, ds=1, n=n, tao2=1e-6, h2=1e-2, taoh=1e-4, taoh2=1e-8,
                      hzx2_1=1.0, max_shots=shots, **more)
    set_model(ctx, nz, nx, n2, nfd)
    ctx.set_wavelet(np.zeros(nt + 1, np.float32))
    return ctx


def set_model(ctx, nz, nx, n2, nfd, v=1500.0):
    import numpy as np
    z = np.full((nz, nx), v, np.float32)
    ctx.set_model(z, z * 0, np.zeros(n2 + 1), np.ones(nfd + 1), None, 1, 1500.0, 1.0)


def shots(ctx, n):
    ctx.set_shots([ctx.n2] * n, [ctx.n2 + 1] * n)


def ragged(ctx, n, widths=None):
    """A ragged batch of n shots (widths: of each, default the grid's)."""
    n2 = ctx.n2
    ctx.set_shot_geometry([dict(nx=w, r_u=n2, r_x=n2 + 1, s_l=n2, s_r=w - n2 - 1, n=w - 2 * n2, x_img=0)
                           for w in widths or [ctx.nx] * n])


def window(ctx, shot, v, nx=None):
    import numpy as np
    a = np.full((ctx.nz, nx or ctx.nx), v, np.float32)
    ctx.set_shot_model(shot, a, a * 0)
