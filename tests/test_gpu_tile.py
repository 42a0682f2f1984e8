"""Whole steps in one launch (the tile kernel of small batches) against the
oracle and against the marching kernels, bit for bit."""
import numpy as np
import pytest

from cases import build_case, hip_context, oracle_engine, synth_gather

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mod_nz,mod_nx,n2,nfdmax,ilste,icompen", [
    (44, 44, 10, 1, 1, 1),     # 64 columns: one tile column, no tile without frame cells
    (45, 107, 10, 4, 0, 1),    # 127 columns, 65 rows: one row into the ninth tile row
    (43, 109, 12, 6, 1, 0),    # 133 columns: 5 into the third tile
    (120, 170, 12, 12, 1, 1),  # the longest operator, tiles with and without frame cells
    (90, 150, 30, 3, 1, 1)])   # a wide frame: tiles of frame cells alone
def test_tile_steps_equal_oracle(mod_nz, mod_nx, n2, nfdmax, ilste, icompen):
    from rtm_gpu_amd import hip
    case = build_case(name="tile", mod_nz=mod_nz, mod_nx=mod_nx, n2=n2, nfdmax=nfdmax, ilste=ilste,
                      nfdmin=min(2, nfdmax), icompen=icompen, nt=100, tao=0.0008, src_x1=20)
    nt, inner = case["cfg"]["nt"], (slice(n2, -n2), slice(n2, -n2))
    seis = synth_gather(case)
    e = oracle_engine(case, record=1)
    ctx = hip_context(case, nshot=1, record=1)
    ctx.set_gathers(seis[None])
    e.forward_begin()
    ctx.forward_begin()
    for n in (1, 40, nt):
        e.forward_advance(n)
        ctx.forward_advance(n)
        assert np.array_equal(ctx.field(hip.FIELD_U), e.field(0)), n
    assert np.array_equal(ctx.records()[0], e.record())
    e.backward_begin(seis)
    ctx.backward_begin()
    for n in (1, 40, nt):
        e.backward_advance(n)
        ctx.backward_advance(n)
        assert np.array_equal(ctx.field(hip.FIELD_Q), e.field(2)), n
        for which, name in ((3, hip.FIELD_I1), (4, hip.FIELD_I2)):
            assert np.array_equal(ctx.field(name)[inner], e.field(which)[inner]), (n, which)
    ctx.close()


@pytest.mark.parametrize("nshot,mod_nz,mod_nx", [(3, 60, 107), (24, 300, 330)])
@pytest.mark.parametrize("ilste,strip_format", [(0, 0), (0, 1), (1, 2)])
def test_tile_passes_equal_marching(nshot, mod_nz, mod_nx, ilste, strip_format):
    """Migration, Born modelling and its adjoint of a small batch and of one
    large enough for tiles of two cells per thread (24 x 320 x 350 cells)."""
    from rtm_gpu_amd import hip
    case = build_case(name="tilemarch", mod_nz=mod_nz, mod_nx=mod_nx, n2=10, nt=60, nshot=nshot,
                      depth_step=2.0, ilste=ilste)
    rng = np.random.default_rng(4)
    n, nt = case["cfg"]["n"], case["cfg"]["nt"]
    seis = (0.01 * rng.standard_normal((nshot, n, nt))).astype(np.float32)
    refl = (0.1 * rng.standard_normal((mod_nz, mod_nx))).astype(np.float32)
    out = []
    for zseg in (0, 16):  # 16 rows per wave: the marching kernels
        ctx = hip_context(case, nshot=nshot, record=1, zseg=zseg, strip_format=strip_format)
        ctx.set_gathers(seis)
        ctx.migrate()
        got = [ctx.field(w, shot=nshot - 1) for w in (hip.FIELD_U, hip.FIELD_Q, hip.FIELD_I1,
                                                     hip.FIELD_I2)]
        got.append(ctx.strip(nshot - 1, nt - 1))
        ctx.set_reflectivity(refl)
        got.append(ctx.born())
        got.append(ctx.field(hip.FIELD_Q, shot=nshot - 1))
        got.append(ctx.adjoint(seis))
        out.append(got)
        ctx.close()
    for i, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), i


@pytest.mark.parametrize("mod_nz,mod_nx,n", [
    (120, 170, 8),    # tiles without frame cells that start at row n2 and that end at nz - n2
    (91, 150, 5),     # rows up to nz - n2 = 96
    (92, 150, 12)])   # ... 104, the longest operator
def test_tile_steps_with_a_frame_as_deep_as_the_operator(mod_nz, mod_nx, n):
    test_tile_steps_equal_oracle(mod_nz, mod_nx, n, n, 1, 1)
