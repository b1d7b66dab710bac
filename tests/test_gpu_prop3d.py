"""GPU parity of the 3D forward propagator against the oracle's FP32 mode.

The HIP kernel and the oracle's FP32 mode evaluate the same expressions in
the same order with contraction off, so agreement is bit for bit.  The
oracle reproduces the reference's block-sequential damping order by running
it (objFuncGradient3d_f.cu:638-667); the kernel reproduces it with the
on-read damping rule, so this test pins that rule too.
"""
import numpy as np
import pytest

from common3d import cij_from, layered_model, rel, ricker

pytestmark = pytest.mark.gpu


def _problem(nz=40, ny=36, nx=44, seed=3):
    v, e, d = layered_model(nz, ny, nx, seed=seed)
    return cij_from(v, e, d)


@pytest.mark.parametrize("levels", [1, 2], ids=["1-level", "2-level"])
@pytest.mark.parametrize("arith", [1, 0], ids=["ref-arith", "fp32-arith"])
@pytest.mark.parametrize("absorbing", [True, False])
@pytest.mark.parametrize("dims", [(40, 36, 44), (48, 29, 70), (43, 30, 40)])
def test_forward_shot_bitexact(vti, orc, ctx, absorbing, dims, arith, levels):
    nz, ny, nx = dims
    c11, c13, c33 = _problem(nz, ny, nx)
    npad, dx, dt = 8, 12.5, 1.0e-3
    nt = 130
    lmax = orc.lmax3d(nt)
    w = ricker(nt, dt, 15.0, 0.08)
    sou = 17 + 15 * nx + 13 * nx * ny
    rec = np.array([ix + (ny // 2) * nx + 9 * nx * ny for ix in range(4, nx - 4)], np.int64)
    sts, nnt = 4, (nt - 1) // 4 + 1
    print(f"case dims={dims} absorbing={absorbing} arith={arith} levels={levels}", flush=True)
    mode = orc.REF if arith == 1 else orc.F32
    tr_ref, tr64, st = orc.forward3d(mode, c11, c13, c33, npad, dx, dx, dx, dt, lmax, w, sou, rec, sts, nnt,
                                     absorbing=absorbing, want_state=True)
    with vti.Prop3D(ctx, nx, ny, nz, npad, dx, dx, dx, dt) as p:
        p.set_zchunk(16)
        p.set_arith(arith)
        p.set_levels(levels)
        p.set_model(c11, c13, c33)
        p.reset(sou, np.float32(np.float32(dt) * np.float32(dt)) * w[0])
        tr = p.forward_shot(lmax, w, sou, rec, sts, nnt, absorbing=absorbing)
        cx, cz, px, pz = p.get_state()
    assert np.array_equal(tr, tr_ref), f"trace mismatch rel={rel(tr, tr_ref)}"
    assert np.array_equal(cx, st[0]) and np.array_equal(cz, st[1])
    if absorbing:
        d = orc.init_damping3d(nx, ny, nz, npad)
        dd = (d[: nx * ny].reshape(ny, nx)[None] * d[nx * ny:][:, None, None]).astype(np.float32)
        inner = np.zeros_like(px, bool)
        inner[:, 4:ny - 4, 4:nx - 4] = True
        px = np.where(inner, px * dd, px)
        pz = np.where(inner, pz * dd, pz)
    assert np.array_equal(px, st[2]) and np.array_equal(pz, st[3])
    assert rel(tr, tr64) < 1e-5


def test_zchunk_invariance(vti, ctx):
    """The z-chunk a workgroup marches over changes nothing in the result."""
    nz, ny, nx = 48, 30, 40
    c11, c13, c33 = _problem(nz, ny, nx, seed=7)
    rng = np.random.default_rng(1)
    st0 = [rng.standard_normal((nz, ny, nx)).astype(np.float32) for _ in range(4)]
    outs = []
    for zc in (4, 12, 48):
        with vti.Prop3D(ctx, nx, ny, nz, 6, 10.0, 10.0, 10.0, 1e-3) as p:
            p.set_zchunk(zc)
            p.set_model(c11, c13, c33)
            p.set_state(*st0)
            p.forward_steps(7, absorbing=True)
            outs.append(p.get_state())
    for o in outs[1:]:
        for a, b in zip(o, outs[0]):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("arith", [1, 0], ids=["ref-arith", "fp32-arith"])
@pytest.mark.parametrize("absorbing", [True, False])
def test_two_levels_equal_one_level(vti, ctx, arith, absorbing):
    """Two levels per launch give the bits of one level per launch from an
    arbitrary state -- nonzero values outside the updated interior included
    -- for odd and even step counts and z-chunks down to one 4-plane block."""
    nz, ny, nx = 47, 30, 71
    c11, c13, c33 = _problem(nz, ny, nx, seed=9)
    rng = np.random.default_rng(2)
    st0 = [rng.standard_normal((nz, ny, nx)).astype(np.float32) for _ in range(4)]
    print(f"two-level arith={arith} absorbing={absorbing}", flush=True)
    for nsteps in (6, 7):
        ref = None
        for levels, zc in ((1, 16), (2, 4), (2, 12), (2, 44)):
            with vti.Prop3D(ctx, nx, ny, nz, 6, 10.0, 10.0, 10.0, 1e-3) as p:
                p.set_zchunk(zc)
                p.set_arith(arith)
                p.set_levels(levels)
                p.set_model(c11, c13, c33)
                p.set_state(*st0)
                p.forward_steps(nsteps, absorbing=absorbing)
                out = p.get_state()
            if ref is None:
                ref = out
                assert np.abs(out[0]).max() > 0
            else:
                for a, b in zip(out, ref):
                    assert np.array_equal(a, b), (nsteps, levels, zc)


def _damping(vti, shape, npad):
    """d = dxy * dz of every point the steps update, 1 elsewhere (the
    propagator holds prev / d of the absorbing side)."""
    nz, ny, nx = shape
    d = vti.init_damping3d(nx, ny, nz, npad)
    out = np.ones(shape, np.float32)
    inner = np.s_[: 4 * (nz // 4), 4:ny - 4, 4:nx - 4]
    out[inner] = (d[: nx * ny].reshape(ny, nx)[None] * d[nx * ny:][:, None, None]).astype(np.float32)[inner]
    return out


@pytest.mark.parametrize("arith", [1, 0], ids=["ref-arith", "fp32-arith"])
@pytest.mark.parametrize("kind,dims", [("fwd", (470, 410, 15)), ("grad", (321, 302, 15)), ("rtm", (331, 351, 13))])
def test_streamed_steps_vs_oracle(vti, orc, ctx, kind, dims, arith):
    """Volumes whose rows fill a fifth of their pitch, so that a step's volumes
    pass the size from which it streams past the caches: 4 levels, bit for bit."""
    c, npad, n = _problem(*dims, seed=5), 5, 4
    rng = np.random.default_rng(dims[1])
    sig, lam = ([(rng.standard_normal(dims) * s).astype(np.float32) for _ in range(4)] for s in (1e-3, 1e-6))
    dd = _damping(vti, dims, npad)
    geo = (npad, 12.5, 12.5, 12.5, 1e-3)
    print("streamed", kind, dims, arith, flush=True)
    mode = 1 if kind == "rtm" else 0
    with vti.Prop3D(ctx, dims[2], dims[1], dims[0], *geo) as p:
        p.set_arith(arith)
        p.set_model(*c)
        p.set_state(cur_x=sig[0], cur_z=sig[2], prev_x=sig[1], prev_z=sig[3])
        if kind == "fwd":
            p.forward_steps(n, absorbing=True)
        else:
            p.set_adjoint(mode, cur_x=lam[0], cur_z=lam[2], prev_x=lam[1], prev_z=lam[3])
            p.backward_steps(n, mode=mode)
            la = p.get_adjoint(mode)
        st = p.get_state()
    if kind == "fwd":
        o = [sig[0], sig[1] * dd, sig[2], sig[3] * dd]
        orc.steps3d(orc.REF if arith else orc.F32, o, *c, *geo, n, absorbing=True)
        st = [st[0], st[1], st[2] * dd, st[3] * dd]
    else:
        acc = [np.zeros(dims, np.float32) for _ in range(3 if mode == 0 else 1)]
        o, lo = orc.bwd_steps3d(mode, arith, sig, [lam[0], lam[1] * dd, lam[2], lam[3] * dd], acc, *c, *geo, n)
        for a, b in zip([la[0], la[1], la[2] * dd, la[3] * dd], (lo[0], lo[2], lo[1], lo[3])):
            assert np.abs(b).max() > 0 and np.array_equal(a, b)
        for a, b in zip(la[4], acc):
            assert np.abs(b).max() > 0 and np.array_equal(a, b)
    for a, b in zip(st, (o[0], o[2], o[1], o[3])):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)


@pytest.mark.parametrize("dims", [(8, 9, 9), (16, 17, 71), (19, 75, 133), (36, 25, 390)])
def test_tile_order_vs_oracle(vti, orc, ctx, dims):
    """1 to 63 tiles a z-chunk, fewer than the XCDs and no multiple of them, in
    1 to 9 chunks: every tile of every chunk is stepped once."""
    c, npad, n = _problem(*dims, seed=dims[2]), 3, 3
    rng = np.random.default_rng(dims[1])
    st = [(rng.standard_normal(dims) * 1e-3).astype(np.float32) for _ in range(4)]
    geo = (npad, 12.5, 12.5, 12.5, 1e-3)
    print("tile order", dims, flush=True)
    want = [a.copy() for a in st]
    orc.steps3d(orc.REF, want, *c, *geo, n, absorbing=False)
    for levels, zc in ((1, 0), (1, 8), (2, 4)):
        with vti.Prop3D(ctx, dims[2], dims[1], dims[0], *geo) as p:
            p.set_levels(levels)
            if zc:
                p.set_zchunk(zc)
            p.set_model(*c)
            p.set_state(cur_x=st[0], cur_z=st[2], prev_x=st[1], prev_z=st[3])
            p.forward_steps(n, absorbing=False)
            got = p.get_state()
        # 3 levels (odd): the oracle's arrays have changed roles
        for a, b in zip(got, (want[1], want[3], want[0], want[2])):
            assert np.abs(b).max() > 0 and np.array_equal(a, b)
