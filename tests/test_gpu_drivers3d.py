"""GPU parity of the 3D reference-signature drivers against the oracle.

objFuncGradientCij3d_f, objFuncCij3d_f, rtmCij3d_f and modelDataCij3d_f on a
small seeded problem.  Single-shot results are bit-exact against the oracle's
REF mode (the reference's own mixed arithmetic, evaluated in the same order); multi-shot gradients differ only by the
cross-shot accumulation, which the library does in FP64 (the reference sums
shots in FP32), and are compared with a tolerance.  Every result also states
its error against the FP64 oracle.
"""
import numpy as np
import pytest

from common3d import rel
from common3d_drivers import problem

pytestmark = pytest.mark.gpu


def _boundaries(vti, P):
    nx, ny, nz, npad = P["nx"], P["ny"], P["nz"], P["npad"]
    nb = P["nbnd"]
    padb = np.zeros(3 * nb, np.float32)
    for k in range(3):
        vti.check(vti.lib.vti_get_boundary(vti.ptr(padb[k * nb:(k + 1) * nb]), vti.ptr(P["cij"][k]), nx, ny, nz, npad))
    randb = (padb * np.tile(P["shell_scale"], 3)).astype(np.float32)
    return padb, randb


def _obs(vti, ctx, P):
    return vti.model_data3d(ctx, P["souloc"], np.arange(len(P["souloc"])), P["recloc"], P["w"], *P["ctrue"], P["nt"],
                            P["npad"], P["o"], P["d"], P["dt"], P["rate"])


def test_model_data_bitexact(vti, orc, ctx):
    P = problem()
    nx, ny, nz = P["nx"], P["ny"], P["nz"]
    dd = _obs(vti, ctx, P)
    sts = int(round(P["rate"] / P["dt"]))
    nnt = (P["nt"] - 1) // sts + 1
    nr = int(P["souloc"][0, 3])
    lmax = orc.lmax3d(P["nt"])
    dx = P["d"][0]
    for s in range(len(P["souloc"])):
        sx, sy, sz = (int(np.float32(P["souloc"][s, k]) / np.float32(dx)) for k in range(3))
        sou = sx + sy * nx + sz * nx * ny
        rb = int(np.float32(P["recloc"][0, 2]) / np.float32(dx) / np.float32(4))
        rec = []
        r0 = int(P["souloc"][s, 4])
        for r in P["recloc"][r0:r0 + nr]:
            ix, iy, iz = (int(np.float32(r[k]) / np.float32(dx)) for k in range(3))
            rec.append(ix + iy * nx + (iz % 4) * nx * ny + 4 * rb * nx * ny)
        tr, _, _ = orc.forward3d(orc.REF, *P["ctrue"], P["npad"], dx, dx, dx, P["dt"], lmax, P["w"], sou,
                                 np.array(rec), sts, nnt, absorbing=True)
        tr[P["recloc"][r0:r0 + nr, 3] == 0] = 0.0
        assert np.array_equal(dd[r0 * nnt:(r0 + nr) * nnt].reshape(nr, nnt), tr)


@pytest.mark.parametrize("obs_kind", ["zero", "model"])
@pytest.mark.parametrize("nshot", [1, 2])
def test_objfunc_gradient_vs_oracle(vti, orc, ctx, nshot, obs_kind):
    """obs 'zero': J = 0.5|d|^2, a well-conditioned gradient, where the FP64
    bar (1e-4) applies.  obs 'model': data of a model 4% different in a blob,
    so the residual is ~1% of the data and every FP32-storage rounding of the
    traces is magnified ~100x in the residual -- the reference's own arithmetic
    sits ~1e-3 from FP64 there; the error is reported, and a loose bound only
    guards against gross mistakes.  Parity with the reference's arithmetic
    is bit-exact in both cases."""
    P = problem()
    if obs_kind == "zero":
        nr_tot = len(P["recloc"])
        obs = np.zeros(nr_tot * ((P["nt"] - 1) // 4 + 1), np.float32)
    else:
        obs = _obs(vti, ctx, P)
    padb, randb = _boundaries(vti, P)
    shots = np.arange(nshot)
    args = (P["souloc"], shots, P["recloc"], P["w"])
    rest = (P["nt"], P["npad"], P["o"], P["d"], P["dt"], P["rate"], obs)
    cg = P["cij"].copy()
    f_gpu, g_gpu = vti.objfunc_gradient3d(ctx, *args, cg, padb, randb, *rest)
    co = P["cij"].copy()
    f_orc, g_orc = orc.gradient3d(orc.REF, *args, co, padb, randb, *rest)
    c64 = P["cij"].copy()
    f64, g64 = orc.gradient3d(orc.F64, *args, c64, padb, randb, *rest)
    e_g, e_f = rel(g_gpu, g64), abs(f_gpu - f64) / abs(f64)
    print(f"nshot={nshot} obs={obs_kind} f_gpu={f_gpu:.9e} f_orc={f_orc:.9e} f64={f64:.9e} "
          f"grad rel vs ref-arith oracle {rel(g_gpu, g_orc):.2e}; vs FP64 oracle: grad {e_g:.2e} f {e_f:.2e}",
          flush=True)
    assert np.array_equal(cg, co), "the caller's cij must end up holding the random boundary shell"
    assert abs(f_gpu - f_orc) <= 2e-7 * abs(f_orc)
    if nshot == 1:
        assert np.array_equal(g_gpu, g_orc)
    else:
        assert rel(g_gpu, g_orc) < 1e-5
    if obs_kind == "zero":
        assert e_g < 1e-4 and e_f < 1e-4
    else:
        assert e_g < 2e-2 and e_f < 2e-3
    f_only = vti.objfunc_gradient3d(ctx, *args, P["cij"].copy(), padb, None, *rest, gradient=False)
    assert f_only == f_gpu


@pytest.mark.parametrize("variant", ["agc", "tpow"])
def test_objective_variants_vs_oracle(vti, orc, ctx, variant):
    """objtype=1 (AGC residual, agc.cpp:70-101, half width 6) and the tpow=
    gain (agc.cpp:103-115): the GPU path against the oracle's restatement in
    the reference arithmetic, one shot.  AGC sums, divisions and square roots
    run in the reference's order and rounding, and the gain is formed with the
    host's powf as the reference forms it, so both gradients are bit-exact."""
    P = problem()
    obs = _obs(vti, ctx, P)
    padb, randb = _boundaries(vti, P)
    args = (P["souloc"], np.arange(1), P["recloc"], P["w"])
    rest = (P["nt"], P["npad"], P["o"], P["d"], P["dt"], P["rate"], obs)
    kw = dict(objtype=1, halfwidth=6) if variant == "agc" else dict(tpow=1.5, ot=0.001)
    print("3d objective variant", variant, flush=True)
    f_gpu, g_gpu = vti.objfunc_gradient3d(ctx, *args, P["cij"].copy(), padb, randb, *rest, **kw)
    f_orc, g_orc = orc.gradient3d(orc.REF, *args, P["cij"].copy(), padb, randb, *rest, **kw)
    f64, g64 = orc.gradient3d(orc.F64, *args, P["cij"].copy(), padb, randb, *rest, **kw)
    print(f"  f_gpu={f_gpu:.9e} f_orc={f_orc:.9e} f64={f64:.9e} grad rel vs FP64 {rel(g_gpu, g64):.2e}",
          flush=True)
    assert np.abs(g_orc).max() > 0
    assert abs(f_gpu - f_orc) <= 2e-6 * abs(f_orc)
    assert np.array_equal(g_gpu, g_orc)
    assert rel(g_gpu, g64) < 3e-2


def test_rtm_vs_oracle(vti, orc, ctx):
    P = problem()
    obs = _obs(vti, ctx, P)
    rec3 = np.ascontiguousarray(P["recloc"][:, :3])
    shots = np.array([0])
    args = (P["souloc"], shots, rec3, P["w"], *P["cij"], P["nt"], P["npad"], P["o"], P["d"], P["dt"], P["rate"], obs)
    img = vti.rtm3d(ctx, *args)
    ref = orc.rtm3d(orc.REF, *args)
    r64 = orc.rtm3d(orc.F64, *args)
    print(f"rtm rel vs FP64 oracle {rel(img, r64):.2e}", flush=True)
    assert np.array_equal(img, ref)
    assert rel(img, r64) < 1e-3


@pytest.mark.parametrize("nz,ny,nx,npad", [(41, 36, 44, 1), (29, 33, 71, 14), (34, 30, 300, 9)])
def test_shells_vs_oracle(vti, orc, ctx, nz, ny, nx, npad):
    """The coefficient volumes get their shells on the device: packed values
    that differ from the model's everywhere, from a shell one point thick to
    one that leaves a single interior plane.  Equal to the oracle bit for bit."""
    P = problem(nz=nz, ny=ny, nx=nx, npad=npad, nt=67, ns=1)
    padb, randb = _boundaries(vti, P)
    padb = (padb * np.random.default_rng(nx).uniform(0.8, 1.0, padb.size)).astype(np.float32)
    obs = np.zeros(len(P["recloc"]) * ((P["nt"] - 1) // 4 + 1), np.float32)
    args = (P["souloc"], np.arange(1), P["recloc"], P["w"])
    rest = (P["nt"], npad, P["o"], P["d"], P["dt"], P["rate"], obs)
    print("3d shells", nz, ny, nx, npad, flush=True)
    cg, co = P["cij"].copy(), P["cij"].copy()
    f, g = vti.objfunc_gradient3d(ctx, *args, cg, padb, randb, *rest)
    fo, go = orc.gradient3d(orc.REF, *args, co, padb, randb, *rest)
    assert np.abs(go).max() > 0
    assert np.array_equal(g, go) and np.array_equal(cg, co)
    assert abs(f - fo) <= 2e-7 * abs(fo)


@pytest.mark.parametrize("edge", [False, True], ids=["interior", "outside"])
def test_receiver_planes_vs_oracle(vti, orc, ctx, edge):
    """Receivers in each of the four planes of their block, the first and the
    last interior column among them ("outside": one past the updated interior,
    which takes the injection as a launch of its own).  Bit for bit."""
    P = problem(nz=40, ny=25, nx=71, npad=6, nt=131, ns=1)
    d = P["d"][0]
    for k in range(len(P["recloc"])):
        P["recloc"][k, 2] = (8 + k % 4) * d + 0.1
    if edge:
        P["recloc"][2, 0] = d + 0.1
    padb, randb = _boundaries(vti, P)
    obs = _obs(vti, ctx, P)
    print("3d receiver planes", edge, flush=True)
    rest = (P["nt"], P["npad"], P["o"], P["d"], P["dt"], P["rate"])
    args = (P["souloc"], np.arange(1), P["recloc"], P["w"])
    _, g = vti.objfunc_gradient3d(ctx, *args, P["cij"].copy(), padb, randb, *rest, np.zeros_like(obs))
    _, go = orc.gradient3d(orc.REF, *args, P["cij"].copy(), padb, randb, *rest, np.zeros_like(obs))
    assert np.abs(go).max() > 0 and np.array_equal(g, go)
    args = (P["souloc"], np.arange(1), np.ascontiguousarray(P["recloc"][:, :3]), P["w"], *P["cij"], *rest, obs)
    img, ref = vti.rtm3d(ctx, *args), orc.rtm3d(orc.REF, *args)
    assert np.abs(ref).max() > 0 and np.array_equal(img, ref)
