"""The resident 2D kernels (one launch per pass, every shot's state on the
chip) against the per-level kernels, which `levels=1` asks for: the same bits
at the edges of their tiles (64 columns, 4 rows to a wavefront's 6), for ragged
last tiles, with several receivers in one column, in waves of several shots,
and through the fallback for a grid that does not fit the chip."""
import ctypes

import numpy as np
import pytest

from common2d import args2d, layered2d, problem2d
from common3d import cij_from, ricker

pytestmark = pytest.mark.gpu


def _probe(vti, ctx, rows=0, raised=0):
    """Has the next passes take `rows` rows a wavefront (0: the fastest) and the
    `raised`th of them start with its abort flag raised (0: none); returns the
    passes launched since the last call, the runs that gave up and the row
    counts that ran."""
    seen = (ctypes.c_int * 3)()
    assert vti.lib.vti_ctx_resident_probe(ctx.h, rows, raised, seen) == 0
    return seen[0], seen[1], {r for r in range(8) if seen[2] >> r & 1}


def _shots(widths, nz, npad, nt, vertical=False, seed=1):
    rng = np.random.default_rng(seed)
    NX = max(widths) + 7
    nnz = nz + 2 * npad
    c = cij_from(*layered2d(nnz, NX + 2 * npad, seed))
    shots, rloc = [], []
    for w in widths:
        w2 = w + 2 * npad
        if vertical:  # a receiver in every interior row of two columns
            cols = sorted({4, w2 - 5})
            r = [(x, z) for x in cols for z in range(4, nnz - 4)]
        else:
            r = [(x, 4 + (nnz - 8) // 2) for x in range(4, w2 - 4)]
        shots.append((int(rng.integers(0, NX - w + 1)), w, 4 + (w2 - 8) // 2, 4, len(r), len(rloc)))
        rloc += r
    nnt = (nt - 1) // 4 + 1
    data = (1e-7 * rng.standard_normal(nnt * len(rloc))).astype(np.float32)
    return data, c, ricker(nt, 1e-3, 25.0, 0.02), np.array(shots, np.int32), np.array(rloc, np.int32), \
        (NX, nz, nt, npad, 10.0, 10.0, 1e-3, 4e-3)


@pytest.mark.parametrize("snap", ["fp32", "s16"])
@pytest.mark.parametrize("widths,nz,npad,nt,vertical", [
    ((1,), 1, 4, 9, False),                    # a single interior point
    ((64,), 4, 4, 21, False),                  # one tile exactly
    ((65, 67, 128), 5, 4, 29, False),          # last tiles of 1, 3 and 64 columns, 5 rows
    ((70, 61), 93, 5, 61, True),               # 97 rows: ragged for every row count; receivers down two columns
    ((200, 90, 131, 64, 177), 60, 12, 81, False),
    ((500,), 300, 20, 61, False),              # several hundred tiles, the waves still apart (a zero gradient)
])
def test_resident_equals_per_level(vti, ctx, widths, nz, npad, nt, vertical, snap):
    data, c, w, shots, rloc, rest = _shots(widths, nz, npad, nt, vertical)
    print("resident", widths, nz, npad, nt, snap, flush=True)
    f0, g0 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest, levels=1, snap=snap)
    f1, g1 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest, snap=snap)
    assert np.isfinite(g0).all() and f0 > 0 and (nt == 61 or g0.any())
    assert f0 == f1 and np.array_equal(g0, g1)


def test_grid_beyond_the_chip(vti, ctx):
    """1.2 M points do not fit: the default call then runs the two-level kernels."""
    data, c, w, shots, rloc, rest = _shots((1500,), 700, 20, 9)
    print("resident fallback by size", flush=True)
    f0, g0 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest, levels=1)
    f1, g1 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest)
    assert f0 == f1 and np.array_equal(g0, g1)


@pytest.mark.parametrize("nx,nz,npad,nt", [(2, 5, 4, 21), (64, 12, 4, 61), (65, 17, 4, 61), (131, 97, 5, 81),
                                           (300, 130, 12, 41)])
def test_resident_product_and_image_vs_oracle(vti, orc, ctx, nx, nz, npad, nt):
    """The Gauss-Newton product and the RTM image of a shot that fits the chip
    equal the oracle's FP32 restatement bit for bit at the edges of the tiles."""
    P = problem2d(vti, nx=nx, nz=nz, npad=npad, nt=nt, ns=1)
    print("resident product and image", nx, nz, npad, nt, flush=True)
    dc = [(1e-2 * (a - b)).astype(np.float32) for a, b in zip(P["ctrue"], P["c"])]
    dc[0][:, ::3] += np.float32(1e3)
    a = args2d(P)
    h = vti.gn_hessian2d(ctx, *P["c"], *dc, P["w"], P["sloc"], P["rloc"], P["taper"], *a)
    ho = orc.fg2d(orc.F32, True, None, *P["c"], dc, P["w"], P["sloc"], P["rloc"], P["taper"], *a)[1]
    assert np.array_equal(h, ho)
    data = (1e-7 * np.random.default_rng(3).standard_normal(((nt - 1) // 4 + 1, P["nr"]))).astype(np.float32)
    img = vti.rtm2d(ctx, data, *P["c"], P["w"], P["sloc"], P["rloc"], P["taper"], *a)
    assert np.array_equal(img, orc.rtm2d(orc.F32, data, *P["c"], P["w"], P["sloc"], P["rloc"], P["taper"], *a))


@pytest.mark.parametrize("max_wave,raised", [(0, 1), (2, 2)])
def test_plan_runs_resident_again_after_giving_up(vti, ctx, max_wave, raised):
    """A plan's run that gives up (in its first wave, in its second) falls back
    to the per-level kernels, and its next run is resident again: same bits."""
    data, c, w, shots, rloc, rest = _shots((70, 61, 90), 12, 5, 61)
    print("resident plan giving up", max_wave, raised, flush=True)
    f0, g0 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest, levels=1)
    assert g0.any()
    waves = 1 if max_wave == 0 else 3
    with vti.BatchPlan(ctx, data, w, shots, rloc, *rest, max_wave=max_wave) as plan:
        for k in range(3):
            _probe(vti, ctx, raised=raised if k == 1 else 0)
            f1, g1 = plan.run(*c)
            passes, gone, _ = _probe(vti, ctx)
            assert f0 == f1 and np.array_equal(g0, g1)
            assert passes == 2 * waves and gone == (1 if k == 1 else 0)
