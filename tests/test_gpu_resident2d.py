"""The resident 2D kernels (one launch per pass, every shot's state on the
chip) against the per-level kernels, which `levels=1` or a context set so asks
for, and the oracle: the same bits at the edges of their tiles (64 columns, 4 to
24 rows), for ragged last tiles, with several receivers in one lane, for every
row count of a wavefront and every pass, in waves of several shots, from several
contexts at once, through the fallback for a grid that does not fit the chip and
after a run that gave up."""
import contextlib
import ctypes
import threading

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


@contextlib.contextmanager
def _by_level(vti):
    with vti.Context(0) as c:
        c.set_resident(False)
        yield c


def _shots(widths, nz, npad, nt, vertical=False, seed=1):
    rng = np.random.default_rng(seed)
    NX = max(widths) + 7
    nnz = nz + 2 * npad
    c = cij_from(*layered2d(nnz, NX + 2 * npad, seed))
    shots, rloc = [], []
    for w in widths:
        w2 = w + 2 * npad
        mid, xs = 4 + (nnz - 8) // 2, 4 + (w2 - 8) // 2
        if vertical:  # a receiver in every interior row of three columns
            cols = sorted({4, min(xs + 3, w2 - 5), w2 - 5})
            r = [(x, z) for x in cols for z in range(4, nnz - 4)]
        else:
            r = [(x, mid) for x in range(4, w2 - 4)]
        shots.append((int(rng.integers(0, NX - w + 1)), w, xs, max(4, mid - 3), len(r), len(rloc)))
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
    ((500,), 300, 20, 161, False),             # several hundred tiles of several rows a wavefront
])
def test_resident_equals_per_level(vti, ctx, widths, nz, npad, nt, vertical, snap):
    data, c, w, shots, rloc, rest = _shots(widths, nz, npad, nt, vertical)
    print("resident", widths, nz, npad, nt, snap, flush=True)
    f0, g0 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest, levels=1, snap=snap)
    _probe(vti, ctx)
    f1, g1 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest, snap=snap)
    passes, gone, rows = _probe(vti, ctx)
    assert np.isfinite(g0).all() and g0.any()
    assert abs(f0 / (0.5 * np.sum(data.astype(np.float64) ** 2)) - 1) > 1e-4  # the traces are seen
    assert f0 == f1 and np.array_equal(g0, g1)
    assert passes == 2 and gone == 0
    if widths == (500,):
        assert max(rows) > 1
        _seen_across_tiles(g1[:, :, shots[0, 0]:], shots[0], nz + 2 * npad, {4, 8, 12, 16, 24})


def _seen_across_tiles(g, shot, nnz, heights):
    """The gradient is nonzero at both sides of the tile edges nearest the source."""
    xs, zs = int(shot[2]), int(shot[3])
    e = 4 + 64 * round((xs - 4) / 64)
    assert abs(e - xs) < 16 and all(g[:, zs - 2:zs + 3, x].any() for x in (e - 1, e))
    for th in heights:
        e = 4 + th * round((zs - 4) / th)
        if 4 < e < nnz - 4:
            assert all(g[:, z, xs - 2:xs + 3].any() for z in (e - 1, e)), th


@pytest.mark.parametrize("snap", ["fp32", "s16"])
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 6])
def test_every_row_count(vti, ctx, rows, snap):
    """The gradient's two passes with each row count of a wavefront, on a
    grid of several tiles either way (95 interior rows: a ragged last tile for all),
    with a receiver in every row of three columns: several to a lane."""
    data, c, w, shots, rloc, rest = _shots((135, 61), 93, 5, 121, vertical=True)
    print("resident rows", rows, snap, flush=True)
    f0, g0 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest, levels=1, snap=snap)
    _probe(vti, ctx, rows)
    f1, g1 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest, snap=snap)
    passes, gone, ran = _probe(vti, ctx)
    assert f0 == f1 and np.array_equal(g0, g1)
    assert passes == 2 and gone == 0 and ran == {rows}
    _seen_across_tiles(g1[:, :, shots[0, 0]:], shots[0], 103, {4 * rows})


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 6])
def test_every_row_count_of_product_and_image(vti, orc, ctx, rows):
    """The same for the Born pass and its adjoint, and for the slices and
    the image, with a dipole in every second row of three columns: both poles in
    a lane, or in two wavefronts, or in two tiles."""
    P = problem2d(vti, nx=131, nz=97, npad=5, nt=81, ns=1)
    print("resident rows of product and image", rows, flush=True)
    a, (sx, sz) = args2d(P), (70, 52)
    dc = [(1e-2 * (x - y)).astype(np.float32) for x, y in zip(P["ctrue"], P["c"])]
    dc[0][:, ::3] += np.float32(1e3)

    def receivers(step):
        return np.array([(x, z) for x in (4, sx + 3, P["nnx"] - 5) for z in range(4, P["nnz"] - 5, step)], np.int32)

    rloc = receivers(1)
    sloc = np.array([[sx, sz, len(rloc), 0]], np.int32)
    ho = orc.fg2d(orc.F32, True, None, *P["c"], dc, P["w"], sloc, rloc, P["taper"], *a)[1]
    _probe(vti, ctx, rows)
    h = vti.gn_hessian2d(ctx, *P["c"], *dc, P["w"], sloc, rloc, P["taper"], *a)
    passes, gone, ran = _probe(vti, ctx, rows)
    assert np.array_equal(h, ho) and passes == 2 and gone == 0 and ran == {rows}
    _seen_across_tiles(h.reshape(3, P["nnz"], P["nnx"]), (0, 0, sx, sz), P["nnz"], {4 * rows})
    rloc = receivers(2)
    sloc = np.array([[sx, sz, len(rloc), 0]], np.int32)
    data = (1e-7 * np.random.default_rng(3).standard_normal((21, len(rloc)))).astype(np.float32)
    io = orc.rtm2d(orc.F32, data, *P["c"], P["w"], sloc, rloc, P["taper"], *a)
    _probe(vti, ctx, rows)
    img = vti.rtm2d(ctx, data, *P["c"], P["w"], sloc, rloc, P["taper"], *a)
    passes, gone, ran = _probe(vti, ctx)
    assert np.array_equal(img, io) and passes == 2 and gone == 0 and ran == {rows}
    _seen_across_tiles(img.reshape(1, P["nnz"], P["nnx"]), (0, 0, sx, sz), P["nnz"], {4 * rows})


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


@pytest.mark.parametrize("snap", ["fp32", "s16"])
@pytest.mark.parametrize("max_wave,raised", [(0, 1), (2, 2)])
def test_plan_runs_resident_again_after_giving_up(vti, ctx, max_wave, raised, snap):
    """A plan's run that gives up (in its first wave, in its second) falls back
    to the per-level kernels, and its next run is resident again: same bits."""
    data, c, w, shots, rloc, rest = _shots((70, 61, 90), 12, 5, 61)
    print("resident plan giving up", max_wave, raised, snap, flush=True)
    f0, g0 = vti.objfunc_gradient2d_batch(ctx, data, *c, w, shots, rloc, *rest, levels=1, snap=snap)
    assert g0.any()
    waves = 1 if max_wave == 0 else 3
    with vti.BatchPlan(ctx, data, w, shots, rloc, *rest, max_wave=max_wave, snap=snap) as plan:
        for k in range(3):
            _probe(vti, ctx, raised=raised if k == 1 else 0)
            f1, g1 = plan.run(*c)
            passes, gone, _ = _probe(vti, ctx)
            assert f0 == f1 and np.array_equal(g0, g1)
            assert passes == 2 * waves and gone == (1 if k == 1 else 0)


@pytest.mark.parametrize("raised", [1, 2, 3, 4])
@pytest.mark.parametrize("call", ["batch", "gradient", "modeling", "product", "image"])
def test_call_that_gives_up_is_done_by_level(vti, ctx, call, raised):
    """A pass of a call finds its wait run out: in the first shot or wave or in a
    later one, in the pass before or after the snapshots.  What the passes before
    it left in the sums, the traces and the images does not reach the result."""
    P = problem2d(vti, nx=290, nz=250, npad=12, nt=61, ns=4) if call == "modeling" else \
        problem2d(vti, nx=90, nz=20, npad=6, nt=81, ns=4)
    a, geo = args2d(P), (P["w"], P["sloc"], P["rloc"], P["taper"])
    print("giving up", call, raised, flush=True)
    dc = [(1e-2 * (x - y)).astype(np.float32) for x, y in zip(P["ctrue"], P["c"])]
    dc[0][:, ::3] += np.float32(1e3)
    data = (1e-7 * np.random.default_rng(3).standard_normal((P["nt"] // 4 + 1, P["nr"]))).astype(np.float32)
    shots = np.array([(0, P["nx"], ix, iz, nr, r0) for ix, iz, nr, r0 in P["sloc"]], np.int32)
    cat = np.concatenate([data[:, r0:r0 + nr].ravel() for _, _, nr, r0 in P["sloc"]])

    def run(c):
        if call == "batch":  # four waves of a shot, two in flight
            return vti.objfunc_gradient2d_batch(c, cat, *P["c"], P["w"], shots, P["rloc"], *a, max_wave=2)
        if call == "gradient":  # one wave
            return vti.objfunc_gradient2d(c, data, *P["c"], *geo, *a)
        if call == "modeling":
            return 0, vti.synthetic2d(c, *P["c"], *geo, *a, data=np.full_like(data, -7))
        if call == "product":  # two passes a shot
            return 0, vti.gn_hessian2d(c, *P["c"], *dc, *geo, *a)
        return 0, vti.rtm2d(c, data, *P["c"], *geo, *a)

    if call == "modeling":
        # shots of one row a wavefront, 5 x 67 tiles: waves of fewer than four
        _probe(vti, ctx, rows=1)
        run(ctx)
        waves = _probe(vti, ctx)[0]
        assert waves >= 2
    else:
        waves = {"batch": 4, "gradient": 1, "product": 8, "image": 8}[call]
    with _by_level(vti) as c:
        f0, g0 = run(c)
        assert _probe(vti, c)[0] == 0
    assert g0.any()
    _probe(vti, ctx, rows=1 if call == "modeling" else 0, raised=raised)
    f1, g1 = run(ctx)
    gone = _probe(vti, ctx)[1]
    assert f0 == f1 and np.array_equal(g0, g1)
    assert gone == (1 if raised <= waves else 0)


def test_contexts_run_resident_at_once(vti):
    """Four contexts in four threads, shots of different sizes: their
    launches share the chip, each call's result is the one it has alone."""
    sizes = [(90, 20), (200, 120), (330, 260), (400, 330)]
    probs = [problem2d(vti, nx=nx, nz=nz, npad=12, nt=121, ns=1, seed=k) for k, (nx, nz) in enumerate(sizes)]
    print("resident contexts at once", flush=True)

    def run(c, P):
        return vti.objfunc_gradient2d(c, np.zeros((31, P["nr"]), np.float32), *P["c"], P["w"], P["sloc"], P["rloc"],
                                      P["taper"], *args2d(P))

    with _by_level(vti) as c:
        alone = [run(c, P) for P in probs]
    bad = []

    def work(k):
        with vti.Context(0) as c:
            for n in range(12):
                f, g = run(c, probs[(k + n) % 4])
                f0, g0 = alone[(k + n) % 4]
                if f != f0 or not np.array_equal(g, g0) or not g.any():
                    bad.append((k, n))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
