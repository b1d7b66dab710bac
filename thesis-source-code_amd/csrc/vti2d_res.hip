// Resident runs of 2D shots: launch shape, tables, launches (vti2d_res.h).
#include "vti2d_res.h"

#include <algorithm>

#include "vti_ctx.h"
#include "vti_internal.h"

namespace vti {

namespace {

template <int NR>
int per_cu(bool adjoint, int snap_fmt)
{
    if (!adjoint) return snap_fmt == 3 ? res_per_cu(fwd2d_res_kernel<NR, 3>) : res_per_cu(fwd2d_res_kernel<NR, 0>);
    return snap_fmt == 3 ? res_per_cu(bwd2d_res_kernel<NR, 3>) : res_per_cu(bwd2d_res_kernel<NR, 0>);
}

__global__ void clear_kernel(u64 *__restrict__ p, long long n, int *__restrict__ flag, int value)
{
    if (flag && blockIdx.x == 0 && threadIdx.x == 0) *flag = value;
    for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < n; k += (long long)gridDim.x * blockDim.x)
        p[k] = 0;
}
}  // namespace

ResGate<ResGateHip> &res_gate(int dev)
{
    static auto *g = new ResGate<ResGateHip>[64];  // outlives static destructors
    return g[dev & 63];
}

void res_clear(const DBuf<u64> &h, int *flag, int value, hipStream_t st)
{
    const unsigned nb = (unsigned)std::max<size_t>(1, std::min<size_t>((h.n + 255) / 256, 4096));
    hipLaunchKernelGGL(clear_kernel, dim3(nb), dim3(256), 0, st, h.p, (long long)h.n, flag, value);
}

ResShape res_rows(const vti_ctx *ctx, const int *nnx, int ns, int nnz, bool adjoint, int snap_fmt)
{
    // us a level takes, from runs of 10 to 984 tiles: the exchange, a
    // wavefront's rows one after the other, and the tiles' traffic
    // (forward 1.50 at 1 row and 56 tiles, 2.81 at 4 and 666, 3.08 at 6 and
    // 450; adjoint 1.64 at 1 and 56, 2.59 at 4 and 407, 3.31 at 6 and 450)
    return res_best_rows(
        nnx, ns, nnz, ctx->probe.rows,
        [&](int nr) { return with_rows(nr, [&](auto n) { return per_cu<n.value>(adjoint, snap_fmt); }); },
        [&](int nr, double t) { return adjoint ? 1.3 + 0.28 * nr + 0.2 * t : 1.15 + 0.22 * nr + 0.38 * t; });
}

bool res_fits(const vti_ctx *ctx, const int *nnx, int ns, int nnz, bool grad, int snap_fmt)
{
    return bool(res_rows(ctx, nnx, ns, nnz, false, snap_fmt)) &&
           (!grad || bool(res_rows(ctx, nnx, ns, nnz, true, snap_fmt)));
}

bool res2d_fits(vti_ctx *ctx, int nnx, int nnz, bool grad)
{
    if (!ctx->resident) return false;
    if (hipSetDevice(ctx->device) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return res_fits(ctx, &nnx, 1, nnz, grad, 0);
}

int res_setup(ResTiles &t, const ResShape &shape, const std::vector<ShotB> &base, int nnz, const int *rxz, const int *r0,
              hipStream_t st, int nf, bool dipole)
{
    VTI_CHECK(shape, "the shots do not fit the chip");
    const int nr = shape.nr, th = kResNW * nr, ns = (int)base.size();
    t.shape = shape;
    t.sb = base;
    t.tile_shot.clear();
    for (int j = 0; j < ns; ++j) {
        ShotB &b = t.sb[j];
        b.ntx = (b.nnx - 8 + 63) / 64;
        b.tile0 = (int)t.tile_shot.size();
        t.tile_shot.insert(t.tile_shot.end(), (size_t)b.ntx * ((nnz - 8 + th - 1) / th), j);
    }
    t.ntiles = (int)t.tile_shot.size();
    struct Item {
        int tile, key;
        ResRec r;
    };
    std::vector<Item> items;
    for (int j = 0; j < ns; ++j)
        for (int k = 0; k < t.sb[j].nr; ++k)
            for (int pole = 0; pole < (dipole ? 2 : 1); ++pole) {
                const int x = rxz[2 * ((size_t)r0[j] + k)] - 4, z = rxz[2 * ((size_t)r0[j] + k) + 1] - 4 + pole;
                if (x < 0 || x >= t.sb[j].nnx - 8 || z < 0 || z >= nnz - 8) continue;
                const int row = z % th, col = x & 63;
                items.push_back({t.sb[j].tile0 + (x >> 6) + (z / th) * t.sb[j].ntx,
                                 ((row / nr) * 64 + col) * nr + row % nr, ResRec{row * 64 + col, pole ? ~k : k}});
            }
    std::stable_sort(items.begin(), items.end(),
                     [](const Item &a, const Item &b) { return a.tile != b.tile ? a.tile < b.tile : a.key < b.key; });
    t.rec_at.assign(t.ntiles + 1, 0);
    t.rec.clear();
    for (const Item &i : items) {
        ++t.rec_at[i.tile + 1];
        t.rec.push_back(i.r);
    }
    for (int k = 0; k < t.ntiles; ++k) t.rec_at[k + 1] += t.rec_at[k];
    int rc = res_upload(t.sbd, t.sb, st);
    if (!rc) rc = res_upload(t.tsd, t.tile_shot, st);
    if (!rc) rc = res_upload(t.rad, t.rec_at, st);
    if (!rc) rc = res_upload(t.recd, t.rec, st);
    if (!rc) rc = t.halo.alloc((size_t)t.ntiles * 2 * nf * (8 * th + 512), st, false);
    return rc;
}

ResArgs res_args(const ResTiles &t, int *abort, const BatchGeo &bg, float dx2, float dz2, float dt2, const float *c11,
                 const float *c13, const float *c33, const float *t0, float *tr)
{
    ResArgs a{};
    a.shots = t.sbd.p;
    a.tile_shot = t.tsd.p;
    a.rec_at = t.rad.p;
    a.rec = t.recd.p;
    a.bg = bg;
    a.dx2 = dx2;
    a.dz2 = dz2;
    a.dt2 = dt2;
    a.halo = t.halo.p;
    a.abort = abort;
    a.c11 = c11;
    a.c13 = c13;
    a.c33 = c33;
    a.t0 = t0;
    a.tr = tr;
    return a;
}

int ResRun::setup(vti_ctx *c, const std::vector<ShotB> &base, int nnz, int snap_fmt, const int *rxz, const int *r0,
                  hipStream_t st)
{
    ctx = c;
    std::vector<int> nnx;
    for (const ShotB &b : base) nnx.push_back(b.nnx);
    const int ns = (int)base.size();
    int rc = res_setup(f, res_rows(ctx, nnx.data(), ns, nnz, false, snap_fmt), base, nnz, rxz, r0, st);
    if (!rc && !lb.empty())
        rc = res_setup(b, res_rows(ctx, nnx.data(), ns, nnz, true, snap_fmt), base, nnz, rxz, r0, st);
    if (!rc) rc = res_upload(lfd, lf, st);
    if (!rc) rc = res_upload(lbd, lb, st);
    if (!rc) rc = abortd.alloc(1, st, false);
    return rc;
}

int ResRun::forward(const BatchGeo &bg, float dx2, float dz2, float dt2, const DBuf<float> *c, const float *t0,
                    float *tr, int nt, bool taper_first, const SnapW &sw, int last_snap, hipStream_t st)
{
    VTI_CHECK(active() && (int)lf.size() >= nt, "resident forward: not set up");
    const ResArgs a = res_args(f, abortd.p, bg, dx2, dz2, dt2, c[0].p, c[1].p, c[2].p, t0, tr);
    const dim3 grid((unsigned)f.ntiles), block(64, kResNW);
    const int tf = taper_first ? 1 : 0;
    return res_launch(ctx, f, abortd.p, st, [&] {
        with_rows(f.shape.nr, [&](auto n) {
            if (sw.s16) fwd2d_res_kernel<n.value, 3><<<grid, block, 0, st>>>(a, lfd.p, nt, tf, sw, last_snap);
            else fwd2d_res_kernel<n.value, 0><<<grid, block, 0, st>>>(a, lfd.p, nt, tf, sw, last_snap);
        });
    });
}

int ResRun::adjoint(const BatchGeo &bg, float dx2, float dz2, float dt2, const DBuf<float> *c, const float *t0,
                    float *tr, const SnapR &sr, int snap_fmt, int last_row, float *g11, float *g13, float *g33,
                    hipStream_t st)
{
    VTI_CHECK(active() && b.shape && (snap_fmt == 0 || snap_fmt == 3), "resident adjoint: not set up");
    const ResArgs a = res_args(b, abortd.p, bg, dx2, dz2, dt2, c[0].p, c[1].p, c[2].p, t0, tr);
    const dim3 grid((unsigned)b.ntiles), block(64, kResNW);
    const int nlev = (int)lb.size();
    return res_launch(ctx, b, nullptr, st, [&] {
        with_rows(b.shape.nr, [&](auto n) {
            if (snap_fmt == 3)
                bwd2d_res_kernel<n.value, 3><<<grid, block, 0, st>>>(a, lbd.p, nlev, sr, last_row, g11, g13, g33);
            else
                bwd2d_res_kernel<n.value, 0><<<grid, block, 0, st>>>(a, lbd.p, nlev, sr, last_row, g11, g13, g33);
        });
    });
}

int res_gave_up(vti_ctx *ctx, const DBuf<int> &abort, bool *yes, hipStream_t st)
{
    int h = 0;
    VTI_HIP(hipMemcpyAsync(&h, abort.p, sizeof h, hipMemcpyDeviceToHost, st));
    VTI_HIP(hipStreamSynchronize(st));
    *yes = h != 0;
    ctx->probe.gave_up += *yes;
    return kOk;
}

int ResRun::aborted(bool *yes, hipStream_t st) const
{
    *yes = false;
    return active() ? res_gave_up(ctx, abortd, yes, st) : kOk;
}

}  // namespace vti
