// One shot of GNhessian_f and of rtm_f / odcig_f run resident (vti2d_res.h).
#include "vti2d_res.h"
#include "vti_ctx.h"
#include "vti_host.h"
#include "vti_internal.h"

namespace vti {

namespace {

template <class Kernels>
ResShape rows_for(const Res2dShot &s, Kernels &&per_cu, double per_row, double per_tile)
{
    return res_best_rows(&s.nnx, 1, s.nnz, s.ctx->probe.rows, per_cu,
                         [&](int nr, double t) { return 1.3 + per_row * nr + per_tile * t; });
}

ResShape rows_born(const Res2dShot &s)
{
    return rows_for(
        s, [](int nr) { return with_rows(nr, [](auto n) { return res_per_cu(born2d_res_kernel<n.value>); }); }, 0.4,
        0.6);
}
ResShape rows_back(const Res2dShot &s, bool image)
{
    return rows_for(
        s,
        [&](int nr) {
            return with_rows(nr, [&](auto n) {
                return image ? res_per_cu(back2d_res_kernel<n.value, 1>) : res_per_cu(back2d_res_kernel<n.value, 0>);
            });
        },
        0.25, 0.3);
}
ResShape rows_slices(const Res2dShot &s)
{
    return rows_for(
        s,
        [](int nr) { return with_rows(nr, [](auto n) { return res_per_cu(fwd2d_res_kernel<n.value, kResSlice>); }); },
        0.22, 0.38);
}

// what a pass needs on the device besides the caller's arrays
struct Pass {
    ResTiles t;
    DBuf<float> t0;
    DBuf<int> abort;
    DBuf<LevF> lf;
    DBuf<LevelB> lb;
    std::vector<float> h0;
    ResArgs a;
    int init(const Res2dShot &s, const ResShape &shape, const std::vector<LevF> &f, const std::vector<LevelB> &b, int nf,
             bool dipole)
    {
        hipStream_t st = s.ctx->stream;
        ShotB sb{};
        sb.nnx = s.nnx;
        sb.nr = s.nr;
        sb.src = (int)s.src;
        const int r0 = 0;
        h0.resize(s.npad + 1);
        taper_profile2d(h0.data(), s.npad);
        h0[s.npad] = 1.f;
        int rc = res_setup(t, shape, {sb}, s.nnz, s.rxz, &r0, st, nf, dipole);
        if (!rc) rc = res_upload(t0, h0, st);
        if (!rc) rc = res_upload(lf, f, st);
        if (!rc) rc = res_upload(lb, b, st);
        if (!rc) rc = abort.alloc(1, st, false);
        if (rc) return rc;
        BatchGeo bg;
        bg.nnz = s.nnz;
        bg.npad = s.npad;
        bg.cpitch = s.nnx;
        bg.rx2 = div_reciprocal(s.dx2);
        bg.rz2 = div_reciprocal(s.dz2);
        bg.nnxz_total = (long long)s.nnx * s.nnz;
        a = res_args(t, abort.p, bg, s.dx2, s.dz2, s.dt2, s.c[0], s.c[1], s.c[2], t0.p, s.tr);
        return kOk;
    }
};

LevelB bracket(double data_t, float image_t)
{
    LevelB l;
    float fr = (float)data_t;
    l.row = (int)fr;
    l.fr = fr - l.row;
    float f = image_t;
    l.slot = (int)f;
    l.f = f - l.slot;
    return l;
}

}  // namespace

bool res2d_fits_gn(const Res2dShot &s) { return rows_born(s) && rows_back(s, false); }
bool res2d_fits_slices(const Res2dShot &s) { return bool(rows_slices(s)); }
bool res2d_fits_image(const Res2dShot &s) { return bool(rows_back(s, true)); }

int res2d_gn(const Res2dShot &s, const float *const *dc, const float *wavelet, float *snap, float *g11, float *g13,
             float *g33, bool *gone)
{
    hipStream_t st = s.ctx->stream;
    const int nnt = (s.nt - 1) / s.ratio + 1;
    std::vector<LevF> lf(s.nt, LevF{0.f, -1, -1, 0});
    for (int it = 1; it < s.nt; ++it)
        lf[it] = LevF{s.dt2 * wavelet[it - 1], it > 1 && (it - 1) % s.ratio == 0 ? (it - 1) / s.ratio : -1,
                      it > 1 && it % s.ratio == 0 ? it / s.ratio : -1, 0};
    Pass f;
    int rc = f.init(s, rows_born(s), lf, {}, 2, false);
    if (rc) return rc;
    const SnapW sw{snap, nullptr, false};
    const dim3 block(64, kResNW);
    rc = res_launch(s.ctx, f.t, f.abort.p, st, [&] {
        with_rows(f.t.shape.nr, [&](auto n) {
            born2d_res_kernel<n.value><<<dim3((unsigned)f.t.ntiles), block, 0, st>>>(f.a, dc[0], dc[1], dc[2], f.lf.p,
                                                                                    s.nt, sw, nnt - 1);
        });
    });
    if (rc) return rc;
    std::vector<LevelB> lb;
    lb.push_back(bracket(0., (float)((s.nt - 2.) / s.ratio)));
    for (int it = s.nt - 3; it >= 0; --it) lb.push_back(bracket((it + 1.) / s.ratio, (float)it / s.ratio));
    Pass b;
    rc = b.init(s, rows_back(s, false), {}, lb, 1, false);
    if (rc) return rc;
    rc = res_launch(s.ctx, b.t, b.abort.p, st, [&] {
        with_rows(b.t.shape.nr, [&](auto n) {
            back2d_res_kernel<n.value, 0><<<dim3((unsigned)b.t.ntiles), block, 0, st>>>(
                b.a, b.lb.p, (int)lb.size(), snap, nnt - 1, g11, g13, g33);
        });
    });
    bool g1 = false, g2 = false;
    if (!rc) rc = res_gave_up(s.ctx, f.abort, &g1, st);
    if (!rc) rc = res_gave_up(s.ctx, b.abort, &g2, st);
    *gone = g1 || g2;
    return rc;
}

int res2d_slices(const Res2dShot &s, const float *wavelet, bool scaled, float *slices, bool *gone)
{
    hipStream_t st = s.ctx->stream;
    std::vector<LevF> lf(s.nt, LevF{0.f, -1, -1, 0});
    for (int it = 1; it < s.nt; ++it)
        lf[it] = LevF{it == 1 || scaled ? s.dt2 * wavelet[it - 1] : wavelet[it - 1], -1,
                      it % s.ratio == 0 ? it / s.ratio : -1, 0};
    Pass f;
    int rc = f.init(s, rows_slices(s), lf, {}, 1, false);
    if (rc) return rc;
    const SnapW sw{slices, nullptr, false};
    rc = res_launch(s.ctx, f.t, f.abort.p, st, [&] {
        with_rows(f.t.shape.nr, [&](auto n) {
            fwd2d_res_kernel<n.value, kResSlice><<<dim3((unsigned)f.t.ntiles), dim3(64, kResNW), 0, st>>>(
                f.a, f.lf.p, s.nt, 1, sw, -1);
        });
    });
    return rc ? rc : res_gave_up(s.ctx, f.abort, gone, st);
}

int res2d_image(const Res2dShot &s, int nt_neg, int last_row, const float *slices, float *image, bool *gone)
{
    hipStream_t st = s.ctx->stream;
    std::vector<LevelB> lb;
    lb.push_back(bracket(0., (float)((s.nt - 2.) / s.ratio)));
    for (int it = s.nt - 3; it >= 0; --it) {
        LevelB l = bracket((it - nt_neg + 1.) / s.ratio, (float)it / s.ratio);
        if (it < nt_neg || !s.nr) l.row = -1;
        lb.push_back(l);
    }
    Pass b;
    int rc = b.init(s, rows_back(s, true), {}, lb, 1, true);
    if (rc) return rc;
    rc = res_launch(s.ctx, b.t, b.abort.p, st, [&] {
        with_rows(b.t.shape.nr, [&](auto n) {
            back2d_res_kernel<n.value, 1><<<dim3((unsigned)b.t.ntiles), dim3(64, kResNW), 0, st>>>(
                b.a, b.lb.p, (int)lb.size(), slices, last_row, image, nullptr, nullptr);
        });
    });
    return rc ? rc : res_gave_up(s.ctx, b.abort, gone, st);
}

}  // namespace vti
