// Resident runs of 2D shots (vti2d_res_kernels.h): the launch shape, the
// tables and the launches.
#pragma once

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "vti2d_res_kernels.h"
#include "vti_ctx.h"
#include "vti_dbuf.h"
#include "vti_res_gate.h"

namespace vti {

// The launch shape of a pass: rows per wavefront (0: the shots do not fit the
// chip), the workgroups that a CU holds for certain, the device's CUs.
struct ResShape {
    int nr = 0, per_cu = 0, cus = 0;
    explicit operator bool() const { return nr > 0; }
};

// A pass of a resident run: the tiles of its launch.
struct ResTiles {
    ResShape shape;
    int ntiles = 0;
    std::vector<ShotB> sb;
    std::vector<int> tile_shot, rec_at;
    std::vector<ResRec> rec;
    DBuf<ShotB> sbd;
    DBuf<int> tsd, rad;
    DBuf<ResRec> recd;
    DBuf<u64> halo;
};

// Workgroups of a kernel that a CU holds for certain.  Other kernels may
// come and go while a launch's workgroups are placed, so registers and LDS can
// be left in pieces; with k-1 workgroups anywhere in a CU, the largest of the
// k gaps holds another one if each takes at most 1/(2k-1) of it.  (Filling the
// CUs to the last register has left workgroups outside, and the others
// waiting for them.)  A workgroup has one wavefront on each SIMD.
template <class F>
int res_per_cu(F *kernel)
{
    hipFuncAttributes fa;
    if (hipFuncGetAttributes(&fa, reinterpret_cast<const void *>(kernel)) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    if (fa.localSizeBytes) return 0;  // scratch would be another thing to wait for
    const int regs = std::max(1, (fa.numRegs + 7) / 8 * 8), lds = std::max<int>(1, (int)fa.sharedSizeBytes);
    int k = 0;
    while (regs * (2 * k + 1) <= 512 && lds * (2 * k + 1) <= 160 * 1024 && k < 8) ++k;
    return k;
}

// f(integral constant NR) for one of the built row counts
template <class F>
auto with_rows(int nr, F &&f)
{
    switch (nr) {
    case 1: return f(std::integral_constant<int, 1>());
    case 2: return f(std::integral_constant<int, 2>());
    case 3: return f(std::integral_constant<int, 3>());
    case 4: return f(std::integral_constant<int, 4>());
    default: return f(std::integral_constant<int, 6>());
    }
}

// The shape of the least cost(rows, tiles per CU) among those whose tiles
// of these shots are all on the current device at once, cap(rows) on a CU;
// no rows when there is none.  only: the one row count to look at, 0 for all.
template <class Cap, class Cost>
ResShape res_best_rows(const int *nnx, int ns, int nnz, int only, Cap &&cap, Cost &&cost)
{
    int dev = 0, cus = 0;
    ResShape best;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
        (void)hipGetLastError();
        return best;
    }
    double least = 0;
    for (int nr : {1, 2, 3, 4, 6}) {
        if (only && nr != only) continue;
        const int th = kResNW * nr;
        long long tiles = 0;
        for (int s = 0; s < ns; ++s) tiles += (long long)((nnx[s] - 8 + 63) / 64) * ((nnz - 8 + th - 1) / th);
        const int k = cap(nr);
        if (tiles > (long long)cus * k) continue;
        const double c = cost(nr, (double)tiles / cus);
        if (best && c >= least) continue;
        best = ResShape{nr, k, cus};
        least = c;
    }
    return best;
}

struct ResGateHip {
    using Stream = hipStream_t;
    using Event = hipEvent_t;
    static bool make(Event *e) { return hipEventCreateWithFlags(e, hipEventDisableTiming) == hipSuccess; }
    static bool record(Event e, Stream s) { return hipEventRecord(e, s) == hipSuccess; }
    static bool wait(Stream s, Event e) { return hipStreamWaitEvent(s, e, 0) == hipSuccess; }
    static bool done(Event e) { return hipEventQuery(e) != hipErrorNotReady; }
};
ResGate<ResGateHip> &res_gate(int dev);
void res_clear(const DBuf<u64> &halo, int *flag, int value, hipStream_t st);
// Clears the strips of t and the abort flag, then launch(), behind those
// resident launches of the device that it may not run beside.  flag: null for a pass that goes on from
// another's results and is void with it.  (It is cleared by every run, not once
// where it is allocated: a plan's runs share it.)
template <class Launch>
int res_launch(vti_ctx *ctx, const ResTiles &t, int *flag, hipStream_t st, Launch &&launch)
{
    int dev = 0;
    VTI_HIP(hipGetLastError());
    VTI_HIP(hipGetDevice(&dev));
    auto &g = res_gate(dev);
    std::lock_guard<std::mutex> lk(g.mu);
    VTI_CHECK(g.enter(t.ntiles, t.shape.per_cu, t.shape.cus, st), "resident launch: waiting for others failed");
    auto &probe = ctx->probe;
    res_clear(t.halo, flag, flag && probe.raise && --probe.raise == 0, st);
    ++probe.passes;
    probe.ran |= 1 << t.shape.nr;
    (void)hipGetLastError();  // (an event not ready yet)
    launch();
    VTI_HIP(hipGetLastError());
    VTI_CHECK(g.leave(), "resident launch: event record failed");
    return kOk;
}

// The shape in which shots of these padded widths (nnz rows each) are all on
// the current device at once in a pass (adjoint or forward; snap_fmt 0 or 3),
// the fastest; no rows when there is none.
ResShape res_rows(const vti_ctx *ctx, const int *nnx, int ns, int nnz, bool adjoint, int snap_fmt);
// whether the shots fit in the forward pass and, with grad, in the adjoint
bool res_fits(const vti_ctx *ctx, const int *nnx, int ns, int nnz, bool grad, int snap_fmt);

// Tables of the shots base (all fields but tile0/ntx as the caller keeps
// them) in tiles of that shape, and the receivers of each: rxz[2 r0[j]
// ..] holds shot j's (ix, iz).  Points outside the interior, where the fields
// stay 0, are left out.  nf: field pairs exchanged; dipole: the point below
// each receiver is its negative pole.  The host tables stay in place until the
// stream has read them.
int res_setup(ResTiles &t, const ResShape &shape, const std::vector<ShotB> &base, int nnz, const int *rxz, const int *r0,
              hipStream_t st, int nf = 1, bool dipole = false);
ResArgs res_args(const ResTiles &t, int *abort, const BatchGeo &bg, float dx2, float dz2, float dt2, const float *c11,
                 const float *c13, const float *c33, const float *t0, float *tr);
// after the stream is idle: whether a wait ran out
int res_gave_up(vti_ctx *ctx, const DBuf<int> &abort, bool *yes, hipStream_t st);

template <class T>
int res_upload(DBuf<T> &d, const std::vector<T> &h, hipStream_t st)
{
    const int rc = d.alloc(h.size(), st, false);
    if (rc) return rc;
    if (!h.empty()) VTI_HIP(hipMemcpyAsync(d.p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, st));
    return kOk;
}

// One set of shots run resident.
struct ResRun {
    vti_ctx *ctx = nullptr;
    ResTiles f, b;
    std::vector<LevF> lf;    // set by the caller before setup
    std::vector<LevelB> lb;  // the same; empty without an adjoint pass
    DBuf<int> abortd;
    DBuf<LevF> lfd;
    DBuf<LevelB> lbd;

    bool active() const { return f.shape.nr > 0; }
    // the tables of both passes (res_setup)
    int setup(vti_ctx *c, const std::vector<ShotB> &base, int nnz, int snap_fmt, const int *rxz, const int *r0,
              hipStream_t st);
    int forward(const BatchGeo &bg, float dx2, float dz2, float dt2, const DBuf<float> *c, const float *t0, float *tr,
                int nt, bool taper_first, const SnapW &sw, int last_snap, hipStream_t st);
    int adjoint(const BatchGeo &bg, float dx2, float dz2, float dt2, const DBuf<float> *c, const float *t0, float *tr,
                const SnapR &sr, int snap_fmt, int last_row, float *g11, float *g13, float *g33, hipStream_t st);
    // after the stream is idle: whether a wait ran out, so that the results
    // are void and the call has to be run on the per-level kernels
    int aborted(bool *yes, hipStream_t st) const;
};

}  // namespace vti
