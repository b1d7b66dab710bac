// Resident runs of 2D shots (vti2d_res_kernels.h): the launch shape, the
// tables and the launches.
#pragma once

#include <vector>

#include "vti2d_res_kernels.h"
#include "vti_dbuf.h"

namespace vti {

// A pass of a resident run: the tiles of its launch.
struct ResTiles {
    int nr = 0, ntiles = 0;  // rows per wavefront (0: the shots do not fit the chip), tiles
    std::vector<ShotB> sb;
    std::vector<int> tile_shot, rec_at;
    std::vector<ResRec> rec;
    DBuf<ShotB> sbd;
    DBuf<int> tsd, rad;
    DBuf<ResRec> recd;
    DBuf<u64> halo;
};

// The rows per wavefront with which shots of these padded widths (nnz rows
// each) are all on the current device at once in a pass (adjoint or forward;
// snap_fmt 0 or 3), the fastest of them; 0 when there is none.
int res_rows(const int *nnx, int ns, int nnz, bool adjoint, int snap_fmt);
// whether the shots fit in the forward pass and, with grad, in the adjoint
bool res_fits(const int *nnx, int ns, int nnz, bool grad, int snap_fmt);

// One set of shots run resident.
struct ResRun {
    ResTiles f, b;
    std::vector<LevF> lf;    // set by the caller before setup
    std::vector<LevelB> lb;  // the same; empty without an adjoint pass
    DBuf<int> abortd;
    DBuf<LevF> lfd;
    DBuf<LevelB> lbd;

    bool active() const { return f.nr > 0; }
    // Tables for the shots base (all fields but tile0/ntx as the caller keeps
    // them) and the receivers of each: rxz[2 r0[j] ..] holds shot j's (ix, iz).
    // Points outside the interior, where the fields stay 0, are left out.
    // The host tables stay in place until the stream has read them.
    int setup(const std::vector<ShotB> &base, int nnz, int snap_fmt, const int *rxz, const int *r0, hipStream_t st);
    int forward(const BatchGeo &bg, float dx2, float dz2, float dt2, const DBuf<float> *c, const float *t0, float *tr,
                int nt, bool taper_first, const SnapW &sw, int last_snap, hipStream_t st);
    int adjoint(const BatchGeo &bg, float dx2, float dz2, float dt2, const DBuf<float> *c, const float *t0, float *tr,
                const SnapR &sr, int snap_fmt, int last_row, float *g11, float *g13, float *g33, hipStream_t st);
    // after the stream is idle: whether a wait ran out, so that the results
    // are void and the call has to be run on the per-level kernels
    int aborted(bool *yes, hipStream_t st) const;
};

}  // namespace vti
