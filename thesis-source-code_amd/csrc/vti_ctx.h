// Execution context: one device and the stream every launch of a call goes on.
#pragma once

#include <hip/hip_runtime.h>

struct vti_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    // arithmetic of the 3D bulk stencil for objects created on this context:
    // 1 = the reference's mixed FP64 arithmetic (default), 0 = FP32
    int arith = 1;
    // snapshot storage of 2D gradients on this context: 0 = FP32 (default),
    // 1 = FP16, 2 = BF16, 3 = S16 (16-bit integers, power-of-two scale per
    // 64 points), for the calls the batched driver can take
    int snap_fmt = 0;
    bool resident = true;  // whether 2D passes may run resident (vti2d_res.h), vti_ctx_set_resident
    // the resident passes' side of vti_ctx_resident_probe
    struct {
        int rows = 0;    // rows of a wavefront to take where the shots then fit, 0: the fastest
        int raise = 0;   // which pass from now on (1: the next) starts with its abort flag raised, 0: none;
                         // those with a flag of their own count, not an adjoint's, which is its forward pass's
        int passes = 0;  // launched
        int gave_up = 0; // runs found void
        int ran = 0;     // bit r: some pass took r rows
    } probe;
};

// For the tests of the resident 2D passes: sets what the next ones do
// (vti_ctx::probe) and returns in seen[0..2] the passes launched, the runs
// that gave up and the row counts taken since the last call.  A raised flag
// is what a pass finds whose wait has run out: every kernel ends as usual, and the
// host takes the results for void.
extern "C" int vti_ctx_resident_probe(vti_ctx *ctx, int rows, int raise, int *seen);
