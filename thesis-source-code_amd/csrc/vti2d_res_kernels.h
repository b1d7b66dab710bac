// Resident 2D kernels: one launch runs every time level of a set of shots.
//
// A 2D shot's state is small next to the chip: four wavefield values, three
// coefficients and the taper per point, 2-20 MB for the grids of a survey,
// against 128 MB of vector registers.  So each workgroup keeps its tile of the
// grid in registers for the whole run, and per level only the tile edges
// travel: p (or, in the adjoint, c11 p + c13 q) of 4 columns to the tiles at
// either side, q (c13 p + c33 q) of 4 rows to the tiles above and below.  The
// launches per level, and every read and write of the wavefields, the
// coefficients and the gradient, drop out; what remains per level is the
// arithmetic and one exchange with four neighbours, about 1.1 us.
//
// Tile: 64 columns (a wavefront's lanes) by 4 NR rows, NR rows to each of 4
// wavefronts.  The x stencil reads p from LDS (4 halo columns at either
// side), the z stencil q.  The LDS planes are double-buffered by level, so a
// level needs one workgroup barrier.  Two workgroups share a CU, so one
// computes while the other waits for its neighbours.
//
// Exchange: an edge value goes out as one 8-byte word {value, level}, with an
// agent-scope store, and the neighbour polls the words it needs until they
// carry the level it waits for.  Value and level arrive together, so no
// fence, flag or ordering between different words is needed, and words of
// level L-1 and L sit in different slots: a tile sends level L+1 only after
// it has read all of its neighbours' level L, so a neighbour that is one
// level ahead cannot overwrite a word that is still to be read.
//
// All workgroups of a launch must be on the chip at once, since they wait for
// one another: the host launches no more than fit (res_per_cu), also of
// several launches at a time (vti_res_gate.h).  Every wait is bounded: after
// kResWait without its word (something else holds the CUs) a wavefront raises
// the abort flag and waits no more, the others see the flag and do the same,
// and the host, which finds it raised, runs the call on the per-level kernels
// instead.
//
// Per point the arithmetic is that of vti2d_kernels.h, operation for
// operation, so the results are the per-level kernels' bit for bit.
//
// What bounds a level: at a few tiles the exchange (1.1 of 1.5 us); at several
// hundred the instructions of the rows.  One shot of 592 x 1104 points takes 2.9 us
// a forward level (666 tiles of 4 rows) and 3.4 us an adjoint level (450 of 6), where
// the two-level launches take 7.6 us for the pair's mean and the one-level launches
// 10.4.  In a probe of these loops at that size the levels took 3.15 and 3.7 us, and
// 1.9 and 2.55 with the exchange left out.  Scalar registers are short: the
// row and lane masks and the strips' addresses of three bodies keep 78 of them in
// vector lanes in the 4-row forward kernel and 119 in the 6-row adjoint.
#pragma once

#include "vti2d_batch_kernels.h"

#pragma clang fp contract(off)

namespace vti {

typedef unsigned long long u64;

// the longest wait for a neighbour's word, in ticks of the 100 MHz wall clock
constexpr long long kResWait = 5000000LL;
constexpr int kResNW = 4;  // wavefronts of a workgroup, one per SIMD

// LDS planes and strips of tiles of 4 NR rows.  Words of a tile's strips at
// one level parity: its left and its right 4 columns, its top and its bottom 4
// rows.
template <int NR>
struct ResDim {
    static constexpr int TH = kResNW * NR, PW = 72, QW = 64;
    static constexpr int P = TH * PW, Q = (TH + 8) * QW;  // floats of a plane
    static constexpr int L = 0, R = 4 * TH, T = 8 * TH, B = 8 * TH + 256, WORDS = 8 * TH + 512;
};

// What one forward level does besides the step.
struct LevF {
    float src;  // added at the source
    int snap;   // snapshot slot of the level read, or -1
    int row;    // trace row the new level is recorded in, or -1
    int pad;
};

// A receiver within its tile: point (row * 64 + column) and trace column; ~ir
// at the negative pole of a dipole receiver (the point below it).
struct ResRec {
    int pt, ir;
};

struct ResArgs {
    const ShotB *shots;    // tile0/ntx for this launch's tiles
    const int *tile_shot;  // tile -> shot
    const int *rec_at;     // tile -> first of its receivers in rec (one more than tiles)
    const ResRec *rec;     // by tile, then wavefront, lane, row
    BatchGeo bg;
    float dx2, dz2, dt2;
    u64 *halo;  // strips: tile x parity x ResDim::WORDS
    int *abort;
    const float *c11, *c13, *c33;  // row pitch bg.cpitch
    const float *t0;               // taper profile, t0[npad] = 1
    float *tr;                     // traces, ShotB.r_off
};

// word `word` of the strips, by a 32-bit offset from their uniform base
__device__ __forceinline__ u64 *res_word(u64 *halo, unsigned word)
{
    return reinterpret_cast<u64 *>(reinterpret_cast<char *>(halo) + word * 8u);
}
__device__ __forceinline__ void res_put(u64 *p, float v, unsigned tag)
{
    __hip_atomic_store(p, ((u64)tag << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 res_get(const u64 *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A wavefront's place in its tile and the tile's in the exchange.  Word
// numbers are for parity 0, from the base of all strips (32 bits: a launch
// holds a few hundred tiles).
template <int NR>
struct ResTile {
    using D = ResDim<NR>;
    int lane, w, row0;
    int nk;            // rows of the wavefront inside the interior
    bool send_c;       // this lane sends a word of the wavefront's rows of an edge column
    unsigned wc;
    int lc;            // LDS place of the value
    int kt, kb;        // rows [0, kt) are top edge rows, rows [kb, NR) bottom ones
    unsigned wt, wb;   // words of top row row0 and of bottom row row0, at this lane
    bool get_x;        // this lane fetches a word of the halo columns beside the wavefront's rows
    bool get_u, get_d; // the wavefront fetches halo row w above, w below
    unsigned wx, wu, wd;
    int lx;            // LDS place of the halo column value

    // nf: field pairs exchanged, each with strips of its own
    __device__ __forceinline__ void init(const ResArgs &a, const ShotB &sh, int tile, int z0, int nf = 1)
    {
        const int tl = tile - sh.tile0, tx = tl % sh.ntx;
        lane = threadIdx.x;
        w = __builtin_amdgcn_readfirstlane(threadIdx.y);
        row0 = w * NR;
        const int rows = a.bg.nnz - 4 - z0;  // interior rows from the tile's first
        const int nact = min(D::TH, rows), below = rows - D::TH;
        nk = max(0, min(NR, nact - row0));
        const bool lf = tx > 0, rt = tx + 1 < sh.ntx, up = tl >= sh.ntx, dn = below > 0;
        const unsigned tw = 2u * D::WORDS * nf, own = tw * tile;
        // lanes in the order of the strips' words: 4 NR of the left columns, 4 NR of the right ones
        const bool right = lane >= 4 * NR;
        const int r = row0 + ((right ? lane - 4 * NR : lane) >> 2), c = lane & 3;
        send_c = lane < 8 * NR && r < nact && (right ? rt : lf);
        wc = own + (right ? D::R : D::L) + 4 * r + c;
        lc = r * D::PW + (right ? 64 : 4) + c;
        kt = up ? min(nk, max(0, 4 - row0)) : 0;
        kb = dn ? max(0, D::TH - 4 - row0) : NR;
        wt = own + D::T + row0 * 64 + lane;
        wb = own + D::B + (row0 - (D::TH - 4)) * 64 + lane;
        get_x = send_c;
        wx = (right ? tw * (tile + 1) + D::L : tw * (tile - 1) + D::R) + 4 * r + c;
        lx = r * D::PW + (right ? 68 : 0) + c;
        get_u = up;
        wu = tw * (tile - sh.ntx) + D::B + w * 64 + lane;
        get_d = w < min(4, below);
        wd = tw * (tile + sh.ntx) + D::T + w * 64 + lane;
    }
};

// The wavefront's rows of a level into the tile's LDS planes and, where they
// are edge values, to the neighbours.  a: x-stencil quantity, b: z-stencil's.
template <int NR>
__device__ __forceinline__ void res_send(const ResTile<NR> &t, u64 *halo, float *pl, float *ql, const float (&a)[NR],
                                         const float (&b)[NR], unsigned tag)
{
    using D = ResDim<NR>;
    const unsigned par = (tag & 1) * D::WORDS;
#pragma unroll
    for (int k = 0; k < NR; ++k) pl[(t.row0 + k) * D::PW + t.lane + 4] = a[k];
    // (the wavefront reads back what it has just written: LDS keeps its order)
    __builtin_amdgcn_wave_barrier();
    if (t.send_c) res_put(res_word(halo, t.wc + par), pl[t.lc], tag);
    if (t.kt > 0) {
        u64 *wt = res_word(halo, t.wt + par);
#pragma unroll
        for (int k = 0; k < (NR < 4 ? NR : 4); ++k)
            if (k < t.kt) res_put(wt + 64 * k, b[k], tag);
    }
    if (t.kb < NR) {
        u64 *wb = res_word(halo, t.wb + par);
#pragma unroll
        for (int k = NR < 4 ? 0 : NR - 4; k < NR; ++k)
            if (k >= t.kb) res_put(wb + 64 * k, b[k], tag);
    }
#pragma unroll
    for (int k = 0; k < NR; ++k) ql[(t.row0 + k + 4) * D::QW + t.lane] = b[k];
}

// The neighbours' edge values of level `tag` into the halos of the LDS
// planes: each wavefront waits for the halo columns beside its own rows and
// for one halo row above the tile and one below.
template <int NR>
__device__ __forceinline__ void res_recv(const ResTile<NR> &t, u64 *halo, int *abort, bool &gone, float *pl,
                                         float *ql, unsigned tag)
{
    using D = ResDim<NR>;
    const unsigned par = (tag & 1) * D::WORDS;
    const u64 *wx = res_word(halo, t.wx + par), *wu = res_word(halo, t.wu + par), *wd = res_word(halo, t.wd + par);
    u64 vx = (u64)tag << 32, vu = vx, vd = vx;
    int spin = 0;
    long long t0 = 0;
    bool wait_x = t.get_x && !gone, wait_u = t.get_u && !gone, wait_d = t.get_d && !gone;
    while (wait_x || wait_u || wait_d) {
        if (wait_x) vx = res_get(wx);
        if (wait_u) vu = res_get(wu);
        if (wait_d) vd = res_get(wd);
        wait_x = (unsigned)(vx >> 32) != tag;
        wait_u = (unsigned)(vu >> 32) != tag;
        wait_d = (unsigned)(vd >> 32) != tag;
        __builtin_amdgcn_s_sleep(1);
        if ((++spin & 255) == 0) {
            const long long now = wall_clock64();
            if (spin == 256) t0 = now;
            if (now - t0 > kResWait || __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                __hip_atomic_store(abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                gone = true;
                break;
            }
        }
    }
    gone = __any(gone);
    if (t.get_x) pl[t.lx] = __uint_as_float((unsigned)vx);
    if (t.get_u) ql[t.w * D::QW + t.lane] = __uint_as_float((unsigned)vu);
    if (t.get_d) ql[(D::TH + 4 + t.w) * D::QW + t.lane] = __uint_as_float((unsigned)vd);
}

// x[k] / d for every k < nk, as qdiv (vti2d_kernels.h) gives it: with
// y = RN(1/d), Markstein's correction where every |x[k]| is 0 or lies in
// [2^-100, 2^100), which one minimum and one maximum over all k decide, else the
// division.  (2 bits - 1 orders the magnitudes as unsigned integers with 0 as
// the largest.  The remainder is formed as q0 d - x and taken off: a zero x
// then keeps its sign.)
template <int N>
__device__ __forceinline__ void res_div(float (&x)[N], float d, float y, int nk, bool on)
{
    float t[N], mx = 0.f;
    unsigned mn = 0xffffffffu;
#pragma unroll
    for (int k = 0; k < N; ++k)
        if (k < nk) {
            mn = min(mn, (__float_as_uint(x[k]) << 1) - 1u);
            mx = fmaxf(mx, fabsf(x[k]));
        }
    if (on && (y == 0.f || mn < (0x0d800000u << 1) - 1u || !(mx < 0x1p100f))) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            // (keeps the compiler from dividing in every lane and selecting)
            float xs = x[k];
            asm volatile("" : "+v"(xs));
            t[k] = xs / d;
        }
    } else {
        float q0[N], r[N];
#pragma unroll
        for (int k = 0; k < N; ++k) q0[k] = x[k] * y;
#pragma unroll
        for (int k = 0; k < N; ++k) r[k] = __builtin_fmaf(q0[k], d, -x[k]);
#pragma unroll
        for (int k = 0; k < N; ++k) t[k] = __builtin_fmaf(-r[k], y, q0[k]);
    }
#pragma unroll
    for (int k = 0; k < N; ++k) x[k] = t[k];
}

// Second differences of the wavefront's rows: tp along x of plane pl, tq
// along z of plane ql; pc, qc: the planes' own values.  Several rows are
// worked on at a time, each step for all of them, because a wavefront can
// start a dependent operation only 8 cycles after the one it waits for.
template <int NR>
__device__ __forceinline__ void res_d(const ResTile<NR> &t, const ResArgs &A, const float *pl, const float *ql, int nk,
                                      bool act, float (&tp)[NR], float (&tq)[NR], float (&pc)[NR], float (&qc)[NR])
{
    using D = ResDim<NR>;
    constexpr int G = NR % 3 == 0 ? 3 : NR % 2 == 0 ? 2 : 1;
    const float *r = pl + t.row0 * D::PW + t.lane;
#pragma unroll
    for (int k = 0; k < NR; k += G) {
        float v[9][G];
#pragma unroll
        for (int j = 0; j < 9; ++j)
#pragma unroll
            for (int g = 0; g < G; ++g) v[j][g] = r[(k + g) * D::PW + j];
        float acc[G], s[G];
        auto term = [&](float c, int a, int b) {
#pragma unroll
            for (int g = 0; g < G; ++g) s[g] = v[a][g] + v[b][g];
#pragma unroll
            for (int g = 0; g < G; ++g) s[g] = c * s[g];
#pragma unroll
            for (int g = 0; g < G; ++g) acc[g] = acc[g] + s[g];
        };
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g] = VTI_C0 * v[4][g];
        term(VTI_C1, 3, 5);
        term(VTI_C2, 2, 6);
        term(VTI_C3, 1, 7);
        term(VTI_C4, 0, 8);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            tp[k + g] = acc[g];
            pc[k + g] = v[4][g];
        }
    }
    res_div(tp, A.dx2, A.bg.rx2, nk, act);
    const float *c = ql + t.row0 * D::QW + t.lane;
    float e[NR + 8];
#pragma unroll
    for (int j = 0; j < NR + 8; ++j) e[j] = c[j * D::QW];
    {
        float s[NR];
        auto term = [&](float c, int o) {
#pragma unroll
            for (int k = 0; k < NR; ++k) s[k] = e[k + 4 - o] + e[k + 4 + o];
#pragma unroll
            for (int k = 0; k < NR; ++k) s[k] = c * s[k];
#pragma unroll
            for (int k = 0; k < NR; ++k) tq[k] = tq[k] + s[k];
        };
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            qc[k] = e[k + 4];
            tq[k] = VTI_C0 * e[k + 4];
        }
        term(VTI_C1, 1);
        term(VTI_C2, 2);
        term(VTI_C3, 3);
        term(VTI_C4, 4);
    }
    res_div(tq, A.dz2, A.bg.rz2, nk, act);
}

// How a wavefront's points lie: all inside the interior with the taper 1, all
// inside the interior, or any.
enum { kResInner, kResFull, kResAny };

// The taper of a wavefront's points: a factor per lane and one per row.
template <int NR>
struct ResTaper {
    float x, z[NR];
    // returns whether every factor is 1
    __device__ __forceinline__ bool init(const ResArgs &a, const ShotB &sh, const ResTile<NR> &t, int x0, int z0)
    {
        bool one = true;
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const TapF f = taper_ld(a.t0, a.bg.npad, sh.nnx, a.bg.nnz, min(x0 + t.lane, sh.nnx - 1),
                                    min(z0 + t.row0 + k, a.bg.nnz - 1));
            x = f.x;
            z[k] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(f.z)));
            one = one && f.x == 1.f && f.z == 1.f;
        }
        return __all(one);
    }
    template <int KIND>
    __device__ __forceinline__ float at(int k) const
    {
        return KIND == kResInner ? 1.f : x * z[k];
    }
};

// Forward pass: levels 2..nt-1 of every shot from its level 1, dt2*w[0] at
// the source (objFuncGradient_f.cu:160-210, synthetic_f.cu:86-110), with the
// source, the taper, the recorded traces and the D snapshots.
// lev[it]: what level it does; last_snap: the slot of D of the last level.
// SF: the snapshots' format (0 also for none); kResSlice: no D snapshots, but
// 0.5 (p + q) of the recorded levels into the planes of sw.d
// (recordWavefieldSlice, kernels.cu:335-343), one shot, from a dipole source.
enum { kResSlice = 4 };

template <int NR, int SF, int KIND>
__device__ __forceinline__ void fwd2d_res_body(const ResArgs &A, const ResTile<NR> &t, const ShotB &sh,
                                               const ResTaper<NR> &tap, int tile, int x, int z0, float *lds,
                                               const LevF *__restrict__ lev, int nt, bool taper_first,
                                               const SnapW &sw, int last_snap)
{
    using D = ResDim<NR>;
    const int nnx = sh.nnx, tid = t.lane + 64 * t.w;
    const int nk = KIND == kResAny ? t.nk : NR;
    const bool act = KIND == kResAny ? x < nnx - 4 : true;
    const unsigned i0 = x + (z0 + t.row0) * nnx;
    auto pl = [&](int it) { return lds + (it & 1) * D::P; };
    auto ql = [&](int it) { return lds + 2 * D::P + (it & 1) * D::Q; };
    // the two levels are those of the LDS planes; registers hold the coefficients
    float p[NR], q[NR], a11[NR], a13[NR], a33[NR];
    const float v1 = lev[1].src;
    unsigned smask = 0, nmask = 0;  // this lane's rows that hold the source, a dipole's second pole
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        p[k] = q[k] = a11[k] = a13[k] = a33[k] = 0.f;
        if (k < nk && act) {
            const long long c = sh.c_off + x + (long long)(z0 + t.row0 + k) * A.bg.cpitch;
            a11[k] = A.c11[c];
            a13[k] = A.c13[c];
            a33[k] = A.c33[c];
            if ((int)(i0 + k * nnx) == sh.src) {
                smask |= 1u << k;
                p[k] = taper_first ? v1 * tap.template at<KIND>(k) : v1;
                q[k] = p[k];
            }
            if (SF == kResSlice && (int)(i0 + k * nnx) == sh.src + nnx) {
                nmask |= 1u << k;
                p[k] = -v1 * tap.template at<KIND>(k);
                q[k] = p[k];
            }
        }
    }
    const bool has_src = __ballot((smask | nmask) != 0) != 0;
    const int rec0 = A.rec_at[tile], rec1 = A.rec_at[tile + 1];
    auto record = [&](int it, int row) {
        const float *pr = pl(it) + 4, *qr = ql(it) + 4 * D::QW;
        float *out = A.tr + sh.r_off + (long long)row * sh.nr;
        for (int e = rec0 + tid; e < rec1; e += 64 * kResNW) {
            const ResRec r = A.rec[e];
            out[r.ir] = 0.5f * (pr[(r.pt >> 6) * D::PW + (r.pt & 63)] + qr[r.pt]);
        }
    };
    auto put_snap = [&](int slot, const float (&tp)[NR], const float (&tq)[NR]) {
#pragma unroll
        for (int k = 0; k < NR; ++k)
            if (k < nk) {
                if (SF == 3)
                    snap_put_s16(sw, sh, A.bg.nnz, slot, x, z0 + t.row0 + k, act, tp[k], tq[k]);
                else if (act)
                    snap_put32(sw, sh, (long long)nnx * A.bg.nnz, slot, i0 + k * nnx, tp[k], tq[k]);
            }
    };
    bool gone = false;
    auto put_slice = [&](int slot) {
        float *out = sw.d + (long long)slot * nnx * A.bg.nnz;
#pragma unroll
        for (int k = 0; k < NR; ++k)
            if (k < nk && act) st32(out, i0 + k * nnx, 0.5f * (p[k] + q[k]));
    };
    res_send<NR>(t, A.halo, pl(1), ql(1), p, q, 1);
    LevF l = lev[min(2, nt - 1)];
    res_recv<NR>(t, A.halo, A.abort, gone, pl(1), ql(1), 1);
    lds_barrier();
    if (lev[1].row >= 0) {
        if (SF == kResSlice) put_slice(lev[1].row);
        else record(1, lev[1].row);
    }
    // Level it from the current (pc, qc) over the previous (p, q).  The next
    // level's entry is read ahead of the wait: a scalar load still in flight
    // holds up every LDS read after it.
    auto step = [&](int it) {
        const LevF cur = l;
        float tp[NR], tq[NR], pc[NR], qc[NR];
        __builtin_amdgcn_s_setprio(1);
        res_d<NR>(t, A, pl(it - 1), ql(it - 1), nk, act, tp, tq, pc, qc);
        const float *pv = pl(it) + t.row0 * D::PW + t.lane + 4, *qv = ql(it) + (t.row0 + 4) * D::QW + t.lane;
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const float tk = tap.template at<KIND>(k), pp = pv[k * D::PW], qp = qv[k * D::QW];
            float pn = 2.f * pc[k] + A.dt2 * (a11[k] * tp[k] + a13[k] * tq[k]) - (KIND == kResInner ? pp : pp * tk);
            float qn = 2.f * qc[k] + A.dt2 * (a13[k] * tp[k] + a33[k] * tq[k]) - (KIND == kResInner ? qp : qp * tk);
            if (has_src && (smask >> k & 1)) {
                pn += cur.src;
                qn += cur.src;
            }
            if (SF == kResSlice && has_src && (nmask >> k & 1)) {
                pn -= cur.src;
                qn -= cur.src;
            }
            const bool on = KIND != kResAny || (act && k < nk);
            p[k] = KIND == kResInner ? pn : on ? pn * tk : 0.f;
            q[k] = KIND == kResInner ? qn : on ? qn * tk : 0.f;
        }
        res_send<NR>(t, A.halo, pl(it), ql(it), p, q, it);
        __builtin_amdgcn_s_setprio(0);
        l = lev[min(it + 1, nt - 1)];
        if (SF == kResSlice) {
            if (cur.row >= 0) put_slice(cur.row);
        } else if (cur.snap >= 0) {
            put_snap(cur.snap, tp, tq);
        }
        res_recv<NR>(t, A.halo, A.abort, gone, pl(it), ql(it), it);
        lds_barrier();
        if (SF != kResSlice && cur.row >= 0 && rec0 < rec1) record(it, cur.row);
    };
    for (int it = 2; it < nt; ++it) step(it);
    if (last_snap >= 0) {
        float tp[NR], tq[NR], pc[NR], qc[NR];
        res_d<NR>(t, A, pl(nt - 1), ql(nt - 1), nk, act, tp, tq, pc, qc);
        put_snap(last_snap, tp, tq);
    }
}

// Registers: res_per_cu (vti2d_res.hip) counts on 2 workgroups a CU where none
// takes over a third of a SIMD's registers, on 3 where none takes over a fifth.
template <int NR, int SF>
static __global__ __launch_bounds__(64 * kResNW) __attribute__((amdgpu_waves_per_eu(NR == 4 && SF == 0 ? 5 : 3))) void fwd2d_res_kernel(
    ResArgs A, const LevF *__restrict__ lev, int nt, int taper_first, SnapW sw, int last_snap)
{
    using D = ResDim<NR>;
    __shared__ float lds[2 * D::P + 2 * D::Q];
    const int tid = threadIdx.x + 64 * threadIdx.y;
    for (int k = tid; k < 2 * D::P + 2 * D::Q; k += 64 * kResNW) lds[k] = 0.f;
    const int tile = xcd_tile();
    const ShotB sh = A.shots[A.tile_shot[tile]];
    const int tl = tile - sh.tile0;
    const int x0 = 4 + (tl % sh.ntx) * 64, z0 = 4 + (tl / sh.ntx) * D::TH;
    ResTile<NR> t;
    t.init(A, sh, tile, z0);
    ResTaper<NR> tap;
    const bool one = tap.init(A, sh, t, x0, z0), full = t.nk == NR && x0 + 64 <= sh.nnx - 4;
    __syncthreads();
    if (full && one)
        fwd2d_res_body<NR, SF, kResInner>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, lev, nt, taper_first, sw,
                                          last_snap);
    else if (full)
        fwd2d_res_body<NR, SF, kResFull>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, lev, nt, taper_first, sw,
                                         last_snap);
    else
        fwd2d_res_body<NR, SF, kResAny>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, lev, nt, taper_first, sw,
                                        last_snap);
}

// Adjoint pass: the last residual injected at the receivers, then levels
// nt-3..0 of the exact transpose (backwardDC, kernels.cu:104-148) with the
// residual injected between trace rows, the taper and gradientCrossCor
// against the interpolated snapshots (objFuncGradient_f.cu:225-300).  The
// gradient stays in registers until the end; each snapshot slot is read
// once, when the levels reach it.
// lev[n]: trace rows and slots of the nth level (n = 0: the first image, of
// the injected last residual).
template <int NR, int SF, int KIND>
__device__ __forceinline__ void bwd2d_res_body(const ResArgs &A, const ResTile<NR> &t, const ShotB &sh,
                                               const ResTaper<NR> &tap, int tile, int x, int z0, float *lds,
                                               const LevelB *__restrict__ lev, int nlev, const SnapR &sr, int last_row,
                                               float *__restrict__ G11, float *__restrict__ G13,
                                               float *__restrict__ G33)
{
    using D = ResDim<NR>;
    const int nnx = sh.nnx;
    const int nk = KIND == kResAny ? t.nk : NR;
    const bool act = KIND == kResAny ? x < nnx - 4 : true;
    const unsigned i0 = x + (z0 + t.row0) * nnx;
    auto pl = [&](unsigned n) { return lds + (n & 1) * D::P; };
    auto ql = [&](unsigned n) { return lds + 2 * D::P + (n & 1) * D::Q; };
    float p[NR], q[NR], pp[NR], qp[NR];
    // (the coefficients in LDS: registers are short)
    float *const a11 = lds + 2 * D::P + 2 * D::Q + t.row0 * 64 + t.lane, *const a13 = a11 + D::TH * 64,
                 *const a33 = a13 + D::TH * 64;
    float g11[NR], g13[NR], g33[NR], d0p[NR], d0q[NR], d1p[NR], d1q[NR];
    // this lane's receivers: its rows of them, and the first in the tile's
    // list, which is ordered by wavefront, lane and row
    unsigned rmask = 0;
    int rbase = A.rec_at[tile];
    const int rec1 = A.rec_at[tile + 1];
    auto key = [&](int pt) { return (((pt >> 6) / NR) * 64 + (pt & 63)) * NR + (pt >> 6) % NR; };
    for (int hi = rec1; rbase < hi;) {
        const int m = (rbase + hi) >> 1;
        if (key(A.rec[m].pt) < (t.w * 64 + t.lane) * NR) rbase = m + 1;
        else hi = m;
    }
    int at = rbase;
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        p[k] = q[k] = pp[k] = qp[k] = 0.f;
        g11[k] = g13[k] = g33[k] = d0p[k] = d0q[k] = d1p[k] = d1q[k] = 0.f;
        if (k < nk && act) {
            const long long c = sh.c_off + x + (long long)(z0 + t.row0 + k) * A.bg.cpitch;
            a11[k * 64] = A.c11[c];
            a13[k * 64] = A.c13[c];
            a33[k * 64] = A.c33[c];
            if (at < rec1 && A.rec[at].pt == (t.row0 + k) * 64 + t.lane) {
                rmask |= 1u << k;
                // injectData of the last row into zero fields
                const float r0 = A.tr[sh.r_off + (long long)last_row * sh.nr + A.rec[at++].ir];
                const float s = 0.5f * ((1.f - 0.f) * r0 + 0.f * 0.f);
                p[k] += A.dt2 * s;
                q[k] += A.dt2 * s;
            }
        }
    }
    const bool anyrec = __ballot(rmask != 0) != 0;
    const int ir0 = rmask ? A.rec[rbase].ir : 0;
    int slot = -2;
    auto load_slot = [&](int s, float (&dp)[NR], float (&dq)[NR]) {
#pragma unroll
        for (int k = 0; k < NR; ++k)
            if (k < nk && act) {
                dp[k] = snap_raw32<SF>(sr, sh, (long long)nnx * A.bg.nnz, s, 0, i0 + k * nnx);
                dq[k] = snap_raw32<SF>(sr, sh, (long long)nnx * A.bg.nnz, s, 1, i0 + k * nnx);
            }
        if (SF == 3) {
#pragma unroll
            for (int k = 0; k < NR; ++k)
                if (k < nk) {
                    const long long sg = __builtin_amdgcn_readfirstlane((int)s16_seg(nnx, x - t.lane, z0 + t.row0 + k));
                    dp[k] = snap_mul<SF>(sr, sh, A.bg.nnz, s, 0, sg, dp[k]);
                    dq[k] = snap_mul<SF>(sr, sh, A.bg.nnz, s, 1, sg, dq[k]);
                }
        }
    };
    auto slots = [&](int s) {  // the snapshots around a level, before they are used
        if (s == slot) return;
        if (s == slot - 1) {
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                d1p[k] = d0p[k];
                d1q[k] = d0q[k];
            }
        } else {
            load_slot(s + 1, d1p, d1q);
        }
        load_slot(s, d0p, d0q);
        slot = s;
    };
    auto image = [&](float f, const float (&pn)[NR], const float (&qn)[NR]) {
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const float Dp = (1.f - f) * d0p[k] + f * d1p[k];
            const float Dq = (1.f - f) * d0q[k] + f * d1q[k];
            g11[k] = g11[k] + pn[k] * Dp;
            g13[k] = g13[k] + (pn[k] * Dq + qn[k] * Dp);
            g33[k] = g33[k] + qn[k] * Dq;
        }
    };
    auto send = [&](unsigned tag, const float (&pn)[NR], const float (&qn)[NR]) {
        float a[NR], b[NR];
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const float c13 = a13[k * 64];
            a[k] = a11[k * 64] * pn[k] + c13 * qn[k];
            b[k] = c13 * pn[k] + a33[k * 64] * qn[k];
        }
        res_send<NR>(t, A.halo, pl(tag), ql(tag), a, b, tag);
    };
    bool gone = false;
    send(1, p, q);
    slots(lev[0].slot);
    image(lev[0].f, p, q);
    LevelB l = lev[min(1, nlev - 1)];
    res_recv<NR>(t, A.halo, A.abort, gone, pl(1), ql(1), 1);
    lds_barrier();
    // The nth level from the current (pc, qc) over the previous (p, q); the
    // next level's entry is read ahead of the wait, as in the forward pass.
    auto step = [&](int n) {
        const LevelB cur = l;
        const unsigned tag = n + 1;
        __builtin_amdgcn_s_setprio(1);
        slots(cur.slot);
        // the residual rows at the lane's first receiver, ahead of their use
        const float *row = A.tr + sh.r_off + (long long)cur.row * sh.nr;
        float r0 = 0.f, r1 = 0.f;
        if (anyrec && rmask) {
            r0 = row[ir0];
            r1 = row[ir0 + sh.nr];
        }
        float tp[NR], tq[NR], unused_p[NR], unused_q[NR];
        res_d<NR>(t, A, pl(n), ql(n), nk, act, tp, tq, unused_p, unused_q);
        int e = rbase;
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const float tk = tap.template at<KIND>(k);
            float pn = 2.f * p[k] + A.dt2 * tp[k] - (KIND == kResInner ? pp[k] : pp[k] * tk);
            float qn = 2.f * q[k] + A.dt2 * tq[k] - (KIND == kResInner ? qp[k] : qp[k] * tk);
            if (anyrec && (rmask >> k & 1)) {
                if (e != rbase) {  // further receivers of the lane
                    const int ir = A.rec[e].ir;
                    r0 = row[ir];
                    r1 = row[ir + sh.nr];
                }
                ++e;
                const float s = 0.5f * ((1.f - cur.fr) * r0 + cur.fr * r1);
                pn += A.dt2 * s;
                qn += A.dt2 * s;
            }
            const bool on = KIND != kResAny || (act && k < nk);
            pp[k] = p[k];
            qp[k] = q[k];
            p[k] = KIND == kResInner ? pn : on ? pn * tk : 0.f;
            q[k] = KIND == kResInner ? qn : on ? qn * tk : 0.f;
        }
        if (n + 1 < nlev) send(tag, p, q);
        __builtin_amdgcn_s_setprio(0);
        l = lev[min(n + 1, nlev - 1)];
        image(cur.f, p, q);
        if (n + 1 < nlev) {
            res_recv<NR>(t, A.halo, A.abort, gone, pl(tag), ql(tag), tag);
            lds_barrier();
        }
    };
    for (int n = 1; n < nlev; ++n) step(n);
#pragma unroll
    for (int k = 0; k < NR; ++k)
        if (k < nk && act) {
            const long long i = sh.f_off + i0 + k * nnx;
            G11[i] = g11[k];
            G13[i] = g13[k];
            G33[i] = g33[k];
        }
}

template <int NR, int SF>
static __global__ __launch_bounds__(64 * kResNW) __attribute__((amdgpu_waves_per_eu(3))) void bwd2d_res_kernel(
    ResArgs A, const LevelB *__restrict__ lev, int nlev, SnapR sr, int last_row, float *__restrict__ G11,
    float *__restrict__ G13, float *__restrict__ G33)
{
    using D = ResDim<NR>;
    __shared__ float lds[2 * D::P + 2 * D::Q + 3 * D::TH * 64];
    const int tid = threadIdx.x + 64 * threadIdx.y;
    for (int k = tid; k < 2 * D::P + 2 * D::Q + 3 * D::TH * 64; k += 64 * kResNW) lds[k] = 0.f;
    const int tile = xcd_tile();
    const ShotB sh = A.shots[A.tile_shot[tile]];
    const int tl = tile - sh.tile0;
    const int x0 = 4 + (tl % sh.ntx) * 64, z0 = 4 + (tl / sh.ntx) * D::TH;
    ResTile<NR> t;
    t.init(A, sh, tile, z0);
    ResTaper<NR> tap;
    const bool one = tap.init(A, sh, t, x0, z0), full = t.nk == NR && x0 + 64 <= sh.nnx - 4;
    __syncthreads();
    if (full && one)
        bwd2d_res_body<NR, SF, kResInner>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, lev, nlev, sr, last_row, G11,
                                          G13, G33);
    else if (full)
        bwd2d_res_body<NR, SF, kResFull>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, lev, nlev, sr, last_row, G11,
                                         G13, G33);
    else
        bwd2d_res_body<NR, SF, kResAny>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, lev, nlev, sr, last_row, G11,
                                        G13, G33);
}


// Forward pass of GNhessian_f (hessian_f.cu:735-806): the background field as
// above, and the Born field with the scattering source dt2 * (dC * D p)
// (kernels.cu:282-291), which is the one recorded; the background's D snapshots
// in FP32.  One shot.
template <int NR, int KIND>
__device__ __forceinline__ void born2d_res_body(const ResArgs &A, const ResTile<NR> &t, const ShotB &sh,
                                                const ResTaper<NR> &tap, int tile, int x, int z0, float *lds,
                                                const float *__restrict__ dc11, const float *__restrict__ dc13,
                                                const float *__restrict__ dc33, const LevF *__restrict__ lev, int nt,
                                                const SnapW &sw, int last_snap)
{
    using D = ResDim<NR>;
    const int nnx = sh.nnx, tid = t.lane + 64 * t.w;
    const int nk = KIND == kResAny ? t.nk : NR;
    const bool act = KIND == kResAny ? x < nnx - 4 : true;
    const unsigned i0 = x + (z0 + t.row0) * nnx;
    constexpr int F = 2 * D::P + 2 * D::Q;  // the Born field's planes follow the background's
    auto pl = [&](int it) { return lds + (it & 1) * D::P; };
    auto ql = [&](int it) { return lds + 2 * D::P + (it & 1) * D::Q; };
    ResTile<NR> tb = t;  // and so do its strips
    tb.wc += 2 * D::WORDS;
    tb.wt += 2 * D::WORDS;
    tb.wb += 2 * D::WORDS;
    tb.wx += 2 * D::WORDS;
    tb.wu += 2 * D::WORDS;
    tb.wd += 2 * D::WORDS;
    float p[NR], q[NR], dp[NR], dq[NR], a11[NR], a13[NR], a33[NR], b11[NR], b13[NR], b33[NR];
    unsigned smask = 0;
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        p[k] = q[k] = dp[k] = dq[k] = a11[k] = a13[k] = a33[k] = b11[k] = b13[k] = b33[k] = 0.f;
        if (k < nk && act) {
            const unsigned i = i0 + k * nnx;
            a11[k] = A.c11[i];
            a13[k] = A.c13[i];
            a33[k] = A.c33[i];
            b11[k] = dc11[i];
            b13[k] = dc13[i];
            b33[k] = dc33[i];
            if ((int)i == sh.src) {
                smask |= 1u << k;
                p[k] = q[k] = lev[1].src;
            }
        }
    }
    const bool has_src = __ballot(smask != 0) != 0;
    const int rec0 = A.rec_at[tile], rec1 = A.rec_at[tile + 1];
    auto put_snap = [&](int slot, const float (&tp)[NR], const float (&tq)[NR]) {
#pragma unroll
        for (int k = 0; k < NR; ++k)
            if (k < nk && act) snap_put32(sw, sh, (long long)nnx * A.bg.nnz, slot, i0 + k * nnx, tp[k], tq[k]);
    };
    bool gone = false;
    res_send<NR>(t, A.halo, pl(1), ql(1), p, q, 1);
    res_send<NR>(tb, A.halo, pl(1) + F, ql(1) + F, dp, dq, 1);
    LevF l = lev[min(2, nt - 1)];
    res_recv<NR>(t, A.halo, A.abort, gone, pl(1), ql(1), 1);
    res_recv<NR>(tb, A.halo, A.abort, gone, pl(1) + F, ql(1) + F, 1);
    lds_barrier();
    for (int it = 2; it < nt; ++it) {
        const LevF cur = l;
        float tp[NR], tq[NR], bp[NR], bq[NR], pc[NR], qc[NR];
        const int own_p = t.row0 * D::PW + t.lane + 4, own_q = (t.row0 + 4) * D::QW + t.lane;
        res_d<NR>(t, A, pl(it - 1), ql(it - 1), nk, act, tp, tq, pc, qc);
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const float tk = tap.template at<KIND>(k), pp = pl(it)[own_p + k * D::PW], qp = ql(it)[own_q + k * D::QW];
            float pn = 2.f * pc[k] + A.dt2 * (a11[k] * tp[k] + a13[k] * tq[k]) - (KIND == kResInner ? pp : pp * tk);
            float qn = 2.f * qc[k] + A.dt2 * (a13[k] * tp[k] + a33[k] * tq[k]) - (KIND == kResInner ? qp : qp * tk);
            if (has_src && (smask >> k & 1)) {
                pn += cur.src;
                qn += cur.src;
            }
            const bool on = KIND != kResAny || (act && k < nk);
            p[k] = KIND == kResInner ? pn : on ? pn * tk : 0.f;
            q[k] = KIND == kResInner ? qn : on ? qn * tk : 0.f;
        }
        res_send<NR>(t, A.halo, pl(it), ql(it), p, q, it);
        res_d<NR>(t, A, pl(it - 1) + F, ql(it - 1) + F, nk, act, bp, bq, pc, qc);
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const float tk = tap.template at<KIND>(k), pp = (pl(it) + F)[own_p + k * D::PW],
                        qp = (ql(it) + F)[own_q + k * D::QW];
            float pn = 2.f * pc[k] + A.dt2 * (a11[k] * bp[k] + a13[k] * bq[k]) - (KIND == kResInner ? pp : pp * tk);
            float qn = 2.f * qc[k] + A.dt2 * (a13[k] * bp[k] + a33[k] * bq[k]) - (KIND == kResInner ? qp : qp * tk);
            pn += A.dt2 * (b11[k] * tp[k] + b13[k] * tq[k]);
            qn += A.dt2 * (b13[k] * tp[k] + b33[k] * tq[k]);
            const bool on = KIND != kResAny || (act && k < nk);
            dp[k] = KIND == kResInner ? pn : on ? pn * tk : 0.f;
            dq[k] = KIND == kResInner ? qn : on ? qn * tk : 0.f;
        }
        res_send<NR>(tb, A.halo, pl(it) + F, ql(it) + F, dp, dq, it);
        l = lev[min(it + 1, nt - 1)];
        if (cur.snap >= 0) put_snap(cur.snap, tp, tq);
        res_recv<NR>(t, A.halo, A.abort, gone, pl(it), ql(it), it);
        res_recv<NR>(tb, A.halo, A.abort, gone, pl(it) + F, ql(it) + F, it);
        lds_barrier();
        if (cur.row >= 0 && rec0 < rec1) {
            const float *pr = pl(it) + F + 4, *qr = ql(it) + F + 4 * D::QW;
            float *out = A.tr + sh.r_off + (long long)cur.row * sh.nr;
            for (int e = rec0 + tid; e < rec1; e += 64 * kResNW) {
                const ResRec r = A.rec[e];
                out[r.ir] = 0.5f * (pr[(r.pt >> 6) * D::PW + (r.pt & 63)] + qr[r.pt]);
            }
        }
    }
    float tp[NR], tq[NR], pc[NR], qc[NR];
    res_d<NR>(t, A, pl(nt - 1), ql(nt - 1), nk, act, tp, tq, pc, qc);
    put_snap(last_snap, tp, tq);
}

template <int NR>
static __global__ __launch_bounds__(64 * kResNW) __attribute__((amdgpu_waves_per_eu(NR == 6 ? 2 : 3))) void born2d_res_kernel(
    ResArgs A, const float *__restrict__ dc11, const float *__restrict__ dc13, const float *__restrict__ dc33,
    const LevF *__restrict__ lev, int nt, SnapW sw, int last_snap)
{
    using D = ResDim<NR>;
    __shared__ float lds[4 * D::P + 4 * D::Q];
    const int tid = threadIdx.x + 64 * threadIdx.y;
    for (int k = tid; k < 4 * D::P + 4 * D::Q; k += 64 * kResNW) lds[k] = 0.f;
    const int tile = xcd_tile();
    const ShotB sh = A.shots[A.tile_shot[tile]];
    const int tl = tile - sh.tile0;
    const int x0 = 4 + (tl % sh.ntx) * 64, z0 = 4 + (tl / sh.ntx) * D::TH;
    ResTile<NR> t;
    t.init(A, sh, tile, z0, 2);
    ResTaper<NR> tap;
    const bool one = tap.init(A, sh, t, x0, z0), full = t.nk == NR && x0 + 64 <= sh.nnx - 4;
    __syncthreads();
    if (full && one)
        born2d_res_body<NR, kResInner>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, dc11, dc13, dc33, lev, nt, sw,
                                       last_snap);
    else if (full)
        born2d_res_body<NR, kResFull>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, dc11, dc13, dc33, lev, nt, sw,
                                      last_snap);
    else
        born2d_res_body<NR, kResAny>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, dc11, dc13, dc33, lev, nt, sw,
                                     last_snap);
}

// Backward pass on the forward operator (forwardCD), one shot.  IMG 0:
// GNhessian_f's adjoint (hessian_f.cu:834-900), the Born traces injected and
// imaged as in the adjoint above.  IMG 1: rtm_f's receiver side
// (rtm_f.cu:152-216), data injected as dipoles and
// image += 0.5 (p + q) * the interpolated slice.
// lev[n]: as for the adjoint; row < 0: nothing injected at this level.
template <int NR, int IMG, int KIND>
__device__ __forceinline__ void back2d_res_body(const ResArgs &A, const ResTile<NR> &t, const ShotB &sh,
                                                const ResTaper<NR> &tap, int tile, int x, int z0, float *lds,
                                                const LevelB *__restrict__ lev, int nlev,
                                                const float *__restrict__ snap, int last_row, float *__restrict__ G11,
                                                float *__restrict__ G13, float *__restrict__ G33)
{
    using D = ResDim<NR>;
    constexpr int NI = IMG ? 1 : 3, NS = IMG ? 1 : 2;  // images, planes of a slot
    const int nnx = sh.nnx;
    const int nk = KIND == kResAny ? t.nk : NR;
    const bool act = KIND == kResAny ? x < nnx - 4 : true;
    const unsigned i0 = x + (z0 + t.row0) * nnx;
    const long long plane = (long long)nnx * A.bg.nnz;
    auto pl = [&](unsigned n) { return lds + (n & 1) * D::P; };
    auto ql = [&](unsigned n) { return lds + 2 * D::P + (n & 1) * D::Q; };
    float p[NR], q[NR], a11[NR], a13[NR], a33[NR], g[NI][NR], d0[NS][NR], d1[NS][NR];
    unsigned rmask = 0, nmask = 0;  // rows with a receiver; those of a negative pole
    int rbase = A.rec_at[tile];
    const int rec1 = A.rec_at[tile + 1];
    auto key = [&](int pt) { return (((pt >> 6) / NR) * 64 + (pt & 63)) * NR + (pt >> 6) % NR; };
    for (int hi = rec1; rbase < hi;) {
        const int m = (rbase + hi) >> 1;
        if (key(A.rec[m].pt) < (t.w * 64 + t.lane) * NR) rbase = m + 1;
        else hi = m;
    }
    auto column = [](int ir) { return ir < 0 ? ~ir : ir; };
    int at = rbase;
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        p[k] = q[k] = a11[k] = a13[k] = a33[k] = 0.f;
#pragma unroll
        for (int j = 0; j < NI; ++j) g[j][k] = 0.f;
#pragma unroll
        for (int j = 0; j < NS; ++j) d0[j][k] = d1[j][k] = 0.f;
        if (k < nk && act) {
            a11[k] = A.c11[i0 + k * nnx];
            a13[k] = A.c13[i0 + k * nnx];
            a33[k] = A.c33[i0 + k * nnx];
            if (at < rec1 && A.rec[at].pt == (t.row0 + k) * 64 + t.lane) {
                const int ir = A.rec[at++].ir;
                rmask |= 1u << k;
                if (ir < 0) nmask |= 1u << k;
                // the last row into zero fields; the taper follows in rtm_f alone
                const float r0 = A.tr[(long long)last_row * sh.nr + column(ir)];
                const float s = 0.5f * ((1.f - 0.f) * r0 + 0.f * 0.f), v = A.dt2 * s;
                if (IMG) p[k] = ir < 0 ? -v * tap.template at<KIND>(k) : v * tap.template at<KIND>(k);
                else p[k] += v;
                q[k] = p[k];
            }
        }
    }
    const bool anyrec = __ballot(rmask != 0) != 0;
    const int ir0 = rmask ? column(A.rec[rbase].ir) : 0;
    int slot = -2;
    auto load_slot = [&](int s, float (&d)[NS][NR]) {
#pragma unroll
        for (int j = 0; j < NS; ++j)
#pragma unroll
            for (int k = 0; k < NR; ++k)
                if (k < nk && act) d[j][k] = ld32(snap + ((long long)s * NS + j) * plane, i0 + k * nnx);
    };
    auto slots = [&](int s) {
        if (s == slot) return;
        if (s == slot - 1) {
#pragma unroll
            for (int j = 0; j < NS; ++j)
#pragma unroll
                for (int k = 0; k < NR; ++k) d1[j][k] = d0[j][k];
        } else {
            load_slot(s + 1, d1);
        }
        load_slot(s, d0);
        slot = s;
    };
    auto image = [&](float f) {
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const float Dp = (1.f - f) * d0[0][k] + f * d1[0][k];
            if (IMG) {
                g[0][k] = g[0][k] + 0.5f * (p[k] + q[k]) * Dp;
            } else {
                const float Dq = (1.f - f) * d0[NS - 1][k] + f * d1[NS - 1][k];
                g[0][k] = g[0][k] + p[k] * Dp;
                g[NI / 2][k] = g[NI / 2][k] + (p[k] * Dq + q[k] * Dp);
                g[NI - 1][k] = g[NI - 1][k] + q[k] * Dq;
            }
        }
    };
    bool gone = false;
    res_send<NR>(t, A.halo, pl(1), ql(1), p, q, 1);
    slots(lev[0].slot);
    image(lev[0].f);
    LevelB l = lev[min(1, nlev - 1)];
    res_recv<NR>(t, A.halo, A.abort, gone, pl(1), ql(1), 1);
    lds_barrier();
    for (int n = 1; n < nlev; ++n) {
        const LevelB cur = l;
        const unsigned tag = n + 1;
        slots(cur.slot);
        const bool inject = anyrec && cur.row >= 0;
        const float *row = A.tr + (long long)cur.row * sh.nr;
        float r0 = 0.f, r1 = 0.f;
        if (inject && rmask) {
            r0 = row[ir0];
            r1 = row[ir0 + sh.nr];
        }
        float tp[NR], tq[NR], pc[NR], qc[NR];
        res_d<NR>(t, A, pl(n), ql(n), nk, act, tp, tq, pc, qc);
        const float *pv = pl(tag) + t.row0 * D::PW + t.lane + 4, *qv = ql(tag) + (t.row0 + 4) * D::QW + t.lane;
        int e = rbase;
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const float tk = tap.template at<KIND>(k), pp = pv[k * D::PW], qp = qv[k * D::QW];
            float pn = 2.f * pc[k] + A.dt2 * (a11[k] * tp[k] + a13[k] * tq[k]) - (KIND == kResInner ? pp : pp * tk);
            float qn = 2.f * qc[k] + A.dt2 * (a13[k] * tp[k] + a33[k] * tq[k]) - (KIND == kResInner ? qp : qp * tk);
            if (inject && (rmask >> k & 1)) {
                if (e != rbase) {  // further receivers of the lane
                    const int ir = column(A.rec[e].ir);
                    r0 = row[ir];
                    r1 = row[ir + sh.nr];
                }
                ++e;
                const float s = 0.5f * ((1.f - cur.fr) * r0 + cur.fr * r1);
                if (IMG && (nmask >> k & 1)) {
                    pn -= A.dt2 * s;
                    qn -= A.dt2 * s;
                } else {
                    pn += A.dt2 * s;
                    qn += A.dt2 * s;
                }
            }
            const bool on = KIND != kResAny || (act && k < nk);
            p[k] = KIND == kResInner ? pn : on ? pn * tk : 0.f;
            q[k] = KIND == kResInner ? qn : on ? qn * tk : 0.f;
        }
        if (n + 1 < nlev) res_send<NR>(t, A.halo, pl(tag), ql(tag), p, q, tag);
        l = lev[min(n + 1, nlev - 1)];
        image(cur.f);
        if (n + 1 < nlev) {
            res_recv<NR>(t, A.halo, A.abort, gone, pl(tag), ql(tag), tag);
            lds_barrier();
        }
    }
#pragma unroll
    for (int k = 0; k < NR; ++k)
        if (k < nk && act) {
            G11[i0 + k * nnx] = g[0][k];
            if (!IMG) {
                G13[i0 + k * nnx] = g[NI / 2][k];
                G33[i0 + k * nnx] = g[NI - 1][k];
            }
        }
}

template <int NR, int IMG>
static __global__ __launch_bounds__(64 * kResNW) __attribute__((amdgpu_waves_per_eu(3))) void back2d_res_kernel(
    ResArgs A, const LevelB *__restrict__ lev, int nlev, const float *__restrict__ snap, int last_row,
    float *__restrict__ G11, float *__restrict__ G13, float *__restrict__ G33)
{
    using D = ResDim<NR>;
    __shared__ float lds[2 * D::P + 2 * D::Q];
    const int tid = threadIdx.x + 64 * threadIdx.y;
    for (int k = tid; k < 2 * D::P + 2 * D::Q; k += 64 * kResNW) lds[k] = 0.f;
    const int tile = xcd_tile();
    const ShotB sh = A.shots[A.tile_shot[tile]];
    const int tl = tile - sh.tile0;
    const int x0 = 4 + (tl % sh.ntx) * 64, z0 = 4 + (tl / sh.ntx) * D::TH;
    ResTile<NR> t;
    t.init(A, sh, tile, z0);
    ResTaper<NR> tap;
    const bool one = tap.init(A, sh, t, x0, z0), full = t.nk == NR && x0 + 64 <= sh.nnx - 4;
    __syncthreads();
    if (full && one)
        back2d_res_body<NR, IMG, kResInner>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, lev, nlev, snap, last_row, G11,
                                            G13, G33);
    else if (full)
        back2d_res_body<NR, IMG, kResFull>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, lev, nlev, snap, last_row, G11,
                                           G13, G33);
    else
        back2d_res_body<NR, IMG, kResAny>(A, t, sh, tap, tile, x0 + t.lane, z0, lds, lev, nlev, snap, last_row, G11,
                                          G13, G33);
}

}  // namespace vti
