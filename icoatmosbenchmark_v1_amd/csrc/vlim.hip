// vertical_limiter_thuburn on gfx950.
//
// Reference: kernels/NICAM/dyn_vert_adv_limiter/src/mod_src_tracer.f90:41-243.
//
// The limited half-level value q_h(k) needs the allowable ranges Qout of
// levels k-1 and k; the reference carries Qout(k-1) from one level to the
// next (:140-141, :182-183), but every (g, k) is independent.  One work-item
// handles a run of KC consecutive levels of one column: it recomputes Qout of
// the level just below its run (the reference's peel at kmin plays that role
// for the first run), then marches up carrying Qout, q(k-1), q(k) and
// ck(k,1) in registers.  A wavefront covers 64 consecutive g at one level, so
// every load and store is contiguous.  The pole columns are appended as the
// last work-items.
//
// Many tracers (q(gall,kall,lall,ntr), NICAM's tracer-last layout) share ck
// and d: a work-group limits one tracer, and the tracers of one column block
// and run are consecutive work-groups on one XCD, whose L2 serves ck and d to
// all but the first (eight FP32 tracers on four grids 1.15 ms, against 1.25 ms
// with four tracers per work-item and their levels loaded one at a time, which
// stays the better form for other short runs than the default's).
#include <type_traits>

#include "internal.h"

namespace nicam {
namespace {

constexpr int BLOCK = 256;
constexpr int RUN_KC = 4;  // levels per run; gl7: 4 164 us, 8 168, 16 168, runtime-length 169 (FP64)
constexpr int LONG_KC = 8; // the other length known at compile time; of the masked kernel: a byte of a mask word
constexpr int VTB = 4;     // tracers per work-item of the multi-tracer kernel
constexpr int WIN = 4;     // column blocks an XCD takes at a time (gl7: 1 541 us for the vertical half, 4 530, 8 540)

template <class T>
__device__ __forceinline__ T dmin(T a, T b) { return (b < a) ? b : a; }
template <class T>
__device__ __forceinline__ T dmax(T a, T b) { return (b > a) ? b : a; }
__device__ __forceinline__ double sign_half(double x) { return copysign(0.5, x); }
__device__ __forceinline__ float sign_half(float x) { return copysignf(0.5f, x); }
__device__ __forceinline__ double tabs(double x) { return fabs(x); }
__device__ __forceinline__ float tabs(float x) { return fabsf(x); }

template <class T>
struct VlimArgs {
    T *q_h;
    const T *q, *d, *ck;
    T *q_h_pl;
    const T *q_pl, *d_pl, *ck_pl;
    int gall, kall, lall, gall_pl, have_pl;
    int kc, nrun;  // levels per work-item, runs per column
    int ngrp, multi;  // work-groups of one column block and run: a tracer each, or VTB tracers (multi)
    T eps, big;
    int ntr;          // tracers
    long ts, tps;     // tracer strides of the regular and pole fields
    unsigned ncol;    // columns, the poles' last
    unsigned unit, win, wfull;  // work-groups of a column block, of a window of 8 * WIN blocks, of all whole windows
    uint32_t *mask, *mask_pl;  // clip bits (masked variant only; kc = 8)
};

// Levels [kb, ke) of one column are limited (kb >= kmin+1, 0-based).
// base = offset of level 0, s = stride between levels, ck2 = offset of the
// upper-face plane of ck.  POLE selects the pole loop's product grouping of
// CQin (VLIM:212-215 versus :126-129).
template <bool POLE, class T>
__device__ __forceinline__ void vlim_run(T *__restrict__ q_h, const T *__restrict__ q, const T *__restrict__ d,
                                         const T *__restrict__ ck, size_t base, size_t s, size_t ck2, int kb,
                                         int ke, T EPS, T BIG)
{
    int k = kb - 1;  // first level whose Qout is needed
    T qkm1 = q[base + (size_t)(k - 1) * s];
    T qk = q[base + (size_t)k * s];
    T ck1k = ck[base + (size_t)k * s];
    T Qmin_km1 = T(0), Qmax_km1 = T(0);
    for (; k < ke; ++k) {
        const size_t o = base + (size_t)k * s;
        const T qkp1 = q[o + s];
        const T ck1kp1 = ck[o + s];
        const T ck2k = ck[ck2 + o];
        const T dk = d[o];
        const T inflagL = T(0.5) - sign_half(ck1k);
        const T inflagU = T(0.5) + sign_half(ck1kp1);
        const T Qin_minL = dmin(qk, qkm1) + (T(1) - inflagL) * BIG;
        const T Qin_minU = dmin(qk, qkp1) + (T(1) - inflagU) * BIG;
        const T Qin_maxL = dmax(qk, qkm1) - (T(1) - inflagL) * BIG;
        const T Qin_maxU = dmax(qk, qkp1) - (T(1) - inflagU) * BIG;
        const T qnext_min = dmin(dmin(Qin_minL, Qin_minU), qk);
        const T qnext_max = dmax(dmax(Qin_maxL, Qin_maxU), qk);
        const T Cin = (inflagL)*ck1k + (inflagU)*ck2k;
        const T Cout = (T(1) - inflagL) * ck1k + (T(1) - inflagU) * ck2k;
        T CQin_min, CQin_max;
        if constexpr (POLE) {
            CQin_max = (inflagL) * (ck1k * Qin_maxL) + (inflagU) * (ck2k * Qin_maxU);
            CQin_min = (inflagL) * (ck1k * Qin_minL) + (inflagU) * (ck2k * Qin_minU);
        } else {
            CQin_min = (inflagL)*ck1k * Qin_minL + (inflagU)*ck2k * Qin_minU;
            CQin_max = (inflagL)*ck1k * Qin_maxL + (inflagU)*ck2k * Qin_maxU;
        }
        const T zerosw = T(0.5) - sign_half(tabs(Cout) - EPS);
        const T Qmin_k = ((qk - qnext_max) + qnext_max * (Cin + Cout - dk) - CQin_max) / (Cout + zerosw) *
                                  (T(1) - zerosw) + qk * zerosw;
        const T Qmax_k = ((qk - qnext_min) + qnext_min * (Cin + Cout - dk) - CQin_min) / (Cout + zerosw) *
                                  (T(1) - zerosw) + qk * zerosw;
        if (k >= kb) {  // VLIM:179-180
            const T qh = q_h[o];
            const T out = (inflagL)*dmax(dmin(qh, Qmax_km1), Qmin_km1) + (T(1) - inflagL) * dmax(dmin(qh, Qmax_k), Qmin_k);
            stream_store(&q_h[o], out);
        }
        Qmin_km1 = Qmin_k;
        Qmax_km1 = Qmax_k;
        qkm1 = qk;
        qk = qkp1;
        ck1k = ck1kp1;
    }
}

// vlim_run with the run's length fixed at KC levels at compile time: every
// input of the run (q on kb-2..ke, ck on kb-1..ke, d on kb-1..ke-1, q_h on
// kb..ke-1) is loaded before the first level is formed, so a work-item waits
// for memory once per run rather than once per level, and runs can be long
// (fewer levels re-read at run edges) without losing loads in flight.  A
// shorter last run (ke - kb < KC) reads level ke in place of the levels past
// it and stores nothing there.  Same operations, in the same order, as
// vlim_run.  Returns a bit per face of the run, set where the limited value
// differs from q_h's input (dead code unless the caller stores it).
template <bool POLE, class T, int KC>
__device__ __forceinline__ uint32_t vlim_run_kc(T *__restrict__ q_h, const T *__restrict__ q, const T *__restrict__ d,
                                            const T *__restrict__ ck, size_t base, size_t s, size_t ck2, int kb,
                                            int ke, T EPS, T BIG)
{
    auto at = [&](int k) { return base + (size_t)(k < ke ? k : ke) * s; };
    T qv[KC + 3], c1[KC + 2], c2[KC + 1], dv[KC + 1], qh[KC];
#pragma unroll
    for (int t = 0; t < KC + 3; ++t) qv[t] = q[at(kb - 2 + t)];
#pragma unroll
    for (int t = 0; t < KC + 2; ++t) c1[t] = ck[at(kb - 1 + t)];
#pragma unroll
    for (int t = 0; t < KC + 1; ++t) {
        c2[t] = ck[ck2 + at(kb - 1 + t)];
        dv[t] = d[at(kb - 1 + t)];
    }
#pragma unroll
    for (int t = 0; t < KC; ++t) qh[t] = q_h[at(kb + t)];
    uint32_t bits = 0;
    T Qmin_km1 = T(0), Qmax_km1 = T(0);
#pragma unroll
    for (int t = 0; t <= KC; ++t) {  // level k = kb - 1 + t
        const int k = kb - 1 + t;
        const T qkm1 = qv[t], qk = qv[t + 1], qkp1 = qv[t + 2];
        const T ck1k = c1[t], ck1kp1 = c1[t + 1], ck2k = c2[t], dk = dv[t];
        const T inflagL = T(0.5) - sign_half(ck1k);
        const T inflagU = T(0.5) + sign_half(ck1kp1);
        const T Qin_minL = dmin(qk, qkm1) + (T(1) - inflagL) * BIG;
        const T Qin_minU = dmin(qk, qkp1) + (T(1) - inflagU) * BIG;
        const T Qin_maxL = dmax(qk, qkm1) - (T(1) - inflagL) * BIG;
        const T Qin_maxU = dmax(qk, qkp1) - (T(1) - inflagU) * BIG;
        const T qnext_min = dmin(dmin(Qin_minL, Qin_minU), qk);
        const T qnext_max = dmax(dmax(Qin_maxL, Qin_maxU), qk);
        const T Cin = (inflagL)*ck1k + (inflagU)*ck2k;
        const T Cout = (T(1) - inflagL) * ck1k + (T(1) - inflagU) * ck2k;
        T CQin_min, CQin_max;
        if constexpr (POLE) {
            CQin_max = (inflagL) * (ck1k * Qin_maxL) + (inflagU) * (ck2k * Qin_maxU);
            CQin_min = (inflagL) * (ck1k * Qin_minL) + (inflagU) * (ck2k * Qin_minU);
        } else {
            CQin_min = (inflagL)*ck1k * Qin_minL + (inflagU)*ck2k * Qin_minU;
            CQin_max = (inflagL)*ck1k * Qin_maxL + (inflagU)*ck2k * Qin_maxU;
        }
        const T zerosw = T(0.5) - sign_half(tabs(Cout) - EPS);
        const T Qmin_k = ((qk - qnext_max) + qnext_max * (Cin + Cout - dk) - CQin_max) / (Cout + zerosw) *
                                  (T(1) - zerosw) + qk * zerosw;
        const T Qmax_k = ((qk - qnext_min) + qnext_min * (Cin + Cout - dk) - CQin_min) / (Cout + zerosw) *
                                  (T(1) - zerosw) + qk * zerosw;
        if (t >= 1 && k < ke) {  // VLIM:179-180
            const T qhv = qh[t - 1];
            const T out = (inflagL)*dmax(dmin(qhv, Qmax_km1), Qmin_km1) + (T(1) - inflagL) * dmax(dmin(qhv, Qmax_k), Qmin_k);
            stream_store(&q_h[base + (size_t)k * s], out);
            bits |= (out != qhv ? 1u : 0u) << (t - 1);
        }
        Qmin_km1 = Qmin_k;
        Qmax_km1 = Qmax_k;
    }
    return bits;
}

// vlim_run for up to TB tracers (nb of them) of one column run, which share the
// loads of ck and d and what is formed from them; tracer b's fields start b*ts
// elements after q / q_h.
template <bool POLE, int TB, class T>
__device__ __forceinline__ void vlim_run_multi(T *__restrict__ q_h, const T *__restrict__ q,
                                               const T *__restrict__ d, const T *__restrict__ ck, size_t base,
                                               size_t s, size_t ck2, int kb, int ke, T EPS, T BIG, int nb, long ts)
{
    int k = kb - 1;
    T qkm1[TB], qk[TB], Qmin_km1[TB], Qmax_km1[TB];
#pragma unroll
    for (int b = 0; b < TB; ++b) {
        const int bb = b < nb ? b : 0;  // idle slots repeat tracer 0 and store nothing
        qkm1[b] = q[bb * ts + base + (size_t)(k - 1) * s];
        qk[b] = q[bb * ts + base + (size_t)k * s];
        Qmin_km1[b] = T(0);
        Qmax_km1[b] = T(0);
    }
    T ck1k = ck[base + (size_t)k * s];
    for (; k < ke; ++k) {
        const size_t o = base + (size_t)k * s;
        const T ck1kp1 = ck[o + s];
        const T ck2k = ck[ck2 + o];
        const T dk = d[o];
        const T inflagL = T(0.5) - sign_half(ck1k);
        const T inflagU = T(0.5) + sign_half(ck1kp1);
        const T Cin = (inflagL)*ck1k + (inflagU)*ck2k;
        const T Cout = (T(1) - inflagL) * ck1k + (T(1) - inflagU) * ck2k;
        const T zerosw = T(0.5) - sign_half(tabs(Cout) - EPS);
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            const int bb = b < nb ? b : 0;
            const T qkp1 = q[bb * ts + o + s];
            const T Qin_minL = dmin(qk[b], qkm1[b]) + (T(1) - inflagL) * BIG;
            const T Qin_minU = dmin(qk[b], qkp1) + (T(1) - inflagU) * BIG;
            const T Qin_maxL = dmax(qk[b], qkm1[b]) - (T(1) - inflagL) * BIG;
            const T Qin_maxU = dmax(qk[b], qkp1) - (T(1) - inflagU) * BIG;
            const T qnext_min = dmin(dmin(Qin_minL, Qin_minU), qk[b]);
            const T qnext_max = dmax(dmax(Qin_maxL, Qin_maxU), qk[b]);
            T CQin_min, CQin_max;
            if constexpr (POLE) {
                CQin_max = (inflagL) * (ck1k * Qin_maxL) + (inflagU) * (ck2k * Qin_maxU);
                CQin_min = (inflagL) * (ck1k * Qin_minL) + (inflagU) * (ck2k * Qin_minU);
            } else {
                CQin_min = (inflagL)*ck1k * Qin_minL + (inflagU)*ck2k * Qin_minU;
                CQin_max = (inflagL)*ck1k * Qin_maxL + (inflagU)*ck2k * Qin_maxU;
            }
            const T Qmin_k = ((qk[b] - qnext_max) + qnext_max * (Cin + Cout - dk) - CQin_max) / (Cout + zerosw) *
                                 (T(1) - zerosw) + qk[b] * zerosw;
            const T Qmax_k = ((qk[b] - qnext_min) + qnext_min * (Cin + Cout - dk) - CQin_min) / (Cout + zerosw) *
                                 (T(1) - zerosw) + qk[b] * zerosw;
            if (k >= kb && b < nb) {  // VLIM:179-180
                const T qh = q_h[b * ts + o];
                const T out = (inflagL)*dmax(dmin(qh, Qmax_km1[b]), Qmin_km1[b]) +
                              (T(1) - inflagL) * dmax(dmin(qh, Qmax_k), Qmin_k);
                stream_store(&q_h[b * ts + o], out);
            }
            Qmin_km1[b] = Qmin_k;
            Qmax_km1[b] = Qmax_k;
            qkm1[b] = qk[b];
            qk[b] = qkp1;
        }
        ck1k = ck1kp1;
    }
}

// A work-group is BLOCK consecutive columns at one run of levels for one
// tracer.  The tracers and runs of one column block are consecutive
// work-groups on one XCD: the tracers read the same ck and d, and each run
// also reads the two levels below it, which the run below has just brought
// into that XCD's L2.  KC > 0: runs of KC levels known at compile time
// (vlim_run_kc); 0: of A.kc levels (vlim_run).
// MASK: with runs of eight faces, a byte of the 32-face mask words each (face
// p is bit p % 32 of word p / 32); the last run clears its word's other bytes.
// (18x18x42x40, where runs of a whole word leave 102 work-groups: 58 -> 12 us.)
// MULTI: VTB tracers to a work-group, their levels loaded one at a time
// (vlim_run_multi).
template <class T, int KC, bool MASK = false, bool MULTI = false>
__device__ __forceinline__ void vlim_block(const VlimArgs<T> &A, unsigned blk)
{
    // every argument at once: behind the branches below they would come one batch after the other
    asm volatile("" ::"s"(A.q_h), "s"(A.q), "s"(A.d), "s"(A.ck), "s"(A.gall), "s"(A.kall), "s"(A.lall), "s"(A.ncol),
                 "s"(A.unit), "s"(A.win), "s"(A.wfull), "s"(A.ngrp), "s"(A.ts), "s"(A.eps), "s"(A.big));
    const unsigned ncol_reg = (unsigned)A.gall * A.lall;
    const unsigned w = blk / A.win, r = blk - w * A.win;
    const unsigned L = blk < A.wfull ? w * A.win + (r & 7) * (A.win >> 3) + (r >> 3) : blk;
    const unsigned cb = L / A.unit, ru = L - cb * A.unit;
    const int run = A.ngrp == 1 ? ru : ru / A.ngrp, grp = ru - run * A.ngrp;
    const unsigned col = cb * BLOCK + threadIdx.x;
    if (col >= A.ncol) return;
    const int kmin = 1, kmax = A.kall - 2;  // 0-based
    const int kc = KC > 0 ? KC : A.kc;
    const int kb = kmin + 1 + run * kc;
    const int ke = min(kmax + 1, kb + kc);
    if (kb >= ke) return;
    const int tr = MULTI ? grp * VTB : grp;
    auto go = [&](auto pole, T *q_h, const T *q, const T *d, const T *ck, unsigned t, int gall, int lall, long ts,
                  uint32_t *mask) {
        constexpr bool POLE = decltype(pole)::value;
        const unsigned l = t / gall, g = t - l * gall;
        const size_t base = (size_t)l * A.kall * gall + g;
        const size_t ck2 = (size_t)gall * A.kall * lall;
        q_h += tr * ts;
        q += tr * ts;
        if constexpr (MULTI) {
            vlim_run_multi<POLE, VTB, T>(q_h, q, d, ck, base, gall, ck2, kb, ke, A.eps, A.big, min(VTB, A.ntr - tr), ts);
        } else if constexpr (KC > 0) {
            const uint32_t bits = vlim_run_kc<POLE, T, KC>(q_h, q, d, ck, base, gall, ck2, kb, ke, A.eps, A.big);
            if constexpr (MASK) {
                static_assert(KC == 8, "a run is one byte of a mask word");
                const int nword = (A.nrun + 3) / 4;
                uint8_t *byte = reinterpret_cast<uint8_t *>(mask + ((size_t)l * nword + run / 4) * gall + g);
                byte[run % 4] = (uint8_t)bits;
                if (run == A.nrun - 1)
                    for (int r = run % 4 + 1; r < 4; ++r) byte[r] = 0;
            }
        } else {
            vlim_run<POLE, T>(q_h, q, d, ck, base, gall, ck2, kb, ke, A.eps, A.big);
        }
    };
    if (col < ncol_reg)
        go(std::false_type{}, A.q_h, A.q, A.d, A.ck, col, A.gall, A.lall, A.ts, A.mask);
    else
        go(std::true_type{}, A.q_h_pl, A.q_pl, A.d_pl, A.ck_pl, col - ncol_reg, A.gall_pl, kLallPl, A.tps, A.mask_pl);
}

template <class T, int KC, bool MASK = false, bool MULTI = false>
__global__ void __launch_bounds__(BLOCK) vlim_kernel(VlimArgs<T> A)
{
    vlim_block<T, KC, MASK, MULTI>(A, blockIdx.x);
}

// several grids in one launch: work-groups [off[n], off[n+1]) belong to grid n
template <class T>
struct VlimGroup {
    VlimArgs<T> a[kMaxGroup];
    int off[kMaxGroup + 1];
    int n;
};

// TUNED: a grid has another run length than RUN_KC (their registers would cost
// the default's occupancy)
template <class T, bool TUNED>
__global__ void __launch_bounds__(BLOCK) vlim_group_kernel(VlimGroup<T> G)
{
    const int b = blockIdx.x;
    int n = 0;
    while (n + 1 < G.n && b >= G.off[n + 1]) ++n;
    const VlimArgs<T> &A = G.a[n];
    const unsigned blk = b - G.off[n];
    if constexpr (!TUNED) {
        vlim_block<T, RUN_KC>(A, blk);
    } else {
        if (A.multi) vlim_block<T, 0, false, true>(A, blk);
        else if (A.kc == RUN_KC) vlim_block<T, RUN_KC>(A, blk);
        else if (A.kc == LONG_KC) vlim_block<T, LONG_KC>(A, blk);
        else vlim_block<T, 0>(A, blk);
    }
}

}  // namespace

namespace {

template <class T>
int vlim_make_args(nicam_ctx c, VlimArgs<T> &A, long &nblk, T *q_h, T *q_h_pl, const T *q, const T *q_pl,
                   const T *d, const T *d_pl, const T *ck, const T *ck_pl, T eps, T big, uint32_t *mask,
                   uint32_t *mask_pl, int ntr)
{
    const Dims &D = c->d;
    if (ntr < 1 || (mask && ntr != 1)) return fail(NICAM_ERR_ARG, "tracer count must be >= 1 (1 with a mask)");
    A.ntr = ntr;
    A.ts = (long)D.nreg();
    A.tps = (long)D.npl();
    A.q_h = q_h;
    A.q = q;
    A.d = d;
    A.ck = ck;
    A.q_h_pl = q_h_pl;
    A.q_pl = q_pl;
    A.d_pl = d_pl;
    A.ck_pl = ck_pl;
    A.gall = D.gall;
    A.kall = D.kall;
    A.lall = D.lall;
    A.gall_pl = D.gall_pl;
    A.have_pl = D.have_pl;
    A.eps = eps;
    A.big = big;
    A.mask = mask;
    A.mask_pl = mask_pl;
    nblk = 0;
    const int nlev = D.kall - 3;  // limited levels kmin+1..kmax
    if (nlev <= 0) return NICAM_OK;
    const long ncol = (long)D.gall * D.lall + (D.have_pl ? (long)D.gall_pl * kLallPl : 0);
    // fields beyond the Infinity Cache (256 MB): q, q_h and its result per tracer, ck's two planes and d
    const bool large = sizeof(T) * (3.0 * ntr + 3.0) * ncol * D.kall > 256e6;
    // Short runs give more independent work-items.  Eight FP64 tracers beyond the cache pay for every run's three
    // extra levels of q and ck: 130x130x42x40 1413 us in runs of 4, 1327 in runs of 8; 66x66x58x40 513 and 484.
    const int dflt = sizeof(T) == 8 && ntr > 1 && large ? LONG_KC : RUN_KC;
    int kc = mask ? LONG_KC : (c->tune.vlim_kchunk > 0 ? c->tune.vlim_kchunk : dflt);
    const bool fixed = kc == RUN_KC || kc == LONG_KC;  // lengths known at compile time
    if (!fixed) kc = std::min(kc, nlev);
    // Other short runs of many tracers: ck and d loaded once for VTB of them outweighs the loads in flight of a
    // work-group each (eight FP32 tracers, 130x130x42x40: runs of 2 806 us against 1027, of 5 741 against 817; of 16
    // 789 against 783; eight FP64 tracers there, runs of 4 1322 against 1408).
    A.multi = ntr > 1 && !mask && kc < LONG_KC && (kc != RUN_KC || dflt != RUN_KC);
    A.ngrp = A.multi ? (ntr + VTB - 1) / VTB : ntr;
    A.kc = kc;
    A.nrun = (nlev + kc - 1) / kc;
    const long ncb = (ncol + BLOCK - 1) / BLOCK, unit = (long)A.nrun * A.ngrp;  // column blocks, work-groups of each
    nblk = ncb * unit;
    // 2^32 columns of four levels are more than the device's memory
    if (nblk > 0x7fffffffL || ncol > 0xffffffffL) return fail(NICAM_ERR_ARG, "grid too large for one launch");
    A.ncol = (unsigned)ncol;
    A.unit = (unsigned)unit;
    // Large: each XCD takes WIN column blocks at a time, next to the other XCDs' (gl7 FP64 154 us against 163 with an
    // eighth of the launch to each XCD, FP32 67 against 71; 130x130x42x40 250 against 270).  In the cache: an eighth of
    // the launch (90x90x97x3 20.2 us against 22.0 in windows, FP32 12.9 against 13.4; 66x66x42x40 FP32 27.7 and 28.7), and of
    // the multi-tracer kernel (18x18x98x40, eight FP64 tracers, runs of 2: 61.8 us against 69).
    const long win = large && !A.multi ? 8 * WIN * unit : nblk / 8 * 8, nwin = win > 0 ? nblk / win : 0;
    A.win = nwin > 0 ? (unsigned)win : 8;
    A.wfull = (unsigned)(nwin * win);
    return NICAM_OK;
}

template <class T>
int launch_vlim_t(nicam_ctx c, T *q_h, T *q_h_pl, const T *q, const T *q_pl, const T *d, const T *d_pl,
                  const T *ck, const T *ck_pl, T eps, T big, uint32_t *mask = nullptr, uint32_t *mask_pl = nullptr,
                  int ntr = 1)
{
    VlimArgs<T> A;
    long nblk = 0;
    const int rc = vlim_make_args(c, A, nblk, q_h, q_h_pl, q, q_pl, d, d_pl, ck, ck_pl, eps, big, mask, mask_pl, ntr);
    if (rc != NICAM_OK || nblk == 0) return rc;
    const dim3 grid((unsigned)nblk), blk(BLOCK);
    if (mask) hipLaunchKernelGGL((vlim_kernel<T, LONG_KC, true>), grid, blk, 0, c->stream, A);
    else if (A.multi) hipLaunchKernelGGL((vlim_kernel<T, 0, false, true>), grid, blk, 0, c->stream, A);
    else if (A.kc == RUN_KC) hipLaunchKernelGGL((vlim_kernel<T, RUN_KC>), grid, blk, 0, c->stream, A);
    else if (A.kc == LONG_KC) hipLaunchKernelGGL((vlim_kernel<T, LONG_KC>), grid, blk, 0, c->stream, A);
    else hipLaunchKernelGGL((vlim_kernel<T, 0>), grid, blk, 0, c->stream, A);
    NICAM_HIP(hipGetLastError());
    return NICAM_OK;
}

}  // namespace

int launch_vlim(nicam_ctx c, double *q_h, double *q_h_pl, const double *q, const double *q_pl,
                const double *d, const double *d_pl, const double *ck, const double *ck_pl)
{
    return launch_vlim_t<double>(c, q_h, q_h_pl, q, q_pl, d, d_pl, ck, ck_pl, c->eps, c->big);
}

int launch_vlim_mask(nicam_ctx c, double *q_h, double *q_h_pl, const double *q, const double *q_pl,
                     const double *d, const double *d_pl, const double *ck, const double *ck_pl, uint32_t *mask,
                     uint32_t *mask_pl)
{
    return launch_vlim_t<double>(c, q_h, q_h_pl, q, q_pl, d, d_pl, ck, ck_pl, c->eps, c->big, mask, mask_pl);
}

int launch_vlim_f32(nicam_ctx c, float *q_h, float *q_h_pl, const float *q, const float *q_pl, const float *d,
                    const float *d_pl, const float *ck, const float *ck_pl)
{
    // the FP32 CONST_EPS and CONST_HUGE (nicam_set_const_f32; by default the -DSINGLE build's)
    return launch_vlim_t<float>(c, q_h, q_h_pl, q, q_pl, d, d_pl, ck, ck_pl, c->eps32, c->big32);
}

}  // namespace nicam

namespace nicam {

int launch_vlim_batch(nicam_ctx c, int ntr, double *q_h, double *q_h_pl, const double *q, const double *q_pl,
                      const double *d, const double *d_pl, const double *ck, const double *ck_pl)
{
    return launch_vlim_t<double>(c, q_h, q_h_pl, q, q_pl, d, d_pl, ck, ck_pl, c->eps, c->big, nullptr, nullptr, ntr);
}

int launch_vlim_batch_f32(nicam_ctx c, int ntr, float *q_h, float *q_h_pl, const float *q, const float *q_pl,
                          const float *d, const float *d_pl, const float *ck, const float *ck_pl)
{
    return launch_vlim_t<float>(c, q_h, q_h_pl, q, q_pl, d, d_pl, ck, ck_pl, c->eps32, c->big32, nullptr, nullptr,
                                ntr);
}

}  // namespace nicam

namespace nicam {

int launch_vlim_group_f32(const nicam_ctx *cs, int n, int ntr, const nicam_tracer_step_f32 *g, hipStream_t stream)
{
    if (n < 1 || n > kMaxGroup) return fail(NICAM_ERR_ARG, "a group holds 1..8 grids");
    VlimGroup<float> G;
    G.n = n;
    G.off[0] = 0;
    for (int i = 0; i < n; ++i) {
        const nicam_tracer_step_f32 &p = g[i];
        long nb = 0;
        const int rc = vlim_make_args<float>(cs[i], G.a[i], nb, p.q_h, p.q_h_pl, p.qv, p.qv_pl, p.dv, p.dv_pl, p.ck,
                                             p.ck_pl, cs[i]->eps32, cs[i]->big32, nullptr, nullptr, ntr);
        if (rc != NICAM_OK) return rc;
        if ((long)G.off[i] + nb > 0x7fffffffL) return fail(NICAM_ERR_ARG, "group too large for one launch");
        G.off[i + 1] = G.off[i] + (int)nb;
    }
    if (G.off[n] == 0) return NICAM_OK;
    bool tuned = false;
    for (int i = 0; i < n; ++i) tuned |= G.off[i + 1] > G.off[i] && (G.a[i].kc != RUN_KC || G.a[i].multi);
    hipLaunchKernelGGL((tuned ? vlim_group_kernel<float, true> : vlim_group_kernel<float, false>),
                       dim3((unsigned)G.off[n]), dim3(BLOCK), 0, stream, G);
    NICAM_HIP(hipGetLastError());
    return NICAM_OK;
}

}  // namespace nicam
