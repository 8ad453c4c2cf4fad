// lanes.hpp -- resumable per-lane programs shared by the one-shot kernels and
// the batched engine.
//
// Every program advances one grid point over a range of "ticks" [g0, g1) of
// its job and can stop anywhere: the one-shot kernels run [0, total) in one
// launch, the engine runs a few thousand ticks per launch and parks the lane
// state in HBM in between.  Both paths execute the same arithmetic in the
// same order, so a point's result does not depend on how its work was split.
#pragma once

#include <hip/hip_runtime.h>

#include "lle.hpp"
#include "peaks.hpp"
#include "sweep.hpp"
#include "systems.hpp"

namespace chaos {

// ---------------------------------------------------------------------------
// shared checks (Bifurcation/src/bifurcationCUDA.cu:445-466,
// Basins/src/basinsCUDA.cu:350-376)
// ---------------------------------------------------------------------------

__device__ __forceinline__ bool diverged_exact(double v, double M, int check)
{
    if (check == CHK_BIF_REF) {
        if (v != v || v == v + 1.0) return true;
        if (M != 0 && (double)fabsf((float)v) > M) return true;
    } else if (check == CHK_BASINS_REF) {
        if (isnan(v) || isinf(v)) return true;
        if (M != 0 && (double)fabsf((float)v) > M) return true;
    } else {
        if (!isfinite(v)) return true;
        if (M != 0 && fabs(v) > M) return true;
    }
    return false;
}

__device__ __forceinline__ bool fixed_point(double t, int check)
{
    if (check == CHK_BIF_REF) return (double)sqrtf(fabsf((float)t)) < 1e-9;
    if (check == CHK_BASINS_REF) return sqrt(fabs(t)) < 1e-9;
    return sqrt(t) < 1e-9;
}

template <int NX>
__device__ __forceinline__ double step_delta2(const double* X, const double* xp)
{
    double t = 0;
#pragma unroll
    for (int j = 0; j < NX; ++j) t += ((X[j] - xp[j]) * (X[j] - xp[j]));
    return t;
}

// X[wv] for a compile-time wv (WVT >= 0) or a run-time one (WVT < 0).
template <int NX, int WVT>
__device__ __forceinline__ double pick(const double* X, int wv)
{
    if constexpr (WVT >= 0) {
        return X[WVT];
    } else {
        double v = X[0];
#pragma unroll
        for (int k = 1; k < NX; ++k) v = (wv == k) ? X[k] : v;
        return v;
    }
}

// n steps of one trajectory, four to a trip: the loop's scalar instructions
// and taken branch are issue slots to a lone wavefront (LLE preview of 17^2
// points 403 -> 384 us with the pairs of LleProg::ticks).
template <class Sy>
__host__ __device__ __forceinline__ void plain_steps(double* X, const double* a, const StepConst& c, long long n)
{
    for (; n >= 4; n -= 4) {
        Sy::step(X, a, c);
        Sy::step(X, a, c);
        Sy::step(X, a, c);
        Sy::step(X, a, c);
    }
    for (; n > 0; --n) Sy::step(X, a, c);
}

// Lane state parked in HBM between engine launches (SoA, k-major).
struct LaneStore {
    double* d;     // [nd][np]
    int* i;        // [ni][np]
    long long np;  // lanes (multiple of 64)
};

// ---------------------------------------------------------------------------
// LLE: Benettin with two trajectories (LLE/src/LLECUDA.cu:56-166)
// ticks [0, S): transient on X; tick S starts with the perturbation; ticks
// [S, S + W*NTp) step X and Xp once each, renormalising after every NTp.
// Host-callable as well, so the tick-split invariance and the progress guard
// are checked on the CPU.
// ---------------------------------------------------------------------------
template <int SYS>
struct LleProg {
    using Sy = System<SYS>;
    static constexpr int NX = Sy::NX, NA = Sy::NA;
    static constexpr int ND = 2 * NX + 1;   // parked state: X, Xp, sum
    static constexpr int NDIR = NX;         // engine: eps * direction, after the parked state
    double X[NX], Xp[NX], a[NA], sum;

    __host__ __device__ __forceinline__ static long long total(const LleArgs& p)
    {
        return (long long)p.S + (long long)p.W * p.NTp;
    }

    __host__ __device__ __forceinline__ void params(const LleArgs& p, int i, int j)
    {
        build_params<NA>(a, p.values, p.idxA, grid_value(i, p.nPts, p.rA0, p.rA1), p.idxB,
                         grid_value(j, p.nPts, p.rB0, p.rB1));
    }
    __host__ __device__ __forceinline__ void init(const LleArgs& p)
    {
#pragma unroll
        for (int k = 0; k < NX; ++k) {
            X[k] = p.ic[k];
            Xp[k] = 0.0;
        }
        sum = 0.0;
    }
    // The perturbation added at tick S: eps * v with v the point's seeded
    // unit vector (LLE/src/LLECUDA.cu:88-102 draws it from curand instead).
    __host__ __device__ __forceinline__ static void offset(const LleArgs& p, long long point, double* d)
    {
        double v[NX];
        unit_vector<NX>(p.seed, point, v);
#pragma unroll
        for (int k = 0; k < NX; ++k) d[k] = p.eps * v[k];
    }

    // Advance over ticks [g0, g1).  The perturbation at tick S comes from
    // offset() (DIR_STORED false) or is read from dir[k * dstride] (the
    // engine stores it when the job starts, which keeps the unit-vector code
    // out of its tile loop).  Returns false without stepping when the range
    // cannot make progress -- NTp < 1 would leave every window empty and the
    // window loop would never advance -- so a caller handed a malformed job
    // reports it instead of spinning.
    template <bool DIR_STORED = false>
    __host__ __device__ __forceinline__ bool ticks(const LleArgs& p, long long point, long long g0, long long g1,
                                                   const double* dir = nullptr, long long dstride = 0)
    {
        if (p.NTp < 1 || p.S < 0 || g0 < 0 || g1 < g0) return false;
        long long g = g0;
        if (g < p.S) {
            const long long e = g1 < p.S ? g1 : p.S;
            plain_steps<Sy>(X, a, p.sc, e - g);
            g = e;
        }
        if (g == p.S && g < g1) {
            double d[NX];
            if (DIR_STORED) {
#pragma unroll
                for (int k = 0; k < NX; ++k) d[k] = dir[k * dstride];
            } else {
                offset(p, point, d);
            }
#pragma unroll
            for (int k = 0; k < NX; ++k) Xp[k] = X[k] + d[k];
        }
        int local = g < g1 ? (int)((g - p.S) % p.NTp) : 0;  // position in the first window
        while (g < g1) {
            const long long left = g1 - g;
            const int n = (p.NTp - local) < left ? (p.NTp - local) : (int)left;  // >= 1: local < NTp
            int s = 0;
            for (; s + 1 < n; s += 2) {
                Sy::step(X, a, p.sc);
                Sy::step(Xp, a, p.sc);
                Sy::step(X, a, p.sc);
                Sy::step(Xp, a, p.sc);
            }
            if (s < n) {
                Sy::step(X, a, p.sc);
                Sy::step(Xp, a, p.sc);
            }
            g += n;
            const bool window_end = local + n == p.NTp;
            local = 0;
            if (window_end) {
                double d2 = 0.0;
#pragma unroll
                for (int l = 0; l < NX; ++l) {
                    const double diff = X[l] - Xp[l];
                    d2 = d2 + diff * diff;
                }
                const double dist = sqrt(d2) / p.eps;
                sum = sum + log(dist);
#pragma unroll
                for (int l = 0; l < NX; ++l) Xp[l] = X[l] - ((X[l] - Xp[l]) / dist);
            }
        }
        return true;
    }
    __host__ __device__ __forceinline__ double result(const LleArgs& p) const { return sum / p.tMax; }

    __host__ __device__ __forceinline__ void load(const LaneStore& L, long long q)
    {
#pragma unroll
        for (int k = 0; k < NX; ++k) {
            X[k] = L.d[k * L.np + q];
            Xp[k] = L.d[(NX + k) * L.np + q];
        }
        sum = L.d[2 * NX * L.np + q];
    }
    __host__ __device__ __forceinline__ void store(const LaneStore& L, long long q) const
    {
#pragma unroll
        for (int k = 0; k < NX; ++k) {
            L.d[k * L.np + q] = X[k];
            L.d[(NX + k) * L.np + q] = Xp[k];
        }
        L.d[2 * NX * L.np + q] = sum;
    }
    // Stored perturbation of lane q (engine): dir[k * np] for k < NX.
    __host__ __device__ __forceinline__ static const double* dir_of(const LaneStore& L, long long q)
    {
        return L.d + ND * L.np + q;
    }
};

// ---------------------------------------------------------------------------
// Sweep (Bifurcation / Basins): ticks [0, S) transient, [S, S+B) samples
// (each sample = pre steps).  Kernels and engine must keep all 64 lanes of
// a wave in the loop (append_peaks is a wave-level operation).
// ---------------------------------------------------------------------------
template <int SYS, int KIND>
struct SweepProg {
    using Sy = System<SYS>;
    static constexpr int NX = Sy::NX, NA = Sy::NA;
    static constexpr int ND = NX + 7;  // X, p, first, last, s0, s1, sx, sz
    static constexpr int NI = 4;       // pstart, cnt, prev_t, bits
    double X[NX], a[NA];
    static constexpr bool BIF = stores_peaks(KIND);
    // peak times: the intervals of the bifurcation lists and of the
    // reference basins features; the other kinds use peak values only
    static constexpr bool DET_TIMES = KIND == KIND_BIF || KIND == KIND_BASINS_REF;
    WavePeakDetector<DET_TIMES> det;
    int cnt, prev_t;
    unsigned long long alive;  // wave mask of the lanes still integrating
    bool fixed;
    double s0, s1, sx, sz, first, last;

    __device__ __forceinline__ static long long total(const SweepArgs& A) { return (long long)A.S + A.B; }

    __device__ __forceinline__ static void grid(const SweepArgs& A, long long pq, double& g0, double& g1)
    {
        const int i = (int)(pq % A.nPts);
        const int j = A.dims == 2 ? (int)(pq / A.nPts) : 0;
        g0 = grid_value(i, A.nPts, A.r[0], A.r[1]);
        g1 = A.dims == 2 ? grid_value(j, A.nPts, A.r[2], A.r[3]) : 0.0;
    }
    // Parameter vector of point pq.
    __device__ __forceinline__ void params(const SweepArgs& A, long long pq)
    {
        if (BIF && !A.ic_sweep) {
            // swept entries of the parameter vector (bifurcationCUDA.cu:282-284)
            double g0, g1;
            grid(A, pq, g0, g1);
            build_params<NA>(a, A.values, A.idx0, g0, A.idx1, g1);
        } else {
#pragma unroll
            for (int k = 0; k < NA; ++k) a[k] = A.values[k];
        }
    }
    // Parameters and the initial lane state of point pq.
    __device__ __forceinline__ void init(const SweepArgs& A, long long pq, bool in_range)
    {
        params(A, pq);
        if (BIF && !A.ic_sweep) {
#pragma unroll
            for (int k = 0; k < NX; ++k) X[k] = A.ic[k];
        } else {
            // swept entries of the initial condition (basinsCUDA.cu:253-262,
            // debri/cudaLibrary.cu:1022-1062)
            double g0, g1;
            grid(A, pq, g0, g1);
#pragma unroll
            for (int k = 0; k < NX; ++k) X[k] = (k == A.idx0) ? g0 : ((k == A.idx1) ? g1 : A.ic[k]);
        }
        det.reset();
        cnt = 0;
        prev_t = 0;
        alive = wave_mask(in_range);
        fixed = false;
        s0 = s1 = sx = sz = first = last = 0.0;
    }

    // Divergence test of the recorded variable.  The band test |v| < L is
    // exact-safe (no lane inside it can fail the exact test); the exact test
    // runs only when some lane of the wave is outside it, behind a uniform
    // branch.  Callers keep the wave's control flow uniform.
    template <int WVT>
    __device__ __forceinline__ void check(const SweepArgs& A, int wv)
    {
        const double v = pick<NX, WVT>(X, wv);
        const unsigned long long out = wave_mask(!(fabs(v) < A.L)) & alive;
        if (out) alive &= ~wave_mask(lane_bit(out) && diverged_exact(v, A.maxValue, A.check));
    }

    // n steps, each followed by the divergence test.  Pairs of steps share one
    // band test -- the larger magnitude of the two -- and its mask is branched
    // on after the next pair's steps, as in body().  A NaN stays NaN, so one
    // that v_max drops from its pair is seen with the next pair or at the end.
    template <int WVT>
    __device__ __forceinline__ void checked_steps(const SweepArgs& A, int wv, long long n)
    {
        if (n <= 0) return;
        double v0 = 0.0, v1 = 0.0, m = -1.0;  // no pair yet: inside any band (L >= 0)
        auto exact = [&](unsigned long long out) {
            alive &= ~wave_mask(lane_bit(out) && (diverged_exact(v0, A.maxValue, A.check) ||
                                                  diverged_exact(v1, A.maxValue, A.check)));
        };
        auto pair = [&] {
            const unsigned long long out = wave_mask(!(m < A.L)) & alive;
            Sy::step(X, a, A.sc);
            const double w0 = pick<NX, WVT>(X, wv);
            Sy::step(X, a, A.sc);
            const double w1 = pick<NX, WVT>(X, wv);
            pin_state();
            if (__builtin_expect(out != 0ull, 0)) exact(out);
            v0 = w0;
            v1 = w1;
            m = fmax(fabs(w0), fabs(w1));
        };
        for (; n >= 4; n -= 4) {
            pair();
            pair();
        }
        const unsigned long long out = wave_mask(!(m < A.L)) & alive;
        if (out) exact(out);
        for (; n > 0; --n) {
            Sy::step(X, a, A.sc);
            check<WVT>(A, wv);
        }
        // a NaN of the last pair's second step when no step followed it
        check<WVT>(A, wv);
    }

    // The kind's work for the lanes em with a peak (value pv, time pt); em is
    // wave-uniform and not empty.
    __device__ __forceinline__ void on_peaks(const SweepArgs& A, WaveCursor& cur, int wave, unsigned long long em,
                                             double pv, int pt)
    {
        const bool e = lane_bit(em);
        if (BIF) {
            append_peaks(A.pool, cur, wave, em, pv, pt, cnt);
            if (e) ++cnt;
        } else if (KIND == KIND_BASINS_REF) {
            // running sums of the kept peaks and intervals
            // (avgPeakFinderCUDA, basinsCUDA.cu:841-861)
            if (e) {
                if (cnt >= 1) {
                    s0 = s0 + pv;
                    s1 = s1 + (double)(pt - prev_t) * A.hp;
                }
                prev_t = pt;
                ++cnt;
            }
        } else {
            if (e) {
                if (cnt >= 1) {
                    s0 = s0 + pv;
                    s1 = fma(pv, pv, s1);
                }
                ++cnt;
            }
        }
    }

    // One recorded sample t at the ends of the record (t < 2, t = B - 1):
    // peak detection on the sample, the kind's per-peak work, then preScaller
    // steps and the divergence check.
    template <int WVT>
    __device__ __forceinline__ void sample(const SweepArgs& A, int wv, WaveCursor& cur, int wave, int t)
    {
        const double v = pick<NX, WVT>(X, wv);
        if (t == 0) first = v;
        if (KIND == KIND_BASINS_CFG) {
            sx = sx + X[0];
            sz = sz + X[NX - 1];
        }
        double pv = 0.0;
        int pt = 0;
        const unsigned long long em = det.feed(t, v, pv, pt) & alive;
        if (em) on_peaks(A, cur, wave, em, pv, pt);
        double xp[NX];
#pragma unroll
        for (int k = 0; k < NX; ++k) xp[k] = X[k];
        for (int r = 0; r < A.pre; ++r) Sy::step(X, a, A.sc);
        check<WVT>(A, wv);
        if (t == A.B - 1) {
            last = v;
            fixed = lane_bit(alive) && fixed_point(step_delta2<NX>(X, xp), A.check);
        }
    }

    // The value sampled now, added to the sums that every sample feeds.
    template <int WVT>
    __device__ __forceinline__ double take(int wv)
    {
        if (KIND == KIND_BASINS_CFG) {
            sx = sx + X[0];
            sz = sz + X[NX - 1];
        }
        return pick<NX, WVT>(X, wv);
    }

    // Sample t = value v with its masks: divergence first (a value is tested
    // when it is sampled, which is after the step that made it), then its
    // peaks.
    __device__ __forceinline__ void settle(const SweepArgs& A, WaveCursor& cur, int wave, int t, double v,
                                           unsigned long long c2, unsigned long long tiny, unsigned long long out)
    {
        out &= alive;
        if (out) alive &= ~wave_mask(lane_bit(out) && diverged_exact(v, A.maxValue, A.check));
        double pv = 0.0;
        int pt = 0;
        const unsigned long long em = det.decide(t - 1, v, c2, tiny, pv, pt) & alive;
        if (em) on_peaks(A, cur, wave, em, pv, pt);
    }

    // Recorded samples t, t + 1, ... inside the record (2 <= t, t + 1 < end),
    // two to a trip; returns the first sample not taken.
    //
    // A peak needs a rising sample followed by a fall (up & c2 & ~tiny) and
    // nothing more unless a plateau is open or begins or an index is skipped;
    // such a peak only joins its lane's pending slot (to_slots).  The slots
    // are emptied together -- one append, or one masked update of the sums --
    // when a lane with a full slot peaks again: lanes peak every 30 to 600
    // samples but some lane of the 64 nearly every sample, so that work runs
    // once for tens of peaks.  A pair with anything else to it -- a plateau, a
    // value outside the divergence band, a second peak -- goes sample by sample
    // (settle).  Its mask is branched on after the second sample's steps, which
    // do not depend on it (a compare that is branched on at once stalls a lone
    // wavefront for the time of about six instructions), and the pairs that do
    // not need it run in a loop of their own, so that the state of the detector
    // and of the peak store is not merged back on every trip.
    //
    // A lone wavefront pays an issue slot per instruction of any kind, so fewer
    // scalar instructions and branches a sample count there: the Rossler diagram
    // of 1000 points 28.9 -> 21.1 ms a call with the pairs (20.6 with the slots),
    // BASINS basins of 200^2 73.5 -> 57.9 ms.  The pending slots: Lorenz peak map 88.8 -> 86.2 ms at
    // 1024^2 points and (sweep alone) 8.1 -> 6.9 ms at 200^2, basins 93.1 ->
    // 91.6 ms at 1024^2; full grids are bound by FP64 issue.  Chameleon's long
    // steps leave them nothing to gain (31.2 -> 31.3 ms at 300^2).
    template <int WVT, bool PRE1>
    __device__ __forceinline__ int body(const SweepArgs& A, int wv, WaveCursor& cur, int wave, int t, int end)
    {
        auto advance = [&] {
            if (PRE1) Sy::step(X, a, A.sc);
            else
                for (int r = 0; r < A.pre; ++r) Sy::step(X, a, A.sc);
        };
        unsigned long long busy = det.m.busy() & alive;
        double p = det.p;
        unsigned long long up = det.m.up;
        unsigned long long pend = 0ull;  // lanes with a full slot (value pend_v, time pend_t)
        double pend_v = 0.0;
        int pend_t = 0;
        while (t + 1 < end) {
            double v0, v1;
            SamplePair m;
            do {
                det.p = p;  // the history before the pair
                det.m.up = up;
                v0 = take<WVT>(wv);
                const double d0 = v0 - p;
                m.c0 = wave_mask(d0 <= 0.0);
                m.y0 = wave_mask(fabs(d0) <= 1e-13);
                m.o0 = wave_mask(!(fabs(v0) < A.L));
                advance();
                v1 = take<WVT>(wv);
                const double d1 = v1 - v0;
                m.c1 = wave_mask(d1 <= 0.0);
                m.y1 = wave_mask(fabs(d1) <= 1e-13);
                m.o1 = wave_mask(!(fabs(v1) < A.L));
                const bool events = m.events(up, busy, alive);
                advance();
                pin_state();
                t += 2;
                if (events) {
                    unsigned long long e0, e1;
                    m.peaks(alive, pend, e0, e1);
                    if (m.other) break;
                    // the peaks are the samples t - 3 and t - 2 now
                    to_slots(pend_v, pend_t, p, t - 3, e0, v0, t - 2, e1);
                    pend |= e0 | e1;
                }
                p = v1;
                up = ~(m.c1 | m.y1);
            } while (t + 1 < end);
            if (m.other) {
                if (pend) on_peaks(A, cur, wave, pend, pend_v, pend_t);
                pend = 0ull;
                settle(A, cur, wave, t - 2, v0, m.c0, m.y0, m.o0);
                settle(A, cur, wave, t - 1, v1, m.c1, m.y1, m.o1);
                busy = det.m.busy() & alive;
                p = det.p;
                up = det.m.up;
            }
        }
        if (pend) on_peaks(A, cur, wave, pend, pend_v, pend_t);
        det.p = p;
        det.m.up = up;
        check<WVT>(A, wv);  // the last pair's second step
        return t;
    }

    // A pair's peaks to their lanes' pending slots: value va and time ta on lanes
    // m, vb and tb on lanes n; m and n are disjoint and, as ballots, hold active
    // lanes only.  Values alone are moved under the masks in exec, which then
    // gets back the lanes it had; with times the selects cost no more than that
    // (1-D Rossler diagram 20.8 -> 20.6 ms, Chameleon peak map of 300^2 points
    // 31.3 ms both ways; values only, 1024^2 Lorenz map: selects 1 to 2 % slower).
    __device__ __forceinline__ static void to_slots(double& v, int& t, double va, int ta, unsigned long long m,
                                                    double vb, int tb, unsigned long long n)
    {
        if (DET_TIMES) {
            v = lane_bit(m) ? va : v;
            v = lane_bit(n) ? vb : v;
            t = lane_bit(m) ? ta : t;
            t = lane_bit(n) ? tb : t;
        } else {
            unsigned long long active;
            asm volatile("s_mov_b64 %1, exec\n\ts_mov_b64 exec, %4\n\tv_mov_b64 %0, %2\n\ts_mov_b64 exec, %5\n\t"
                         "v_mov_b64 %0, %3\n\ts_mov_b64 exec, %1"
                         : "+&v"(v), "=&s"(active)
                         : "v"(va), "v"(vb), "s"(m), "s"(n));
        }
    }

    // Keeps the steps before this point ahead of the branch that follows.
    __device__ __forceinline__ void pin_state()
    {
#pragma unroll
        for (int k = 0; k < NX; ++k) asm volatile("" : "+v"(X[k]));
    }

    template <int WVT>
    __device__ __forceinline__ void ticks(const SweepArgs& A, int wv, WaveCursor& cur, int wave, long long g0,
                                          long long g1)
    {
        long long g = g0;
        // ---- transient ----
        if (BIF && A.legacy_transient) {
            // legacy IC sweeps (debri/cudaLibrary.cu:1063-1070): the transient
            // tests X[0] for NaN/inf only (maxValue 0) and a fixed point at its
            // end is still recorded
            if (g < A.S) {
                const long long e = g1 < A.S ? g1 : A.S;
                for (long long s = g; s < e; ++s) {
                    Sy::step(X, a, A.sc);
                    alive &= ~wave_mask(!isfinite(X[0]));
                }
                g = e;
            }
        } else if (BIF) {
            // checked every step; a transient that ends diverged or at a
            // fixed point is not recorded and reports 0 (bifurcationCUDA.cu:334-342)
            if (g < A.S - 1) {
                const long long e = g1 < A.S - 1 ? g1 : A.S - 1;
                checked_steps<WVT>(A, wv, e - g);
                g = e;
            }
            if (g == A.S - 1 && g < g1) {
                double xp[NX];
#pragma unroll
                for (int k = 0; k < NX; ++k) xp[k] = X[k];
                Sy::step(X, a, A.sc);
                check<WVT>(A, wv);
                alive &= ~wave_mask(fixed_point(step_delta2<NX>(X, xp), A.check));
                ++g;
            }
        } else if (g < A.S) {
            // no checks during the Basins transient (basinsCUDA.cu:264-271)
            const long long e = g1 < A.S ? g1 : A.S;
            plain_steps<Sy>(X, a, A.sc, e - g);
            g = e;
        }
        // ---- record ----
        // head (t < 2: detector warm-up, first sample), body, tail (t = B-1)
        const int B = A.B;
        int t = (int)(g - A.S);
        const int te = (int)(g1 - A.S);
        const int body_end = te < B - 1 ? te : B - 1;
        for (; t < te && t < 2; ++t) sample<WVT>(A, wv, cur, wave, t);
        if (t + 1 < body_end)
            t = A.pre == 1 ? body<WVT, true>(A, wv, cur, wave, t, body_end)
                           : body<WVT, false>(A, wv, cur, wave, t, body_end);
        for (; t < te; ++t) sample<WVT>(A, wv, cur, wave, t);
    }

    __device__ __forceinline__ void finish(const SweepArgs& A, long long q) const
    {
        const int flag = this->flag();
        if (A.flags) A.flags[q] = flag;
        if (BIF) {
            A.counts[q] = cnt;
            A.first[q] = first;
        } else if (KIND == KIND_BASINS_REF) {
            double f0, f1;
            if (flag == 0) {
                f0 = 999;
                f1 = 999;
            } else if (flag == -1) {
                f0 = last;
                f1 = -1.0;
            } else {
                const int P = cnt > 1 ? cnt - 1 : 0;
                if (P <= 0) {
                    f0 = 1000;
                    f1 = 1000;
                } else {
                    f0 = s0 / P;
                    f1 = s1 / P;
                }
            }
            A.f0[q] = f0;
            A.f1[q] = f1;
            if (A.f2) A.f2[q] = 0.0;
            if (A.counts) A.counts[q] = cnt;
        } else {
            double f[3];
            config_features(A, flag, f);
            A.f0[q] = f[0];
            A.f1[q] = f[1];
            A.f2[q] = f[2];
            if (A.counts) A.counts[q] = cnt;
        }
    }

    // Lane flag (1 alive, -1 fixed point, 0 diverged).
    __device__ __forceinline__ int flag() const { return lane_bit(alive) ? (fixed ? -1 : 1) : 0; }

    // CONFIG features (mean X[0], mean X[NX-1], population std of the kept
    // peaks), all 0 for a diverged lane.
    __device__ __forceinline__ void config_features(const SweepArgs& A, int flag, double* f) const
    {
        const int B = A.B;
        f[0] = f[1] = f[2] = 0.0;
        if (flag != 0) {
            f[0] = sx / B;
            f[1] = sz / B;
            const int n = cnt > 1 ? cnt - 1 : 0;
            if (n >= 2) {
                const double m = s0 / n;
                const double var = s1 / n - m * m;
                f[2] = var > 0 ? sqrt(var) : 0.0;
            }
        }
    }

    // Parked state.  A kind parks what it uses: anything more stays in registers
    // across the ticks between a load and the next store, and the engine's kernels
    // have none to spare (all of it: 2 to 7 VGPRs spilled in the basins kernels).
    // `last` and `fixed` are set by the record's last sample, after which nothing
    // is parked.
    static constexpr bool FIRST = BIF, SUMS = !BIF, MEANS = KIND == KIND_BASINS_CFG, LAST_T = KIND == KIND_BASINS_REF;
    __device__ __forceinline__ void load(const LaneStore& L, long long q)
    {
#pragma unroll
        for (int k = 0; k < NX; ++k) X[k] = L.d[k * L.np + q];
        const double* d = L.d + NX * L.np + q;
        det.p = d[0];
        first = FIRST ? d[L.np] : 0.0;
        last = 0.0;
        s0 = SUMS ? d[3 * L.np] : 0.0;
        s1 = SUMS ? d[4 * L.np] : 0.0;
        sx = MEANS ? d[5 * L.np] : 0.0;
        sz = MEANS ? d[6 * L.np] : 0.0;
        det.pstart = DET_TIMES ? L.i[q] : 0;
        cnt = L.i[L.np + q];
        prev_t = LAST_T ? L.i[2 * L.np + q] : 0;
        const int bits = L.i[3 * L.np + q];
        alive = wave_mask(bits & 1);
        fixed = false;
        det.m.plat = wave_mask(bits & 4);
        det.m.skip = wave_mask(bits & 8);
        det.m.up = wave_mask(bits & 16);
    }
    __device__ __forceinline__ void store(const LaneStore& L, long long q) const
    {
#pragma unroll
        for (int k = 0; k < NX; ++k) L.d[k * L.np + q] = X[k];
        double* d = L.d + NX * L.np + q;
        d[0] = det.p;
        if (FIRST) d[L.np] = first;
        if (SUMS) {
            d[3 * L.np] = s0;
            d[4 * L.np] = s1;
        }
        if (MEANS) {
            d[5 * L.np] = sx;
            d[6 * L.np] = sz;
        }
        if (DET_TIMES) L.i[q] = det.pstart;
        L.i[L.np + q] = cnt;
        if (LAST_T) L.i[2 * L.np + q] = prev_t;
        L.i[3 * L.np + q] =
            (lane_bit(alive) ? 1 : 0) | (lane_bit(det.m.plat) ? 4 : 0) |
            (lane_bit(det.m.skip) ? 8 : 0) | (lane_bit(det.m.up) ? 16 : 0);
    }
};

// Where a sweep group's state is parked between calls.
struct SweepPark {
    LaneStore st;
    WaveCursor* cursors;  // per group, for the kinds that store peaks
    long long total;      // ticks of the whole run
};

// Ticks [g0, g1) of one 64-point group of a sweep whose lane state is parked
// between calls; writes the outputs when g1 is the last tick.  park() gives the
// SweepPark and is called anew after the ticks, so that it need not stay in
// registers across them.  All 64 lanes of the wave call it.
template <int SYS, int KIND, int WV, class Park, class G>
__device__ __forceinline__ void sweep_group_ticks(const SweepArgs& A, const Park& park, const G& group_of, int lane,
                                                  long long g0, long long g1)
{
    SweepProg<SYS, KIND> L;
    WaveCursor cur{A.pool.nchunks, kChunk};
    const long long group = group_of();
    {
        const SweepPark P = park();
        const long long q = group * 64 + lane;
        const bool in_range = q < A.n_points;
        const long long pq = A.p0 + (in_range ? q : 0);
        if (g0 == 0) {
            L.init(A, pq, in_range);
        } else {
            L.params(A, pq);
            L.load(P.st, q);
            if (stores_peaks(KIND)) {
                const WaveCursor c = P.cursors[group];
                cur.chunk = __builtin_amdgcn_readfirstlane(c.chunk);
                cur.fill = __builtin_amdgcn_readfirstlane(c.fill);
            }
        }
    }
    const bool last = g1 == park().total;
    L.template ticks<WV>(A, WV, cur, (int)group, g0, g1);
    const long long after = group_of();
    const long long q = after * 64 + lane;
    if (last) {
        if (stores_peaks(KIND)) close_chunk(A.pool, cur);
        if (q < A.n_points) L.finish(A, q);
    } else {
        const SweepPark P = park();
        L.store(P.st, q);
        if (stores_peaks(KIND) && lane == 0) P.cursors[after] = cur;
    }
}

}  // namespace chaos
