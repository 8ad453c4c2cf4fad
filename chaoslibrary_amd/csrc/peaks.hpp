// peaks.hpp -- online peak detection over a lane's sample stream, plus the
// wavefront-compacted peak store.
//
// The detector replays the reference peakFinder
// (Bifurcation/src/bifurcationCUDA.cu:469-514, same text in
// Basins/src/basinsCUDA.cu:382-440) one sample at a time, in registers,
// instead of re-reading a stored trajectory:
//   candidate at i:   d[i]-d[i-1] > 1e-13  &&  d[i] >= d[i+1]
//   plateau scan j:   d[j] < d[j+1]          -> reject, next candidate i = j+2
//                     d[j]-d[j+1] > 1e-13    -> peak (d[j], trunc((i+j)/2)),
//                                               next candidate i = j+2
// (the reference's i = j+1 followed by the loop's ++i skips index j+1).
// All comparisons are on exact differences of adjacent samples:
// d[c]-d[c+1] == -(d[c+1]-d[c]) and d[c] >= d[c+1] <=> d[c+1]-d[c] <= 0 for
// finite samples, so one subtraction per sample feeds all three tests.
#pragma once

#include <hip/hip_runtime.h>

namespace chaos {

struct PeakDetector {
    double p;      // last sample d[t-1]
    double dn;     // d[t-1] - d[t-2]
    int pstart;    // plateau start index
    bool plat;     // scanning a plateau
    bool skip;     // next index is not a candidate

    __device__ __forceinline__ void reset()
    {
        p = 0.0;
        dn = 0.0;
        pstart = 0;
        plat = false;
        skip = false;
    }

    // Feed sample d[t] = cur (t >= 0).  For t >= 2 the index c = t-1 is
    // examined; on a peak, returns true with its value (d[c]) and time.
    __device__ __forceinline__ bool feed(int t, double cur, double& val, int& time)
    {
        const double dnx = cur - p;  // d[c+1] - d[c]
        bool emit = false;
        if (t >= 2) {
            const int c = t - 1;
            const bool c1 = dn > 1e-13;     // d[c] - d[c-1] > 1e-13
            const bool c2 = dnx <= 0.0;     // d[c] >= d[c+1]
            const bool c3 = dnx < -1e-13;   // d[c] - d[c+1] > 1e-13
            if (plat) {
                if (!c2) {
                    plat = false;
                    skip = true;
                } else if (c3) {
                    emit = true;
                    val = p;
                    time = (pstart + c) >> 1;
                    plat = false;
                    skip = true;
                }
            } else if (skip) {
                skip = false;
            } else if (c1 && c2) {
                if (c3) {
                    emit = true;
                    val = p;
                    time = c;
                    skip = true;
                } else {
                    plat = true;
                    pstart = c;
                }
            }
        }
        dn = dnx;
        p = cur;
        return emit;
    }
};

// Lane mask <-> lane predicate: a compare written straight into a wave mask,
// and a wave mask used as a lane predicate, both without VALU work.  Every
// lane of the wave must be active where a mask is formed.
__device__ __forceinline__ unsigned long long wave_mask(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ bool lane_bit(unsigned long long m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// PeakDetector's state for a whole wave as lane masks (SGPRs).  With
// dnx = d[t] - d[t-1], two compares a sample give all three tests: c2 =
// (dnx <= 0) and tiny = (|dnx| <= 1e-13), for d[c] - d[c+1] > 1e-13 is
// c2 & ~tiny, and the rising test of the next sample, dn > 1e-13, is
// ~(c2 | tiny).  (Of a NaN difference both compares are false; the next
// difference is NaN too, so no candidate comes of it.)  The state machine runs
// on the scalar unit -- a per-lane bool state costs two VALU instructions per
// sample to form each ballot.
struct PeakMasks {
    unsigned long long up;    // lanes with d[t-1] - d[t-2] > 1e-13
    unsigned long long plat;  // lanes scanning a plateau
    unsigned long long skip;  // lanes whose next index is not a candidate

    struct Found {
        unsigned long long emit;    // lanes with a peak at c = t - 1
        unsigned long long closed;  // of them, those that end a plateau
        unsigned long long opened;  // lanes that begin a plateau at c
    };

    // PeakDetector::feed for every lane (t >= 2).  skip is kept only
    // where it matters, after a plateau that rose again: after a peak
    // dnx < -1e-13, so the next index fails its own rising test.  So with
    // no plateau open and nothing skipped (quiet), a sample finds no peak and
    // opens no plateau unless up & c2.
    __host__ __device__ __forceinline__ Found step(unsigned long long c2, unsigned long long tiny)
    {
        const unsigned long long c3 = c2 & ~tiny;
        const unsigned long long cand = ~plat & ~skip & up & c2;
        const unsigned long long act = plat | cand;
        const Found f = {act & c3, plat & c3, cand & ~c3};
        skip = plat & ~c2;
        plat = act & c2 & tiny;
        up = ~(c2 | tiny);
        return f;
    }
    __host__ __device__ __forceinline__ unsigned long long busy() const { return plat | skip; }
};

// Two samples of a wave, one after the other, by their lane masks: c (not above
// the sample before), y (within 1e-13 of it), o (outside the divergence band).
// Says whether the pair is plain -- its peaks, if any, only join their lanes'
// pending slots -- or goes sample by sample.  Lanes that no longer integrate
// cannot make it do so: what their detector holds is never used.
struct SamplePair {
    unsigned long long c0, y0, o0, c1, y1, o1;
    unsigned long long f0, f1;  // rising samples followed by one that does not rise
    unsigned long long other;   // lanes for which the pair goes sample by sample

    // `up` and `busy` are PeakMasks' before the pair, busy of lanes alive.
    __host__ __device__ __forceinline__ bool events(unsigned long long up, unsigned long long busy,
                                                    unsigned long long alive)
    {
        f0 = up & c0;
        f1 = c1 & ~(c0 | y0);
        other = ((o0 | o1) & alive) | busy;
        return (f0 | f1 | other) != 0ull;
    }
    // The lanes with a peak at the pair's first (e0) and second sample (e1),
    // where events() said that there may be any; pend: lanes whose slot is full.
    __host__ __device__ __forceinline__ void peaks(unsigned long long alive, unsigned long long pend,
                                                   unsigned long long& e0, unsigned long long& e1)
    {
        e0 = f0 & ~y0 & alive;
        e1 = f1 & ~y1 & alive;
        other |= (((f0 & y0) | (f1 & y1)) & alive) | ((e0 | e1) & pend);
    }
};

// PeakDetector for a whole wave, as the sweeps use it: the masks, the last
// sample's value and the plateau starts.  The compares are written into masks
// and the emit mask feeds the wave's append directly.  All 64 lanes must take
// every call (wave-uniform control flow).  TIMES: track the plateau start and
// report peak times (not needed when only peak values are used).
template <bool TIMES>
struct WavePeakDetector {
    double p;    // last sample d[t-1]
    int pstart;  // plateau start index
    PeakMasks m;

    __device__ __forceinline__ void reset()
    {
        p = 0.0;
        pstart = 0;
        m.up = m.plat = m.skip = 0ull;
    }

    // t >= 2, c = t - 1: the sample cur with its masks c2 and tiny; returns
    // the mask of lanes with a peak at c (value val, time time).
    __device__ __forceinline__ unsigned long long decide(int c, double cur, unsigned long long c2,
                                                         unsigned long long tiny, double& val, int& time)
    {
        const unsigned long long plat = m.plat;
        const PeakMasks::Found f = m.step(c2, tiny);
        val = p;
        time = 0;
        if (TIMES) {
            // a peak's time is its sample index, or the middle of the
            // plateau for a lane that ends one; plateaus are rare, so both
            // lane updates sit behind wave-uniform branches
            time = c;
            if (f.closed) time = lane_bit(plat) ? (pstart + c) >> 1 : c;
            if (f.opened) pstart = lane_bit(f.opened) ? c : pstart;
        }
        p = cur;
        return f.emit;
    }

    // Any t: sample 0 only fills the history, sample 1 only the rising test.
    __device__ __forceinline__ unsigned long long feed(int t, double cur, double& val, int& time)
    {
        const double dnx = cur - p;
        const unsigned long long c2 = wave_mask(dnx <= 0.0), tiny = wave_mask(fabs(dnx) <= 1e-13);
        if (t >= 2) return decide(t - 1, cur, c2, tiny, val, time);
        m.up = ~(c2 | tiny);
        p = cur;
        val = 0.0;
        time = 0;
        return 0ull;
    }
};

// One stored peak: value, sample index, and (sequence number << 6 | lane).
struct PeakEntry {
    double v;
    unsigned t;
    unsigned kl;
};

constexpr int kChunk = 256;  // entries per chunk (4 KiB)

// Pool of fixed-size chunks handed out to waves by an atomic head.  A wave
// appends the peaks that wait in its lanes' slots together, with one mbcnt prefix
// over their mask, so a chunk holds one wave's entries densely: those of a lane
// in time order, with consecutive sequence numbers (the scatter relies on that),
// those of different lanes in no order.
// The bookkeeping sits in one array meta[2 * nchunks + 2] (owner, fill,
// head, overflow), so a sweep loop holds one pointer for it, not four.
struct PeakPool {
    PeakEntry* entries;     // [nchunks * kChunk]
    int* meta;              // owner[nchunks], fill[nchunks], head, overflow
    unsigned nchunks;
    __host__ __device__ int* owner() const { return meta; }                    // global wave id per chunk
    __host__ __device__ int* fill() const { return meta + nchunks; }           // entries used per chunk
    __host__ __device__ unsigned* head() const { return (unsigned*)(meta + 2 * (size_t)nchunks); }  // next free chunk
    __host__ __device__ int* overflow() const { return meta + 2 * (size_t)nchunks + 1; }  // pool ran out
};

// Place in its chunk of an entry with sequence number seq, the chunk put in
// order of (lane, sequence): the lane's entries take the `count` places from
// `base`, consecutive from the smallest sequence number `first`.  -1 for an
// entry that is not one of them, as a chunk that no wave filled may hold.
__host__ __device__ inline int chunk_place(int base, int count, unsigned first, unsigned seq)
{
    return seq - first < (unsigned)count ? base + (int)(seq - first) : -1;
}

struct WaveCursor {
    unsigned chunk;  // current chunk (nchunks when none / exhausted)
    int fill;        // entries used in it
};

__device__ __forceinline__ unsigned lane_prefix(unsigned long long mask)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

__device__ __forceinline__ int first_lane(unsigned long long active) { return __ffsll((long long)active) - 1; }

// Close the cursor's chunk (record its fill) -- call from all active lanes.
__device__ __forceinline__ void close_chunk(const PeakPool& pool, WaveCursor& cur)
{
    const unsigned long long act = __ballot(1);
    if (cur.chunk < pool.nchunks && (int)__lane_id() == first_lane(act)) pool.fill()[cur.chunk] = cur.fill;
}

// Append the entries of the lanes in mask m (wave-uniform control flow
// required).
__device__ __forceinline__ void append_peaks(const PeakPool& pool, WaveCursor& cur, int wave,
                                             unsigned long long m, double v, int t, int k)
{
    if (m == 0ull) return;
    const bool emit = lane_bit(m);
    const int n = __popcll(m);
    if (cur.fill + n > kChunk) {
        const unsigned long long act = __ballot(1);
        const bool leader = (int)__lane_id() == first_lane(act);
        if (cur.chunk < pool.nchunks && leader) pool.fill()[cur.chunk] = cur.fill;
        unsigned nc = 0;
        if (leader) nc = atomicAdd(pool.head(), 1u);
        // the leader is the first active lane: the cursor stays wave-uniform (SGPRs)
        nc = __builtin_amdgcn_readfirstlane(nc);
        if (nc < pool.nchunks) {
            if (leader) pool.owner()[nc] = wave;
        } else {
            if (leader) atomicExch(pool.overflow(), 1);
            nc = pool.nchunks;
        }
        cur.chunk = nc;
        cur.fill = 0;
    }
    // the cursor moves on before the divergent store, which keeps it in SGPRs
    // (moved after it, it is merged from both sides of the store's condition)
    const unsigned base_fill = (unsigned)cur.fill;
    cur.fill += n;
    if (emit && cur.chunk < pool.nchunks) {
        // wave-uniform chunk base + a 32-bit byte offset inside the chunk
        const unsigned off = (base_fill + lane_prefix(m)) * (unsigned)sizeof(PeakEntry);
        char* base = (char*)(pool.entries + (size_t)cur.chunk * kChunk);
        PeakEntry e;
        e.v = v;
        e.t = (unsigned)t;
        e.kl = ((unsigned)k << 6) | (unsigned)__lane_id();
        *(PeakEntry*)(base + off) = e;
    }
}

}  // namespace chaos
