// The sweeps' loop over pairs of samples (SweepProg::body,
// chaoslibrary_amd/csrc/lanes.hpp) on the host, one bit a lane, from the masks
// of SamplePair and PeakMasks (peaks.hpp): pending slots, their flush when a
// lane peaks again, and pairs that go sample by sample.
#include <cmath>

#include "peaks.hpp"

// data[64][n]; a lane stops at the first sample with |v| > bound or not finite;
// |v| < band is sure to be inside.  counts[64]; values and times [64][n].
// Returns the pairs that went sample by sample.
extern "C" int host_sample_pairs(const double* data, int n, double bound, double band, int* counts, double* values,
                                 int* times)
{
    typedef unsigned long long u64;
    chaos::PeakMasks m{0ull, 0ull, 0ull};
    u64 alive = ~0ull, pend = 0ull;
    int pstart[64] = {0}, pend_t[64], slow = 0;
    double pend_v[64];
    auto at = [&](int l, int t) { return data[(size_t)l * n + t]; };
    auto mask = [&](auto f) {
        u64 r = 0;
        for (int l = 0; l < 64; ++l)
            if (f(l)) r |= 1ull << l;
        return r;
    };
    auto falls = [&](int t) { return mask([&](int l) { return at(l, t) - at(l, t - 1) <= 0.0; }); };
    auto near = [&](int t) { return mask([&](int l) { return std::fabs(at(l, t) - at(l, t - 1)) <= 1e-13; }); };
    auto outside = [&](int t) { return mask([&](int l) { return !(std::fabs(at(l, t)) < band); }); };
    auto diverge = [&](int t, u64 out) {
        alive &= ~mask([&](int l) { return (out >> l & 1) && (!std::isfinite(at(l, t)) || std::fabs(at(l, t)) > bound); });
    };
    auto emit = [&](int l, double v, int t) {
        values[(size_t)l * n + counts[l]] = v;
        times[(size_t)l * n + counts[l]++] = t;
    };
    auto flush = [&] {
        for (int l = 0; l < 64; ++l)
            if (pend >> l & 1) emit(l, pend_v[l], pend_t[l]);
        pend = 0ull;
    };
    auto settle = [&](int t, u64 c, u64 y, u64 o) {
        diverge(t, o & alive);
        if (t < 2) {
            m.up = ~(c | y);
            return;
        }
        const u64 plat = m.plat;
        const chaos::PeakMasks::Found f = m.step(c, y);
        for (int l = 0; l < 64; ++l) {
            const u64 b = 1ull << l;
            if (f.emit & alive & b) emit(l, at(l, t - 1), (f.closed & plat & b) ? (pstart[l] + t - 1) >> 1 : t - 1);
            if (f.opened & b) pstart[l] = t - 1;
        }
    };
    for (int l = 0; l < 64; ++l) counts[l] = 0;
    int t = 0;
    for (; t < n && t < 2; ++t) {
        if (t == 0) diverge(0, outside(0));
        else settle(t, falls(t), near(t), outside(t));
    }
    u64 busy = m.busy() & alive;
    for (; t + 1 < n; t += 2) {
        chaos::SamplePair s;
        s.c0 = falls(t);
        s.y0 = near(t);
        s.o0 = outside(t);
        s.c1 = falls(t + 1);
        s.y1 = near(t + 1);
        s.o1 = outside(t + 1);
        if (s.events(m.up, busy, alive)) {
            u64 e0, e1;
            s.peaks(alive, pend, e0, e1);
            if (s.other) {
                flush();
                settle(t, s.c0, s.y0, s.o0);
                settle(t + 1, s.c1, s.y1, s.o1);
                busy = m.busy() & alive;
                ++slow;
                continue;
            }
            for (int l = 0; l < 64; ++l) {
                if (e0 >> l & 1) pend_v[l] = at(l, t - 1), pend_t[l] = t - 1;
                if (e1 >> l & 1) pend_v[l] = at(l, t), pend_t[l] = t;
            }
            pend |= e0 | e1;
        }
        m.up = ~(s.c1 | s.y1);
    }
    flush();
    for (; t < n; ++t) settle(t, falls(t), near(t), outside(t));
    return slow;
}
