// Host build of the wave peak detector's mask logic (PeakMasks,
// chaoslibrary_amd/csrc/peaks.hpp): 64 rows of samples advance together, one
// bit each, as the sweeps' lanes do -- with the sweeps' shortcut (a sample with
// no lane up & c2 and nothing busy only moves the rising mask on) or without.
#include <cmath>

#include "peaks.hpp"

// data[64][n]; counts[64]; values and times [64][n].
extern "C" void host_peak_masks(const double* data, int n, int shortcut, int* counts, double* values, int* times)
{
    chaos::PeakMasks m{0ull, 0ull, 0ull};
    int pstart[64] = {0};
    for (int l = 0; l < 64; ++l) counts[l] = 0;
    for (int t = 1; t < n; ++t) {
        unsigned long long c2 = 0, tiny = 0;
        for (int l = 0; l < 64; ++l) {
            const double d = data[(size_t)l * n + t] - data[(size_t)l * n + t - 1];
            if (d <= 0.0) c2 |= 1ull << l;
            if (std::fabs(d) <= 1e-13) tiny |= 1ull << l;
        }
        if (t < 2 || (shortcut && (((m.up & c2) | m.busy()) == 0ull))) {
            m.up = ~(c2 | tiny);
            continue;
        }
        const int c = t - 1;
        const unsigned long long plat = m.plat;
        const chaos::PeakMasks::Found f = m.step(c2, tiny);
        for (int l = 0; l < 64; ++l) {
            const unsigned long long b = 1ull << l;
            if (f.emit & b) {
                const int k = counts[l]++;
                values[(size_t)l * n + k] = data[(size_t)l * n + c];
                times[(size_t)l * n + k] = (f.closed & b) && (plat & b) ? (pstart[l] + c) >> 1 : c;
            }
            if (f.opened & b) pstart[l] = c;
        }
    }
}
