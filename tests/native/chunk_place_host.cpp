// The order in which a chunk of the peak store is scattered
// (chunk_place, chaoslibrary_amd/csrc/peaks.hpp), for
// tests/test_chunk_place_cpu.py: the kernel's steps for one chunk of n entries.
#include "peaks.hpp"

extern "C" void chunk_places(const unsigned* kl, int n, int* place)
{
    unsigned first[64];
    int count[64] = {0}, base[64];
    for (int l = 0; l < 64; ++l) first[l] = ~0u;
    for (int s = 0; s < n; ++s) {
        const unsigned l = kl[s] & 63u;
        if ((kl[s] >> 6) < first[l]) first[l] = kl[s] >> 6;
        ++count[l];
    }
    for (int l = 0, b = 0; l < 64; b += count[l++]) base[l] = b;
    for (int s = 0; s < n; ++s) {
        const unsigned l = kl[s] & 63u;
        place[s] = chaos::chunk_place(base[l], count[l], first[l], kl[s] >> 6);
    }
}
