// rotate_plan.hpp -- when a grid's wavefronts take turns on the SIMDs, as
// plain host C++ (no HIP types), so that it runs and is tested on machines
// without a GPU.
#pragma once

namespace chaos {

// The two kinds of per-lane program: exponent maps (two trajectories, no
// per-sample work: two wavefronts on a SIMD already fill its FP64 unit) and
// sweeps (per-sample scalar work and branches, which more wavefronts hide).
enum RotateKind { ROTATE_LLE, ROTATE_SWEEP };

constexpr long long kRotateChunk = 2000;  // fewest ticks per chunk
constexpr int kRotateMinChunks = 12, kRotateMaxChunks = 48;
// Most steps of a trajectory in a chunk, and tickets (groups * chunks) in a run.
// A wavefront waits for the chunk before its own and gives up after about a
// minute or two (kRotatePolls, rotate.hpp), which must mean that the chunk's
// wavefront is gone and not that the run is a long one: a step is at most 4 us
// (the slowest map, two trajectories a lane, two wavefronts on the SIMD), so a
// chunk stays below 10 s.
constexpr long long kRotateChunkSteps = 1LL << 21, kRotateTickets = 1LL << 25;

// Ticks per chunk: a run of `ticks` in at most kRotateMaxChunks chunks of at
// least kRotateChunk ticks, rounded up to a multiple of `unit`; more chunks, of
// one unit or more, where `steps` steps a tick (0: not asked) would make that
// more than kRotateChunkSteps steps.
inline long long rotate_chunk_ticks(long long ticks, long long unit, long long steps = 0)
{
    long long c = (ticks + kRotateMaxChunks - 1) / kRotateMaxChunks;
    if (c < kRotateChunk) c = kRotateChunk;
    if (unit < 1) unit = 1;
    c = (c + unit - 1) / unit;
    if (steps > 0 && c > kRotateChunkSteps / steps / unit) c = kRotateChunkSteps / steps / unit;
    return c < 1 ? unit : c * unit;
}

// Wavefronts per SIMD of a rotating launch (rotate.hpp) over `groups`
// wavefronts of work, or 0 to launch them all at once.
//
// At once, the SIMDs that hold ceil(w) wavefronts (w = groups / simds) finish
// last and the others idle meanwhile; rotating, simds * k wavefronts take the
// groups' chunks in turn and every SIMD does w of the work.  In units of a
// wavefront's share of a full SIMD the times were, on 1024 SIMDs over w = 1 to
// 8 (Rossler, Lorenz and Chameleon maps of 258^2 to 720^2 points, 80,000 and
// 60,000 ticks):
//   exponent maps: at once ceil(w); k = 1: 1.03 w; k = 2: 0.92 w + 0.6
//   sweeps:        at once ceil(w) + 0.34; k = 1: 1.33 w; k = 2: w + 0.38
// (with k = 2 a chunk's predecessor has only just finished when w is little
// above 2, and k = 3 or 4 were never ahead).  For instance, at once / rotating:
// Rossler exponents 258^2 (w = 1.02) 18.7 / 9.7 ms, 300^2 (1.37) 17.2 / 12.7,
// 400^2 (2.44) 26.7 / 22.1, 600^2 (5.49) 52.8 / 49.6; Lorenz peak map 300^2
// 13.6 / 11.5, 400^2 19.7 / 16.4, 600^2 36.5 / 33.8; Chameleon peak map 300^2
// 16.4 / 13.3.  The plain launch stays where it is within 2 %, above eight
// wavefronts a SIMD (the most that reside: the hardware's refill evens the
// load), and for runs of fewer than 12 chunks of 2000 ticks (`ticks` per
// group): shorter chunks cost too much to hand over and fewer leave an uneven
// end of their own.  Chunks of one long `unit` each may be fewer; the rounds in
// which they are run then count whole (lane pairs on 1.22 and 1.76 wavefronts a
// SIMD, 40,000 window ticks, at once / in turns: one window 6.15 / 6.21 and 5.82
// / 6.16 ms, two 6.14 / 4.84 and 5.84 / 6.23, four 5.99 / 3.97 and 5.81 / 6.16,
// six 5.97 / 4.18 and 5.83 / 5.70).  The plain launch stays, too, where the chunks
// would be too long to wait for or too many.
struct RotatePlan {
    int waves;    // wavefronts per SIMD, 0: all at once
    double time;  // in the units above
};

inline RotatePlan rotate_plan(RotateKind kind, long long groups, long long simds, long long ticks, long long unit,
                              long long steps)
{
    if (simds <= 0) return {0, 1e30};
    const double c = (double)((groups + simds - 1) / simds);
    const double at_once = kind == ROTATE_LLE ? c : c + 0.34;
    const RotatePlan plain{0, at_once};
    if (groups <= simds || groups > 8 * simds) return plain;
    if (ticks < kRotateChunk * kRotateMinChunks) return plain;
    const long long chunk = rotate_chunk_ticks(ticks, unit, steps), chunks = (ticks + chunk - 1) / chunk;
    if (steps > 0 && chunk > kRotateChunkSteps / steps) return plain;
    if (chunks >= kRotateTickets / groups) return plain;
    const long long units = groups * chunks;
    double w = (double)groups / (double)simds, w2 = w;
    if (chunks < kRotateMinChunks) {
        w = (double)((units + simds - 1) / simds) / (double)chunks;
        w2 = 2.0 * (double)((units + 2 * simds - 1) / (2 * simds)) / (double)chunks;
    }
    const double one = kind == ROTATE_LLE ? 1.03 * w : 1.33 * w;
    const double two = groups < 2 * simds ? 1e30 : kind == ROTATE_LLE ? 0.92 * w2 + 0.6 : w2 + 0.38;
    const double best = one < two ? one : two;
    if (best >= 0.98 * at_once) return plain;
    return {one < two ? 1 : 2, best};
}

inline int rotate_waves(RotateKind kind, long long groups, long long simds, long long ticks, long long unit = 1,
                        long long steps = 0)
{
    return rotate_plan(kind, groups, simds, ticks, unit, steps).waves;
}

// Blocks of `block` threads (a multiple of 64) that hold `waves` wavefronts for
// each of a CU's four SIMDs; a wavefront takes tickets by itself, so the block's
// size is the caller's choice.
inline unsigned rotate_blocks(long long cus, int waves, int block)
{
    return (unsigned)((cus * waves * 256 + block - 1) / block);
}

// Window ticks of an exponent map, for the rules on it: none for a transient of
// negative length, whose run LleProg::ticks refuses (the map is 0), so such a
// call keeps to the plain kernel, which asks LleProg::ticks.
inline long long lle_window_ticks(long long S, long long W, long long NTp)
{
    return S < 0 ? 0 : W * NTp;
}

// Exponent maps: whether the windows run with the base and the perturbed
// trajectory of a point on two neighbouring lanes instead of one after the
// other on the same lane.  That halves each wavefront's steps and doubles the
// wavefronts.  Both lanes do a window's end (the distance and its logarithm), so
// a wavefront's work falls to (NTp + end) / (2 NTp + end), `end` in steps; up to
// one wavefront of pairs a SIMD that is the gain (17^2 points, 2100 window
// ticks: 384 -> 251 us; Rossler with half its 80,000 ticks in windows 128^2 9.2 ->
// 6.4 ms).  Above, the SIMD does that work twice, which gains where the pairs'
// wavefronts take turns (200^2 9.3 -> 7.6 ms, 230^2 (0.81 wavefronts per SIMD) 9.2
// -> 8.8; none when the SIMDs are full, 256^2: 9.7 -> 10.0, so the line is at
// 0.9), or where two wavefronts at once take `two` < 1 times the time of one with
// both trajectories.  Too few ticks for turns, on one lane / on pairs:
// 200^2 and 240^2 Rossler, 2000 window ticks in windows of 1, 8, 50 steps 1.50 /
// 2.10, 0.84 / 1.01, 0.67 / 0.70 ms; BASINS in windows of 1, 4, 8, 50 steps
// 2.9 / 3.4, 1.89 / 1.89, 1.80 / 1.71, 1.70 / 1.58.
// Below 200 window ticks the second launch costs what it saves.
inline bool lle_split(long long groups, long long simds, long long window_ticks, long long NTp, double end, double two)
{
    if (simds <= 0 || 10 * groups > 9 * simds || window_ticks < 200) return false;
    const long long pairs = 2 * groups;
    const RotatePlan plan = rotate_plan(ROTATE_LLE, pairs, simds, window_ticks, NTp, 1);
    const double time = plan.waves || pairs <= simds ? plan.time : two * plan.time;
    return time * ((double)NTp + end) / (2.0 * (double)NTp + end) < 0.98;
}

}  // namespace chaos
