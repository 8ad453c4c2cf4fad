// Host build of the rotating launches' planning (chaoslibrary_amd/csrc/
// rotate_plan.hpp), for tests/test_rotate_limits_cpu.py.
#include "rotate_plan.hpp"

extern "C" int plan_waves(int kind, long long groups, long long simds, long long ticks, long long unit,
                          long long steps)
{
    return chaos::rotate_waves((chaos::RotateKind)kind, groups, simds, ticks, unit, steps);
}

extern "C" long long plan_chunk(long long ticks, long long unit, long long steps)
{
    return chaos::rotate_chunk_ticks(ticks, unit, steps);
}
