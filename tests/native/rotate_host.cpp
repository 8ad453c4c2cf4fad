// Host build of the rotating launches' planning (chaoslibrary_amd/csrc/
// rotate_plan.hpp), for tests/test_rotate_plan_cpu.py.
#include "rotate_plan.hpp"

extern "C" int rotate_waves_host(int kind, long long groups, long long simds, long long ticks)
{
    return chaos::rotate_waves((chaos::RotateKind)kind, groups, simds, ticks);
}

extern "C" long long rotate_chunk_host(long long ticks, long long unit)
{
    return chaos::rotate_chunk_ticks(ticks, unit);
}
