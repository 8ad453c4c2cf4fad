// Host build of the exponent maps' launch rules (chaoslibrary_amd/csrc/
// rotate_plan.hpp), for tests/test_lle_plan_cpu.py.
#include "rotate_plan.hpp"

extern "C" int lle_split_host(long long groups, long long simds, long long S, long long W, long long NTp)
{
    return chaos::lle_split(groups, simds, chaos::lle_window_ticks(S, W, NTp), NTp, 4.0, 1.0);
}

extern "C" int lle_turn_host(long long groups, long long simds, long long S, long long W, long long NTp)
{
    return chaos::rotate_waves(chaos::ROTATE_LLE, groups, simds, S + chaos::lle_window_ticks(S, W, NTp));
}
