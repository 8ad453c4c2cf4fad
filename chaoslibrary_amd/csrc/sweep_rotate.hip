// sweep_rotate.hip -- the Bifurcation and Basins sweeps for grids that do not
// fill the SIMDs evenly: the wavefronts take turns (rotate.hpp), chunks of
// ticks of 64-point groups with the lane state parked in between.  The
// Chameleon peak map of 300^2 points (1.4 wavefronts per SIMD) 40.2 -> 31.2 ms.
#include "dispatch.hpp"
#include "lanes.hpp"
#include "moments.hpp"
#include "rotate.hpp"
#include "rotate_plan.hpp"
#include "sweep.hpp"

namespace chaos {

template <int SYS, int WV, int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void sweep_rotate_kernel(const SweepArgs A, const RotateCtl ctl, long long chunk, const LaneStore st,
                         WaveCursor* __restrict__ cursors)
{
    const long long total = SweepProg<SYS, KIND>::total(A);
    const InVgprs<SweepPark> park(SweepPark{st, cursors, total});
    const InVgprs<long long> len(chunk);
    rotate(ctl, [&](unsigned g, unsigned c, int lane) {
        const InVgprs<long long> group((long long)g);
        const long long n = len.get(), g0 = (long long)c * n, left = park.get().total - g0;
        sweep_group_ticks<SYS, KIND, WV>(
            A, [&] { return park.get(); }, [&] { return group.get(); }, lane, g0, g0 + (n < left ? n : left));
    });
}

// The z-score's first pass over the stored features, block for block what
// sweep_kernel's epilogue forms from registers (a rotating wavefront ends a
// group at a time, not the 256 points of a block together).
__global__ __launch_bounds__(256) void feature_moments_kernel(const SweepArgs A)
{
    const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
    const bool in_range = q < A.n_points;
    double f[3] = {0.0, 0.0, 0.0};
    bool m = false;
    if (in_range) {
        f[0] = A.f0[q];
        f[1] = A.f1[q];
        f[2] = A.f2[q];
        m = A.flags[q] != 0;
    }
    block256_moments(f, 3, m, A.zb, A.zsum, A.zcnt, A.zmm);
}

void launch_sweep_rotating(CallCtx& ctx, int system, int writableVar, int kind, const SweepArgs& A, int waves)
{
    const long long groups = (A.n_points + 63) / 64, np = groups * 64;
    const long long total = (long long)A.S + A.B, chunk = rotate_chunk_ticks(total, 1, A.pre);
    const RotateCtl ctl = make_rotate_ctl(ctx, groups, (total + chunk - 1) / chunk);
    dispatch_system(system, [&](auto tag) {
        constexpr int S = decltype(tag)::value;
        constexpr int NXs = System<S>::NX;
        auto go = [&](auto wvtag, auto kindtag) {
            constexpr int WV = decltype(wvtag)::value, KIND = decltype(kindtag)::value;
            if constexpr (WV < NXs) {
                using P = SweepProg<S, KIND>;
                const LaneStore st{
                    static_cast<double*>(ctx.scratch(CallCtx::SCRATCH_STATE, (size_t)P::ND * np * sizeof(double))),
                    static_cast<int*>(ctx.scratch(CallCtx::SCRATCH_INTS, (size_t)P::NI * np * sizeof(int))), np};
                WaveCursor* cursors = static_cast<WaveCursor*>(
                    ctx.scratch(CallCtx::SCRATCH_CURSORS, (size_t)groups * sizeof(WaveCursor)));
                hipLaunchKernelGGL((sweep_rotate_kernel<S, WV, KIND>), dim3(rotate_grid(ctx, waves)), dim3(256), 0,
                                   ctx.stream(), A, ctl, chunk, st, cursors);
            }
        };
        auto pick_wv = [&](auto kindtag) {
            if (writableVar == 0) go(std::integral_constant<int, 0>{}, kindtag);
            else if (writableVar == 1) go(std::integral_constant<int, 1>{}, kindtag);
            else go(std::integral_constant<int, 2>{}, kindtag);
        };
        if (kind == KIND_BIF) pick_wv(std::integral_constant<int, KIND_BIF>{});
        else if (kind == KIND_BIF_VALS) pick_wv(std::integral_constant<int, KIND_BIF_VALS>{});
        else if (kind == KIND_BASINS_REF) pick_wv(std::integral_constant<int, KIND_BASINS_REF>{});
        else pick_wv(std::integral_constant<int, KIND_BASINS_CFG>{});
    });
    CHAOS_HIP(hipGetLastError());
    ctx.add_launch();
    if (kind == KIND_BASINS_CFG && A.zsum) {
        hipLaunchKernelGGL(feature_moments_kernel, dim3(ceil_div((unsigned long long)A.n_points, 256)), dim3(256), 0,
                           ctx.stream(), A);
        CHAOS_HIP(hipGetLastError());
        ctx.add_launch();
    }
}

}  // namespace chaos
