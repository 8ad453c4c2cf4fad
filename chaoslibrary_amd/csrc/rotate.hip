// rotate.hip -- host side of the rotating launches (rotate.hpp).
#include "rotate.hpp"
#include "rotate_plan.hpp"

namespace chaos {

__global__ void rotate_clear_kernel(unsigned* p, unsigned n)
{
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

RotateCtl make_rotate_ctl(CallCtx& ctx, long long groups, long long chunks)
{
    CHAOS_REQUIRE(groups > 0 && chunks > 0 && groups * chunks < kRotateTickets, "rotating launch too large");
    ctx.check_watched();  // an earlier launch of this call used the same block
    // the ticket counter and the error word on a cache line of their own
    constexpr unsigned kPad = 32;
    unsigned* buf = static_cast<unsigned*>(ctx.scratch(CallCtx::SCRATCH_CTL, ((size_t)groups + kPad) * sizeof(unsigned)));
    const unsigned n = (unsigned)groups + kPad;
    hipLaunchKernelGGL(rotate_clear_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, ctx.stream(), buf, n);
    CHAOS_HIP(hipGetLastError());
    int* err = reinterpret_cast<int*>(buf + 1);
    ctx.watch(err);
    return RotateCtl{buf, err, buf + kPad, (unsigned)groups, (unsigned)chunks};
}

long long device_simds(CallCtx& ctx) { return 4LL * device_props(ctx.device()).multiProcessorCount; }

unsigned rotate_grid(CallCtx& ctx, int waves, int block)
{
    return rotate_blocks(device_props(ctx.device()).multiProcessorCount, waves, block);
}

}  // namespace chaos
