// lle.hip -- largest Lyapunov exponent maps (Benettin, two trajectories per
// lane), the path of LLE/src/LLECUDA.cu:56-166 (kernels) and :205-428 (host).
//
// One lane per (A_i, B_j) grid point.  The base and perturbed trajectories
// are stepped in the same loop iteration, which gives the scheduler two
// independent FP64 dependency chains per lane; all state stays in VGPRs and
// nothing but the final FP64 exponent touches HBM (the reference keeps the
// state in shared memory and hands it between two kernels via semi_result).
#include <cmath>
#include <memory>
#include <vector>

#include "csv.hpp"
#include "dispatch.hpp"
#include "lanes.hpp"
#include "lle.hpp"
#include "rotate.hpp"
#include "rotate_plan.hpp"

namespace chaos {

// Benettin loop for one point.  Shared by the one-shot kernel below and the
// batched engine, which stores (X, Xp, sum) between launches.
template <int SYS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(Occupancy<SYS>::waves)))
void lle_map_kernel(const LleArgs p, double* __restrict__ out)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= p.n_points) return;
    const int i = (int)(q % p.nPts);
    const int j = (int)(p.row0 + q / p.nPts);
    // transient (LLE/src/LLECUDA.cu:86), perturbation (:88-102) and the
    // Benettin windows (:147-163) in one pass
    LleProg<SYS> L;
    L.params(p, i, j);
    L.init(p);
    L.ticks(p, (long long)j * p.nPts + i, 0, LleProg<SYS>::total(p));
    out[q] = L.result(p);
}

// The map with the wavefronts taking turns (rotate.hpp): chunks of `chunk`
// ticks of 64-point groups, the lane state parked in st between them.  Rossler
// map of 300^2 points (1.4 wavefronts per SIMD, 240,100 ticks): 41.0 -> 29.3 ms.
template <int SYS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void lle_rotate_kernel(const LleArgs p, const RotateCtl ctl, long long chunk, const LaneStore st,
                       double* __restrict__ out)
{
    using P = LleProg<SYS>;
    struct Kept {
        LaneStore st;
        double* out;
        long long chunk;
    };
    const InVgprs<Kept> kept(Kept{st, out, chunk});
    rotate(ctl, [&](unsigned g, unsigned c, int lane) {
        const long long q = (long long)g * 64 + lane;
        const long long qq = q < p.n_points ? q : 0;
        const int i = (int)(qq % p.nPts);
        const int j = (int)(p.row0 + qq / p.nPts);
        const Kept k = kept.get();
        P L;
        L.params(p, i, j);
        if (c == 0) L.init(p);
        else L.load(k.st, q);
        const long long total = P::total(p), g0 = (long long)c * k.chunk;
        const long long g1 = g0 + k.chunk < total ? g0 + k.chunk : total;
        L.ticks(p, (long long)j * p.nPts + i, g0, g1);
        const Kept after = kept.get();
        if (g1 < total) L.store(after.st, q);
        else if (q < p.n_points) after.out[q] = L.result(p);
    });
}

// The transient alone, one lane per point; X to xs[k * xn + q].
template <int SYS>
__global__ __launch_bounds__(256) void lle_transient_kernel(const LleArgs p, double* __restrict__ xs, long long xn)
{
    using P = LleProg<SYS>;
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= p.n_points) return;
    P L;
    L.params(p, (int)(q % p.nPts), (int)(p.row0 + q / p.nPts));
    L.init(p);
    plain_steps<typename P::Sy>(L.X, L.a, p.sc, p.S);
#pragma unroll
    for (int k = 0; k < P::NX; ++k) xs[k * xn + q] = L.X[k];
}

// The other lane's value of an even / odd lane pair.
__device__ __forceinline__ double pair_swap(double v)
{
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0xB1, 0xF, 0xF, true);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}

// Windows [w0, w1) of a point on a lane pair: the even lane steps X, the odd
// lane Xp, in T; each window ends with LleProg::ticks' renormalisation, done
// on both lanes from the same difference (the odd lane has its negative, which
// rounds alike) and applied by the odd one.
template <int SYS>
__device__ __forceinline__ void pair_windows(const LleArgs& p, const double* a, bool odd, double* T, double& sum,
                                             int w0, int w1)
{
    using Sy = System<SYS>;
    constexpr int NX = Sy::NX;
    for (int w = w0; w < w1; ++w) {
        plain_steps<Sy>(T, a, p.sc, p.NTp);
        double o[NX], e[NX], d2 = 0.0;
#pragma unroll
        for (int l = 0; l < NX; ++l) {
            o[l] = pair_swap(T[l]);
            e[l] = o[l] - T[l];
            d2 = d2 + e[l] * e[l];
        }
        const double dist = sqrt(d2) / p.eps;
        sum = sum + log(dist);
#pragma unroll
        for (int l = 0; l < NX; ++l) {
            const double r = o[l] - e[l] / dist;  // on the odd lane: X - (X - Xp) / dist
            T[l] = odd ? r : T[l];
        }
    }
}

// The Benettin windows with a point's two trajectories on two neighbouring
// lanes (lle_split): for grids that leave SIMDs without a wavefront, where the
// time of a tick is its instructions.  xs: the states after the transient, or
// NULL when there was none.  Rossler preview of 17^2 points 384 -> 251 us,
// Chameleon map of 200^2 23.1 -> 20.7 ms.
template <int SYS>
__device__ __forceinline__ void pair_begin(const LleArgs& p, long long q, bool odd, const double* xs, long long xn,
                                           double* a, double* T)
{
    using P = LleProg<SYS>;
    P L;
    const int i = (int)(q % p.nPts), j = (int)(p.row0 + q / p.nPts);
    L.params(p, i, j);
#pragma unroll
    for (int k = 0; k < P::NA; ++k) a[k] = L.a[k];
    if (T == nullptr) return;
    double d[P::NX];
    P::offset(p, (long long)j * p.nPts + i, d);
#pragma unroll
    for (int k = 0; k < P::NX; ++k) {
        const double x = xs ? xs[k * xn + q] : p.ic[k];
        T[k] = odd ? x + d[k] : x;
    }
}

template <int SYS>
__global__ __launch_bounds__(256) void lle_pair_kernel(const LleArgs p, const double* __restrict__ xs, long long xn,
                                                       double* __restrict__ out)
{
    using P = LleProg<SYS>;
    const long long h = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long q = h >> 1;
    if (q >= p.n_points) return;
    const bool odd = h & 1;
    double a[P::NA], T[P::NX], sum = 0.0;
    pair_begin<SYS>(p, q, odd, xs, xn, a, T);
    pair_windows<SYS>(p, a, odd, T, sum, 0, p.W);
    if (!odd) out[q] = sum / p.tMax;
}

// The same with the wavefronts taking turns: groups of 32 points, chunks of
// `chunk` windows.
template <int SYS>
__global__ __launch_bounds__(256) void lle_pair_rotate_kernel(const LleArgs p, const RotateCtl ctl, int chunk,
                                                              const double* __restrict__ xs, long long xn,
                                                              const LaneStore st, double* __restrict__ out)
{
    using P = LleProg<SYS>;
    rotate(ctl, [&](unsigned g, unsigned c, int lane) {
        const long long h = (long long)g * 64 + lane;
        const long long q = (h >> 1) < p.n_points ? h >> 1 : 0;
        const bool odd = h & 1;
        double a[P::NA], T[P::NX], sum = 0.0;
        if (c == 0) {
            pair_begin<SYS>(p, q, odd, xs, xn, a, T);
        } else {
            pair_begin<SYS>(p, q, odd, xs, xn, a, nullptr);
#pragma unroll
            for (int k = 0; k < P::NX; ++k) T[k] = st.d[k * st.np + h];
            sum = st.d[P::NX * st.np + h];
        }
        const int w0 = (int)c * chunk, w1 = w0 + chunk < p.W ? w0 + chunk : p.W;
        pair_windows<SYS>(p, a, odd, T, sum, w0, w1);
        if (w1 < p.W) {
#pragma unroll
            for (int k = 0; k < P::NX; ++k) st.d[k * st.np + h] = T[k];
            st.d[P::NX * st.np + h] = sum;
        } else if (!odd && (h >> 1) < p.n_points) {
            out[q] = sum / p.tMax;
        }
    });
}

LleArgs make_lle_args(const chaos_options& o, double tMax, double NT, int nPts, double h, double eps,
                      const double* ic, int nx, const double* ranges, const int* idx,
                      double transientTime, const double* values, int na)
{
    check_system(o.system, nx, na);
    CHAOS_REQUIRE(nPts >= 1, "nPts must be >= 1 (got %d)", nPts);
    CHAOS_REQUIRE(h > 0 && std::isfinite(h), "h must be positive");
    CHAOS_REQUIRE(ic && ranges && idx && values, "NULL input array");
    CHAOS_REQUIRE(idx[0] >= 0 && idx[0] < na && idx[1] >= 0 && idx[1] < na,
                  "indicesOfMutVars out of range [0,%d)", na);
    CHAOS_REQUIRE(eps > 0, "eps must be positive");
    CHAOS_REQUIRE(tMax > 0, "tMax must be positive");
    LleArgs p{};
    for (int k = 0; k < na; ++k) p.values[k] = values[k];
    for (int k = 0; k < nx; ++k) p.ic[k] = ic[k];
    p.rA0 = ranges[0];
    p.rA1 = ranges[1];
    p.rB0 = ranges[2];
    p.rB1 = ranges[3];
    p.idxA = idx[0];
    p.idxB = idx[1];
    p.nPts = nPts;
    p.S = horizon_steps(transientTime, h, o.semantics);
    p.NTp = horizon_steps(NT, h, o.semantics);
    const int all = horizon_steps(tMax, h, o.semantics);
    CHAOS_REQUIRE(p.NTp >= 1, "NT/h must be >= 1");
    // The reference runs amountOfCalcBlocks + 1 = all/NTp + 2 windows
    // (LLE/src/LLECUDA.cu:227,147); CONFIG runs exactly all/NTp.
    p.W = (o.semantics == CHAOS_SEM_REFERENCE) ? all / p.NTp + 2 : all / p.NTp;
    p.eps = eps;
    p.tMax = tMax;
    p.sc = make_step_const(h);
    p.seed = o.seed;
    return p;
}

double lle_steps_per_point(const LleArgs& p) { return (double)p.S + 2.0 * p.W * (double)p.NTp; }

static double* lane_state(CallCtx& ctx, int nd, long long groups)
{
    return static_cast<double*>(ctx.scratch(CallCtx::SCRATCH_STATE, (size_t)nd * groups * 64 * sizeof(double)));
}

// lle_split's measured costs: the steps a window's end takes, and the time of
// two wavefronts on a SIMD at once with one trajectory a lane over that of one
// wavefront with two.  The long steps of BASINS and DAMIR, with their sines and
// exponentials, leave a lone wavefront waiting (DAMIR 240^2, 2000 window ticks
// in windows of 1 and 50 steps, on one lane / on pairs: 8.0 / 7.3, 7.0 / 5.6 ms).
template <int SYS>
struct PairCost {
    static constexpr double end = 4.0, two = 1.0;
};
template <>
struct PairCost<SYS_BASINS> {
    static constexpr double end = 1.0, two = 0.92;
};
template <>
struct PairCost<SYS_DAMIR> {
    static constexpr double end = 0.5, two = 0.8;
};

// Transient on one lane per point, then the windows on lane pairs.
static void launch_lle_split(CallCtx& ctx, int system, const LleArgs& p, int block, double* d_out)
{
    const long long n = p.n_points, pairs = (2 * n + 63) / 64;
    const long long windows = (long long)p.W * p.NTp;
    const int turn = rotate_waves(ROTATE_LLE, pairs, device_simds(ctx), windows, p.NTp, 1);
    dispatch_system(system, [&](auto tag) {
        constexpr int S = decltype(tag)::value;
        constexpr int NX = System<S>::NX;
        // the transient's states, then the rotating windows' lane state
        double* mem = lane_state(ctx, NX + (turn ? NX + 1 : 0), pairs);
        double* xs = nullptr;
        const long long xn = pairs * 64;
        if (p.S > 0) {
            xs = mem;
            hipLaunchKernelGGL(lle_transient_kernel<S>, dim3(ceil_div(n, block)), dim3(block), 0, ctx.stream(), p, xs,
                               xn);
            ctx.add_launch();
        }
        if (turn) {
            const int chunk = (int)(rotate_chunk_ticks(windows, p.NTp, 1) / p.NTp);
            const RotateCtl ctl = make_rotate_ctl(ctx, pairs, (p.W + chunk - 1) / chunk);
            const LaneStore st{mem + NX * xn, nullptr, xn};
            hipLaunchKernelGGL(lle_pair_rotate_kernel<S>, dim3(rotate_grid(ctx, turn, block)), dim3(block), 0,
                               ctx.stream(), p, ctl, chunk, xs, xn, st, d_out);
        } else {
            hipLaunchKernelGGL(lle_pair_kernel<S>, dim3(ceil_div(2 * n, block)), dim3(block), 0, ctx.stream(), p, xs,
                               xn, d_out);
        }
    });
    CHAOS_HIP(hipGetLastError());
    ctx.add_launch();
}

void launch_lle_rows(CallCtx& ctx, int system, LleArgs p, long long row0, long long rows, double* d_out)
{
    p.row0 = row0;
    p.n_points = rows * p.nPts;
    const int block = ctx.opt().block > 0 ? ctx.opt().block : 256;
    CHAOS_REQUIRE(block % 64 == 0 && block <= 256, "block must be a multiple of 64 and <= 256");
    const long long groups = (p.n_points + 63) / 64, simds = device_simds(ctx);
    const long long windows = lle_window_ticks(p.S, p.W, p.NTp), total = (long long)p.S + windows;
    bool split = false;
    dispatch_system(system, [&](auto tag) {
        using Cost = PairCost<decltype(tag)::value>;
        split = lle_split(groups, simds, windows, p.NTp, Cost::end, Cost::two);
    });
    if (split) {
        launch_lle_split(ctx, system, p, block, d_out);
        return;
    }
    const int turn = rotate_waves(ROTATE_LLE, groups, simds, total, 1, 2);
    dispatch_system(system, [&](auto tag) {
        constexpr int S = decltype(tag)::value;
        if (turn) {
            const long long chunk = rotate_chunk_ticks(total, 1, 2);
            const RotateCtl ctl = make_rotate_ctl(ctx, groups, (total + chunk - 1) / chunk);
            const LaneStore st{lane_state(ctx, LleProg<S>::ND, groups), nullptr, groups * 64};
            hipLaunchKernelGGL(lle_rotate_kernel<S>, dim3(rotate_grid(ctx, turn, block)), dim3(block), 0, ctx.stream(), p,
                               ctl, chunk, st, d_out);
        } else {
            hipLaunchKernelGGL(lle_map_kernel<S>, dim3(ceil_div(p.n_points, block)), dim3(block), 0, ctx.stream(), p,
                               d_out);
        }
    });
    CHAOS_HIP(hipGetLastError());
    ctx.add_launch();
}

}  // namespace chaos

using namespace chaos;

extern "C" int chaos_lle2d(const chaos_options* opt, double tMax, double NT, int nPts, double h,
                           double eps, const double* initialConditions, int amountOfInitialConditions,
                           const double* ranges, const int* indicesOfMutVars, int writableVar,
                           double maxValue, double transientTime, const double* values,
                           int amountOfValues, double* out)
{
    (void)writableVar;
    (void)maxValue;  // never read by the reference either (LLE/src/LLECUDA.cu:205-428)
    return guarded("chaos_lle2d", [&] {
        chaos_options o = resolve_options(opt);
        CHAOS_REQUIRE(out, "out is NULL");
        LleArgs p = make_lle_args(o, tMax, NT, nPts, h, eps, initialConditions, amountOfInitialConditions,
                                  ranges, indicesOfMutVars, transientTime, values, amountOfValues);
        CallCtx ctx(o);
        const long long n = (long long)nPts * nPts;
        DevBuf<double> tmp;
        double* d_out = out;
        if (!o.device_buffers) {
            tmp.alloc((size_t)n);
            d_out = tmp.get();
        }
        ctx.begin();
        launch_lle_rows(ctx, o.system, p, 0, nPts, d_out);
        const double ms = ctx.end();
        ctx.add_kernel_ms(ms);
        ctx.add_steps(lle_steps_per_point(p) * (double)n);
        if (!o.device_buffers)
            CHAOS_HIP(hipMemcpyAsync(out, d_out, (size_t)n * sizeof(double), hipMemcpyDeviceToHost, ctx.stream()));
        ctx.sync();
        ctx.finish();
    });
}

namespace chaos {

void write_lle_file(TextFile* f, const char* path, const double* ranges, int nPts, const double* v, int output)
{
    // two range lines, then the map at the default precision with NaN
    // written as 0 (LLE/src/LLECUDA.cu:252-253, 383-398)
    MapSpec m;
    m.ranges = ranges;
    m.header_lines = 2;
    m.nPts = nPts;
    m.count = (long long)nPts * nPts;
    m.nan_to_zero = true;
    m.dv = v;
    if (f) {
        write_map_text(*f, m);
        f->close();
    }
    if (out_bin(output)) write_map_bin(std::string(path) + ".bin", m);
}

}  // namespace chaos

extern "C" int chaos_LLE2D(const chaos_options* opt, double tMax, double NT, int nPts, double h,
                           double eps, const double* initialConditions, int amountOfInitialConditions,
                           const double* ranges, const int* indicesOfMutVars, int writableVar,
                           double maxValue, double transientTime, const double* values,
                           int amountOfValues, const char* OUT_FILE_PATH)
{
    return guarded("chaos_LLE2D", [&] {
        CHAOS_REQUIRE(OUT_FILE_PATH, "OUT_FILE_PATH is NULL");
        chaos_options o = resolve_options(opt);
        o.device_buffers = 0;
        const long long n = (long long)nPts * (nPts > 0 ? nPts : 0);
        // Open first: the reference exits before computing when the file
        // cannot be opened (LLE/src/LLECUDA.cu:245-251).
        std::unique_ptr<TextFile> f;
        if (out_csv(o.output)) f.reset(new TextFile(OUT_FILE_PATH));
        std::vector<double> res((size_t)n);
        int rc = chaos_lle2d(&o, tMax, NT, nPts, h, eps, initialConditions, amountOfInitialConditions, ranges,
                             indicesOfMutVars, writableVar, maxValue, transientTime, values, amountOfValues,
                             res.data());
        if (rc != CHAOS_OK) throw Error(rc, chaos_last_error());
        write_lle_file(f.get(), OUT_FILE_PATH, ranges, nPts, res.data(), o.output);
    });
}
