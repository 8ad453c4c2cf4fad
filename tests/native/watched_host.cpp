// The call context (chaoslibrary_amd/csrc/runtime.cpp) over a stand-in HIP
// runtime whose device memory is host memory, for tests/test_watched_cpu.py.
#include <cstring>

#include "runtime.hpp"

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.0f; return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
}

// A call as the sweeps make it: a region whose launch is watched, then the
// stage that reads its outputs, then finish().  Returns 1 when that stage ran,
// plus 2 when the call failed.
extern "C" int watched_call(int word)
{
    using namespace chaos;
    int stage = 0;
    try {
        CallCtx ctx(resolve_options(nullptr));
        ctx.begin();
        ctx.watch(&word);
        ctx.end();
        stage = 1;
        ctx.finish();
    } catch (const Error&) {
        return stage + 2;
    }
    return stage;
}
