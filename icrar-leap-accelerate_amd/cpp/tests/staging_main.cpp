// Host test of the staging of host-resident visibilities (csrc/staging.cpp) where a copy fails half way.
// The HIP calls that it makes are defined here: copies wait in a queue until a call that the runtime
// promises to finish them (a stream's or a recorded event's synchronisation), as late as a copy engine
// may be, and one of them can be made to fail.  No GPU and no HIP runtime is involved.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "leap_internal.h"

namespace {

struct Copy {
    void* dst;
    const void* src;
    size_t bytes;
};
std::vector<Copy> queue;                 // of the copy stream, in order
size_t finished = 0;                     // copies of it that have been made
std::map<hipEvent_t, size_t> recorded;   // an event's place in it
int calls = 0, fail_at = 0;              // copies asked for; the one that fails (0: none)

void finish(size_t n) {
    for (; finished < n; ++finished) std::memcpy(queue[finished].dst, queue[finished].src, queue[finished].bytes);
}

}  // namespace

extern "C" {
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t) {
    if (++calls == fail_at) return hipErrorUnknown;
    queue.push_back({dst, src, bytes});
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    finish(queue.size());
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    recorded[e] = queue.size();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    finish(recorded.count(e) ? recorded[e] : 0);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
}

namespace leap {
void hip_check(hipError_t e, const char* what, const char*, int) {
    if (e != hipSuccess) throw Error(LEAP_ERR_HIP, what);
}
DeviceBuffer::~DeviceBuffer() { std::free(ptr); }
void DeviceBuffer::reserve(size_t n) {
    if (n <= bytes) return;
    std::free(ptr);
    ptr = std::malloc(n);
    bytes = n;
}
PinnedBuffer::~PinnedBuffer() {}
CapturedSequence::~CapturedSequence() {}
void launch_widen_c64(hipStream_t, const void*, size_t, double*) {}
}  // namespace leap

namespace {

int failures = 0;
void expect(bool ok, const char* what, int route, int at) {
    if (ok) return;
    ++failures;
    std::printf("FAILED route %d, copy %d: %s\n", route, at, what);
}

// Stages 20 MiB of ones with copy `at` failing, then the same of twos to another place.
// Routes: 0 whole rows, 1 pol 0 of complex128, 2 pol 0 of complex64.
void run(int route, int at) {
    queue.clear();
    recorded.clear();
    finished = 0;
    calls = 0;
    leap_ctx ctx;
    for (int b = 0; b < 2; ++b) {
        ctx.ev_h2d[b] = reinterpret_cast<hipEvent_t>(uintptr_t(8 + b));
        ctx.ev_widened[b] = reinterpret_cast<hipEvent_t>(uintptr_t(16 + b));
    }
    ctx.ev_copy_fork = reinterpret_cast<hipEvent_t>(uintptr_t(24));
    ctx.ev_copy_join = reinterpret_cast<hipEvent_t>(uintptr_t(25));
    const size_t n = size_t(20) << 17;  // doubles in 20 MiB
    std::vector<double> ones(n, 1.0), twos(n, 2.0), to1(n, 0.0), to2(n, 0.0);
    std::vector<float> ones32, twos32;
    if (route == 2) {
        ones32.assign(n, 1.0f);
        twos32.assign(n, 2.0f);
    }
    auto stage = [&](const double* wide, const float* narrow, double* to) {
        if (route == 0) leap::stage_copy(&ctx, wide, n * 8, to);
        if (route == 1) leap::stage_pol0(&ctx, wide, LEAP_VIS_C128, 1, n / 2, to);
        if (route == 2) leap::stage_pol0(&ctx, narrow, LEAP_VIS_C64, 1, n / 2, to);
    };
    fail_at = at;
    bool threw = false;
    try {
        stage(ones.data(), ones32.data(), to1.data());
    } catch (const leap::Error&) {
        threw = true;
    }
    expect(threw, "the failed copy is reported", route, at);
    const size_t left = queue.size();
    fail_at = 0;
    stage(twos.data(), twos32.data(), to2.data());
    finish(queue.size());
    expect(left == size_t(at - 1), "the copies before it were sent", route, at);
    // what was sent is what the call was given, not the next call's (route 2 sends both to one buffer)
    for (size_t k = 0; k < left && route != 2; ++k) {
        const Copy& c = queue[k];
        const double* p = static_cast<const double*>(c.dst);
        for (size_t i = 0; i < c.bytes / 8; ++i)
            if (p[i] != 1.0) {
                expect(false, "a copy in flight took the next call's data", route, at);
                break;
            }
    }
    const bool whole = route == 2 ? std::memcmp(ctx.d_widen[0].ptr, twos32.data(), n * sizeof(float)) == 0 : to2 == twos;
    expect(whole, "the next call's data", route, at);
    for (void* p : ctx.h_pinned) std::free(p);
}

}  // namespace

int main() {
    for (int route = 0; route < 3; ++route)
        for (int at : {1, 2}) run(route, at);
    if (failures == 0) std::printf("staging ok\n");
    return failures == 0 ? 0 : 1;
}
