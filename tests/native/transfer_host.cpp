// The copies of transfer.hip on the host: the HIP calls it makes are plain
// memory operations here, and some of them refuse on demand.
//   transfer_host MODE BYTES...   MODE: all, no_pinned, no_event or threads N (N thread creations succeed)
// prints one line per copy: OK or what went wrong, and which way it went.
#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <string>

#include "internal.h"

static bool pinned_ok = true, event_ok = true;
static int threads_left = 1 << 20, started = 0;
static hipError_t last = hipSuccess;

extern "C" {
int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
    if (threads_left-- <= 0) return EAGAIN;
    ++started;
    return real(t, a, f, arg);
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = pinned_ok ? std::malloc(n) : nullptr;
    return *p ? hipSuccess : last = hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(1);
    return event_ok ? hipSuccess : last = hipErrorOutOfMemory;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return last = hipErrorInvalidValue; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(to, from, n);
    return hipSuccess;
}
}

int main(int argc, char **argv) {
    const std::string mode = argv[1];
    int a = 2;
    pinned_ok = mode != "no_pinned";
    event_ok = mode != "no_event";
    if (mode == "threads") threads_left = std::atoi(argv[a++]);
    fk_context ctx;
    for (; a < argc; ++a) {
        const size_t want = std::strtoull(argv[a], nullptr, 10);
        std::vector<unsigned char> from(want), to(want, 0);
        for (size_t i = 0; i < want; ++i) from[i] = static_cast<unsigned char>(i * 2654435761u >> 13);
        try {
            fk::copy_out(&ctx, to.data(), from.data(), want);
            std::printf("%s %s threads %d%s\n", from == to ? "OK" : "WRONG", ctx.link ? "ring" : "plain", started,
                        last != hipSuccess ? " error left behind" : "");
        } catch (const fk::Error &e) {
            std::printf("THROWN %s\n", e.msg.c_str());
        }
        std::fflush(stdout);
    }
    ctx.link.reset();
    return 0;
}
