// HostRing (stzpp_amd/csrc/host_copy.hpp) on the host alone: the HIP calls it
// makes are stubs on ordinary memory, and memory for a thread can be made to
// run out.  Prints OK when every copy arrived whole.
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../../stzpp_amd/csrc/host_copy.hpp"

static thread_local int g_allow = -1;  // allocations until the next one fails (-1: none fails)

void *operator new(size_t n) {
    if (g_allow == 0) throw std::bad_alloc();
    if (g_allow > 0) g_allow--;
    void *p = std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::malloc(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
}

int main() {
    // 1 byte, a short last chunk, fewer chunks than slots, many chunks
    const size_t chunk = stz::HostRing::kChunk;
    for (size_t n : {size_t(1), stz::HostRing::kDownMin, 17 * chunk - 5, 40 * chunk})
        for (int allow = -1; allow < 9; allow++) {
            std::vector<unsigned char> a(n), b(n, 0), c(n, 0);
            for (size_t i = 0; i < n; i++) a[i] = (unsigned char)(i * 2654435761u >> 13);
            stz::HostRing ring;
            g_allow = allow;
            const hipError_t e = ring.download(b.data(), a.data(), n, nullptr);
            g_allow = allow;
            const hipError_t u = ring.upload(c.data(), a.data(), n, nullptr);
            g_allow = -1;
            if (e != hipSuccess || u != hipSuccess || a != b || a != c) {
                std::printf("FAIL %zu bytes, %d allocations\n", n, allow);
                return 1;
            }
        }
    std::printf("OK\n");
    return 0;
}
