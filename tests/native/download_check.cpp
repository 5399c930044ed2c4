// Host harness for the download of results (gpview_amd/csrc/gpv_download.hpp):
// tests/test_downloads.py drives it with the HIP calls below in place of the
// runtime's, "device" memory being host memory.  Test tooling only.
#include "gpv_download.hpp"

#include <cstdlib>

namespace {
// what the stand-ins did, and what they are told to refuse
struct Log {
    int64_t kernels = 0, kernel_bytes = 0, copies = 0, copy_bytes = 0, waits = 0;
    bool no_locked_memory = false, no_events = false;
    hipError_t last = hipSuccess;
} g;
struct Range {
    const char* p;
    size_t n;
    hipMemoryType type;
};
std::vector<Range> g_known;   // memory that the runtime knows

hipError_t note(hipError_t e)
{
    if (e != hipSuccess) g.last = e;
    return e;
}
}  // namespace

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned int)
{
    if (g.no_locked_memory) return note(hipErrorOutOfMemory);
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    for (const Range& r : g_known)
        if ((const char*)p >= r.p && (const char*)p < r.p + r.n) {
            *a = hipPointerAttribute_t{};
            a->type = r.type;
            a->devicePointer = a->hostPointer = const_cast<void*>(p);
            return hipSuccess;
        }
    return note(hipErrorInvalidValue);
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    ++g.copies;
    g.copy_bytes += (int64_t)n;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    ++g.waits;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    if (g.no_events) return note(hipErrorOutOfMemory);
    *e = (hipEvent_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::free((void*)e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t)
{
    ++g.waits;
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = g.last;
    g.last = hipSuccess;
    return e;
}
}

namespace gpv {
void launch_copy_out(const CopyOut& L, int pieces, hipStream_t)
{
    ++g.kernels;
    for (int k = 0; k < pieces; ++k) {
        g.kernel_bytes += L.n[k];
        std::memcpy(L.dst[k], L.src[k], (size_t)L.n[k]);
    }
}
}  // namespace gpv

extern "C" {
void* dl_new() { return new gpv::Downloader(); }
void dl_delete(void* d) { delete static_cast<gpv::Downloader*>(d); }
// type 0: page-locked host memory, 1: device memory
void dl_known(const void* p, int64_t n, int type)
{
    g_known.push_back(Range{(const char*)p, (size_t)n, type ? hipMemoryTypeDevice : hipMemoryTypeHost});
}
void dl_reset(int no_locked_memory, int no_events)
{
    g = Log{};
    g.no_locked_memory = no_locked_memory != 0;
    g.no_events = no_events != 0;
    g_known.clear();
}
// log: kernels, their bytes, copies, their bytes, waits, the error left behind
int dl_run(void* d, int count, void* const* dst, const void* const* src, const int64_t* n, int64_t* log)
{
    std::vector<gpv::Downloader::Piece> p;
    for (int k = 0; k < count; ++k) p.push_back({dst[k], src[k], (size_t)n[k]});
    const int r = (int)static_cast<gpv::Downloader*>(d)->run(p.data(), count, nullptr);
    const int64_t v[6] = {g.kernels, g.kernel_bytes, g.copies, g.copy_bytes, g.waits, (int64_t)g.last};
    std::memcpy(log, v, sizeof v);
    return r;
}
}
