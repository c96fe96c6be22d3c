// split_scratch_check.cpp — the pool of split-k partition buffers and the
// workspace that may fail (stream_scratch, try_workspace, runtime.cpp) on the
// CPU, against a model of the HIP calls they make. The model refuses what HIP refuses while a stream is captured:
// allocating and freeing unless the thread's capture mode is relaxed, and any
// wait for a captured stream or the device. Prints "ok", or what went wrong.
#include "../../blis_amd/csrc/runtime.cpp"

#include <cstdlib>
#include <map>
#include <set>

namespace {

std::map<hipStream_t, unsigned long long> capturing;   // stream -> capture id
hipStreamCaptureMode thread_mode = hipStreamCaptureModeGlobal;
std::set<void*> live, held;      // allocations; those that a graph holds
size_t live_bytes = 0;
std::map<void*, size_t> sizes;
uintptr_t next_address = 4096;
bool memory_left = true;

void fail(const char* what) {
    std::printf("failed: %s\n", what);
    std::fflush(stdout);
    std::_Exit(1);
}

bool refused() { return !capturing.empty() && thread_mode != hipStreamCaptureModeRelaxed; }

hipStream_t stream_no(int i) { return (hipStream_t)(uintptr_t)(i + 1); }

// A product's call, as gemm.hip makes it; what a capture gets, its graph holds.
void* take(size_t mib, int st) {
    void* p = blis_amd::stream_scratch(mib << 20, stream_no(st));
    if (p != nullptr) {
        if (!live.count(p) || sizes[p] < (mib << 20)) fail("buffer freed or too small");
        if (capturing.count(stream_no(st))) held.insert(p);
    }
    return p;
}

bool shares_with_graph(size_t mib, int st) {
    const std::set<void*> before = held;
    return before.count(take(mib, st)) != 0;
}

void begin(int st, unsigned long long id) { capturing[stream_no(st)] = id; }
void end(int st) { capturing.erase(stream_no(st)); }

} // namespace

extern "C" {
const char* bli_error_string_for_code(gint_t) { return "error"; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "refused during capture"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = stream_no(99); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemGetAddressRange(hipDeviceptr_t*, size_t*, hipDeviceptr_t) { return hipErrorInvalidValue; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    return capturing.count(s) || refused() ? hipErrorStreamCaptureUnsupported : hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    return capturing.empty() ? hipSuccess : hipErrorStreamCaptureUnsupported;
}
hipError_t hipMalloc(void** p, size_t n) {
    if (refused()) return hipErrorStreamCaptureUnsupported;
    if (!memory_left) return hipErrorOutOfMemory;
    *p = (void*)next_address;
    next_address += n;
    live.insert(*p);
    sizes[*p] = n;
    live_bytes += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (refused()) return hipErrorStreamCaptureUnsupported;
    if (p == nullptr) return hipSuccess;
    if (held.count(p)) fail("freed a buffer that a graph holds");
    if (!live.erase(p)) fail("freed twice");
    live_bytes -= sizes[p];
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) {
    *c = capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamGetCaptureInfo(hipStream_t s, hipStreamCaptureStatus* c,
                                   unsigned long long* id) {
    if (id && capturing.count(s)) *id = capturing[s];
    return hipStreamIsCapturing(s, c);
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    std::swap(*m, thread_mode);
    return hipSuccess;
}
}

int main() {
    // Warm up on one stream, capture on another.
    void* eager0 = take(4, 0);
    begin(1, 7);
    void* graph1 = take(4, 1);
    if (graph1 == nullptr) fail("no buffer for a captured stream");
    if (graph1 == eager0) fail("a graph shares an eager stream's buffer");
    if (take(3, 1) != graph1) fail("products of one captured stream run in turn");
    if (take(40, 1) == nullptr) fail("a larger product in the same capture");
    begin(2, 7);                                   // a stream forked into the capture
    if (take(4, 2) == graph1) fail("two streams of a capture share a buffer");
    end(2);
    // An eager product on another stream while this one is captured, growing.
    if (take(40, 0) == nullptr || take(40, 3) == nullptr) fail("eager beside a capture");
    end(1);
    if (shares_with_graph(4, 1)) fail("an eager product shares a graph's buffer");
    begin(1, 8);
    if (shares_with_graph(4, 1)) fail("two graphs share a buffer");
    end(1);
    // A capture of a stream whose own eager buffer is too small.
    take(4, 4);
    begin(4, 9);
    if (take(40, 4) == nullptr) fail("a captured product larger than the eager ones");
    end(4);
    // More streams than buffers, captured and not.
    for (int st = 10; st < 22; ++st) take(4, st);
    begin(30, 10);
    if (take(4, 30) == nullptr) fail("a capture after many streams");
    if (take(4, 31) == nullptr) fail("a new stream beside a capture");
    end(30);
    // No memory: the caller makes one pass; later calls ask again.
    memory_left = false;
    if (blis_amd::try_workspace(4 << 20, 13) != nullptr) fail("a workspace without memory");
    if (take(4, 40) != nullptr) fail("a buffer without memory");
    begin(41, 11);
    if (take(4, 41) != nullptr) fail("a captured buffer without memory");
    end(41);
    memory_left = true;
    if (take(4, 40) == nullptr || blis_amd::try_workspace(4 << 20, 13) == nullptr)
        fail("memory is back");
    hipFree(blis_amd::workspace(4 << 20, 13));
    // What graphs hold is bounded, and so are the streams' buffers.
    bool refused_one = false;
    for (unsigned long long id = 100; id < 200; ++id) {
        begin(50, id);
        refused_one = take(32, 50) == nullptr || refused_one;
        end(50);
    }
    size_t held_bytes = 0;
    for (void* p : held) held_bytes += sizes[p];
    if (!refused_one || held_bytes > ((size_t)1 << 30)) fail("graphs hold more than 1 GiB");
    if (live_bytes - held_bytes > (size_t)8 * 48 << 20) fail("streams hold more than eight buffers");
    if (thread_mode != hipStreamCaptureModeGlobal) fail("the thread's capture mode was changed");
    std::printf("ok\n");
    return 0;
}
