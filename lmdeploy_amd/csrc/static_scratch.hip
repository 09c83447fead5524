// Scratch memory for callers that cannot allocate (code under HIP graph capture, serving loops and
// harnesses that forbid hipMalloc): a file-scope device array that the split-K kernels use for their
// partial tiles and arrival counters instead of a handle's workspace.
//
// Every GPU the library runs on holds its own copy of the array, at its own address, from the
// moment the code object is loaded there until the process ends.  In host code the array's name is
// only a stand-in for those copies: its device address comes from hipGetSymbolAddress, once per
// device with that device current, and only that address is ever handed to a kernel.
#include "w4a16_internal.h"

#include <algorithm>
#include <atomic>
#include <mutex>

namespace w4a16 {

namespace {

constexpr size_t kCounterBytes = kStaticCounterInts * sizeof(int);
constexpr size_t kStaticBytes  = kCounterBytes + kStaticWorkspaceBytes;
constexpr int    kMaxDevices   = 64;

// [arrival counters, in three parts (kStaticCounters)][fp32 partial tiles: kStaticWorkspaceBytes]
static __device__ __align__(256) unsigned char scratch[kStaticBytes];

std::mutex     g_mutex;
unsigned char* g_ptr[kMaxDevices];  // device address of `scratch` on each device, null until looked up
int            g_cus[kMaxDevices];  // and the device's compute units

// A launch made at once tags its counts with a number of its own (arrive_last); zero, a handle's tag, is that of launches
// recorded into a graph.
std::atomic<unsigned> g_launches{0};

__global__ void __launch_bounds__(256) fill_zero_kernel(int* p, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

}  // namespace

hipError_t static_scratch(Scratch* out)
{
    int        dev = 0;
    hipError_t e   = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    unsigned char* ptr;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (!g_ptr[dev]) {
            void* p = nullptr;
            e       = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (e != hipSuccess) return e;
            if (!p) return hipErrorInvalidSymbol;
            e = hipDeviceGetAttribute(&g_cus[dev], hipDeviceAttributeMultiprocessorCount, dev);
            if (e != hipSuccess) return e;
            g_ptr[dev] = static_cast<unsigned char*>(p);
        }
        ptr      = g_ptr[dev];
        out->cus = g_cus[dev];
    }
    out->cnt      = reinterpret_cast<int*>(ptr);
    out->cnt_len  = (int)kStaticCounters;
    out->ws       = reinterpret_cast<float*>(ptr + kCounterBytes);
    out->ws_bytes = kStaticWorkspaceBytes;
    out->epoch    = 1 + (int)(g_launches.fetch_add(1, std::memory_order_relaxed) % ((1u << (31 - kEpochShift)) - 1));
    return hipSuccess;
}

// Before a launch that counts arrivals in `sc`, of static_scratch, with `n` counters.  A launch made at once has a tag that no
// earlier one used, and starts from whatever is there.  The replays of a recorded launch all carry one tag, and a count that
// overlapping calls left under it would be taken for the replay's own, each time: there the counters are cleared first, by a
// kernel (not hipMemsetAsync, whose nodes a graph may replay wrongly), and counted without a tag.
hipError_t prepare_static_counters(Scratch* sc, int n, hipStream_t st)
{
    // (the null stream cannot be captured, and must not be asked while another one is)
    if (st == nullptr) return hipSuccess;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    const hipError_t       e  = hipStreamIsCapturing(st, &cs);
    if (e != hipSuccess) return e;
    if (cs == hipStreamCaptureStatusNone) return hipSuccess;
    sc->epoch = 0;
    sc->cnt += kStaticRecorded;
    n = 2 * std::min(n, sc->cnt_len);  // (eight bytes each)
    return launch_kernel(fill_zero_kernel, dim3((n + 255) / 256), dim3(256), 0, st, sc->cnt, n);
}

}  // namespace w4a16
