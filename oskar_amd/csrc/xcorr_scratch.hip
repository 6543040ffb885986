/*
 * Split partials of the direct correlator's allocation-free entry point: a
 * fixed array in a device's code object.  It has a source file, and so a code
 * object, of its own: the runtime loads that when the array's address is first
 * asked for, so only processes that call the entry point hold its memory.
 */
#include <hip/hip_runtime.h>

#include <mutex>

#include "xcorr_common.h"

/* Host code never passes this name to a kernel: it is a host-side stand-in,
 * not a device address; the device address comes from hipGetSymbolAddress. */
static __device__ __align__(256)
        double scratch[oskar_amd::XCORR_PARTIAL_BYTES / sizeof(double)];

namespace oskar_amd {

namespace {

/* The address, looked up once per device (with that device current). */
constexpr int MAX_DEVICES = 64;
std::mutex g_lock;
void* g_address[MAX_DEVICES];

} /* namespace */

hipError_t xcorr_scratch(double** out)
{
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> guard(g_lock);
    if (!g_address[dev])
    {
        void* p = nullptr;
        err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (err != hipSuccess) return err;
        if (!p) return hipErrorInvalidSymbol;
        g_address[dev] = p;
    }
    *out = (double*) g_address[dev];
    return hipSuccess;
}

} /* namespace oskar_amd */
