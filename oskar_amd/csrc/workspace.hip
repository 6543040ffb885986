/* Per-(kind, device, stream) device workspaces (see workspace.h). */
#include <new>

#include "workspace.h"

namespace oskar_amd {

namespace {

struct Entry
{
    int kind, dev;
    hipStream_t stream;
    void* ptr;
    size_t size;
    Entry* next;
};

Entry* g_entries = nullptr;
std::mutex g_lock;
std::mutex g_launch_lock;

} /* namespace */

void* ws_acquire(int kind, int dev, hipStream_t stream, size_t bytes,
        hipError_t* err)
{
    std::lock_guard<std::mutex> guard(g_lock);
    Entry* e = g_entries;
    while (e && !(e->kind == kind && e->dev == dev && e->stream == stream))
        e = e->next;
    if (!e)
    {
        e = new (std::nothrow) Entry{kind, dev, stream, nullptr, 0,
                g_entries};
        if (!e)
        {
            *err = hipErrorOutOfMemory;
            return nullptr;
        }
        g_entries = e;
    }
    if (e->size < bytes)
    {
        if (e->ptr) (void) hipFree(e->ptr);
        e->ptr = nullptr;
        e->size = 0;
        *err = hipMalloc(&e->ptr, bytes > 0 ? bytes : 1);
        if (*err != hipSuccess)
        {
            e->ptr = nullptr;
            return nullptr;
        }
        e->size = bytes;
    }
    *err = hipSuccess;
    return e->ptr;
}

void* ws_acquire_here(int kind, hipStream_t stream, size_t bytes,
        hipError_t* err)
{
    int dev = 0;
    *err = hipGetDevice(&dev);
    return *err == hipSuccess ? ws_acquire(kind, dev, stream, bytes, err) :
            nullptr;
}

std::mutex& ws_launch_lock() { return g_launch_lock; }

} /* namespace oskar_amd */
