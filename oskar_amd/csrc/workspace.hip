/* Per-(kind, device, stream) device workspaces (see workspace.h). */
#include "workspace.h"

namespace oskar_amd {

namespace {

struct Entry
{
    int kind, dev;
    hipStream_t stream;
    void* ptr;
    size_t size;
    unsigned long long used;     /* when it was last acquired */
};

constexpr int MAX_ENTRIES = 1024;
Entry g_entries[MAX_ENTRIES];
int g_count = 0;
unsigned long long g_clock = 0;
std::mutex g_lock;
std::mutex g_launch_lock;

} /* namespace */

void* ws_acquire(int kind, int dev, hipStream_t stream, size_t bytes,
        hipError_t* err)
{
    std::lock_guard<std::mutex> guard(g_lock);
    Entry* e = nullptr;
    for (int i = 0; i < g_count; ++i)
    {
        Entry& x = g_entries[i];
        if (x.kind == kind && x.dev == dev && x.stream == stream)
        {
            e = &x;
            break;
        }
    }
    if (!e)
    {
        if (g_count < MAX_ENTRIES) e = &g_entries[g_count++];
        else
        {
            /* The least recently used (hipFree waits for its device). */
            e = &g_entries[0];
            for (int i = 1; i < MAX_ENTRIES; ++i)
                if (g_entries[i].used < e->used) e = &g_entries[i];
            if (e->ptr) (void) hipFree(e->ptr);
        }
        e->kind = kind;
        e->dev = dev;
        e->stream = stream;
        e->ptr = nullptr;
        e->size = 0;
    }
    e->used = ++g_clock;
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
