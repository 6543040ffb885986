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

/* Buffers for captured calls, newest first. */
struct Capture
{
    int kind, dev;
    void* ptr;
    size_t size;
    Capture* next;
};

Capture* g_captures = nullptr;
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
    if (*err != hipSuccess) return nullptr;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (stream)
    {
        *err = hipStreamIsCapturing(stream, &capture);
        if (*err != hipSuccess) return nullptr;
    }
    Capture* c = nullptr;
    {
        std::lock_guard<std::mutex> guard(g_lock);
        for (c = g_captures; c && !(c->kind == kind && c->dev == dev);)
            c = c->next;
        if (!c || c->size < bytes)
        {
            /* Newest first, at least twice the last; the last stays. */
            Capture* n = new (std::nothrow) Capture{kind, dev, nullptr,
                    c && 2 * c->size > bytes ? 2 * c->size : bytes,
                    g_captures};
            *err = n ? hipMalloc(&n->ptr, n->size > 0 ? n->size : 1) :
                    hipErrorOutOfMemory;
            if (*err != hipSuccess)
            {
                delete n;
                return nullptr;
            }
            g_captures = c = n;
        }
    }
    if (capture != hipStreamCaptureStatusNone) return c->ptr;
    return ws_acquire(kind, dev, stream, bytes, err);
}

std::mutex& ws_launch_lock() { return g_launch_lock; }

} /* namespace oskar_amd */
