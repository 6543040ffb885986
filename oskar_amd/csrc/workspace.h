/*
 * Device workspaces of the kernels, one per (device, stream, kind).  Calls
 * on different streams get different buffers, so concurrent calls on two
 * streams do not share partial sums; calls on one stream are ordered by the
 * stream and reuse its buffer.  A buffer grows (hipFree, which waits for the
 * device, then hipMalloc) when a call needs more.  Buffers live until the
 * process ends: a captured graph may hold their addresses.
 */
#ifndef OSKAR_AMD_WORKSPACE_H_
#define OSKAR_AMD_WORKSPACE_H_

#include <hip/hip_runtime.h>
#include <stddef.h>

#include <mutex>

namespace oskar_amd {

enum WorkspaceKind
{
    WS_XCORR_SPLIT = 0,      /* direct correlator: FP64 split-K partials */
    WS_FACT_SOURCES,         /* shared-beam factorised: stations, sources */
    WS_FACT_PARTIALS,        /* shared-beam factorised: FP32 part tiles */
    WS_FACT_STATIONS,        /* per-station factorised: everything */
    WS_ACORR,                /* auto-correlator: FP64 partial sums */
    WS_SKY_COUNTS,           /* horizon clip, prefix sum: tiles' counts */
    WS_KINDS
};

/* A buffer of at least `bytes` for this (kind, device, stream), or NULL
 * with *err set. */
void* ws_acquire(int kind, int dev, hipStream_t stream, size_t bytes,
        hipError_t* err);

/* The same on the current device, for kernels whose calls may be captured on
 * a stream that has not run them before: under capture, where nothing can be
 * allocated, the buffer is one that all captures of the device share, made by
 * an earlier call of at least this size on any stream, and never freed or
 * moved, since graphs hold its address. */
void* ws_acquire_here(int kind, hipStream_t stream, size_t bytes,
        hipError_t* err);

/* Held from acquiring a buffer to the last launch that uses it, so that
 * host threads which share a stream do not interleave their launches. */
std::mutex& ws_launch_lock();

} /* namespace oskar_amd */

#endif /* OSKAR_AMD_WORKSPACE_H_ */
