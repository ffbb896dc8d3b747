// A host stand-in of the HIP calls that pinned_pool.h makes: streams that can be captured or
// destroyed, work that is done when the test says so, and an event that, asked for after its
// last stream is being captured or has gone, answers with an error as the runtime does.
#pragma once
#include <cstdlib>

enum hipError_t { hipSuccess = 0, hipErrorInvalidHandle = 400, hipErrorNotReady = 600, hipErrorCapturedEvent = 907 };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
struct Stream {
    bool gone = false, captured = false;
    int queued = 0, done = 0;
};
struct Event {
    Stream *st = nullptr;
    int at = 0;
};
using hipStream_t = Stream *;
using hipEvent_t = Event *;
inline int g_mallocs = 0, g_frees = 0, g_events = 0;

inline hipError_t hipHostMalloc(void **p, size_t n, int) { ++g_mallocs; *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void *p) { ++g_frees; std::free(p); return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t *e) { ++g_events; *e = new Event; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, int) { return hipEventCreate(e); }
inline hipError_t hipEventDestroy(hipEvent_t e) { --g_events; delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (s->gone) return hipErrorInvalidHandle;
    e->st = s;
    e->at = s->queued;
    return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e)
{
    if (!e->st) return hipSuccess;
    if (e->st->gone) return hipErrorInvalidHandle;
    if (e->st->captured) return hipErrorCapturedEvent;
    return e->st->done >= e->at ? hipSuccess : hipErrorNotReady;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) { return e->st && e->st->gone ? hipErrorInvalidHandle : hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) { s->done = s->queued; return s->gone ? hipErrorInvalidHandle : hipSuccess; }
