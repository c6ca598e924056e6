// CPU harness of the batched calls' descriptor blocks (rocrand_amd/csrc/rr_staging.hpp) for
// tests/test_staging.py: the product's class over a stand-in for the HIP runtime that keeps a
// last error and answers event queries as the test says.
#include "rr_staging.hpp"

#include <cstdint>
#include <cstdlib>
#include <map>

namespace
{
hipError_t                last = hipSuccess;
std::map<void*, hipError_t> answer; // per event
int                       mallocs, syncs, queries;
hipError_t                sync_result = hipSuccess;

hipError_t done(hipError_t e)
{
    if(e != hipSuccess)
        last = e;
    return e;
}
} // namespace

extern "C" {

hipError_t hipMalloc(void** p, size_t n)
{
    mallocs++;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    static uintptr_t next = 0;
    *e                    = reinterpret_cast<hipEvent_t>(++next);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    answer.erase(e);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e)
{
    queries++;
    return done(answer[e]);
}
hipError_t hipDeviceSynchronize()
{
    syncs++;
    return done(sync_result);
}
hipError_t hipPeekAtLastError() { return last; }
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last               = hipSuccess;
    return e;
}

void* staging_new()
{
    last = sync_result = hipSuccess;
    mallocs = syncs = queries = 0;
    return new rr::staging_pool();
}

// One call's use of a block, captured into a graph or with an event that answers `query`
// from then on; returns its device address.
void* staging_use(void* pool, size_t bytes, int captured, int query)
{
    rr::staging_pool::block b;
    hipEvent_t              ev = nullptr;
    auto*                   p  = static_cast<rr::staging_pool*>(pool);
    if(p->acquire(0, bytes, captured != 0, b, ev) != hipSuccess)
        return nullptr;
    if(captured)
        p->leave_to_graph(b, ev);
    else
    {
        answer[ev] = static_cast<hipError_t>(query);
        p->release_after(b, ev);
    }
    return b.dev;
}
void staging_collect(void* pool) { static_cast<rr::staging_pool*>(pool)->collect(); }
void staging_set(int last_error, int sync) { last = static_cast<hipError_t>(last_error), sync_result = static_cast<hipError_t>(sync); }
void staging_counts(int* out) { out[0] = mallocs, out[1] = syncs, out[2] = queries, out[3] = last; }

} // extern "C"
