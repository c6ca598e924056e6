// Device blocks with pinned host twins for the one-shot batched call's descriptor images,
// recycled once the call that used them has completed (its event has fired).  Blocks come in
// power-of-two sizes from 64 KiB and stay allocated for the process lifetime, so a steady
// stream of calls allocates nothing and never waits for the device.
#pragma once

#include <hip/hip_runtime_api.h>

#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace rr
{

class staging_pool
{
public:
    struct block
    {
        char*  dev    = nullptr;
        char*  host   = nullptr;
        size_t size   = 0;
        int    device = 0;
    };

    // A block of at least `bytes` on `device` (the current one) and an event for its use.  A
    // call that is being captured takes a free block as it is: asking an event of the
    // capturing stream, or waiting, would end the capture.
    hipError_t acquire(int device, size_t bytes, bool captured, block& b, hipEvent_t& ev)
    {
        size_t size = 64 << 10;
        while(size < bytes)
            size *= 2;
        std::lock_guard<std::mutex> lock(mu_);
        auto& fl = free_[std::make_pair(device, size)];
        if(!captured)
        {
            reclaim();
            if(fl.empty())
                recover(device);
        }
        if(!fl.empty())
        {
            b = fl.back();
            fl.pop_back();
        }
        else
        {
            b            = block{};
            b.size       = size;
            b.device     = device;
            hipError_t e = hipMalloc(reinterpret_cast<void**>(&b.dev), size);
            if(e != hipSuccess)
                return e;
            e = hipHostMalloc(reinterpret_cast<void**>(&b.host), size, hipHostMallocDefault);
            if(e != hipSuccess)
            {
                (void)hipFree(b.dev);
                return e;
            }
        }
        auto& evs = events_[device];
        if(!evs.empty())
        {
            ev = evs.back();
            evs.pop_back();
            return hipSuccess;
        }
        return hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    }

    // Hands the block back once `ev` (recorded after the block's last use) has fired.
    void release_after(const block& b, hipEvent_t ev)
    {
        std::lock_guard<std::mutex> lock(mu_);
        pending_.push_back(std::make_pair(b, ev));
    }

    // The block stays with a captured graph, which may be replayed at any time; its event
    // was not recorded.
    void leave_to_graph(const block& b, hipEvent_t ev)
    {
        std::lock_guard<std::mutex> lock(mu_);
        events_[b.device].push_back(ev);
    }

    // Takes back the blocks whose events have fired (a caller whose streams are drained and
    // about to be destroyed: an event cannot be asked once its stream is gone).
    void collect()
    {
        std::lock_guard<std::mutex> lock(mu_);
        reclaim();
    }

private:
    // An error that the caller has not read yet stays for it: nothing is asked then, and
    // otherwise the queries' own errors are not left for the next launch to report.
    void reclaim()
    {
        if(pending_.empty() || hipPeekAtLastError() != hipSuccess)
            return;
        size_t keep   = 0;
        bool   failed = false;
        for(size_t i = 0; i < pending_.size(); i++)
        {
            const hipError_t e = hipEventQuery(pending_[i].second);
            failed             = failed || e != hipSuccess;
            if(e == hipSuccess)
            {
                give_back(pending_[i].first);
                events_[pending_[i].first.device].push_back(pending_[i].second);
            }
            else if(e == hipErrorNotReady)
                pending_[keep++] = pending_[i];
            else // its stream is gone
                lost_.push_back(pending_[i]);
        }
        pending_.resize(keep);
        if(failed)
            (void)hipGetLastError();
    }

    // Blocks whose streams are gone: a wait for the whole device covers their last use.  Only
    // called where a block would have to be allocated otherwise.
    void recover(int device)
    {
        size_t of_device = 0;
        for(const auto& l : lost_)
            of_device += l.first.device == device ? 1 : 0;
        if(of_device == 0 || hipPeekAtLastError() != hipSuccess)
            return;
        if(hipDeviceSynchronize() != hipSuccess)
        {
            (void)hipGetLastError();
            return;
        }
        size_t keep = 0;
        for(size_t i = 0; i < lost_.size(); i++)
            if(lost_[i].first.device == device)
            {
                give_back(lost_[i].first);
                (void)hipEventDestroy(lost_[i].second);
            }
            else
                lost_[keep++] = lost_[i];
        lost_.resize(keep);
    }

    void give_back(const block& b) { free_[std::make_pair(b.device, b.size)].push_back(b); }

    std::mutex                                           mu_;
    std::map<std::pair<int, size_t>, std::vector<block>> free_;
    std::map<int, std::vector<hipEvent_t>>               events_;
    std::vector<std::pair<block, hipEvent_t>>            pending_;
    std::vector<std::pair<block, hipEvent_t>>            lost_;
};

} // namespace rr
