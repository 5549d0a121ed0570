// Bookkeeping of the device-array pool (rrtmgp_hip_pool_malloc / _free, runtime.hip), kept free of HIP calls
// so that its rules can be unit-tested on the host.
//
// Unlike the scratch cache (cache_policy.h), the pool knows nothing of the streams that use an array: its
// callers hand arrays to any stream of the library and to other libraries.  hipFree, which it stands in for,
// waits for the whole device before memory changes hands; the pool keeps that promise at the reuse instead.
// A free takes the current generation; a device synchronisation starts a new generation, and once it has
// completed every block freed in an earlier one may be handed out again without waiting.  One wait so serves
// all arrays freed before it.  Blocks that need no wait are preferred.
//
// What the free list holds is bounded per device (the oldest blocks leave first and are given back to the
// driver); requests are served from blocks at most an eighth larger.
#ifndef RRTMGP_HIP_DEVICE_POOL_H
#define RRTMGP_HIP_DEVICE_POOL_H

#include <cstddef>
#include <cstdint>
#include <deque>
#include <unordered_map>
#include <vector>

namespace rrtmgp_hip
{
struct PoolBlock
{
    void* ptr = nullptr;
    size_t bytes = 0;
    int device = 0;
    uint64_t freed = 0;              // generation of the free
};

// Calls free_block for every block with its device current, by way of set_device, and leaves `current` so again.
// An error (a value other than 0) of either ends nothing; the first one is returned.
template<typename SetDevice, typename FreeBlock>
int for_each_on_device(const std::vector<PoolBlock>& blocks, int current, SetDevice set_device, FreeBlock free_block)
{
    int first = 0, device = current;
    const auto note = [&](int rc) { if (first == 0) first = rc; return rc == 0; };
    for (const PoolBlock& b : blocks)
    {
        if (b.device != device)
        {
            if (!note(set_device(b.device))) continue;
            device = b.device;
        }
        note(free_block(b));
    }
    if (device != current) note(set_device(current));
    return first;
}

class PoolPolicy
{
    public:
        // Allocation granularity: 512 B below 1 MiB, 2 MiB above (large mappings are cheaper whole).  Sizes that
        // no device holds, and whose rounding (or an eighth more) could wrap around, stay as they are.
        static size_t round_block(size_t bytes)
        {
            if (bytes > SIZE_MAX / 4) return bytes;
            const size_t q = bytes > (size_t(1) << 20) ? (size_t(2) << 20) : size_t(512);
            return (bytes + q - 1) / q * q;
        }

        // Takes a free block of the device for `bytes` (rounded): the smallest that needs no wait, else the
        // smallest at all, with wait = true.  The block becomes live.
        bool take(int device, size_t bytes, PoolBlock& out, bool& wait)
        {
            if (bytes > SIZE_MAX / 4) return false;
            const size_t most = bytes + (bytes >> 3);
            size_t best = free_.size();
            bool best_waits = true;
            for (size_t i = 0; i < free_.size(); ++i)
            {
                const PoolBlock& b = free_[i];
                if (b.device != device || b.bytes < bytes || b.bytes > most) continue;
                const bool w = b.freed >= safe_[device];
                if (best == free_.size() || (best_waits && !w) || (best_waits == w && b.bytes < free_[best].bytes))
                {
                    best = i;
                    best_waits = w;
                }
            }
            if (best == free_.size()) return false;
            out = free_[best];
            wait = best_waits;
            free_.erase(free_.begin() + std::ptrdiff_t(best));
            held_[device] -= out.bytes;
            live_[out.ptr] = out;
            return true;
        }

        void add_live(void* ptr, size_t bytes, int device)
        {
            PoolBlock b;
            b.ptr = ptr; b.bytes = bytes; b.device = device;
            live_[ptr] = b;
        }

        // A device synchronisation that is about to start; its number goes to waited() once it is done.
        uint64_t start_wait() { return ++generation_; }
        void waited(int device, uint64_t number)
        {
            uint64_t& s = safe_[device];
            if (number > s) s = number;
        }

        // Returns a live block to the free list; blocks that the bound pushes out go to `out` for the caller to
        // free (the block itself when it alone exceeds the bound).  False for a pointer that is not live.
        bool give(void* ptr, size_t bound, std::vector<PoolBlock>& out)
        {
            auto it = live_.find(ptr);
            if (it == live_.end()) return false;
            PoolBlock b = it->second;
            live_.erase(it);
            b.freed = generation_;
            if (b.bytes > bound)
            {
                out.push_back(b);
                return true;
            }
            size_t& held = held_[b.device];
            for (size_t i = 0; i < free_.size() && held + b.bytes > bound;)
            {
                if (free_[i].device != b.device) { ++i; continue; }
                held -= free_[i].bytes;
                out.push_back(free_[i]);
                free_.erase(free_.begin() + std::ptrdiff_t(i));
            }
            held += b.bytes;
            free_.push_back(b);
            return true;
        }

        // Empties the free list of every device.
        std::vector<PoolBlock> drain()
        {
            std::vector<PoolBlock> out(free_.begin(), free_.end());
            free_.clear();
            held_.clear();
            return out;
        }

        size_t held(int device) const
        {
            auto it = held_.find(device);
            return it == held_.end() ? 0 : it->second;
        }
        size_t n_live() const { return live_.size(); }

    private:
        // Generation 0 is never safe: the first reuse waits.
        uint64_t generation_ = 0;
        std::unordered_map<int, uint64_t> safe_;
        std::unordered_map<int, size_t> held_;
        std::deque<PoolBlock> free_;
        std::unordered_map<void*, PoolBlock> live_;
};
}  // namespace rrtmgp_hip

#endif
