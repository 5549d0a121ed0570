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
#include <map>
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
            const auto at = devices_.find(device);
            if (at == devices_.end()) return false;
            Device& d = at->second;
            // A size's oldest block is the one that a wait has most likely covered.
            auto best = d.by_size.lower_bound(bytes);
            const auto end = d.by_size.upper_bound(bytes + (bytes >> 3));
            if (best == end) return false;
            const auto waits = [&](const std::deque<uint64_t>& ages) { return d.by_age.at(ages.front()).freed >= d.safe; };
            auto it = best;
            while (it != end && waits(it->second)) ++it;
            wait = it == end;
            if (!wait) best = it;
            const auto block = d.by_age.find(best->second.front());
            out = block->second;
            live_[out.ptr] = out;                        // before the block leaves the list: this may throw
            forget(d, block);
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
            uint64_t& s = devices_[device].safe;
            if (number > s) s = number;
        }

        // Returns a live block to the free list (the block stays live if there is no host memory for that); blocks that the bound pushes out go to `out` for the caller to
        // free (the block itself when it alone exceeds the bound).  False for a pointer that is not live.
        bool give(void* ptr, size_t bound, std::vector<PoolBlock>& out)
        {
            const auto it = live_.find(ptr);
            if (it == live_.end()) return false;
            PoolBlock b = it->second;
            b.freed = generation_;
            if (b.bytes > bound) out.push_back(b);
            else
            {
                Device& d = devices_[b.device];
                while (d.held + b.bytes > bound)
                {
                    out.push_back(d.by_age.begin()->second);
                    forget(d, d.by_age.begin());
                }
                const auto block = d.by_age.emplace(age_, b).first;
                try { d.by_size[b.bytes].push_back(age_); }
                catch (...) { d.by_age.erase(block); throw; }
                ++age_;
                d.held += b.bytes;
            }
            live_.erase(it);
            return true;
        }

        // Empties the free list of every device.
        std::vector<PoolBlock> drain()
        {
            std::vector<PoolBlock> out;
            size_t n = 0;
            for (const auto& d : devices_) n += d.second.by_age.size();
            out.reserve(n);
            for (auto& d : devices_)
            {
                for (const auto& b : d.second.by_age) out.push_back(b.second);
                d.second.by_age.clear();
                d.second.by_size.clear();
                d.second.held = 0;
            }
            return out;
        }

        size_t held(int device) const
        {
            const auto it = devices_.find(device);
            return it == devices_.end() ? 0 : it->second.held;
        }
        size_t held() const
        {
            size_t n = 0;
            for (const auto& d : devices_) n += d.second.held;
            return n;
        }
        size_t n_live() const { return live_.size(); }
        size_t live_bytes() const
        {
            size_t n = 0;
            for (const auto& b : live_) n += b.second.bytes;
            return n;
        }

    private:
        // A device's free blocks by their age (a running number) and, for each size, the ages oldest first: a
        // request looks at the sizes within an eighth of it, not at every block.
        struct Device
        {
            std::map<uint64_t, PoolBlock> by_age;
            std::map<size_t, std::deque<uint64_t>> by_size;
            size_t held = 0;
            uint64_t safe = 0;
        };

        // Only a size's oldest block is ever taken out.
        static void forget(Device& d, std::map<uint64_t, PoolBlock>::iterator block)
        {
            d.held -= block->second.bytes;
            const auto s = d.by_size.find(block->second.bytes);
            s->second.pop_front();
            if (s->second.empty()) d.by_size.erase(s);
            d.by_age.erase(block);
        }

        // Generation 0 is never safe: the first reuse waits.
        uint64_t generation_ = 0, age_ = 0;
        std::unordered_map<int, Device> devices_;
        std::unordered_map<void*, PoolBlock> live_;
};
}  // namespace rrtmgp_hip

#endif
