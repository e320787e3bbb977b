// Device memory kept for reuse; the memory itself comes from `Mem` (hipMalloc
// and hipFree in the library).
#pragma once
#include <algorithm>
#include <cstddef>
#include <map>
#include <mutex>
#include <unordered_map>

namespace dmhm {

// Device memory of destroyed matrices and buffers, kept for the next ones: a
// product or a copy per step of a user's loop otherwise pays hipMalloc and
// hipFree (about 0.1 ms each, and a device synchronisation) every time. At most
// kHoldMax bytes are held, in blocks of at most kBlockMax; a request takes the
// smallest held block that is at most a quarter larger. All work of the library
// is ordered on one stream, so a block's old users are done before its new
// ones start. Everything held is given back by trim (dmhm_trim), by close
// (dmhm_finalize) and before an allocation is reported as failed; a block that
// outlives a close, whose device may then no longer be the library's, is given
// back when it is put. Batch of 24 products and applications (FP32, 48^2 and
// 64^2): 22 ms without, 12.4 with.
//
// Mem::alloc(bytes) returns null when memory is short and throws on other
// errors, Mem::free(p) does not throw, Mem::short_of_memory() throws.
template <typename Mem>
class BlockPool {
public:
    static constexpr size_t kHoldMax = size_t(4) << 30, kBlockMax = size_t(2) << 30;

    void* get(size_t bytes)
    {
        bytes = (std::max<size_t>(bytes, 1) + 255) & ~size_t(255);
        std::lock_guard<std::mutex> lk(mu_);
        auto it = held_.lower_bound(bytes);
        if (it != held_.end() && it->first - bytes <= bytes / 4) {
            void* p = it->second;
            holding_ -= it->first;
            held_.erase(it);
            return p;
        }
        void* p = raw(bytes);
        blocks_[p] = {bytes, epoch_};
        return p;
    }
    void put(void* p)
    {
        std::lock_guard<std::mutex> lk(mu_);
        const Block b = blocks_.at(p);
        if (open_ && b.epoch == epoch_ && b.bytes <= kBlockMax && holding_ + b.bytes <= kHoldMax) {
            held_.emplace(b.bytes, p);
            holding_ += b.bytes;
            return;
        }
        blocks_.erase(p);
        Mem::free(p);
    }
    // Memory that is not pooled (Mem::free gives it back), for plans' tables.
    void* outside(size_t bytes)
    {
        std::lock_guard<std::mutex> lk(mu_);
        return raw(bytes);
    }
    void trim()
    {
        std::lock_guard<std::mutex> lk(mu_);
        drop();
    }
    // Blocks put are held from open to close.
    void open()
    {
        std::lock_guard<std::mutex> lk(mu_);
        open_ = true;
    }
    void close()
    {
        std::lock_guard<std::mutex> lk(mu_);
        drop();
        open_ = false;
        ++epoch_;
    }

private:
    struct Block { size_t bytes; long epoch; };

    void* raw(size_t bytes)
    {
        void* p = Mem::alloc(bytes);
        if (!p && !held_.empty()) {
            drop();
            p = Mem::alloc(bytes);
        }
        if (!p) Mem::short_of_memory();
        return p;
    }
    void drop()
    {
        for (auto& h : held_) { blocks_.erase(h.second); Mem::free(h.second); }
        held_.clear();
        holding_ = 0;
    }

    std::mutex mu_;
    std::multimap<size_t, void*> held_;
    std::unordered_map<void*, Block> blocks_;   // every block handed out or held
    size_t holding_ = 0;
    long epoch_ = 0;                            // closes so far
    bool open_ = false;
};

} // namespace dmhm
