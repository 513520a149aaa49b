// Memory that is kept between calls, and its return where memory is short.
// Nothing here names HIP: Memory is { static int alloc(void** p, size_t bytes,
// bool pinned) (0: done); static void release(void* p, bool pinned); }.
#pragma once

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <vector>

namespace bh {

// A holder of memory that no call needs to finish.
struct Spare {
    virtual void give_back() = 0;  // from any thread; at most what is idle
    virtual ~Spare() = default;
};

// Every holder, asked for its memory when an allocation fails.
class SpareList {
    std::mutex mu;
    std::vector<Spare*> all;

public:
    void add(Spare* s) {
        std::lock_guard<std::mutex> lk(mu);
        all.push_back(s);
    }
    void remove(Spare* s) {
        std::lock_guard<std::mutex> lk(mu);
        all.erase(std::remove(all.begin(), all.end(), s), all.end());
    }
    void give_back() {
        std::lock_guard<std::mutex> lk(mu);
        for (Spare* s : all) s->give_back();
    }
};
inline SpareList& spares() {
    static SpareList& list = *new SpareList;  // outlives whatever is destroyed at exit
    return list;
}

// Allocates; when that fails once more with what the holders gave back.
template <class Memory>
int alloc_or_reclaim(void** p, size_t bytes, bool pinned) {
    int rc = Memory::alloc(p, bytes, pinned);
    if (rc != 0) {
        spares().give_back();
        rc = Memory::alloc(p, bytes, pinned);
    }
    return rc;
}

// Device memory that its owner can do without: taken only where it is there
// without others giving theirs back, and given back when an allocation fails
// (an owner holds the lock while it queues work on the buffers; releasing them
// waits for that work).
template <class Memory>
class Extra : public Spare {
    std::mutex mu;
    std::vector<void*> bufs;

    void drop() {
        for (void* p : bufs) Memory::release(p, false);
        bufs.clear();
    }

public:
    Extra() = default;
    Extra(const Extra&) = delete;
    Extra& operator=(const Extra&) = delete;
    ~Extra() override {
        spares().remove(this);
        drop();
    }
    // the buffers of these sizes, or none
    void take(const std::vector<size_t>& bytes) {
        {
            std::lock_guard<std::mutex> lk(mu);
            for (size_t n : bytes) {
                void* p = nullptr;
                if (Memory::alloc(&p, n, false) != 0) return drop();
                bufs.push_back(p);
            }
        }
        spares().add(this);
    }
    std::unique_lock<std::mutex> hold() { return std::unique_lock<std::mutex>(mu); }
    bool there() const { return !bufs.empty(); }
    template <class T>
    T* as(size_t i) const {
        return static_cast<T*>(bufs[i]);
    }
    void give_back() override {
        std::unique_lock<std::mutex> lk(mu, std::try_to_lock);
        if (lk) drop();
    }
};

// Device and pinned host memory that a context's calls use while they run.
// A call used to allocate and free each of its buffers and to copy each result
// down by itself (a copy to pageable memory costs ~9 us of the host's time, a
// wait 11): draws, densities and estimates of 65,536 values took 247 us in six
// calls of which the kernels are 75, and take 137 with this.  The blocks are
// kept between calls, at most kDevMax + kPinMax bytes of them, the last ones
// used, and freed with the context; a call holds its blocks until its stream
// is idle, so any call on any stream of the context may use them next.
template <class Memory>
struct Pool : Spare {
    // kept at most, all blocks together and the largest of them; sizes up to
    // the latter are rounded to the next power of two
    static constexpr size_t kDevMax = (size_t)128 << 20, kDevBlock = (size_t)64 << 20;
    static constexpr size_t kPinMax = (size_t)4 << 20, kPinBlock = kPinMax;
    static constexpr size_t kBlocks = 64;
    struct Block {
        void* p;
        size_t bytes;
        bool pinned;
    };
    std::mutex mu;
    std::vector<Block> kept;  // the one put back last at the end
    size_t kept_bytes[2] = {0, 0};

    Pool() {
        kept.reserve(kBlocks);
        spares().add(this);
    }
    Pool(const Pool&) = delete;
    Pool& operator=(const Pool&) = delete;
    ~Pool() override {
        spares().remove(this);
        give_back();
    }
    static void release(const Block& b) { Memory::release(b.p, b.pinned); }
    void give_back() override {
        std::lock_guard<std::mutex> lk(mu);
        for (const Block& b : kept) release(b);
        kept.clear();
        kept_bytes[0] = kept_bytes[1] = 0;
    }
    int get(size_t bytes, bool pinned, Block* out) {
        size_t want = bytes;
        if (bytes <= (pinned ? kPinBlock : kDevBlock))
            for (want = 4096; want < bytes;) want *= 2;
        {
            std::lock_guard<std::mutex> lk(mu);
            for (size_t i = kept.size(); i-- > 0;) {
                if (kept[i].pinned != pinned || kept[i].bytes != want) continue;
                *out = kept[i];
                kept_bytes[pinned] -= want;
                kept.erase(kept.begin() + i);
                return 0;
            }
        }
        *out = Block{nullptr, want, pinned};
        return alloc_or_reclaim<Memory>(&out->p, want, pinned);
    }
    // Keeps the block; the oldest ones make room for it.  Without that the
    // first large block, or 64 blocks of sizes that do not come again, took the
    // room for good, and every later call allocated and freed as before.
    void put(const Block& b) {
        if (b.bytes > (b.pinned ? kPinBlock : kDevBlock)) return release(b);
        const size_t most = b.pinned ? kPinMax : kDevMax;
        std::lock_guard<std::mutex> lk(mu);
        for (size_t i = 0; i < kept.size();) {
            const bool room = kept_bytes[b.pinned] + b.bytes <= most;
            if (room && kept.size() < kBlocks) break;
            if (!room && kept[i].pinned != b.pinned) {
                ++i;
                continue;
            }
            release(kept[i]);
            kept_bytes[kept[i].pinned] -= kept[i].bytes;
            kept.erase(kept.begin() + i);
        }
        kept_bytes[b.pinned] += b.bytes;
        kept.push_back(b);
    }
};

}  // namespace bh
