// Blocks of memory that runs gave back, kept for the next ones. Mem::alloc(void **,
// size_t) returns 0 or an error, Mem::free(void *) takes a block back for good.
//
// At most `limit` bytes are kept idle. A block that comes back is the one most
// likely to be asked for again, so room for it is made by freeing the largest
// other idle ones. Safe with several threads; blocks are allocated and freed
// outside the lock (freeing waits for the device).
#pragma once
#include <algorithm>
#include <cstddef>
#include <mutex>
#include <unordered_map>
#include <vector>

// Requests from this size on take any idle block that holds them, smaller ones
// only a block of at most twice their size (or 1 MiB): a small array must not
// occupy the block that a run's one large array needs.
constexpr size_t POOL_BIG = size_t(256) << 20;

template<typename Mem> class BlockPool {
    struct Block {
        void *p;
        size_t n;
    };
    std::mutex mu;
    std::vector<Block> idle;
    std::unordered_map<void *, size_t> size;    // of every block handed out or idle
    size_t idle_bytes = 0, limit;

    void *take(size_t i)
    {
        void *p = idle[i].p;
        idle_bytes -= idle[i].n;
        idle.erase(idle.begin() + (std::ptrdiff_t)i);
        return p;
    }

public:
    explicit BlockPool(size_t limit_) : limit(limit_) {}
    BlockPool(const BlockPool &) = delete;
    BlockPool &operator=(const BlockPool &) = delete;
    ~BlockPool() { trim(); }

    // (before the first block is handed out)
    void set_limit(size_t n) { limit = n; }

    // A block of at least n bytes: 0, or Mem::alloc's error.
    int get(void **p, size_t n)
    {
        n = (n + 255) / 256 * 256;
        const size_t most = n >= POOL_BIG ? (size_t)-1 : std::max(2 * n, size_t(1) << 20);
        {
            std::lock_guard<std::mutex> lk(mu);
            size_t best = idle.size();
            for(size_t i = 0; i < idle.size(); ++i)
                if(idle[i].n >= n && idle[i].n <= most && (best == idle.size() || idle[i].n < idle[best].n)) best = i;
            if(best < idle.size()) {
                *p = take(best);
                return 0;
            }
        }
        const int e = Mem::alloc(p, n);
        if(e) return e;
        std::lock_guard<std::mutex> lk(mu);
        size[*p] = n;
        return 0;
    }

    // Give a block of get() back (null: nothing).
    void put(void *p)
    {
        if(!p) return;
        std::vector<void *> gone;
        {
            std::lock_guard<std::mutex> lk(mu);
            const size_t n = size[p];
            if(n <= limit) {
                while(idle_bytes + n > limit) {
                    const auto it = std::max_element(idle.begin(), idle.end(),
                                                     [](const Block &a, const Block &b) { return a.n < b.n; });
                    gone.push_back(take((size_t)(it - idle.begin())));
                }
                idle.push_back({p, n});
                idle_bytes += n;
            } else {
                gone.push_back(p);
            }
            for(void *q : gone) size.erase(q);
        }
        for(void *q : gone) Mem::free(q);
    }

    // Free every idle block.
    void trim()
    {
        std::vector<Block> gone;
        {
            std::lock_guard<std::mutex> lk(mu);
            gone.swap(idle);
            idle_bytes = 0;
            for(const Block &b : gone) size.erase(b.p);
        }
        for(const Block &b : gone) Mem::free(b.p);
    }

    size_t held()
    {
        std::lock_guard<std::mutex> lk(mu);
        return idle_bytes;
    }
};
