// Test harness only: the product's block pool (csrc/devpool.h) over a counted
// stand-in for device memory.
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>

#include "../../bellhopcuda_amd/csrc/devpool.h"

namespace {
// Addresses only (a block may be said to have gigabytes), each of its own.
struct FakeMem {
    static std::atomic<long long> live, allocs, frees, bad;
    static std::atomic<size_t> left;                // bytes before alloc fails
    static std::mutex mu;
    static std::unordered_map<void *, size_t> blocks;
    static int alloc(void **p, size_t n)
    {
        std::lock_guard<std::mutex> lk(mu);
        *p = nullptr;
        if(n > left) return 2;
        left -= n;
        *p = malloc(16);
        blocks[*p] = n;
        live += (long long)n;
        ++allocs;
        return 0;
    }
    static void free(void *p)
    {
        std::lock_guard<std::mutex> lk(mu);
        const auto it = blocks.find(p);
        if(it == blocks.end()) {
            ++bad;
            return;
        }
        left += it->second;
        live -= (long long)it->second;
        ++frees;
        blocks.erase(it);
        ::free(p);
    }
};
std::atomic<long long> FakeMem::live{0}, FakeMem::allocs{0}, FakeMem::frees{0}, FakeMem::bad{0};
std::atomic<size_t> FakeMem::left{0};
std::mutex FakeMem::mu;
std::unordered_map<void *, size_t> FakeMem::blocks;
typedef BlockPool<FakeMem> Pool;
} // namespace

extern "C" {
void *pool_new(long long limit) { return new Pool((size_t)limit); }
void pool_delete(void *p) { delete static_cast<Pool *>(p); }
void mem_set(long long bytes) { FakeMem::left = (size_t)bytes; }
// address, or 0
long long pool_get(void *p, long long n)
{
    void *q = nullptr;
    return static_cast<Pool *>(p)->get(&q, (size_t)n) ? 0 : (long long)(intptr_t)q;
}
void pool_put(void *p, long long q) { static_cast<Pool *>(p)->put((void *)(intptr_t)q); }
void pool_trim(void *p) { static_cast<Pool *>(p)->trim(); }
long long pool_held(void *p) { return (long long)static_cast<Pool *>(p)->held(); }
// live bytes, allocations, frees, frees of what was not allocated
void mem_counts(long long *c)
{
    c[0] = FakeMem::live;
    c[1] = FakeMem::allocs;
    c[2] = FakeMem::frees;
    c[3] = FakeMem::bad;
}
// `threads` threads take and give back blocks of mixed sizes; returns how often
// one block was in two hands, or did not hold what was asked for.
int pool_stress(void *p, int threads, int rounds)
{
    std::mutex mu;
    std::unordered_map<void *, int> out;
    std::atomic<int> wrong{0};
    auto work = [&](int t) {
        unsigned r = 12345u + 7919u * (unsigned)t;
        for(int i = 0; i < rounds; ++i) {
            void *q[3];
            for(auto &b : q) {
                r = 1664525u * r + 1013904223u;
                const size_t n = (size_t)1 << (8 + r / 65536u % 22);
                if(static_cast<Pool *>(p)->get(&b, n)) {
                    ++wrong;
                    b = nullptr;
                    continue;
                }
                std::lock_guard<std::mutex> lk(mu);
                if(out[b]++) ++wrong;
                std::lock_guard<std::mutex> lm(FakeMem::mu);
                if(FakeMem::blocks[b] < n) ++wrong;
            }
            for(auto b : q) {
                if(!b) continue;
                {
                    std::lock_guard<std::mutex> lk(mu);
                    --out[b];
                }
                static_cast<Pool *>(p)->put(b);
            }
        }
    };
    std::vector<std::thread> ts;
    for(int t = 0; t < threads; ++t) ts.emplace_back(work, t);
    for(auto &t : ts) t.join();
    return wrong;
}
}
