// The kept device blocks (burn_automata_amd/csrc/npa_blocks.hpp) over a host allocator with a budget.
#include "../../burn_automata_amd/csrc/npa_blocks.hpp"

#include <stdio.h>
#include <stdlib.h>

#include <map>
#include <thread>

struct FakeMemory {
    using Error = int;  // 0 success, 2 out of memory
    static std::mutex mutex;
    static std::map<void*, size_t> live;
    static size_t used, budget;
    static int frees;
    static Error alloc(void** p, size_t bytes) {
        std::lock_guard<std::mutex> lock(mutex);
        *p = nullptr;
        if (used + bytes > budget) return 2;
        used += bytes;
        *p = malloc(1);
        live[*p] = bytes;
        return 0;
    }
    static void free(void* p) {
        std::lock_guard<std::mutex> lock(mutex);
        if (!live.count(p)) {
            printf("freed twice\n");
            exit(1);
        }
        used -= live[p];
        live.erase(p);
        ::free(p);
        ++frees;
    }
    static bool ok(Error e) { return e == 0; }
    static bool out_of_memory(Error e) { return e == 2; }
};
std::mutex FakeMemory::mutex;
std::map<void*, size_t> FakeMemory::live;
size_t FakeMemory::used = 0, FakeMemory::budget = 0;
int FakeMemory::frees = 0;

using Pool = npa::BlockPool<FakeMemory>;
using Block = Pool::Block;
constexpr size_t MB = (size_t)1 << 20;

#define CHECK(c)                                                   \
    do {                                                           \
        if (!(c)) {                                                \
            printf("line %d: %s\n", __LINE__, #c);                 \
            exit(1);                                               \
        }                                                          \
    } while (0)

static Block take(Pool& pool, size_t bytes) {
    Block b;
    CHECK(pool.acquire(bytes, &b) == 0 && b.ptr && b.bytes >= bytes);
    return b;
}

static void reuse() {
    FakeMemory::budget = 100000 * MB;
    Pool pool;
    Block a = take(pool, 100 * MB + 1);
    CHECK(a.bytes == 102 * MB);
    pool.release(a);
    CHECK(take(pool, 102 * MB).ptr == a.ptr);
    pool.release(a);
    Block b = take(pool, 50 * MB);  // less than half of it
    CHECK(b.ptr != a.ptr);
    Block c = take(pool, 51 * MB);
    CHECK(c.ptr == a.ptr);
    pool.release(b);
    pool.release(c);
    CHECK(FakeMemory::used == 152 * MB);
}

static void out_of_memory() {
    FakeMemory::budget = 1000 * MB;
    Pool one, two;
    one.release(take(one, 400 * MB));
    two.release(take(two, 500 * MB));
    void* p = nullptr;
    CHECK(Pool::allocate(&p, 700 * MB) == 0 && p && FakeMemory::used == 700 * MB);  // a workspace: both pools give back
    void* q = nullptr;
    CHECK(Pool::allocate(&q, 400 * MB) == 2 && !q);
    FakeMemory::free(p);
    one.release(take(one, 600 * MB));
    Block b = take(two, 900 * MB);  // a state of another context
    CHECK(FakeMemory::used == b.bytes);
    FakeMemory::free(b.ptr);
    Block none{(void*)&b, 1};
    CHECK(one.acquire(2000 * MB, &none) == 2 && !none.ptr && !none.bytes);
}

static void bounds() {
    FakeMemory::budget = 100000 * MB;
    Pool pool;
    Block b[6];
    for (int k = 0; k < 6; ++k) b[k] = take(pool, (size_t)(k + 1) * 40 * MB);
    for (int k = 0; k < 6; ++k) pool.release(b[k]);
    CHECK(FakeMemory::live.size() == Pool::kBlocks);
    Block big = take(pool, 3000 * MB);
    pool.release(big);
    CHECK(FakeMemory::used <= Pool::kBytes);
    Block x = take(pool, 700 * MB), y = take(pool, 600 * MB);
    pool.release(x);
    pool.release(y);
    CHECK(FakeMemory::used <= Pool::kBytes);
}

static void oldest_leaves() {  // sizes that are no longer asked for make room
    FakeMemory::budget = 100000 * MB;
    Pool pool;
    Block b[5];
    for (int k = 0; k < 4; ++k) b[k] = take(pool, (size_t)(k + 1) * 4 * MB);
    for (int k = 0; k < 4; ++k) pool.release(b[k]);
    b[4] = take(pool, 200 * MB);
    pool.release(b[4]);
    CHECK(FakeMemory::live.size() == 4 && !FakeMemory::live.count(b[0].ptr));
    CHECK(take(pool, 200 * MB).ptr == b[4].ptr);
    pool.release(b[4]);
    Block wide = take(pool, 900 * MB);
    pool.release(wide);
    CHECK(FakeMemory::used <= Pool::kBytes && take(pool, 900 * MB).ptr == wide.ptr);
    pool.release(wide);
}

static void threads() {
    FakeMemory::budget = 2000 * MB;
    Pool one, two;
    auto work = [](Pool* pool, size_t mb) {
        for (int k = 0; k < 2000; ++k) {
            Block b;
            if (pool->acquire((mb + (size_t)k % 7 * 30) * MB, &b) == 0) pool->release(b);
            void* p = nullptr;
            if (Pool::allocate(&p, 900 * MB) == 0) FakeMemory::free(p);
        }
    };
    std::thread t[4] = {std::thread(work, &one, 100), std::thread(work, &one, 200), std::thread(work, &two, 300),
                        std::thread(work, &two, 50)};
    for (auto& x : t) x.join();
}

int main() {
    for (auto f : {reuse, out_of_memory, bounds, oldest_leaves, threads}) {
        f();
        CHECK(FakeMemory::live.empty() && FakeMemory::used == 0);  // the pools gave everything back
    }
    printf("blocks ok\n");
    return 0;
}
