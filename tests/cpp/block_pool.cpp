// BlockPool (device memory kept for reuse) on a counted, bounded host memory:
// reuse and its slack, the bounds on what is held, the give-back on trim, on
// close, on a failed allocation, and of blocks that outlive a close.
#include <cstdio>
#include <cstdlib>
#include <set>
#include <stdexcept>
#include "pool.hpp"

struct Memory {
    static std::map<char*, size_t> live;
    static size_t used, capacity;
    static void* alloc(size_t bytes)
    {
        if (used + bytes > capacity) return nullptr;
        char* p = new char[1];
        live[p] = bytes;
        used += bytes;
        return p;
    }
    static void free(void* q)
    {
        char* p = static_cast<char*>(q);
        if (!live.count(p)) { std::puts("freed twice"); std::exit(1); }
        used -= live[p];
        live.erase(p);
        delete[] p;
    }
    [[noreturn]] static void short_of_memory() { throw std::bad_alloc(); }
};
std::map<char*, size_t> Memory::live;
size_t Memory::used = 0, Memory::capacity = size_t(16) << 30;

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main()
{
    typedef dmhm::BlockPool<Memory> Pool;
    const size_t G = size_t(1) << 30;
    Pool pool;
    pool.open();
    // Reuse up to a quarter larger, never smaller.
    void* a = pool.get(1000);
    CHECK(Memory::used == 1024);
    pool.put(a);
    CHECK(Memory::used == 1024);
    CHECK(pool.get(820) == a);              // 1,024 bytes for 1,024
    pool.put(a);
    CHECK(pool.get(1025) != a);
    CHECK(pool.get(512) != a);              // twice as large
    CHECK(pool.get(1024) == a);
    // One user at a time.
    CHECK(pool.get(1024) != a);
    // Bounds: blocks of at most 2 GiB, 4 GiB in all.
    void* big = pool.get(2 * G + 1);
    size_t before = Memory::used;
    pool.put(big);
    CHECK(Memory::used == before - (2 * G + 256));
    void* b[4];
    for (void*& p : b) p = pool.get(3 * G / 2);
    before = Memory::used;
    for (void* p : b) pool.put(p);
    CHECK(Memory::used == before - 3 * G);  // two of the four are held
    // Given back on request, ...
    pool.trim();
    CHECK(Memory::used == before - 6 * G);
    // ... before an allocation fails, ...
    void* c = pool.get(2 * G);
    pool.put(c);
    void* d = pool.get(Memory::capacity - Memory::used + G);
    pool.put(d);
    c = pool.get(2 * G);
    pool.put(c);
    d = pool.outside(Memory::capacity - Memory::used + G);
    Memory::free(d);
    c = pool.get(2 * G);
    pool.put(c);
    bool thrown = false;
    try { pool.get(Memory::capacity); } catch (const std::bad_alloc&) { thrown = true; }
    CHECK(thrown);
    before = Memory::used;
    pool.trim();
    CHECK(Memory::used == before);          // the failed one had given it back
    // ... and on close; what is put later, also after another open, is not held:
    // its device may be another one.
    void* e = pool.get(G);
    void* f = pool.get(G);
    pool.put(pool.get(G));
    pool.close();
    before = Memory::used;
    pool.put(e);
    CHECK(Memory::used == before - G);
    pool.open();
    pool.put(f);
    CHECK(Memory::used == before - 2 * G);
    void* h = pool.get(G);
    pool.put(h);
    CHECK(pool.get(G) == h);
    std::puts("ok");
    return 0;
}
