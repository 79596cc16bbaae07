// The leased scratch (sme-gemm_amd/csrc/lease_pool.h) on the CPU with a recording
// allocator: one holder at a time per (device, stream), other streams
// independent, outgrown and evicted buffers given back, both bounds kept. Built
// and run by tests/test_host_logic.py under AddressSanitizer and UBSan.
#include <atomic>
#include <cassert>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "../../sme-gemm_amd/csrc/lease_pool.h"

struct Recorder {
    std::atomic<int> *held;
    bool *fail;
    void *acquire(int, size_t bytes) {
        if (*fail) return nullptr;
        ++*held;
        return std::malloc(bytes);
    }
    void release(int, void *p) {
        --*held;
        std::free(p);
    }
};
typedef smg::LeasePool<Recorder> Pool;
static Pool::Lease take(Pool &p, int device, size_t stream, size_t bytes) {
    return p.take(device, (const void *)(stream * 16), bytes);
}

int main() {
    std::atomic<int> held{0};
    bool fail = false;
    {
        Pool pool(3, (size_t)8 << 20, Recorder{&held, &fail});
        void *a;
        {
            Pool::Lease l = take(pool, 0, 1, 1000);
            assert((a = l.buf()) != nullptr);
            // another stream and another device while it is held: their own
            Pool::Lease l2 = take(pool, 0, 2, 10), l3 = take(pool, 1, 1, 10);
            assert(l2.buf() && l3.buf() && l2.buf() != a && l3.buf() != a && l2.buf() != l3.buf());
            // a fourth stream while all are held: no room
            assert(!take(pool, 0, 3, 10).buf() && pool.streams() == 3);
        }
        assert(take(pool, 0, 1, 1 << 20).buf() == a);
        // a fourth stream evicts the least recently used (0, 2)
        assert(take(pool, 0, 3, 10).buf() && pool.streams() == 3 && held == 3);
        assert(take(pool, 0, 1, 10).buf() == a);
        // growth gives the outgrown buffer back (as many are held), sizes
        // are powers of two
        assert(take(pool, 0, 1, (3 << 20) + 5).buf() && pool.bytes() == (size_t)6 << 20 && held == 3);
        // past the byte bound others go first; one that can never fit is refused
        assert(take(pool, 0, 1, (size_t)8 << 20).buf() && pool.bytes() == (size_t)8 << 20 && held == 1);
        assert(!take(pool, 0, 1, ((size_t)8 << 20) + 1).buf());
        // a failed allocation: empty, and the next call tries again
        fail = true;
        assert(!take(pool, 0, 9, 10).buf());
        fail = false;
        assert(take(pool, 0, 9, 10).buf());
    }
    assert(held == 0);
    // Threads on one stream: nobody sees the buffer change while it is held
    // (as pack and product must not be parted by another call's pack).
    {
        Pool pool(2, (size_t)64 << 20, Recorder{&held, &fail});
        std::atomic<int> wrong{0};
        std::vector<std::thread> ts;
        for (int t = 0; t < 8; t++)
            ts.emplace_back([&, t] {
                for (int i = 0; i < 400; i++) {
                    const size_t n = 64 + (size_t)(i % 7 == 0 ? i : 0) * 8192;
                    Pool::Lease l = take(pool, 0, t % 3, n);
                    unsigned char *p = (unsigned char *)l.buf();
                    if (!p) continue;  // three streams on two entries
                    std::memset(p, t, 64);
                    std::this_thread::yield();
                    for (int j = 0; j < 64; j++) wrong += p[j] != t;
                }
            });
        for (std::thread &t : ts) t.join();
        assert(wrong == 0);
    }
    assert(held == 0);
    std::printf("lease pool ok\n");
    return 0;
}
