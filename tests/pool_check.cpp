// Checks of libsais_amd/csrc/copy_pool.h that need its parts: test_copy_pool_parts.py builds
// this with a sanitizer and runs one check by name.  Prints "ok" and returns 0, or says
// what is wrong.
#include "../libsais_amd/csrc/copy_pool.h"

#include <chrono>
#include <new>
#include <stdio.h>
#include <stdlib.h>

static std::atomic<int> g_fail_after{-1};   // allocations until every one fails; -1: none does

void *operator new(size_t n)
{
    if (g_fail_after >= 0 && g_fail_after-- == 0) {
        g_fail_after = 0;
        throw std::bad_alloc();
    }
    if (void *p = malloc(n)) return p;
    throw std::bad_alloc();
}
void *operator new[](size_t n) { return operator new(n); }
void operator delete(void *p) noexcept { free(p); }
void operator delete[](void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
void operator delete[](void *p, size_t) noexcept { free(p); }

namespace {

#define EXPECT(c)                                                                                  \
    do {                                                                                           \
        if (!(c)) {                                                                                \
            printf("line %d: %s\n", __LINE__, #c);                                                 \
            return 1;                                                                              \
        }                                                                                          \
    } while (0)

CopyPool &pool = *new CopyPool;   // (its workers live as long as the process)
// The stretch of a download by DMA: a slot of the staged copies' ring.
constexpr u64 SLOT = 8ull << 20;

// Every form of a staged copy, in the stretches that the engine grants: its parts fit the
// room that the job was given, and every entry arrives.
int copy_form(bool tiny, int conv, u64 entries, bool up, bool shared, bool dma = false)
{
    const u64 bytes = 4 * entries;
    const CopyForm f{tiny, conv, shared, !tiny && bytes >= (shared ? COPY_SHARED_LARGE : COPY_LARGE), dma};
    std::vector<u32> dev(entries);
    std::vector<int64_t> wide(entries);
    for (u64 i = 0; i < entries; i++) {
        dev[i] = up ? 0u : (u32)(i * 2654435761ull);
        wide[i] = up ? (int64_t)(u32)(i * 2654435761ull) : -1;
    }
    std::vector<u32> plain(entries);
    uint8_t *host = conv ? (uint8_t *)wide.data() : (uint8_t *)plain.data();
    if (up && !conv)
        for (u64 i = 0; i < entries; i++) plain[i] = (u32)wide[i];
    CopyPool::Job j(f.room(bytes));
    pool.begin(j, 4);
    u64 off = 0;
    for (int k = 0; off < bytes; k++) {
        u64 len = up ? f.up_chunk(k) : dma ? SLOT : f.down_chunk(bytes);
        len = bytes - off < len ? bytes - off : len;
        const bool ok = up ? pool.grant(j, {(uint8_t *)dev.data() + off, host + f.taken(off), len, conv}, f.up_part())
                           : pool.grant(j, {host + f.written(off), (const uint8_t *)dev.data() + off, f.written(len), conv},
                                        f.shared ? f.shared_part() : f.down_part(bytes));
        if (!ok) break;
        off += len;
    }
    pool.end(j);
    EXPECT(off == bytes);
    for (u64 i = 0; i < entries; i++) {
        const u32 v = (u32)(i * 2654435761ull);
        EXPECT(dev[i] == v);
        EXPECT(conv ? wide[i] == (int64_t)v : plain[i] == v);
    }
    return 0;
}

int forms()
{
    const u64 sizes[] = {1, 4095, 4096, 100003, 300007, 1u << 20, (8u << 20) + 1, (10u << 20) - 1, (10u << 20) + 4097};
    for (u64 n : sizes)
        for (int tiny = 0; tiny < 2; tiny++)
            for (int conv = 0; conv < 3; conv++)
                for (int how = 0; how < 5; how++) {   // upload or download, alone or beside others (4: by DMA)
                    const bool up = how < 2;
                    if (conv == (up ? 2 : 1)) continue;
                    if (n > 1u << 20 && tiny) continue;   // (the sizes of larger chunks and parts)
                    if (copy_form(tiny != 0, conv, n, up, how % 2 != 0 || how == 4, how == 4)) {
                        printf("entries %llu, tiny %d, conv %d, way %d\n", n, tiny, conv, how);
                        return 1;
                    }
                }
    return 0;
}

// A stretch of more parts than the job has left is refused whole.
int refused()
{
    std::vector<uint8_t> a(1 << 20, 7), b(1 << 20, 0);
    CopyPool::Job j(3);
    pool.begin(j, 2);
    EXPECT(pool.grant(j, {b.data(), a.data(), 100, 0}, 64));            // two parts
    EXPECT(!pool.grant(j, {b.data() + 100, a.data(), 128, 0}, 64));     // two more
    EXPECT(j.granted.load() == 2);
    EXPECT(pool.grant(j, {b.data() + 100, a.data(), 64, 0}, 64));
    EXPECT(!pool.grant(j, {b.data() + 164, a.data(), 1, 0}, 64));
    pool.end(j);
    for (int i = 0; i < 200; i++) EXPECT(b[i] == (i < 164 ? 7 : 0));
    return 0;
}

// Callers with different thread counts at once: one waits for its parts while another
// starts more workers.
int counts()
{
    CopyPool &p = *new CopyPool;
    constexpr u64 LEN = 8ull << 20;
    std::vector<std::thread> ts;
    std::atomic<int> wrong{0};
    for (int k = 1; k <= 6; k++)
        ts.emplace_back([&, k] {
            std::vector<uint8_t> a(LEN + k, (uint8_t)k), b(LEN + k, 0);
            for (int q = 0; q < 4; q++) {
                p.copy(b.data(), a.data(), a.size(), 2 * k);
                if (a != b) wrong++;
                memset(b.data(), 0, b.size());
            }
        });
    for (auto &t : ts) t.join();
    EXPECT(wrong == 0);
    return 0;
}

// A job's thread count caps the workers that take its parts, however many there are:
// with one thread the caller copies alone.
int limits()
{
    CopyPool &p = *new CopyPool;
    constexpr u64 LEN = 64ull << 20, PER = 64 << 10;
    std::vector<uint8_t> a(LEN, 5), b(LEN, 0);
    p.copy(b.data(), a.data(), LEN, 8);   // seven workers from here on
    for (int threads = 1; threads <= 4; threads++) {
        memset(b.data(), 0, LEN);
        CopyPool::Job j(CopyPool::parts_of(LEN, PER));
        p.begin(j, threads);
        EXPECT(p.grant(j, {b.data(), a.data(), LEN / 2, 0}, PER));
        EXPECT(p.grant(j, {b.data() + LEN / 2, a.data() + LEN / 2, LEN / 2, 0}, PER));
        int most = 0, done = 0;
        for (int k = 0; k < 50; k++) {   // the workers by themselves
            std::this_thread::sleep_for(std::chrono::milliseconds(1));
            most = std::max(most, j.users.load());
        }
        for (u64 k = 0; k < LEN / PER; k++) done += j.done[k].load();
        EXPECT(most <= threads - 1);
        EXPECT(threads > 1 ? done > 0 : done == 0);
        p.end(j);
        EXPECT(a == b);
    }
    // a job without workers beside one that has them
    CopyPool::Job j1(1), j2(1);
    p.begin(j1, 1);
    p.begin(j2, 2);
    EXPECT(p.grant(j1, {b.data(), a.data(), 64, 0}, 64));
    EXPECT(p.grant(j2, {b.data() + 64, a.data(), 64, 0}, 64));
    for (int k = 0; k < 5000 && !j2.done[0].load(); k++) std::this_thread::sleep_for(std::chrono::milliseconds(1));
    EXPECT(j2.done[0].load() && !j1.done[0].load());
    p.end(j1);
    p.end(j2);
    return 0;
}

// A copy finishes, and throws nothing, wherever the memory for its job or its threads ends.
int no_memory()
{
    constexpr u64 LEN = 3ull << 20;
    std::vector<uint8_t> a(LEN, 9), b(LEN);
    for (int k = 0; k < 8; k++) {
        CopyPool &p = *new CopyPool;
        memset(b.data(), 0, LEN);
        bool threw = false;
        g_fail_after = k;
        try {
            p.copy(b.data(), a.data(), LEN, 3);
        } catch (...) {
            threw = true;
        }
        g_fail_after = -1;
        EXPECT(!threw && a == b);
    }
    return 0;
}

} // namespace

int main(int argc, char **argv)
{
    const struct { const char *name; int (*run)(); } checks[] = {{"forms", forms}, {"refused", refused}, {"counts", counts}, {"limits", limits},
                                                         {"no_memory", no_memory}};
    for (const auto &c : checks)
        if (argc > 1 && !strcmp(argv[1], c.name)) {
            const int rc = c.run();
            if (!rc) printf("ok\n");
            return rc;
        }
    printf("no such check\n");
    return 2;
}
