// copy_pool.h -- host copies split over worker threads, and the shape of the staged copies
// that use them (engine.hip).  Plain C++ without GPU code, so host programs can include it
// by itself.
#pragma once

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

typedef unsigned long long u64;
typedef uint32_t u32;

namespace {

// Copies split over worker threads.  Workers are detached and live until the process
// ends; a forked child starts a new pool.  Parts are small (128 KiB take a thread about
// 40 us while 16 of them share the memory), so that the first ones are soon ready for
// the DMA; they are taken and reported without a lock, and a thread looks for the next
// one for some time before it sleeps (waking one takes longer than a part).
class CopyPool {
  public:
    struct Part {
        uint8_t *d;
        const uint8_t *s;
        u64 len;     // bytes written
        int conv;    // 0: bytes; 1: int64 narrowed to u32; 2: u32 widened to int64
    };
    // At most `most` parts, granted by the owner in order as they become ready, taken in
    // that order, and done in any.
    struct Job {
        explicit Job(u64 most) : part(most), done(new std::atomic<char>[most])
        {
            for (u64 k = 0; k < most; k++) done[k].store(0, std::memory_order_relaxed);
        }
        std::vector<Part> part;
        std::unique_ptr<std::atomic<char>[]> done;
        std::atomic<int> granted{0}, next{0}, users{0};
        std::atomic<bool> closing{false};
        int limit = 0;    // workers that may be on it at once; set before it is opened
        int prefix = 0;   // the owner's: parts [0, prefix) are done
    };

  private:
    std::mutex m;   // open, sleeping; workers grow under it
    std::condition_variable work_cv;
    std::vector<Job *> open;
    std::atomic<int> sleeping{0};
    std::atomic<u32> epoch{0};   // grants so far, of all jobs
    std::atomic<int> opens{0};   // jobs in `open`
    std::atomic<int> workers{0};

    static void run(const Part &p)
    {
        if (p.conv == 1) {
            const int64_t *s = (const int64_t *)p.s;
            u32 *d = (u32 *)p.d;
            for (u64 i = 0; i < p.len / 4; i++) d[i] = (u32)s[i];
        } else if (p.conv == 2) {
            const u32 *s = (const u32 *)p.s;
            int64_t *d = (int64_t *)p.d;
            for (u64 i = 0; i < p.len / 8; i++) d[i] = (int64_t)s[i];
        } else {
            memcpy(p.d, p.s, p.len);
        }
    }
    // Takes and runs one part, if there is one.
    static bool take(Job &j)
    {
        int k = j.next.load();
        while (k < j.granted.load())
            if (j.next.compare_exchange_weak(k, k + 1)) {
                run(j.part[k]);
                j.done[k].store(1, std::memory_order_release);
                return true;
            }
        return false;
    }
    // m is held (users only grow under it): of the jobs with parts to take and room for one
    // more thread, one with the fewest threads
    Job *find()
    {
        Job *best = nullptr;
        for (Job *j : open)
            if (j->next.load() < j->granted.load() && j->users.load() < j->limit &&
                (!best || j->users.load() < best->users.load()))
                best = j;
        return best;
    }
    void loop()
    {
        std::unique_lock<std::mutex> lk(m);
        for (;;) {
            Job *j = find();
            if (!j) {   // look out for a grant for some 50 us, then sleep
                const u32 seen = epoch.load();
                lk.unlock();
                for (int k = 0; k < 2000 && epoch.load() == seen; k++) __builtin_ia32_pause();
                lk.lock();
                if (epoch.load() != seen) continue;
                sleeping++;
                work_cv.wait(lk, [&] { return (j = find()) != nullptr; });
                sleeping--;
            }
            j->users++;
            lk.unlock();
            // (with other jobs open, back to look there at once)
            for (int idle = 0; idle < (opens.load() > 1 ? 20 : 2000) && !j->closing.load(); idle++) {
                if (take(*j)) idle = 0;
                else __builtin_ia32_pause();
            }
            j->users--;
            lk.lock();
        }
    }

  public:
    // Opens a job (no parts yet) for up to `threads` threads, the owner (who takes parts, too)
    // among them; fewer where the system gives no more.
    void begin(Job &j, int threads)
    {
        j.limit = threads - 1;
        std::lock_guard<std::mutex> lk(m);
        open.push_back(&j);
        opens++;
        try {
            while (workers.load() < threads - 1) {
                std::thread([this] { loop(); }).detach();
                workers++;
            }
        } catch (const std::exception &) {
        }
    }
    void end(Job &j)   // waits for every part granted, and for the workers to leave the job
    {
        wait(j, j.granted.load());
        j.closing.store(true);
        {
            std::lock_guard<std::mutex> lk(m);
            open.erase(std::find(open.begin(), open.end(), &j));
            opens--;
        }
        while (j.users.load() > 0) __builtin_ia32_pause();
    }
    // Grants a stretch in parts of `per` written bytes.  False, and nothing granted, when
    // the job has no room for them.
    bool grant(Job &j, Part all, u64 per)
    {
        const u64 sper = all.conv == 1 ? 2 * per : all.conv == 2 ? per / 2 : per;
        int g = j.granted.load();
        const int g0 = g;
        if (parts_of(all.len, per) > j.part.size() - (u64)g) return false;
        for (; all.len; all.d += per, all.s += sper) {
            Part p = all;
            p.len = all.len < per ? all.len : per;
            all.len -= p.len;
            j.part[g++] = p;
        }
        j.granted.store(g);
        // All workers that may join it are called (more parts follow soon), and beside other
        // jobs at most one a part.  (At the limit none: a worker that leaves the job looks for
        // parts again.)
        int call = j.limit - j.users.load();
        if (call <= 0) return true;
        epoch++;
        if (sleeping.load() > 0) {
            { std::lock_guard<std::mutex> lk(m); }
            if (opens.load() <= 1) work_cv.notify_all();
            else for (call = std::min(call, g - g0); call > 0; call--) work_cv.notify_one();
        }
        return true;
    }
    // Waits until parts [0, upto) are done; takes parts itself when that is not soon, or at
    // once while other jobs want the workers, too.
    void wait(Job &j, int upto)
    {
        for (int idle = 0; j.prefix < upto; idle++) {
            if (j.done[j.prefix].load(std::memory_order_acquire)) {
                j.prefix++;
                idle = 0;
            } else if (idle < 2000 && workers.load() > 0 && j.limit > 0 && opens.load() <= 1) {
                __builtin_ia32_pause();
            } else if (!take(j)) {
                std::this_thread::yield();
            }
        }
    }
    static u64 parts_of(u64 len, u64 per) { return (len + per - 1) / per; }
    // (where there is no memory for the job, the caller copies alone)
    void copy(void *d, const void *s, u64 len, int threads)
    try {
        if (threads <= 1 || len < (1u << 20)) {
            memcpy(d, s, len);
            return;
        }
        // parts of whole pages, at least 1 MiB
        u64 per = (len + threads - 1) / threads;
        per = per < (1u << 20) ? (1u << 20) : (per + 4095) & ~(u64)4095;
        Job j(parts_of(len, per));
        begin(j, threads);
        if (!grant(j, Part{(uint8_t *)d, (const uint8_t *)s, len, 0}, per)) memcpy(d, s, len);
        end(j);
    } catch (const std::bad_alloc &) {
        memcpy(d, s, len);
    }
    void lock() { m.lock(); }
    void unlock() { m.unlock(); }
};

constexpr u64 COPY_MID = 32ull << 20, COPY_LARGE = 40ull << 20, COPY_SHARED_LARGE = 8ull << 20;   // device bytes

// The shape of one staged copy: settled when it starts, since the options may change while
// it runs.  Sizes are device bytes where nothing else is said; conv is Part::conv.
struct CopyForm {
    bool tiny;    // 64 KiB chunks of 16 KiB parts, whatever the size (host_staging 2)
    int conv;
    bool shared;  // other calls are under way
    bool large;   // passes through the larger ring
    bool dma;     // a download by DMA, in slots (else by a kernel, in chunks)

    u64 written(u64 bytes) const { return conv == 2 ? 2 * bytes : bytes; }   // by the host copies
    u64 taken(u64 bytes) const { return conv == 1 ? 2 * bytes : bytes; }     // from the caller's array
    // Upload chunk k.  The first ones are small, so that DMA and host copies overlap from
    // early on; later ones keep the DMA's start-up small beside it (a 4 MiB chunk takes 73 us).
    // Beside other calls, whose DMAs run meanwhile, whole stretches.
    u64 up_chunk(int k) const
    {
        if (tiny) return 64u << 10;
        if (shared) return 16ull << 20;
        if (large) return k < 3 ? (2ull << 20) << k : 16ull << 20;
        return k < 4 ? (512ull << 10) << k : k < 8 ? 4ull << 20 : 8ull << 20;
    }
    // Chunk of a download of `bytes`.
    u64 down_chunk(u64 bytes) const { return tiny ? 64u << 10 : bytes < COPY_MID ? 1u << 20 : 4u << 20; }
    // Written bytes of a part: of an upload (beside other calls larger ones: 8 threads in
    // libsais_lcp of 4 M entries each 42 ms with 128 KiB, 37 with 1 MiB),
    u64 up_part() const { return written(tiny ? 16u << 10 : shared ? 1u << 20 : 128u << 10); }
    // of a download of `bytes` (larger parts from COPY_MID on, so that fewer threads fault in
    // one huge page of an array not touched before: 64 MB 1.69 -> 1.45 ms, 192 MB 4.75 -> 3.96,
    // touched arrays the same; 16 MB 0.38 -> 0.51 ms, as the threads then have too few; nor for
    // 64-bit arrays, which wait for the threads: libsais64, libsais64_plcp and libsais64_lcp of
    // 12,000,001 symbols 10.7 -> 11.2 ms, and 12.7 -> 11.9 into arrays not touched before),
    u64 down_part(u64 bytes) const
    {
        return written(tiny ? 16u << 10 : bytes < COPY_MID || conv == 2 ? 128u << 10 : 512u << 10);
    }
    // and of one beside other calls.
    u64 shared_part() const { return tiny ? written(16u << 10) : 1u << 20; }
    // Room for the parts of a copy of `bytes`: every stretch that is granted may end in a
    // short one, and no part or stretch but the last is smaller than the least of any form.
    u64 room(u64 bytes) const
    {
        return CopyPool::parts_of(written(bytes), tiny ? 16u << 10 : 128u << 10) +
               CopyPool::parts_of(bytes, tiny ? 64u << 10 : 512u << 10);
    }
};

} // namespace
