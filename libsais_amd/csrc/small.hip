// small.hip -- a whole build of a short byte text in one kernel.
//
// A text of a few thousand bytes has nothing to spread over 256 CUs: the general engine
// takes 40 to 70 launches and 5 to 7 host waits for it, of which each launch costs
// about 4.5 us whatever it does and each wait 10 to 30 us.  Up to SMALL_MAX bytes one
// workgroup of 1024 threads keeps everything in LDS and does all of it -- alphabet,
// initial sort, doubling rounds, BWT, PLCP, LCP -- with barriers (well under 1 us) in
// the place of launches.  libsais_bwt of 4001 bytes on host buffers: 415 -> 53 us; a GSA
// build (SA, LCP) of a 22,347-byte string on the device: 237 -> 111 us, 41 of them the
// three passes of the initial sort.  What bounds it is one CU: about 45 vector and 7 LDS
// instructions per element and pass.
//
// LDS (ROWS * 1024 positions, 6 bytes each, 160 KB hold 24 rows):
//   s_sa    u16  suffix of every slot
//   s_rank  u16  sort key of every suffix, then its rank (first slot of its group)
//   s_x     2 B  codes (1 B) and low key bytes (1 B) of the initial sort; key2 of every
//                slot in a round; codes again for BWT and PLCP
//   s_cnt        digit counters of every wave
//   s_bits       bit p: slot p starts a group (slots from n on count as starts)
//
// Order: element e of a pass is position w * 64 * ROWS + r * 64 + lane (wave w, row r),
// so that a wave's elements are consecutive and one ballot per row is one word of
// s_bits.
//
// 1. Codes of the present bytes, and keys of the first k0 symbols in base sigma
//    (sigma^k0 <= 2^24), in GSA mode zero from the first separator on: three stable
//    8-bit LSD passes in LDS.  GSA keys with a separator are alone in their group, in
//    order of position, as in the general engine.
// 2. Rounds with h = k0, 2 k0, ...: members of a group are ordered by the rank of the
//    suffix h further on (a suffix that ends before that comes first, the shorter one
//    first).  Groups of at most SM_COUNT members are ranked by counting; if a larger
//    one is left, the round sorts all slots by (group, key2), four LSD passes.
// 3. PLCP by Kasai's recurrence, every thread over its own stretch of the text: the
//    first position of a stretch compares from nothing, 8 symbols a step; a match past
//    32 symbols is finished by the whole wave, 512 symbols a step.
#include "engine.h"

namespace {

constexpr int SM_THREADS = 1024, SM_WAVES = SM_THREADS / SAGPU_WAVE;
// Largest group ranked by counting: a member costs its group's size in LDS reads (a round
// of 24 rows whose groups are below this takes 9 to 13 us); the four-pass sort of all
// slots takes 60 us there, whatever the groups are.
constexpr u32 SM_COUNT = 96;

template <int ROWS> struct SmallLds {
    static constexpr u32 N = ROWS * SM_THREADS;
    u16 sa[N];
    u16 rank[N];
    union {
        struct {
            uint8_t code[N + 64];   // zero past the text
            uint8_t low[N];
        } c;
        u16 key[N];
    } x;
    u16 cnt[SM_WAVES * 256];
    u64 bits[N / 64 + 1];
    u16 part[4][256];
    u32 present[256];
    uint8_t lut[256], inv[256];
    u64 ball[4];
    u32 flags, active, bad, wsum[4];
};

// Eight bytes at p + i of an LDS array (p 8-byte aligned), from three aligned words.
__device__ __forceinline__ u64 load8(const uint8_t *p, u32 i)
{
    const u32 *q = (const u32 *)p + (i >> 2);
    const u32 a = q[0], b = q[1], c = q[2];
    return (u64)__builtin_amdgcn_alignbyte(c, b, i & 3) << 32 | __builtin_amdgcn_alignbyte(b, a, i & 3);
}

// The compiler keeps what depends on a row's number in registers across the round loop
// (24 rows of addresses and bounds; it spilled 150 registers): a value it cannot see
// through at the start of each phase makes it compute them there.
__device__ __forceinline__ u32 opaque(u32 v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// Stable LSD pass over the n elements in slot order: src(p) = the suffix in slot p,
// digit(i) = suffix i's digit.
template <int ROWS, class Src, class Digit>
__device__ void small_pass(SmallLds<ROWS> &l, u32 n, Src src, Digit digit)
{
    const u32 tid = threadIdx.x, w = tid / SAGPU_WAVE, lane = lane_id();
    const u32 base = opaque(w * SAGPU_WAVE * ROWS + lane);
    for (u32 k = tid; k < SM_WAVES * 128; k += SM_THREADS) ((u32 *)l.cnt)[k] = 0;
    __syncthreads();
    u32 item[ROWS];   // suffix | rank among the wave's equal digits << 16
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const u32 p = base + r * SAGPU_WAVE;
        const bool ok = p < n;
        const u32 i = ok ? src(p) : 0u;
        const u32 d = ok ? digit(i) : 0u;
        const u64 m = wave_peers<8>(d, __ballot(ok));
        const u32 below = mask_below(m);
        u32 old = 0;
        if (ok) {
            old = l.cnt[w * 256 + d];
            l.cnt[w * 256 + d] = (u16)(old + (u32)__popcll(m));   // the same value from every peer
        }
        item[r] = i | (old + below) << 16;
    }
    __syncthreads();
    // First slot of every wave's run of every digit, into cnt: four threads per digit sum
    // four waves' counts each.
    constexpr u32 QW = SM_WAVES / 4;
    const u32 d = tid & 255, quarter = tid >> 8;
    u32 own[QW], sum = 0;
#pragma unroll
    for (u32 q = 0; q < QW; q++) {
        own[q] = l.cnt[(quarter * QW + q) * 256 + d];
        sum += own[q];
    }
    l.part[quarter][d] = (u16)sum;
    __syncthreads();
    u32 tot = 0, before = 0;   // the digit's count, and that of the waves before this quarter's
#pragma unroll
    for (u32 q = 0; q < 4; q++) {
        const u32 c = l.part[q][d];
        tot += c;
        before += q < quarter ? c : 0u;
    }
    const u32 inc = wave_incl_sum(tot);   // (waves 4 q .. 4 q + 3 hold the digits in order)
    if (quarter == 0 && lane == SAGPU_WAVE - 1) l.wsum[w] = inc;
    __syncthreads();
    u32 at = inc - tot + before;
#pragma unroll
    for (u32 q = 0; q < 3; q++) at += q < (w & 3) ? l.wsum[q] : 0u;
#pragma unroll
    for (u32 q = 0; q < QW; q++) {
        l.cnt[(quarter * QW + q) * 256 + d] = (u16)at;
        at += own[q];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const u32 p = base + r * SAGPU_WAVE;
        if (p < n) {
            const u32 d = digit(item[r] & 0xFFFFu);   // read again: it would cost a register per row
            l.sa[l.cnt[w * 256 + d] + (item[r] >> 16)] = (u16)item[r];
        }
    }
    __syncthreads();
}

// The last group start before word `word` of s_bits (word > 0; slot 0 is a start).
template <int ROWS> __device__ u32 small_carry(const SmallLds<ROWS> &l, u32 word)
{
    const u32 lane = lane_id();
    for (int at = (int)word - 1;; at -= SAGPU_WAVE) {
        const int q = at - (int)lane;
        const u64 v = q >= 0 ? l.bits[q] : 0ull;
        const u64 m = __ballot(v != 0);
        if (m) {
            const int first = __ffsll((unsigned long long)m) - 1;
            const u64 bw = __shfl(v, first, SAGPU_WAVE);
            return (u32)(at - first) * 64 + 63 - (u32)__clzll((long long)bw);
        }
        if (at < SAGPU_WAVE) return 0;   // no start below (slot 0 always is one)
    }
}

// rank of every suffix from the group starts in s_bits.
template <int ROWS> __device__ void small_ranks(SmallLds<ROWS> &l, u32 n)
{
    const u32 w = threadIdx.x / SAGPU_WAVE, lane = lane_id();
    u32 carry = w ? small_carry(l, w * ROWS) : 0u;
    const u32 wrow = __builtin_amdgcn_readfirstlane(opaque(w * ROWS));
#pragma unroll 4
    for (int r = 0; r < ROWS; r++) {
        const u32 word = wrow + r, p = word * 64 + lane;
        const u64 b = l.bits[word];
        const u64 upto = b & (lanemask_lt() | 1ull << lane);
        const u32 head = upto ? word * 64 + 63 - (u32)__clzll((long long)upto) : carry;
        if (p < n) l.rank[l.sa[p]] = (u16)head;
        if (b) carry = word * 64 + 63 - (u32)__clzll((long long)b);
    }
}

// First group start after slot p (p < n; the bits from n on are set).
template <int ROWS> __device__ __forceinline__ u32 small_next(const SmallLds<ROWS> &l, u32 p)
{
    u32 word = (p + 1) >> 6;
    u64 v = l.bits[word] & (~0ull << ((p + 1) & 63));
    while (!v) v = l.bits[++word];
    return word * 64 + (u32)__ffsll((unsigned long long)v) - 1;
}

__device__ __forceinline__ void put_index(void *out, u32 i, u32 v, int wide)
{
    if (wide) ((int64_t *)out)[i] = (int64_t)v;
    else ((u32 *)out)[i] = v;
}

template <int ROWS>
__global__ __launch_bounds__(SM_THREADS) void k_small_build(SmallJob j)
{
    __shared__ SmallLds<ROWS> l;
    constexpr u32 N = SmallLds<ROWS>::N;
    const u32 tid = threadIdx.x, w = tid / SAGPU_WAVE, lane = lane_id(), n = j.n;
    const u32 base = w * SAGPU_WAVE * ROWS + lane;

    // ---- alphabet and codes
    if (tid < 256) l.present[tid] = 0;
    if (tid == 0) l.bad = 0;
    // this thread's symbols: words of W bytes, the next SM_THREADS words further on
    constexpr int W = ROWS < 8 ? ROWS : 8, WORDS = ROWS / W;
    u64 t[WORDS];
#pragma unroll
    for (int q = 0; q < WORDS; q++) {
        const u32 p = (q * SM_THREADS + tid) * W;
        t[q] = 0;
        if (p + W <= n) {
            __builtin_memcpy(&t[q], j.T + p, W);
        } else {
            for (u32 b = 0; b < W && p + b < n; b++) t[q] |= (u64)j.T[p + b] << (8 * b);
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < WORDS; q++) {
#pragma unroll
        for (int b = 0; b < W; b++) {
            const u32 c = (u32)(t[q] >> (8 * b)) & 255u;
            if ((q * SM_THREADS + tid) * W + b >= n) continue;
            if (j.want_freq) atomicAdd(&l.present[c], 1u);
            else l.present[c] = 1u;
        }
    }
    __syncthreads();
    if (tid < 256) {
        const u64 b = __ballot(l.present[tid] != 0);
        if (lane == 0) l.ball[w] = b;
        if (j.want_freq) j.out->freq[tid] = l.present[tid];
    }
    __syncthreads();
    const bool gsa = j.gsa && l.present[0];   // separators are code 0
    u32 sigma = 0;
    for (int q = 0; q < 4; q++) sigma += (u32)__popcll(l.ball[q]);
    if (tid < 256) {
        u32 c = (u32)__popcll(l.ball[w] & lanemask_lt());
        for (u32 q = 0; q < w; q++) c += (u32)__popcll(l.ball[q]);
        l.lut[tid] = (uint8_t)c;
        if (l.present[tid]) l.inv[c] = (uint8_t)tid;
    }
    __syncthreads();
    auto store_codes = [&]() {   // zero past the text
#pragma unroll
        for (int q = 0; q < WORDS; q++) {
            const u32 p = (q * SM_THREADS + tid) * W;
            u64 v = 0;
#pragma unroll
            for (int b = 0; b < W; b++)
                v |= (u64)(p + b < n ? l.lut[(u32)(t[q] >> (8 * b)) & 255u] : 0u) << (8 * b);
            __builtin_memcpy(l.x.c.code + p, &v, W);
        }
        if (tid < 64) l.x.c.code[N + tid] = 0;
    };
    store_codes();
    __syncthreads();
    if (j.gsa && !j.in_SA) {   // separators: the last symbol, none first or after another
        u32 bad = 0;
#pragma unroll
        for (int q = 0; q < WORDS; q++) {
            const u32 p = (q * SM_THREADS + tid) * W;
            u32 before = p > 0 && p <= n ? l.x.c.code[p - 1] : 0u;   // (0 is there: code 0 is it)
#pragma unroll
            for (int b = 0; b < W; b++) {
                const u32 c = (u32)(t[q] >> (8 * b)) & 255u;
                if (p + b < n && c == 0 && before == 0) bad |= 1u;
                if (p + b == n - 1 && c != 0) bad |= 2u;   // not terminated: the general engine's case
                before = c;
            }
        }
        if (bad) atomicOr(&l.bad, bad);
        __syncthreads();
        if (l.bad) {
            if (tid == 0) j.out->status = l.bad & 2u ? SMALL_NOT_TAKEN : SAGPU_EINVAL;
            return;
        }
    }
    const u32 radix = sigma < 2 ? 2u : sigma;
    u32 k0 = 0;
    for (u32 v = 1; k0 < 16 && v <= (1u << 24) / radix; v *= radix) k0++;
    // key / radix = umulhi(key, magic): exact, since key < 2^24 and radix <= 256 leave
    // key * (magic - 2^32 / radix) / 2^32 < 2^-8 <= 1 / radix
    const u32 magic = (u32)((0x100000000ull + radix - 1) / radix);
    u32 rounds = 0, h = k0;

    if (j.in_SA) {
        // ---- a suffix array of the caller's: only PLCP is asked for
#pragma unroll 4
        for (int r = 0; r < ROWS; r++) {
            const u32 p = base + r * SAGPU_WAVE;
            if (p < n) {
                u64 v = j.wide ? ((const u64 *)j.in_SA)[p] : ((const u32 *)j.in_SA)[p];
                if (v >= n) v = n - 1;   // not an index: no result is defined, no access leaves LDS
                l.sa[p] = (u16)v;
                l.rank[p] = 0;
            }
        }
        __syncthreads();
#pragma unroll 4
        for (int r = 0; r < ROWS; r++) {
            const u32 p = base + r * SAGPU_WAVE;
            if (p < n) l.rank[l.sa[p]] = (u16)p;
        }
        __syncthreads();
    } else {
        // ---- initial keys, every thread over a stretch of its own from right to left:
        // key(i) = code(i) sigma^(k0-1) + key(i+1) / sigma
        const u32 lo = tid * ROWS;
        u32 key = 0, top = 1;
        {
            const u64 a = load8(l.x.c.code, lo + ROWS), b = load8(l.x.c.code, lo + ROWS + 8);
            bool sep = false;
            for (u32 q = 0; q < k0; q++) {
                const u32 c = (u32)((q < 8 ? a : b) >> (8 * (q & 7))) & 255u;
                sep = sep || (gsa && c == 0);
                key = key * radix + (sep ? 0u : c);
                if (q) top *= radix;
            }
        }
#pragma unroll
        for (int r = ROWS - 1; r >= 0; r--) {
            const u32 c = l.x.c.code[lo + r];
            key = c * top + __umulhi(key, magic);
            if (gsa && c == 0) key = 0;
            l.x.c.low[lo + r] = (uint8_t)key;
            l.rank[lo + r] = (u16)(key >> 8);
        }
        __syncthreads();
        // ---- sorts and doubling rounds.  The sort's passes are one piece of code for
        // the initial keys (passes 0-2) and for a round over all slots (3-6): unrolled
        // over the rows it is the bulk of the kernel, and fetched cold.
        bool first = true, sort = true;
        auto key2 = [&](u32 i) {
            const u32 q = i + h;
            return q < n ? h + (u32)l.rank[q] : n - 1 - i;
        };
        for (;;) {
            if (sort) {
                for (int pass = first ? 0 : 3; pass < (first ? 3 : 7); pass++) {
                    const int down = pass == 2 || pass == 4 || pass == 6 ? 8 : 0;
                    small_pass<ROWS>(l, n, [&](u32 p) { return pass == 0 ? p : (u32)l.sa[p]; }, [&](u32 i) {
                        const u32 v = pass == 0 ? (u32)l.x.c.low[i] : pass == 3 || pass == 4 ? key2(i) : (u32)l.rank[i];
                        return v >> down & 255u;
                    });
                }
                auto whole = [&](u32 p) {   // what sets the suffix in slot p apart
                    const u32 i = l.sa[p];
                    return first ? (u32)l.rank[i] << 8 | l.x.c.low[i] : (u32)l.rank[i] << 16 | key2(i);
                };
                const u32 base = opaque(w * SAGPU_WAVE * ROWS + lane);
#pragma unroll 4
                for (int r = 0; r < ROWS; r++) {
                    const u32 p = base + r * SAGPU_WAVE;
                    const u32 k = p < n ? whole(p) : 0u;
                    u32 kp = __shfl_up(k, 1, SAGPU_WAVE);
                    if (lane == 0 && p > 0 && p < n) kp = whole(p - 1);
                    const u64 b = __ballot(p >= n || p == 0 || k != kp || (first && gsa && k == __umulhi(k, magic) * radix));
                    if (lane == 0) l.bits[w * ROWS + r] = b;
                }
                if (tid == 0) {
                    l.bits[N / 64] = ~0ull;
                    l.flags = l.active = 0;
                }
                __syncthreads();
                small_ranks<ROWS>(l, n);
                __syncthreads();
                if (!first) h *= 2;
                first = sort = false;
            }

            // key2 of the members of groups; flags: 1 a group is left, 2 a large one is
            u32 fl = 0, act = 0;
            const u32 base = opaque(w * SAGPU_WAVE * ROWS + lane), wrow = __builtin_amdgcn_readfirstlane(base >> 6);
#pragma unroll 4
            for (int r = 0; r < ROWS; r++) {
                const u32 p = base + r * SAGPU_WAVE, word = wrow + r;
                const u64 b = l.bits[word], nb = b >> 1 | l.bits[word + 1] << 63;
                if (!~(b & nb)) continue;   // every slot of the row is alone
                act += (u32)__popcll(~(b & nb));
                if (!(b >> lane & 1) || !(nb >> lane & 1)) {
                    const u32 i = l.sa[p], q = i + h;
                    l.x.key[p] = (u16)(q < n ? h + l.rank[q] : n - 1 - i);
                    if ((b >> lane & 1) && small_next(l, p) - p > SM_COUNT) fl = 2u;
                }
            }
            if (act) {
                fl = __any(fl != 0) ? 3u : 1u;
                if (lane == 0) {
                    atomicOr(&l.flags, fl);
                    atomicAdd(&l.active, act);
                }
            }
            __syncthreads();
            const u32 f = l.flags;
            if (!f || h > 4 * n + 64) break;
            if (tid == 0 && rounds < 64) j.out->active[rounds] = l.active;
            rounds++;
            if (f & 2u) {
                sort = true;
                continue;
            }
            {
                const u32 base = opaque(w * SAGPU_WAVE * ROWS + lane), wrow = __builtin_amdgcn_readfirstlane(base >> 6);
                u32 to[ROWS];   // new slot << 16 | new group start
#pragma unroll
                for (int r = 0; r < ROWS; r++) {
                    const u32 p = base + r * SAGPU_WAVE, word = wrow + r;
                    const u64 b = l.bits[word], nb = b >> 1 | l.bits[word + 1] << 63;
                    to[r] = ~0u;
                    if (!~(b & nb)) continue;
                    if (!(b >> lane & 1) || !(nb >> lane & 1)) {
                        const u32 head = l.rank[l.sa[p]], end = small_next(l, p), k = l.x.key[p];
                        u32 less = 0, same = 0;
                        u32 e = head;
                        for (; e + 4 <= end; e += 4) {   // four reads under way at a time
                            const u32 o0 = l.x.key[e], o1 = l.x.key[e + 1], o2 = l.x.key[e + 2], o3 = l.x.key[e + 3];
                            less += (o0 < k) + (o1 < k) + (o2 < k) + (o3 < k);
                            same += (o0 == k && e < p) + (o1 == k && e + 1 < p) + (o2 == k && e + 2 < p) +
                                    (o3 == k && e + 3 < p);
                        }
                        for (; e < end; e++) {
                            const u32 o = l.x.key[e];
                            less += o < k;
                            same += o == k && e < p;
                        }
                        to[r] = (head + less + same) << 16 | (head + less);
                    }
                }
                __syncthreads();
                if (tid == 0) l.flags = l.active = 0;
#pragma unroll
                for (int r = 0; r < ROWS; r++) {   // keys are done with: they take the new order
                    if (to[r] == ~0u) continue;
                    const u32 slot = to[r] >> 16, head = to[r] & 0xFFFFu, i = l.sa[base + r * SAGPU_WAVE];
                    l.x.key[slot] = (u16)i;
                    l.rank[i] = (u16)head;
                    if (slot == head) atomicOr((u32 *)l.bits + (slot >> 5), 1u << (slot & 31));
                }
                __syncthreads();
#pragma unroll
                for (int r = 0; r < ROWS; r++)
                    if (to[r] != ~0u) l.sa[base + r * SAGPU_WAVE] = l.x.key[base + r * SAGPU_WAVE];
                __syncthreads();
            }
            h *= 2;
        }
        __syncthreads();
        store_codes();
        __syncthreads();
    }

    // ---- outputs
    if (j.SA) {
#pragma unroll 4
        for (int r = 0; r < ROWS; r++) {
            const u32 p = base + r * SAGPU_WAVE;
            if (p < n) put_index(j.SA, p, l.sa[p], j.wide);
        }
    }
    const u32 j0 = l.rank[0];
    if (j.U) {
#pragma unroll 4
        for (int r = 0; r < ROWS; r++) {
            const u32 p = base + r * SAGPU_WAVE;
            if (p >= n) continue;
            const u32 i = l.sa[p];
            if (i == 0) j.U[0] = l.inv[l.x.c.code[n - 1]];
            else j.U[p + (p < j0)] = l.inv[l.x.c.code[i - 1]];
        }
    }
    if (j.I) {   // auxiliary samples: 1-based row of every r-th suffix
        for (u32 k = tid; k <= (n - 1) / j.r; k += SM_THREADS) put_index(j.I, k, l.rank[k * j.r] + 1u, j.wide);
    }
    if (tid == 0) {
        j.out->primary = j0 + 1;
        j.out->rounds = rounds;
        j.out->ksym = k0;
        j.out->sigma = sigma;
        j.out->status = h > 4 * n + 64 ? SAGPU_EDEVICE : SAGPU_OK;
    }
    if (!j.PLCP && !j.LCP) return;
    __syncthreads();   // rank[0] is read
    {
        // bytes the 8 at i and at k share, from the left (a separator in GSA mode is shared
        // by nothing); 8 when all
        auto shared = [&](u32 i, u32 k) {
            const u64 a = load8(l.x.c.code, i), b = load8(l.x.c.code, k);
            u64 z = a ^ b;
            // 0x80 in every zero byte of a (exact up to the first one)
            if (gsa) z |= (a - 0x0101010101010101ull) & ~a & 0x8080808080808080ull;
            return z ? (u32)(__ffsll((unsigned long long)z) - 1) / 8 : 8u;
        };
        u32 lcp = 0;
        const u32 lo = tid * ROWS;
        for (u32 i = lo; i < lo + ROWS; i++) {
            const u32 r = i < n ? l.rank[i] : 0u;
            u32 k = 0, most = 0;
            if (r) {
                k = l.sa[r - 1];
                most = n - (i > k ? i : k);
            }
            lcp = r && lcp ? lcp - 1 : 0u;
            // a few steps alone, then the wave together on each match that goes on
            bool open = lcp < most;
            for (int step = 0; step < 4 && open; step++) {
                const u32 c = shared(i + lcp, k + lcp);
                lcp += c;
                open = c == 8 && lcp < most;
            }
            for (u64 m = __ballot(open); m; m &= m - 1) {
                const int src = __ffsll((unsigned long long)m) - 1;
                const u32 wi = __shfl(i, src, SAGPU_WAVE), wk = __shfl(k, src, SAGPU_WAVE);
                const u32 end = __shfl(most, src, SAGPU_WAVE);
                u32 o = __shfl(lcp, src, SAGPU_WAVE);
                for (; o < end; o += 8 * SAGPU_WAVE) {
                    const u32 at = o + 8 * lane;
                    const u32 c = at < end ? shared(wi + at, wk + at) : 0u;
                    const u64 stop = __ballot(c < 8);
                    if (stop) {
                        const int first = __ffsll((unsigned long long)stop) - 1;
                        o += 8 * (u32)first + __shfl(c, first, SAGPU_WAVE);
                        break;
                    }
                }
                if ((int)lane == src) lcp = o;
            }
            if (lcp > most) lcp = most;
            if (i < n) l.rank[i] = (u16)lcp;
        }
    }
    __syncthreads();
#pragma unroll 4
    for (int r = 0; r < ROWS; r++) {
        const u32 p = base + r * SAGPU_WAVE;
        if (p >= n) continue;
        if (j.PLCP) put_index(j.PLCP, p, l.rank[p], j.wide);
        if (j.LCP) put_index(j.LCP, p, l.rank[l.sa[p]], j.wide);
    }
}

} // namespace

int launch_small_build(const SmallJob &j, hipStream_t s)
{
    if (j.n < 2 || j.n > SMALL_MAX) {
        sagpu_set_error("small build: text length out of range", __FILE__, __LINE__);
        return SAGPU_EDEVICE;
    }
    const u32 rows = (j.n + SM_THREADS - 1) / SM_THREADS;
#define SMALL_CASE(R) hipLaunchKernelGGL(k_small_build<R>, dim3(1), dim3(SM_THREADS), 0, s, j)
    if (rows <= 1) SMALL_CASE(1);
    else if (rows <= 2) SMALL_CASE(2);
    else if (rows <= 4) SMALL_CASE(4);
    else if (rows <= 8) SMALL_CASE(8);
    else if (rows <= 16) SMALL_CASE(16);
    else SMALL_CASE(24);
#undef SMALL_CASE
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}
