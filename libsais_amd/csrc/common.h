// common.h -- shared device helpers for the gfx950 suffix-array engine.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define SAGPU_WAVE 64

typedef unsigned long long u64;
typedef uint32_t u32;
typedef uint16_t u16;

// Status codes used inside the engine; they map 1:1 onto the libsais return codes.
enum { SAGPU_OK = 0, SAGPU_EINVAL = -1, SAGPU_ENOMEM = -2, SAGPU_EDEVICE = -3 };

#define SAGPU_CHECK(expr)                                                      \
    do {                                                                       \
        hipError_t _e = (expr);                                                \
        if (_e != hipSuccess) {                                                \
            sagpu_set_error(hipGetErrorString(_e), __FILE__, __LINE__);        \
            return (_e == hipErrorOutOfMemory) ? SAGPU_ENOMEM : SAGPU_EDEVICE; \
        }                                                                      \
    } while (0)

#define SAGPU_TRY(expr)                 \
    do {                                \
        int _rc = (expr);               \
        if (_rc != SAGPU_OK) return _rc; \
    } while (0)

void sagpu_set_error(const char *msg, const char *file, int line);

__device__ __forceinline__ u32 lane_id() { return __lane_id(); }

__device__ __forceinline__ u64 lanemask_lt() { return (1ull << lane_id()) - 1ull; }

// Lanes of `active` that hold the same low BITS bits of d as this lane.  Four vector
// instructions per bit: the bit spread over a word (x), its ballot, and for each half
// of the mask m & ~(ballot ^ x), one three-input operation (the empty asm keeps the
// compiler from testing the bit a second way).  Written as m &= bit ? ballot : ~ballot
// it compiled to nine; a radix pass ranks every key with eight of these, and a pass over
// 2^28 u32 pairs went from 1.21 to 1.12 ms with the four (116 to 75 vector instructions
// per key).
template <int BITS> __device__ __forceinline__ u64 wave_peers(u32 d, u64 active)
{
    u32 lo = (u32)active, hi = (u32)(active >> 32);
#pragma unroll
    for (int b = 0; b < BITS; b++) {
        u32 x = (u32)__builtin_amdgcn_sbfe((int)d, b, 1);
        asm("" : "+v"(x));
        const u64 bb = __ballot(x != 0);
        lo &= ~((u32)bb ^ x);
        asm("" : "+v"(lo));
        hi &= ~((u32)(bb >> 32) ^ x);
        asm("" : "+v"(hi));
    }
    return (u64)hi << 32 | lo;
}

// Set bits of m below this lane.
__device__ __forceinline__ u32 mask_below(u64 m)
{
    return __builtin_amdgcn_mbcnt_hi((u32)(m >> 32), __builtin_amdgcn_mbcnt_lo((u32)m, 0u));
}

// Lane moves inside the wave by DPP, which costs a vector instruction where a shuffle
// takes a trip through LDS.  Lanes without a source get `old`.
template <int CTRL, int ROWS> __device__ __forceinline__ u32 dpp(u32 old, u32 v)
{
    return (u32)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS> __device__ __forceinline__ u64 dpp(u64 old, u64 v)
{
    return (u64)dpp<CTRL, ROWS>((u32)(old >> 32), (u32)(v >> 32)) << 32 | dpp<CTRL, ROWS>((u32)old, (u32)v);
}
// The value of the lane below (lane 0: old) and above (lane 63: old).
template <typename V> __device__ __forceinline__ V lane_up(V old, V v) { return dpp<0x138, 0xf>(old, v); }
template <typename V> __device__ __forceinline__ V lane_down(V old, V v) { return dpp<0x130, 0xf>(old, v); }
// The value of one lane, in a scalar register.
__device__ __forceinline__ u32 lane_value(u32 v, int l) { return (u32)__builtin_amdgcn_readlane((int)v, l); }
__device__ __forceinline__ u64 lane_value(u64 v, int l)
{
    return (u64)lane_value((u32)(v >> 32), l) << 32 | lane_value((u32)v, l);
}

// Inclusive wave-level scans over 64 lanes: within rows of 16 lanes, then the last lane of
// each row (and of the lower half) to the rows after it.
template <typename V, class OP> __device__ __forceinline__ V wave_scan(V v, OP op)
{
    v = op(v, dpp<0x111, 0xf>((V)0, v));
    v = op(v, dpp<0x112, 0xf>((V)0, v));
    v = op(v, dpp<0x114, 0xf>((V)0, v));
    v = op(v, dpp<0x118, 0xf>((V)0, v));
    v = op(v, dpp<0x142, 0xa>((V)0, v));
    v = op(v, dpp<0x143, 0xc>((V)0, v));
    return v;
}
__device__ __forceinline__ u32 wave_incl_sum(u32 v)
{
    return wave_scan(v, [](u32 a, u32 b) { return a + b; });
}
__device__ __forceinline__ u32 wave_incl_max(u32 v)
{
    return wave_scan(v, [](u32 a, u32 b) { return a > b ? a : b; });
}
__device__ __forceinline__ u64 wave_incl_sum64(u64 v)
{
    return wave_scan(v, [](u64 a, u64 b) { return a + b; });
}
__device__ __forceinline__ u64 wave_incl_max64(u64 v)
{
    return wave_scan(v, [](u64 a, u64 b) { return a > b ? a : b; });
}

// An order of `count` work items that gives each XCD (workgroups go to the XCDs
// round-robin) runs of neighbouring items, which share its L2: up to 256 items (what an XCD
// has in flight), at least 8 runs an XCD, so that uneven work evens out.  b < xcd_runs(count);
// an item of count or more is none.
__host__ __device__ __forceinline__ int xcd_run_log2(u64 count)
{
    const int l = count ? 63 - __builtin_clzll(count) : 0;
    return l < 6 ? 0 : l > 14 ? 8 : l - 6;
}
__host__ __device__ __forceinline__ u64 xcd_runs(u64 count)
{
    const int s = xcd_run_log2(count) + 3;
    return (count + (1ull << s) - 1) >> s << s;
}
__device__ __forceinline__ u64 xcd_run(u64 b, u64 count)
{
    const int s = xcd_run_log2(count);
    const u64 j = b >> 3;   // the XCD's j-th
    return (((j >> s) << 3 | (b & 7)) << s) | (j & ((1ull << s) - 1));
}
// Workgroups for b of them: whole rounds of the XCDs.
inline unsigned xcd_grid(u64 b) { return (unsigned)(b < 8 ? 8 : b < 65528 ? b : 65528); }

// row + the highest set bit of m, or `none`.
__device__ __forceinline__ u32 last_set(u64 m, u32 row, u32 none)
{
    return m ? row + 63u - (u32)__clzll((long long)m) : none;
}

// p[i] of memory that nothing writes while the kernel runs, at an index that is the same
// in all lanes: a scalar load.
__device__ __forceinline__ u32 const_word(const u32 *p, int i)
{
    typedef const __attribute__((address_space(4))) u32 *cptr;
    return ((cptr)(uintptr_t)p)[i];
}

// Device-scope relaxed atomics on 64-bit look-back words.
__device__ __forceinline__ u64 ld_acquire_u64(const u64 *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void st_release_u64(u64 *p, u64 v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

static inline unsigned ceil_div_u(u64 a, u64 b) { return (unsigned)((a + b - 1) / b); }
