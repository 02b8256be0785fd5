// unbwt.hip -- BWT auxiliary samples and the inverse BWT.
//
// Inverse BWT.  Rows 0..n of the sorted rotations of T$: row 0 starts with $, row
// x >= 1 is SA slot x-1.  The libsais BWT layout stores the last column without the
// $ of row p (the 1-based primary index): U[q] is the last symbol of row
// x(q) = q + (q >= p).  Walking LF from row 0 reads T backwards, and
//   LF(x(q)) = 1 + #{bytes < U[q]} + #{q' < q : U[q'] == U[q]},
// a stable counting rank.  k_ub_count / scan / k_ub_succ turn that into a
// successor array S over BWT positions (S[q] = position of the next row, or
// UB_END when the next row is the $ row).
//
// Decoding, two ways:
//   - aux samples (libsais_unbwt_aux with many samples): sample k+1 gives the row
//     of suffix (k+1)*r, so chunk [k*r, (k+1)*r) is an independent walk of r
//     steps; one thread per chunk;
//   - list ranking (plain libsais_unbwt, or few samples): a hashed 1/G subset of the
//     positions (always including position 0, the start) are samples; every sample
//     walks to the next sample and keeps the symbols it meets (k_ub_lr_walk), pointer
//     jumping over the samples gives each one its distance to the end, and a copy puts
//     every sample's symbols in their place (k_ub_lr_copy).  The sample test is a
//     bijective hash of the position, so a sample's number and its position follow
//     from each other without a table.  The hash keeps the gaps geometric (mean G)
//     whatever the text; a gap longer than UB_CAP steps is reported as an error instead
//     of running on.
//
// A walk is a chain of dependent 4-byte reads from all over S, bound by their latency
// and, with enough walks at once, by the rate of random reads (about 53 G/s).  So it
// reads nothing but S: the symbol of a position is the bucket its successor's row lies
// in, found in LDS while the next read is under way (16-bit symbols read U beside S).
// And the text is walked once: a 32 MiB block took 1.27 ms for the walk that measured
// the gaps (131,000 walks of mean 256) and 2.40 ms for the one that wrote the text
// byte by byte; see UbPlan for the figures of the present form.
#include "engine.h"

namespace {

constexpr int UB_THREADS = 256, UB_ITEMS = 16, UB_TILE = UB_THREADS * UB_ITEMS;
constexpr int UB_WAVES = UB_THREADS / SAGPU_WAVE;
constexpr u32 UB_END = 0xFFFFFFFFu;
constexpr u32 UB_CAP = 1u << 16;

// Bijective hash of [0, 2^k): position q is a sample iff its hash is below m, and the
// hash is then the sample's number.  Multiplications by odd numbers and xor-shifts by
// at least half the width are bijections, the latter their own inverse; 0 maps to 0.
struct UbHash {
    u64 mask;   // 2^k - 1, 2^k >= n, k <= 32
    u32 sh;     // (k + 1) / 2
    u32 m;      // sample numbers: 2^k / G
    u32 i1, i2; // inverses of the two multipliers modulo 2^32
    __host__ __device__ u32 of(u32 q) const
    {
        u32 x = q;
        x = (u32)((u64)(x ^ (x >> sh)) * 0x9E3779B1u & mask);
        x = (u32)((u64)(x ^ (x >> sh)) * 0x85EBCA77u & mask);
        return x ^ (x >> sh);
    }
    __host__ __device__ u32 inverse(u32 x) const
    {
        x ^= x >> sh;
        x = (u32)((u64)x * i2 & mask);
        x ^= x >> sh;
        x = (u32)((u64)x * i1 & mask);
        return x ^ (x >> sh);
    }
};

// Inverse of an odd number modulo 2^32 (Newton: each step doubles the correct bits).
u32 ub_inverse(u32 a)
{
    u32 x = a;
    for (int k = 0; k < 5; k++) x *= 2u - a * x;
    return x;
}

// Byte counts per tile, digit-major (counts[d * tiles + t]), for the stable rank.
__global__ __launch_bounds__(UB_THREADS) void k_ub_count(const uint8_t *__restrict__ U, u64 n,
                                                         u32 *__restrict__ counts, u64 tiles)
{
    __shared__ u32 s_h[UB_WAVES][256];
    const u32 tid = threadIdx.x, w = tid / SAGPU_WAVE;
#pragma unroll
    for (int q = 0; q < UB_WAVES; q++) s_h[q][tid] = 0;
    __syncthreads();
    const u64 base = (u64)blockIdx.x * UB_TILE;
#pragma unroll
    for (int j = 0; j < UB_ITEMS; j++) {
        u64 pos = base + (u64)j * UB_THREADS + tid;
        if (pos < n) atomicAdd(&s_h[w][U[pos]], 1u);
    }
    __syncthreads();
    u32 c = 0;
#pragma unroll
    for (int q = 0; q < UB_WAVES; q++) c += s_h[q][tid];
    counts[(u64)tid * tiles + blockIdx.x] = c;
}

// S[q] from the stable rank of U[q]: scanned[d * tiles + t] = bytes < d overall plus
// bytes == d in earlier tiles; inside the tile the rank is position order (wave,
// item, lane), found with a ballot peer mask as in the radix pass.
__global__ __launch_bounds__(UB_THREADS) void k_ub_succ(const uint8_t *__restrict__ U, u64 n, u64 p,
                                                        const u32 *__restrict__ scanned, u64 tiles,
                                                        u32 *__restrict__ S)
{
    __shared__ u32 s_wcnt[UB_WAVES][256];
    const u32 tid = threadIdx.x, w = tid / SAGPU_WAVE, lane = lane_id();
#pragma unroll
    for (int q = 0; q < UB_WAVES; q++) s_wcnt[q][tid] = 0;
    __syncthreads();
    const u64 tile = blockIdx.x;
    const u64 wbase = tile * UB_TILE + (u64)w * (SAGPU_WAVE * UB_ITEMS);
    u32 dig[UB_ITEMS], rank[UB_ITEMS];
#pragma unroll
    for (int j = 0; j < UB_ITEMS; j++) {
        u64 pos = wbase + (u64)j * SAGPU_WAVE + lane;
        bool ok = pos < n;
        u32 d = ok ? (u32)U[pos] : 0u;
        const u64 m = wave_peers<8>(d, __ballot(ok));
        const u32 below = mask_below(m);
        u32 old = 0;
        if (ok) {
            old = s_wcnt[w][d];
            s_wcnt[w][d] = old + (u32)__popcll(m);   // the same value from every peer
        }
        dig[j] = d;
        rank[j] = old + below;
    }
    __syncthreads();
    {
        const u32 d = tid;
        u32 run = 0;
#pragma unroll
        for (int q = 0; q < UB_WAVES; q++) {
            u32 c = s_wcnt[q][d];
            s_wcnt[q][d] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < UB_ITEMS; j++) {
        u64 pos = wbase + (u64)j * SAGPU_WAVE + lane;
        if (pos >= n) continue;
        const u32 d = dig[j];
        const u64 x = (u64)scanned[(u64)d * tiles + tile] + s_wcnt[w][d] + rank[j] + 1;  // next row
        S[pos] = x == p ? UB_END : (u32)(x - (x > p));
    }
}

// Symbols from successors: position q's symbol is the bucket of row LF(x(q)).  first[c]
// = symbols below c in the whole text; block b of 2^sh rows starts in bucket tab[b].
constexpr int UB_BLOCKS = 4096;
struct UbDecode {
    const u32 *scanned;   // the scanned counts of launch_unbwt_succ: first[c] = scanned[c * tiles]
    u64 tiles;
    u64 n, p;
    int sh;
};

template <typename ST> struct UbSymbols;

template <> struct UbSymbols<uint8_t> {
    struct Lds {
        u32 first[257];
        uint8_t tab[UB_BLOCKS];
    };
    const Lds &l;
    int sh;
    u32 p;
    __device__ UbSymbols(Lds &lds, const UbDecode &d, const uint8_t *) : l(lds), sh(d.sh), p((u32)d.p)
    {
        for (u32 c = threadIdx.x; c < 257; c += blockDim.x)
            lds.first[c] = c < 256 ? d.scanned[(u64)c * d.tiles] : (u32)d.n;
        __syncthreads();
        for (u32 b = threadIdx.x; b < UB_BLOCKS; b += blockDim.x) {
            const u64 x = (u64)b << sh;   // the last bucket that starts at or before row x
            u32 c = 0;
            for (u32 st = 128; st; st >>= 1)
                if (lds.first[c + st] <= x) c += st;
            lds.tab[b] = (uint8_t)c;
        }
        __syncthreads();
    }
    __device__ u32 fetch(u32) const { return 0; }   // nothing beside the successor
    // s: the successor of the position (UB_END: its row is p)
    __device__ u32 decode(u32 s, u32) const
    {
        const u32 x = (s == UB_END ? p : s + (s >= p)) - 1u;
        u32 c = l.tab[x >> sh];
        while (l.first[c + 1] <= x) c++;
        return c;
    }
};

template <> struct UbSymbols<uint16_t> {
    struct Lds { };
    const uint16_t *U;
    __device__ UbSymbols(Lds &, const UbDecode &, const uint16_t *u) : U(u) {}
    __device__ u32 fetch(u32 q) const { return U[q]; }
    __device__ u32 decode(u32, u32 v) const { return v; }
};

// Aux decoding: one thread per chunk [c*r, min((c+1)*r, n)), walking back from the
// row of suffix (c+1)*r (row 0 for the last chunk).  Symbols are gathered into 8-byte
// words of the output and written a word at a time.
template <typename ST>
__global__ __launch_bounds__(256) void k_ub_walk_aux(const ST *__restrict__ U, const u32 *__restrict__ S, u64 n,
                                                     u64 p, u64 r, const u64 *__restrict__ rows, u64 chunks,
                                                     ST *__restrict__ out, UbDecode dec, u32 *__restrict__ err)
{
    __shared__ typename UbSymbols<ST>::Lds s_l;
    const UbSymbols<ST> sym(s_l, dec, U);
    constexpr u32 W = 8 / sizeof(ST), SB = 8 * sizeof(ST);
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 c = (u64)blockIdx.x * blockDim.x + threadIdx.x; c < chunks; c += stride) {
        const u64 lo = c * r, hi = lo + r < n ? lo + r : n;
        const u64 x = c + 1 < chunks ? rows[c + 1] : 0;
        if (x == p || x > n) {  // a sample that claims the $ row: inconsistent input
            atomicOr(err, 1u);
            continue;
        }
        u32 q = (u32)(x - (x > p));
        u64 acc = 0;
        u64 top = hi;   // symbols [j, top) are in acc, the lowest last
        for (u64 j = hi; j-- > lo;) {
            const u32 s = S[q];
            const u32 v = sym.decode(s, sym.fetch(q));
            acc = acc << SB | v;
            // a whole aligned word of the output
            if (j % W == 0 && top - j == W) {
                *(u64 *)(out + j) = acc;
                top = j;
            } else if (j % W == 0 || j == lo || (s == UB_END && j > lo)) {
                for (u64 k = j; k < top; k++) {
                    out[k] = (ST)acc;
                    acc >>= SB;
                }
                top = j;
            }
            if (s == UB_END && j > lo) {
                atomicOr(err, 1u);
                break;
            }
            q = s;
        }
    }
}

// Room for the symbols of the walks: `cap` symbols per sample, and pages of cap symbols
// for the gaps that are longer (one in twenty at cap = 3 G), taken from `segs` counters
// (a workgroup uses that of its number modulo segs, so they do not queue on one
// address).  A gap's pages are chained: link[id] is the first one, link[m + page] the
// one after a page.  Where no page is left, UB_END stands there and more[id] is the
// position the rest of the gap starts at, to be walked again.  (With that second walk
// for every long gap, its dependent reads were 0.45 of the 0.50 ms that k_ub_lr_copy
// took for a 32 MiB block.)
template <typename ST> struct UbRoom {
    ST *buf;          // [m + pages] chunks of cap symbols
    u32 *link;        // [m + pages]
    u32 *more;        // [m]
    u32 *used;        // [segs] pages taken
    u32 m, cap, pages, segs;
    __device__ u32 page() const
    {
        const u32 g = blockIdx.x % segs, per = pages / segs;
        const u32 k = atomicAdd(&used[g], 1u);
        return k < per ? g * per + k : UB_END;
    }
    __device__ ST *end(u32 chunk) const { return buf + (u64)(chunk + 1) * cap; }
};

// Each sample walks to the next sample and keeps its symbols: nd = (symbols from this
// sample up to the next one or the end) << 32 | next sample's number (UB_END at the
// end).  Symbols go to the sample's chunk and its pages, each filled from its end
// (text order).
template <typename ST>
__global__ __launch_bounds__(256) void k_ub_lr_walk(const ST *__restrict__ U, const u32 *__restrict__ S, UbHash h,
                                                    UbDecode dec, UbRoom<ST> room, u64 *__restrict__ nd,
                                                    u32 *__restrict__ err)
{
    __shared__ typename UbSymbols<ST>::Lds s_l;
    const UbSymbols<ST> sym(s_l, dec, U);
    constexpr u32 W = 8 / sizeof(ST), SB = 8 * sizeof(ST);
    for (u32 id = blockIdx.x * blockDim.x + threadIdx.x; id < h.m; id += gridDim.x * blockDim.x) {
        u32 q = h.inverse(id);
        if (q >= dec.n) {   // no such position
            nd[id] = UB_END;
            continue;
        }
        u32 chunk = id, full = room.cap;   // the current chunk is full after `full` symbols
        ST *at = room.end(id);             // symbols [len - len % W, ..) go below at
        u64 acc = 0;
        u32 len = 0, next;
        for (;;) {
            const u32 s = S[q];
            const u32 v = sym.decode(s, sym.fetch(q));
            if (len == full && chunk != UB_END) {
                const u32 pg = room.page();
                room.link[chunk] = pg;
                if (pg != UB_END) {
                    chunk = h.m + pg;
                    full += room.cap;
                    at = room.end(chunk);
                } else {
                    room.more[id] = q;
                    chunk = UB_END;
                }
            }
            acc = acc << SB | v;
            len++;
            if (len % W == 0 && chunk != UB_END) {
                at -= W;
                *(u64 *)at = acc;
            }
            if (s == UB_END) {
                next = UB_END;
                break;
            }
            next = h.of(s);
            if (next < h.m) break;
            if (len >= UB_CAP) {   // gap over UB_CAP: the host reports an error
                atomicOr(err, 2u);
                next = UB_END;
                break;
            }
            q = s;
        }
        const u32 part = len % W;
        if (part && chunk != UB_END) *(u64 *)(at - W) = acc << (SB * (W - part));
        nd[id] = (u64)len << 32 | next;
    }
}

// One pointer-jumping round: nd (in) -> nd2 (out).
__global__ __launch_bounds__(256) void k_ub_jump(const u64 *__restrict__ nd, u32 m, u64 *__restrict__ nd2)
{
    for (u32 id = blockIdx.x * blockDim.x + threadIdx.x; id < m; id += gridDim.x * blockDim.x) {
        const u64 a = nd[id];
        u64 o = a;
        if ((u32)a != UB_END) {
            const u64 b = nd[(u32)a];
            o = (((a >> 32) + (b >> 32)) << 32) | (u32)b;
        }
        nd2[id] = o;
    }
}

// Samples on the path from position 0 (their pointer reached the end) put their gap in
// its place: step t of the path emits out[n-1-t], and sample id starts at step
// dist[0] - dist[id].  Eight lanes per sample, eight bytes each per step.
constexpr u32 UB_CP = 8;
template <typename ST>
__global__ __launch_bounds__(256) void k_ub_lr_copy(const ST *__restrict__ U, const u32 *__restrict__ S, UbHash h,
                                                    UbDecode dec, UbRoom<ST> room, const u64 *__restrict__ nd0,
                                                    const u64 *__restrict__ nd, ST *__restrict__ out)
{
    __shared__ typename UbSymbols<ST>::Lds s_l;
    const UbSymbols<ST> sym(s_l, dec, U);
    constexpr u32 W = 8 / sizeof(ST);
    const u64 n = dec.n, total = nd[0] >> 32;
    if ((u32)nd[0] != UB_END) return;   // no path from position 0 to the end
    const u32 sub = threadIdx.x % UB_CP;
    for (u64 g = ((u64)blockIdx.x * blockDim.x + threadIdx.x) / UB_CP; g < h.m;
         g += (u64)gridDim.x * blockDim.x / UB_CP) {
        const u32 id = (u32)g;
        const u64 d = nd[id];
        const u32 len = (u32)(nd0[id] >> 32);
        if ((u32)d != UB_END || len == 0) continue;   // not on the path from position 0
        const u64 t0 = total - (d >> 32);
        if (t0 >= n) continue;   // inconsistent input: a walk longer than the text
        const u64 top = n - t0;  // symbol j goes to out[top - 1 - j]
        const u32 have = len < top ? len : (u32)top;
        u32 chunk = id;
        for (u32 base = 0; base < have; base += room.cap) {   // symbols [base, stop) from one chunk
            if (base) chunk = room.link[chunk];
            if (chunk == UB_END) {   // no page was left: the rest is walked again
                if (sub == 0) {
                    u32 q = room.more[id];
                    for (u32 j = base; j < have; j++) {
                        const u32 s = S[q];
                        out[top - 1 - j] = (ST)sym.decode(s, sym.fetch(q));
                        q = s;   // the walk met no end before its last symbol
                    }
                }
                break;
            }
            if (base) chunk += h.m;
            const ST *end = room.end(chunk);
            const u32 kept = have - base < room.cap ? have - base : room.cap;
            const u64 tb = top - base;
            for (u32 j = sub * W; j < kept; j += UB_CP * W) {
                if (j + W <= kept) {
                    const u64 w = *(const u64 *)(end - (j + W));
                    __builtin_memcpy(out + (tb - (j + W)), &w, 8);
                } else {
                    for (u32 k = j; k < kept; k++) out[tb - 1 - k] = end[-1 - (int)k];
                }
            }
        }
    }
}

// Successor array from a stable sort of (symbol, position): the position sorted to
// slot k has LF row k + 1 (16-bit symbols, where per-tile counting tables do not fit).
__global__ __launch_bounds__(256) void k_ub_succ_sorted(const u32 *__restrict__ V, u64 n, u64 p, u32 *__restrict__ S)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 k = (u64)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
        const u64 x = k + 1;
        S[V[k]] = x == p ? UB_END : (u32)(x - (x > p));
    }
}

__global__ __launch_bounds__(256) void k_ub_keys16(const uint16_t *__restrict__ U, u64 n, u32 *__restrict__ keys,
                                                   u32 *__restrict__ vals)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 q = (u64)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += stride) {
        keys[q] = U[q];
        vals[q] = (u32)q;
    }
}

__global__ __launch_bounds__(256) void k_aux_samples(const u32 *__restrict__ ISA, u64 n, u64 r, u64 count,
                                                     u32 *__restrict__ out)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 k = (u64)blockIdx.x * blockDim.x + threadIdx.x; k < count; k += stride) out[k] = isa_rank(ISA[k * r], n);
}

unsigned grid_of(u64 work, unsigned per_block, unsigned cap)
{
    u64 b = (work + per_block - 1) / per_block;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (unsigned)b;
}

} // namespace

int launch_aux_samples(const u32 *ISA, u64 n, u64 r, u64 count, u32 *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_aux_samples, dim3(grid_of(count, 256 * 4, 65535)), dim3(256), 0, s, ISA, n, r, count, out);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

u64 unbwt_count_slots(u64 n) { return 256 * ((n + UB_TILE - 1) / UB_TILE); }

int launch_unbwt_succ(const uint8_t *U, u64 n, u64 p, u32 *counts, ScanScratch &sc, u32 *S, hipStream_t s)
{
    const u64 tiles = (n + UB_TILE - 1) / UB_TILE;
    hipLaunchKernelGGL(k_ub_count, dim3((unsigned)tiles), dim3(UB_THREADS), 0, s, U, n, counts, tiles);
    SAGPU_CHECK(hipGetLastError());
    SAGPU_TRY(scan_exclusive_u32(sc, counts, tiles * 256, s));
    hipLaunchKernelGGL(k_ub_succ, dim3((unsigned)tiles), dim3(UB_THREADS), 0, s, U, n, p, counts, tiles, S);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

static UbDecode ub_decode(const u32 *scanned, u64 n, u64 p)
{
    int sh = 0;
    while ((n >> sh) >= (u64)UB_BLOCKS) sh++;
    return UbDecode{scanned, (n + UB_TILE - 1) / UB_TILE, n, p, sh};
}

int launch_unbwt_aux_walk(const void *U, int sym_bytes, const u32 *S, u64 n, u64 p, u64 r, const u64 *rows,
                          u64 chunks, const u32 *scanned, void *out, u32 *err, hipStream_t s)
{
    const UbDecode dec = ub_decode(scanned, n, p);
    if (sym_bytes == 2)
        hipLaunchKernelGGL(k_ub_walk_aux<uint16_t>, dim3(grid_of(chunks, 256, 65535)), dim3(256), 0, s,
                           (const uint16_t *)U, S, n, p, r, rows, chunks, (uint16_t *)out, dec, err);
    else
        hipLaunchKernelGGL(k_ub_walk_aux<uint8_t>, dim3(grid_of(chunks, 256, 65535)), dim3(256), 0, s,
                           (const uint8_t *)U, S, n, p, r, rows, chunks, (uint8_t *)out, dec, err);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_unbwt_succ16(const uint16_t *U, u64 n, u64 p, u32 *keys, u32 *vals, u32 *S, hipStream_t s)
{
    (void)p;
    (void)S;
    hipLaunchKernelGGL(k_ub_keys16, dim3(grid_of(n, 256 * 8, 65535)), dim3(256), 0, s, U, n, keys, vals);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_unbwt_succ_sorted(const u32 *V, u64 n, u64 p, u32 *S, hipStream_t s)
{
    hipLaunchKernelGGL(k_ub_succ_sorted, dim3(grid_of(n, 256 * 8, 65535)), dim3(256), 0, s, V, n, p, S);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

UbPlan unbwt_plan(u64 n)
{
    int k = 1;
    while ((1ull << k) < n) k++;
    const int g = n >= (1ull << 24) ? 6 : n >= (1ull << 22) ? 5 : 4;
    UbPlan pl;
    pl.k = k;
    pl.m = k > g ? 1u << (k - g) : 1u;
    pl.gap = 1u << g;
    // two and a half times the pages that gaps over 3 * gap are expected to take
    pl.segs = pl.m >= (1u << 18) ? 64 : 1;
    pl.pages = pl.m / 8 + 16;
    return pl;
}

template <typename ST>
static int ub_rank(const ST *U, const u32 *S, u64 n, u64 p, const UbPlan &pl, u32 cap, const u32 *scanned,
                   u64 *const nd[3], void *buf, u32 *link, u32 *more, u32 *used, ST *out, u32 *err, hipStream_t s)
{
    const UbDecode dec = ub_decode(scanned, n, p);
    const UbHash h{(1ull << pl.k) - 1, (u32)(pl.k + 1) / 2, pl.m, ub_inverse(0x9E3779B1u), ub_inverse(0x85EBCA77u)};
    const UbRoom<ST> room{(ST *)buf, link, more, used, pl.m, cap, pl.pages, pl.segs};
    const unsigned g = grid_of(pl.m, 256, 65535), gc = grid_of((u64)pl.m * UB_CP, 256, 65535);
    SAGPU_TRY(launch_fill_u32(used, pl.segs, 0, s));
    hipLaunchKernelGGL(k_ub_lr_walk<ST>, dim3(g), dim3(256), 0, s, U, S, h, dec, room, nd[0], err);
    int rounds = 0;
    while ((1ull << rounds) < (u64)pl.m + 1) rounds++;
    int cur = 0;   // nd[0] keeps the gaps
    for (int k = 0; k <= rounds; k++) {
        const int to = cur == 1 ? 2 : 1;
        hipLaunchKernelGGL(k_ub_jump, dim3(g), dim3(256), 0, s, nd[cur], pl.m, nd[to]);
        cur = to;
    }
    hipLaunchKernelGGL(k_ub_lr_copy<ST>, dim3(gc), dim3(256), 0, s, U, S, h, dec, room, nd[0], nd[cur], out);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_unbwt_rank(const void *U, int sym_bytes, const u32 *S, u64 n, u64 p, const UbPlan &pl, u32 cap,
                      const u32 *scanned, u64 *const nd[3], void *buf, u32 *link, u32 *more, u32 *used, void *out,
                      u32 *err, hipStream_t s)
{
    if (sym_bytes == 2)
        return ub_rank((const uint16_t *)U, S, n, p, pl, cap, scanned, nd, buf, link, more, used, (uint16_t *)out, err, s);
    return ub_rank((const uint8_t *)U, S, n, p, pl, cap, scanned, nd, buf, link, more, used, (uint8_t *)out, err, s);
}
