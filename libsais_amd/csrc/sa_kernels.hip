// sa_kernels.hip -- symbol histogram, packed initial keys, doubling-round keys.
#include "engine.h"

namespace {

// 256-bin byte histogram (the libsais `freq` table) with LDS privatisation: one
// sub-histogram per wave so that the few hot bins of DNA text do not serialise
// the whole workgroup.  In GSA mode it also counts the positions that make the
// input invalid (a 0 at position 0 or a 0 directly after another 0).
// Workgroup 0 also clears the 64 bytes of padding after the text.
__global__ __launch_bounds__(256) void k_histogram(const uint8_t *__restrict__ T, u64 n, int gsa,
                                                   u64 *__restrict__ hist, uint8_t *__restrict__ pad)
{
    u32 *bad = (u32 *)(hist + 256);
    if (pad && blockIdx.x == 0 && threadIdx.x < 64) pad[threadIdx.x] = 0;
    // 16 sub-histograms: lanes of a wave spread over 4 copies (lane % 4), so a text of
    // few distinct bytes (DNA) has a quarter of the same-word atomics per step.  Rows
    // of 257 words put the copies of one byte value in different LDS banks.
    __shared__ u32 s_h[16][257];
    for (int i = threadIdx.x; i < 16 * 257; i += 256) (&s_h[0][0])[i] = 0;
    __syncthreads();
    const u32 w = (threadIdx.x / SAGPU_WAVE) * 4 + (threadIdx.x & 3);
    u32 nbad = 0;
    const u64 nvec = n / 16;
    const uint4 *T16 = reinterpret_cast<const uint4 *>(T);
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x; v < nvec; v += stride) {
        uint4 x = T16[v];
        u32 words[4] = {x.x, x.y, x.z, x.w};
        u32 prev = (v == 0) ? 0u : T[16 * v - 1];
#pragma unroll
        for (int q = 0; q < 4; q++) {
#pragma unroll
            for (int b = 0; b < 4; b++) {
                u32 c = (words[q] >> (8 * b)) & 255u;
                atomicAdd(&s_h[w][c], 1u);
                if (gsa) nbad += (c == 0) && (prev == 0);
                prev = c;
            }
        }
    }
    for (u64 i = nvec * 16 + (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        u32 c = T[i];
        atomicAdd(&s_h[w][c], 1u);
        if (gsa) nbad += (c == 0) && (i == 0 || T[i - 1] == 0);
    }
    __syncthreads();
    for (int c = threadIdx.x; c < 256; c += 256) {
        u32 t = 0;
        for (int q = 0; q < 16; q++) t += s_h[q][c];
        if (t) atomicAdd(&hist[c], (u64)t);
    }
    if (gsa && nbad) atomicAdd(bad, nbad);
}

// The counts as dense codes of the present bytes (lut) and back (inv); counts and validity
// to the host (pinned), and cleared for the next text.  It replaces a fill, a copy back
// and two uploads of tables made on the host.  (A kernel of its own: left to the last
// workgroup of k_histogram, the fence that each of up to 2048 workgroups needs took 0.1
// ms on a 48 MiB text.)
__global__ __launch_bounds__(256) void k_alphabet(u64 *__restrict__ hist, uint8_t *__restrict__ lut,
                                                  uint8_t *__restrict__ inv, u64 *__restrict__ host)
{
    __shared__ u64 s_b[4];
    __shared__ uint8_t s_inv[256];
    const u32 c = threadIdx.x, wv = c / SAGPU_WAVE;
    const u64 cnt = hist[c];
    const u64 b = __ballot(cnt != 0);
    if (lane_id() == 0) s_b[wv] = b;
    s_inv[c] = 0;
    __syncthreads();
    u32 code = (u32)__popcll(b & lanemask_lt());
    for (u32 q = 0; q < wv; q++) code += (u32)__popcll(s_b[q]);
    if (cnt) s_inv[code] = (uint8_t)c;
    lut[c] = (uint8_t)code;
    host[c] = cnt;
    hist[c] = 0;
    if (c == 0) {
        host[256] = hist[256] & 0xFFFFFFFFull;
        hist[256] = 0;
    }
    __syncthreads();
    inv[c] = s_inv[c];
}

constexpr int PK_THREADS = 256, PK_ITEMS = 16, PK_TILE = PK_THREADS * PK_ITEMS, PK_HALO = 64;

// Packed keys of the first k symbols of every suffix (k*bits <= 32): symbol t of
// suffix i sits in bits [bits*(k-1-t), bits*(k-t)).  Positions past the end read
// code 0, the smallest code; ties that this creates are broken by the doubling
// rounds, where a suffix shorter than the offset ranks by its length.  In GSA mode
// (separator = code 0, letters >= 1) every symbol after the first separator is
// forced to 0, so keys that contain a separator end in a zero slot.
// keys[p] = codes of T[p .. p+k) (first symbol high), vals[p] = p, or with cb > 0
// (p << cb) | code of T[p-1]: the BWT symbol of suffix p travels with it through
// the initial sort.
__global__ __launch_bounds__(PK_THREADS) void k_pack_keys32(const uint8_t *__restrict__ T, u64 n,
                                                            const uint8_t *__restrict__ lut, int bits, int k,
                                                            int gsa, int cb, u32 *__restrict__ keys,
                                                            u32 *__restrict__ vals, int items)
{
    // items <= PK_ITEMS keys per thread (short texts take fewer, so more workgroups
    // share the k-symbol loops)
    __shared__ uint8_t s_lut[256];
    __shared__ uint8_t s_c[PK_TILE + PK_HALO + 1];   // s_c[i] = code of T[base - 1 + i]
    s_lut[threadIdx.x] = lut[threadIdx.x];
    __syncthreads();
    const int tile = PK_THREADS * items;
    const u64 base = (u64)blockIdx.x * tile;
    for (int i = threadIdx.x; i < tile + PK_HALO + 1; i += PK_THREADS) {
        u64 p = base + i;   // position base - 1 + i, shifted by one
        s_c[i] = (p >= 1 && p - 1 < n) ? s_lut[T[p - 1]] : 0;
    }
    __syncthreads();
#pragma unroll 4
    for (int j = 0; j < items; j++) {
        int li = j * PK_THREADS + threadIdx.x;
        u64 p = base + li;
        if (p >= n) break;
        u32 key = 0;
        bool sep = false;
        for (int t = 0; t < k; t++) {
            u32 c = s_c[li + 1 + t];
            if (gsa) {
                if (sep) c = 0;
                sep = sep || c == 0;
            }
            key = (key << bits) | c;
        }
        keys[p] = key;
        vals[p] = cb ? ((u32)p << cb) | (u32)s_c[li] : (u32)p;
    }
}

// String ids: a workgroup takes SI_TILE positions, four to a thread and step; the
// separators of a tile are counted first, and after a scan of the counts a second read
// of the text writes the ids (the 5 + 1 bytes per position that it takes).  As a flag per
// position and a scan in place over them: 2.6 ms for 2^29 positions, now 0.7.
constexpr int SI_STEPS = 4, SI_STEP = 1024, SI_TILE = SI_STEPS * SI_STEP;
// Zero bytes of x, a bit at the top of each.
__device__ __forceinline__ u32 zero_bytes(u32 x) { return ~(((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x | 0x7F7F7F7Fu); }
// The zero bytes among T[p .. p + 4), none from n on.
__device__ __forceinline__ u32 zeros4(const uint8_t *T, u64 p, u64 n)
{
    if (p >= n) return 0u;
    u32 x;
    __builtin_memcpy(&x, T + p, 4);   // (the text's padding is there)
    const u32 z = zero_bytes(x);
    return n - p < 4 ? z & ((1u << (8 * (u32)(n - p))) - 1u) : z;
}
__global__ __launch_bounds__(256) void k_string_counts(const uint8_t *__restrict__ T, u64 n, u32 *__restrict__ cnt)
{
    __shared__ u32 s_w[256 / SAGPU_WAVE];
    const u64 base = (u64)blockIdx.x * SI_TILE;
    u32 c = 0;
#pragma unroll
    for (int j = 0; j < SI_STEPS; j++) c += (u32)__popc(zeros4(T, base + (u64)j * SI_STEP + 4 * threadIdx.x, n));
    c = wave_incl_sum(c);
    if (lane_id() == SAGPU_WAVE - 1) s_w[threadIdx.x / SAGPU_WAVE] = c;
    __syncthreads();
    if (threadIdx.x == 0) cnt[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}
__global__ __launch_bounds__(256) void k_string_ids(const uint8_t *__restrict__ T, u64 n, const u32 *__restrict__ before,
                                                    u32 *__restrict__ sid)
{
    constexpr int NW = 256 / SAGPU_WAVE;
    __shared__ u32 s_w[SI_STEPS][NW];
    const u64 base = (u64)blockIdx.x * SI_TILE;
    const u32 w = threadIdx.x / SAGPU_WAVE;
    u32 z[SI_STEPS], inc[SI_STEPS];
#pragma unroll
    for (int j = 0; j < SI_STEPS; j++) z[j] = zeros4(T, base + (u64)j * SI_STEP + 4 * threadIdx.x, n);
#pragma unroll
    for (int j = 0; j < SI_STEPS; j++) {
        inc[j] = wave_incl_sum((u32)__popc(z[j]));
        if (lane_id() == SAGPU_WAVE - 1) s_w[j][w] = inc[j];
    }
    __syncthreads();
    u32 c = before[blockIdx.x];
#pragma unroll
    for (int j = 0; j < SI_STEPS; j++) {
        u32 o = c + inc[j] - (u32)__popc(z[j]);
        for (u32 q = 0; q < (u32)NW; q++) {
            if (q < w) o += s_w[j][q];
            c += s_w[j][q];
        }
        const u64 p = base + (u64)j * SI_STEP + 4 * threadIdx.x;
        const u32 id[4] = {o, o + (u32)__popc(z[j] & 0xFFu), o + (u32)__popc(z[j] & 0xFFFFu),
                           o + (u32)__popc(z[j] & 0xFFFFFFu)};
        if (p + 4 <= n) {
            *reinterpret_cast<uint4 *>(sid + p) = make_uint4(id[0], id[1], id[2], id[3]);
        } else {
            for (int t = 0; t < 4; t++)
                if (p + t < n) sid[p + t] = id[t];
        }
    }
}

// Keys of string sets sorted string by string (local: a string's number among those
// sorted together).  Each thread takes PK_ITEMS consecutive positions from right to left,
// key(i) = code(i) in front of key(i + 1) without its last symbol, and zero at a separator;
// the keys are written out through LDS.  Bound by its 4 bytes written and 5 read per
// position.
__global__ __launch_bounds__(PK_THREADS) void k_pack_keys32_sid(const uint8_t *__restrict__ T, u64 n,
                                                                const uint8_t *__restrict__ lut, int bits, int k,
                                                                const u32 *__restrict__ sid,
                                                                const uint8_t *__restrict__ local,
                                                                u32 *__restrict__ keys)
{
    constexpr int ROW = PK_ITEMS + 1;   // (rows a bank apart)
    static_assert(PK_ITEMS == 16 && PK_HALO <= 64, "16 codes a thread");
    __shared__ uint8_t s_lut[256];
    __shared__ __align__(16) uint8_t s_c[PK_TILE + 64];
    __shared__ u32 s_k[PK_THREADS * ROW];
    s_lut[threadIdx.x] = lut[threadIdx.x];
    __syncthreads();
    const u64 base = (u64)blockIdx.x * PK_TILE;
    const int lo = (int)threadIdx.x * PK_ITEMS;
    // codes of 16 positions, 0 from n on (the text's padding may hold anything)
    auto codes16 = [&](u64 p, u64 c[2]) {
        uint8_t b[16];
        c[0] = c[1] = 0;
        if (p >= n) return;
        __builtin_memcpy(b, T + p, 16);
#pragma unroll
        for (int t = 0; t < 16; t++) c[t / 8] |= (u64)(p + t < n ? s_lut[b[t]] : 0u) << (8 * (t % 8));
    };
    u64 c[2];
    codes16(base + lo, c);
    __builtin_memcpy(s_c + lo, c, 16);
    if (threadIdx.x < 4) {
        u64 h[2];
        codes16(base + PK_TILE + 16 * threadIdx.x, h);
        __builtin_memcpy(s_c + PK_TILE + 16 * threadIdx.x, h, 16);
    }
    __syncthreads();
    const int top = bits * (k - 1), kb = bits * k;
    u32 key = 0;   // of position lo + 16
    for (int ch = (k - 1) / 8; ch >= 0; ch--) {
        u64 x;
        __builtin_memcpy(&x, s_c + lo + PK_ITEMS + 8 * ch, 8);
        for (int t = k - 1 - 8 * ch < 7 ? k - 1 - 8 * ch : 7; t >= 0; t--) {
            const u32 s = (u32)(x >> (8 * t)) & 255u;
            key = s ? (s << top) | (key >> bits) : 0u;
        }
    }
#pragma unroll
    for (int j = PK_ITEMS - 1; j >= 0; j--) {
        const u32 s = (u32)(c[j / 8] >> (8 * (j % 8))) & 255u;
        key = s ? (s << top) | (key >> bits) : 0u;
        s_k[threadIdx.x * ROW + j] = key;
    }
    __syncthreads();
    // most tiles lie inside one string
    const u64 last = base + PK_TILE <= n ? base + PK_TILE - 1 : n - 1;
    const u32 q0 = sid[base], q1 = sid[last];
    const u32 l0 = local[q0];
#pragma unroll 4
    for (int j = 0; j < PK_ITEMS; j++) {
        const int li = j * PK_THREADS + (int)threadIdx.x;
        const u64 p = base + li;
        if (p >= n) break;
        const u32 l = q0 == q1 ? l0 : local[sid[p]];
        keys[p] = s_k[li / PK_ITEMS * ROW + li % PK_ITEMS] | (l ? l << kb : 0u);
    }
}

__global__ __launch_bounds__(PK_THREADS) void k_pack_keys64_sid(const uint8_t *__restrict__ T, u64 n,
                                                                const uint8_t *__restrict__ lut, int bits, int k,
                                                                const u32 *__restrict__ sid, u64 *__restrict__ keys,
                                                                u32 *__restrict__ vals)
{
    __shared__ uint8_t s_lut[256];
    __shared__ uint8_t s_c[PK_TILE + PK_HALO];
    s_lut[threadIdx.x] = lut[threadIdx.x];
    __syncthreads();
    const u64 base = (u64)blockIdx.x * PK_TILE;
    for (int i = threadIdx.x; i < PK_TILE + PK_HALO; i += PK_THREADS) {
        u64 p = base + i;
        s_c[i] = p < n ? s_lut[T[p]] : 0;
    }
    __syncthreads();
#pragma unroll 4
    for (int j = 0; j < PK_ITEMS; j++) {
        int li = j * PK_THREADS + threadIdx.x;
        u64 p = base + li;
        if (p >= n) break;
        u32 key = 0;
        bool sep = false;
        for (int t = 0; t < k; t++) {
            u32 c = s_c[li + t];
            if (sep) c = 0;
            sep = sep || c == 0;
            key = (key << bits) | c;
        }
        keys[p] = ((u64)sid[p] << 32) | key;
        vals[p] = (u32)p;
    }
}

__global__ void k_check_offsets(const uint8_t *__restrict__ T, const u32 *__restrict__ sid,
                                const int64_t *__restrict__ off, u32 count, u32 *bad)
{
    for (u32 q = blockIdx.x * blockDim.x + threadIdx.x; q < count; q += gridDim.x * blockDim.x) {
        int64_t o = off[q];
        bool ok = sid[o] == q && off[q + 1] > o + 1 && T[off[q + 1] - 1] == 0 && (q == 0 || T[o - 1] == 0);
        // no separator before the string's last symbol (that of the last string would make
        // ids past every table that is read by id)
        ok = ok && sid[off[q + 1] - 1] == q;
        if (!ok) atomicOr(bad, 1u);
    }
}

// out[j] = SA[j] less its string's first position.  The slots of a string are its own
// positions; most tiles of 4096 lie inside one string and take its offset once.
constexpr u64 LZ_TILE = 4096;
__global__ __launch_bounds__(256) void k_localize(const u32 *__restrict__ SA, const u32 *__restrict__ sid,
                                                  const int64_t *__restrict__ off, u64 n, u32 *__restrict__ out)
{
    const u64 base = (u64)blockIdx.x * LZ_TILE;
    const u64 last = n - base < LZ_TILE ? n - 1 : base + LZ_TILE - 1;
    const u32 q0 = sid[base], q1 = sid[last];
    const u32 o0 = (u32)off[q0];
#pragma unroll
    for (u64 j = base + threadIdx.x; j < base + LZ_TILE; j += 256)
        if (j <= last) out[j] = SA[j] - (q0 == q1 ? o0 : (u32)off[sid[j]]);
}

__global__ __launch_bounds__(256) void k_batch_extract(const u32 *__restrict__ gSA, const u32 *__restrict__ gLCP,
                                                       const u32 *__restrict__ sid, const int64_t *__restrict__ off,
                                                       const u32 *__restrict__ ISA, const uint8_t *__restrict__ T,
                                                       u64 N, u32 *__restrict__ outSA, u32 *__restrict__ outLCP,
                                                       uint8_t *__restrict__ outU)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 j = (u64)blockIdx.x * blockDim.x + threadIdx.x; j < N; j += stride) {
        const u32 k = sid[j];
        const u64 o = (u64)off[k];
        if (j == o) continue;                 // the separator's own suffix
        const u64 jj = j - o - 1;             // slot inside job k's suffix array
        const u64 po = o - k;                 // packed output offset of job k
        const u32 v = gSA[j] - (u32)o;        // suffix index inside job k
        outSA[po + jj] = v;
        if (outLCP) outLCP[po + jj] = gLCP[j];
        if (outU) {
            const u64 nk = (u64)off[k + 1] - o - 1;
            const u64 j0 = (u64)isa_rank(ISA[o], N) - o - 1;
            if (v == 0) outU[po] = T[o + nk - 1];
            else outU[po + jj + (jj < j0)] = T[o + v - 1];
        }
    }
}

__global__ void k_batch_primary(const u32 *__restrict__ ISA, const int64_t *__restrict__ off, u32 count, u64 N,
                                u32 *__restrict__ prim)
{
    for (u32 q = blockIdx.x * blockDim.x + threadIdx.x; q < count; q += gridDim.x * blockDim.x)
        prim[q] = isa_rank(ISA[off[q]], N) - (u32)off[q];
}

// Plain device copy, 16 bytes per lane per step (the copy-bandwidth yardstick).
__global__ __launch_bounds__(256) void k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, u64 count)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) dst[i] = src[i];
}

__global__ void k_copy_tail(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, u64 count)
{
    for (u64 i = threadIdx.x; i < count; i += blockDim.x) dst[i] = src[i];
}

__global__ void k_fill_u32(u32 *p, u64 count, u32 v)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) p[i] = v;
}

__global__ void k_fill_u8(uint8_t *p, u64 count, uint8_t v)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) p[i] = v;
}

__global__ void k_fill_u64(u64 *p, u64 count, u64 v)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) p[i] = v;
}

// Integer alphabet: packed keys of `k` symbols of `bits` bits each read from a u32
// symbol array (values < 2^bits).  Past the end reads 0, as for bytes.
__global__ __launch_bounds__(PK_THREADS) void k_pack_int(const u32 *__restrict__ S, u64 n, int bits, int k, int gsa,
                                                         u32 *__restrict__ keys, u32 *__restrict__ vals)
{
    __shared__ u32 s_c[PK_TILE + PK_HALO];
    const u64 base = (u64)blockIdx.x * PK_TILE;
    for (int i = threadIdx.x; i < PK_TILE + PK_HALO; i += PK_THREADS) {
        u64 p = base + i;
        s_c[i] = p < n ? S[p] : 0u;
    }
    __syncthreads();
    for (int j = 0; j < PK_ITEMS; j++) {
        int li = j * PK_THREADS + threadIdx.x;
        u64 p = base + li;
        if (p >= n) break;
        u32 key = 0;
        bool sep = false;
        for (int t = 0; t < k; t++) {
            u32 c = s_c[li + t];
            if (gsa) {  // code 0 is the separator: everything after the first one reads 0
                if (sep) c = 0;
                sep = sep || c == 0;
            }
            key = (bits >= 32 ? 0u : key << bits) | c;
        }
        keys[p] = key;
        vals[p] = (u32)p;
    }
}

// Largest symbol value (as unsigned), for the symbol width.  One atomic per workgroup:
// the maxima of all waves land on one address, and 16384 of them (one per wave of 4096
// workgroups) took 137 us for 6 M symbols, where the reads take about 5 us.
template <typename ST>
__global__ __launch_bounds__(256) void k_max_sym(const ST *__restrict__ T, u64 n, u64 *__restrict__ out)
{
    __shared__ u64 s_m[256 / SAGPU_WAVE];
    u64 m = 0;
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        u64 v = sizeof(ST) == 4 ? (u64)(u32)T[i] : (u64)T[i];
        m = v > m ? v : m;
    }
    m = wave_incl_max64(m);
    if (lane_id() == SAGPU_WAVE - 1) s_m[threadIdx.x / SAGPU_WAVE] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < 256 / SAGPU_WAVE; q++) m = s_m[q] > m ? s_m[q] : m;
        m = s_m[0] > m ? s_m[0] : m;
        if (m) atomicMax((unsigned long long *)out, (unsigned long long)m);
    }
}

// Symbols as sort keys (u32 narrowing when the values are known to fit, or u64)
// with their positions for dense ranking (vals may be null).
template <typename ST, typename K>
__global__ __launch_bounds__(256) void k_sym_keys(const ST *__restrict__ T, u64 n, K *__restrict__ keys,
                                                  u32 *__restrict__ vals)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        keys[i] = sizeof(ST) == 4 ? (K)(u32)T[i] : (K)(u64)T[i];
        if (vals) vals[i] = (u32)i;
    }
}

// After sorting (value, position): flag[e] = 1 where a new value starts.
template <typename K>
__global__ __launch_bounds__(256) void k_run_flags(const K *__restrict__ keys, u64 n, u32 *__restrict__ flags)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 e = (u64)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride)
        flags[e] = (e == 0 || keys[e] != keys[e - 1]) ? 1u : 0u;
}

// S[position] = dense rank (number of distinct smaller values), from the exclusive
// scan of the run flags.
template <typename K>
__global__ __launch_bounds__(256) void k_dense_scatter(const K *__restrict__ keys, const u32 *__restrict__ vals,
                                                       const u32 *__restrict__ excl, u64 n, u32 *__restrict__ S)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 e = (u64)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) {
        const u32 f = (e == 0 || keys[e] != keys[e - 1]) ? 1u : 0u;
        S[vals[e]] = excl[e] + f - 1;
    }
}

// Dense ranks of an integer alphabet through a table of its values: table[v] = 1 where
// value v occurs, an exclusive scan turns that into v's rank, and a gather replaces
// the symbols.  The flag is read before it is written: in Zipf-like texts most symbols
// find it set, and the few hot words would otherwise take every write.
template <typename ST>
__global__ __launch_bounds__(256) void k_mark_values(const ST *__restrict__ T, u64 n, u32 *__restrict__ table)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        u32 *f = table + (u32)T[i];
        if (!*f) *f = 1u;
    }
}

template <typename ST>
__global__ __launch_bounds__(256) void k_value_ranks(const ST *__restrict__ T, u64 n, const u32 *__restrict__ table,
                                                     u32 *__restrict__ S)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) S[i] = table[(u32)T[i]];
}

// 65536-bin histogram of 16-bit symbols.  Each workgroup counts stretches of at most
// H16_TILE symbols in LDS, two 16-bit counters per word (H16_TILE < 65536, so a half
// never carries), and adds the bins it met to the global table: a symbol of a
// Zipf-like text costs one LDS atomic instead of a global one on a few hot addresses
// (4 M token ids: 790 us with one global atomic per distinct symbol of a wave step).
// 128 KB of counters are one workgroup per CU, so it has 1024 threads.  In GSA mode it
// also counts the invalid positions (a 0 first, or two adjacent 0s).
constexpr u32 H16_TILE = 16384, H16_THREADS = 1024;

__global__ __launch_bounds__(H16_THREADS) void k_hist16(const uint16_t *__restrict__ T, u64 n, u64 span, int gsa,
                                                        u64 *__restrict__ hist, u32 *__restrict__ bad)
{
    __shared__ u32 s_h[32768];
    u32 nbad = 0;
    const u64 lo = (u64)blockIdx.x * span, hi = lo + span < n ? lo + span : n;
    for (u64 base = lo; base < hi; base += H16_TILE) {
        for (u32 b = threadIdx.x; b < 32768; b += H16_THREADS) s_h[b] = 0;
        __syncthreads();
        const u64 end = base + H16_TILE < hi ? base + H16_TILE : hi;
        for (u64 i = base + threadIdx.x; i < end; i += H16_THREADS) {
            const u32 v = T[i];
            if (gsa && v == 0 && (i == 0 || T[i - 1] == 0)) nbad++;
            atomicAdd(&s_h[v >> 1], 1u << (16 * (v & 1)));
        }
        __syncthreads();
        for (u32 b = threadIdx.x; b < 32768; b += H16_THREADS) {
            const u32 x = s_h[b];
            if (x & 0xFFFFu) atomicAdd((unsigned long long *)&hist[2 * b], (unsigned long long)(x & 0xFFFFu));
            if (x >> 16) atomicAdd((unsigned long long *)&hist[2 * b + 1], (unsigned long long)(x >> 16));
        }
        __syncthreads();
    }
    if (gsa && nbad) atomicAdd(bad, nbad);
}

// Dense codes of 16-bit symbols through a 65536-entry table.
__global__ __launch_bounds__(256) void k_map16(const uint16_t *__restrict__ T, u64 n, const u32 *__restrict__ lut,
                                               u32 *__restrict__ S)
{
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) S[i] = lut[T[i]];
}

unsigned grid_for(u64 work, unsigned per_block, unsigned cap)
{
    u64 b = (work + per_block - 1) / per_block;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (unsigned)b;
}

} // namespace

int launch_histogram(const uint8_t *T, u64 n, int gsa, u64 *hist, uint8_t *pad, uint8_t *lut, uint8_t *inv, u64 *host,
                     hipStream_t s)
{
    hipLaunchKernelGGL(k_histogram, dim3(grid_for(n, 256 * 16 * 8, 2048)), dim3(256), 0, s, T, n, gsa, hist, pad);
    hipLaunchKernelGGL(k_alphabet, dim3(1), dim3(256), 0, s, hist, lut, inv, host);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_pack_keys32(const uint8_t *T, u64 n, const uint8_t *lut, int bits, int k, int gsa, int cb, u32 *keys,
                       u32 *vals, hipStream_t s)
{
    if (k > PK_HALO || k * bits > 32 || (cb && (u64)(n - 1) >> (32 - cb))) {
        sagpu_set_error("pack32: bad symbol count", __FILE__, __LINE__);
        return SAGPU_EDEVICE;
    }
    const int items = n < (1u << 20) ? 1 : PK_ITEMS;
    hipLaunchKernelGGL(k_pack_keys32, dim3(ceil_div_u(n, (u64)PK_THREADS * items)), dim3(PK_THREADS), 0, s, T, n, lut,
                       bits, k, gsa, cb, keys, vals, items);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_hist16(const uint16_t *T, u64 n, int gsa, u64 *hist65536, u32 *bad, hipStream_t s)
{
    // whole tiles per workgroup, at most 1024 workgroups (four rounds over the 256 CUs)
    const u64 tiles = (n + H16_TILE - 1) / H16_TILE;
    const u64 per = (tiles + 1023) / 1024;
    hipLaunchKernelGGL(k_hist16, dim3(ceil_div_u(tiles, per)), dim3(H16_THREADS), 0, s, T, n, per * H16_TILE, gsa,
                       hist65536, bad);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_map16(const uint16_t *T, u64 n, const u32 *lut, u32 *S, hipStream_t s)
{
    hipLaunchKernelGGL(k_map16, dim3(grid_for(n, 256 * 8, 65535)), dim3(256), 0, s, T, n, lut, S);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_pack_int(const u32 *S, u64 n, int bits, int k, int gsa, u32 *keys, u32 *vals, hipStream_t s)
{
    if (k > PK_HALO || k * bits > 32 || k < 1) {
        sagpu_set_error("pack_int: bad symbol count", __FILE__, __LINE__);
        return SAGPU_EDEVICE;
    }
    hipLaunchKernelGGL(k_pack_int, dim3(ceil_div_u(n, PK_TILE)), dim3(PK_THREADS), 0, s, S, n, bits, k, gsa, keys,
                       vals);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_max_sym(const void *T, int width, u64 n, u64 *out, hipStream_t s)
{
    if (width == 4)
        hipLaunchKernelGGL(k_max_sym<int32_t>, dim3(grid_for(n, 256 * 16, 1024)), dim3(256), 0, s, (const int32_t *)T,
                           n, out);
    else
        hipLaunchKernelGGL(k_max_sym<int64_t>, dim3(grid_for(n, 256 * 16, 1024)), dim3(256), 0, s, (const int64_t *)T,
                           n, out);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_sym_narrow(const void *T, int width, u64 n, u32 *S, hipStream_t s)
{
    if (width == 4)
        hipLaunchKernelGGL((k_sym_keys<int32_t, u32>), dim3(grid_for(n, 256 * 8, 65535)), dim3(256), 0, s,
                           (const int32_t *)T, n, S, (u32 *)nullptr);
    else
        hipLaunchKernelGGL((k_sym_keys<int64_t, u32>), dim3(grid_for(n, 256 * 8, 65535)), dim3(256), 0, s,
                           (const int64_t *)T, n, S, (u32 *)nullptr);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_sym_keys64(const void *T, int width, u64 n, u64 *keys, u32 *vals, hipStream_t s)
{
    if (width == 4)
        hipLaunchKernelGGL((k_sym_keys<int32_t, u64>), dim3(grid_for(n, 256 * 8, 65535)), dim3(256), 0, s,
                           (const int32_t *)T, n, keys, vals);
    else
        hipLaunchKernelGGL((k_sym_keys<int64_t, u64>), dim3(grid_for(n, 256 * 8, 65535)), dim3(256), 0, s,
                           (const int64_t *)T, n, keys, vals);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_mark_values(const void *T, int width, u64 n, u32 *table, hipStream_t s)
{
    const dim3 g(grid_for(n, 256 * 8, 65535));
    if (width == 4) hipLaunchKernelGGL(k_mark_values<int32_t>, g, dim3(256), 0, s, (const int32_t *)T, n, table);
    else hipLaunchKernelGGL(k_mark_values<int64_t>, g, dim3(256), 0, s, (const int64_t *)T, n, table);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_value_ranks(const void *T, int width, u64 n, const u32 *table, u32 *S, hipStream_t s)
{
    const dim3 g(grid_for(n, 256 * 8, 65535));
    if (width == 4) hipLaunchKernelGGL(k_value_ranks<int32_t>, g, dim3(256), 0, s, (const int32_t *)T, n, table, S);
    else hipLaunchKernelGGL(k_value_ranks<int64_t>, g, dim3(256), 0, s, (const int64_t *)T, n, table, S);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_run_flags64(const u64 *keys, u64 n, u32 *flags, hipStream_t s)
{
    hipLaunchKernelGGL(k_run_flags<u64>, dim3(grid_for(n, 256 * 8, 65535)), dim3(256), 0, s, keys, n, flags);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_dense_scatter64(const u64 *keys, const u32 *vals, const u32 *excl, u64 n, u32 *S, hipStream_t s)
{
    hipLaunchKernelGGL(k_dense_scatter<u64>, dim3(grid_for(n, 256 * 8, 65535)), dim3(256), 0, s, keys, vals, excl, n,
                       S);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

static u64 string_tiles(u64 n) { return (n + SI_TILE - 1) / SI_TILE; }
u64 string_ids_words(u64 n) { return string_tiles(n) + string_tiles(n) / 4096 + 2; }
int launch_string_ids(const uint8_t *T, u64 n, u32 *sid, u32 *part, hipStream_t s)
{
    const u64 tiles = string_tiles(n);
    hipLaunchKernelGGL(k_string_counts, dim3((unsigned)tiles), dim3(256), 0, s, T, n, part);
    ScanScratch sc{part + tiles, tiles / 4096 + 2};
    SAGPU_TRY(scan_exclusive_u32(sc, part, tiles, s));
    hipLaunchKernelGGL(k_string_ids, dim3((unsigned)tiles), dim3(256), 0, s, T, n, (const u32 *)part, sid);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_pack_keys32_sid(const uint8_t *T, u64 n, const uint8_t *lut, int bits, int k, const u32 *sid,
                           const uint8_t *local, u32 *keys, hipStream_t s)
{
    if (k > PK_HALO || k < 1 || k * bits > 32) {
        sagpu_set_error("pack_keys: bad symbol count", __FILE__, __LINE__);
        return SAGPU_EDEVICE;
    }
    hipLaunchKernelGGL(k_pack_keys32_sid, dim3(ceil_div_u(n, PK_TILE)), dim3(PK_THREADS), 0, s, T, n, lut, bits, k, sid,
                       local, keys);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_pack_keys64_sid(const uint8_t *T, u64 n, const uint8_t *lut, int bits, int k, const u32 *sid, u64 *keys,
                           u32 *vals, hipStream_t s)
{
    if (k > PK_HALO || k * bits > 32) {
        sagpu_set_error("pack64: bad symbol count", __FILE__, __LINE__);
        return SAGPU_EDEVICE;
    }
    hipLaunchKernelGGL(k_pack_keys64_sid, dim3(ceil_div_u(n, PK_TILE)), dim3(PK_THREADS), 0, s, T, n, lut, bits, k,
                       sid, keys, vals);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_check_offsets(const uint8_t *T, const u32 *sid, const int64_t *offsets, u32 count, u32 *bad, hipStream_t s)
{
    hipLaunchKernelGGL(k_check_offsets, dim3(grid_for(count, 256, 4096)), dim3(256), 0, s, T, sid, offsets, count,
                       bad);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_localize(const u32 *SA, const u32 *sid, const int64_t *offsets, u64 n, u32 *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_localize, dim3((unsigned)((n + LZ_TILE - 1) / LZ_TILE)), dim3(256), 0, s, SA, sid, offsets, n, out);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_batch_extract(const u32 *gSA, const u32 *gLCP, const u32 *sid, const int64_t *off, const u32 *ISA,
                         const uint8_t *T, u64 N, u32 *outSA, u32 *outLCP, uint8_t *outU, hipStream_t s)
{
    hipLaunchKernelGGL(k_batch_extract, dim3(grid_for(N, 256 * 8, 65535)), dim3(256), 0, s, gSA, gLCP, sid, off, ISA,
                       T, N, outSA, outLCP, outU);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_batch_primary(const u32 *ISA, const int64_t *off, u32 count, u64 N, u32 *prim, hipStream_t s)
{
    hipLaunchKernelGGL(k_batch_primary, dim3(grid_for(count, 256, 4096)), dim3(256), 0, s, ISA, off, count, N, prim);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_fill_u32(u32 *p, u64 count, u32 value, hipStream_t s)
{
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(count, 256 * 4, 16384)), dim3(256), 0, s, p, count, value);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_copy(void *dst, const void *src, u64 bytes, hipStream_t s)
{
    const u64 vec = ((uintptr_t)dst % 16 == 0 && (uintptr_t)src % 16 == 0) ? bytes / 16 : 0;
    if (vec) {
        u64 blocks = (vec + 256 * 4 - 1) / (256 * 4);
        if (blocks > 8192) blocks = 8192;
        hipLaunchKernelGGL(k_copy16, dim3((unsigned)blocks), dim3(256), 0, s, (const uint4 *)src, (uint4 *)dst, vec);
    }
    if (bytes > vec * 16)
        hipLaunchKernelGGL(k_copy_tail, dim3(1), dim3(256), 0, s, (const uint8_t *)src + vec * 16,
                           (uint8_t *)dst + vec * 16, bytes - vec * 16);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_fill_u8(uint8_t *p, u64 count, uint8_t value, hipStream_t s)
{
    if (!count) return SAGPU_OK;
    hipLaunchKernelGGL(k_fill_u8, dim3(grid_for(count, 256 * 16, 16384)), dim3(256), 0, s, p, count, value);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}

int launch_fill_u64(u64 *p, u64 count, u64 value, hipStream_t s)
{
    hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(count, 256 * 4, 16384)), dim3(256), 0, s, p, count, value);
    SAGPU_CHECK(hipGetLastError());
    return SAGPU_OK;
}
