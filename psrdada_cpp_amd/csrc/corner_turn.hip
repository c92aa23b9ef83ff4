// corner_turn.hip -- the byte reorders either side of the beamformer.
//
//   fbf_tuse_transpose  TUSE beam corner turn after it
//                       (meerkat/tuse/src/transpose_to_dada.cpp:19-48)
//   fbf_feng_to_dada    F-engine heap reorder before it
//                       (meerkat/tools/src/feng_to_dada.cu:54-80)
//
// Both are, per batch, the transpose of an R x C matrix of E-byte elements.
// A work-group stages a TR x TC tile of elements through LDS so that global
// reads are runs of input rows (TC elements, contiguous) and global writes
// runs of output rows, moving 16-, 4- or 1-byte units.  HBM-bound: every byte
// is read once and written once.
//
// In 16-byte units a block of 8 MiB or more is stored past the cache, which
// leaves the cache to what is read, and one of 128 MiB or more is read past it
// too.  On blocks that are not in the cache yet (us: all cached, stores past it,
// both; F-engine channels / heaps or TUSE channels / samples / bands / beams /
// groups):
//   1280/9,            12 MB     5.2    4.4    5.1
//   4096/16,           67 MB    26.7   19.9   24.0
//   64/64/16/128/8,    67 MB    31.2   20.6   24.4
//   128/64/32/64/10,  168 MB    63.3   61.5   54.3
//   4096/64,          268 MB    99.3   95.1   94.0
// Word tiles whose output rows are not whole 128-byte lines are stored past it
// from 16 MiB (132/96, 13 MB 5.9 cached and 7.3 past; 3152/16, 52 MB 22.8 and
// 16.1), 4-byte units never (3394/10, 35 MB 14.4 and 16.3).
#include "fbf_internal.hpp"

#include <algorithm>

#include <climits>

namespace fbf {
namespace {

// A tile's input or output rows of n units, walked by 256 threads a step.
struct CtRow {
    uint32_t inv;   // ceil(2^32 / n)
    int rows, k;    // 256 = rows * n + k
};

struct CtArgs {
    const uint8_t* in;
    uint8_t* out;
    long long n2;                  // batch index z = i1 * n2 + i2
    long long in_s1, in_s2;        // byte offsets of batch (i1, i2)
    long long out_s1, out_s2;
    int R, C;                      // input rows and columns (elements)
    int EU;                        // units per element
    int TR, TC;                    // tile rows and columns (elements)
    int tiles_r, tiles_c;
    int sh_ru, sh_eu;              // square tiles: log2(TC * EU), log2(EU) (when powers of two)
    uint32_t inv_eu;               // ceil(2^32 / EU)
    CtRow in_row[2], out_row[2];   // of a full and of the last tile
};

// Past the cache: neither loads nor stores, the stores, both.
enum { CT_CACHED = 0, CT_STORE = 1, CT_BOTH = 2 };

// A store and a load, of 16 bytes past the cache or not.
template <int PAST, typename U>
__device__ __forceinline__ void store_unit(const U& v, U* p)
{
    if constexpr (PAST != CT_CACHED) {
        static_assert(sizeof(U) == 16, "units past the cache");
        typedef uint32_t v4u __attribute__((ext_vector_type(4)));
        __builtin_nontemporal_store(v4u{v.x, v.y, v.z, v.w}, reinterpret_cast<v4u*>(p));
    } else {
        *p = v;
    }
}

template <int PAST, typename U>
__device__ __forceinline__ U load_unit(const U* p)
{
    if constexpr (PAST == CT_BOTH) {
        const int4 v = load_stream(p);
        return U{(uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w};
    } else {
        return *p;
    }
}

// i / n of a unit index with inv = ceil(2^32 / n) (exact: both are below 2^16).
__device__ __forceinline__ int ct_div(int i, int n, uint32_t inv) { return n == 1 ? i : (int)__umulhi((uint32_t)i, inv); }

// A work-group's tile: its corner in the input and the output, and its size.
template <typename U>
struct CtTile {
    const U* src;
    U* dst;
    size_t in_row, out_row;   // units
    int nr, nc, ru, ou;       // rows, columns, units of an input and of an output row
};

template <typename U>
__device__ __forceinline__ CtTile<U> ct_tile(const CtArgs& a, long long bid)
{
    const int tc = (int)(bid % a.tiles_c);
    bid /= a.tiles_c;
    const int tr = (int)(bid % a.tiles_r);
    bid /= a.tiles_r;
    const long long i2 = bid % a.n2;
    const long long i1 = bid / a.n2;
    const int r0 = tr * a.TR, c0 = tc * a.TC;
    CtTile<U> t;
    t.in_row = (size_t)a.C * a.EU;
    t.out_row = (size_t)a.R * a.EU;
    t.src = reinterpret_cast<const U*>(a.in + i1 * a.in_s1 + i2 * a.in_s2) + (size_t)r0 * t.in_row + (size_t)c0 * a.EU;
    t.dst = reinterpret_cast<U*>(a.out + i1 * a.out_s1 + i2 * a.out_s2) + (size_t)c0 * t.out_row + (size_t)r0 * a.EU;
    t.nr = min(a.TR, a.R - r0);
    t.nc = min(a.TC, a.C - c0);
    t.ru = t.nc * a.EU;
    t.ou = t.nr * a.EU;
    return t;
}

// The tile's row pitch in LDS is TC * EU + 1 units, so that the transposed
// reads of the write phase (threads stepping down the tile rows) fall in
// distinct banks.
//
// Three ways to walk a tile, none best everywhere (us, the block in the cache):
//                                   units   rows   steps
//   16 bytes, 192/64/32/64/4         38.2   70.6    42.7
//   16 bytes, 80/128/20/40/8         22.1      -    23.6
//    4 bytes, 8/22/3/412/6            4.8    6.0     5.1
//    4 bytes, 52/62/21/61/9          28.7   18.4    25.4
//    4 bytes, 999/100                47.0   37.5    45.4
//    4 bytes, 132/467/8/3/3           5.9    8.1     5.9
//    4 bytes, 191/12                  4.0    4.3     3.6
//    1 byte,  23/92/44/72/1          12.3   10.8    11.9
//    1 byte,  21/222/21/2/8           6.1    7.2     5.4

// 16-byte units, and tiles of up to two units a thread: the threads take
// consecutive units, each split into (row, unit of the row) by a multiplication.
// POW2: shifts where the tile is full, TC * EU and EU being powers of two.
template <typename U, bool POW2, int PAST>
__global__ __launch_bounds__(256) void corner_turn_units_k(CtArgs a)
{
    extern __shared__ __align__(16) uint8_t ct_lds[];
    U* tile = reinterpret_cast<U*>(ct_lds);
    const CtTile<U> t = ct_tile<U>(a, blockIdx.x);
    const int EU = a.EU, pitch = a.TC * EU + 1, n = t.nr * t.ru;
    if (POW2 && t.nr == a.TR && t.nc == a.TC) {
        const int mu = (1 << a.sh_ru) - 1, me = EU - 1;
        for (int i = threadIdx.x; i < n; i += 256) {
            const int r = i >> a.sh_ru, k = i & mu;
            tile[r * pitch + k] = load_unit<PAST>(t.src + (size_t)r * t.in_row + k);
        }
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += 256) {
            const int c = i >> a.sh_ru, k = i & mu;
            const int r = k >> a.sh_eu, e = k & me;
            store_unit<PAST>(tile[r * pitch + c * EU + e], t.dst + (size_t)c * t.out_row + k);
        }
        return;
    }
    const uint32_t inv_ru = a.in_row[t.nc != a.TC].inv, inv_ou = a.out_row[t.nr != a.TR].inv;
    for (int i = threadIdx.x; i < n; i += 256) {
        const int r = ct_div(i, t.ru, inv_ru), k = i - r * t.ru;
        tile[r * pitch + k] = load_unit<PAST>(t.src + (size_t)r * t.in_row + k);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 256) {
        const int c = ct_div(i, t.ou, inv_ou), k = i - c * t.ou;
        const int r = ct_div(k, EU, a.inv_eu);
        store_unit<PAST>(tile[r * pitch + c * EU + k - r * EU], t.dst + (size_t)c * t.out_row + k);
    }
}

// 4- and 1-byte units in few or small tiles: the threads take consecutive
// units, so none is idle in tiles of few or narrow rows; a thread finds its
// first unit's row by multiplication and steps on from there by additions.
template <typename U>
__global__ __launch_bounds__(256) void corner_turn_steps_k(CtArgs a)
{
    extern __shared__ __align__(16) uint8_t ct_lds[];
    U* tile = reinterpret_cast<U*>(ct_lds);
    const CtTile<U> t = ct_tile<U>(a, blockIdx.x);
    const int EU = a.EU, pitch = a.TC * EU + 1, n = t.nr * t.ru;
    const int tid = threadIdx.x;
    {
        const CtRow w = a.in_row[t.nc != a.TC];
        const int r = ct_div(tid, t.ru, w.inv);
        int k = tid - r * t.ru;
        const U* src = t.src + (size_t)r * t.in_row + k;
        int l = r * pitch + k;
        const size_t step = (size_t)w.rows * t.in_row + w.k;
        const int lstep = w.rows * pitch + w.k;
        for (int i = tid; i < n; i += 256) {
            tile[l] = *src;
            k += w.k;
            src += step;
            l += lstep;
            if (k >= t.ru) {
                k -= t.ru;
                src += t.in_row - t.ru;
                l += pitch - t.ru;
            }
        }
    }
    __syncthreads();
    {
        const CtRow w = a.out_row[t.nr != a.TR];
        const int c = ct_div(tid, t.ou, w.inv), k = tid - c * t.ou;
        int r = ct_div(k, EU, a.inv_eu), e = k - r * EU;
        U* dst = t.dst + (size_t)c * t.out_row + k;
        int l = r * pitch + c * EU + e;
        const int rstep = ct_div(w.k, EU, a.inv_eu), estep = w.k - rstep * EU;
        const size_t step = (size_t)w.rows * t.out_row + w.k;
        const int lstep = rstep * pitch + w.rows * EU + estep;
        for (int i = tid; i < n; i += 256) {
            *dst = tile[l];
            e += estep;
            r += rstep;
            dst += step;
            l += lstep;
            if (e >= EU) {
                e -= EU;
                ++r;
                l += pitch - EU;
            }
            if (r >= t.nr) {
                r -= t.nr;
                dst += t.out_row - t.ou;
                l += EU - t.nr * pitch;
            }
        }
    }
}

// 4- and 1-byte units in many tiles of more than 1024: a wave takes rows, its
// lanes the units of a row.
template <typename U>
__global__ __launch_bounds__(256) void corner_turn_rows_k(CtArgs a)
{
    extern __shared__ __align__(16) uint8_t ct_lds[];
    U* tile = reinterpret_cast<U*>(ct_lds);
    const CtTile<U> t = ct_tile<U>(a, blockIdx.x);
    const int EU = a.EU, pitch = a.TC * EU + 1;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (t.nr < 4) {
        // A wave per row would leave some without one.
        for (int r = 0; r < t.nr; ++r)
            for (int k = threadIdx.x; k < t.ru; k += 256) tile[r * pitch + k] = t.src[(size_t)r * t.in_row + k];
    } else {
        for (int r = wave; r < t.nr; r += 16) {   // up to four rows' loads in flight
            for (int k = lane; k < t.ru; k += 64) {
                U v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (r + 4 * j < t.nr) v[j] = t.src[(size_t)(r + 4 * j) * t.in_row + k];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (r + 4 * j < t.nr) tile[(r + 4 * j) * pitch + k] = v[j];
            }
        }
    }
    __syncthreads();
    if (t.ou <= 16) {
        // Output rows of few units: a wave of the loop below would be nearly
        // empty (1 channel, 4000 samples, 2 bands, 200 beams, 4 groups: 94 us
        // through it, 9.4 here).
        const uint32_t inv_ou = a.out_row[t.nr != a.TR].inv;
        for (int i = threadIdx.x; i < t.nc * t.ou; i += 256) {
            const int c = ct_div(i, t.ou, inv_ou), k = i - c * t.ou;
            const int r = ct_div(k, EU, a.inv_eu);
            t.dst[(size_t)c * t.out_row + k] = tile[r * pitch + c * EU + k - r * EU];
        }
        return;
    }
    for (int k = lane; k < t.ou; k += 64) {
        const int r = ct_div(k, EU, a.inv_eu);
        const U* u = tile + r * pitch + (k - r * EU);
        for (int c = wave; c < t.nc; c += 4) t.dst[(size_t)c * t.out_row + k] = u[c * EU];
    }
}

// 4-byte elements, 64 x 64 tiles: 16-byte global loads (4 words of an
// input row) and stores (4 words of an output row); the tile stays in
// 4-byte LDS words with a 65-word pitch, which keeps both the row writes
// and the column reads free of bank conflicts.  Rows and columns come in
// fours, so edge tiles do the same, with what lies past them left out (word by
// word, 176 channels, 2 heaps took 5.3 us, 3.2 so).
template <int PAST>
__global__ __launch_bounds__(256) void corner_turn_w4_k(CtArgs a)
{
    extern __shared__ __align__(16) uint8_t ct_lds[];
    uint32_t* tile = reinterpret_cast<uint32_t*>(ct_lds);
    constexpr int P = 65;
    const CtTile<uint32_t> t = ct_tile<uint32_t>(a, blockIdx.x);
    const int i16 = threadIdx.x >> 4, k4 = (threadIdx.x & 15) << 2;
    // Loads past the tile's edge read its last row or columns again.
    uint4 v[4];
    const int kc = min(k4, t.nc - 4);
#pragma unroll
    for (int j = 0; j < 4; ++j)
        v[j] = load_unit<PAST>(reinterpret_cast<const uint4*>(t.src + (size_t)min(i16 + 16 * j, t.nr - 1) * t.in_row + kc));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t* l = tile + (i16 + 16 * j) * P + k4;
        l[0] = v[j].x;
        l[1] = v[j].y;
        l[2] = v[j].z;
        l[3] = v[j].w;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int c = i16 + 16 * j;
        const uint4 o{tile[k4 * P + c], tile[(k4 + 1) * P + c], tile[(k4 + 2) * P + c], tile[(k4 + 3) * P + c]};
        if (c < t.nc && k4 < t.nr) store_unit<PAST>(o, reinterpret_cast<uint4*>(t.dst + (size_t)c * t.out_row + k4));
    }
}

inline int ilog2_exact(long long v)
{
    if (v <= 0 || (v & (v - 1)) != 0) return -1;
    int s = 0;
    while ((1ll << s) < v) ++s;
    return s;
}

// Tile: square, the edge the largest power of two up to 64 whose rows hold
// at most 1 KiB within the LDS budget; where the matrix has fewer rows than
// that, all of them and as many more columns.  Rows of 64 units left 1- and
// 4-byte units with tiles of one or two elements (23 channels, 92 samples, 44
// bands, 72 beams, 1 group, 13 MB moved: 75 us, 11 us so).
constexpr size_t kCtLdsMax = 32 * 1024;
constexpr size_t kCtRow = 1024;

inline size_t ct_tile_bytes(int TR, int TC, int EU, size_t U)
{
    return (size_t)TR * ((size_t)TC * EU + 1) * U;
}

// Tile and row constants, and the number of tiles.
int ct_plan(CtArgs& a, long long n1, int E, size_t U, long long* nblocks)
{
    a.EU = E / (int)U;
    int T = 64;
    while (T > 1 && ((size_t)T * E > kCtRow || ct_tile_bytes(T, T, a.EU, U) > kCtLdsMax)) T >>= 1;
    auto tiles = [&](int tr, int tc) { return n1 * a.n2 * ((a.R + tr - 1) / tr) * ((a.C + tc - 1) / tc); };
    // A small block takes smaller tiles, down to two units a thread, to fill
    // the chip (7 channels, 900 samples, 40 bands, 2 beams, 1 group: 13.3 us in
    // tiles of 256-byte rows, 4.0 so).
    while (T > 1 && T * T * a.EU > 512 && tiles(T, T) < 512) T >>= 1;
    a.TR = a.TC = T;
    if (a.R < T) {
        a.TR = a.R;
        for (int tc = std::min(T * T / a.R, (a.C + T - 1) / T * T); tc > T && a.TC == T; tc -= T)
            if (ct_tile_bytes(a.TR, tc, a.EU, U) <= kCtLdsMax && tiles(a.TR, tc) >= 512) a.TC = tc;
    }
    FBF_REQUIRE(ct_tile_bytes(1, 1, a.EU, U) <= kCtLdsMax, FBF_ERR_UNSUPPORTED,
                "corner turn: element too large (at most 32 KiB - 16 B)");
    a.tiles_r = (a.R + a.TR - 1) / a.TR;
    a.tiles_c = (a.C + a.TC - 1) / a.TC;
    *nblocks = n1 * a.n2 * a.tiles_r * a.tiles_c;
    FBF_REQUIRE(*nblocks < INT_MAX, FBF_ERR_UNSUPPORTED, "corner turn: too many tiles for one launch");
    a.sh_ru = ilog2_exact((long long)a.TC * a.EU);
    a.sh_eu = ilog2_exact(a.EU);
    auto inverse = [](long long n) { return (uint32_t)(((1ull << 32) + n - 1) / n); };   // (0 for 1, unused)
    auto row = [&](long long n) { return CtRow{inverse(n), (int)(256 / n), (int)(256 % n)}; };
    a.inv_eu = inverse(a.EU);
    a.in_row[0] = row((long long)a.TC * a.EU);
    a.in_row[1] = row((long long)(a.C - (a.tiles_c - 1) * a.TC) * a.EU);
    a.out_row[0] = row((long long)a.TR * a.EU);
    a.out_row[1] = row((long long)(a.R - (a.tiles_r - 1) * a.TR) * a.EU);
    return FBF_OK;
}

template <int PAST>
void ct_launch_units(const CtArgs& a, bool pow2, dim3 grid, size_t shm, hipStream_t s)
{
    if (pow2)
        corner_turn_units_k<uint4, true, PAST><<<grid, 256, shm, s>>>(a);
    else
        corner_turn_units_k<uint4, false, PAST><<<grid, 256, shm, s>>>(a);
}

template <typename U>
int ct_launch_u(CtArgs a, long long n1, int E, int past, hipStream_t s)
{
    long long nblocks = 0;
    const int st = ct_plan(a, n1, E, sizeof(U), &nblocks);
    if (st) return st;
    if (nblocks == 0) return FBF_OK;
    const size_t shm = ct_tile_bytes(a.TR, a.TC, a.EU, sizeof(U));
    const dim3 grid((unsigned)nblocks);
    const long long units = (long long)a.TR * std::min(a.TC, a.C) * a.EU;   // of a tile
    if constexpr (sizeof(U) == 16) {
        // (From tiles of four elements a row: of one or two, the shifts gain
        // nothing; 1024/64/32/8/3 41.2 us without, 48.7 with.)
        const bool pow2 = a.TR == a.TC && a.TC >= 4 && a.sh_ru >= 0 && a.sh_eu >= 0;
        if (past == CT_BOTH)
            ct_launch_units<CT_BOTH>(a, pow2, grid, shm, s);
        else if (past == CT_STORE)
            ct_launch_units<CT_STORE>(a, pow2, grid, shm, s);
        else
            ct_launch_units<CT_CACHED>(a, pow2, grid, shm, s);
    } else if (units <= 512) {
        corner_turn_units_k<U, false, CT_CACHED><<<grid, 256, shm, s>>>(a);
    } else if (units > 1024 && nblocks >= 512) {
        corner_turn_rows_k<U><<<grid, 256, shm, s>>>(a);
    } else {
        corner_turn_steps_k<U><<<grid, 256, shm, s>>>(a);
    }
    FBF_HIP_TRY(hipGetLastError());
    return FBF_OK;
}

// 16-byte units when every element and base is 16-byte aligned, else 4, else 1.
int ct_launch(CtArgs a, long long n1, int E, hipStream_t s)
{
    const long long bytes = n1 * a.n2 * a.R * a.C * E;
    const int past = bytes >= (128ll << 20) ? CT_BOTH : bytes >= (8ll << 20) ? CT_STORE : CT_CACHED;
    const uintptr_t al = reinterpret_cast<uintptr_t>(a.in) | reinterpret_cast<uintptr_t>(a.out) |
                         (uintptr_t)a.in_s1 | (uintptr_t)a.in_s2 | (uintptr_t)a.out_s1 | (uintptr_t)a.out_s2;
    if (E == 4 && ((al | (uintptr_t)a.R * 4 | (uintptr_t)a.C * 4) & 15) == 0) {
        // word transposes with 16-byte global accesses (rows 16-byte aligned)
        a.EU = 1;
        a.TR = a.TC = 64;
        a.tiles_r = (a.R + 63) / 64;
        a.tiles_c = (a.C + 63) / 64;
        const long long nblocks = n1 * a.n2 * a.tiles_r * a.tiles_c;
        if (nblocks == 0) return FBF_OK;
        FBF_REQUIRE(nblocks < INT_MAX, FBF_ERR_UNSUPPORTED, "corner turn: too many tiles for one launch");
        const dim3 grid((unsigned)nblocks);
        constexpr size_t shm = 64 * 65 * 4;
        if (past == CT_BOTH)
            corner_turn_w4_k<CT_BOTH><<<grid, 256, shm, s>>>(a);
        else if (past == CT_STORE && (a.R % 32 == 0 || bytes >= (16ll << 20)))
            corner_turn_w4_k<CT_STORE><<<grid, 256, shm, s>>>(a);
        else
            corner_turn_w4_k<CT_CACHED><<<grid, 256, shm, s>>>(a);
        FBF_HIP_TRY(hipGetLastError());
        return FBF_OK;
    }
    if (E % 16 == 0 && (al & 15) == 0) return ct_launch_u<uint4>(a, n1, E, past, s);
    if (E % 4 == 0 && (al & 3) == 0) return ct_launch_u<uint32_t>(a, n1, E, past, s);
    return ct_launch_u<uint8_t>(a, n1, E, past, s);
}

}  // namespace
}  // namespace fbf

using namespace fbf;

extern "C" int fbf_tuse_transpose(const void* in, size_t in_bytes, void* out, size_t out_bytes, int nchans,
                                  int nsamples, int nfreq, int nbeams, int ngroups, int beam0, int nbeams_out,
                                  fbf_stream_t stream)
{
    FBF_REQUIRE(nchans > 0 && nsamples > 0 && nfreq > 0 && nbeams > 0 && ngroups > 0, FBF_ERR_ARG,
                "fbf_tuse_transpose: geometry values must be positive");
    FBF_REQUIRE(beam0 >= 0 && nbeams_out >= 0 && beam0 + nbeams_out <= nbeams, FBF_ERR_ARG,
                "fbf_tuse_transpose: beam range outside [0, nbeams)");
    const long long per_beam = (long long)nchans * nsamples * nfreq;   // one beam of one group
    const long long need_in = per_beam * nbeams * ngroups;
    const long long need_out = per_beam * ngroups * nbeams_out;
    FBF_REQUIRE((long long)in_bytes >= need_in, FBF_ERR_SIZE,
                "fbf_tuse_transpose: input holds " + std::to_string(in_bytes) + " bytes, the geometry needs " +
                    std::to_string(need_in));
    FBF_REQUIRE((long long)out_bytes == need_out, FBF_ERR_SIZE,
                "fbf_tuse_transpose: output must be nbeams_out * ngroups * nsamples * nfreq * nchans = " +
                    std::to_string(need_out) + " bytes");
    if (nbeams_out == 0) return FBF_OK;
    FBF_REQUIRE(in && out, FBF_ERR_ARG, "fbf_tuse_transpose: null buffer");
    CtArgs a{};
    // batch (beam bo, group g): input [g][beam0 + bo][f][s][c], output [bo][g][s][f][c]
    a.in = static_cast<const uint8_t*>(in) + (size_t)beam0 * per_beam;
    a.out = static_cast<uint8_t*>(out);
    a.n2 = ngroups;
    a.in_s1 = per_beam;
    a.in_s2 = per_beam * nbeams;
    a.out_s1 = per_beam * ngroups;
    a.out_s2 = per_beam;
    a.R = nfreq;
    a.C = nsamples;
    return ct_launch(a, nbeams_out, nchans, static_cast<hipStream_t>(stream));
}

extern "C" int fbf_feng_to_dada(const void* in, void* out, size_t bytes, int nchans, fbf_stream_t stream)
{
    FBF_REQUIRE(nchans > 0, FBF_ERR_ARG, "fbf_feng_to_dada: nchans must be positive");
    const size_t per_ts = (size_t)nchans * 256 * 4;   // MEERKAT_FENG_NSAMPS_PER_HEAP x 2 pols x char2
    FBF_REQUIRE(bytes % per_ts == 0, FBF_ERR_SIZE,
                "fbf_feng_to_dada: number of bytes is not a multiple of the bytes per timestamp "
                "(feng_to_dada.cu:30-35)");
    if (bytes == 0) return FBF_OK;
    FBF_REQUIRE(in && out, FBF_ERR_ARG, "fbf_feng_to_dada: null buffer");
    FBF_REQUIRE(in != out, FBF_ERR_ARG, "fbf_feng_to_dada: input and output must be distinct buffers");
    CtArgs a{};
    a.in = static_cast<const uint8_t*>(in);
    a.out = static_cast<uint8_t*>(out);
    a.n2 = 1;
    a.in_s1 = (long long)per_ts;
    a.out_s1 = (long long)per_ts;
    a.R = nchans;
    a.C = 256;
    return ct_launch(a, (long long)(bytes / per_ts), 4, static_cast<hipStream_t>(stream));
}
