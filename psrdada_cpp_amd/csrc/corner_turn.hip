// corner_turn.hip -- the byte reorders either side of the beamformer.
//
//   fbf_tuse_transpose  TUSE beam corner turn after it
//                       (meerkat/tuse/src/transpose_to_dada.cpp:19-48)
//   fbf_feng_to_dada    F-engine heap reorder before it
//                       (meerkat/tools/src/feng_to_dada.cu:54-80)
//
// Both are, per batch, the transpose of an R x C matrix of E-byte elements.
// corner_turn_k stages a TR x TC tile of elements through LDS so that global
// reads are runs of input rows (TC elements, contiguous) and global writes
// runs of output rows, moving 16-, 4- or 1-byte units.  HBM-bound: every byte
// is read once and written once.  A block of 16 MiB or more is stored past the
// cache, which leaves the cache to what is read, and one of 128 MiB or more
// is read past it too (64 beams, 128 channels, 64 samples, 32 bands, 10 groups,
// 336 MB moved: 65.7 us all cached, 61.5 us with the stores past the cache,
// 56.0 us with both; 16 heaps of 4096 channels, 134 MB moved: 25.6, 20.0 and
// 23.8 us).
#include "fbf_internal.hpp"

#include <algorithm>

#include <climits>

namespace fbf {
namespace {

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
    uint32_t inv_ou;               // ceil(2^32 / (TR * EU)): the units of a full tile's output row
    bool load_past, store_past;    // the block is read, and written, past the cache
};

// A store past the cache where `past` says so (units of 16 and 4 bytes; a
// wave's 64 single bytes leave half a line for a later store).
template <typename U>
__device__ __forceinline__ void store_unit(U v, U* p, bool past)
{
    if constexpr (sizeof(U) == 16) {
        typedef uint32_t v4u __attribute__((ext_vector_type(4)));
        if (past)
            __builtin_nontemporal_store(v4u{v.x, v.y, v.z, v.w}, reinterpret_cast<v4u*>(p));
        else
            *p = v;
    } else if constexpr (sizeof(U) == 4) {
        if (past)
            __builtin_nontemporal_store(v, p);
        else
            *p = v;
    } else {
        *p = v;
    }
}

// 16-byte loads of a block too large for the cache go past it (`past`).
__device__ __forceinline__ uint4 load_unit(const uint4* p, bool past)
{
    if (past) {
        const int4 v = load_stream(p);
        return uint4{(uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w};
    }
    return *p;
}
template <typename U>
__device__ __forceinline__ U load_unit(const U* p, bool)
{
    return *p;
}

// Tile row pitch in units: TC * EU + 1, so that the transposed reads of the
// write phase (threads stepping down the tile rows) fall in distinct banks.
// POW2: square tiles with TC * EU and EU powers of two take shifts where the
// tile is full; else a wave takes rows, its lanes the units of a row, and the
// write phase splits a unit index into (row, unit of the element) with one
// multiplication.
template <typename U, bool POW2>
__global__ __launch_bounds__(256) void corner_turn_k(CtArgs a)
{
    extern __shared__ __align__(16) uint8_t ct_lds[];
    U* tile = reinterpret_cast<U*>(ct_lds);
    const int EU = a.EU;
    const int pitch = a.TC * EU + 1;
    long long bid = blockIdx.x;
    const int tc = (int)(bid % a.tiles_c);
    bid /= a.tiles_c;
    const int tr = (int)(bid % a.tiles_r);
    bid /= a.tiles_r;
    const long long i2 = bid % a.n2;
    const long long i1 = bid / a.n2;
    const U* in = reinterpret_cast<const U*>(a.in + i1 * a.in_s1 + i2 * a.in_s2);
    U* out = reinterpret_cast<U*>(a.out + i1 * a.out_s1 + i2 * a.out_s2);
    const int r0 = tr * a.TR, c0 = tc * a.TC;
    const int nr = min(a.TR, a.R - r0), nc = min(a.TC, a.C - c0);
    const size_t in_row = (size_t)a.C * EU, out_row = (size_t)a.R * EU;
    const U* src = in + (size_t)r0 * in_row + (size_t)c0 * EU;
    U* dst = out + (size_t)c0 * out_row + (size_t)r0 * EU;

    if (POW2 && nr == a.TR && nc == a.TC) {
        // Full tile, TC * EU and EU powers of two: shifts instead of divisions.
        const int n = a.TR << a.sh_ru;
        const int mu = (1 << a.sh_ru) - 1, me = EU - 1;
        for (int i = threadIdx.x; i < n; i += 256) {
            const int r = i >> a.sh_ru, k = i & mu;
            tile[r * pitch + k] = load_unit(src + (size_t)r * in_row + k, a.load_past);
        }
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += 256) {
            const int c = i >> a.sh_ru, k = i & mu;
            const int r = k >> a.sh_eu, e = k & me;
            store_unit(tile[r * pitch + c * EU + e], dst + (size_t)c * out_row + k, a.store_past);
        }
        return;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int ru = nc * EU;
    if (ru < 64 && nr * ru <= 256) {
        // A matrix of few units: all of it at once (8 channels, 22 samples, 3
        // bands, 412 beams, 6 groups: 6.4 us through the loop below, 5.1 so).
        const int r = (int)threadIdx.x / ru, k = (int)threadIdx.x - r * ru;
        if (r < nr) tile[r * pitch + k] = load_unit(src + (size_t)r * in_row + k, a.load_past);
    } else if (nr < 4) {
        // A wave per row would leave some without one: 64 channels, 512
        // samples, 1 band, 256 beams, 4 groups (34 MB) 17.8 us so, 12.4 here.
        for (int r = 0; r < nr; ++r)
            for (int k = threadIdx.x; k < ru; k += 256)
                tile[r * pitch + k] = load_unit(src + (size_t)r * in_row + k, a.load_past);
    } else {
        for (int r = wave; r < nr; r += 16) {   // up to four rows' loads in flight
            for (int k = lane; k < ru; k += 64) {
                U v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (r + 4 * j < nr) v[j] = load_unit(src + (size_t)(r + 4 * j) * in_row + k, a.load_past);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (r + 4 * j < nr) tile[(r + 4 * j) * pitch + k] = v[j];
            }
        }
    }
    __syncthreads();
    const int ou = nr * EU;
    if (ou <= 16 && nr == a.TR) {
        // Few rows: a wave of the loop below would be nearly empty.  1 channel,
        // 300 samples, 2 bands, 100 beams, 4 groups: 10.2 us through it, 4.5
        // here; but 26 units (13, 64,
        // 2, 500, 4) 9.6 and 10.1.
        for (int i = threadIdx.x; i < nc * ou; i += 256) {
            const int c = ou == 1 ? i : (int)__umulhi((uint32_t)i, a.inv_ou), k = i - c * ou;
            const int r = EU == 1 ? k : (int)__umulhi((uint32_t)k, a.inv_eu);
            store_unit(tile[r * pitch + c * EU + k - r * EU], dst + (size_t)c * out_row + k, a.store_past);
        }
        return;
    }
    for (int k = lane; k < ou; k += 64) {
        const int r = EU == 1 ? k : (int)__umulhi((uint32_t)k, a.inv_eu);
        const U* t = tile + r * pitch + (k - r * EU);
        for (int c = wave; c < nc; c += 4) store_unit(t[c * EU], dst + (size_t)c * out_row + k, a.store_past);
    }
}

// 4-byte elements, full 64 x 64 tiles: 16-byte global loads (4 words of an
// input row) and stores (4 words of an output row); the tile stays in
// 4-byte LDS words with a 65-word pitch, which keeps both the row writes
// and the column reads free of bank conflicts.  Edge tiles take the general
// path of corner_turn_k.
__global__ __launch_bounds__(256) void corner_turn_w4_k(CtArgs a)
{
    extern __shared__ __align__(16) uint8_t ct_lds[];
    uint32_t* tile = reinterpret_cast<uint32_t*>(ct_lds);
    constexpr int T = 64, P = 65;
    long long bid = blockIdx.x;
    const int tc = (int)(bid % a.tiles_c);
    bid /= a.tiles_c;
    const int tr = (int)(bid % a.tiles_r);
    bid /= a.tiles_r;
    const long long i2 = bid % a.n2;
    const long long i1 = bid / a.n2;
    const uint32_t* in = reinterpret_cast<const uint32_t*>(a.in + i1 * a.in_s1 + i2 * a.in_s2);
    uint32_t* out = reinterpret_cast<uint32_t*>(a.out + i1 * a.out_s1 + i2 * a.out_s2);
    const int r0 = tr * T, c0 = tc * T;
    const int nr = min(T, a.R - r0), nc = min(T, a.C - c0);
    const uint32_t* src = in + (size_t)r0 * a.C + c0;
    uint32_t* dst = out + (size_t)c0 * a.R + r0;
    if (nr == T && nc == T) {
        // One uniform branch around all four loads: a branch for each kept them
        // from being in flight together (64 channels, 146 heaps 4.9 us, 4.5
        // so).
        uint4 v[4];
        auto load = [&](bool past) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = threadIdx.x + 256 * j;
                v[j] = load_unit(reinterpret_cast<const uint4*>(src + (size_t)(i >> 4) * a.C + ((i & 15) << 2)), past);
            }
        };
        if (a.load_past)
            load(true);
        else
            load(false);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = threadIdx.x + 256 * j;
            uint32_t* l = tile + (i >> 4) * P + ((i & 15) << 2);
            l[0] = v[j].x;
            l[1] = v[j].y;
            l[2] = v[j].z;
            l[3] = v[j].w;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = threadIdx.x + 256 * j;
            const int c = i >> 4, r = (i & 15) << 2;
            uint4 v;
            v.x = tile[r * P + c];
            v.y = tile[(r + 1) * P + c];
            v.z = tile[(r + 2) * P + c];
            v.w = tile[(r + 3) * P + c];
            store_unit(v, reinterpret_cast<uint4*>(dst + (size_t)c * a.R + r), a.store_past);
        }
    } else {
        for (int i = threadIdx.x; i < nr * nc; i += 256) {
            const int r = i / nc, c = i - r * nc;
            tile[r * P + c] = src[(size_t)r * a.C + c];
        }
        __syncthreads();
        for (int i = threadIdx.x; i < nr * nc; i += 256) {
            const int c = i / nr, r = i - c * nr;
            dst[(size_t)c * a.R + r] = tile[r * P + c];
        }
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
// bands, 72 beams and groups, 13 MB moved: 75 us, 13.2 us now).
constexpr size_t kCtLdsMax = 32 * 1024;
constexpr size_t kCtRow = 1024;

inline size_t ct_tile_bytes(int TR, int TC, int EU, size_t U)
{
    return (size_t)TR * ((size_t)TC * EU + 1) * U;
}

template <typename U>
int ct_launch_u(CtArgs a, long long n1, int E, hipStream_t s)
{
    a.EU = E / (int)sizeof(U);
    int T = 64;
    while (T > 1 && ((size_t)T * E > kCtRow || ct_tile_bytes(T, T, a.EU, sizeof(U)) > kCtLdsMax)) T >>= 1;
    auto tiles = [&](int tr, int tc) { return n1 * a.n2 * ((a.R + tr - 1) / tr) * ((a.C + tc - 1) / tc); };
    // A small block takes smaller tiles, down to 256-byte rows, to fill the chip.
    while (T > 1 && (size_t)T * E >= 512 && tiles(T, T) < 512) T >>= 1;
    a.TR = a.TC = T;
    if (a.R < T) {
        a.TR = a.R;
        for (int tc = std::min(T * T / a.R, (a.C + T - 1) / T * T); tc > T && a.TC == T; tc -= T)
            if (ct_tile_bytes(a.TR, tc, a.EU, sizeof(U)) <= kCtLdsMax && tiles(a.TR, tc) >= 512) a.TC = tc;
    }
    const size_t shm = ct_tile_bytes(a.TR, a.TC, a.EU, sizeof(U));
    FBF_REQUIRE(ct_tile_bytes(1, 1, a.EU, sizeof(U)) <= kCtLdsMax, FBF_ERR_UNSUPPORTED,
                "corner turn: element too large (at most 32 KiB - 16 B)");
    a.tiles_r = (a.R + a.TR - 1) / a.TR;
    a.tiles_c = (a.C + a.TC - 1) / a.TC;
    const long long nblocks = n1 * a.n2 * a.tiles_r * a.tiles_c;
    if (nblocks == 0) return FBF_OK;
    FBF_REQUIRE(nblocks < INT_MAX, FBF_ERR_UNSUPPORTED, "corner turn: too many tiles for one launch");
    a.sh_ru = ilog2_exact((long long)T * a.EU);
    a.sh_eu = ilog2_exact(a.EU);
    a.inv_eu = (uint32_t)(((1ull << 32) + a.EU - 1) / a.EU);   // (0 for EU = 1, unused)
    const unsigned long long row = (unsigned long long)a.TR * a.EU;   // exact below 2^16 units
    a.inv_ou = (uint32_t)(((1ull << 32) + row - 1) / row);
    const bool pow2 = a.TR == T && a.sh_ru >= 0 && a.sh_eu >= 0;
    if (pow2)
        corner_turn_k<U, true><<<dim3((unsigned)nblocks), 256, shm, s>>>(a);
    else
        corner_turn_k<U, false><<<dim3((unsigned)nblocks), 256, shm, s>>>(a);
    FBF_HIP_TRY(hipGetLastError());
    return FBF_OK;
}

// 16-byte units when every element and base is 16-byte aligned, else 4, else 1.
int ct_launch(CtArgs a, long long n1, int E, hipStream_t s)
{
    const long long bytes = n1 * a.n2 * a.R * a.C * E;
    a.load_past = bytes >= (128ll << 20);
    a.store_past = bytes >= (16ll << 20);
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
        corner_turn_w4_k<<<dim3((unsigned)nblocks), 256, 64 * 65 * 4, s>>>(a);
        FBF_HIP_TRY(hipGetLastError());
        return FBF_OK;
    }
    if (E % 16 == 0 && (al & 15) == 0) return ct_launch_u<uint4>(a, n1, E, s);
    if (E % 4 == 0 && (al & 3) == 0) return ct_launch_u<uint32_t>(a, n1, E, s);
    return ct_launch_u<uint8_t>(a, n1, E, s);
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
