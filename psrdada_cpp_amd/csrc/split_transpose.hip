// Split transpose TAFTP -> FTPA for a contiguous antenna subset.
//
// Behaviour follows SplitTranspose.cu:11-126 (reference kernel and host
// wrapper): out[f][hg*S + s][p][a] = in[hg][start + a][f][s][p].
//
// MI355X design: for one (heap group, channel) the input is A_used rows of
// 2*S complex samples (1 KiB each for S = 256) at a stride of F KiB, and the
// output is one contiguous [2*S][A_used] block.  A 256-thread block moves a
// tile of 64 antennas x 128 (sample, pol) or 128 x 64: 16-byte coalesced row
// loads into LDS, then each thread gathers 8 consecutive elements of the
// output block and writes them as one 16-byte vector, across columns where
// the antennas are no multiple of 4 (the tile holds them all; multiples of 4
// take 8-byte vectors), so the output side is coalesced for any antennas.
// HBM-bound.  These stores are nontemporal: the block written is as large as the
// one read, and leaves the cache to it.  44 of 64 antennas, 64 channels, 12
// heaps (69 MB moved): 13.8 us with cached stores from 64-column tiles, 12.6 us
// now; 13 of 17 antennas, 83 channels, 39 heaps: 36.9 us with 2-byte stores,
// 14.7 us now.  Full tiles and large blocks keep to cached stores from 64 x 64
// tiles (NEAR, st_near).
//
// A launch can also generate the block's beamforming weights: its first
// work-groups run the weights generator (weights_run) and leave, and the
// rest do the transpose.  The generator's arithmetic then runs beside the
// transpose's memory traffic, in the same launch, with no dependency
// between the two.
#include "fbf_internal.hpp"

namespace fbf {
namespace {

constexpr int kIbSamples = 32;   // samples whose windows a tile is sure to hold whole
constexpr int kPad = 2;          // int16 padding per LDS row (an odd number of dwords)

template <int U>
struct VecOf;
template <> struct VecOf<8> { using T = int4; };
template <> struct VecOf<4> { using T = int2; };
template <> struct VecOf<2> { using T = int; };
template <> struct VecOf<1> { using T = int16_t; };

__device__ __forceinline__ void store_stream(int4 v, int16_t* dst)
{
    typedef int v4 __attribute__((ext_vector_type(4)));
    __builtin_nontemporal_store(v4{v.x, v.y, v.z, v.w}, reinterpret_cast<v4*>(dst));
}
__device__ __forceinline__ void store_stream(int2 v, int16_t* dst)
{
    typedef int v2 __attribute__((ext_vector_type(2)));
    __builtin_nontemporal_store(v2{v.x, v.y}, reinterpret_cast<v2*>(dst));
}
__device__ __forceinline__ void store_stream(int v, int16_t* dst)
{
    __builtin_nontemporal_store(v, reinterpret_cast<int*>(dst));
}
__device__ __forceinline__ void store_stream(int16_t v, int16_t* dst) { __builtin_nontemporal_store(v, dst); }

template <bool NEAR, typename V>
__device__ __forceinline__ void store_out(V v, int16_t* dst)
{
    if constexpr (NEAR)
        *reinterpret_cast<V*>(dst) = v;
    else
        store_stream(v, dst);
}

// Incoherent beam computed from the same tiles (all antennas of the block):
// output [sample_out][channel] int8, tscrunch dividing the tile's 32 samples,
// fscrunch 1 (IncoherentBeamformer.cu:10-69).
struct IbTile {
    int8_t* out;            // null: no incoherent beam
    const float* offsets;
    const float* scales;
    int tscrunch, quant;
};

// SP: columns of the tile (its antennas are 8192 / SP).  U > 0: vectors of U
// antennas of one column (U divides used_nantennas); U = 0: 16-byte vectors
// of the whole output block, all antennas in one tile; `inv` is then
// ceil(2^32 / used_nantennas).  NEAR: tiles of 64 antennas, neighbours on one
// XCD, cached stores.
template <int U, int SP, bool IB, bool NEAR>
__global__ __launch_bounds__(256) void split_transpose_k(
    const int16_t* __restrict__ in, int16_t* __restrict__ out,
    int nheap_groups, int total_nantennas, int used_nantennas, int start_antenna,
    int nchans, int sp_per_heap, int n_sp_tiles, uint32_t inv, IbTile ib, WeightsJob wj)
{
    constexpr int kTileA = NEAR ? 64 : 8192 / SP;
    constexpr int TPR = SP / 8;         // threads per row
    constexpr int RPP = 256 / TPR;      // rows per pass
    __shared__ int16_t tile[kTileA][SP + kPad];
    __shared__ int ibsum[4][SP / 2];
    const int tid = threadIdx.x;
    if (weights_job_run(wj, tid)) return;   // uniform over the work-group
    const int logical = NEAR ? xcd_remap((int)blockIdx.x - wj.nblocks, (int)gridDim.x - wj.nblocks)
                             : (int)blockIdx.x - wj.nblocks;
    const int spt = logical % n_sp_tiles;
    const int rest = logical / n_sp_tiles;
    const int hg = rest % nheap_groups;
    const int f = rest / nheap_groups;
    if (f >= nchans) return;

    const size_t out_block = ((size_t)f * nheap_groups + hg) * sp_per_heap + (size_t)spt * SP;
    // Incoherent beam: a 16-byte row load holds 4 samples x 2 pols of one
    // antenna, and one sdot4 of a 4-byte word with itself is the power of
    // both pols of a sample.  This thread sums its 4 samples over the rows it
    // loads.  A word squares to at most 4 * 128^2 = 2^16, so even the sum of
    // a sample over all A antennas (below) is exact in int32 for A < 2^15,
    // which the incoherent-beam plan requires.
    int ibacc[4] = {0, 0, 0, 0};

    for (int ab = 0; ab < used_nantennas; ab += kTileA) {
        const int na = min(kTileA, used_nantennas - ab);
        const int col = (tid % TPR) * 8;
        auto load = [&](int r) {
            const size_t row = ((size_t)hg * total_nantennas + start_antenna + ab + r) * nchans + f;
            return *reinterpret_cast<const int4*>(in + row * sp_per_heap + (size_t)spt * SP + col);
        };
        auto stage = [&](int r, const int4& v) {
            if (IB) {
                ibacc[0] = __builtin_amdgcn_sdot4(v.x, v.x, ibacc[0], false);
                ibacc[1] = __builtin_amdgcn_sdot4(v.y, v.y, ibacc[1], false);
                ibacc[2] = __builtin_amdgcn_sdot4(v.z, v.z, ibacc[2], false);
                ibacc[3] = __builtin_amdgcn_sdot4(v.w, v.w, ibacc[3], false);
            }
            uint32_t* dst = reinterpret_cast<uint32_t*>(&tile[r][col]);
            dst[0] = (uint32_t)v.x;
            dst[1] = (uint32_t)v.y;
            dst[2] = (uint32_t)v.z;
            dst[3] = (uint32_t)v.w;
        };
        if constexpr (NEAR) {
#pragma unroll
            for (int pass = 0; pass < kTileA / RPP; ++pass) {
                const int r = pass * RPP + tid / TPR;
                if (r < na) stage(r, load(r));
            }
        } else {
            int4 v[kTileA / RPP];
#pragma unroll
            for (int pass = 0; pass < kTileA / RPP; ++pass) {
                const int r = pass * RPP + tid / TPR;
                if (r < na) v[pass] = load(r);
            }
#pragma unroll
            for (int pass = 0; pass < kTileA / RPP; ++pass) {
                const int r = pass * RPP + tid / TPR;
                if (r < na) stage(r, v[pass]);
            }
        }
        __syncthreads();
        if constexpr (U > 0) {
            const int units = na / U;
            for (int idx = tid; idx < SP * units; idx += 256) {
                const int sp = idx / units;
                const int u = idx - sp * units;
                union {
                    typename VecOf<U>::T v;
                    int16_t e[U];
                } pack;
#pragma unroll
                for (int i = 0; i < U; ++i) pack.e[i] = tile[u * U + i][sp];
                store_out<NEAR>(pack.v, out + (out_block + sp) * used_nantennas + ab + u * U);
            }
        } else {
            // SP is a multiple of 8, so the block is whole 16-byte vectors
            // and starts at one.
            for (int idx = tid; idx < SP / 8 * used_nantennas; idx += 256) {
                int sp = (int)__umulhi((uint32_t)idx * 8u, inv);
                int a = idx * 8 - sp * used_nantennas;
                union {
                    int4 v;
                    int16_t e[8];
                } pack;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    pack.e[i] = tile[a][sp];
                    if (++a == used_nantennas) {
                        a = 0;
                        ++sp;
                    }
                }
                store_out<NEAR>(pack.v, out + out_block * used_nantennas + (size_t)idx * 8);
            }
        }
        __syncthreads();
    }
    if (IB) {
        // Lanes with the same tid % TPR hold the same 4 samples for different
        // rows: sum over them in the wave, then over the 4 waves.
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int m = TPR; m < 64; m <<= 1) ibacc[q] += __shfl_xor(ibacc[q], m);
        const int lane = tid & 63;
        if (lane < TPR) {
#pragma unroll
            for (int q = 0; q < 4; ++q) ibsum[tid >> 6][lane * 4 + q] = ibacc[q];
        }
        __syncthreads();
        // SP / 2 samples per tile -> SP / 2 / tscrunch outputs.
        const int nout = (SP / 2) / ib.tscrunch;
        if (tid < nout) {
            long long P = 0;
            for (int c = tid * ib.tscrunch; c < (tid + 1) * ib.tscrunch; ++c)
                P += (long long)ibsum[0][c] + ibsum[1][c] + ibsum[2][c] + ibsum[3][c];
            const long long t0 = ((long long)hg * sp_per_heap + (long long)spt * SP) / 2;
            const long long to = t0 / ib.tscrunch + tid;
            ib.out[to * nchans + f] = quantise((double)P, ib.offsets[f], ib.scales[f], ib.quant);
        }
    }
}

}  // namespace
}  // namespace fbf

using namespace fbf;

namespace {

template <int SP, bool IB, bool NEAR = false>
int st_launch_t(const void* taftp, void* ftpa, int total_nantennas, int used_nantennas, int start_antenna,
                int nchans, int nsamples_per_heap, int nhg, IbTile ib, WeightsJob wj, fbf_stream_t stream)
{
    const int sp_per_heap = 2 * nsamples_per_heap;
    const int n_sp_tiles = sp_per_heap / SP;
    const size_t nblocks = (size_t)nchans * nhg * n_sp_tiles + (size_t)wj.nblocks;
    FBF_REQUIRE(nblocks < (1ull << 31), FBF_ERR_UNSUPPORTED, "fbf_split_transpose: grid too large");
    // Vectors of 8 antennas where they divide; else, while one tile holds
    // every antenna, 16-byte vectors across columns; else what divides.
    const uint32_t inv = (uint32_t)(((1ull << 32) + used_nantennas - 1) / used_nantennas);
    const auto kernel = [&] {
        if constexpr (NEAR)
            return used_nantennas % 8 == 0   ? split_transpose_k<8, SP, IB, true>
                   : used_nantennas % 4 == 0 ? split_transpose_k<4, SP, IB, true>
                                             : split_transpose_k<0, SP, IB, true>;
        else
            return used_nantennas % 8 == 0       ? split_transpose_k<8, SP, IB, false>
                   : used_nantennas % 4 == 0     ? split_transpose_k<4, SP, IB, false>
                   : used_nantennas == 1         ? split_transpose_k<1, SP, IB, false>
                   : used_nantennas <= 8192 / SP ? split_transpose_k<0, SP, IB, false>
                   : used_nantennas % 2 == 0     ? split_transpose_k<2, SP, IB, false>
                                                 : split_transpose_k<1, SP, IB, false>;
    }();
    kernel<<<dim3((unsigned)nblocks), 256, 0, static_cast<hipStream_t>(stream)>>>(
        static_cast<const int16_t*>(taftp), static_cast<int16_t*>(ftpa), nhg, total_nantennas, used_nantennas,
        start_antenna, nchans, sp_per_heap, n_sp_tiles, inv, ib, wj);
    FBF_LAUNCH_CHECK("split_transpose_k");
    return FBF_OK;
}

// Whether a block takes 64 x 64 tiles with cached stores: antennas that fill such
// tiles, and copies that outgrow the cache.  us, these tiles against 64 x 128 with
// nontemporal stores (antennas / channels / heaps of 256 samples; with the
// incoherent beam in brackets): 64/64/32 46 against 61 (46, 66), 64/64/12 16.2
// against 17.0, 56/64/32 41 against 45 (42, 46), 128/64/32 116 against 128 (116,
// 125), 60/64/32 46 against 49, 40/64/48 (252 MB moved) 43 against 48; but
// 40/64/32 (168 MB) 31 against 25 (37, 28), and with the incoherent beam 40/64/48
// 53 against 49.  Antennas not in fours, whose vectors run across columns, where one tile
// holds them and the copy outgrows the cache without being far beyond it:
// 62/64/32 45.7 against 53.0 (46.5, 53.6), 62/64/40 59.0 against 64.4 (60.0, 65.5),
// 58/64/28 37.0 against 40.3, 50/64/32 38.2 against 41.0 (42.9, 42.4); but 62/64/20
// 30.4 against 27.2 (32.0, 29.1), 62/64/52 84.7 against 82.4, 58/64/46 with the
// incoherent beam 68.5 against 65.7, 46/64/32 35.2 against 35.4 (41.5, 37.1).
//
// A copy that the next launch reads (`read_next`: the library's own calls) takes
// them too from 24 antennas, and smaller copies sooner: the coherent kernel
// finds its channels in the L2 of its XCD.  Both launches, us, cached 64 x 64
// tiles against the others (antennas / channels / heaps, 64 beams): 32/64/8 17.1
// against 24.6, 24/64/16 25.8 and 30.0, 16/64/8 15.0 and 16.2, 48/16/8 10.4 and
// 12.2; but 8/64/32 33.0 and 28.0, 12/64/8 with the incoherent beam 18.4 and 17.2.
// With the incoherent beam small copies are launches and latency either way:
// 52/16/1 5.0 against 5.9, but 16/64/8 10.3 and 7.4.
bool st_near(bool ib, int used_nantennas, size_t moved, bool read_next)
{
    // (Columns of whole 64-byte lines, 32 antennas, gain from the cache sooner:
    // 32/64/32, 128 MiB, 21.5 against 22.9; 32/64/16 11.6 against 11.4.)
    const size_t near_bytes = (size_t)(used_nantennas % 32 == 0 ? 128 : 192) << 20;
    if (used_nantennas % 4 != 0)
        return used_nantennas >= (ib ? 54 : 48) && used_nantennas < 64 && moved >= near_bytes &&
               moved < (size_t)320 << 20;
    if (used_nantennas > 64) return true;
    if (used_nantennas >= 56 && used_nantennas % 8 == 0) return true;
    const size_t copy_mib = (moved / 2) >> 20;
    if (read_next && (used_nantennas >= 24 || copy_mib < 2 || (used_nantennas >= 16 && copy_mib < 16))) return true;
    if (ib && used_nantennas >= 20 && copy_mib < 4) return true;
    return moved >= near_bytes && (!ib || used_nantennas >= 56);
}

template <bool IB>
int st_launch_sp(const void* taftp, void* ftpa, int total_nantennas, int used_nantennas, int start_antenna,
                 int nchans, int nsamples_per_heap, int nhg, IbTile ib, WeightsJob wj, fbf_stream_t stream,
                 bool read_next)
{
    if (st_near(IB, used_nantennas, (size_t)8 * used_nantennas * nchans * nsamples_per_heap * nhg, read_next))
        return st_launch_t<64, IB, true>(taftp, ftpa, total_nantennas, used_nantennas, start_antenna, nchans,
                                         nsamples_per_heap, nhg, ib, wj, stream);
    // Tiles of 128 columns where 64 antennas hold a subset and they divide a
    // heap, else of 64 columns and 128 antennas.
    if (used_nantennas <= 64 && nsamples_per_heap % 64 == 0)
        return st_launch_t<128, IB>(taftp, ftpa, total_nantennas, used_nantennas, start_antenna, nchans,
                                    nsamples_per_heap, nhg, ib, wj, stream);
    return st_launch_t<64, IB>(taftp, ftpa, total_nantennas, used_nantennas, start_antenna, nchans,
                               nsamples_per_heap, nhg, ib, wj, stream);
}

int st_launch(const void* taftp, void* ftpa, int total_nantennas, int used_nantennas, int start_antenna, int nchans,
              int nsamples_per_heap, int nhg, IbTile ib, fbf_stream_t stream, bool read_next,
              WeightsJob wj = WeightsJob{})
{
    if (ib.out)
        return st_launch_sp<true>(taftp, ftpa, total_nantennas, used_nantennas, start_antenna, nchans,
                                 nsamples_per_heap, nhg, ib, wj, stream, read_next);
    return st_launch_sp<false>(taftp, ftpa, total_nantennas, used_nantennas, start_antenna, nchans,
                              nsamples_per_heap, nhg, ib, wj, stream, read_next);
}

int st_run(const void* taftp, size_t taftp_bytes, void* ftpa, size_t ftpa_bytes, int total_nantennas,
           int used_nantennas, int start_antenna, int nchans, int nsamples_per_heap, fbf_stream_t stream,
           bool read_next)
{
    FBF_REQUIRE(taftp && ftpa, FBF_ERR_ARG, "fbf_split_transpose: null buffer");
    FBF_REQUIRE(total_nantennas > 0 && used_nantennas > 0 && start_antenna >= 0 &&
                    start_antenna + used_nantennas <= total_nantennas,
                FBF_ERR_ARG, "fbf_split_transpose: antenna subset outside the input");
    FBF_REQUIRE(nchans > 0 && nsamples_per_heap > 0, FBF_ERR_ARG,
                "fbf_split_transpose: nchans and nsamples_per_heap must be positive");
    FBF_REQUIRE(nsamples_per_heap % 32 == 0, FBF_ERR_UNSUPPORTED,
                "fbf_split_transpose: nsamples_per_heap must be a multiple of 32");
    const size_t hg_bytes = (size_t)4 * total_nantennas * nchans * nsamples_per_heap;
    FBF_REQUIRE(taftp_bytes % hg_bytes == 0, FBF_ERR_SIZE,
                "fbf_split_transpose: input is not a whole number of heap groups");
    const size_t nhg = taftp_bytes / hg_bytes;
    const size_t expect_out = (size_t)4 * used_nantennas * nchans * nsamples_per_heap * nhg;
    FBF_REQUIRE(ftpa_bytes == expect_out, FBF_ERR_SIZE,
                "fbf_split_transpose: output size " + std::to_string(ftpa_bytes) +
                    " != expected " + std::to_string(expect_out));
    FBF_REQUIRE((reinterpret_cast<uintptr_t>(taftp) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(ftpa) & 15) == 0,
                FBF_ERR_ARG, "fbf_split_transpose: buffers must be 16-byte aligned");
    if (nhg == 0) return FBF_OK;
    FBF_REQUIRE(nhg < (1u << 20), FBF_ERR_UNSUPPORTED, "fbf_split_transpose: too many heap groups");

    return st_launch(taftp, ftpa, total_nantennas, used_nantennas, start_antenna, nchans, nsamples_per_heap,
                     (int)nhg, IbTile{nullptr, nullptr, nullptr, 1, 0}, stream, read_next);
}

// Checks a fused split-transpose + incoherent-beam call and returns the
// launch arguments.
int st_ib_params(const void* taftp, size_t taftp_bytes, const void* ftpa, size_t ftpa_bytes, int nchans,
                        int nsamples_per_heap, const fbf_ib_plan* ib_plan, void* tf, size_t tf_bytes, int* nhg_out,
                        int* nantennas, IbTile* tile)
{
    FBF_REQUIRE(taftp && ftpa && ib_plan && tf, FBF_ERR_ARG, "fbf_split_transpose_ib: null argument");
    IbFuseParams ibp;
    int st = ib_fuse_params(ib_plan, &ibp);
    if (st) return st;
    FBF_REQUIRE(ibp.nchans == nchans && ibp.nsamples_per_heap == nsamples_per_heap, FBF_ERR_ARG,
                "fbf_split_transpose_ib: incoherent-beam plan geometry differs from the block's");
    FBF_REQUIRE(ibp.fscrunch == 1 && ibp.tscrunch > 0 && kIbSamples % ibp.tscrunch == 0, FBF_ERR_UNSUPPORTED,
                "fbf_split_transpose_ib: needs fscrunch 1 and a tscrunch dividing 32");
    const int A = ibp.nantennas;
    FBF_REQUIRE(nsamples_per_heap > 0 && nsamples_per_heap % 32 == 0, FBF_ERR_UNSUPPORTED,
                "fbf_split_transpose_ib: nsamples_per_heap must be a multiple of 32");
    const size_t hg_bytes = (size_t)4 * A * nchans * nsamples_per_heap;
    FBF_REQUIRE(taftp_bytes % hg_bytes == 0 && ftpa_bytes == taftp_bytes, FBF_ERR_SIZE,
                "fbf_split_transpose_ib: input and output must be the same whole number of heap groups");
    const size_t nhg = taftp_bytes / hg_bytes;
    const size_t expect_tf = nhg * nsamples_per_heap / ibp.tscrunch * nchans;
    FBF_REQUIRE(tf_bytes == expect_tf, FBF_ERR_SIZE,
                "fbf_split_transpose_ib: incoherent-beam output size " + std::to_string(tf_bytes) +
                    " != expected " + std::to_string(expect_tf));
    FBF_REQUIRE((reinterpret_cast<uintptr_t>(taftp) & 15) == 0 && (reinterpret_cast<uintptr_t>(ftpa) & 15) == 0,
                FBF_ERR_ARG, "fbf_split_transpose_ib: buffers must be 16-byte aligned");
    FBF_REQUIRE(nhg < (1u << 20), FBF_ERR_UNSUPPORTED, "fbf_split_transpose_ib: too many heap groups");
    *nhg_out = (int)nhg;
    *nantennas = A;
    *tile = IbTile{static_cast<int8_t*>(tf), ibp.offsets, ibp.scales, ibp.tscrunch, ibp.quant};
    return FBF_OK;
}

int st_ib_run(const void* taftp, size_t taftp_bytes, void* ftpa, size_t ftpa_bytes, int nchans,
              int nsamples_per_heap, fbf_ib_plan* ib_plan, void* tf, size_t tf_bytes, fbf_stream_t stream,
              bool read_next)
{
    int nhg = 0, A = 0;
    IbTile ib{};
    const int st = st_ib_params(taftp, taftp_bytes, ftpa, ftpa_bytes, nchans, nsamples_per_heap, ib_plan, tf,
                                tf_bytes, &nhg, &A, &ib);
    if (st) return st;
    if (nhg == 0) return FBF_OK;
    return st_launch(taftp, ftpa, A, A, 0, nchans, nsamples_per_heap, nhg, ib, stream, read_next);
}

}  // namespace

extern "C" int fbf_split_transpose(const void* taftp, size_t taftp_bytes, void* ftpa,
                                   size_t ftpa_bytes, int total_nantennas, int used_nantennas,
                                   int start_antenna, int nchans, int nsamples_per_heap,
                                   fbf_stream_t stream)
{
    return st_run(taftp, taftp_bytes, ftpa, ftpa_bytes, total_nantennas, used_nantennas, start_antenna, nchans,
                  nsamples_per_heap, stream, false);
}

int fbf::split_transpose_read_next(const void* taftp, size_t taftp_bytes, void* ftpa, size_t ftpa_bytes,
                                   int total_nantennas, int used_nantennas, int start_antenna, int nchans,
                                   int nsamples_per_heap, fbf_stream_t stream)
{
    return st_run(taftp, taftp_bytes, ftpa, ftpa_bytes, total_nantennas, used_nantennas, start_antenna, nchans,
                  nsamples_per_heap, stream, true);
}

extern "C" int fbf_split_transpose_ib(const void* taftp, size_t taftp_bytes, void* ftpa, size_t ftpa_bytes,
                                      int nchans, int nsamples_per_heap, fbf_ib_plan* ib_plan, void* tf,
                                      size_t tf_bytes, fbf_stream_t stream)
{
    return st_ib_run(taftp, taftp_bytes, ftpa, ftpa_bytes, nchans, nsamples_per_heap, ib_plan, tf, tf_bytes, stream,
                     false);
}

int fbf::split_transpose_ib_read_next(const void* taftp, size_t taftp_bytes, void* ftpa, size_t ftpa_bytes,
                                      int nchans, int nsamples_per_heap, fbf_ib_plan* ib_plan, void* tf,
                                      size_t tf_bytes, fbf_stream_t stream)
{
    return st_ib_run(taftp, taftp_bytes, ftpa, ftpa_bytes, nchans, nsamples_per_heap, ib_plan, tf, tf_bytes, stream,
                     true);
}

extern "C" int fbf_split_transpose_ib_weights(const void* taftp, size_t taftp_bytes, void* ftpa, size_t ftpa_bytes,
                                              int nchans, int nsamples_per_heap, fbf_ib_plan* ib_plan, void* tf,
                                              size_t tf_bytes, fbf_weights_plan* weights_plan, const void* delays,
                                              size_t delays_bytes, double epoch, void* weights,
                                              size_t weights_bytes, fbf_stream_t stream)
{
    int nhg = 0, A = 0;
    IbTile ib{};
    int st = st_ib_params(taftp, taftp_bytes, ftpa, ftpa_bytes, nchans, nsamples_per_heap, ib_plan, tf, tf_bytes,
                          &nhg, &A, &ib);
    if (st) return st;
    WeightsJob wj{};
    st = weights_launch_params(weights_plan, delays, delays_bytes, epoch, weights, weights_bytes, &wj.w);
    if (st) return st;
    FBF_REQUIRE(wj.w.F == nchans, FBF_ERR_ARG,
                "fbf_split_transpose_ib_weights: the weights plan's channels differ from the block's");
    FBF_REQUIRE((unsigned long long)wj.w.gx * wj.w.gy < (1ull << 30), FBF_ERR_UNSUPPORTED,
                "fbf_split_transpose_ib_weights: too many weights work-groups");
    wj.nblocks = (int)(wj.w.gx * wj.w.gy);
    if (nhg == 0) return fbf_weights_generate(weights_plan, delays, delays_bytes, epoch, weights, weights_bytes,
                                              nullptr, stream);
    return st_launch(taftp, ftpa, A, A, 0, nchans, nsamples_per_heap, nhg, ib, stream, false, wj);
}
