// Incoherent beam: detected power summed over all antennas.
//
// Behaviour follows IncoherentBeamformer.cu:10-117 (icbf_taftp_general_k and
// IncoherentBeamformer::beamform) and its host reference
// IncoherentBeamformerTester.cu:36-97:
//   P(to, fo) = sum over antennas, fscrunch channels, tscrunch samples and
//               pols of re^2 + im^2,  out = quantise(P, offset[fo], scale[fo])
// written TF: [heap_group * S / ts + window][fo].
//
// MI355X design: HBM-bound read of the whole TAFTP block.  A work-group owns
// one heap group and output channel; its waves share the rows (channel,
// antenna) out in contiguous runs, and each reads whole 1 KiB (channel, antenna) rows as
// 16-byte vectors (4 samples x 2 pols a lane) and squares with v_dot4_i32_i8
// (exact int32).  tscrunch is reduced in-lane and across lanes with shuffles,
// the waves' sums through LDS, in int64 (exact).  Blocks that the cache is not
// likely to hold are read past it, and work-groups that follow each other in a
// heap group stay on one XCD.  64 antennas, 64 channels, 32 heaps, fscrunch 2:
// 26.0 us with cached loads and a wave to each of four channels, 21.5 us now
// (6.2 TB/s).
//
// fbf_ib_beamform_weights also generates the block's beamforming weights in
// the same launch (its first work-groups), as the split-transpose launch can.
#include "fbf_internal.hpp"

namespace fbf {
namespace {

enum { IB_INT8 = 0, IB_POWER = 1 };

struct IbArgs {
    const int8_t* taftp;
    void* out;
    const float* offsets;
    const float* scales;
    int nhg, A, F, Fo, ts, fs, quant;
};

__device__ __forceinline__ int sq4(int x, int acc)
{
    return __builtin_amdgcn_sdot4(x, x, acc, false);
}

// NW waves per work-group: 4, 8 or 16 (ib_waves); PAST: the block
// is read past the cache (ib_run); ONE: a wave per output channel, NW of them
// to a work-group, instead of the waves sharing one's rows out.
template <int MODE, int NW, bool PAST, bool ONE>
__global__ __launch_bounds__(64 * NW) void ib_k(IbArgs p, WeightsJob wj)
{
    constexpr int S = 256;
    __shared__ long long part[NW][S];
    const int tid = threadIdx.x;
    if (NW == 4 && weights_job_run(wj, tid)) return;   // uniform over the work-group
    const int sc = tid & 63;   // 16-byte chunk: samples 4*sc .. 4*sc+3
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int logical = xcd_remap((int)blockIdx.x - wj.nblocks, (int)gridDim.x - wj.nblocks);
    const int groups = ONE ? (p.Fo + NW - 1) / NW : p.Fo;
    const int fo = ONE ? logical % groups * NW + wave : logical % groups;
    const int hg = logical / groups;
    if (hg >= p.nhg) return;

    // Rows (channel k, antenna a) of the output channel, antennas fastest; this
    // wave's are [r, r1).  One word squared is at most 4 * 128^2 = 2^16, so
    // int32 sums over kRun = 2^14 rows are exact; each run's are then added in
    // int64.
    constexpr int kRun = 1 << 14;
    long long s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    const size_t row_bytes = (size_t)S * 4;
    const size_t astride = (size_t)p.F * row_bytes;
    const int rows = ONE && fo >= p.Fo ? 0 : p.fs * p.A;   // (1 KiB each: below 2^31)
    const int per = ONE ? rows : (rows + NW - 1) / NW;
    int r = ONE ? 0 : min(wave * per, rows);
    const int r1 = min(r + per, rows);
    const int k0 = r / p.A;
    int a = r - k0 * p.A;
    const int8_t* row = p.taftp + ((size_t)hg * p.A * p.F + (size_t)fo * p.fs + k0) * row_bytes +
                        (size_t)a * astride + (size_t)sc * 16;
    auto next = [&]() {   // the current row, and on to the next
        const int8_t* q = row;
        row += astride;
        if (++a == p.A) {
            a = 0;
            row += row_bytes - (size_t)p.A * astride;
        }
        return q;
    };
    auto load = [](const int8_t* q) { return PAST ? load_stream(q) : *reinterpret_cast<const int4*>(q); };
    while (r < r1) {
        int c0 = 0, c1 = 0, c2 = 0, c3 = 0;
        const int n = min(r1 - r, kRun);
        auto add = [&](int4 x) {
            c0 = sq4(x.x, c0);
            c1 = sq4(x.y, c1);
            c2 = sq4(x.z, c2);
            c3 = sq4(x.w, c3);
        };
        int i = 0;
        for (; i + 4 <= n; i += 4) {
            int4 x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = load(next());
#pragma unroll
            for (int u = 0; u < 4; ++u) add(x[u]);
        }
        for (; i < n; ++i) add(load(next()));
        s0 += c0;
        s1 += c1;
        s2 += c2;
        s3 += c3;
        r += n;
    }

    // tscrunch: per-sample sums s0..s3 cover samples 4*sc + {0..3}.
    const int nwin = S / p.ts;
    if (p.ts >= 4) {
        long long v = s0 + s1 + s2 + s3;
        for (int m = 1; m < p.ts / 4; m <<= 1) v += __shfl_xor(v, m, 64);
        if ((sc % (p.ts / 4)) == 0) part[wave][sc / (p.ts / 4)] = v;
    } else if (p.ts == 2) {
        part[wave][2 * sc] = s0 + s1;
        part[wave][2 * sc + 1] = s2 + s3;
    } else {
        part[wave][4 * sc] = s0;
        part[wave][4 * sc + 1] = s1;
        part[wave][4 * sc + 2] = s2;
        part[wave][4 * sc + 3] = s3;
    }
    __syncthreads();

    // The waves' sums of a window.
    for (int w = ONE ? sc : tid; w < nwin && fo < p.Fo; w += ONE ? 64 : 64 * NW) {
        long long v = 0;
        if constexpr (ONE) {
            v = part[wave][w];
        } else {
#pragma unroll
            for (int r = 0; r < NW; ++r) v += part[r][w];
        }
        const size_t t = (size_t)hg * nwin + w;
        if (MODE == IB_POWER) {
            static_cast<double*>(p.out)[t * p.Fo + fo] = (double)v;
        } else {
            static_cast<int8_t*>(p.out)[t * p.Fo + fo] = quantise((double)v, p.offsets[fo], p.scales[fo], p.quant);
        }
    }
}

// Waves that share the rows of a work-group (`work` of them), on blocks in turn
// (us; antennas / channels / heaps / fscrunch):
//                      work  rows     4     8    16
//   120/16/4/1          64   120    6.5   4.8   4.2   16 where few work-groups
//   64/40/4/8           20   512   14.2   8.5   7.8   have many rows;
//   40/40/30/4         300   160    9.2   9.7   9.8   4 where few compute units
//   64/40/30/4         300   256   13.1  14.1  13.9   would have two work-groups
//   68/56/39/4         546   272   26.1  27.8  27.4   and the others one, longer
//                                                     so past the cache;
//   24/64/60/1        3840    24   16.0  17.5  26.1   4 where rows are few;
//   40/16/60/1         960    40    8.0   7.7   8.9   else 8
//   96/64/12/1         768    96   12.8  12.4  13.1
inline int ib_waves(long long work, long long rows, bool past)
{
    if (rows >= 112 && work <= 96) return 16;
    if (rows < 16 || (rows < 32 && work >= 1024)) return 4;
    return work > 256 && work < (past ? 1024 : 384) ? 4 : 8;
}

template <int MODE, int NW, bool ONE>
void launch_ib_nw(const IbArgs& a, const WeightsJob& wj, dim3 grid, bool past, hipStream_t s)
{
    past ? ib_k<MODE, NW, true, ONE><<<grid, 64 * NW, 0, s>>>(a, wj)
         : ib_k<MODE, NW, false, ONE><<<grid, 64 * NW, 0, s>>>(a, wj);
}

template <int MODE>
void launch_ib(const IbArgs& a, const WeightsJob& wj, dim3 grid, bool one, int waves, bool past, hipStream_t s)
{
    if (one)
        launch_ib_nw<MODE, 4, true>(a, wj, grid, past, s);
    else if (waves == 16)
        launch_ib_nw<MODE, 16, false>(a, wj, grid, past, s);
    else if (waves == 8)
        launch_ib_nw<MODE, 8, false>(a, wj, grid, past, s);
    else
        launch_ib_nw<MODE, 4, false>(a, wj, grid, past, s);
}

}  // namespace
}  // namespace fbf

using namespace fbf;

struct fbf_ib_plan {
    fbf_ib_desc d;
    float* d_levels;
};

extern "C" int fbf_ib_plan_create(const fbf_ib_desc* desc, const float* offsets, const float* scales,
                                  fbf_ib_plan** plan)
{
    FBF_REQUIRE(plan, FBF_ERR_ARG, "fbf_ib_plan_create: null plan pointer");
    *plan = nullptr;
    FBF_REQUIRE(desc && offsets && scales, FBF_ERR_ARG, "fbf_ib_plan_create: null argument");
    const fbf_ib_desc& d = *desc;
    FBF_REQUIRE(d.nantennas > 0 && d.nchans > 0 && d.tscrunch > 0 && d.fscrunch > 0, FBF_ERR_ARG,
                "fbf_ib: geometry values must be positive");
    // Per-channel partial power sums are int32: a word (one sample, both
    // pols) squares to at most 2^16, so A antennas stay below 2^31 for A < 2^15.
    FBF_REQUIRE(d.nantennas < 32768, FBF_ERR_UNSUPPORTED,
                "fbf_ib: nantennas must be below 32768 (int32 per-channel partial power sums)");
    FBF_REQUIRE(d.nsamples_per_heap == 256, FBF_ERR_UNSUPPORTED,
                "fbf_ib: nsamples_per_heap must be 256 (FBFUSE_NSAMPLES_PER_HEAP)");
    FBF_REQUIRE(256 % d.tscrunch == 0, FBF_ERR_UNSUPPORTED, "fbf_ib: tscrunch must divide 256");
    FBF_REQUIRE(d.nchans % d.fscrunch == 0, FBF_ERR_ARG, "fbf_ib: fscrunch must divide nchans");
    FBF_REQUIRE((d.fscrunch <= 4 && 4 % d.fscrunch == 0) || d.fscrunch % 4 == 0, FBF_ERR_UNSUPPORTED,
                "fbf_ib: fscrunch must be 1, 2 or a multiple of 4");
    const int cpb = d.fscrunch > 4 ? d.fscrunch : 4;
    FBF_REQUIRE(d.nchans % cpb == 0, FBF_ERR_UNSUPPORTED, "fbf_ib: nchans must be a multiple of 4 and of fscrunch");
    FBF_REQUIRE(d.quant_mode == FBF_QUANT_ROUND || d.quant_mode == FBF_QUANT_TRUNC, FBF_ERR_ARG,
                "fbf_ib: bad quant_mode");
    auto* p = new fbf_ib_plan{d, nullptr};
    const int Fo = d.nchans / d.fscrunch;
    hipError_t e = hipMalloc(&p->d_levels, sizeof(float) * 2 * Fo);
    if (e != hipSuccess) {
        delete p;
        return hip_status(e, "hipMalloc(levels)");
    }
    int st = fbf_ib_plan_set_levels(p, offsets, scales);
    if (st) {
        (void)hipFree(p->d_levels);
        delete p;
        return st;
    }
    *plan = p;
    return FBF_OK;
}

extern "C" int fbf_ib_plan_set_levels(fbf_ib_plan* plan, const float* offsets, const float* scales)
{
    FBF_REQUIRE(plan && offsets && scales, FBF_ERR_ARG, "fbf_ib_plan_set_levels: null argument");
    const int Fo = plan->d.nchans / plan->d.fscrunch;
    // Work still running on any stream may read the levels being replaced.
    FBF_HIP_TRY(hipDeviceSynchronize());
    FBF_HIP_TRY(hipMemcpy(plan->d_levels, offsets, sizeof(float) * Fo, hipMemcpyHostToDevice));
    FBF_HIP_TRY(hipMemcpy(plan->d_levels + Fo, scales, sizeof(float) * Fo, hipMemcpyHostToDevice));
    return FBF_OK;
}

extern "C" int fbf_ib_plan_destroy(fbf_ib_plan* plan)
{
    if (!plan) return FBF_OK;
    hipError_t e = hipFree(plan->d_levels);
    delete plan;
    if (e != hipSuccess) return hip_status(e, "hipFree(levels)");
    return FBF_OK;
}

static int ib_nhg(const fbf_ib_plan* plan, size_t taftp_bytes, long long* nhg)
{
    const size_t hg_bytes = (size_t)4 * plan->d.nantennas * plan->d.nchans * plan->d.nsamples_per_heap;
    FBF_REQUIRE(taftp_bytes % hg_bytes == 0, FBF_ERR_SIZE,
                "fbf_ib: input is not a multiple of AFTP blocks (IncoherentBeamformer.cu:95)");
    *nhg = (long long)(taftp_bytes / hg_bytes);
    return FBF_OK;
}

extern "C" int fbf_ib_output_bytes(const fbf_ib_plan* plan, size_t taftp_bytes, size_t* tf_bytes)
{
    FBF_REQUIRE(plan && tf_bytes, FBF_ERR_ARG, "fbf_ib_output_bytes: null argument");
    long long nhg = 0;
    int st = ib_nhg(plan, taftp_bytes, &nhg);
    if (st) return st;
    *tf_bytes = (size_t)nhg * (plan->d.nsamples_per_heap / plan->d.tscrunch) * (plan->d.nchans / plan->d.fscrunch);
    return FBF_OK;
}

static int ib_run(fbf_ib_plan* plan, int mode, const void* taftp, size_t taftp_bytes, void* out, size_t out_bytes,
                  fbf_stream_t stream, WeightsJob wj = WeightsJob{})
{
    FBF_REQUIRE(plan && taftp && out, FBF_ERR_ARG, "fbf_ib: null argument");
    long long nhg = 0;
    int st = ib_nhg(plan, taftp_bytes, &nhg);
    if (st) return st;
    const fbf_ib_desc& d = plan->d;
    const int Fo = d.nchans / d.fscrunch;
    const size_t nout = (size_t)nhg * (d.nsamples_per_heap / d.tscrunch) * Fo;
    const size_t expect = mode == IB_INT8 ? nout : nout * sizeof(double);
    FBF_REQUIRE(out_bytes == expect, FBF_ERR_SIZE,
                "fbf_ib: output size " + std::to_string(out_bytes) + " != expected " + std::to_string(expect));
    FBF_REQUIRE((reinterpret_cast<uintptr_t>(taftp) & 15) == 0, FBF_ERR_ARG, "fbf_ib: input must be 16-byte aligned");
    if (nhg == 0 && wj.nblocks == 0) return FBF_OK;
    IbArgs a;
    a.taftp = static_cast<const int8_t*>(taftp);
    a.out = out;
    a.offsets = plan->d_levels;
    a.scales = plan->d_levels + Fo;
    a.nhg = (int)nhg;
    a.A = d.nantennas;
    a.F = d.nchans;
    a.Fo = Fo;
    a.ts = d.tscrunch;
    a.fs = d.fscrunch;
    a.quant = d.quant_mode;
    // A wave per output channel where there are few rows and many outputs:
    // one row or two to a wave left mostly the sums over the waves (us, shared
    // out against a wave each; antennas / channels / heaps, tscrunch 16:
    // 4/128/48 10.3 against 6.1, 8/64/32 5.7 against 4.8, 12/64/32 6.4 against 5.8).
    const bool one = (long long)d.nantennas * d.fscrunch <= 12 && nhg * Fo >= 1024;
    const long long work = one ? nhg * ((Fo + 3) / 4) : nhg * Fo;
    const long long nblocks = work + wj.nblocks;
    FBF_REQUIRE(nblocks < (1ll << 31), FBF_ERR_UNSUPPORTED, "fbf_ib: grid too large");
    hipStream_t s = static_cast<hipStream_t>(stream);
    // Past the cache (256 MiB) from 96 MiB: with three blocks in turn smaller
    // ones are read from it (us, cached and past; 64 antennas, 40 channels, 30
    // heaps, fscrunch 4, 75 MiB 13.1 and 15.1; 96/40/30, 112 MiB 22.0 and 19.3).
    const bool past = taftp_bytes >= ((size_t)96 << 20);
    // (The weights job is made of work-groups of 4 waves.)
    const int waves = wj.nblocks ? 4 : ib_waves(work, (long long)d.nantennas * d.fscrunch, past);
    const dim3 grid((unsigned)nblocks);
    if (mode == IB_INT8)
        launch_ib<IB_INT8>(a, wj, grid, one, waves, past, s);
    else
        launch_ib<IB_POWER>(a, wj, grid, one, waves, past, s);
    FBF_LAUNCH_CHECK("ib_k");
    return FBF_OK;
}

int fbf::ib_finish_job(const fbf_ib_plan* plan, const int* partials, int nparts, long long T, void* tf,
                       size_t tf_bytes, IbFinishJob* out)
{
    FBF_REQUIRE(plan && partials && tf && out, FBF_ERR_ARG, "fbf_ib: null argument");
    const fbf_ib_desc& d = plan->d;
    FBF_REQUIRE(T % 16 == 0 && T % d.tscrunch == 0, FBF_ERR_SIZE, "fbf_ib: partials of a partial tile");
    FBF_REQUIRE(d.tscrunch < 16 ? 16 % d.tscrunch == 0 : d.tscrunch % 16 == 0, FBF_ERR_UNSUPPORTED,
                "fbf_ib: tscrunch must divide 16 or be a multiple of it");
    const int Fo = d.nchans / d.fscrunch;
    const long long nwin = T / d.tscrunch;
    const long long nout = nwin * Fo;
    FBF_REQUIRE(tf_bytes == (size_t)nout, FBF_ERR_SIZE,
                "fbf_ib: output size " + std::to_string(tf_bytes) + " != expected " + std::to_string(nout));
    const long long nblocks = (4 * nout + 255) / 256;
    FBF_REQUIRE(nblocks < (1ll << 30) && T / 16 < (1ll << 31), FBF_ERR_UNSUPPORTED, "fbf_ib: grid too large");
    *out = IbFinishJob{partials, static_cast<int8_t*>(tf), plan->d_levels, plan->d_levels + Fo, nwin, (int)(T / 16),
                       Fo, d.tscrunch, d.fscrunch, d.quant_mode, nparts, (int)nblocks};
    return FBF_OK;
}

int fbf::ib_fuse_params(const fbf_ib_plan* plan, IbFuseParams* out)
{
    FBF_REQUIRE(plan && out, FBF_ERR_ARG, "fbf_ib: null plan");
    const int fo = plan->d.nchans / plan->d.fscrunch;
    out->offsets = plan->d_levels;
    out->scales = plan->d_levels + fo;
    out->nantennas = plan->d.nantennas;
    out->nchans = plan->d.nchans;
    out->nsamples_per_heap = plan->d.nsamples_per_heap;
    out->tscrunch = plan->d.tscrunch;
    out->fscrunch = plan->d.fscrunch;
    out->quant = plan->d.quant_mode;
    return FBF_OK;
}

extern "C" int fbf_ib_beamform(fbf_ib_plan* plan, const void* taftp, size_t taftp_bytes, void* tf, size_t tf_bytes,
                               fbf_stream_t stream)
{
    return ib_run(plan, IB_INT8, taftp, taftp_bytes, tf, tf_bytes, stream);
}

extern "C" int fbf_ib_beamform_weights(fbf_ib_plan* plan, const void* taftp, size_t taftp_bytes, void* tf,
                                       size_t tf_bytes, fbf_weights_plan* weights_plan, const void* delays,
                                       size_t delays_bytes, double epoch, void* weights, size_t weights_bytes,
                                       fbf_stream_t stream)
{
    FBF_REQUIRE(plan, FBF_ERR_ARG, "fbf_ib_beamform_weights: null plan");
    WeightsJob wj{};
    int st = weights_launch_params(weights_plan, delays, delays_bytes, epoch, weights, weights_bytes, &wj.w);
    if (st) return st;
    FBF_REQUIRE(wj.w.F == plan->d.nchans, FBF_ERR_ARG,
                "fbf_ib_beamform_weights: the weights plan's channels differ from the block's");
    FBF_REQUIRE((unsigned long long)wj.w.gx * wj.w.gy < (1ull << 30), FBF_ERR_UNSUPPORTED,
                "fbf_ib_beamform_weights: too many weights work-groups");
    wj.nblocks = (int)(wj.w.gx * wj.w.gy);
    return ib_run(plan, IB_INT8, taftp, taftp_bytes, tf, tf_bytes, stream, wj);
}

extern "C" int fbf_ib_power(fbf_ib_plan* plan, const void* taftp, size_t taftp_bytes, double* power,
                            size_t power_bytes, fbf_stream_t stream)
{
    return ib_run(plan, IB_POWER, taftp, taftp_bytes, power, power_bytes, stream);
}
