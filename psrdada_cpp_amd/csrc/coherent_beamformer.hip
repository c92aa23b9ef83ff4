// Coherent beamformer on CDNA4 int8 MFMA.
//
// Behaviour follows CoherentBeamformer.cu:48-225 (kernel bf_aptf_general_k and
// CoherentBeamformer::beamform):
//   beam(b, f, t, p) = sum_a w[f][b][a] * v[f][t][p][a]      (no conjugate)
//   P(b, fo, to)     = sum over fscrunch, tscrunch, pol of |beam|^2
//   out              = quantise(P, offset[fo], scale[fo])   written TBTF
//
// The int8 output leaves the beamformer kernel as [Fo][To][B] (beams
// contiguous: each work-group writes whole 64-byte runs) and a second kernel
// (tbtf_k) moves it to TBTF [To/ohs][B][ohs][Fo].  Writing TBTF directly from
// the beamformer (done for small blocks only, cb_tbtf_direct) scatters single
// bytes 1 channel apart across work-groups (one work-group owns one channel),
// which the memory system turns into 32-byte partial writes: 32x the output
// size in HBM writes.
//
// MI355X design.  Per channel the contraction is a real GEMM
//   C[2B x T*P] = W'[2B x 2A] * V'[2A x T*P]
// with the [Re, -Im; Im, Re] embedding: row Re_b = [wr_a, -wi_a] and
// row Im_b = [wi_a, wr_a] over k = (antenna, re/im).  k is interleaved exactly
// as FTPA stores a column (char2 per antenna), so every 16-byte K slice of a
// voltage column is one contiguous 16-byte load straight into the MFMA B
// operand -- no de-interleave and no LDS staging.  The weights are embedded in
// registers from the raw FBA char2 bytes (byte swap for Im rows, negation
// of the odd bytes for Re rows), once per channel per wave; waves whose
// weights hold a wi = -128, whose negation int8 cannot hold, take an exact
// path instead (cb_exact_outputs), so the sums are exact for every int8
// weight.
//
// v_mfma_i32_16x16x64_i8: A (16 rows x 64 k) = weights, B (64 k x 16 cols) =
// voltages, D lane l holds rows 4*(l/16)+i, column l%16.  Rows are ordered
// (beam, re/im) so one lane holds Re and Im of two beams for one column, and
// the 16 columns of a tile are 16 different output samples: column c of the
// j-th tile is input column (t0 + c) * tscrunch * P + j.  Detection and the
// whole tscrunch x pol x fscrunch integration therefore happen in-lane with no
// cross-lane traffic.  Power is accumulated exactly in int64 with
// v_mad_i64_i32 (one instruction per squared int32 sum; |r| < 2^22 for
// A <= 128) and handed to the quantiser as a double, like the oracle.
#include "cb_tr.hpp"

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace fbf {
namespace {

__global__ __launch_bounds__(256) void cb_thresholds_k(const float* offsets, const float* scales, int mode,
                                                       long long* thr)
{
    const int fo = blockIdx.x;
    const float off = offsets[fo], sc = scales[fo];
    long long* t = thr + (size_t)fo * kThr;
    const int j = threadIdx.x + 1;   // 1 .. 256
    if (j == 256) {
        t[0] = LLONG_MIN;
        t[256] = LLONG_MAX;
        return;
    }
    const int k = j - 128;
    long long lo = 0, hi = 1ll << 62;
    if (quantise((double)hi, off, sc, mode) < k) {
        t[j] = LLONG_MAX;
        return;
    }
    while (lo < hi) {   // least P in [lo, hi] with quantise(P) >= k
        const long long mid = lo + (hi - lo) / 2;
        if (quantise((double)mid, off, sc, mode) >= k)
            hi = mid;
        else
            lo = mid + 1;
    }
    t[j] = lo;
}

// ---------------------------------------------------------------------------
// Staged [Fo][To][B] int8 -> TBTF [To/ohs][B][ohs][Fo]
//
// A work-group moves a tile of up to 128 beams x tt samples (within one
// output heap) x up to 64 channels.  Loads are 8-byte runs of beams (a tile
// row is a whole 128-byte line, so no line is fetched by two work-groups);
// the tile is scattered into LDS as [t][b][f] (channel bytes contiguous) and
// written out as 4-byte words of channels, so one wave stores whole rows of
// tt * Fo contiguous bytes per beam.  LDS dword layout: b pitch BP (odd),
// t pitch TP = 128 * BP + 16, so that the word reads of a wave (16 words of
// one (t, b) row x 4 samples) fall in distinct banks.
// ---------------------------------------------------------------------------
constexpr int kTrBeams = 128;
constexpr int kTrMaxChans = 64;
constexpr int kTrLdsBudget = 40 * 1024;

// Tile bid of one reorder.
__device__ __forceinline__ void tbtf_tile(const TbtfArgs& a, long long bid, int8_t* tr_lds)
{
    const int bt = (int)(bid % a.n_btiles);
    bid /= a.n_btiles;
    const int ftile = (int)(bid % a.n_ftiles);
    bid /= a.n_ftiles;
    const int ttile = (int)(bid % a.n_ttiles);
    const long long heap = bid / a.n_ttiles;
    const int b0 = bt * kTrBeams, f0 = ftile * a.ft, t0 = ttile * a.tt;
    const int bv = min(kTrBeams, a.B - b0), fv = min(a.ft, a.Fo - f0), tv = min(a.tt, a.ohs - t0);
    const long long tg0 = heap * a.ohs + t0;

    // 16-byte path: beams, channels, B and Fo multiples of 16 (the tile's
    // beams and channels then start 16-aligned, and so do the rows).
    const bool wide = ((bv | fv | a.B | a.Fo) & 15) == 0;
    if (wide) {
        // Load item: 16 beams x 4 channels as four 16-byte loads (beam
        // sixteens fastest, so a wave reads whole 128-byte rows); four 4 x 4
        // byte transposes with v_perm_b32; sixteen words of 4 channels to
        // LDS.
        const int nb16 = bv >> 4, nfg = fv >> 2;
        const int nitems = nb16 * tv * nfg;
        const size_t fstep = (size_t)a.To * a.B;
        for (int i = threadIdx.x; i < nitems; i += 256) {
            const int bs = i % nb16;
            const int rest = i / nb16;
            const int t = rest % tv;
            const int fg = rest / tv;
            const int8_t* src = a.src + ((size_t)(f0 + 4 * fg) * a.To + tg0 + t) * a.B + b0 + 16 * bs;
            const uint4 q0 = *reinterpret_cast<const uint4*>(src);
            const uint4 q1 = *reinterpret_cast<const uint4*>(src + fstep);
            const uint4 q2 = *reinterpret_cast<const uint4*>(src + 2 * fstep);
            const uint4 q3 = *reinterpret_cast<const uint4*>(src + 3 * fstep);
            uint32_t* l = reinterpret_cast<uint32_t*>(tr_lds) + (size_t)t * a.tp + (size_t)(16 * bs) * a.bp + fg;
            auto quad = [&](uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3, uint32_t* lq) {
                const uint32_t t0 = __builtin_amdgcn_perm(r1, r0, 0x05010400u);
                const uint32_t t1 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
                const uint32_t t2 = __builtin_amdgcn_perm(r3, r2, 0x05010400u);
                const uint32_t t3 = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
                lq[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
                lq[a.bp] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
                lq[2 * a.bp] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
                lq[3 * a.bp] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
            };
            quad(q0.x, q1.x, q2.x, q3.x, l);
            quad(q0.y, q1.y, q2.y, q3.y, l + 4 * a.bp);
            quad(q0.z, q1.z, q2.z, q3.z, l + 8 * a.bp);
            quad(q0.w, q1.w, q2.w, q3.w, l + 12 * a.bp);
        }
    } else if ((fv & 3) == 0 && (f0 & 3) == 0) {
        // Load 4 channels x 4 beams as four 4-byte words (beam quads
        // fastest, so a wave reads whole 128-byte rows), transpose the 4 x 4
        // bytes with v_perm_b32 and write four words of 4 channels.
        const int nbq = bv >> 2, nfg = fv >> 2;
        const int nitems = nbq * tv * nfg;
        for (int i = threadIdx.x; i < nitems; i += 256) {
            const int bq = i % nbq;
            const int rest = i / nbq;
            const int t = rest % tv;
            const int fg = rest / tv;
            const int8_t* src = a.src + ((size_t)(f0 + 4 * fg) * a.To + tg0 + t) * a.B + b0 + 4 * bq;
            const size_t fstep = (size_t)a.To * a.B;
            const uint32_t r0 = *reinterpret_cast<const uint32_t*>(src);
            const uint32_t r1 = *reinterpret_cast<const uint32_t*>(src + fstep);
            const uint32_t r2 = *reinterpret_cast<const uint32_t*>(src + 2 * fstep);
            const uint32_t r3 = *reinterpret_cast<const uint32_t*>(src + 3 * fstep);
            const uint32_t t0 = __builtin_amdgcn_perm(r1, r0, 0x05010400u);   // r0.0 r1.0 r0.1 r1.1
            const uint32_t t1 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);   // r0.2 r1.2 r0.3 r1.3
            const uint32_t t2 = __builtin_amdgcn_perm(r3, r2, 0x05010400u);   // r2.0 r3.0 r2.1 r3.1
            const uint32_t t3 = __builtin_amdgcn_perm(r3, r2, 0x07030602u);   // r2.2 r3.2 r2.3 r3.3
            uint32_t* l = reinterpret_cast<uint32_t*>(tr_lds) + (size_t)t * a.tp + (size_t)(4 * bq) * a.bp + fg;
            l[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);               // beam 0: channels 0..3
            l[a.bp] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);            // beam 1
            l[2 * a.bp] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);        // beam 2
            l[3 * a.bp] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);        // beam 3
        }
    } else {
    // Load: (piece of 8 beams, t, f), pieces fastest.
    const int nb8 = bv >> 3;
    const int nload = fv * tv * nb8;
    for (int i = threadIdx.x; i < nload; i += 256) {
        const int pb = i % nb8;
        const int rest = i / nb8;
        const int t = rest % tv;
        const int f = rest / tv;
        const uint2 v = *reinterpret_cast<const uint2*>(a.src + ((size_t)(f0 + f) * a.To + tg0 + t) * a.B + b0 +
                                                        8 * pb);
        int8_t* l = tr_lds + ((size_t)t * a.tp + (size_t)(8 * pb) * a.bp) * 4 + f;
        const size_t bstep = (size_t)a.bp * 4;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            l[k * bstep] = (int8_t)(v.x >> (8 * k));
            l[(k + 4) * bstep] = (int8_t)(v.y >> (8 * k));
        }
    }
    }
    __syncthreads();

    // Store: (word of 4 channels, t, b), words fastest; a beam's tv rows of
    // Fo channels are contiguous in TBTF when the tile holds every channel.
    int8_t* out = a.dst + (((size_t)heap * a.B + b0) * a.ohs + t0) * a.Fo + f0;
    const size_t brow = (size_t)a.ohs * a.Fo;
    if (wide) {
        // Store item: 16 channels of one (beam, sample) as one 16-byte store
        // (channel sixteens fastest, then samples: a beam's tv rows are one
        // contiguous run).
        const int n16 = fv >> 4;
        const int nstore = bv * tv * n16;
        for (int i = threadIdx.x; i < nstore; i += 256) {
            const int w = i % n16;
            const int rest = i / n16;
            const int t = rest % tv;
            const int b = rest / tv;
            const uint32_t* l = reinterpret_cast<const uint32_t*>(tr_lds) + (size_t)t * a.tp + (size_t)b * a.bp + 4 * w;
            uint4 v;
            v.x = l[0];
            v.y = l[1];
            v.z = l[2];
            v.w = l[3];
            typedef uint32_t v4u __attribute__((ext_vector_type(4)));
            __builtin_nontemporal_store(v4u{v.x, v.y, v.z, v.w},
                                        reinterpret_cast<v4u*>(out + b * brow + (size_t)t * a.Fo + 16 * w));
        }
    } else if ((a.Fo & 3) == 0) {
        const int nw = fv >> 2;
        const int nstore = bv * tv * nw;
        for (int i = threadIdx.x; i < nstore; i += 256) {
            const int w = i % nw;
            const int rest = i / nw;
            const int t = rest % tv;
            const int b = rest / tv;
            const uint32_t word =
                *reinterpret_cast<const uint32_t*>(tr_lds + ((size_t)t * a.tp + (size_t)b * a.bp + w) * 4);
            *reinterpret_cast<uint32_t*>(out + b * brow + (size_t)t * a.Fo + 4 * w) = word;
        }
    } else {
        const int nstore = bv * tv * fv;
        for (int i = threadIdx.x; i < nstore; i += 256) {
            const int f = i % fv;
            const int rest = i / fv;
            const int t = rest % tv;
            const int b = rest / tv;
            out[b * brow + (size_t)t * a.Fo + f] = tr_lds[((size_t)t * a.tp + (size_t)b * a.bp) * 4 + f];
        }
    }
}

// The first wj.nblocks work-groups generate weights (the next block's,
// weights_job_run), the next job.nblocks finish the incoherent beam from the
// coherent kernel's partials (ib_finish_run), both beside the reorder; the
// rest reorder, numbered from 0.
__global__ __launch_bounds__(256) void tbtf_k(TbtfArgs a, IbFinishJob job, WeightsJob wj)
{
    extern __shared__ __align__(16) int8_t tr_lds[];
    if (weights_job_run(wj, threadIdx.x)) return;   // uniform over the work-group
    const int b1 = (int)blockIdx.x - wj.nblocks;
    if (b1 < job.nblocks) {
        ib_finish_run(job, (long long)b1 * 256 + threadIdx.x);
        return;
    }
    tbtf_tile(a, (long long)b1 - job.nblocks, tr_lds);
}

// The reorders of up to kTbtfJobs subarrays of a batch in one launch (after
// the incoherent beam's finish): each by itself fills the chip for a few
// microseconds at most, and starts and drains alone.  Subarrays of 40, 16 and 8
// antennas (768, 256, 64 beams, 64 channels, 8192 samples) took 253.8 us with a
// launch for each and 247.3 us with one; 8, 16, 8, 32 antennas (72, 112, 16, 32
// beams, 44 channels, 2304 samples) 64.5 and 52.0 us.
constexpr int kTbtfJobs = 8;

struct TbtfJobs {
    TbtfArgs a[kTbtfJobs];
    int first[kTbtfJobs];   // first work-group of each
    int n;
};

__global__ __launch_bounds__(256) void tbtf_jobs_k(TbtfJobs jobs, IbFinishJob job)
{
    extern __shared__ __align__(16) int8_t tr_lds[];
    const int b1 = (int)blockIdx.x;
    if (b1 < job.nblocks) {
        ib_finish_run(job, (long long)b1 * 256 + threadIdx.x);
        return;
    }
    const int b = b1 - job.nblocks;
    int k = jobs.n - 1;
    while (k > 0 && b < jobs.first[k]) --k;
    const TbtfArgs a = jobs.a[k];
    tbtf_tile(a, b - jobs.first[k], tr_lds);
}

// Tile shape and grid for tbtf_k.
TbtfArgs tbtf_args(const int8_t* src, int8_t* dst, long long To, int B, int Fo, int ohs)
{
    TbtfArgs a{};
    a.src = src;
    a.dst = dst;
    a.To = To;
    a.B = B;
    a.Fo = Fo;
    a.ohs = ohs;
    a.ft = Fo < kTrMaxChans ? Fo : kTrMaxChans;
    a.bp = (a.ft + 3) / 4 + 1;
    if ((a.bp & 1) == 0) ++a.bp;
    a.tp = kTrBeams * a.bp + 16;
    // Samples per tile: the fewest that still give each beam one 128-byte
    // output run (tt * Fo bytes when the tile holds every channel), so the
    // grid has as many work-groups as that allows (2 samples at 64
    // channels measured 1.5 % faster over the CB window than 4).
    int tt = 1;
    if (a.ft == Fo)
        while (tt < 16 && tt * Fo < 128) tt <<= 1;
    while (tt > 1 && (size_t)tt * a.tp * 4 > (size_t)kTrLdsBudget) tt >>= 1;
    a.tt = tt < ohs ? tt : ohs;
    a.n_ttiles = (ohs + a.tt - 1) / a.tt;
    a.n_ftiles = (Fo + a.ft - 1) / a.ft;
    a.n_btiles = (B + kTrBeams - 1) / kTrBeams;
    return a;
}

long long tbtf_blocks(const TbtfArgs& a) { return a.To / a.ohs * a.n_ttiles * a.n_ftiles * a.n_btiles; }

hipError_t launch_tbtf(const TbtfArgs& a, hipStream_t s, const IbFinishJob& job, const WeightsJob& wj)
{
    const long long nblocks = tbtf_blocks(a) + job.nblocks + wj.nblocks;
    if (nblocks <= 0) return hipSuccess;
    if (nblocks >= (1ll << 31)) return hipErrorInvalidConfiguration;
    const size_t shm = (size_t)a.tt * a.tp * 4;
    tbtf_k<<<dim3((unsigned)nblocks), 256, shm, s>>>(a, job, wj);
    return hipGetLastError();
}

}  // namespace
}  // namespace fbf

// ---------------------------------------------------------------------------
// Plan and C ABI
// ---------------------------------------------------------------------------
using namespace fbf;

struct fbf_cb_plan {
    fbf_cb_desc d;
    int ohs;
    int variant;
    int chunk;        // LDS chunk length in columns, 0 = automatic
    float* d_levels;  // device: offsets[Fo], scales[Fo], then the thresholds [Fo][kThr] (int64)
    void* staging;    // [Fo][To][B] int8 between the beamformer and tbtf_k
    size_t staging_bytes;
    void* ftpa;       // FTPA of fbf_cb_beamform_taftp's split-transpose path
    size_t ftpa_bytes;
    void* ibp;        // incoherent-beam partials of fbf_cb_ib_beamform_taftp
    size_t ibp_bytes;
    hipEvent_t t_before, t_after;   // recorded around the coherent kernel (fbf_cb_plan_set_timing)
};

static long long* cb_thr(const fbf_cb_plan* plan)
{
    return reinterpret_cast<long long*>(plan->d_levels + 2 * (plan->d.nchans / plan->d.fscrunch));
}

// Grows one of the plan's device buffers (not while the stream is being
// captured).
static int cb_grow(void** buf, size_t* have, size_t bytes, hipStream_t s, void** out)
{
    if (*have < bytes) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        FBF_HIP_TRY(hipStreamIsCapturing(s, &cs));
        FBF_REQUIRE(cs == hipStreamCaptureStatusNone, FBF_ERR_STATE,
                    "fbf_cb: the plan's buffers must be sized (fbf_cb_plan_reserve) before stream capture");
        // Earlier launches on any stream may still use the old buffer.
        if (*buf) {
            FBF_HIP_TRY(hipDeviceSynchronize());
            FBF_HIP_TRY(hipFree(*buf));
        }
        *buf = nullptr;
        *have = 0;
        FBF_HIP_TRY(hipMalloc(buf, bytes));
        *have = bytes;
    }
    *out = *buf;
    return FBF_OK;
}

// Whether a call wants more of a buffer than there is while its stream is
// being captured, which leaves cb_grow only its error.
static int cb_cannot_grow(size_t have, size_t bytes, hipStream_t s, bool* out)
{
    *out = false;
    if (have >= bytes) return FBF_OK;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    FBF_HIP_TRY(hipStreamIsCapturing(s, &cs));
    *out = cs != hipStreamCaptureStatusNone;
    return FBF_OK;
}

static int cb_staging(fbf_cb_plan* plan, size_t bytes, hipStream_t s, void** out)
{
    return cb_grow(&plan->staging, &plan->staging_bytes, bytes, s, out);
}

static int cb_validate(const fbf_cb_desc* d)
{
    FBF_REQUIRE(d, FBF_ERR_ARG, "fbf_cb: null descriptor");
    FBF_REQUIRE(d->nantennas > 0 && d->nbeams > 0 && d->nchans > 0 && d->tscrunch > 0 && d->fscrunch > 0,
                FBF_ERR_ARG, "fbf_cb: geometry values must be positive");
    FBF_REQUIRE(d->nantennas % 4 == 0 && d->nantennas <= 128, FBF_ERR_UNSUPPORTED,
                "fbf_cb: nantennas must be a multiple of 4 and <= 128 (CoherentBeamformer.cu:60-70)");
    FBF_REQUIRE(d->nbeams % 8 == 0, FBF_ERR_UNSUPPORTED, "fbf_cb: nbeams must be a multiple of 8");
    FBF_REQUIRE(d->nchans % d->fscrunch == 0, FBF_ERR_ARG, "fbf_cb: fscrunch must divide nchans");
    FBF_REQUIRE(d->quant_mode == FBF_QUANT_ROUND || d->quant_mode == FBF_QUANT_TRUNC, FBF_ERR_ARG,
                "fbf_cb: bad quant_mode");
    FBF_REQUIRE(d->nsamples_per_heap_out >= 0, FBF_ERR_ARG, "fbf_cb: bad nsamples_per_heap_out");
    return FBF_OK;
}

// Process-wide autotuning table: geometry -> (variant, chunk).
namespace {
std::mutex g_tune_mutex;
std::map<std::string, std::pair<int, int>> g_tune_table;

std::string tune_key(const fbf_cb_desc& d)
{
    return std::to_string(d.nantennas) + "/" + std::to_string(d.nbeams) + "/" + std::to_string(d.nchans) + "/" +
           std::to_string(d.tscrunch) + "/" + std::to_string(d.fscrunch);
}
}  // namespace

extern "C" int fbf_cb_plan_create(const fbf_cb_desc* desc, const float* offsets, const float* scales,
                                  fbf_cb_plan** plan)
{
    FBF_REQUIRE(plan, FBF_ERR_ARG, "fbf_cb_plan_create: null plan pointer");
    *plan = nullptr;
    int st = cb_validate(desc);
    if (st) return st;
    FBF_REQUIRE(offsets && scales, FBF_ERR_ARG, "fbf_cb_plan_create: null offsets/scales");
    const int Fo = desc->nchans / desc->fscrunch;
    int ohs = desc->nsamples_per_heap_out ? desc->nsamples_per_heap_out : 8192 / Fo;
    FBF_REQUIRE(ohs > 0, FBF_ERR_ARG, "fbf_cb_plan_create: output heap holds no samples");
    auto* p = new fbf_cb_plan{*desc, ohs, 0, 0, nullptr, nullptr, 0, nullptr, 0, nullptr, 0, nullptr, nullptr};
    hipError_t e = hipMalloc(&p->d_levels, sizeof(float) * 2 * Fo + sizeof(long long) * kThr * Fo);
    if (e != hipSuccess) {
        delete p;
        return hip_status(e, "hipMalloc(levels)");
    }
    st = fbf_cb_plan_set_levels(p, offsets, scales);
    if (st) {
        (void)hipFree(p->d_levels);
        delete p;
        return st;
    }
    {
        std::lock_guard<std::mutex> lock(g_tune_mutex);
        auto it = g_tune_table.find(tune_key(*desc));
        if (it != g_tune_table.end()) {
            p->variant = it->second.first;
            p->chunk = it->second.second;
        }
    }
    *plan = p;
    return FBF_OK;
}

extern "C" int fbf_cb_plan_set_levels(fbf_cb_plan* plan, const float* offsets, const float* scales)
{
    FBF_REQUIRE(plan && offsets && scales, FBF_ERR_ARG, "fbf_cb_plan_set_levels: null argument");
    const int Fo = plan->d.nchans / plan->d.fscrunch;
    // A beamform still running on any stream reads the levels and thresholds
    // being replaced (the library's streams do not wait for the null stream):
    // it finishes first.
    FBF_HIP_TRY(hipDeviceSynchronize());
    FBF_HIP_TRY(hipMemcpy(plan->d_levels, offsets, sizeof(float) * Fo, hipMemcpyHostToDevice));
    FBF_HIP_TRY(hipMemcpy(plan->d_levels + Fo, scales, sizeof(float) * Fo, hipMemcpyHostToDevice));
    cb_thresholds_k<<<Fo, 256, 0, nullptr>>>(plan->d_levels, plan->d_levels + Fo, plan->d.quant_mode,
                                             cb_thr(plan));
    FBF_HIP_TRY(hipGetLastError());
    FBF_HIP_TRY(hipStreamSynchronize(nullptr));
    return FBF_OK;
}

extern "C" int fbf_cb_plan_destroy(fbf_cb_plan* plan)
{
    if (!plan) return FBF_OK;
    hipError_t e = hipFree(plan->d_levels);
    if (plan->staging) {
        const hipError_t e2 = hipFree(plan->staging);
        if (e == hipSuccess) e = e2;
    }
    if (plan->ftpa) {
        const hipError_t e2 = hipFree(plan->ftpa);
        if (e == hipSuccess) e = e2;
    }
    if (plan->ibp) {
        const hipError_t e2 = hipFree(plan->ibp);
        if (e == hipSuccess) e = e2;
    }
    delete plan;
    if (e != hipSuccess) return hip_status(e, "hipFree(levels)");
    return FBF_OK;
}

// Kernel variants: MFMA shape and beams per wave.  Variant 0 picks
// automatically (the tuned choice for the geometry).
struct CbVariant {
    int mfma;        // 32: v_mfma_i32_32x32x32_i8, 16: v_mfma_i32_16x16x64_i8
    int rows;        // row tiles per wave (RT for 32x32, ROWT for 16x16)
    bool lds;        // voltage tile staged through LDS and shared by the work-group
    bool tr;         // transposed tiles (cb_tr_k): voltages as the A operand
    bool ws;         // transposed tiles with wave-private staging (cb_ws_k)
    bool few = false;   // transposed: one beam group, four time slots to a work-group (cb_tr_few.hip)
};
static const CbVariant kCbVariants[] = {
    {0, 0, false, false, false},   // auto
    {32, 4, false, false, false},  // 64 beams x 32 samples per wave
    {32, 2, false, false, false},  // 32 beams x 32 samples per wave
    {16, 8, false, false, false},  // 64 beams x 16 samples per wave
    {16, 4, false, false, false},  // 32 beams x 16 samples per wave
    {32, 1, true, false, false},   // LDS: 16 beams per wave, 64 per work-group
    {32, 2, true, false, false},   // LDS: 32 beams per wave, 128 per work-group
    {32, 4, true, false, false},   // LDS: 64 beams per wave, 256 per work-group
    {32, 2, true, true, false},    // transposed: 32 beams per wave
    {32, 4, true, true, false},    // transposed: 64 beams per wave
    {32, 4, true, true, true},     // transposed, wave-private staging: 64 beams per wave
    {32, 8, true, true, false},    // transposed: 128 beams per wave, two waves per SIMD
};
constexpr int kCbVariantLds = 5;
constexpr int kCbVariantTr2 = 8;
constexpr int kCbVariantTr4 = 9;
constexpr int kCbVariantTr8 = 11;

static bool cb_tr_applies(const fbf_cb_desc& d, int rt, int mode, long long T)
{
    return mode == MODE_INT8 && T % 16 == 0 && 2 * T / 32 < (1ll << 31) && T / d.tscrunch < (1ll << 31) &&
           cb_tr_supported(d.nantennas, d.tscrunch, d.fscrunch, rt);
}

static bool cb_ws_applies(const fbf_cb_desc& d, int mode, long long T)
{
    return mode == MODE_INT8 && T % 16 == 0 && 2 * T / 32 < (1ll << 31) &&
           cb_ws_supported(d.nantennas, d.tscrunch, d.fscrunch);
}

// Work-groups of the transposed kernel with waves of 16 rt beams, `beams` beams
// and `slots` time slots to a work-group and one pass on every slot.
static long long cb_groups(const fbf_cb_desc& d, long long T, int rt, int beams, int slots)
{
    const int W = 2 * d.tscrunch;
    const int spt = W >= 32 ? 1 : 32 / W, tps = W >= 32 ? W / 32 : 1;
    const long long ntp = (long long)(cb_tr_nslot(rt, W) / spt) * tps;
    const long long passes = (2 * T / 32 + ntp - 1) / ntp;
    return (long long)(d.nchans / d.fscrunch) * ((d.nbeams + beams - 1) / beams) * ((passes + slots - 1) / slots);
}

// Whether the few-beam form (cb_tr_few.hip: waves of 16 rt beams, four time slots
// to a work-group) runs all its waves in `rounds` rounds of one pass each.
//
// A pass is two windows or more in a row, whatever else of the chip is idle, and
// a wave of 128 beams takes twice as long over it as one of 64.  So small blocks
// take waves of 64 beams, and where the windows are long and there is room even
// for those waves of 32 (us; 128, 64 and 32 beams a wave, and the wave-private
// kernel from FTPA; antennas / beams / channels / samples / tscrunch, TAFTP
// marked t): 48/96/4/1024/256 t 33.8, 24.3, 20.2; 16/96/4/1024/64 12.6, 7.1,
// 6.1, 10.7; 48/96/16/2048/128 20.5, 13.4, 11.0, 15.0; 40/256/16/2048/16 14.4,
// 10.4, -, 14.0; but with 32 beams 56/208/8/256/8 7.4 against 6.1, and in four
// rounds of 64 40/512/64/4096/128 64.0 against 52.2 with 128.
static bool cb_few_fit(const fbf_cb_desc& d, long long T, int rt, int rounds)
{
    return cb_groups(d, T, rt, 16 * rt, 4) <= (long long)rounds * tr_wgs(rt, 1) * device_cu_count();
}

// Beam tiles of the few-beam form for a block, 0: it takes another form.
static int cb_few_rows(const fbf_cb_desc& d, long long T)
{
    if (d.nbeams <= 32 || (d.tscrunch >= 32 && cb_few_fit(d, T, 2, 1))) return 2;
    return d.nbeams <= 64 || cb_few_fit(d, T, 4, 2) ? 4 : 0;
}

// Automatic choice from FTPA: the transposed kernel, up to 64 antennas with
// 128 beams per wave or with 32 or 64 for few beams and small blocks
// (cb_few_rows), above with 64 (32 for at most 32: a 64-beam wave would be half
// empty); the LDS-staged kernel for the rest (tscrunch below 4 or no power of
// two, fscrunch above 4, also int32 sums and power output).  Measured against the
// wave-private kernel and the earlier picks (us; antennas / beams / channels /
// samples / tscrunch): 16/256/64/8192/16 40.6 against 44.7, 48/512/64/8192/16 111
// against 128, 40/768/64/8192/4 250 against 272, 8/64/64/8192/16 16.4 against
// 17.4, 16/32/16/2048/16 8.3 against 9.4 (5.4 in one launch, cb_tbtf_direct); but
// 8/768/64/8192/128, whose units fill the rounds of the grid to 87 %, 92 against
// 85.  fscrunch 2 and 4: 128 beams per wave above 96 beams, or where the forms
// with several time slots per work-group end (two K steps of four channels);
// 44/1024/64/8192/16 at fscrunch 4 took 205 against 348 of the LDS-staged kernel,
// 44/64 32 against 50, but 24/64 26.7 against 24.5 with 32 beams per wave.  Small
// blocks of them in FTPA: cb_pick_ftpa.
static CbVariant cb_pick_variant(const fbf_cb_desc& d, int variant, int mode, long long T)
{
    if (variant <= 0) {
        const int ksteps = (2 * d.nantennas + 31) / 32;
        const bool tr8 = cb_tr_applies(d, 8, mode, T);
        const int few = tr8 && d.fscrunch == 1 ? cb_few_rows(d, T) : 0;
        if (few) return {32, few, true, true, false, true};
        if (tr8 && (d.fscrunch == 1 || d.nbeams > 96 || d.fscrunch * ksteps > 8)) return kCbVariants[kCbVariantTr8];
        if ((ksteps <= 4 || d.nbeams > 32) && cb_tr_applies(d, 4, mode, T)) return kCbVariants[kCbVariantTr4];
        if (cb_tr_applies(d, 2, mode, T)) return kCbVariants[kCbVariantTr2];
        return kCbVariants[kCbVariantLds];
    }
    const CbVariant v = kCbVariants[variant];
    if (v.ws && !cb_ws_applies(d, mode, T)) return cb_pick_variant(d, 0, mode, T);
    if (v.tr && !v.ws && !cb_tr_applies(d, v.rows, mode, T)) return kCbVariants[kCbVariantLds];
    return v;
}

// The kernel of a block in FTPA.  As cb_pick_variant, but automatic blocks with
// channels summed over and more than 96 beams take waves of 32 beams where the
// kernel has them (three time slots to a work-group: of eight K slices over the
// summed channels, which 44 to 64 antennas at fscrunch 2 and 20 to 32 at 4 have,
// and windows of 32 columns or more) and one round of one pass each holds the
// block.
//
// With 128 beams a wave, such a block is a few waves that each take four times
// as long over a pass (us, 32 beams against 128; antennas / beams / channels /
// samples / tscrunch / fscrunch): 64/264/6/1024/256/2 26.0 against 35.6,
// 52/512/4/256/128/2 16.2 against 22.3, 64/304/16/1024/128/2 20.5 against 24.0,
// 56/256/4/3072/32/2 13.2 against 14.3, 20/400/8/1536/256/4 25.9 against 28.8; but
// in two rounds 32/232/24/4096/128/4 31.0 against 25.2.  From TAFTP only 128
// beams a wave stage the block, and the split-transpose costs what the narrow
// waves give: 64/136/6/2048/64/2 18.3 staged, 21.0 split.
static CbVariant cb_pick_ftpa(const fbf_cb_desc& d, int variant, int mode, long long T)
{
    if (variant <= 0 && d.fscrunch > 1 && d.nbeams > 96 && cb_tr_applies(d, 2, mode, T) &&
        cb_groups(d, T, 2, 128 / d.fscrunch, 3) <= device_cu_count())
        return kCbVariants[kCbVariantTr2];
    return cb_pick_variant(d, variant, mode, T);
}

extern "C" int fbf_cb_variant_count(int* count)
{
    FBF_REQUIRE(count, FBF_ERR_ARG, "fbf_cb_variant_count: null pointer");
    *count = (int)(sizeof(kCbVariants) / sizeof(kCbVariants[0]));
    return FBF_OK;
}

extern "C" int fbf_cb_plan_set_variant(fbf_cb_plan* plan, int variant)
{
    int n = 0;
    fbf_cb_variant_count(&n);
    FBF_REQUIRE(plan && variant >= 0 && variant < n, FBF_ERR_ARG, "fbf_cb_plan_set_variant: bad variant");
    plan->variant = variant;
    return FBF_OK;
}

static int cb_nsamples(const fbf_cb_plan* plan, size_t ftpa_bytes, long long* nsamples)
{
    const size_t per_sample = (size_t)2 * 2 * plan->d.nantennas * plan->d.nchans;
    FBF_REQUIRE(ftpa_bytes % per_sample == 0, FBF_ERR_SIZE,
                "fbf_cb: input is not a whole number of samples (CoherentBeamformer.cu:197)");
    const long long T = (long long)(ftpa_bytes / per_sample);
    FBF_REQUIRE(T % plan->d.tscrunch == 0, FBF_ERR_SIZE, "fbf_cb: nsamples is not a multiple of tscrunch");
    *nsamples = T;
    return FBF_OK;
}

extern "C" int fbf_cb_output_bytes(const fbf_cb_plan* plan, size_t ftpa_bytes, size_t* tbtf_bytes)
{
    FBF_REQUIRE(plan && tbtf_bytes, FBF_ERR_ARG, "fbf_cb_output_bytes: null argument");
    long long T = 0;
    int st = cb_nsamples(plan, ftpa_bytes, &T);
    if (st) return st;
    *tbtf_bytes = (size_t)(T / plan->d.tscrunch) * plan->d.nbeams * (plan->d.nchans / plan->d.fscrunch);
    return FBF_OK;
}

// The transposed kernel that stages a TAFTP block itself: RT beam tiles (16
// RT beams) per wave, 0 where none does; `few` as in CbVariant.
struct TaftpForm {
    int rt;
    bool few;
};

// A TAFTP block read directly by the coherent beamformer: S samples per
// heap, Atot antennas, the beamformer's antennas from antenna a0.
struct TaftpView {
    int S, Atot, a0;
    TaftpForm form;   // the kernel (cb_taftp_form)
    int* ibp;      // incoherent-beam partials to leave (cb_ib_fused), or null
};

// Work for the reorder's launch beside the reorder: the finish of the
// incoherent-beam partials, and weights generated there (the next block's:
// the coherent kernel has read this block's by then).
struct TailJobs {
    IbFinishJob ib;
    WeightsJob weights;
    TbtfArgs* defer = nullptr;   // leave the reorder's arguments here instead of launching it
};

static hipError_t cb_reorder(const TbtfArgs& a, hipStream_t s, const TailJobs& tail)
{
    if (!tail.defer) return launch_tbtf(a, s, tail.ib, tail.weights);
    *tail.defer = a;
    return hipSuccess;
}

struct Span {
    const void* p;
    size_t n;
};

static bool spans_overlap(const Span& a, const Span& b)
{
    const uintptr_t x = reinterpret_cast<uintptr_t>(a.p), y = reinterpret_cast<uintptr_t>(b.p);
    return a.n && b.n && x < y + b.n && y < x + a.n;
}

// Whether a few-beam form of the kernel writes TBTF itself, with the tail's
// jobs in its own launch (CbTrArgs::tbtf): outputs of at most kTbtfDirect
// bytes, none of them over the kernel's inputs (next weights written over the
// block's, say: those are read until the launch ends), and an incoherent beam
// of this block alone in windows within a tile.
//
// Such blocks are launches and latency: the reorder's launch costs more than
// its scattered bytes.  One launch against two (us; antennas / beams /
// channels / heaps, output size): both beams and the next weights 16/32/16/8,
// 64 KiB 7.0 against 9.5, 48/64/64/4, 256 KiB 10.6 against 12.9, 48/64/64/8,
// 512 KiB 13.9 against 15.0, but 48/64/64/16, 1 MiB 20.8 against 20.5; the
// coherent beams alone 5.3 against 8.9, 8.7 against 11.2, 11.3 against 13.4, and
// 2 MiB 33.7 against 30.7.  Above 64 antennas the coherent beams alone 96/128/64/4,
// 512 KiB 14.8 against 17.6, but with the incoherent beam, whose outputs a wave
// with beams sums and quantises tile by tile, only up to 65536 channels x
// samples: 72/16/64/4 14.3 against 14.8, 72/16/64/8 20.0 against 19.1.
constexpr size_t kTbtfDirect = 1 << 19;
constexpr long long kTbtfDirectIb = 1 << 16;

static bool cb_tbtf_direct(int ksteps, const Span& volts, const Span& weights, const Span& out, const TailJobs& tail)
{
    auto clear = [&](const Span& o) { return !spans_overlap(o, volts) && !spans_overlap(o, weights); };
    if (out.n > kTbtfDirect || !clear(out)) return false;
    const IbFinishJob& ib = tail.ib;
    if (ib.nblocks && (ib.nparts != 1 || ib.fs != 1 || ib.ts > 16 ||
                       (ksteps > 4 && ib.nwin * ib.ts * ib.Fo > kTbtfDirectIb) ||
                       !clear(Span{ib.out, (size_t)ib.nwin * ib.Fo})))
        return false;
    const WeightsLaunch& w = tail.weights.w;
    return !tail.weights.nblocks || clear(Span{w.weights, (size_t)2 * w.F * w.nd});
}

// Validates and launches one coherent-beam kernel over T samples of voltage
// columns that are `vstride` bytes apart, the beamformer's antennas starting
// `voff` bytes into each column; or, with `tv`, over the TAFTP block `ftpa`
// (the caller has checked cb_taftp_direct).
static int cb_launch(fbf_cb_plan* plan, int mode, const void* ftpa, long long T, int vstride, int voff,
                     const void* fba, size_t weights_bytes, void* out, size_t out_bytes, fbf_stream_t stream,
                     void* workspace = nullptr, size_t workspace_bytes = 0, const TaftpView* tv = nullptr,
                     const TailJobs& tail = TailJobs{})
{
    FBF_REQUIRE(plan, FBF_ERR_ARG, "fbf_cb: null plan");
    FBF_REQUIRE(ftpa && fba && out, FBF_ERR_ARG, "fbf_cb: null buffer");
    const fbf_cb_desc& d = plan->d;
    FBF_REQUIRE(T % d.tscrunch == 0, FBF_ERR_SIZE, "fbf_cb: nsamples is not a multiple of tscrunch");
    FBF_REQUIRE(vstride >= 2 * d.nantennas + voff && voff >= 0 && vstride % 8 == 0 && voff % 8 == 0,
                FBF_ERR_ARG, "fbf_cb: bad voltage column stride/offset");
    const bool al16_view = (vstride % 16 == 0) && (voff % 16 == 0);
    const size_t wbytes = (size_t)2 * d.nchans * d.nbeams * d.nantennas;
    FBF_REQUIRE(weights_bytes == wbytes, FBF_ERR_SIZE,
                "fbf_cb: weights size " + std::to_string(weights_bytes) + " != expected " +
                    std::to_string(wbytes) + " (CoherentBeamformer.cu:209)");
    const int Fo = d.nchans / d.fscrunch;
    const long long To = T / d.tscrunch;
    size_t expect = 0;
    if (mode == MODE_INT8) {
        FBF_REQUIRE(To % plan->ohs == 0, FBF_ERR_SIZE,
                    "fbf_cb: output samples " + std::to_string(To) + " are not a multiple of the output heap (" +
                        std::to_string(plan->ohs) + ") (CoherentBeamformer.cu:204)");
        expect = (size_t)To * d.nbeams * Fo;
    } else if (mode == MODE_SUMS) {
        expect = (size_t)d.nchans * T * 2 * d.nbeams * 2 * sizeof(int32_t);
    } else {
        expect = (size_t)Fo * To * d.nbeams * sizeof(double);
    }
    FBF_REQUIRE(out_bytes == expect, FBF_ERR_SIZE,
                "fbf_cb: output size " + std::to_string(out_bytes) + " != expected " + std::to_string(expect));
    FBF_REQUIRE((reinterpret_cast<uintptr_t>(ftpa) & 15) == 0 && (reinterpret_cast<uintptr_t>(fba) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(out) & 15) == 0,
                FBF_ERR_ARG, "fbf_cb: buffers must be 16-byte aligned");
    if (T == 0) return FBF_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const CbVariant var =
        tv ? CbVariant{32, tv->form.rt, true, true, false, tv->form.few} : cb_pick_ftpa(d, plan->variant, mode, T);
    const size_t vbytes = tv ? (size_t)4 * tv->Atot * d.nchans * T : (size_t)2 * vstride * d.nchans * T;
    const int wsteps = (2 * d.nantennas + 31) / 32;   // 32-byte K steps
    const bool four_waves = var.few || (var.tr && !var.ws && var.rows == 4 && tr_four_waves(4, wsteps));
    const bool direct = four_waves && mode == MODE_INT8 && d.fscrunch == 1 && !plan->t_before && !plan->t_after &&
                        cb_tbtf_direct(wsteps, Span{ftpa, vbytes}, Span{fba, wbytes}, Span{out, expect}, tail);
    void* kout = out;
    if (mode == MODE_INT8) {
        if (workspace) {
            FBF_REQUIRE(workspace_bytes >= expect && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
                        FBF_ERR_SIZE, "fbf_cb: workspace too small or not 16-byte aligned");
            kout = workspace;
        } else {
            // Also where the kernel writes TBTF itself (at most kTbtfDirect
            // bytes): the plan's next call on such a block may be captured and
            // need it (beams over its inputs, timing events).
            bool skip = false;
            if (direct) {
                const int st = cb_cannot_grow(plan->staging_bytes, expect, s, &skip);
                if (st) return st;
            }
            if (!skip) {
                const int st = cb_staging(plan, expect, s, &kout);
                if (st) return st;
            }
        }
    }
    // The timing events (fbf_cb_plan_set_timing), around the coherent kernel only.
    auto mark = [&](hipEvent_t ev) { return ev ? hipEventRecord(ev, s) : hipSuccess; };
    if (var.ws) {
        CbWsArgs wa{};
        CbArgs& a = wa.p;
        a.ftpa = static_cast<const int8_t*>(ftpa);
        a.fba = static_cast<const int8_t*>(fba);
        a.out = kout;
        a.offsets = plan->d_levels;
        a.scales = plan->d_levels + Fo;
        a.thr = cb_thr(plan);
        a.nsamples = T;
        a.nsamples_out = To;
        a.A = d.nantennas;
        a.B = d.nbeams;
        a.F = d.nchans;
        a.Fo = Fo;
        a.ts = d.tscrunch;
        a.fs = d.fscrunch;
        a.ohs = plan->ohs;
        a.quant = d.quant_mode;
        a.vstride = vstride;
        a.voff = voff;
        const int W = 2 * d.tscrunch;
        const int spt = W >= 32 ? 1 : 32 / W;
        wa.tps = W >= 32 ? W / 32 : 1;
        wa.ntp = (cb_ws_nslot(W) / spt) * wa.tps;
        wa.ntiles = (int)(2 * T / 32);
        wa.nbg = (d.nbeams + 63) / 64;
        const int ksteps = (2 * d.nantennas + 31) / 32;
        hipError_t e = mark(plan->t_before);
        if (e == hipSuccess) e = cb_launch_ws(wa, W, ksteps, s);
        if (e == hipSuccess) e = mark(plan->t_after);
        if (e != hipSuccess) return hip_status(e, "cb_ws_k launch");
        e = cb_reorder(tbtf_args(static_cast<const int8_t*>(kout), static_cast<int8_t*>(out), To, d.nbeams, Fo, plan->ohs), s,
                   tail);
        if (e != hipSuccess) return hip_status(e, "tbtf_k launch");
        return FBF_OK;
    }
    if (var.tr) {
        CbTrArgs ta{};
        CbArgs& a = ta.p;
        a.ftpa = static_cast<const int8_t*>(ftpa);
        a.fba = static_cast<const int8_t*>(fba);
        a.out = kout;
        a.offsets = plan->d_levels;
        a.scales = plan->d_levels + Fo;
        a.thr = cb_thr(plan);
        a.nsamples = T;
        a.nsamples_out = To;
        a.A = d.nantennas;
        a.B = d.nbeams;
        a.F = d.nchans;
        a.Fo = Fo;
        a.ts = d.tscrunch;
        a.fs = d.fscrunch;
        a.ohs = plan->ohs;
        a.quant = d.quant_mode;
        a.vstride = vstride;
        a.voff = voff;
        if (tv) {
            a.S = tv->S;
            a.Atot = tv->Atot;
            a.a0 = tv->a0;
            ta.hstride = (size_t)4 * tv->Atot * d.nchans * tv->S;
            ta.lgtph = __builtin_ctz((unsigned)(tv->S / 16));
            ta.ibp = tv->ibp;
        }
        if (direct) {
            ta.tbtf = static_cast<int8_t*>(out);
            ta.ib = tail.ib;
            ta.weights = tail.weights;
        }
        const int rt = var.rows;
        const int W = 2 * d.tscrunch;
        const int spt = W >= 32 ? 1 : 32 / W;
        ta.tps = W >= 32 ? W / 32 : 1;
        const int nslot = cb_tr_nslot(rt, W);
        ta.ntp = (nslot / spt) * ta.tps;
        ta.ntiles = (int)(2 * T / 32);
        const int passes = (ta.ntiles + ta.ntp - 1) / ta.ntp;
        const int ksteps = (2 * d.nantennas + 31) / 32;
        hipError_t e = mark(plan->t_before);
        if (e == hipSuccess)
            e = var.few             ? cb_launch_tr_few(ta, rt, W, ksteps, passes, s)
                : rt == 2           ? cb_launch_tr2(ta, d.fscrunch, W, ksteps, passes, s)
                : rt == 4           ? cb_launch_tr4(ta, d.fscrunch, W, ksteps, passes, s)
                : d.fscrunch == 1   ? cb_launch_tr8(ta, W, ksteps, passes, s)
                                    : cb_launch_tr8_fs(ta, d.fscrunch, W, ksteps, passes, s);
        if (e == hipSuccess) e = mark(plan->t_after);
        if (e != hipSuccess) return hip_status(e, "cb_tr_k launch");
        if (direct) return FBF_OK;
        e = cb_reorder(tbtf_args(static_cast<const int8_t*>(kout), static_cast<int8_t*>(out), To, d.nbeams, Fo, plan->ohs), s,
                   tail);
        if (e != hipSuccess) return hip_status(e, "tbtf_k launch");
        return FBF_OK;
    }
    const int kbytes = var.mfma == 32 ? 32 : 64;
    const int ksteps = (2 * d.nantennas + kbytes - 1) / kbytes;
    const int beams_per_wave = var.mfma == 32 ? 16 * var.rows : 8 * var.rows;
    const int t_per_wave = var.mfma == 32 ? 32 : 16;
    const bool al16 = d.nantennas % 8 == 0;
    FBF_REQUIRE(!al16 || al16_view, FBF_ERR_ARG,
                "fbf_cb: a multiple-of-8 antenna subset needs a 16-byte aligned column stride and offset");
    int jc = cb_lds_chunk(2 * d.tscrunch, 2 * d.nantennas, al16);
    if (plan->chunk > 0) {
        FBF_REQUIRE((2 * d.tscrunch) % plan->chunk == 0 && plan->chunk <= jc, FBF_ERR_ARG,
                    "fbf_cb: chunk must divide 2*tscrunch and fit the prefetch registers");
        jc = plan->chunk;
    }
    CbArgs a{};
    a.ftpa = static_cast<const int8_t*>(ftpa);
    a.fba = static_cast<const int8_t*>(fba);
    a.out = kout;
    a.offsets = plan->d_levels;
    a.scales = plan->d_levels + Fo;
    a.thr = cb_thr(plan);
    a.nsamples = T;
    a.nsamples_out = To;
    a.A = d.nantennas;
    a.B = d.nbeams;
    a.F = d.nchans;
    a.Fo = Fo;
    a.ts = d.tscrunch;
    a.fs = d.fscrunch;
    a.ohs = plan->ohs;
    a.quant = d.quant_mode;
    a.vstride = vstride;
    a.voff = voff;
    a.n_bchunks = (d.nbeams + beams_per_wave - 1) / beams_per_wave;
    a.n_tchunks = (int)((To + t_per_wave - 1) / t_per_wave);
    if (var.lds) {
        // Four waves share the samples and split the beams.
        a.wb = 4;
        a.n_bgroups = (a.n_bchunks + 3) / 4;
        a.n_tgroups = a.n_tchunks;
    } else {
        a.wb = a.n_bchunks >= 4 ? 4 : (a.n_bchunks >= 2 ? 2 : 1);
        a.n_bgroups = (a.n_bchunks + a.wb - 1) / a.wb;
        const int wt = 4 / a.wb;
        a.n_tgroups = (a.n_tchunks + wt - 1) / wt;
    }
    const long long nblocks = (long long)Fo * a.n_tgroups * a.n_bgroups;
    FBF_REQUIRE(nblocks > 0 && nblocks < (1ll << 31), FBF_ERR_UNSUPPORTED, "fbf_cb: grid too large");
    dim3 grid((unsigned)nblocks);
    hipError_t e = mark(plan->t_before);
    if (e != hipSuccess) return hip_status(e, "hipEventRecord");
    if (var.lds)
        e = cb_launch_lds(a, mode, var.rows, ksteps, jc, grid, s);
    else if (var.mfma == 32)
        e = cb_launch_mfma32(a, mode, var.rows, ksteps, grid, s);
    else
        e = cb_launch_mfma16(a, mode, var.rows, ksteps, grid, s);
    if (e == hipSuccess) e = mark(plan->t_after);
    if (e != hipSuccess) return hip_status(e, "cb_mfma_k launch");
    if (mode == MODE_INT8) {
        e = cb_reorder(tbtf_args(static_cast<const int8_t*>(kout), static_cast<int8_t*>(out), To, d.nbeams, Fo, plan->ohs), s,
                   tail);
        if (e != hipSuccess) return hip_status(e, "tbtf_k launch");
    }
    return FBF_OK;
}

static int cb_run(fbf_cb_plan* plan, int mode, const void* ftpa, size_t ftpa_bytes, const void* fba,
                  size_t weights_bytes, void* out, size_t out_bytes, fbf_stream_t stream)
{
    FBF_REQUIRE(plan, FBF_ERR_ARG, "fbf_cb: null plan");
    long long T = 0;
    int st = cb_nsamples(plan, ftpa_bytes, &T);
    if (st) return st;
    return cb_launch(plan, mode, ftpa, T, 2 * plan->d.nantennas, 0, fba, weights_bytes, out, out_bytes, stream);
}

extern "C" int fbf_cb_beamform_subarray(fbf_cb_plan* plan, const void* ftpa_block, size_t block_bytes,
                                        int block_nantennas, int antenna_offset, const void* fba_weights,
                                        size_t weights_bytes, void* tbtf, size_t tbtf_bytes, fbf_stream_t stream)
{
    FBF_REQUIRE(plan, FBF_ERR_ARG, "fbf_cb_beamform_subarray: null plan");
    FBF_REQUIRE(block_nantennas > 0 && antenna_offset >= 0 &&
                    antenna_offset + plan->d.nantennas <= block_nantennas,
                FBF_ERR_ARG, "fbf_cb_beamform_subarray: subarray outside the block's antennas");
    const size_t per_sample = (size_t)2 * 2 * block_nantennas * plan->d.nchans;
    FBF_REQUIRE(block_bytes % per_sample == 0, FBF_ERR_SIZE,
                "fbf_cb_beamform_subarray: block is not a whole number of samples");
    const long long T = (long long)(block_bytes / per_sample);
    return cb_launch(plan, MODE_INT8, ftpa_block, T, 2 * block_nantennas, 2 * antenna_offset, fba_weights,
                     weights_bytes, tbtf, tbtf_bytes, stream);
}

// The kernel that stages a TAFTP block itself for the plan's coherent beams
// (rt 0: none, the block is split-transposed): the plan's variant, or when
// that is automatic 128 beams per wave up to 64 antennas (32 or 64 for few beams
// and small blocks, cb_few_rows) and 64 beams per wave above.
//
// Staging the block itself was the faster at every size measured.  Blocks of
// both beams, direct against split-transposed (us; antennas / beams / channels
// / heaps, tscrunch 16; the reorder in a launch of its own, which the first two
// now do without, cb_tbtf_direct): 16/32/16/8 8.6 against 17.1, 48/64/64/8 13.0
// against 27.8, 64/64/64/32 33.7 against 79.5, 128/32/64/8 22.9 against 45.0.  Waves
// of 32 or 64 beams for so few took 8.6 and 33.7 us where 128-beam waves took
// 10.8 and 41.0.
// Not for speed, blocks of at most kTaftpSmall channels x samples are
// split-transposed where fbf_cb_taftp_direct and fbf_cb_ib_fused tell callers,
// who choose their calls and reserve their buffers by it, that they are: at most
// 96 beams of up to 48 antennas (unless both beams of the whole block are
// formed), at most 32 of more than 64 on their own.  It costs one launch of the
// small ones (16 of 64 antennas, 32 beams, 4 channels, 4 heaps 7.9 us) and much
// above 64 antennas (96/32/4/4 23.5 us, 6.4 staged; 128/32/2/1 16.4 and 6.9).
constexpr long long kTaftpSmall = 4096;

enum TaftpUse {
    kTaftpAlone,     // fbf_cb_beamform_taftp
    kTaftpOnePass,   // with the incoherent beam of the whole block
    kTaftpBatch      // one of a batch's subarrays
};

static TaftpForm cb_taftp_form(const fbf_cb_plan* plan, long long T, int nantennas_total, TaftpUse use)
{
    const fbf_cb_desc& d = plan->d;
    const TaftpForm none{0, false};
    const CbVariant v = cb_pick_variant(d, plan->variant, MODE_INT8, T);
    const int ksteps = (2 * d.nantennas + 31) / 32;
    if (plan->variant <= 0 && use != kTaftpBatch && (long long)d.nchans * T <= kTaftpSmall) {
        if (ksteps > 4 && d.nbeams <= 32 && use == kTaftpAlone) return none;
        const bool whole = d.fscrunch == 1 && nantennas_total == d.nantennas;
        if ((ksteps <= 3 || (ksteps == 4 && d.fscrunch > 1)) && d.nbeams <= 96 && !whole) return none;
    }
    // Above 64 antennas no other form stages TAFTP.
    if (plan->variant <= 0 && ksteps > 4 && d.fscrunch == 1 && cb_tr_applies(d, 4, MODE_INT8, T))
        return TaftpForm{4, false};
    return v.tr && !v.ws && (v.rows == 8 || v.few || (v.rows == 4 && d.fscrunch == 1)) ? TaftpForm{v.rows, v.few}
                                                                                        : none;
}

// Whether the block's geometry lets cb_tr_k stage it: a heap of a power-of-two
// number of samples, at least one tile (16 samples; two where other heaps were
// refused by the split-transpose), a heap group's bytes within a 31-bit offset
// and 32-bit tile offsets.
static bool cb_taftp_stages(const fbf_cb_plan* plan, long long T, int nantennas_total, int S)
{
    const fbf_cb_desc& d = plan->d;
    const bool one_tile = d.nantennas % 8 == 0 && d.nantennas <= 64 && d.fscrunch == 1 &&
                          (plan->variant > 0 || d.nantennas > 48);
    return S >= (one_tile ? 16 : 32) && (S & (S - 1)) == 0 && (long long)4 * nantennas_total * d.nchans * S < (1ll << 31) &&
           (long long)4 * nantennas_total * d.nchans * T < (1ll << 32);
}

// Whether fbf_cb_beamform_taftp stages the TAFTP block itself.
static bool cb_taftp_direct(const fbf_cb_plan* plan, long long T, int nantennas_total, int S)
{
    return cb_taftp_form(plan, T, nantennas_total, kTaftpAlone).rt > 0 && cb_taftp_stages(plan, T, nantennas_total, S);
}

// The form in which a call on the block stages it (rt 0: split-transposed).  A
// block that would be split-transposed under capture, without the FTPA buffer
// that needs, is staged where its geometry allows it: calls of other sizes or
// of both beams, which size no FTPA buffer, may have been the plan's first.
static int cb_taftp_takes(const fbf_cb_plan* plan, long long T, int nantennas_total, int S, hipStream_t s,
                          TaftpForm* form)
{
    *form = TaftpForm{0, false};
    if (!cb_taftp_stages(plan, T, nantennas_total, S)) return FBF_OK;
    *form = cb_taftp_form(plan, T, nantennas_total, kTaftpAlone);
    if (form->rt > 0) return FBF_OK;
    bool fixed = false;
    const int st = cb_cannot_grow(plan->ftpa_bytes, (size_t)4 * plan->d.nantennas * plan->d.nchans * T, s, &fixed);
    if (st) return st;
    if (fixed) *form = cb_taftp_form(plan, T, nantennas_total, kTaftpBatch);
    return FBF_OK;
}

// The incoherent beam of the block formed in the split-transpose's pass.
struct SplitIb {
    fbf_ib_plan* plan;
    void* tf;
    size_t tf_bytes;
};

// fbf_cb_beamform_taftp, with work for the reorder's launch and, when the
// block is split-transposed (all its antennas), the incoherent beam in that
// pass.
static int cb_taftp_run(fbf_cb_plan* plan, const void* taftp, size_t taftp_bytes, int nantennas_total,
                        int start_antenna, int nsamples_per_heap, const void* fba_weights, size_t weights_bytes,
                        void* tbtf, size_t tbtf_bytes, fbf_stream_t stream, const TailJobs& tail,
                        const SplitIb* split_ib)
{
    FBF_REQUIRE(plan, FBF_ERR_ARG, "fbf_cb_beamform_taftp: null plan");
    FBF_REQUIRE(taftp && fba_weights && tbtf, FBF_ERR_ARG, "fbf_cb_beamform_taftp: null buffer");
    const fbf_cb_desc& d = plan->d;
    FBF_REQUIRE(nantennas_total > 0 && start_antenna >= 0 && start_antenna + d.nantennas <= nantennas_total,
                FBF_ERR_ARG, "fbf_cb_beamform_taftp: the plan's antennas lie outside the block's");
    FBF_REQUIRE(nsamples_per_heap > 0, FBF_ERR_ARG, "fbf_cb_beamform_taftp: nsamples_per_heap must be positive");
    const size_t hg_bytes = (size_t)4 * nantennas_total * d.nchans * nsamples_per_heap;
    FBF_REQUIRE(taftp_bytes % hg_bytes == 0, FBF_ERR_SIZE,
                "fbf_cb_beamform_taftp: input is not a whole number of heap groups");
    const long long T = (long long)(taftp_bytes / hg_bytes) * nsamples_per_heap;
    FBF_REQUIRE((reinterpret_cast<uintptr_t>(taftp) & 15) == 0, FBF_ERR_ARG,
                "fbf_cb_beamform_taftp: buffers must be 16-byte aligned");
    TaftpForm form{0, false};
    int st = cb_taftp_takes(plan, T, nantennas_total, nsamples_per_heap, static_cast<hipStream_t>(stream), &form);
    if (st) return st;
    if (T == 0 || form.rt > 0) {
        const TaftpView tv{nsamples_per_heap, nantennas_total, start_antenna, form, nullptr};
        return cb_launch(plan, MODE_INT8, taftp, T, 2 * d.nantennas, 0, fba_weights, weights_bytes, tbtf,
                         tbtf_bytes, stream, nullptr, 0, T ? &tv : nullptr, tail);
    }
    // Otherwise the plan's antennas are split-transposed into the plan's FTPA
    // buffer for the FTPA kernels.  Sizes are checked before any launch.
    const size_t fbytes = (size_t)4 * d.nantennas * d.nchans * T;
    FBF_REQUIRE(weights_bytes == (size_t)2 * d.nchans * d.nbeams * d.nantennas, FBF_ERR_SIZE,
                "fbf_cb_beamform_taftp: weights size " + std::to_string(weights_bytes) + " != expected " +
                    std::to_string((size_t)2 * d.nchans * d.nbeams * d.nantennas));
    size_t expect = 0;
    st = fbf_cb_output_bytes(plan, fbytes, &expect);
    if (st) return st;
    FBF_REQUIRE(tbtf_bytes == expect && (T / d.tscrunch) % plan->ohs == 0, FBF_ERR_SIZE,
                "fbf_cb_beamform_taftp: output size " + std::to_string(tbtf_bytes) + " != expected " +
                    std::to_string(expect) + ", or not whole output heaps");
    void* ftpa = nullptr;
    st = cb_grow(&plan->ftpa, &plan->ftpa_bytes, fbytes, static_cast<hipStream_t>(stream), &ftpa);
    if (st) return st;
    st = split_ib ? split_transpose_ib_read_next(taftp, taftp_bytes, ftpa, fbytes, d.nchans, nsamples_per_heap,
                                                 split_ib->plan, split_ib->tf, split_ib->tf_bytes, stream)
                  : split_transpose_read_next(taftp, taftp_bytes, ftpa, fbytes, nantennas_total, d.nantennas,
                                              start_antenna, d.nchans, nsamples_per_heap, stream);
    if (st) return st;
    return cb_launch(plan, MODE_INT8, ftpa, T, 2 * d.nantennas, 0, fba_weights, weights_bytes, tbtf, tbtf_bytes,
                     stream, nullptr, 0, nullptr, tail);
}

extern "C" int fbf_cb_beamform_taftp(fbf_cb_plan* plan, const void* taftp, size_t taftp_bytes, int nantennas_total,
                                     int start_antenna, int nsamples_per_heap, const void* fba_weights,
                                     size_t weights_bytes, void* tbtf, size_t tbtf_bytes, fbf_stream_t stream)
{
    return cb_taftp_run(plan, taftp, taftp_bytes, nantennas_total, start_antenna, nsamples_per_heap, fba_weights,
                        weights_bytes, tbtf, tbtf_bytes, stream, TailJobs{}, nullptr);
}

// Whether fbf_cb_ib_beamform_taftp forms the incoherent beam inside the
// coherent beamformer: the block staged by four-wave work-groups (every
// automatic form at fscrunch 1; 128 beams per wave, or 64 above 64 antennas),
// and an incoherent-beam plan of the same block (antennas, channels, heap
// size).  In a small block (kTaftpSmall) of up to 48 antennas and 96 beams an
// incoherent beam of several channels keeps its own pass, as fbf_cb_ib_fused
// has always answered.
static bool cb_ib_fused(const fbf_cb_plan* plan, const IbFuseParams& ibp, long long T, int S)
{
    const fbf_cb_desc& d = plan->d;
    const TaftpForm form = cb_taftp_form(plan, T, d.nantennas, kTaftpOnePass);
    const int ksteps = (2 * d.nantennas + 31) / 32;
    if (form.rt == 0 || d.fscrunch != 1 || !(form.few || tr_four_waves(form.rt, ksteps))) return false;
    if ((long long)d.nchans * T <= kTaftpSmall && ksteps <= 3 && d.nbeams <= 96 && ibp.fscrunch > 1 &&
        plan->variant <= 0)
        return false;
    return cb_taftp_stages(plan, T, d.nantennas, S) && ibp.nantennas == d.nantennas && ibp.nchans == d.nchans &&
           ibp.nsamples_per_heap == S;
}

// Both beams of a TAFTP block in one pass, or where the plans do not allow it
// the incoherent beam in the split-transpose's pass or on its own; `next` (a
// fbf_weights_generate call) runs in the reorder's launch.
struct NextWeights {
    fbf_weights_plan* plan;
    const void* delays;
    size_t delays_bytes;
    double epoch;
    void* weights;
    size_t weights_bytes;
};

static int cb_ib_run(fbf_cb_plan* plan, fbf_ib_plan* ib_plan, const void* taftp, size_t taftp_bytes,
                     int nsamples_per_heap, const void* fba_weights, size_t weights_bytes, void* tbtf,
                     size_t tbtf_bytes, void* tf, size_t tf_bytes, fbf_stream_t stream, const NextWeights* next)
{
    FBF_REQUIRE(plan && ib_plan, FBF_ERR_ARG, "fbf_cb_ib_beamform_taftp: null plan");
    FBF_REQUIRE(taftp && fba_weights && tbtf && tf, FBF_ERR_ARG, "fbf_cb_ib_beamform_taftp: null buffer");
    IbFuseParams ibp;
    int st = ib_fuse_params(ib_plan, &ibp);
    if (st) return st;
    const fbf_cb_desc& d = plan->d;
    FBF_REQUIRE(nsamples_per_heap > 0, FBF_ERR_ARG, "fbf_cb_ib_beamform_taftp: nsamples_per_heap must be positive");
    const size_t hg_bytes = (size_t)4 * d.nantennas * d.nchans * nsamples_per_heap;
    FBF_REQUIRE(taftp_bytes % hg_bytes == 0, FBF_ERR_SIZE,
                "fbf_cb_ib_beamform_taftp: input is not a whole number of heap groups of the plan's antennas");
    const long long T = (long long)(taftp_bytes / hg_bytes) * nsamples_per_heap;
    WeightsJob wj{};
    if (next) {
        // Checked before anything is launched.
        st = weights_launch_params(next->plan, next->delays, next->delays_bytes, next->epoch, next->weights,
                                   next->weights_bytes, &wj.w);
        if (st) return st;
        FBF_REQUIRE(next->weights_bytes == weights_bytes, FBF_ERR_SIZE,
                    "fbf_cb_ib_beamform_taftp_next: the next weights differ in size from the block's");
        FBF_REQUIRE(wj.w.F == d.nchans && (long long)wj.w.nd == (long long)d.nantennas * d.nbeams, FBF_ERR_ARG,
                    "fbf_cb_ib_beamform_taftp_next: the weights plan's geometry differs from the coherent plan's");
        FBF_REQUIRE((unsigned long long)wj.w.gx * wj.w.gy < (1ull << 30), FBF_ERR_UNSUPPORTED,
                    "fbf_cb_ib_beamform_taftp_next: too many weights work-groups");
        wj.nblocks = (int)(wj.w.gx * wj.w.gy);
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    bool fused = T > 0 && cb_ib_fused(plan, ibp, T, nsamples_per_heap);
    const size_t part_bytes = (size_t)d.nchans * T * 4 * sizeof(int);
    if (fused) {
        // Under capture without the partials' buffer (the coherent beams alone
        // were the plan's first call, say) the incoherent beam runs on its own.
        bool fixed = false;
        st = cb_cannot_grow(plan->ibp_bytes, part_bytes, s, &fixed);
        if (st) return st;
        fused = !fixed;
    }
    if (!fused) {
        // The incoherent beam comes out of the split-transpose's pass where
        // there is one and the plan's scrunch allows it (one read of the
        // block and one launch less: a block of 16 antennas, 16 channels,
        // 2048 spectra and 32 beams, which is launches and latency, took
        // 21.4 us in five launches and takes 17.2 us in three); else it runs
        // first.
        TaftpForm form{0, false};
        st = cb_taftp_takes(plan, T, d.nantennas, nsamples_per_heap, s, &form);
        if (st) return st;
        const bool split_ib = T > 0 && form.rt == 0 && ibp.nantennas == d.nantennas && ibp.nchans == d.nchans &&
                              ibp.nsamples_per_heap == nsamples_per_heap && split_ib_applies(ibp);
        if (split_ib) {
            size_t tf_expect = 0;
            st = fbf_ib_output_bytes(ib_plan, taftp_bytes, &tf_expect);
            if (st) return st;
            FBF_REQUIRE(tf_bytes == tf_expect, FBF_ERR_SIZE,
                        "fbf_cb_ib_beamform_taftp: incoherent-beam output size " + std::to_string(tf_bytes) +
                            " != expected " + std::to_string(tf_expect));
        } else {
            st = fbf_ib_beamform(ib_plan, taftp, taftp_bytes, tf, tf_bytes, stream);
            if (st) return st;
        }
        const SplitIb sib{ib_plan, tf, tf_bytes};
        st = cb_taftp_run(plan, taftp, taftp_bytes, d.nantennas, 0, nsamples_per_heap, fba_weights, weights_bytes,
                          tbtf, tbtf_bytes, stream, TailJobs{IbFinishJob{}, wj, nullptr}, split_ib ? &sib : nullptr);
        if (st || !next || T > 0) return st;
        return fbf_weights_generate(next->plan, next->delays, next->delays_bytes, next->epoch, next->weights,
                                    next->weights_bytes, nullptr, stream);
    }
    size_t tf_expect = 0;
    st = fbf_ib_output_bytes(ib_plan, taftp_bytes, &tf_expect);
    if (st) return st;
    FBF_REQUIRE(tf_bytes == tf_expect, FBF_ERR_SIZE,
                "fbf_cb_ib_beamform_taftp: incoherent-beam output size " + std::to_string(tf_bytes) +
                    " != expected " + std::to_string(tf_expect));
    FBF_REQUIRE((reinterpret_cast<uintptr_t>(taftp) & 15) == 0, FBF_ERR_ARG,
                "fbf_cb_ib_beamform_taftp: buffers must be 16-byte aligned");
    void* part = nullptr;
    st = cb_grow(&plan->ibp, &plan->ibp_bytes, part_bytes, s, &part);
    if (st) return st;
    IbFinishJob ibj{};
    st = ib_finish_job(ib_plan, static_cast<const int*>(part), 1, T, tf, tf_bytes, &ibj);
    if (st) return st;
    const TaftpView tv{nsamples_per_heap, d.nantennas, 0, cb_taftp_form(plan, T, d.nantennas, kTaftpOnePass),
                       static_cast<int*>(part)};
    return cb_launch(plan, MODE_INT8, taftp, T, 2 * d.nantennas, 0, fba_weights, weights_bytes, tbtf, tbtf_bytes,
                     stream, nullptr, 0, &tv, TailJobs{ibj, wj, nullptr});
}

std::pair<int, int> fbf::cb_plan_tuning(const fbf_cb_plan* plan) { return {plan->variant, plan->chunk}; }

bool fbf::cb_batch_stages(const fbf_cb_plan* plan, long long T, int nantennas_total, int S, bool partials)
{
    const fbf_cb_desc& d = plan->d;
    const TaftpForm form = cb_taftp_form(plan, T, nantennas_total, kTaftpBatch);
    if (form.rt == 0 || T % d.tscrunch != 0 || !cb_taftp_stages(plan, T, nantennas_total, S)) return false;
    return !partials || (d.fscrunch == 1 && (form.few || tr_four_waves(form.rt, (2 * d.nantennas + 31) / 32)));
}

int fbf::cb_batch_beamform(fbf_cb_plan* plan, const void* taftp, long long T, int nantennas_total, int start_antenna,
                           int S, const void* fba_weights, size_t weights_bytes, void* tbtf, size_t tbtf_bytes,
                           hipStream_t s, int* partials, TbtfArgs* reorder)
{
    *reorder = TbtfArgs{};
    const TaftpView tv{S, nantennas_total, start_antenna, cb_taftp_form(plan, T, nantennas_total, kTaftpBatch),
                       partials};
    return cb_launch(plan, MODE_INT8, taftp, T, 2 * plan->d.nantennas, 0, fba_weights, weights_bytes, tbtf,
                     tbtf_bytes, s, nullptr, 0, &tv, TailJobs{IbFinishJob{}, WeightsJob{}, reorder});
}

int fbf::cb_batch_reorder(const TbtfArgs* reorders, int n, const IbFinishJob& ib, hipStream_t s)
{
    TbtfJobs jobs{};
    IbFinishJob job = ib;   // (in the first launch)
    long long nblocks = 0;
    size_t shm = 0;
    auto flush = [&]() {
        const long long all = nblocks + job.nblocks;
        if (all == 0) return hipSuccess;
        if (all >= (1ll << 31)) return hipErrorInvalidConfiguration;
        tbtf_jobs_k<<<dim3((unsigned)all), 256, shm, s>>>(jobs, job);
        jobs = TbtfJobs{};
        job = IbFinishJob{};
        nblocks = 0;
        shm = 0;
        return hipGetLastError();
    };
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess; ++i) {
        const TbtfArgs& a = reorders[i];
        if (!a.src) continue;   // (written by the coherent kernel itself)
        const long long nb = tbtf_blocks(a);
        if (jobs.n == kTbtfJobs || nblocks + nb + job.nblocks >= (1ll << 31)) e = flush();
        jobs.a[jobs.n] = a;
        jobs.first[jobs.n++] = (int)nblocks;
        nblocks += nb;
        shm = std::max(shm, (size_t)a.tt * a.tp * 4);
    }
    if (e == hipSuccess) e = flush();
    return e == hipSuccess ? FBF_OK : hip_status(e, "tbtf_jobs_k launch");
}

extern "C" int fbf_cb_ib_beamform_taftp(fbf_cb_plan* plan, fbf_ib_plan* ib_plan, const void* taftp,
                                        size_t taftp_bytes, int nsamples_per_heap, const void* fba_weights,
                                        size_t weights_bytes, void* tbtf, size_t tbtf_bytes, void* tf,
                                        size_t tf_bytes, fbf_stream_t stream)
{
    return cb_ib_run(plan, ib_plan, taftp, taftp_bytes, nsamples_per_heap, fba_weights, weights_bytes, tbtf,
                     tbtf_bytes, tf, tf_bytes, stream, nullptr);
}

extern "C" int fbf_cb_ib_beamform_taftp_next(fbf_cb_plan* plan, fbf_ib_plan* ib_plan, const void* taftp,
                                             size_t taftp_bytes, int nsamples_per_heap, const void* fba_weights,
                                             size_t weights_bytes, void* tbtf, size_t tbtf_bytes, void* tf,
                                             size_t tf_bytes, fbf_weights_plan* weights_plan, const void* delays,
                                             size_t delays_bytes, double next_epoch, void* next_weights,
                                             size_t next_weights_bytes, fbf_stream_t stream)
{
    const NextWeights next{weights_plan, delays, delays_bytes, next_epoch, next_weights, next_weights_bytes};
    return cb_ib_run(plan, ib_plan, taftp, taftp_bytes, nsamples_per_heap, fba_weights, weights_bytes, tbtf,
                     tbtf_bytes, tf, tf_bytes, stream, &next);
}

extern "C" int fbf_cb_ib_fused(const fbf_cb_plan* plan, const fbf_ib_plan* ib_plan, int nsamples_per_heap,
                               long long nsamples, int* fused)
{
    FBF_REQUIRE(plan && ib_plan && fused, FBF_ERR_ARG, "fbf_cb_ib_fused: null argument");
    IbFuseParams ibp;
    const int st = ib_fuse_params(ib_plan, &ibp);
    if (st) return st;
    *fused = nsamples > 0 && nsamples % plan->d.tscrunch == 0 && cb_ib_fused(plan, ibp, nsamples, nsamples_per_heap);
    return FBF_OK;
}

extern "C" int fbf_cb_taftp_direct(const fbf_cb_plan* plan, int nantennas_total, int nsamples_per_heap,
                                   long long nsamples, int* direct)
{
    FBF_REQUIRE(plan && direct, FBF_ERR_ARG, "fbf_cb_taftp_direct: null argument");
    *direct = nsamples > 0 && nsamples % plan->d.tscrunch == 0 &&
              cb_taftp_direct(plan, nsamples, nantennas_total, nsamples_per_heap);
    return FBF_OK;
}

extern "C" int fbf_cb_plan_set_timing(fbf_cb_plan* plan, fbf_event_t before, fbf_event_t after)
{
    FBF_REQUIRE(plan, FBF_ERR_ARG, "fbf_cb_plan_set_timing: null plan");
    FBF_REQUIRE((before == nullptr) == (after == nullptr), FBF_ERR_ARG,
                "fbf_cb_plan_set_timing: give both events or neither");
    plan->t_before = static_cast<hipEvent_t>(before);
    plan->t_after = static_cast<hipEvent_t>(after);
    return FBF_OK;
}

extern "C" int fbf_cb_plan_set_chunk(fbf_cb_plan* plan, int chunk)
{
    FBF_REQUIRE(plan && chunk >= 0 && chunk <= 16 && (chunk & (chunk - 1)) == 0, FBF_ERR_ARG,
                "fbf_cb_plan_set_chunk: chunk must be 0 (auto) or a power of two <= 16");
    plan->chunk = chunk;
    return FBF_OK;
}

extern "C" int fbf_cb_beamform(fbf_cb_plan* plan, const void* ftpa, size_t ftpa_bytes, const void* fba_weights,
                               size_t weights_bytes, void* tbtf, size_t tbtf_bytes, fbf_stream_t stream)
{
    return cb_run(plan, MODE_INT8, ftpa, ftpa_bytes, fba_weights, weights_bytes, tbtf, tbtf_bytes, stream);
}

extern "C" int fbf_cb_beamform_ws(fbf_cb_plan* plan, const void* ftpa, size_t ftpa_bytes, const void* fba_weights,
                                  size_t weights_bytes, void* tbtf, size_t tbtf_bytes, void* workspace,
                                  size_t workspace_bytes, fbf_stream_t stream)
{
    FBF_REQUIRE(plan, FBF_ERR_ARG, "fbf_cb: null plan");
    FBF_REQUIRE(workspace, FBF_ERR_ARG, "fbf_cb_beamform_ws: null workspace");
    long long T = 0;
    int st = cb_nsamples(plan, ftpa_bytes, &T);
    if (st) return st;
    return cb_launch(plan, MODE_INT8, ftpa, T, 2 * plan->d.nantennas, 0, fba_weights, weights_bytes, tbtf,
                     tbtf_bytes, stream, workspace, workspace_bytes);
}

extern "C" int fbf_cb_plan_reserve(fbf_cb_plan* plan, long long nsamples)
{
    FBF_REQUIRE(plan && nsamples >= 0, FBF_ERR_ARG, "fbf_cb_plan_reserve: bad argument");
    FBF_REQUIRE(nsamples % plan->d.tscrunch == 0, FBF_ERR_SIZE, "fbf_cb_plan_reserve: nsamples % tscrunch != 0");
    const size_t bytes = (size_t)(nsamples / plan->d.tscrunch) * plan->d.nbeams * (plan->d.nchans / plan->d.fscrunch);
    if (bytes == 0) return FBF_OK;
    void* p = nullptr;
    const int st = cb_staging(plan, bytes, nullptr, &p);
    if (st) return st;
    // The incoherent-beam partials of fbf_cb_ib_beamform_taftp (16 bytes per
    // channel and sample).
    return cb_grow(&plan->ibp, &plan->ibp_bytes, (size_t)plan->d.nchans * nsamples * 4 * sizeof(int), nullptr, &p);
}

extern "C" int fbf_cb_beam_sums(fbf_cb_plan* plan, const void* ftpa, size_t ftpa_bytes, const void* fba_weights,
                                size_t weights_bytes, int32_t* sums, size_t sums_bytes, fbf_stream_t stream)
{
    return cb_run(plan, MODE_SUMS, ftpa, ftpa_bytes, fba_weights, weights_bytes, sums, sums_bytes, stream);
}

extern "C" int fbf_cb_beam_power(fbf_cb_plan* plan, const void* ftpa, size_t ftpa_bytes, const void* fba_weights,
                                 size_t weights_bytes, double* power, size_t power_bytes, fbf_stream_t stream)
{
    return cb_run(plan, MODE_POWER, ftpa, ftpa_bytes, fba_weights, weights_bytes, power, power_bytes, stream);
}

// ---------------------------------------------------------------------------
// Autotuner: times every (variant, chunk) candidate on synthetic data of the
// plan's geometry.  The voltage values do not change the instruction stream,
// so constant bytes are enough for timing.
// ---------------------------------------------------------------------------
extern "C" int fbf_cb_autotune(fbf_cb_plan* plan, long long nsamples, int reps, int* best_variant, int* best_chunk,
                               float* best_ms)
{
    FBF_REQUIRE(plan && nsamples > 0 && reps > 0, FBF_ERR_ARG, "fbf_cb_autotune: bad argument");
    const fbf_cb_desc& d = plan->d;
    FBF_REQUIRE(nsamples % d.tscrunch == 0 && (nsamples / d.tscrunch) % plan->ohs == 0, FBF_ERR_ARG,
                "fbf_cb_autotune: nsamples must fill whole output heaps");
    const size_t vbytes = (size_t)nsamples * 2 * 2 * d.nantennas * d.nchans;
    const size_t wbytes = (size_t)2 * d.nchans * d.nbeams * d.nantennas;
    const size_t obytes = (size_t)(nsamples / d.tscrunch) * d.nbeams * (d.nchans / d.fscrunch);
    void *v = nullptr, *w = nullptr, *o = nullptr;
    hipStream_t s = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto cleanup = [&]() {
        if (v) (void)hipFree(v);
        if (w) (void)hipFree(w);
        if (o) (void)hipFree(o);
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        if (s) (void)hipStreamDestroy(s);
    };
    hipError_t e = hipMalloc(&v, vbytes);
    if (e == hipSuccess) e = hipMalloc(&w, wbytes);
    if (e == hipSuccess) e = hipMalloc(&o, obytes);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    if (e == hipSuccess) e = hipMemsetAsync(v, 0x11, vbytes, s);
    if (e == hipSuccess) e = hipMemsetAsync(w, 0x5A, wbytes, s);
    if (e != hipSuccess) {
        cleanup();
        return hip_status(e, "fbf_cb_autotune setup");
    }
    const int nvar = (int)(sizeof(kCbVariants) / sizeof(kCbVariants[0]));
    const bool al16 = d.nantennas % 8 == 0;
    const int jc_max = cb_lds_chunk(2 * d.tscrunch, 2 * d.nantennas, al16);
    const int saved_variant = plan->variant, saved_chunk = plan->chunk;
    int bv = saved_variant, bc = saved_chunk;
    float bms = 1e30f;
    float auto_ms = 1e30f;   // the automatic pick (variant 0)
    for (int var = 0; var < nvar; ++var) {
        std::vector<int> chunks{0};
        if (kCbVariants[var].lds && !kCbVariants[var].tr)
            for (int jc = jc_max / 2; jc >= 1; jc >>= 1) chunks.push_back(jc);
        for (int jc : chunks) {
            plan->variant = var;
            plan->chunk = jc;
            int st = cb_launch(plan, MODE_INT8, v, nsamples, 2 * d.nantennas, 0, w, wbytes, o, obytes, s);
            if (st != FBF_OK) continue;   // candidate not applicable to this geometry
            (void)hipEventRecord(e0, s);
            for (int r = 0; r < reps; ++r)
                cb_launch(plan, MODE_INT8, v, nsamples, 2 * d.nantennas, 0, w, wbytes, o, obytes, s);
            (void)hipEventRecord(e1, s);
            e = hipEventSynchronize(e1);
            if (e != hipSuccess) {
                plan->variant = saved_variant;
                plan->chunk = saved_chunk;
                cleanup();
                return hip_status(e, "fbf_cb_autotune timing");
            }
            float ms = 0.0f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            ms /= (float)reps;
            if (var == 0) {
                auto_ms = ms;
            } else if (ms < bms) {
                bms = ms;
                bv = var;
                bc = jc;
            }
        }
    }
    // The automatic pick stays unless a variant beats it: it may be a form that
    // no variant names (few beams), and leaves fbf_cb_beamform_taftp its own
    // choice.  It is reported as the variant of its kernel.
    const bool keep_auto = auto_ms <= 1.01f * bms;
    if (keep_auto) {
        const CbVariant v = cb_pick_ftpa(d, 0, MODE_INT8, nsamples);
        bv = !v.tr ? kCbVariantLds : v.rows == 2 ? kCbVariantTr2 : v.rows == 4 ? kCbVariantTr4 : kCbVariantTr8;
        bc = 0;
        bms = auto_ms;
    }
    plan->variant = keep_auto ? 0 : bv;
    plan->chunk = bc;
    {
        std::lock_guard<std::mutex> lock(g_tune_mutex);
        g_tune_table[tune_key(d)] = {plan->variant, bc};
    }
    cleanup();
    if (best_variant) *best_variant = bv;
    if (best_chunk) *best_chunk = bc;
    if (best_ms) *best_ms = bms;
    return FBF_OK;
}
