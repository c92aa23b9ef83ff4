// Internal helpers shared by the HIP kernels and the C ABI implementation.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <string>
#include <utility>

#include "../../include/fbfuse_hip.h"

namespace fbf {

// Records `msg` as the calling thread's last error and returns `code`.
int set_error(int code, const std::string& msg);
void clear_error();

// Returns FBF_ERR_HIP (and records the HIP error string) when `e` failed.
int hip_status(hipError_t e, const char* what);

}  // namespace fbf

#define FBF_HIP_TRY(expr)                                              \
    do {                                                               \
        hipError_t fbf_e_ = (expr);                                    \
        if (fbf_e_ != hipSuccess) return ::fbf::hip_status(fbf_e_, #expr); \
    } while (0)

#define FBF_REQUIRE(cond, code, msg)                                   \
    do {                                                               \
        if (!(cond)) return ::fbf::set_error((code), (msg));           \
    } while (0)

// Per-launch check: hipGetLastError after a kernel launch.
#define FBF_LAUNCH_CHECK(name)                                         \
    do {                                                               \
        hipError_t fbf_e_ = hipGetLastError();                         \
        if (fbf_e_ != hipSuccess) return ::fbf::hip_status(fbf_e_, name); \
    } while (0)

namespace fbf {

// What the fused split-transpose + incoherent-beam path needs from an
// incoherent-beam plan (incoherent_beamformer.hip).
struct IbFuseParams {
    const float* offsets;   // device, [nchans / fscrunch]
    const float* scales;
    int nantennas, nchans, nsamples_per_heap, tscrunch, fscrunch, quant;
};
int ib_fuse_params(const fbf_ib_plan* plan, IbFuseParams* out);

// Whether the split-transpose can form this incoherent beam in its pass: one
// channel to an output channel, whole windows in its 32-sample tiles.
inline bool split_ib_applies(const IbFuseParams& p)
{
    return p.fscrunch == 1 && p.tscrunch > 0 && 32 % p.tscrunch == 0 && p.nsamples_per_heap % 32 == 0;
}
// fbf_split_transpose and fbf_split_transpose_ib of a copy that the coherent
// beamformer reads in the next launch (st_near).
int split_transpose_read_next(const void* taftp, size_t taftp_bytes, void* ftpa, size_t ftpa_bytes,
                              int total_nantennas, int used_nantennas, int start_antenna, int nchans,
                              int nsamples_per_heap, fbf_stream_t stream);
int split_transpose_ib_read_next(const void* taftp, size_t taftp_bytes, void* ftpa, size_t ftpa_bytes, int nchans,
                                 int nsamples_per_heap, fbf_ib_plan* ib_plan, void* tf, size_t tf_bytes,
                                 fbf_stream_t stream);

// The incoherent beam from the partials that the coherent beamformer left
// ([F][T / 16][2 halves][32 columns] int32; sample j of a tile is the sum of
// columns 2j, 2j + 1 of both halves), int8 TF of T samples with the IB
// plan's scrunch and quantiser, as a job for nblocks work-groups of 256
// threads of another launch (ib_finish_run).  nparts partials one after the
// other (the subarrays that share the block's antennas out) are added up.
struct IbFinishJob {
    const int* part;
    int8_t* out;
    const float* offsets;
    const float* scales;
    long long nwin;   // output windows (T / tscrunch)
    int ntiles, Fo, ts, fs, quant;
    int nparts;
    int nblocks;      // 0: none
};
int ib_finish_job(const fbf_ib_plan* plan, const int* partials, int nparts, long long T, void* tf, size_t tf_bytes,
                  IbFinishJob* out);

// A coherent plan's kernel variant and chunk length.
std::pair<int, int> cb_plan_tuning(const fbf_cb_plan* plan);

// One reorder of staged beams to TBTF (tbtf_k).
struct TbtfArgs {
    const int8_t* src;
    int8_t* dst;
    long long To;
    int B, Fo, ohs;
    int tt, ft, bp, tp;           // tile samples / channels, LDS pitches (dwords)
    int n_ttiles, n_ftiles, n_btiles;
};

// A batch's subarray beamformed from the TAFTP block itself: whether the
// plan's kernel stages such a block (with `partials`: and leaves the
// incoherent beam's partials of its antennas); the call, which leaves its
// reorder in *reorder (src null: none is needed); and the reorders of the
// batch's subarrays with the incoherent beam's finish.
bool cb_batch_stages(const fbf_cb_plan* plan, long long T, int nantennas_total, int S, bool partials);
int cb_batch_beamform(fbf_cb_plan* plan, const void* taftp, long long T, int nantennas_total, int start_antenna,
                      int S, const void* fba_weights, size_t weights_bytes, void* tbtf, size_t tbtf_bytes,
                      hipStream_t s, int* partials, TbtfArgs* reorder);
int cb_batch_reorder(const TbtfArgs* reorders, int n, const IbFinishJob& ib, hipStream_t s);

// Weights generation (weights.hip), shared by weights_k and by launches that
// generate the weights beside other work.  A thread takes one (beam,
// antenna) di over the run of kWChans channels starting at f0.
constexpr int kWChans = 8;

struct WeightsLaunch {
    const float2* delays;   // [B][A] (rate, offset)
    const double* freqs;    // device, [F]
    double epoch;
    int F, nd;              // channels; beams x antennas
    char2* weights;         // [F][B][A]
    unsigned gx, gy;        // work-groups over (beam, antenna) pairs and channel runs
};
// Checks a generate call's arguments against its plan and fills the launch.
int weights_launch_params(const fbf_weights_plan* plan, const void* delays, size_t delays_bytes, double epoch,
                          void* weights, size_t weights_bytes, WeightsLaunch* out);

// phase = (rate * t + offset) * f in FP64 (contraction off, the oracle's
// order), the whole-cycle part removed, then 127 times the FP32 cosine and sine
// of the reduced phase, rounded to the nearest integer, ties to even: the bytes
// that sincospif gives.
//
// The generator was bound by VALU issue, two thirds of it sincospif.  The
// hardware's v_sin_f32 / v_cos_f32 take a phase in cycles, and over every
// float in [-1/2, 1/2] 127 times either is within 1.9e-5 of 127 times
// sincospif's value (all 2 * 0x3f000001 of them compared on gfx950).  So where
// neither component lies within kWAmbig (five times that) of a half-integer
// the rounded weight is sincospif's, bit for bit; the other lanes (one in
// 2500, and any NaN) call sincospif.
// The channel frequencies are read through the constant address space
// (scalar loads): as vector loads each waited for the previous channel's
// store as well.
// 64 antennas, 1024 beams, 64 channels: 7.7 us a call with sincospif alone, 5.4 us now.
constexpr float kWAmbig = 1e-4f;

__device__ __forceinline__ void weights_run(const WeightsLaunch& w, float* phase_out, int di, int f0)
{
#pragma clang fp contract(off)
    const float2 d = w.delays[di];
    double tau = (double)d.x * w.epoch;
    tau = tau + (double)d.y;
    const int f1 = f0 + kWChans < w.F ? f0 + kWChans : w.F;
    const auto* freqs = (const __attribute__((address_space(4))) double*)w.freqs;
    for (int f = f0; f < f1; ++f) {
        const double phase = tau * freqs[f];
        const double frac = phase - rint(phase);
        const float x = (float)frac;
        float re = 127.0f * __builtin_amdgcn_cosf(x);
        float im = 127.0f * __builtin_amdgcn_sinf(x);
        const float off = fmaxf(fabsf(re - rintf(re)), fabsf(im - rintf(im)));
        if (!(off <= 0.5f - kWAmbig)) {   // (true for NaN)
            float s, c;
            sincospif(2.0f * x, &s, &c);
            re = 127.0f * c;
            im = 127.0f * s;
        }
        char2 v;
        v.x = (signed char)(int)rintf(re);
        v.y = (signed char)(int)rintf(im);
        const size_t idx = (size_t)f * w.nd + di;
        w.weights[idx] = v;
        if (phase_out) phase_out[idx] = x;
    }
}

// Weights generated by the first nblocks work-groups (of 256 threads) of
// another kernel's launch (nblocks = 0: none); the rest of the launch does
// that kernel's own work, numbered from 0 again.
struct WeightsJob {
    WeightsLaunch w;
    int nblocks;   // w.gx * w.gy
};

// Runs this work-group's share of the job and returns true when the
// work-group is one of the job's.
__device__ __forceinline__ bool weights_job_run(const WeightsJob& wj, int tid)
{
    if ((int)blockIdx.x >= wj.nblocks) return false;
    const int wb = blockIdx.x;
    const int di = (wb % (int)wj.w.gx) * 256 + tid;
    if (di < wj.w.nd) weights_run(wj.w, nullptr, di, (wb / (int)wj.w.gx) * kWChans);
    return true;
}

// Number of XCDs on MI355X; work-groups are dispatched round robin over them.
constexpr int kNumXcd = 8;

// Maps a hardware block id to a logical tile id so that logical neighbours
// (tiles that share input through L2) run on the same XCD.  Bijective on
// [0, nblocks).
__device__ __forceinline__ int xcd_remap(int bid, int nblocks)
{
    const int per = nblocks / kNumXcd;
    if (bid >= per * kNumXcd) return bid;
    return (bid % kNumXcd) * per + bid / kNumXcd;
}

// A 16-byte load of data that is read once, and the matching store.
__device__ __forceinline__ int4 load_stream(const void* p)
{
    typedef int v4 __attribute__((ext_vector_type(4)));
    const v4 v = __builtin_nontemporal_load(static_cast<const v4*>(p));
    return int4{v.x, v.y, v.z, v.w};
}

// Quantiser shared by every output path: (P - offset) / scale in IEEE double,
// round half away from zero (mode 0) or truncate (mode 1), saturate to int8.
__device__ __forceinline__ int8_t quantise(double power, float offset, float scale, int mode)
{
    double v = (power - (double)offset) / (double)scale;
    double q = mode ? trunc(v) : round(v);
    q = fmax(q, -128.0);  // fmax maps NaN to -128
    q = fmin(q, 127.0);
    return (int8_t)(int)q;
}

// One thread of an IbFinishJob (gi = work-group * 256 + thread): four lanes
// per output (window, output channel), each adding every fourth 16-byte
// piece (8-byte pair of a column pair) of the window's partials over the
// fscrunch channels in int64, then the four sums folded with two shuffles
// and quantised by the first lane.  Consecutive outputs are consecutive
// windows of one output channel, so a wave reads one contiguous run of
// partials.  Every lane of the work-group reaches the shuffles.
__device__ __forceinline__ void ib_finish_run(const IbFinishJob& j, long long gi)
{
    const long long i = gi >> 2;   // output
    const int q = (int)(gi & 3);   // lane of the output's four
    const bool valid = i < j.nwin * j.Fo;
    const int fo = valid ? (int)(i / j.nwin) : 0;
    const long long w = valid ? i - (long long)fo * j.nwin : 0;
    long long P = 0;
    if (valid) {
        const int* base = j.part;
        for (int k = 0; k < j.nparts; ++k, base += (size_t)j.Fo * j.fs * j.ntiles * 64) {
            for (int fc = 0; fc < j.fs; ++fc) {
                const int* pf = base + (size_t)(fo * j.fs + fc) * j.ntiles * 64;
                if (j.ts >= 16) {
                    // Whole tiles: the ts / 16 records, ts 16-byte pieces.
                    const int4* r = reinterpret_cast<const int4*>(pf + (size_t)(w * (j.ts / 16)) * 64);
                    for (int q4 = q; q4 < j.ts; q4 += 4) {
                        const int4 v = r[q4];
                        P += (long long)v.x + v.y + v.z + v.w;
                    }
                } else {
                    // Samples j0 .. j0 + ts - 1 of one tile: the column pairs
                    // j0 .. j0 + ts - 1 of both halves (8 bytes each).
                    const long long t0 = w * j.ts;
                    const int2* r = reinterpret_cast<const int2*>(pf + (size_t)(t0 >> 4) * 64) + (t0 & 15);
                    for (int q4 = q; q4 < 2 * j.ts; q4 += 4) {
                        const int2 v = r[(q4 & 1) * 16 + (q4 >> 1)];
                        P += (long long)v.x + v.y;
                    }
                }
            }
        }
    }
    P += __shfl_xor(P, 1, 4);
    P += __shfl_xor(P, 2, 4);
    if (valid && q == 0) j.out[w * j.Fo + fo] = quantise((double)P, j.offsets[fo], j.scales[fo], j.quant);
}

}  // namespace fbf
