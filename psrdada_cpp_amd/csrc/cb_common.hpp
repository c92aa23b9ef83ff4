// Coherent beamformer: the arguments, launchers and device helpers that its
// translation units share.  coherent_beamformer.hip has the overview and the
// C ABI.
#pragma once

#include "fbf_internal.hpp"

#include <climits>
#include <type_traits>

namespace fbf {

enum { MODE_INT8 = 0, MODE_SUMS = 1, MODE_POWER = 2 };

struct CbArgs {
    const int8_t* ftpa;
    const int8_t* fba;
    void* out;
    const float* offsets;
    const float* scales;
    const long long* thr;   // quantiser thresholds [Fo][kThr] (cb_thresholds_k)
    long long nsamples;   // T
    long long nsamples_out;
    int A, B, F, Fo, ts, fs, ohs, quant;
    int n_bchunks, n_tchunks, n_bgroups, n_tgroups, wb;
    // Voltage columns are `vstride` bytes apart and this beamformer's
    // 2*A bytes start `voff` bytes into each column (vstride = 2*A and
    // voff = 0 for a split-transposed subset; a subarray reading a full
    // FTPA block uses the block's column stride and its antenna offset).
    int vstride, voff;
    // S > 0: the voltages are instead a TAFTP block, [heap group][Atot][F][S
    // samples][2 pols] char2, and this beamformer's antennas start at its
    // antenna a0 (read so by cb_tr_k<..., TA = true> and cb_exact_outputs).
    int S, Atot, a0;
};

struct CbTrArgs {
    CbArgs p;
    int ntiles;                // 32-column tiles per channel
    int tps;                   // tiles per window (W >= 32), else 1
    int npasses;               // passes per work-group
    int ntp;                   // tiles per pass
    int n_bgroups, n_tgroups;
    // TAFTP staging: bytes per heap group of the block, log2 of the tiles
    // (16 samples) per heap.
    size_t hstride;
    int lgtph;
    // Incoherent-beam partials (cb_tr_k with IBF): [F][ntiles][2 halves][32
    // columns] int32; sample j of a tile has the power over the block's
    // antennas and both pols split over columns 2j, 2j + 1 (its pols) of
    // both halves (ib_finish_run adds the four).
    int* ibp;
    // The few-beam forms for a small block (cb_tbtf_direct): the outputs go
    // straight to TBTF at `tbtf` (else null), the incoherent beam of `ib`
    // (ib.out null: none, or partials) to its output, and the first
    // weights.nblocks work-groups generate weights.
    int8_t* tbtf;
    IbFinishJob ib;
    WeightsJob weights;
};

struct CbWsArgs {
    CbArgs p;
    int ntiles;      // 32-column tiles per channel
    int tps;         // tiles per window (W >= 32), else 1
    int ntp;         // tiles per pass
    int ct;          // tiles per chunk: a whole number of passes, >= NB
    int nbg;         // 64-beam groups
    int ntr;         // time ranges per (channel, beam group)
    int tr_chunks;   // chunks per time range
    int nunits;      // Fo * nbg * ntr
    int U;           // units per work-group
};

// The kernels' launchers, one translation unit each (the template instances
// compile side by side): cb_tr2, cb_tr4, cb_tr8, cb_tr8_fs, cb_tr_few, cb_ws and cb_lds.
hipError_t cb_launch_tr2(const CbTrArgs& a, int fs, int W, int ksteps, int passes, hipStream_t s);
hipError_t cb_launch_tr4(const CbTrArgs& a, int fs, int W, int ksteps, int passes, hipStream_t s);
hipError_t cb_launch_tr8(const CbTrArgs& a, int W, int ksteps, int passes, hipStream_t s);
hipError_t cb_launch_tr8_fs(const CbTrArgs& a, int fs, int W, int ksteps, int passes, hipStream_t s);
hipError_t cb_launch_tr_few(const CbTrArgs& a, int rt, int W, int ksteps, int passes, hipStream_t s);
hipError_t cb_launch_ws(const CbWsArgs& a, int W, int ksteps, hipStream_t s);
hipError_t cb_launch_lds(const CbArgs& a, int mode, int rt, int ksteps, int jc, dim3 grid, hipStream_t s);
hipError_t cb_launch_mfma32(const CbArgs& a, int mode, int rt, int ksteps, dim3 grid, hipStream_t s);
hipError_t cb_launch_mfma16(const CbArgs& a, int mode, int rowt, int ksteps, dim3 grid, hipStream_t s);

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// Two adjacent beams' int8 outputs as one 16-bit store (b is even, B % 8 == 0).
__device__ __forceinline__ void store_pair(int8_t* dst, int8_t a, int8_t b)
{
    *reinterpret_cast<uint16_t*>(dst) = (uint16_t)((uint8_t)a | ((uint16_t)(uint8_t)b << 8));
}


// Loads of one 16-byte K slice [k0, k0 + 16) of a column of K bytes.  They
// are unconditional and branch-free (divergent branches around loads force
// the compiler to wait for every load in flight): addresses are clamped
// inside the column instead.  K is a multiple of 8; AL16 means K % 16 == 0.
//
// Voltage slices: bytes at k >= K may hold anything, because the weights
// there are zero.  A slice past the column end re-reads the column start; the
// upper half of a slice straddling K (K % 16 == 8) re-reads its lower half.
template <bool AL16>
__device__ __forceinline__ v4i load_vslice(const int8_t* col, int k0, int K)
{
    if (AL16) {
        const int kk = k0 < K ? k0 : 0;
        return *reinterpret_cast<const v4i*>(col + kk);
    } else {
        const int klo = k0 < K ? k0 : 0;
        const int khi = k0 + 8 < K ? k0 + 8 : klo;
        const int2 lo = *reinterpret_cast<const int2*>(col + klo);
        const int2 hi = *reinterpret_cast<const int2*>(col + khi);
        return v4i{lo.x, lo.y, hi.x, hi.y};
    }
}

// Weight slices: bytes at k >= K, and every byte of a row past the last
// beam (row_valid false), are zero.
template <bool AL16>
__device__ __forceinline__ v4i load_wslice(const int8_t* col, int k0, int K, bool row_valid)
{
    const v4i r = load_vslice<AL16>(col, k0, K);
    const bool lo_ok = row_valid && k0 < K;
    const bool hi_ok = row_valid && k0 + 8 < K;
    return v4i{lo_ok ? r.x : 0, lo_ok ? r.y : 0, hi_ok ? r.z : 0, hi_ok ? r.w : 0};
}

// Im row: [wr, wi] -> [wi, wr] per antenna (swap the bytes of each 16-bit
// half: one byte permutation).
__device__ __forceinline__ uint32_t swap_pairs(uint32_t x)
{
    return __builtin_amdgcn_perm(x, x, 0x02030001u);
}

typedef unsigned short us2_t __attribute__((ext_vector_type(2)));

// Re row: [wr, wi] -> [wr, -wi] per antenna.  The odd byte of each 16-bit
// half is negated by a packed 16-bit subtract from zero: its low byte is
// zero, so no borrow reaches the even byte.  -wi is exact for wi != -128
// (wi = -128 gives -128 again); weights holding -128 never reach the
// embedded form (below).
__device__ __forceinline__ uint32_t neg_odd(uint32_t x)
{
    const us2_t n = us2_t{0, 0} - __builtin_bit_cast(us2_t, x & 0xFF00FF00u);
    return (x & 0x00FF00FFu) | __builtin_bit_cast(uint32_t, n);
}

// Embedded 16-byte weight slice of an Im row (swap_pairs) or a Re row
// (neg_odd).  The callers pass im_row as a constant, so only one form is
// compiled.
__device__ __forceinline__ v4i embed_slice(v4i raw, bool im_row)
{
    v4i e;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t x = (uint32_t)raw[q];
        e[q] = (int)(im_row ? swap_pairs(x) : neg_odd(x));
    }
    return e;
}

// Weight components wi = -128.  The Re row would carry -wi = 128, which
// int8 cannot hold, while the reference's int32 sums
// (r = xx - yy, CoherentBeamformer.cu:150-155) are exact for every int8
// weight.  Weights round(127 e^{i theta}) never hold -128, so the MFMA paths
// stay as they are and every kernel first checks the weights it will use:
// a wave (or a work-group, where its waves share staging) that finds a
// wi = -128 computes its outputs with cb_exact_outputs instead.
//
// Flag dword from a dword x: 0x01 at the odd byte of every 16-bit pair of x
// whose even byte is 0x80, else 0.  e's even byte is zero exactly for 0x80,
// and adding 0xFF to it carries into bit 8 exactly when it is not zero (at
// most 0x1FE, so the pairs do not interact).
__device__ __forceinline__ int m128_corr(uint32_t x)
{
    const uint32_t e = (x & 0x00FF00FFu) ^ 0x00800080u;
    return (int)(((e + 0x00FF00FFu) & 0x01000100u) ^ 0x01000100u);
}

// Whether a raw FBA slice [wr, wi, ...] holds a wi = -128 (an odd byte 0x80).
__device__ __forceinline__ bool raw_has_m128(v4i raw)
{
    int any = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) any |= m128_corr((uint32_t)raw[q] >> 8);
    return any != 0;
}

// The same over a wave: uniform, so the exact path is a scalar branch.
__device__ __forceinline__ bool wave_any(bool x)
{
    return __builtin_amdgcn_ballot_w64(x) != 0;
}

// Exact outputs of output channel fo for beams [b0, b0 + nb) and output
// windows [w0, w1): the int32 sums of every column (MODE_SUMS,
// [F][T][P][B][2]), the power (MODE_POWER, double [Fo][To][B]) or the staged
// int8 output (MODE_INT8, [Fo][To][B]).  Thread t of nt takes (beam, window)
// pairs t, t + nt, ... and forms plain int32 dot products:
// r = sum wr vr - wi vi and i = sum wr vi + wi vr are exact for every int8
// weight (CoherentBeamformer.cu:150-155); the power is exact in int64 and the
// quantiser is the exact one.  The path of waves (or work-groups) whose
// weights hold a wi = -128; consecutive threads take consecutive beams, so a
// wave's voltage reads are one broadcast column.  TBTF: the int8 output goes to
// TBTF instead ([To/ohs][B][ohs][Fo]).
template <int MODE, bool TBTF = false>
__device__ __forceinline__ void cb_exact_outputs(const CbArgs& p, int fo, int b0, int nb, long long w0,
                                                 long long w1, int t, int nt)
{
    if (w1 > p.nsamples_out) w1 = p.nsamples_out;
    if (w1 <= w0) return;
    const int K = 2 * p.A;
    const size_t TP = (size_t)2 * p.nsamples;
    const int W = 2 * p.ts;
    const float off = p.offsets[fo], sc = p.scales[fo];
    const long long n = (long long)nb * (w1 - w0);
    for (long long idx = t; idx < n; idx += nt) {
        const int b = b0 + (int)(idx % nb);
        const long long w = w0 + idx / nb;
        if (b >= p.B) continue;
        long long P = 0;
        for (int fc = 0; fc < p.fs; ++fc) {
            const int f = fo * p.fs + fc;
            const int8_t* wrow = p.fba + ((size_t)f * p.B + b) * K;
            for (int j = 0; j < W; ++j) {
                // Column (sample, pol) jc of channel f; antenna a at col + a * astep.
                const long long jc = w * W + j;
                const int8_t* col;
                size_t astep;
                if (p.S > 0) {
                    const long long t = jc >> 1;
                    col = p.ftpa + (((size_t)(t / p.S) * p.Atot + p.a0) * p.F + f) * p.S * 4 +
                          (size_t)(t % p.S) * 4 + 2 * (jc & 1);
                    astep = (size_t)p.F * p.S * 4;
                } else {
                    col = p.ftpa + ((size_t)f * TP + (size_t)jc) * p.vstride + p.voff;
                    astep = 2;
                }
                int re = 0, im = 0;
                for (int a = 0; a < p.A; ++a) {
                    const int vr = col[a * astep], vi = col[a * astep + 1];
                    const int wr = wrow[2 * a], wi = wrow[2 * a + 1];
                    re += wr * vr - wi * vi;
                    im += wr * vi + wi * vr;
                }
                if (MODE == MODE_SUMS) {
                    int32_t* dst = static_cast<int32_t*>(p.out) + (((size_t)f * TP + (size_t)w * W + j) * p.B + b) * 2;
                    dst[0] = re;
                    dst[1] = im;
                }
                P += (long long)re * re + (long long)im * im;
            }
        }
        const size_t o = ((size_t)fo * p.nsamples_out + (size_t)w) * p.B + b;
        if (MODE == MODE_POWER) static_cast<double*>(p.out)[o] = (double)P;
        if constexpr (TBTF) {
            const long long heap = w / p.ohs;
            const size_t ot = ((size_t)(heap * p.B + b) * p.ohs + (size_t)(w - heap * p.ohs)) * p.Fo + fo;
            static_cast<int8_t*>(p.out)[ot] = quantise((double)P, off, sc, p.quant);
        } else if (MODE == MODE_INT8) {
            static_cast<int8_t*>(p.out)[o] = quantise((double)P, off, sc, p.quant);
        }
    }
}

// Whether any weight of beams [b0, b0 + nb) over the fscrunch channels of
// output channel fo holds a wi = -128, as seen by this lane (lanes take
// 16-byte pieces t, t + nt, ...).  K = 2A is a multiple of 8: pieces are
// 16 bytes, or 8 at the end of a row.
__device__ __forceinline__ bool cb_weights_have_m128(const CbArgs& p, int fo, int b0, int nb, int t, int nt)
{
    const int K = 2 * p.A;
    const int kp = (K + 15) / 16;
    bool m = false;
    const int n = p.fs * nb * kp;
    for (int i = t; i < n; i += nt) {
        const int fc = i / (nb * kp);
        const int r = i - fc * nb * kp;
        const int b = b0 + r / kp;
        const int k0 = 16 * (r % kp);
        if (b >= p.B) continue;
        const int8_t* row = p.fba + ((size_t)(fo * p.fs + fc) * p.B + b) * K;
        const int2 lo = *reinterpret_cast<const int2*>(row + k0);
        const int2 hi = k0 + 8 < K ? *reinterpret_cast<const int2*>(row + k0 + 8) : int2{0, 0};
        m |= raw_has_m128(v4i{lo.x, lo.y, hi.x, hi.y});
    }
    return m;
}

constexpr int kLdsMaxPieces = 4;   // per-thread prefetch registers (pieces) of cb_lds_k

// Chunk length: the largest power of two <= 16 that divides tsp and keeps
// one chunk within kLdsMaxPieces pieces per thread.
inline int cb_lds_chunk(int tsp, int K, bool al16)
{
    const int pb = al16 ? 16 : 8;
    int jc = 16;
    while (jc > 1 && (tsp % jc != 0 || 32 * jc * K / pb > 256 * kLdsMaxPieces)) jc >>= 1;
    return jc;
}

}  // namespace
}  // namespace fbf
