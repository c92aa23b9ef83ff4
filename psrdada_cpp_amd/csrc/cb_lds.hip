// Coherent beamformer with the weights as the A operand: the register-fed
// kernels (cb_mfma_k, cb_mfma32_k) and the LDS-staged one (cb_lds_k), which also
// serve int32 sums, power output and every scrunch.
#include "cb_common.hpp"

namespace fbf {
namespace {

template <int ROWT, int KSTEPS, int MODE, bool AL16>
__global__ __launch_bounds__(256) void cb_mfma_k(CbArgs p)
{
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int g = lane >> 4;   // K group of the operands, row group of D
    const int c = lane & 15;   // A row / B,D column
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int bgroup = logical % p.n_bgroups;
    const int rest = logical / p.n_bgroups;
    const int tgroup = rest % p.n_tgroups;
    const int fo = rest / p.n_tgroups;
    const int wt = 4 / p.wb;
    const int bc = bgroup * p.wb + (wave % p.wb);
    const int tc = tgroup * wt + (wave / p.wb);
    if (bc >= p.n_bchunks || tc >= p.n_tchunks || fo >= p.Fo) return;

    const int K = 2 * p.A;
    const int beam_base = bc * (8 * ROWT);
    const long long t_out = (long long)tc * 16 + c;
    const bool t_valid = t_out < p.nsamples_out;
    // Lanes past the last output sample read (and never store) the last one.
    const long long t_addr = t_valid ? t_out : p.nsamples_out - 1;
    const int tsp = 2 * p.ts;
    const long long TP = 2 * p.nsamples;

    // A wave whose weights hold a wi = -128 takes the exact path.
    if (wave_any(cb_weights_have_m128(p, fo, beam_base, 8 * ROWT, lane, 64))) {
        cb_exact_outputs<MODE>(p, fo, beam_base, 8 * ROWT, (long long)tc * 16, (long long)tc * 16 + 16, lane, 64);
        return;
    }

    long long pw[ROWT][2];
#pragma unroll
    for (int r = 0; r < ROWT; ++r) pw[r][0] = pw[r][1] = 0;

    for (int fc = 0; fc < p.fs; ++fc) {
        const int f = fo * p.fs + fc;
        // Embedded weights for this channel: lane holds row c of each 16-row tile.
        v4i w[ROWT][KSTEPS];
#pragma unroll
        for (int r = 0; r < ROWT; ++r) {
            const int b = beam_base + r * 8 + (c >> 1);
            const bool bvalid = b < p.B;
            const int8_t* wcol = p.fba + ((size_t)f * p.B + (bvalid ? b : p.B - 1)) * K;
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) w[r][s] = load_wslice<AL16>(wcol, s * 64 + g * 16, K, bvalid);
        }
        // Every load is in flight before the first is used.
#pragma unroll
        for (int r = 0; r < ROWT; ++r)
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) w[r][s] = embed_slice(w[r][s], c & 1);

        const int8_t* vcol = p.ftpa + ((size_t)f * TP + (size_t)t_addr * tsp) * p.vstride + p.voff;
        v4i v[KSTEPS];
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) v[s] = load_vslice<AL16>(vcol, s * 64 + g * 16, K);

        for (int j = 0; j < tsp; ++j) {
            // Prefetch the next column while this one is multiplied (the last
            // step re-reads its own column).
            v4i vn[KSTEPS];
            const int jn = j + 1 < tsp ? j + 1 : j;
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) vn[s] = load_vslice<AL16>(vcol + (size_t)jn * p.vstride, s * 64 + g * 16, K);
#pragma unroll
            for (int r = 0; r < ROWT; ++r) {
                v4i acc = {0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < KSTEPS; ++s)
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[r][s], v[s], acc, 0, 0, 0);
                if (MODE == MODE_SUMS) {
                    const int b0 = beam_base + r * 8 + 2 * g;
                    if (t_valid && b0 < p.B) {
                        const long long n = t_out * tsp + j;
                        int32_t* dst = static_cast<int32_t*>(p.out) +
                                       (((size_t)f * TP + (size_t)n) * p.B + b0) * 2;
                        *reinterpret_cast<v4i*>(dst) = acc;
                    }
                }
                pw[r][0] += (long long)acc[0] * acc[0];
                pw[r][0] += (long long)acc[1] * acc[1];
                pw[r][1] += (long long)acc[2] * acc[2];
                pw[r][1] += (long long)acc[3] * acc[3];
            }
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) v[s] = vn[s];
        }
    }

    if (MODE == MODE_SUMS || !t_valid) return;
    if (MODE == MODE_POWER) {
        double* dst = static_cast<double*>(p.out) + ((size_t)fo * p.nsamples_out + t_out) * p.B;
#pragma unroll
        for (int r = 0; r < ROWT; ++r) {
            const int b0 = beam_base + r * 8 + 2 * g;
            if (b0 < p.B) {
                dst[b0] = (double)pw[r][0];
                dst[b0 + 1] = (double)pw[r][1];
            }
        }
        return;
    }
    // int8, staged [fo][to][b]
    const float off = p.offsets[fo];
    const float sc = p.scales[fo];
    int8_t* row = static_cast<int8_t*>(p.out) + ((size_t)fo * p.nsamples_out + t_out) * p.B;
#pragma unroll
    for (int r = 0; r < ROWT; ++r) {
        const int b0 = beam_base + r * 8 + 2 * g;
        if (b0 < p.B)
            store_pair(row + b0, quantise((double)pw[r][0], off, sc, p.quant),
                       quantise((double)pw[r][1], off, sc, p.quant));
    }
}

// ---------------------------------------------------------------------------
// v2: v_mfma_i32_32x32x32_i8 (the full-rate int8 MFMA on gfx950).
//
// A (32 rows x 32 k) = embedded weights, lane l: row l%32, K half h = l/32.
// B (32 k x 32 cols) = voltages, lane l: column l%32, K half h.
// D lane l: column l%32, rows 8*(i/4) + 4*h + i%4 for i = 0..15, so a lane
// holds Re and Im of beams 4*q + 2*h + {0, 1} (q = 0..3) of its row tile.
// K is split into 16-byte slices; slice (h, s) covers bytes
// [16 * (h * KSTEPS + s), +16) of a column, so each lane reads one contiguous
// 16*KSTEPS-byte half of every voltage column.  The 32 columns of a tile are
// 32 output samples; column j of the integration window is processed at
// step j, with two columns in flight (va / vb) so that loads overlap the
// MFMAs and the FP64 detection of the previous column.
// ---------------------------------------------------------------------------

template <int KSTEPS, bool AL16>
__device__ __forceinline__ void cb32_load_col(v4i (&v)[KSTEPS], const int8_t* col, int h, int K)
{
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) v[s] = load_vslice<AL16>(col, 16 * (h * KSTEPS + s), K);
}

template <int RT, int KSTEPS, int MODE>
__device__ __forceinline__ void cb32_column(const v4i (&w)[RT][KSTEPS], const v4i (&v)[KSTEPS],
                                            long long (&pw)[RT][4][2], const CbArgs& p, int f, long long n,
                                            int beam_base, int h, bool t_valid)
{
    v16i acc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        acc[r] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
            acc[r] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[r][s], v[s], acc[r], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        if (MODE == MODE_SUMS) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int b0 = beam_base + r * 16 + 4 * q + 2 * h;
                if (t_valid && b0 < p.B) {
                    int32_t* dst = static_cast<int32_t*>(p.out) +
                                   (((size_t)f * 2 * p.nsamples + (size_t)n) * p.B + b0) * 2;
                    *reinterpret_cast<v4i*>(dst) = v4i{acc[r][4 * q], acc[r][4 * q + 1], acc[r][4 * q + 2],
                                                       acc[r][4 * q + 3]};
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int xr = acc[r][4 * q + 2 * e];
                const int xi = acc[r][4 * q + 2 * e + 1];
                pw[r][q][e] += (long long)xr * xr;
                pw[r][q][e] += (long long)xi * xi;
            }
        }
    }
}

// MFMA half of cb32_column: acc[r] = W'[r] x column.
template <int RT, int KSTEPS>
__device__ __forceinline__ void cb32_mfma(v16i (&acc)[RT], const v4i (&w)[RT][KSTEPS], const v4i (&v)[KSTEPS])
{
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        acc[r] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
            acc[r] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[r][s], v[s], acc[r], 0, 0, 0);
    }
}

// Detection half of cb32_column: |beam|^2 into the exact int64 accumulators
// (and, in MODE_SUMS, the raw int32 sums to memory).
template <int RT, int MODE>
__device__ __forceinline__ void cb32_detect(const v16i (&acc)[RT], long long (&pw)[RT][4][2], const CbArgs& p,
                                            int f, long long n, int beam_base, int h, bool t_valid)
{
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        if (MODE == MODE_SUMS) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int b0 = beam_base + r * 16 + 4 * q + 2 * h;
                if (t_valid && b0 < p.B) {
                    int32_t* dst = static_cast<int32_t*>(p.out) +
                                   (((size_t)f * 2 * p.nsamples + (size_t)n) * p.B + b0) * 2;
                    *reinterpret_cast<v4i*>(dst) = v4i{acc[r][4 * q], acc[r][4 * q + 1], acc[r][4 * q + 2],
                                                       acc[r][4 * q + 3]};
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int xr = acc[r][4 * q + 2 * e];
                const int xi = acc[r][4 * q + 2 * e + 1];
                pw[r][q][e] += (long long)xr * xr;
                pw[r][q][e] += (long long)xi * xi;
            }
    }
}

template <int KSTEPS>
__device__ __forceinline__ void lds_col(v4i (&v)[KSTEPS], const int8_t* src, int jj, int c, int h, int kp)
{
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s)
        v[s] = *reinterpret_cast<const v4i*>(src + (jj * 32 + c) * kp + 16 * (h * KSTEPS + s));
}

template <int RT, int KSTEPS, int MODE, bool AL16>
__global__ __launch_bounds__(256) void cb_mfma32_k(CbArgs p)
{
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int h = lane >> 5;
    const int c = lane & 31;
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int bgroup = logical % p.n_bgroups;
    const int rest = logical / p.n_bgroups;
    const int tgroup = rest % p.n_tgroups;
    const int fo = rest / p.n_tgroups;
    const int wt = 4 / p.wb;
    const int bc = bgroup * p.wb + (wave % p.wb);
    const int tc = tgroup * wt + (wave / p.wb);
    if (bc >= p.n_bchunks || tc >= p.n_tchunks || fo >= p.Fo) return;

    const int K = 2 * p.A;
    const int beam_base = bc * (16 * RT);
    const long long t_out = (long long)tc * 32 + c;
    const bool t_valid = t_out < p.nsamples_out;
    // Lanes past the last output sample read (and never store) the last one.
    const long long t_addr = t_valid ? t_out : p.nsamples_out - 1;
    const int tsp = 2 * p.ts;
    const long long TP = 2 * p.nsamples;

    // A wave whose weights hold a wi = -128 takes the exact path.
    if (wave_any(cb_weights_have_m128(p, fo, beam_base, 16 * RT, lane, 64))) {
        cb_exact_outputs<MODE>(p, fo, beam_base, 16 * RT, (long long)tc * 32, (long long)tc * 32 + 32, lane, 64);
        return;
    }

    long long pw[RT][4][2];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q) pw[r][q][0] = pw[r][q][1] = 0;

    for (int fc = 0; fc < p.fs; ++fc) {
        const int f = fo * p.fs + fc;
        v4i w[RT][KSTEPS];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int b = beam_base + r * 16 + (c >> 1);
            const bool bvalid = b < p.B;
            const int8_t* wcol = p.fba + ((size_t)f * p.B + (bvalid ? b : p.B - 1)) * K;
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) w[r][s] = load_wslice<AL16>(wcol, 16 * (h * KSTEPS + s), K, bvalid);
        }
        // Every load is in flight before the first is used.
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) w[r][s] = embed_slice(w[r][s], c & 1);

        const int8_t* vcol = p.ftpa + ((size_t)f * TP + (size_t)t_addr * tsp) * p.vstride + p.voff;
        const long long n0 = t_out * tsp;
        v4i va[KSTEPS], vb[KSTEPS];
        cb32_load_col<KSTEPS, AL16>(va, vcol, h, K);
        cb32_load_col<KSTEPS, AL16>(vb, vcol + p.vstride, h, K);
        for (int j = 0; j < tsp; j += 2) {
            // Two columns in flight; the last steps re-read the final column.
            const int j2 = j + 2 < tsp ? j + 2 : tsp - 1;
            const int j3 = j + 3 < tsp ? j + 3 : tsp - 1;
            v4i cur[KSTEPS];
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) cur[s] = va[s];
            cb32_load_col<KSTEPS, AL16>(va, vcol + (size_t)j2 * p.vstride, h, K);
            cb32_column<RT, KSTEPS, MODE>(w, cur, pw, p, f, n0 + j, beam_base, h, t_valid);
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) cur[s] = vb[s];
            cb32_load_col<KSTEPS, AL16>(vb, vcol + (size_t)j3 * p.vstride, h, K);
            cb32_column<RT, KSTEPS, MODE>(w, cur, pw, p, f, n0 + j + 1, beam_base, h, t_valid);
        }
    }

    if (MODE == MODE_SUMS || !t_valid) return;
    if (MODE == MODE_POWER) {
        double* dst = static_cast<double*>(p.out) + ((size_t)fo * p.nsamples_out + t_out) * p.B;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int b0 = beam_base + r * 16 + 4 * q + 2 * h;
                if (b0 < p.B) {
                    dst[b0] = (double)pw[r][q][0];
                    dst[b0 + 1] = (double)pw[r][q][1];
                }
            }
        return;
    }
    // int8, staged [fo][to][b]
    const float off = p.offsets[fo];
    const float sc = p.scales[fo];
    int8_t* row = static_cast<int8_t*>(p.out) + ((size_t)fo * p.nsamples_out + t_out) * p.B;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int b0 = beam_base + r * 16 + 4 * q + 2 * h;
            if (b0 < p.B)
                store_pair(row + b0, quantise((double)pw[r][q][0], off, sc, p.quant),
                           quantise((double)pw[r][q][1], off, sc, p.quant));
        }
}

// ---------------------------------------------------------------------------
// v3: 32x32x32 MFMA with the voltage tile staged through LDS.
//
// The four waves of a work-group share the same 32 output samples and take
// 16*RT beams each, so one copy of the voltage columns in LDS feeds all four.
// The integration window of the 32 samples is streamed in chunks of JC
// columns: every thread loads its share of the next chunk from HBM/L2 with
// wide coalesced loads (each sample's JC columns are contiguous) while the
// current chunk is multiplied out of the other LDS buffer.  LDS rows are
// padded to 32*KSTEPS + 16 bytes so that the ds_read_b128 of consecutive
// lanes fall on distinct bank groups.
// ---------------------------------------------------------------------------

template <int RT, int KSTEPS, int MODE, bool AL16>
__global__ __launch_bounds__(256) void cb_lds_k(CbArgs p, int jc)
{
    extern __shared__ __align__(16) int8_t lds[];
    constexpr int KP = 32 * KSTEPS + 16;
    constexpr int PB = AL16 ? 16 : 8;   // bytes per fill piece
    using Piece = typename std::conditional<AL16, v4i, int2>::type;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int h = lane >> 5;
    const int c = lane & 31;
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int bgroup = logical % p.n_bgroups;
    const int rest = logical / p.n_bgroups;
    const int tgroup = rest % p.n_tgroups;
    const int fo = rest / p.n_tgroups;
    if (fo >= p.Fo) return;   // uniform over the work-group

    const int K = 2 * p.A;
    const int beam_base = (bgroup * 4 + wave) * (16 * RT);
    const bool wave_active = beam_base < p.B;
    const long long t0 = (long long)tgroup * 32;
    const long long t_out = t0 + c;
    const bool t_valid = t_out < p.nsamples_out;
    const int tsp = 2 * p.ts;
    const long long TP = 2 * p.nsamples;
    const int buf_bytes = jc * 32 * KP;
    const int pieces_per_run = jc * K / PB;   // one output sample's jc columns
    const int npieces = 32 * pieces_per_run;
    const int nchunks = tsp / jc;

    // A work-group any of whose weights hold a wi = -128 takes the exact
    // path (its waves share the voltage staging, so all of them).
    if (__syncthreads_or(cb_weights_have_m128(p, fo, bgroup * 4 * 16 * RT, 4 * 16 * RT, tid, 256) ? 1 : 0)) {
        cb_exact_outputs<MODE>(p, fo, bgroup * 4 * 16 * RT, 4 * 16 * RT, t0, t0 + 32, tid, 256);
        return;
    }

    long long pw[RT][4][2];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q) pw[r][q][0] = pw[r][q][1] = 0;

    for (int fc = 0; fc < p.fs; ++fc) {
        const int f = fo * p.fs + fc;
        v4i w[RT][KSTEPS];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int b = beam_base + r * 16 + (c >> 1);
            const bool bvalid = b < p.B;
            const int8_t* wcol = p.fba + ((size_t)f * p.B + (bvalid ? b : p.B - 1)) * K;
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) w[r][s] = load_wslice<AL16>(wcol, 16 * (h * KSTEPS + s), K, bvalid);
        }
        // Every load is in flight before the first is used.
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) w[r][s] = embed_slice(w[r][s], c & 1);

        const int8_t* vbase = p.ftpa + (size_t)f * TP * p.vstride + p.voff;
        Piece pre[kLdsMaxPieces];
        auto fetch = [&](int chunk) {
#pragma unroll
            for (int u = 0; u < kLdsMaxPieces; ++u) {
                const int i = tid + 256 * u;
                const int ii = i < npieces ? i : npieces - 1;
                const int cc = ii / pieces_per_run;
                const int o = (ii - cc * pieces_per_run) * PB;
                long long tc = t0 + cc;
                tc = tc < p.nsamples_out ? tc : p.nsamples_out - 1;
                const int jj = o / K;
                pre[u] = *reinterpret_cast<const Piece*>(vbase + ((size_t)tc * tsp + (size_t)chunk * jc + jj) * p.vstride +
                                                         (o - jj * K));
            }
        };
        auto stash = [&](int buf) {
            int8_t* dst = lds + buf * buf_bytes;
#pragma unroll
            for (int u = 0; u < kLdsMaxPieces; ++u) {
                const int i = tid + 256 * u;
                if (i < npieces) {
                    const int cc = i / pieces_per_run;
                    const int o = (i - cc * pieces_per_run) * PB;
                    const int jj = o / K;
                    const int kb = o - jj * K;
                    *reinterpret_cast<Piece*>(dst + (jj * 32 + cc) * KP + kb) = pre[u];
                }
            }
        };

        fetch(0);
        stash(0);
        __syncthreads();
        for (int k = 0; k < nchunks; ++k) {
            if (k + 1 < nchunks) fetch(k + 1);
            if (wave_active) {
                // One column at a time: with three waves per SIMD the
                // hardware interleaves MFMA and detection of different waves
                // (a two-deep software pipeline costs a wave of occupancy and
                // measured slower).
                const int8_t* src = lds + (k & 1) * buf_bytes;
                const long long n0 = t_out * tsp + (long long)k * jc;
                for (int jj = 0; jj < jc; ++jj) {
                    v4i v[KSTEPS];
                    lds_col<KSTEPS>(v, src, jj, c, h, KP);
                    v16i acc[RT];
                    cb32_mfma<RT, KSTEPS>(acc, w, v);
                    cb32_detect<RT, MODE>(acc, pw, p, f, n0 + jj, beam_base, h, t_valid);
                }
            }
            if (k + 1 < nchunks) stash((k + 1) & 1);
            __syncthreads();
        }
    }

    if (MODE == MODE_SUMS || !t_valid || !wave_active) return;
    if (MODE == MODE_POWER) {
        double* dst = static_cast<double*>(p.out) + ((size_t)fo * p.nsamples_out + t_out) * p.B;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int b0 = beam_base + r * 16 + 4 * q + 2 * h;
                if (b0 < p.B) {
                    dst[b0] = (double)pw[r][q][0];
                    dst[b0 + 1] = (double)pw[r][q][1];
                }
            }
        return;
    }
    // int8, staged [fo][to][b]
    const float off = p.offsets[fo];
    const float sc = p.scales[fo];
    int8_t* row = static_cast<int8_t*>(p.out) + ((size_t)fo * p.nsamples_out + t_out) * p.B;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int b0 = beam_base + r * 16 + 4 * q + 2 * h;
            if (b0 < p.B)
                store_pair(row + b0, quantise((double)pw[r][q][0], off, sc, p.quant),
                           quantise((double)pw[r][q][1], off, sc, p.quant));
        }
}

inline size_t cb_lds_bytes(int ksteps, int jc) { return (size_t)2 * jc * 32 * (32 * ksteps + 16); }

template <int RT, int MODE, bool AL16>
hipError_t launch_lds_rt(const CbArgs& a, int ksteps, int jc, dim3 grid, hipStream_t s)
{
    const size_t shm = cb_lds_bytes(ksteps, jc);
    switch (ksteps) {
    case 1: cb_lds_k<RT, 1, MODE, AL16><<<grid, 256, shm, s>>>(a, jc); break;
    case 2: cb_lds_k<RT, 2, MODE, AL16><<<grid, 256, shm, s>>>(a, jc); break;
    case 3: cb_lds_k<RT, 3, MODE, AL16><<<grid, 256, shm, s>>>(a, jc); break;
    case 4: cb_lds_k<RT, 4, MODE, AL16><<<grid, 256, shm, s>>>(a, jc); break;
    case 5: cb_lds_k<RT, 5, MODE, AL16><<<grid, 256, shm, s>>>(a, jc); break;
    case 6: cb_lds_k<RT, 6, MODE, AL16><<<grid, 256, shm, s>>>(a, jc); break;
    case 7: cb_lds_k<RT, 7, MODE, AL16><<<grid, 256, shm, s>>>(a, jc); break;
    case 8: cb_lds_k<RT, 8, MODE, AL16><<<grid, 256, shm, s>>>(a, jc); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int MODE>
hipError_t launch_lds_mode(const CbArgs& a, int rt, int ksteps, int jc, dim3 grid, hipStream_t s)
{
    const bool al16 = (a.A % 8) == 0;
    switch (rt) {
    case 1: return al16 ? launch_lds_rt<1, MODE, true>(a, ksteps, jc, grid, s)
                        : launch_lds_rt<1, MODE, false>(a, ksteps, jc, grid, s);
    case 2: return al16 ? launch_lds_rt<2, MODE, true>(a, ksteps, jc, grid, s)
                        : launch_lds_rt<2, MODE, false>(a, ksteps, jc, grid, s);
    case 4: return al16 ? launch_lds_rt<4, MODE, true>(a, ksteps, jc, grid, s)
                        : launch_lds_rt<4, MODE, false>(a, ksteps, jc, grid, s);
    default: return hipErrorInvalidValue;
    }
}

template <int RT, int MODE, bool AL16>
hipError_t launch32_rt(const CbArgs& a, int ksteps, dim3 grid, hipStream_t s)
{
    switch (ksteps) {
    case 1: cb_mfma32_k<RT, 1, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 2: cb_mfma32_k<RT, 2, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 3: cb_mfma32_k<RT, 3, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 4: cb_mfma32_k<RT, 4, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 5: cb_mfma32_k<RT, 5, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 6: cb_mfma32_k<RT, 6, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 7: cb_mfma32_k<RT, 7, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 8: cb_mfma32_k<RT, 8, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int MODE>
hipError_t launch32_mode(const CbArgs& a, int rt, int ksteps, dim3 grid, hipStream_t s)
{
    const bool al16 = (a.A % 8) == 0;
    if (rt == 4)
        return al16 ? launch32_rt<4, MODE, true>(a, ksteps, grid, s) : launch32_rt<4, MODE, false>(a, ksteps, grid, s);
    return al16 ? launch32_rt<2, MODE, true>(a, ksteps, grid, s) : launch32_rt<2, MODE, false>(a, ksteps, grid, s);
}

template <int ROWT, int MODE, bool AL16>
hipError_t launch_rowt(const CbArgs& a, int ksteps, dim3 grid, hipStream_t s)
{
    switch (ksteps) {
    case 1: cb_mfma_k<ROWT, 1, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 2: cb_mfma_k<ROWT, 2, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 3: cb_mfma_k<ROWT, 3, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    case 4: cb_mfma_k<ROWT, 4, MODE, AL16><<<grid, 256, 0, s>>>(a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int MODE>
hipError_t launch_mode(const CbArgs& a, int rowt, int ksteps, dim3 grid, hipStream_t s)
{
    const bool al16 = (a.A % 8) == 0;
    if (rowt == 8)
        return al16 ? launch_rowt<8, MODE, true>(a, ksteps, grid, s) : launch_rowt<8, MODE, false>(a, ksteps, grid, s);
    return al16 ? launch_rowt<4, MODE, true>(a, ksteps, grid, s) : launch_rowt<4, MODE, false>(a, ksteps, grid, s);
}

}  // namespace
}  // namespace fbf

hipError_t fbf::cb_launch_lds(const CbArgs& a, int mode, int rt, int ksteps, int jc, dim3 grid, hipStream_t s)
{
    if (mode == MODE_INT8) return launch_lds_mode<MODE_INT8>(a, rt, ksteps, jc, grid, s);
    if (mode == MODE_SUMS) return launch_lds_mode<MODE_SUMS>(a, rt, ksteps, jc, grid, s);
    return launch_lds_mode<MODE_POWER>(a, rt, ksteps, jc, grid, s);
}

hipError_t fbf::cb_launch_mfma32(const CbArgs& a, int mode, int rt, int ksteps, dim3 grid, hipStream_t s)
{
    if (mode == MODE_INT8) return launch32_mode<MODE_INT8>(a, rt, ksteps, grid, s);
    if (mode == MODE_SUMS) return launch32_mode<MODE_SUMS>(a, rt, ksteps, grid, s);
    return launch32_mode<MODE_POWER>(a, rt, ksteps, grid, s);
}

hipError_t fbf::cb_launch_mfma16(const CbArgs& a, int mode, int rowt, int ksteps, dim3 grid, hipStream_t s)
{
    if (mode == MODE_INT8) return launch_mode<MODE_INT8>(a, rowt, ksteps, grid, s);
    if (mode == MODE_SUMS) return launch_mode<MODE_SUMS>(a, rowt, ksteps, grid, s);
    return launch_mode<MODE_POWER>(a, rowt, ksteps, grid, s);
}
