// Coherent beamformer: the transposed-tile kernel (cb_tr_k), its detection and
// its quantiser.
#pragma once

#include "cb_common.hpp"
#include "cb_stage.hpp"

namespace fbf {
namespace {

// ---------------------------------------------------------------------------
// Transposed tiles: voltages as the A operand, weights as the B operand.
//
//   D[m][n] = sum_k V[m][k] W'[n][k]
//
// Rows m are 32 consecutive input columns (t, p) of one channel, columns n
// are 16 beams x (Re, Im) embedding rows.  Lane l holds column n = l % 32
// and rows 8*(i/4) + 4*(l/32) + i%4 (i = 0..15).  For an integration window
// of W = 2*tscrunch = 8, 16 or 32 columns, or a multiple of 32, every window
// a lane touches is a fixed group of its 16 values, so the squares sum into
// one int64 per (beam tile, window) in the lane.  The four lanes holding
// {Re, Im} x {row halves} of a beam are combined once per pass of windows by
// a reduce-scatter (exchange with lane ^ 1, then lane ^ 32) that leaves each
// lane a distinct (beam, window) total to quantise.
//
// A wave keeps RT beam tiles (16 RT beams) of weights in registers for its
// channel and reads each voltage tile once from LDS for all of them: LDS
// traffic is 1/RT of a tile per MFMA.  With fscrunch FS = 2 or 4 the waves of
// a work-group take different channels of the fscrunch group (each with its
// own weights) and add their window totals through LDS before quantising.
//
// Voltage staging is a ring of NB tile sets in LDS (one tile per channel of
// the fscrunch group per set) filled by direct global->LDS loads issued
// NB - 1 tiles ahead.  Every step issues one set (past the work-group's last
// tile the loads repeat the last tile into a slot nobody reads), so the
// number of loads in flight after a wave's loads of the current set is the
// constant (NB - 2) * M and the wait is a fixed s_waitcnt.
// ---------------------------------------------------------------------------

// s_waitcnt vmcnt(N) lgkmcnt(0).
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0()
{
    static_assert(N >= 0 && N <= 63, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

// One 16-byte global->LDS load per lane: lane i's 16 bytes land at
// lds_run + 16 * i (lds_run is wave-uniform).
__device__ __forceinline__ void dma16(const int8_t* src, int8_t* lds_run)
{
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)lds_run, 16, 0, 0);
}

// A wave-uniform pointer as scalar registers, so that a load from it plus a
// 32-bit lane offset takes the scalar-base address form (no 64-bit vector
// address arithmetic per load).
template <typename T>
__device__ __forceinline__ T* uniform_ptr(T* ptr)
{
    const unsigned long long v = reinterpret_cast<unsigned long long>(ptr);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return reinterpret_cast<T*>(((unsigned long long)hi << 32) | lo);
}

// A pointer known to address global memory, so that stores through it are
// global (not flat: a flat store also counts against the LDS wait counter).
__device__ __forceinline__ __attribute__((address_space(1))) int8_t* global_ptr(int8_t* ptr)
{
    return (__attribute__((address_space(1))) int8_t*)ptr;
}

// Work-group barrier without the memory fence of __syncthreads (which would
// wait for every outstanding global load, including the LDS prefetches).
// Callers wait for their own LDS and global->LDS traffic first; the empty
// asm statements keep the compiler from moving memory accesses across.
__device__ __forceinline__ void block_barrier()
{
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

// The incoherent-beam partials of tiles [t0, t1) of channel f straight from
// the TAFTP block, for the work-groups on the exact path (which leave the
// tile loop): per sample the power over all antennas and both pols in
// column 2j of half 0, zeros in its other three places.
__device__ __forceinline__ void cb_exact_ib_partials(const CbArgs& p, int* ibp, int ntiles, int f, int t0, int t1,
                                                  int tid, int nt)
{
    const size_t astep = (size_t)p.F * p.S * 4;
    for (int i = tid; i < (t1 - t0) * 16; i += nt) {
        const int tile = t0 + i / 16, j = i % 16;
        const long long t = (long long)tile * 16 + j;
        const int8_t* v = p.ftpa + (((size_t)(t / p.S) * p.Atot + p.a0) * p.F + f) * p.S * 4 + (size_t)(t % p.S) * 4;
        int sum = 0;
        for (int a = 0; a < p.A; ++a) {
            const int w = *reinterpret_cast<const int*>(v + a * astep);
            sum = __builtin_amdgcn_sdot4(w, w, sum, false);
        }
        int* dst = ibp + ((size_t)f * ntiles + tile) * 64 + 2 * j;
        dst[0] = sum;
        dst[1] = 0;
        dst[32] = 0;
        dst[33] = 0;
    }
}

// The same work-groups' incoherent-beam outputs where the kernel writes them
// itself (windows within a tile): one window per thread.
__device__ __forceinline__ void cb_exact_ib_outputs(const CbArgs& p, const IbFinishJob& ib, int f, int t0, int t1,
                                                 int tid, int nt)
{
    const size_t astep = (size_t)p.F * p.S * 4;
    const int per_tile = 16 / ib.ts;
    for (int i = tid; i < (t1 - t0) * per_tile; i += nt) {
        const long long w = (long long)t0 * per_tile + i;
        int sum = 0;
        for (int j = 0; j < ib.ts; ++j) {
            const long long t = w * ib.ts + j;
            const int8_t* v = p.ftpa + (((size_t)(t / p.S) * p.Atot + p.a0) * p.F + f) * p.S * 4 + (size_t)(t % p.S) * 4;
            for (int a = 0; a < p.A; ++a) {
                const int x = *reinterpret_cast<const int*>(v + a * astep);
                sum = __builtin_amdgcn_sdot4(x, x, sum, false);
            }
        }
        ib.out[w * p.F + f] = quantise((double)sum, ib.offsets[f], ib.scales[f], ib.quant);
    }
}

// The 16-byte A operands of one step's K slices (8 antennas x char2 of one
// column each) from an LDS tile laid out [antenna][32 columns] int16, 64
// bytes a row: two ds_read_b64_tr_b16 of 4 antenna rows each per slice.
// Within every 16-lane group G the instruction gives lane i, as its element
// r, element i % 4 of the 8 bytes read by lane 16 G + 4 r + i / 4.  So when
// lane L reads the 4 columns 16 (G % 2) + 4 (L % 4) .. + 3 of antenna row
// base + (L / 4) % 4, lane c + 32 h (c < 32) receives column c of rows
// base .. base + 3, in row order.  `src` is that row piece of slice 0 for
// this lane; slice s is 8 rows (512 bytes) further on, its second read 4
// rows (256 bytes) after its first.
//
// The reads of up to four slices are issued in one asm block that ends with
// their LDS wait.
// Issued through the builtin, every transposed read is preceded by a wait
// for all outstanding global->LDS loads (the compiler cannot tell that they
// fill other ring slots), which cost the kernel a memory round trip per
// step; the ring's own vmcnt wait and barrier already order them.  The
// outputs are complete when the block ends (lgkmcnt(0) inside it).
typedef int v2i __attribute__((ext_vector_type(2)));

// 2 * N transposed reads of N slices from `addr` on, and their LDS wait.
template <int N>
__device__ __forceinline__ void tr_reads(uint32_t addr, v2i* r)
{
    static_assert(N >= 1 && N <= 4, "slices per block");
    if constexpr (N == 1) {
        __asm__ volatile(
            "ds_read_b64_tr_b16 %0, %2\n\t"
            "ds_read_b64_tr_b16 %1, %2 offset:256\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(r[0]), "=&v"(r[1])
            : "v"(addr)
            : "memory");
    } else if constexpr (N == 2) {
        __asm__ volatile(
            "ds_read_b64_tr_b16 %0, %4\n\t"
            "ds_read_b64_tr_b16 %1, %4 offset:256\n\t"
            "ds_read_b64_tr_b16 %2, %4 offset:512\n\t"
            "ds_read_b64_tr_b16 %3, %4 offset:768\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
            : "v"(addr)
            : "memory");
    } else if constexpr (N == 3) {
        __asm__ volatile(
            "ds_read_b64_tr_b16 %0, %6\n\t"
            "ds_read_b64_tr_b16 %1, %6 offset:256\n\t"
            "ds_read_b64_tr_b16 %2, %6 offset:512\n\t"
            "ds_read_b64_tr_b16 %3, %6 offset:768\n\t"
            "ds_read_b64_tr_b16 %4, %6 offset:1024\n\t"
            "ds_read_b64_tr_b16 %5, %6 offset:1280\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5])
            : "v"(addr)
            : "memory");
    } else {
        __asm__ volatile(
            "ds_read_b64_tr_b16 %0, %8\n\t"
            "ds_read_b64_tr_b16 %1, %8 offset:256\n\t"
            "ds_read_b64_tr_b16 %2, %8 offset:512\n\t"
            "ds_read_b64_tr_b16 %3, %8 offset:768\n\t"
            "ds_read_b64_tr_b16 %4, %8 offset:1024\n\t"
            "ds_read_b64_tr_b16 %5, %8 offset:1280\n\t"
            "ds_read_b64_tr_b16 %6, %8 offset:1536\n\t"
            "ds_read_b64_tr_b16 %7, %8 offset:1792\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]),
              "=&v"(r[7])
            : "v"(addr)
            : "memory");
    }
}

template <int KSTEPS>
__device__ __forceinline__ void tr_operands(const int8_t* src, v4i (&a)[KSTEPS])
{
    const uint32_t addr = (uint32_t)(size_t)(const __attribute__((address_space(3))) int8_t*)src;
    v2i r[2 * KSTEPS];
    static_assert(KSTEPS >= 1 && KSTEPS <= 8, "K steps");
    constexpr int N0 = KSTEPS < 4 ? KSTEPS : 4;
    tr_reads<N0>(addr, r);
    if constexpr (KSTEPS > 4) tr_reads<KSTEPS - 4>(addr + 2048, r + 8);
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) a[s] = v4i{r[2 * s].x, r[2 * s].y, r[2 * s + 1].x, r[2 * s + 1].y};
}

// A tile's incoherent-beam partials from the operands tr_operands gave this
// wave (every K slice): per lane the power of its column over the 8 * KSTEPS
// antennas of its row half, each word (two antennas' re, im) squared with
// v_dot4, antenna groups of 4 past A left out (they re-read antenna 0); the
// 64 lanes store their sums as the tile's [2 halves][32 columns] record
// (ib_tile), or add them up over each window's columns (at most 128 antennas
// x 16 samples x 2 pols x 2^15 < 2^31) and store the window's quantised output
// (ib_tile_outputs).
template <int KSTEPS>
__device__ __forceinline__ int ib_columns(const v4i (&a)[KSTEPS], int A, int lane)
{
    int v = 0;
    if (A == 16 * KSTEPS) {   // uniform: no padded rows, one dot chain
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
            for (int q = 0; q < 4; ++q) v = __builtin_amdgcn_sdot4(a[s][q], a[s][q], v, false);
    } else {
        const int h = lane >> 5;
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
            for (int q = 0; q < 4; q += 2) {
                int t = __builtin_amdgcn_sdot4(a[s][q], a[s][q], 0, false);
                t = __builtin_amdgcn_sdot4(a[s][q + 1], a[s][q + 1], t, false);
                v += 8 * (h * KSTEPS + s) + 2 * q < A ? t : 0;
            }
    }
    return v;
}

template <int KSTEPS>
__device__ __forceinline__ void ib_tile(const v4i (&a)[KSTEPS], int* ibp, int ntiles, int A, int f, int tile,
                                        int lane)
{
    const int v = ib_columns<KSTEPS>(a, A, lane);
    if (tile < ntiles) ibp[((size_t)f * ntiles + tile) * 64 + lane] = v;
}

// v plus its value in the lane that the data-parallel-primitive control names.
template <int CTRL>
__device__ __forceinline__ int add_dpp(int v)
{
    return v + __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

// `off` and `sc` are the channel's levels, read before the tile loop by scalar
// loads.  The sums over a window's 2 ts columns and both halves stay in the
// VALU (four DPP steps and two lane swaps).  With the sums through LDS and the
// levels read per tile, the block of 16 antennas, 16 channels, 2048 spectra
// and 32 beams took 8.2 us against 6.9; keeping the sums for one quantisation
// of all tiles gained nothing more.
template <int KSTEPS>
__device__ __forceinline__ void ib_tile_outputs(const v4i (&a)[KSTEPS], const IbFinishJob& ib, float off, float sc,
                                                int ntiles, int A, int F, int f, int tile, int lane)
{
    int v = ib_columns<KSTEPS>(a, A, lane);
    const auto h = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    v = add_dpp<0xB1>((int)(h[0] + h[1]));     // quad_perm [1, 0, 3, 2]
    if (ib.ts >= 2) v = add_dpp<0x4E>(v);      // quad_perm [2, 3, 0, 1]
    if (ib.ts >= 4) v = add_dpp<0x141>(v);     // row_half_mirror
    if (ib.ts >= 8) v = add_dpp<0x140>(v);     // row_mirror
    if (ib.ts >= 16) {
        const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
        v = (int)(r[0] + r[1]);
    }
    if (tile < ntiles && lane < 32 && (lane & (2 * ib.ts - 1)) == 0)
        ib.out[((long long)tile * (16 / ib.ts) + lane / (2 * ib.ts)) * F + f] =
            quantise((double)v, off, sc, ib.quant);
}

// a + b' where lanes below 32 keep a and take b' = (a of lane + 32), and
// lanes from 32 keep b and take (b of lane - 32): the halves' exchange of a
// reduce-scatter in one v_permlane32_swap per dword.  With a = value for the
// lower half and b = value for the upper half, every lane gets its own sum.
__device__ __forceinline__ long long swap32_sum(long long a, long long b)
{
    const unsigned alo = (uint32_t)(unsigned long long)a, ahi = (uint32_t)((unsigned long long)a >> 32);
    const unsigned blo = (uint32_t)(unsigned long long)b, bhi = (uint32_t)((unsigned long long)b >> 32);
    const auto lo = __builtin_amdgcn_permlane32_swap(alo, blo, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(ahi, bhi, false, false);
    // 64-bit sum as one add and one add-with-carry of the halves.
    const unsigned slo = lo[0] + lo[1];
    const unsigned shi = hi[0] + hi[1] + (slo < lo[0] ? 1u : 0u);
    return (long long)(((unsigned long long)shi << 32) | slo);
}

// Constants of the threshold quantiser's estimates: FP64 (P - offset) * inv
// with inv = RN(1 / scale), and FP32 P * inv_f + c_f with inv_f = RN(1 /
// scale), c_f = RN(-offset * inv_f).
struct QuantConst {
    double off_d, inv;
    float inv_f, c_f;
};

__device__ __forceinline__ QuantConst quant_const(float off, float sc)
{
    const float inv_f = 1.0f / sc;
    return QuantConst{(double)off, 1.0 / (double)sc, inv_f, -off * inv_f};
}

// Quantiser thresholds.  For a positive, normal, finite scale and a finite
// offset, quantise((double)P, offset, scale, mode) is a non-decreasing step
// function of the integer power P: thr[j] is the least P >= 0 that quantises
// to at least j - 128 (thr[0] = INT64_MIN, thr[256] = INT64_MAX, and
// INT64_MAX where no P < 2^62 gets there).  The kernel needs only an
// estimate e within one step of the result q: the two thresholds around e
// then settle q without a division or a branch (P >= thr[e + 129] means
// q = e + 1, P < thr[e + 128] means q = e - 1).  The estimate is
// e = trunc(clamp(y, -128, 127)) for an approximation y of the quotient Y
// that the exact quantiser rounds: whenever |y - Y| < 0.5, truncation moves
// y by less than 1 and the mode's rounding moves Y by at most 0.5 (truncation
// by less than 1, and then |y - Y| < 1 suffices), so |e - q| < 2 in either
// mode (the clamp keeps this), i.e. e is q or a neighbour.
constexpr int kThr = 257;
constexpr int kThrBytes = 2304;   // kThr int64, padded to a multiple of 256 bytes
static_assert(kThrBytes >= kThr * 8, "threshold table");

__device__ __forceinline__ bool thr_applies(float off, float sc)
{
    return isfinite(off) && sc >= 1.17549435e-38f && sc <= 3.40282347e+38f;
}

// Threshold correction of an estimate e in [-128, 127]; thr_mid = thr + 128
// (so thr_mid[e] and thr_mid[e + 1] are one ds_read2_b64).
__device__ __forceinline__ int8_t thr_settle(long long P, int e, const long long* thr_mid)
{
    const long long lo = thr_mid[e], hi = thr_mid[e + 1];
    return (int8_t)(e + (int)(P >= hi) - (int)(P < lo));
}

// FP64 estimate RN(RN((double)P - offset) * RN(1 / scale)): it rounds the
// same difference as the exact quantiser, so it is within 2^-43 of Y for
// |Y| <= 256 at any offset and scale; beyond, both saturate alike.
__device__ __forceinline__ int thr_estimate(long long P, const QuantConst& q)
{
    const double y = ((double)P - q.off_d) * q.inv;
    return (int)fmin(fmax(y, -128.0), 127.0);
}

__device__ __forceinline__ int8_t quantise_thr(long long P, const QuantConst& q, const long long* thr_mid)
{
    return thr_settle(P, thr_estimate(P, q), thr_mid);
}

// FP32 estimate (about a third of the VALU time of the FP64 one).  For
// P >= 0, RN(RN(hi) * 2^32 + RN(lo)) is within 3 * 2^-24 of P relative;
// RN(1 / scale) and c = RN(-offset * inv) are within 2^-24 and 2^-23
// relative, and the fma rounds once, so for |Y| <= 130 the estimate is
// within 2^-24 * (4 |P / scale| + 2 |offset / scale| + 131) <=
// 2^-24 * (651 + 6 |offset / scale|) of Y: below 0.38 when
// |offset / scale| < 2^20 (thr_f32_applies); beyond |Y| = 130 both
// saturate alike.
__device__ __forceinline__ bool thr_f32_applies(float off, float sc)
{
    return fabsf(off / sc) < 1048576.0f;
}

__device__ __forceinline__ int thr_estimate_f32(long long P, const QuantConst& q)
{
    const float pf = (float)(int)(P >> 32) * 4294967296.0f + (float)(uint32_t)P;
    const float y = __builtin_fmaf(pf, q.inv_f, q.c_f);
    return (int)__builtin_amdgcn_fmed3f(y, -128.0f, 127.0f);
}

// One tile step of the transposed kernels: the RT tiles' MFMA chains and the
// detection of their values into the pass accumulators pw[RT / 2][NSLOT]
// (tile r adds to beam group r / 2; values of window q of the tile go to
// slot g * SPT + q), one v_mad_i64_i32 per value.  (Splitting the
// dependent chains into independent partial sums measured 0.7 % slower:
// the other waves of the SIMD already cover their latency.)
template <int RT, int KSTEPS, int SPT, int NSLOT>
__device__ __forceinline__ void detect_step(const v4i (&a)[KSTEPS], const v4i (&w)[RT][KSTEPS],
                                            long long (&pw)[RT / 2][NSLOT], int g)
{
    constexpr int n = 16 / SPT;   // values per window per tile
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        v16i acc = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[s], w[r][s], acc, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < SPT; ++q)
#pragma unroll
            for (int i = 0; i < n; ++i) pw[r >> 1][g * SPT + q] += (long long)acc[q * n + i] * acc[q * n + i];
    }
}

// Four-wave work-groups per compute unit (waves per SIMD): two with 128 beams
// per wave or more than four K steps (256 VGPRs a wave), else three.
constexpr int tr_wgs(int rt, int ksteps) { return rt == 8 || ksteps > 4 ? 2 : 3; }

// Tile sets in the staging ring for ni 1 KiB loads a set: within 60 KiB; in a
// four-wave work-group less the dummy run and, with fscrunch, the 8 KiB of
// its reduction (48 KiB keep whole sets of 16), and within 48 KiB where three
// share a compute unit.
constexpr int tr_nb(int rt, int ksteps, int ni, int fs, int nw)
{
    const int kib = nw > 4 ? 60 : (fs > 1 || tr_wgs(rt, ksteps) > 2 ? 48 : 60) - (ni % nw ? nw : 0);
    const int n = kib / ni;
    return n < 2 ? 2 : (n > 8 ? 8 : n);
}

// Totals per lane that one round of the fscrunch reduction passes through
// LDS: as many as leave a four-wave work-group's ring its 48 KiB.
constexpr int tr_red_vals(int vals) { return vals < 4 ? vals : 4; }

// Staging constants of cb_tr_k for NTS time slots x FS channels x KSTEPS
// 32-byte K steps and NWB beam groups.
template <int RT, int FS, int KSTEPS, int NTS, int NWB>
struct TrStage {
    static constexpr int NW = NTS * NWB * FS;              // waves per work-group
    static constexpr int NI = NTS * FS * KSTEPS;           // 1 KiB loads per set
    static constexpr int M = (NI + NW - 1) / NW;           // per wave (the rest load into a dummy run)
    static constexpr int SET = NI * 1024;                  // bytes per set
    static constexpr int NB = tr_nb(RT, KSTEPS, NI, FS, NW);
    static constexpr int G = NB >= 4 ? 2 : 1;             // steps per barrier
    static constexpr int WAIT = (NB - 2 * G) * M;
    static constexpr int DUMMY = (NI % NW) ? NW * 1024 : 0;
};

template <int RT, int NSLOT>
struct TrRed {
    // totals per lane after the reduce-scatter
    static constexpr int VALS = RT == 2 ? NSLOT / 2 : (RT / 4) * NSLOT;
};

// Forms of at most 64 beams per wave in four-wave work-groups.
constexpr bool tr_writes_tbtf(int rt, int fs, int nw) { return rt <= 4 && fs == 1 && nw == 4; }

// RT: beam tiles per wave (RT / 2 groups of 32 beams, a Re and an Im tile
// each); SPT: windows per tile (1, 2, 4); NSLOT: windows
// per pass held in registers; FS: fscrunch; NTS: time slots and NWB: beam
// groups (of 16 RT beams) per work-group;
// DT: the outputs go straight to TBTF (CbTrArgs::tbtf; an instance of its own:
// as a branch it cost the 128-antenna kernel 5 %);
// TA: the voltages are a TAFTP block (CbArgs::S > 0), staged straight into
// [antenna][column] tiles and read with transposed LDS loads (tr_operands),
// else FTPA columns; IBF (with TA, FS = 1, all antennas of the block): the
// work-groups of beam group 0 also leave the incoherent beam's per-sample
// partials (CbTrArgs::ibp) from the same operands.
//
// A work-group has NTS x NWB x FS waves: NTS time slots (contiguous runs of
// passes of the same channel group and beams) of NWB beam groups x FS
// channels.  With 64 beams per wave a work-group holds every wave of its
// compute unit (4 NTS = 12 or 16), so the per-step
// barrier keeps them in lockstep: waves of separate work-groups sharing a
// SIMD progress at different rates (the issue arbiter prefers older waves),
// which leaves SIMDs with one wave at the end.  With 128 beams per wave
// (two waves per SIMD) a work-group is four waves, two share a compute
// unit, and they take turns at a raised wave priority instead.
template <int RT, int KSTEPS, int SPT, int NSLOT, int FS, int NTS, int NWB, bool TA, bool IBF, bool DT>
__global__ __launch_bounds__(64 * NTS * NWB * FS, NTS * NWB * FS == 4 ? tr_wgs(RT, KSTEPS) : 1) void cb_tr_k(CbTrArgs ta)
{
    using St = TrStage<RT, FS, KSTEPS, NTS, NWB>;
    constexpr int KPAD = 32 * KSTEPS;
    constexpr int VALS = TrRed<RT, NSLOT>::VALS;
    constexpr int NB = St::NB;
    constexpr int NG = RT / 2;                     // groups of 32 beams per wave
    static_assert(RT == 2 || RT == 4 || RT == 8, "RT");
    static_assert(NSLOT % SPT == 0 && (RT != 2 || NSLOT % 2 == 0), "slots");
    static_assert(St::M <= 4 && St::WAIT >= 0, "staging loads per wave per set");
    constexpr int RV = tr_red_vals(VALS);          // totals per round of the fscrunch reduction
    // Waves of a beam group share its totals out: value v goes to the wave of
    // channel v % FS.
    constexpr bool SHARE = FS > 1 && RV % FS == 0;
    constexpr int NV = SHARE ? VALS / FS : VALS;   // values a wave quantises
    static_assert(!IBF || (TA && FS == 1), "incoherent-beam partials");
    static_assert(!DT || tr_writes_tbtf(RT, FS, St::NW), "direct outputs");
    extern __shared__ __align__(16) int8_t lds[];
    const CbArgs& p = ta.p;
    int wjobs = 0;
    if constexpr (DT) {
        if (weights_job_run(ta.weights, threadIdx.x)) return;   // uniform over the work-group
        wjobs = ta.weights.nblocks;
    }

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    const int h = lane >> 5;
    const int c = lane & 31;
    constexpr int WPS = NWB * FS;                 // waves per time slot
    constexpr int NTHR = 64 * St::NW;
    const int tsl = wv / WPS;                     // time slot
    const int wc = (wv - tsl * WPS) % FS;         // channel of the fscrunch group
    const int wb = (wv - tsl * WPS) / FS;         // beam group within the work-group

    const int logical = xcd_remap((int)blockIdx.x - wjobs, (int)gridDim.x - wjobs);
    const int bgroup = logical % ta.n_bgroups;
    const int rest = logical / ta.n_bgroups;
    const int tgroup = rest % ta.n_tgroups;
    const int fo = rest / ta.n_tgroups;
    if (fo >= p.Fo) return;   // uniform over the work-group

    const int K = 2 * p.A;
    const int f = fo * FS + wc;
    const int beam_base = (bgroup * NWB + wb) * 16 * RT;
    const size_t TP = (size_t)2 * p.nsamples;
    const int slot_tiles = ta.npasses * ta.ntp;
    const int tile0 = (tgroup * NTS + tsl) * slot_tiles;

    // Start-up loads first, all in flight together: the channel's quantiser
    // thresholds (to LDS below), the weights, then the first staged tiles.
    // One threshold per thread, two for the first threads of a four-wave
    // work-group (256 threads, kThr = 257).
    static_assert(2 * NTHR >= kThr, "at most two thresholds per thread");
    const long long thr_v = tid < kThr ? p.thr[(size_t)fo * kThr + tid] : 0;
    const long long thr_v2 = tid + NTHR < kThr ? p.thr[(size_t)fo * kThr + tid + NTHR] : 0;

    // Weights (B operand).  Tile r holds the Re (r even) or Im (r odd)
    // embedding rows of the 32 beams beam_base + 32 (r / 2) + n, n = lane %
    // 32, so a lane's Re and Im outputs belong to one beam and its power
    // sums in-lane.
    v4i w[RT][KSTEPS];
    auto load_weights = [&](int g, auto al16) {
        const int b = beam_base + 32 * g + c;
        const bool bvalid = b < p.B;
        const int8_t* wcol = p.fba + ((size_t)f * p.B + (bvalid ? b : p.B - 1)) * K;
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
            w[2 * g][s] = load_wslice<decltype(al16)::value>(wcol, 16 * (h * KSTEPS + s), K, bvalid);
    };
    // Antennas a multiple of 4 only: rows of 8-byte alignment.  One uniform
    // branch around all groups' loads: with one for each group they waited for
    // one another, 0.7 to 1.2 us of a launch.  (The larger work-groups have 128
    // VGPRs a wave and spill two of them that way.)
    if constexpr (St::NW == 4) {
        if (K & 15) {
#pragma unroll
            for (int g = 0; g < NG; ++g) load_weights(g, std::false_type{});
        } else {
#pragma unroll
            for (int g = 0; g < NG; ++g) load_weights(g, std::true_type{});
        }
    } else {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (K & 15)
                load_weights(g, std::false_type{});
            else
                load_weights(g, std::true_type{});
        }
    }

    // Staging.  A wave's 16-byte load lands at LDS offset 16 * lane of a
    // 1 KiB run.  FTPA: staged_load says which 16 bytes that is; where it
    // starts early, the operand is moved down (`tail_s`).  TAFTP: a tile is
    // 16 * KSTEPS antenna rows of 64 bytes (its 32 columns, contiguous in
    // TAFTP), and a load fills 16 rows, 4 lanes a row; rows past A re-read
    // antenna 0.
    // LDS: the channel's thresholds first (at address 0, so that a
    // threshold read takes the table's offset as its immediate), then the
    // ring, the dummy run and the fscrunch reduction.
    long long* thr = reinterpret_cast<long long*>(lds);                   // [kThr] of channel fo
    int8_t* const ring = lds + kThrBytes;
    int8_t* dummy = ring + NB * St::SET;
    long long* red = reinterpret_cast<long long*>(dummy + St::DUMMY);   // [waves][RV][64]
    // A set holds one tile per (time slot, channel): tile index
    // tsl * FS + ch.  Load m of this wave fills 1 KiB of tile ti = u / KSTEPS
    // (u = wave + NW * m, the same tile for the whole wave): the channel's
    // base is wave-uniform (scalar), and each lane adds its column and
    // swizzled K piece as a 32-bit offset.
    const int8_t* cbase[St::M];
    uint32_t goff[St::M];
    uint32_t early[St::M];
    int gtile[St::M];
    int ldst[St::M];
#pragma unroll
    for (int m = 0; m < St::M; ++m) {
        const int u = wv + St::NW * m;
        early[m] = 0;
        if (u < St::NI) {
            const int ti = u / KSTEPS;
            if constexpr (TA) {
                const int kp = u - ti * KSTEPS;
                int an = 16 * kp + (lane >> 2);
                if (an >= p.A) an = 0;
                cbase[m] = p.ftpa + (size_t)(fo * FS + ti % FS) * p.S * 4;
                goff[m] = (uint32_t)(p.a0 + an) * (uint32_t)(p.F * p.S * 4) + 16 * (lane & 3);
            } else {
                const StagedLoad ld = staged_load((u - ti * KSTEPS) * 1024 + lane * 16, KPAD, K, p.vstride);
                cbase[m] = p.ftpa + (size_t)(fo * FS + ti % FS) * TP * p.vstride + p.voff;
                goff[m] = (uint32_t)ld.offset;
                early[m] = fo * FS + ti % FS == p.F - 1 ? ld.early : 0;
            }
            gtile[m] = (tgroup * NTS + ti / FS) * slot_tiles;
            ldst[m] = u * 1024;
        } else {
            cbase[m] = TA ? p.ftpa : p.ftpa + (size_t)(fo * FS) * TP * p.vstride + p.voff;
            goff[m] = 0;
            gtile[m] = 0;
            ldst[m] = -1;
        }
    }
    const size_t tile_stride = (size_t)32 * p.vstride;
    const int tmask = (1 << ta.lgtph) - 1;
    // TAFTP: each load keeps a running 32-bit offset of its next tile (the
    // block is below 4 GiB, fbf_cb_beamform_taftp's condition), since the
    // issues take consecutive tiles: 64 bytes on within a heap, the next
    // heap's first tile at a heap boundary; loads past the last tile keep
    // re-reading it.  A handful of scalar instructions per load instead of a
    // 64-bit tile address (every wave of a compute unit shares one scalar
    // unit, and the loads are issued right after a barrier).
    uint32_t toff_run[St::M];
    int tile_run[St::M];
    if constexpr (TA) {
#pragma unroll
        for (int m = 0; m < St::M; ++m) {
            const int t = gtile[m] < ta.ntiles ? gtile[m] : ta.ntiles - 1;
            tile_run[m] = gtile[m];
            toff_run[m] = (uint32_t)(t >> ta.lgtph) * (uint32_t)ta.hstride + ((uint32_t)(t & tmask) << 6);
            cbase[m] = uniform_ptr(cbase[m]);
        }
    }
    const uint32_t heap_jump = (uint32_t)ta.hstride - (uint32_t)tmask * 64u;
    auto issue = [&](int q, int slot) {
        int8_t* set = ring + slot * St::SET;
#pragma unroll
        for (int m = 0; m < St::M; ++m) {
            int8_t* dst = ldst[m] >= 0 ? set + ldst[m] : dummy + wv * 1024;
            if constexpr (TA) {
                dma16(cbase[m] + toff_run[m] + goff[m], dst);
                ++tile_run[m];
                if (tile_run[m] < ta.ntiles) toff_run[m] += (tile_run[m] & tmask) ? 64u : heap_jump;
            } else {
                const int tt = gtile[m] + q < ta.ntiles - 1 ? gtile[m] + q : ta.ntiles - 1;
                const uint32_t off = tt == ta.ntiles - 1 ? goff[m] - early[m] : goff[m];
                dma16(uniform_ptr(cbase[m] + (size_t)tt * tile_stride) + off, dst);
            }
        }
    };
    // Physical offsets of this lane's K pieces in its column (FTPA), or of
    // the row piece this lane reads for K slice s (TAFTP, tr_operands): rows
    // 8 (h KSTEPS + s) + (lane / 4) % 4, columns 16 ((lane / 16) % 2) +
    // 4 (lane % 4), so lane c + 32 h gets the antennas of K piece
    // h KSTEPS + s, as FTPA's column holds them.
    int aoff[KSTEPS];
    if constexpr (TA) {
        const int rr = (lane >> 2) & 3, xx = lane & 3, gh = (lane >> 4) & 1;
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
            aoff[s] = (tsl * FS + wc) * KSTEPS * 1024 + (8 * (h * KSTEPS + s) + rr) * 64 + 32 * gh + 8 * xx;
    } else {
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
            aoff[s] = (tsl * FS + wc) * 32 * KPAD + staged_piece(c, h * KSTEPS + s, KPAD);
    }

    // The block's last tile (FTPA, K % 16 == 8) and the slice of this lane's
    // operands that was loaded 8 bytes early there.
    const int tail_tile = !TA && (K & 15) && f == p.F - 1 ? ta.ntiles - 1 : -1;
    const int tail_s = c == 31 ? staged_tail_piece(K) - h * KSTEPS : -1;

    const bool wave_active = beam_base < p.B;
#pragma unroll
    for (int q = 0; q < NB - St::G; ++q) issue(q, q);
    int step = 0;
    int rs = 0;              // ring slot read this step
    int is = NB - St::G;     // next ring slot to fill

    bool m128 = false;
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
            m128 |= raw_has_m128(w[2 * g][s]);
            w[2 * g + 1][s] = embed_slice(w[2 * g][s], true);
            w[2 * g][s] = embed_slice(w[2 * g][s], false);
        }
    // A work-group any of whose waves holds a weight wi = -128 computes its
    // outputs on the exact path instead.  The flags pass through the
    // thresholds' LDS before the thresholds are written there: written, a
    // barrier, read by every wave, a barrier.
    {
        int* const flags = reinterpret_cast<int*>(thr);
        const bool wave_m128 = wave_any(m128);   // every lane votes (not inside the lane-0 branch)
        if (lane == 0) flags[wv] = wave_m128 ? 1 : 0;
        wait_vm_lgkm0<63>();
        block_barrier();
        int any = 0;
#pragma unroll
        for (int i = 0; i < St::NW; ++i) any |= flags[i];
        any = __builtin_amdgcn_readfirstlane(any);
        wait_vm_lgkm0<63>();
        block_barrier();
        if (any) {
            wait_vm_lgkm0<0>();   // the staging loads land before LDS is released
            const int tend = (tgroup + 1) * NTS * slot_tiles;
            if constexpr (DT) {
                CbArgs pt = p;
                pt.out = ta.tbtf;
                cb_exact_outputs<MODE_INT8, true>(pt, fo, bgroup * NWB * 16 * RT, NWB * 16 * RT,
                                                  (long long)tgroup * NTS * slot_tiles * SPT / ta.tps,
                                                  (long long)(tend < ta.ntiles ? tend : ta.ntiles) * SPT / ta.tps, tid,
                                                  (int)blockDim.x);
            } else {
                cb_exact_outputs<MODE_INT8>(p, fo, bgroup * NWB * 16 * RT, NWB * 16 * RT,
                                            (long long)tgroup * NTS * slot_tiles * SPT / ta.tps,
                                            (long long)(tend < ta.ntiles ? tend : ta.ntiles) * SPT / ta.tps, tid,
                                            (int)blockDim.x);
            }
            if constexpr (IBF) {
                if (DT && bgroup == 0 && ta.ib.out)
                    cb_exact_ib_outputs(p, ta.ib, fo, tgroup * NTS * slot_tiles, tend < ta.ntiles ? tend : ta.ntiles,
                                        tid, (int)blockDim.x);
                else if (bgroup == 0)
                    cb_exact_ib_partials(p, ta.ibp, ta.ntiles, fo, tgroup * NTS * slot_tiles,
                                         tend < ta.ntiles ? tend : ta.ntiles, tid, (int)blockDim.x);
            }
            return;
        }
    }

    // Quantiser: the thresholds are visible after the tile loop's first
    // barrier.
    const float q_off = p.offsets[fo], q_sc = p.scales[fo];
    const bool q_thr = thr_applies(q_off, q_sc);
    const bool q_f32 = q_thr && thr_f32_applies(q_off, q_sc);
    const QuantConst qz = quant_const(q_off, q_sc);
    const bool ib_out = DT && IBF && ta.ib.out;   // the incoherent beam's outputs are written here
    typedef const __attribute__((address_space(4))) float* scalar_ptr;
    const float ib_off = ib_out ? ((scalar_ptr)ta.ib.offsets)[fo] : 0.0f;
    const float ib_sc = ib_out ? ((scalar_ptr)ta.ib.scales)[fo] : 1.0f;
    if (tid < kThr) thr[tid] = thr_v;
    if (tid + NTHR < kThr) thr[tid + NTHR] = thr_v2;
    const long long* const thr_mid = thr + 128;
    // Quantise and store one pass's totals (staged [fo][to][b] int8); with
    // FS > 1 the waves of a beam group share the totals out.
    // Value v of a lane: slot 2v + h of beam c (RT = 2), else slot
    // v % NSLOT of beam 64 (v / NSLOT) + 32 h + c.  The row of slot 2v
    // (RT = 2) or v % NSLOT is wave-uniform, so its address is scalar and
    // each lane adds a 32-bit offset (the next row for the upper half when
    // RT = 2).
    int8_t* const out_f = static_cast<int8_t*>(p.out) + (size_t)fo * p.nsamples_out * p.B;
    const int b_lane = RT == 2 ? beam_base + c : beam_base + 32 * h + c;
    const int lane_off = (RT == 2 ? h * p.B : 0) + b_lane;
    // Output windows number below 2^31 (cb_tr_applies), so window indices
    // compare as int: a scalar compare for the wave-uniform rows.
    const int nout = (int)p.nsamples_out;
    const bool all_beams = wave_active && beam_base + 16 * RT <= p.B;
    // All of a pass's values are estimated first, then their thresholds
    // read (the LDS reads in flight together, one wait), then stored.
    auto store_pass = [&](const long long (&t)[NV], int w0) {
        int q[NV];   // (ints: no packing into dwords before the byte stores)
        if (q_thr) {
            int e[NV];
            if (q_f32) {
#pragma unroll
                for (int v = 0; v < NV; ++v) e[v] = thr_estimate_f32(t[v], qz);
            } else {
#pragma unroll
                for (int v = 0; v < NV; ++v) e[v] = thr_estimate(t[v], qz);
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) q[v] = thr_settle(t[v], e[v], thr_mid);
        } else {
#pragma unroll
            for (int v = 0; v < NV; ++v) q[v] = quantise((double)t[v], q_off, q_sc, p.quant);
        }
        if constexpr (DT) {   // [To/ohs][B][ohs][Fo], below 2^31 bytes
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int row = w0 + (RT == 2 ? 2 * v + h : v % NSLOT);
                const int b = b_lane + (RT == 2 ? 0 : 64 * (v / NSLOT));
                if (!wave_active || row >= nout || b >= p.B) continue;
                const unsigned heap = (unsigned)row / (unsigned)p.ohs;
                const unsigned in_heap = (unsigned)row - heap * p.ohs;
                global_ptr(ta.tbtf)[((heap * p.B + b) * p.ohs + in_heap) * p.Fo + fo] = (int8_t)q[v];
            }
            return;
        }
        // Every beam of the wave and every window of the pass in range (the
        // usual case, uniform over the wave): the four rows' bases are
        // scalar and the stores need no per-store checks.
        if constexpr (RT != 2 && FS == 1) {
            if (all_beams && w0 + NSLOT <= nout) {
                int8_t* const base = out_f + (size_t)w0 * p.B;
#pragma unroll
                for (int v = 0; v < NV; ++v)
                    global_ptr(uniform_ptr(base + (size_t)(v % NSLOT) * p.B + 64 * (v / NSLOT)))[(unsigned)lane_off] =
                        q[v];
                return;
            }
        }
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int v = SHARE ? k * FS + wc : k;
            if (FS > 1 && !SHARE && v % FS != wc) continue;
            const int row = w0 + (RT == 2 ? 2 * v : v % NSLOT);
            const int bsh = RT == 2 ? 0 : 64 * (v / NSLOT);
            // Uniform bounds first (a scalar branch), then the lane's.
            if (!wave_active || row >= nout) continue;
            if (b_lane + bsh < p.B && (RT != 2 || row + h < nout))
                global_ptr(uniform_ptr(out_f + (size_t)row * p.B + bsh))[(unsigned)lane_off] = q[k];
        }
    };
    const int prio_phase = blockIdx.x >= gridDim.x / 2 ? 1 : 0;
    // First window of the pass; tile0 is a multiple of the slot's tiles, so
    // the division is exact.
    int w0_pass = tile0 * SPT / ta.tps;
    for (int pass = 0; pass < ta.npasses; ++pass) {
        long long pw[NG][NSLOT];
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int sl = 0; sl < NSLOT; ++sl) pw[g][sl] = 0;
        // Passes past the end of the channel (the last slots of a one-round
        // grid) still take part in the staging and the barriers but leave
        // the MFMA pipe to the other waves of the SIMD.
        const bool tiles_live = tile0 + pass * ta.ntp < ta.ntiles;
        const bool live = wave_active && tiles_live;
        // Incoherent-beam partials: in beam group 0, one wave of each time
        // slot per step (whether it holds beams or not) forms the tile's.
        // The role rotates with the step (and, with two time slots, the
        // slot), so that a wave issues one partials store per four steps
        // (stores count against the staging loads' vmcnt wait) and the
        // SIMDs take turns.
        const bool ib_live = IBF && bgroup == 0 && tiles_live;

        // Tiles of the pass: NSLOT/SPT groups of tps tiles (tps = 1 unless
        // a window spans several tiles).
#pragma unroll
        for (int g = 0; g < NSLOT / SPT; ++g) {
            for (int x = 0; x < ta.tps; ++x) {
                // Every G steps: this wave's loads of the next G sets are
                // done once WAIT later loads remain; the barrier makes every
                // wave's loads visible and frees the G slots read since the
                // last barrier, which are refilled NB - G steps ahead.
                // Four-wave work-groups (two per compute unit, one wave each
                // per SIMD): the issue arbiter favours the older wave of a
                // SIMD, so the two work-groups take turns at a raised
                // priority, every 16 steps in opposite phase (the halves of
                // the grid), instead of the older one finishing first and
                // leaving its SIMDs one wave for the rest.
                if constexpr (St::NW == 4) {
                    if (step % 16 == 0) {
                        if (((step >> 4) + prio_phase) & 1) __builtin_amdgcn_s_setprio(2);
                        else __builtin_amdgcn_s_setprio(0);
                    }
                }
                if (step % St::G == 0) {
                    wait_vm_lgkm0<St::WAIT>();
                    block_barrier();
#pragma unroll
                    for (int j = 0; j < St::G; ++j) {
                        issue(step + NB - St::G + j, is);
                        is = is + 1 == NB ? 0 : is + 1;
                    }
                }
                const bool ib_now = ib_live && (step + 2 * tsl) % WPS == wv - tsl * WPS;
                if (live || ib_now) {
                    const int8_t* src = ring + rs * St::SET;
                    v4i a[KSTEPS];
                    if constexpr (TA) {
                        tr_operands<KSTEPS>(src + aoff[0], a);
                    } else {
#pragma unroll
                        for (int s = 0; s < KSTEPS; ++s) a[s] = *reinterpret_cast<const v4i*>(src + aoff[s]);
                        if (tile0 + pass * ta.ntp + g * ta.tps + x == tail_tile) {
#pragma unroll
                            for (int s = 0; s < KSTEPS; ++s)
                                if (s == tail_s) a[s] = v4i{a[s].z, a[s].w, a[s].z, a[s].w};
                        }
                    }
                    if (live) detect_step<RT, KSTEPS, SPT, NSLOT>(a, w, pw, g);
                    if constexpr (IBF) {
                        const int tile = tile0 + pass * ta.ntp + g * ta.tps + x;
                        if (ib_out) {
                            if (ib_now)
                                ib_tile_outputs<KSTEPS>(a, ta.ib, ib_off, ib_sc, ta.ntiles, p.A, p.F, fo, tile, lane);
                        } else if (ib_now) {
                            ib_tile<KSTEPS>(a, ta.ibp, ta.ntiles, p.A, fo, tile, lane);
                        }
                    }
                }
                rs = rs + 1 == NB ? 0 : rs + 1;
                ++step;
            }
        }

        // A window's power is split over the row halves (lane and lane ^ 32):
        // one v_permlane32_swap reduce-scatter per value, lanes below 32
        // keeping the even beam group of each pair (RT >= 4) or the even
        // slots (RT = 2).
        long long tot[VALS];
        if constexpr (RT == 2) {
#pragma unroll
            for (int v = 0; v < VALS; ++v) tot[v] = swap32_sum(pw[0][2 * v], pw[0][2 * v + 1]);
        } else {
#pragma unroll
            for (int gp = 0; gp < NG / 2; ++gp)
#pragma unroll
                for (int sl = 0; sl < NSLOT; ++sl)
                    tot[gp * NSLOT + sl] = swap32_sum(pw[2 * gp][sl], pw[2 * gp + 1][sl]);
        }

        // Sum over the fscrunch channels (one per wave of a beam group), RV
        // totals at a time through LDS; each wave of the group reads back
        // the sums of the values it quantises.
        if constexpr (FS > 1) {
            long long sum[NV];
#pragma unroll
            for (int r = 0; r < VALS; r += RV) {
#pragma unroll
                for (int v = 0; v < RV; ++v) red[(wv * RV + v) * 64 + lane] = tot[r + v];
                wait_vm_lgkm0<63>();
                block_barrier();
#pragma unroll
                for (int k = 0; k < (SHARE ? RV / FS : RV); ++k) {
                    const int v = SHARE ? k * FS + wc : k;
                    long long t = 0;
#pragma unroll
                    for (int ch = 0; ch < FS; ++ch) t += red[((tsl * WPS + wb * FS + ch) * RV + v) * 64 + lane];
                    sum[SHARE ? r / FS + k : r + k] = t;
                }
                wait_vm_lgkm0<63>();
                block_barrier();
            }
            store_pass(sum, w0_pass);
        } else {
            store_pass(tot, w0_pass);
        }
        w0_pass += NSLOT;   // a pass holds NSLOT windows (ta.ntp = NSLOT / SPT * tps tiles)
    }
    // The loads past the last tile are still in flight: LDS must not be
    // released before they land.
    wait_vm_lgkm0<0>();
}

// Launch of cb_tr_k.  Supports 4 | A <= 128, tscrunch a power of two >= 4
// (window 8, 16, 32 or a multiple of 32 columns), fscrunch 1, 2 or 4 (with
// work-groups of several time slots fscrunch * ceil(A / 16) <= 8), int8
// output.
// Windows per pass.  With 64 beams per wave and windows of 16 or more
// columns, two windows per pass keep a wave within 128 VGPRs, so four waves
// share a SIMD (tr_nts).  Windows of 8 columns fill a tile four times, so a
// pass holds at least 4.
inline int cb_tr_nslot(int rt, int W)
{
    if (W == 16 && rt == 4) return 2;
    if (W <= 16) return rt == 2 ? 8 : 4;
    return W == 32 && rt != 4 ? 4 : 2;
}

// Whether a form of the transposed kernel has four-wave work-groups, two per
// compute unit: 128 beams per wave (256 VGPRs, two waves per SIMD), and 64
// beams per wave over more than four K steps (65 to 128 antennas), which
// holds as many weights (up to 128 VGPRs; the wave stays within 256).  With
// 128 beams per wave, one work-group of two time slots kept its two waves of a
// SIMD in lockstep, and the older one waited at every barrier for the
// younger; two work-groups with alternating priority measured 2.0-2.4 %
// faster.  At 128 antennas, 1024 beams, 64 channels, 8192 samples the one-pass
// block took 494 us with 64 beams per wave against 643 us with 32 in
// three-slot work-groups from a split-transposed copy.
//
// The other forms have one work-group per compute unit: four time slots with
// 64 beams per wave and two windows per pass (at most 128 VGPRs a wave, four
// waves per SIMD), else three.  With four waves a SIMD overlaps one wave's
// MFMAs with the others' detection better: at 64 antennas the VALU work per
// step outweighs the MFMA work.
constexpr bool tr_four_waves(int rt, int ksteps) { return rt == 8 || (rt == 4 && ksteps > 4); }

// Fewest beam groups per four-wave work-group: over more than four K steps the
// ring holds two time slots at most.
constexpr int tr_nwb_min(int ksteps) { return ksteps > 4 ? 2 : 1; }

// Time slots per work-group.
constexpr int tr_nts(int rt, int ksteps, int nslot, int fs, int nwb)
{
    return tr_four_waves(rt, ksteps) ? 4 / (fs * nwb) : (rt == 4 && nslot == 2 ? 4 : 3);
}

inline size_t cb_tr_shm(int rt, int fs, int ksteps, int vals, int nts, int nwb)
{
    const int nw = nts * nwb * fs;
    const int ni = nts * fs * ksteps;
    return (size_t)tr_nb(rt, ksteps, ni, fs, nw) * ni * 1024 + ((ni % nw) ? (size_t)nw * 1024 : 0) +
           (fs > 1 ? (size_t)nw * tr_red_vals(vals) * 64 * sizeof(long long) : 0) + kThrBytes;
}

inline bool cb_tr_supported(int A, int ts, int fs, int rt)
{
    if (A % 4 != 0 || A > 128) return false;
    if (ts < 4 || (ts & (ts - 1)) != 0) return false;
    if (!(fs == 1 || fs == 2 || fs == 4)) return false;
    const int ksteps = (2 * A + 31) / 32;
    if (rt == 8 ? ksteps > 4 : rt * ksteps > 16 && (rt != 4 || fs > 2)) return false;
    if (tr_four_waves(rt, ksteps)) return true;   // their rings are sized to fit
    if (fs * ksteps > 8) return false;
    const int nslot = cb_tr_nslot(rt, 2 * ts);
    const int vals = rt == 2 ? nslot / 2 : (rt / 4) * nslot;
    return cb_tr_shm(rt, fs, ksteps, vals, tr_nts(rt, ksteps, nslot, fs, 4 / fs), 4 / fs) <= 65536;
}

// Compute units of the current device (cached per device).
inline int device_cu_count()
{
    static int cus[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cus[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

// Work-groups per (channel group, beam group), each a contiguous run of
// passes on every time slot: `slots` resident work-groups run at a time.  The
// fewest tile steps in a row over the rounds, where a work-group's start-up
// (weights, the first staged tiles) is about five steps long.  That is one
// round wherever it fills the slots; 192 units on 512 slots (40 antennas, 768
// beams, 64 channels) left a quarter of them empty: 185 us in one round, 165 us
// in three (8192 samples, tscrunch 16).
struct TrRounds {
    long long per_unit;   // work-groups per (channel group, beam group)
    long long cost;       // tile steps in a row
};

inline TrRounds tr_rounds(long long units, long long slots, int passes, int nts, int ntp)
{
    constexpr int kStart = 5;
    const long long most = (passes + nts - 1) / nts;
    TrRounds best{1, 0};
    for (int round = 1; round <= 8; ++round) {   // the most work-groups of each number of rounds
        long long n = round * slots / units;
        n = n < 1 ? 1 : n > most ? most : n;
        const long long np = (passes + n * nts - 1) / (n * nts);   // passes per slot
        const long long groups = (passes + np * nts - 1) / (np * nts);
        const long long cost = (units * groups + slots - 1) / slots * (np * ntp + kStart);
        if (best.cost == 0 || cost < best.cost) best = {n, cost};
        if (n == most) break;
    }
    return best;
}

// Beam groups per four-wave work-group: 4 / fs, or fewer (and as many more
// time slots) where that takes fewer tile steps in a row (more beam groups
// would leave waves without beams).  Fewer beam groups stage each tile for
// fewer waves, so they have to win a tenth.
inline int tr_nwb(int rt, int ksteps, int fs, const CbTrArgs& a, int passes)
{
    const long long slots = (long long)tr_wgs(rt, ksteps) * device_cu_count();
    int best = 4 / fs;
    long long best_cost = 0;
    for (int n = best; n >= tr_nwb_min(ksteps); n /= 2) {
        const int beams = 16 * rt * n;
        const long long units = (long long)a.p.Fo * ((a.p.B + beams - 1) / beams);
        const long long cost = tr_rounds(units, slots, passes, 4 / (fs * n), a.ntp).cost;
        if (best_cost == 0 || 10 * cost <= 9 * best_cost) {
            best = n;
            best_cost = cost;
        }
    }
    return best;
}

template <int RT, int KSTEPS, int SPT, int NSLOT, int FS, int NTS, int NWB, bool TA, bool IBF = false, bool DT = false>
hipError_t launch_tr_kt(CbTrArgs a, int passes, hipStream_t s)
{
    if constexpr (!DT && tr_writes_tbtf(RT, FS, NTS * NWB * FS))
        if (a.tbtf) return launch_tr_kt<RT, KSTEPS, SPT, NSLOT, FS, NTS, NWB, TA, IBF, true>(a, passes, s);
    if (a.tbtf && !DT) return hipErrorInvalidValue;
    constexpr int NTHR = 64 * NTS * NWB * FS;
    constexpr auto kernel = cb_tr_k<RT, KSTEPS, SPT, NSLOT, FS, NTS, NWB, TA, IBF, DT>;
    const size_t shm = cb_tr_shm(RT, FS, KSTEPS, TrRed<RT, NSLOT>::VALS, NTS, NWB);
    if (shm > 65536) return hipErrorInvalidConfiguration;
    constexpr int beams_per_wg = 16 * RT * NWB;
    a.n_bgroups = (a.p.B + beams_per_wg - 1) / beams_per_wg;
    static int occ = 0;
    if (occ == 0) {
        int o = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&o, kernel, NTHR, shm) != hipSuccess || o < 1)
            o = 1;
        occ = o;
    }
    const long long units = (long long)a.p.Fo * a.n_bgroups;
    const long long per_unit = tr_rounds(units, (long long)occ * device_cu_count(), passes, NTS, a.ntp).per_unit;
    a.npasses = (int)((passes + per_unit * NTS - 1) / (per_unit * NTS));
    a.n_tgroups = (int)((passes + (long long)a.npasses * NTS - 1) / ((long long)a.npasses * NTS));
    const long long nblocks = units * a.n_tgroups + a.weights.nblocks;
    if (nblocks <= 0 || nblocks >= (1ll << 31)) return hipErrorInvalidConfiguration;
    kernel<<<dim3((unsigned)nblocks), NTHR, shm, s>>>(a);
    return hipGetLastError();
}

// TAFTP staging (a.p.S > 0) is built for 64 beams per wave at fscrunch 1 and
// for 128 (cb_taftp_form).  The incoherent-beam partials (a.ibp) are built
// for the four-wave work-groups at fscrunch 1 (cb_ib_fused).
template <int RT, int KSTEPS, int SPT, int NSLOT, int FS, int NWB>
hipError_t launch_tr_kn(const CbTrArgs& a, int passes, hipStream_t s)
{
    constexpr int NTS = tr_nts(RT, KSTEPS, NSLOT, FS, NWB);
    if (a.p.S > 0) {
        if constexpr (RT == 8 || (RT == 4 && FS == 1)) {
            if (a.ibp) {
                if constexpr (FS == 1 && tr_four_waves(RT, KSTEPS))
                    return launch_tr_kt<RT, KSTEPS, SPT, NSLOT, FS, NTS, NWB, true, true>(a, passes, s);
                return hipErrorInvalidValue;
            }
            return launch_tr_kt<RT, KSTEPS, SPT, NSLOT, FS, NTS, NWB, true>(a, passes, s);
        }
        return hipErrorInvalidValue;
    }
    return launch_tr_kt<RT, KSTEPS, SPT, NSLOT, FS, NTS, NWB, false>(a, passes, s);
}

template <int RT, int KSTEPS, int SPT, int NSLOT, int FS>
hipError_t launch_tr_k(const CbTrArgs& a, int passes, hipStream_t s)
{
    if constexpr (tr_four_waves(RT, KSTEPS)) {
        const int nwb = tr_nwb(RT, KSTEPS, FS, a, passes);
        if constexpr (FS <= 2 && tr_nwb_min(KSTEPS) == 1)
            if (nwb == 1) return launch_tr_kn<RT, KSTEPS, SPT, NSLOT, FS, 1>(a, passes, s);
        if constexpr (FS == 1)
            if (nwb == 2) return launch_tr_kn<RT, KSTEPS, SPT, NSLOT, FS, 2>(a, passes, s);
    }
    return launch_tr_kn<RT, KSTEPS, SPT, NSLOT, FS, 4 / FS>(a, passes, s);
}

template <int RT, int SPT, int NSLOT, int FS>
hipError_t launch_tr_ks(const CbTrArgs& a, int ksteps, int passes, hipStream_t s)
{
    if constexpr (FS * 2 <= 8) {
        if (ksteps == 1) return launch_tr_k<RT, 1, SPT, NSLOT, FS>(a, passes, s);
        if (ksteps == 2) return launch_tr_k<RT, 2, SPT, NSLOT, FS>(a, passes, s);
    }
    if constexpr (RT == 8 || FS * 4 <= 8) {
        if (ksteps == 3) return launch_tr_k<RT, 3, SPT, NSLOT, FS>(a, passes, s);
        if (ksteps == 4) return launch_tr_k<RT, 4, SPT, NSLOT, FS>(a, passes, s);
    }
    if constexpr ((FS == 1 && RT == 2) || (FS <= 2 && RT == 4)) {
        switch (ksteps) {
        case 5: return launch_tr_k<RT, 5, SPT, NSLOT, FS>(a, passes, s);
        case 6: return launch_tr_k<RT, 6, SPT, NSLOT, FS>(a, passes, s);
        case 7: return launch_tr_k<RT, 7, SPT, NSLOT, FS>(a, passes, s);
        case 8: return launch_tr_k<RT, 8, SPT, NSLOT, FS>(a, passes, s);
        default: break;
        }
    }
    return hipErrorInvalidValue;
}

template <int RT, int FS>
hipError_t launch_tr_w(const CbTrArgs& a, int W, int ksteps, int passes, hipStream_t s)
{
    // Windows per pass as cb_tr_nslot
    constexpr int small = RT == 2 ? 8 : 4;
    if (W == 8) return launch_tr_ks<RT, 4, small, FS>(a, ksteps, passes, s);
    if (W == 16) return launch_tr_ks<RT, 2, RT == 4 ? 2 : small, FS>(a, ksteps, passes, s);
    if (W == 32) return launch_tr_ks<RT, 1, RT == 4 ? 2 : 4, FS>(a, ksteps, passes, s);
    return launch_tr_ks<RT, 1, 2, FS>(a, ksteps, passes, s);
}

// Windows per pass of cb_ws_k.
inline int cb_ws_nslot(int W) { return W <= 32 ? 4 : 2; }

// cb_ws_k serves 4 | A <= 64, fscrunch 1, tscrunch a power of two >= 4.
inline bool cb_ws_supported(int A, int ts, int fs)
{
    return A % 4 == 0 && A <= 64 && fs == 1 && ts >= 4 && (ts & (ts - 1)) == 0;
}

}  // namespace
}  // namespace fbf
