// Coherent beamformer with wave-private staging (cb_ws_k).
#include "cb_tr.hpp"

namespace fbf {
namespace {

// ---------------------------------------------------------------------------
// Wave-private staging (cb_ws_k)
//
// The contraction, detection, reduce-scatter and quantiser of cb_tr_k with
// RT = 4 (a wave holds 64 beams, Re and Im tiles) and fscrunch 1, but every
// wave stages its own voltage tiles in a private LDS ring and waits for
// nothing but its own loads: no work-group barrier in the tile loop, so the
// waves of a SIMD drift apart and one wave's MFMAs overlap another wave's
// detection (the 64-bit multiply-adds take as long as the MFMAs at 64
// antennas).  Work is dealt dynamically.  A unit is (output channel, 64-beam
// group, time range); a work-group of 12 waves serves U units, the waves
// starting 12 / U to a unit; a wave takes chunks (whole passes, at least a
// ring's worth of tiles) from its unit's LDS counter and, when the unit runs
// dry, moves to the next unit of the work-group (reloading its weights), so
// the waves of a work-group end within a chunk of each other.
//
// Ring: NB tiles per wave; the tile at sequence position q sits in slot
// q % NB.  Step q waits for its own loads of tile q (a fixed s_waitcnt:
// (NB - 1) tiles issued after it), reads the tile into registers, and then
// reuses the slot for tile q + NB.  A slot is written only after the same
// wave's reads of it have completed, and the loads are issued for every
// step (past the end of the work they re-read a valid tile), so the count
// stays exact.
// ---------------------------------------------------------------------------
// Returns the old value of the LDS word at byte address addr and adds v.
// Written as one asm block that also waits for the result: the compiler
// puts a full vmcnt(0) wait before its own LDS atomics while global->LDS
// loads are in flight, which would drain a wave's staging ring at every
// chunk.
__device__ __forceinline__ int lds_fetch_add(unsigned addr, int v)
{
    int old;
    __asm__ volatile("ds_add_rtn_u32 %0, %1, %2\n\ts_waitcnt lgkmcnt(0)" : "=v"(old) : "v"(addr), "v"(v) : "memory");
    return old;
}

constexpr int kWsWaves = 12;
constexpr int kWsRingBudget = 144 * 1024;
constexpr int kWsMaxUnits = 6;

template <int KSTEPS>
struct WsStage {
    static constexpr int KPAD = 32 * KSTEPS;
    static constexpr int TILE = 32 * KPAD;                  // bytes per tile
    static constexpr int LPT = KSTEPS;                      // 1 KiB loads per tile
    static constexpr int NB0 = kWsRingBudget / (kWsWaves * TILE);
    static constexpr int NB = NB0 < 2 ? 2 : (NB0 > 8 ? 8 : NB0);
    static constexpr int WAIT = (NB - 1) * LPT;
};

// AL16: K = 2A is a multiple of 16 (else of 8: antennas in fours).
template <int KSTEPS, int SPT, int NSLOT, bool AL16>
__global__ __launch_bounds__(64 * kWsWaves) void cb_ws_k(CbWsArgs wa)
{
    using St = WsStage<KSTEPS>;
    constexpr int KPAD = St::KPAD;
    constexpr int NB = St::NB;
    constexpr int RT = 4, NG = 2;
    static_assert(NSLOT % SPT == 0, "slots");
    static_assert(St::WAIT <= 63, "vmcnt");
    extern __shared__ __align__(16) int8_t lds[];
    const CbArgs& p = wa.p;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5;
    const int c = lane & 31;
    const int U = wa.U;
    const int unit0 = xcd_remap(blockIdx.x, gridDim.x) * U;
    int8_t* const ring = lds + wv * NB * St::TILE;
    long long* const thr_all = reinterpret_cast<long long*>(lds + kWsWaves * NB * St::TILE);   // [U][kThr]
    int* const counter = reinterpret_cast<int*>(thr_all + U * kThr);                          // [U]
    int* const m128_flags = counter + U;                                                      // [kWsWaves]

    // Units: id = ((fo * ntr + tr) * nbg + bg).
    auto unit_fo = [&](int gu) { return gu / (wa.ntr * wa.nbg); };
    for (int i = tid; i < U * kThr; i += 64 * kWsWaves) {
        const int gu = unit0 + i / kThr;
        thr_all[i] = gu < wa.nunits ? p.thr[(size_t)unit_fo(gu) * kThr + i % kThr] : 0;
    }
    if (tid < U) counter[tid] = 0;
    // Weights of every unit of the work-group: one holding a wi = -128 sends
    // the work-group to the exact path (before any staging load is issued).
    const int K = 2 * p.A;
    {
        const int kp = (K + 15) / 16;
        const int per_unit = 64 * kp;
        bool m128 = false;
        for (int i = tid; i < U * per_unit; i += 64 * kWsWaves) {
            const int gu = unit0 + i / per_unit;
            const int r = i % per_unit;
            const int b = (gu % wa.nbg) * 64 + r / kp;
            if (gu < wa.nunits && b < p.B)
                m128 |= raw_has_m128(load_wslice<AL16>(p.fba + ((size_t)unit_fo(gu) * p.B + b) * K, 16 * (r % kp), K,
                                                        true));
        }
        const bool wave_m128 = wave_any(m128);   // every lane votes (not inside the lane-0 branch)
        if (lane == 0) m128_flags[wv] = wave_m128 ? 1 : 0;
    }
    __syncthreads();
    {
        int any = 0;
#pragma unroll
        for (int i = 0; i < kWsWaves; ++i) any |= m128_flags[i];
        if (__builtin_amdgcn_readfirstlane(any)) {
            for (int u = 0; u < U; ++u) {
                const int gu = unit0 + u;
                if (gu >= wa.nunits) break;
                const int tr = (gu / wa.nbg) % wa.ntr;
                const long long t0 = (long long)tr * wa.tr_chunks * wa.ct;
                long long t1 = t0 + (long long)wa.tr_chunks * wa.ct;
                if (t1 > wa.ntiles) t1 = wa.ntiles;
                cb_exact_outputs<MODE_INT8>(p, unit_fo(gu), (gu % wa.nbg) * 64, 64, t0 * SPT / wa.tps,
                                            t1 * SPT / wa.tps, tid, (int)blockDim.x);
            }
            return;
        }
    }

    const size_t TP = (size_t)2 * p.nsamples;
    const int chunk_tiles = wa.ct;

    // This lane's part of a tile load m (staged_load), and the offsets of its K
    // pieces.
    int goff[St::LPT];
    int early[St::LPT];
#pragma unroll
    for (int m = 0; m < St::LPT; ++m) {
        const StagedLoad ld = staged_load(m * 1024 + lane * 16, KPAD, K, p.vstride);
        goff[m] = ld.offset;
        early[m] = ld.early;
    }
    int aoff[KSTEPS];
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) aoff[s] = staged_piece(c, h * KSTEPS + s, KPAD);

    // Chunk descriptors: (local unit << 24) | chunk, or -1 once every unit
    // of the work-group is dry.
    int home = (wv * U) / kWsWaves;
    const unsigned counter_lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)counter;
    auto grab = [&]() -> int {
        for (int k = 0; k < U; ++k) {
            int got = 0;
            if (lane == 0) got = lds_fetch_add(counter_lds + 4u * (unsigned)home, 1);
            got = __builtin_amdgcn_readfirstlane(got);
            const int gu = unit0 + home;
            const int tr = (gu / wa.nbg) % wa.ntr;
            if (gu < wa.nunits && got < wa.tr_chunks && (tr * wa.tr_chunks + got) * chunk_tiles < wa.ntiles)
                return (home << 24) | got;
            home = home + 1 == U ? 0 : home + 1;
        }
        return -1;
    };
    // First tile (in its channel) and channel byte offset of a chunk.
    auto chunk_tile0 = [&](int d) {
        const int gu = unit0 + (d >> 24);
        const int tr = (gu / wa.nbg) % wa.ntr;
        return (tr * wa.tr_chunks + (d & 0xFFFFFF)) * chunk_tiles;
    };
    // The issue cursor's chunk as a first-tile address and a count of tiles
    // inside the channel (later tiles re-read the last one; past the end of
    // the work every load re-reads tile 0 of channel 0).
    const size_t tile_bytes = (size_t)32 * p.vstride;
    const int8_t* isrc = p.ftpa + p.voff;
    int ilast = 0;
    int itail = -1;   // the block's last tile within the chunk, if it is there
    auto set_issue_chunk = [&](int d) {
        isrc = p.ftpa + p.voff;
        ilast = 0;
        itail = p.F == 1 && wa.ntiles == 1 ? 0 : -1;
        if (d >= 0) {
            const int t0 = chunk_tile0(d);
            isrc += (size_t)unit_fo(unit0 + (d >> 24)) * TP * p.vstride + (size_t)t0 * tile_bytes;
            ilast = (wa.ntiles - t0 < chunk_tiles ? wa.ntiles - t0 : chunk_tiles) - 1;
            itail = unit_fo(unit0 + (d >> 24)) == p.F - 1 && t0 + ilast == wa.ntiles - 1 ? ilast : -1;
        }
    };
    auto issue = [&](int off, int slot) {
        const int o = off < ilast ? off : ilast;
        const int8_t* src = isrc + (size_t)o * tile_bytes;
#pragma unroll
        for (int m = 0; m < St::LPT; ++m)
            dma16(src + (uint32_t)(!AL16 && o == itail ? goff[m] - early[m] : goff[m]), ring + slot * St::TILE + m * 1024);
    };

    int cdesc = grab();          // chunk of the compute cursor
    int ioff = 0;                // issue cursor's tile within its chunk
    int pend = -1;               // next chunk, taken by the issue cursor
    set_issue_chunk(cdesc);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        issue(ioff, q);
        ++ioff;
    }

    // Weights of the unit being computed (loaded when it changes).
    v4i w[RT][KSTEPS];
    int wunit = -1;
    int fo = 0, beam_base = 0;
    float q_off = 0.f, q_sc = 1.f;
    bool q_thr = false;
    QuantConst qz{0.0, 1.0, 1.0f, 0.0f};
    const long long* thr = thr_all;

    int q = 0;   // sequence position of the compute cursor
    while (cdesc >= 0) {
        const int u = cdesc >> 24;
        if (u != wunit) {
            wunit = u;
            const int gu = unit0 + u;
            fo = unit_fo(gu);
            beam_base = (gu % wa.nbg) * 64;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const int b = beam_base + 32 * g + c;
                const bool bvalid = b < p.B;
                const int8_t* wcol = p.fba + ((size_t)fo * p.B + (bvalid ? b : p.B - 1)) * K;
#pragma unroll
                for (int s = 0; s < KSTEPS; ++s)
                    w[2 * g][s] = load_wslice<AL16>(wcol, 16 * (h * KSTEPS + s), K, bvalid);
            }
#pragma unroll
            for (int g = 0; g < NG; ++g)
#pragma unroll
                for (int s = 0; s < KSTEPS; ++s) {
                    w[2 * g + 1][s] = embed_slice(w[2 * g][s], true);
                    w[2 * g][s] = embed_slice(w[2 * g][s], false);
                }
            q_off = p.offsets[fo];
            q_sc = p.scales[fo];
            q_thr = thr_applies(q_off, q_sc);
            qz = quant_const(q_off, q_sc);
            thr = thr_all + u * kThr;
        }
        const int ctile0 = chunk_tile0(cdesc);
        const int b_out = beam_base + 32 * h + c;
        const bool wave_active = beam_base < p.B;

        for (int pc = 0; pc < chunk_tiles; pc += wa.ntp) {
            long long pw[NG][NSLOT];
#pragma unroll
            for (int g = 0; g < NG; ++g)
#pragma unroll
                for (int sl = 0; sl < NSLOT; ++sl) pw[g][sl] = 0;
#pragma unroll
            for (int g = 0; g < NSLOT / SPT; ++g) {
                for (int x = 0; x < wa.tps; ++x) {
                    const int slot = q % NB;
                    wait_vm_lgkm0<St::WAIT>();
                    const int8_t* src = ring + slot * St::TILE;
                    v4i a[KSTEPS];
#pragma unroll
                    for (int s = 0; s < KSTEPS; ++s) a[s] = *reinterpret_cast<const v4i*>(src + aoff[s]);
                    if (!AL16 && fo == p.F - 1 && ctile0 + pc + g * wa.tps + x == wa.ntiles - 1) {
#pragma unroll
                        for (int s = 0; s < KSTEPS; ++s)
                            if (c == 31 && h * KSTEPS + s == staged_tail_piece(K)) a[s] = v4i{a[s].z, a[s].w, a[s].z, a[s].w};
                    }
                    wait_vm_lgkm0<63>();
                    // The slot is free again: refill it NB positions ahead.
                    if (ioff == chunk_tiles) {
                        pend = grab();
                        set_issue_chunk(pend);
                        ioff = 0;
                    }
                    issue(ioff, slot);
                    ++ioff;
                    detect_step<RT, KSTEPS, SPT, NSLOT>(a, w, pw, g);
                    ++q;
                }
            }
            // Reduce-scatter over the row halves (lanes below 32 keep beam
            // group 0), quantise, store.
            long long tot[NSLOT];
#pragma unroll
            for (int sl = 0; sl < NSLOT; ++sl) tot[sl] = swap32_sum(pw[0][sl], pw[1][sl]);
            const int win0 = (ctile0 + pc) * SPT / wa.tps;
#pragma unroll
            for (int v = 0; v < NSLOT; ++v) {
                const long long to = (long long)win0 + v;
                if (!wave_active || b_out >= p.B || to >= p.nsamples_out) continue;
                int8_t* row = static_cast<int8_t*>(p.out) + ((size_t)fo * p.nsamples_out + (size_t)to) * p.B;
                row[b_out] = q_thr ? quantise_thr(tot[v], qz, thr + 128)
                                   : quantise((double)tot[v], q_off, q_sc, p.quant);
            }
        }
        cdesc = pend;
        pend = -1;
    }
    // Loads issued past the last chunk are still in flight.
    wait_vm_lgkm0<0>();
}

// Units, chunks and units per work-group of cb_ws_k for one launch.
template <int KSTEPS, int SPT, int NSLOT>
hipError_t launch_ws_k(CbWsArgs a, hipStream_t s)
{
    const int nb = WsStage<KSTEPS>::NB;
    a.ct = a.ntp * ((nb + a.ntp - 1) / a.ntp);
    const int chunks = (a.ntiles + a.ct - 1) / a.ct;
    const long long base_units = (long long)a.p.Fo * a.nbg;
    const int ncu = device_cu_count();
    int ntr = 1;
    if (base_units < ncu) ntr = (int)((ncu + base_units - 1) / base_units);
    if (ntr > chunks) ntr = chunks;
    a.tr_chunks = (chunks + ntr - 1) / ntr;
    a.ntr = (chunks + a.tr_chunks - 1) / a.tr_chunks;
    const long long nunits = base_units * a.ntr;
    if (nunits >= (1ll << 24)) return hipErrorInvalidConfiguration;
    a.nunits = (int)nunits;
    static const int kU[] = {1, 2, 3, 4, 6};
    a.U = kWsMaxUnits;
    for (int u : kU)
        if ((nunits + u - 1) / u <= ncu) {
            a.U = u;
            break;
        }
    const long long nblocks = (nunits + a.U - 1) / a.U;
    const size_t shm = (size_t)kWsWaves * nb * WsStage<KSTEPS>::TILE + (size_t)a.U * (kThr * sizeof(long long) + 4) +
                       kWsWaves * sizeof(int);
    if (a.p.A % 8 == 0)
        cb_ws_k<KSTEPS, SPT, NSLOT, true><<<dim3((unsigned)nblocks), 64 * kWsWaves, shm, s>>>(a);
    else
        cb_ws_k<KSTEPS, SPT, NSLOT, false><<<dim3((unsigned)nblocks), 64 * kWsWaves, shm, s>>>(a);
    return hipGetLastError();
}

template <int SPT, int NSLOT>
hipError_t launch_ws_ks(const CbWsArgs& a, int ksteps, hipStream_t s)
{
    switch (ksteps) {
    case 1: return launch_ws_k<1, SPT, NSLOT>(a, s);
    case 2: return launch_ws_k<2, SPT, NSLOT>(a, s);
    case 3: return launch_ws_k<3, SPT, NSLOT>(a, s);
    case 4: return launch_ws_k<4, SPT, NSLOT>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace
}  // namespace fbf

hipError_t fbf::cb_launch_ws(const CbWsArgs& a, int W, int ksteps, hipStream_t s)
{
    if (W == 8) return launch_ws_ks<4, 4>(a, ksteps, s);
    if (W == 16) return launch_ws_ks<2, 4>(a, ksteps, s);
    if (W == 32) return launch_ws_ks<1, 4>(a, ksteps, s);
    return launch_ws_ks<1, 2>(a, ksteps, s);
}
