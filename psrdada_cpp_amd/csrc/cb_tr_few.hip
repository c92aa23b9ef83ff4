// Instances of the transposed kernel (cb_tr_k) for few beams or small blocks of
// up to 64 antennas: one wave of 32 or 64 beams per time slot, four time slots to
// a work-group (cb_few_rows).
#include "cb_tr.hpp"

namespace fbf {
namespace {

template <int RT, int KSTEPS, int SPT, int NSLOT>
hipError_t launch_few(const CbTrArgs& a, int passes, hipStream_t s)
{
    if (a.p.S == 0) return launch_tr_kt<RT, KSTEPS, SPT, NSLOT, 1, 4, 1, false>(a, passes, s);
    return a.ibp ? launch_tr_kt<RT, KSTEPS, SPT, NSLOT, 1, 4, 1, true, true>(a, passes, s)
                 : launch_tr_kt<RT, KSTEPS, SPT, NSLOT, 1, 4, 1, true, false>(a, passes, s);
}

template <int RT, int SPT, int NSLOT>
hipError_t launch_few_ks(const CbTrArgs& a, int ksteps, int passes, hipStream_t s)
{
    switch (ksteps) {
    case 1: return launch_few<RT, 1, SPT, NSLOT>(a, passes, s);
    case 2: return launch_few<RT, 2, SPT, NSLOT>(a, passes, s);
    case 3: return launch_few<RT, 3, SPT, NSLOT>(a, passes, s);
    case 4: return launch_few<RT, 4, SPT, NSLOT>(a, passes, s);
    default: return hipErrorInvalidValue;
    }
}

// Windows per pass as cb_tr_nslot.
template <int RT>
hipError_t launch_few_w(const CbTrArgs& a, int W, int ksteps, int passes, hipStream_t s)
{
    constexpr int small = RT == 2 ? 8 : 4;
    if (W == 8) return launch_few_ks<RT, 4, small>(a, ksteps, passes, s);
    if (W == 16) return launch_few_ks<RT, 2, RT == 4 ? 2 : small>(a, ksteps, passes, s);
    if (W == 32) return launch_few_ks<RT, 1, RT == 4 ? 2 : 4>(a, ksteps, passes, s);
    return launch_few_ks<RT, 1, 2>(a, ksteps, passes, s);
}

}  // namespace
}  // namespace fbf

hipError_t fbf::cb_launch_tr_few(const CbTrArgs& a, int rt, int W, int ksteps, int passes, hipStream_t s)
{
    return rt == 2 ? launch_few_w<2>(a, W, ksteps, passes, s) : launch_few_w<4>(a, W, ksteps, passes, s);
}
