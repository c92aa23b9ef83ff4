// Instances of the transposed kernel (cb_tr_k) with 32 beams per wave.
#include "cb_tr.hpp"

hipError_t fbf::cb_launch_tr2(const CbTrArgs& a, int fs, int W, int ksteps, int passes, hipStream_t s)
{
    if (fs == 1) return launch_tr_w<2, 1>(a, W, ksteps, passes, s);
    if (fs == 2) return launch_tr_w<2, 2>(a, W, ksteps, passes, s);
    return launch_tr_w<2, 4>(a, W, ksteps, passes, s);
}
