// Instances of the transposed kernel (cb_tr_k) with 64 beams per wave.
#include "cb_tr.hpp"

hipError_t fbf::cb_launch_tr4(const CbTrArgs& a, int fs, int W, int ksteps, int passes, hipStream_t s)
{
    if (fs == 1) return launch_tr_w<4, 1>(a, W, ksteps, passes, s);
    if (fs == 2) return launch_tr_w<4, 2>(a, W, ksteps, passes, s);
    return launch_tr_w<4, 4>(a, W, ksteps, passes, s);
}
