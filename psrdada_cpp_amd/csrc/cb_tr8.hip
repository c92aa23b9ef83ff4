// Instances of the transposed kernel (cb_tr_k) with 128 beams per wave,
// fscrunch 1.
#include "cb_tr.hpp"

hipError_t fbf::cb_launch_tr8(const CbTrArgs& a, int W, int ksteps, int passes, hipStream_t s)
{
    return launch_tr_w<8, 1>(a, W, ksteps, passes, s);
}
