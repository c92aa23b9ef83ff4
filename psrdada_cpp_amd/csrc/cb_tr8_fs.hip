// Instances of the transposed kernel (cb_tr_k) with 128 beams per wave,
// fscrunch 2 and 4.
#include "cb_tr.hpp"

hipError_t fbf::cb_launch_tr8_fs(const CbTrArgs& a, int fs, int W, int ksteps, int passes, hipStream_t s)
{
    return fs == 2 ? launch_tr_w<8, 2>(a, W, ksteps, passes, s) : launch_tr_w<8, 4>(a, W, ksteps, passes, s);
}
