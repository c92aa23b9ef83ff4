// Instances of the transposed kernel (cb_tr_k) with 32 beams per wave.
#include "cb_tr.hpp"

hipError_t fbf::cb_launch_tr2(const CbTrArgs& a, int fs, int W, int ksteps, int passes, hipStream_t s)
{
    return launch_tr<2>(a, fs, W, ksteps, passes, s);
}
