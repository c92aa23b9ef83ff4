// Instances of the transposed kernel (cb_tr_k) with 128 beams per wave.
#include "cb_tr.hpp"

hipError_t fbf::cb_launch_tr8(const CbTrArgs& a, int fs, int W, int ksteps, int passes, hipStream_t s)
{
    return launch_tr<8>(a, fs, W, ksteps, passes, s);
}
