// gd_ring_io_f64.hip -- boundary ring passes of the compiled lengths, FP64 rings
#include "gd_ring_io.hpp"

template <> bool gd_launch_ring_plan<double>(hipStream_t st, int mode, const RingArgs &a)
{
    const int nf = a.nfield;
    return mode == RING_SYNTH ? ring_plan_mode<double, RING_SYNTH>(st, a, nf)
                              : ring_plan_mode<double, RING_ANALYSIS>(st, a, nf);
}
