// gd_ring_io_f32.hip -- boundary ring passes of the compiled lengths, FP32 rings
#include "gd_ring_io.hpp"

template <> bool gd_launch_ring_plan<float>(hipStream_t st, int mode, const RingArgs &a)
{
    const int nf = a.nfield;
    return mode == RING_SYNTH ? ring_plan_mode<float, RING_SYNTH>(st, a, nf)
                              : ring_plan_mode<float, RING_ANALYSIS>(st, a, nf);
}
