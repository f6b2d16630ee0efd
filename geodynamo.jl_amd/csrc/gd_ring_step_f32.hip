// gd_ring_step_f32.hip -- step-mode ring passes of the compiled lengths, FP32 rings
#include "gd_ring_step.hpp"

template <> bool gd_launch_ring_step_plan<float>(hipStream_t st, int mode, const RingArgs &a)
{
    switch (mode) {
    case RING_STEP_TANG: return ring_step_mode<float, RING_STEP_TANG>(st, a);
    case RING_STEP_TANG_C: return ring_step_mode<float, RING_STEP_TANG_C>(st, a);
    case RING_ADJ_TANG: return ring_step_mode<float, RING_ADJ_TANG>(st, a);
    case RING_STEP: return ring_step_mode<float, RING_STEP>(st, a);
    default: return false;
    }
}

template <> bool gd_launch_ring_tang_batch_plan<float>(hipStream_t st, const BatchRef<RingArgs> &b, int nblocks, int nlon, bool deal)
{
    return ring_step_batch<float>(st, b, nblocks, nlon, deal);
}
