// gxt_loop.hip -- the step loop of one precision (GXT_LOOP_R) and transport
// mode (GXT_LOOP_MODE); built once for each.
#include "gxt_loop.h"

template hipError_t gxt::prepare_loop_mode<GXT_LOOP_R, GXT_LOOP_MODE>(int);
template hipError_t gxt::launch_loop_mode<GXT_LOOP_R, GXT_LOOP_MODE>(const gxt::LoopArgs &, hipStream_t, hipEvent_t,
                                                                     hipEvent_t);
