// mm_scan_bwd_lanes_f16.hip -- the float16 instances of the P/Q backward kernel of
// mm_scan_bwd_lanes.hip (compiled once per input type, so that the three sets build in parallel).
#define MM_BWD_LANES_TYPE f16_t
#include "mm_scan_bwd_lanes.hip"
