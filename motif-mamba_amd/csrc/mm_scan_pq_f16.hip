// mm_scan_pq_f16.hip -- the float16 instances of the P/Q forward kernels of mm_scan_pq.hip (compiled
// once per input type, so that the three sets build in parallel).
#define MM_PQ_TYPE f16_t
#include "mm_scan_pq.hip"
