// gemm_w4a8_ring_chn_many.hip -- decode-shape W4A8 GEMM, per-channel weights, 64- and 128-token workgroups.
#include "gemm_w4a8_ring.h"

int qs_ring_chn_many(const RingCall& c) { return ring_part<0, false>(c); }
#ifdef QS_RING_TRACE
int qs_ring_trace_chn_many(unsigned long long* p) { return ring_trace_to(p); }
#endif
