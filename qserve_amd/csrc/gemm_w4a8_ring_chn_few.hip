// gemm_w4a8_ring_chn_few.hip -- decode-shape W4A8 GEMM, per-channel weights, 16- and 32-token workgroups.
#include "gemm_w4a8_ring.h"

int qs_ring_chn_few(const RingCall& c) { return ring_part<0, true>(c); }
#ifdef QS_RING_TRACE
int qs_ring_trace_chn_few(unsigned long long* p) { return ring_trace_to(p); }
#endif
