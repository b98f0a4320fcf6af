// gemm_w4a8_ring.hip -- which part of the decode-shape W4A8 GEMM (gemm_w4a8_ring.h) a call is for.
#include "gemm_w4a8_ring.h"

qs_flag g_ring_flags = 0;

#ifdef QS_RING_TRACE
extern "C" int qs_debug_ring_trace(void* buf) {
    unsigned long long* p = reinterpret_cast<unsigned long long*>(buf);
    for (const auto to : {qs_ring_trace_chn_few, qs_ring_trace_chn_many, qs_ring_trace_group_few, qs_ring_trace_group_many})
        if (const int rc = to(p)) return rc;
    return QS_OK;
}
#endif

// Entry used by the dispatcher in gemm_w4a8.hip.  mt = m-tiles per workgroup (1, 2, 4), wn = units per workgroup
// (1, 2, 4); ksplit = K slices (1 = none; > 1 needs the slab / counter workspace: (N/64) * mblocks * ksplit * mt KiB * 4 and
// (N/64) * mblocks counters); preconditions (checked there): N % (64*wn) == 0, qs_ring_fits,
// M*K and N*K/2 below 4 GiB.
int qs_launch_gemm_ring(int mode, int outk, int mt, int wn, const int8_t* A, const uint8_t* W, const int8_t* zeros,
                        const int8_t* scales8, const void* wscales, const void* ascales, const void* wszs,
                        const void* assums, void* out, int M, int N, int K, int mblocks, int ksplit, int* slabs,
                        unsigned* counters, hipStream_t stream) {
    if (g_qs_plan.active) {
        g_qs_plan.family = 3;
        g_qs_plan.p[0] = mt, g_qs_plan.p[1] = wn, g_qs_plan.p[2] = mblocks, g_qs_plan.p[3] = ksplit;
        return QS_OK;
    }
    if (outk == 2 && ksplit > 1) {
        qs_set_error("w4a8 gemm (ring): the activation epilogue has no K-sliced form");
        return QS_ENOSUP;
    }
    if ((outk == 0 || outk == 2) && ((reinterpret_cast<uintptr_t>(wscales) & 3) || (mode == 0 && (reinterpret_cast<uintptr_t>(wszs) & 3)))) {
        // (the reference reads them as half2, gemm_cuda.cu:581-582: the same requirement)
        qs_set_error("w4a8 gemm: wscales / w_szs must be 4-byte aligned");
        return QS_EINVAL;
    }
    const bool even = (K / 64) % ksplit == 0 && (K / 64 / ksplit) % (8 / wn) == 0;
    if (!even && (outk == 2 || mt == 8)) {
        qs_set_error("w4a8 gemm (ring): the stages of K=%d do not divide over the groups", K);
        return QS_ENOSUP;
    }
    const RingCall c = {outk, mt, wn, !even ? 2 : ksplit > 1, A, W, zeros, scales8, wscales, ascales, wszs, assums, out, M, N, K, mblocks, ksplit, slabs, stream};
    if (mode == 0) return mt <= 2 ? qs_ring_chn_few(c) : qs_ring_chn_many(c);
    return mt <= 2 ? qs_ring_group_few(c) : qs_ring_group_many(c);
}
