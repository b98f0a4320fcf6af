// serve_route.h -- the router of a mixture of at most 64 experts for one token: scores by a workgroup of four waves, the choice by one wave, one expert
// per lane.  A kernel that has a token's row at hand routes it on its way out (route_row); the kernel for rows in memory is in serve_moe.hip.  Both add the
// same products in the same order: the same bits.
#pragma once
#include "serve_common.h"

namespace {
__device__ __forceinline__ void load8(const bf16_t* p, float (&v)[8]) {
    const uint4 u = *(const uint4*)p;
    const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}
__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ unsigned order_key(float v) {         // larger key = larger value; -0 = +0, NaN below everything
    const unsigned u = __float_as_uint(v + 0.0f);
    return v != v ? 0u : u >> 31 ? ~u : u | 0x80000000u;
}
// number of lanes j < n in `mask` whose key is larger (or equal at a lower index): unique per lane of the mask
__device__ __forceinline__ int place_of(unsigned key, unsigned long long mask, int n, int lane) {
    int r = 0;
    for (int j = 0; j < n; ++j) {
        const unsigned kj = (unsigned)__builtin_amdgcn_readlane((int)key, j);
        r += (mask >> j & 1) && (kj > key || (kj == key && j < lane));
    }
    return r;
}
template <typename T>
struct Piece {
    typedef uint4 type;
};
struct float8 {
    float4 a, b;
};
template <>
struct Piece<float> {
    typedef float8 type;
};

struct RouteArgs {
    int32_t* idx;                    // [n, top_k]
    float* weight;
    const void *router, *bias;       // [E, D], [E] or NULL, in the storage type
    const float* correction;
    int renorm, E, top_k, G, keep, score_fn, group_top;
    float scale;
};

// s: lane e < E has the product of router row e with token t's row; cs: 64 floats of this wave.  Scores s = softmax over all experts (score_fn 0) or the
// sigmoid (1); the choice goes by s + correction inside the `keep` best of G groups, the weights are the chosen s (renorm: over their sum) times scale.
__device__ __forceinline__ void select_experts(float s, float lane_bias, float lane_corr, const RouteArgs& a, size_t t, float* cs, int lane) {
    const bool mine = lane < a.E;
    s = mine ? s : -INFINITY;
    if (mine && a.bias) s += lane_bias;
    if (a.score_fn == 0) {
        const float mx = wave_max(s);
        s = mine ? expf(s - mx) : 0.f;
        s *= 1.0f / wave_sum(s);
    } else {
        s = 1.0f / (1.0f + expf(-s));
    }
    const float c = mine ? (a.correction ? s + lane_corr : s) : 0.f;
    unsigned long long ok = a.E == 64 ? ~0ull : (1ull << a.E) - 1;   // experts that may be chosen
    if (a.keep < a.G) {
        cs[lane] = c;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int per = a.E / a.G;
        float gs = 0.f;
        if (lane < a.G) {
            float v1 = cs[lane * per], v2 = -INFINITY;        // the two largest
            for (int e = 1; e < per; ++e) {
                const float v = cs[lane * per + e];
                if (v > v1) {
                    v2 = v1;
                    v1 = v;
                } else if (v > v2) {
                    v2 = v;
                }
            }
            gs = (a.group_top == 2 && per > 1) ? v1 + v2 : v1;
        }
        const unsigned long long all = a.G == 64 ? ~0ull : (1ull << a.G) - 1;
        const int place = place_of(order_key(gs), all, a.G, lane);
        const unsigned long long kept = __ballot(lane < a.G && place < a.keep);
        ok = __ballot(mine && (kept >> (min(lane, a.E - 1) / per) & 1));
    }
    const int place = place_of(order_key(c), ok, a.E, lane);
    const bool chosen = mine && (ok >> lane & 1) && place < a.top_k;
    float wt = s;
    if (a.renorm) {                                                // over the chosen only, summed from the best down
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (chosen) cs[place] = s;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        float sum = 0.f;
        for (int k = 0; k < a.top_k; ++k) sum += cs[k];
        wt /= sum;
    }
    if (a.renorm || a.scale != 1.0f) wt *= a.scale;
    if (chosen) {
        a.idx[t * a.top_k + place] = lane;
        a.weight[t * a.top_k + place] = wt;
    }
}

template <typename T, int EC>
struct RouteHead {                                               // router columns 8 tid .. of the first EC experts, requested before the row is there
    typename Piece<T>::type r[EC];
    __device__ __forceinline__ void request(const RouteArgs& a, int D) {
        const int c = min((int)threadIdx.x * 8, D - 8);
#pragma unroll
        for (int e = 0; e < EC; ++e) r[e] = *(const typename Piece<T>::type*)((const T*)a.router + (size_t)min(e, a.E - 1) * D + c);
    }
};
template <typename T, int P, int EC>
struct RouteRoom {
    T row[P * 1024];
    float part[4][64], cs[64];
};
template <typename T, int P>
struct RouteRoom<T, P, 0> {};
inline bool route_ok(const RouteArgs& r) {
    return r.idx && r.weight && r.router && (uintptr_t)r.router % 16 == 0 && r.E > 0 && r.E <= 64 && r.G > 0 && r.E % r.G == 0 && r.keep > 0 && r.keep <= r.G &&
           r.top_k > 0 && r.top_k <= r.keep * (r.E / r.G) && (r.score_fn == 0 || r.score_fn == 1) && (r.group_top == 1 || r.group_top == 2);
}
// Token t's row (D elements in LDS, written by this workgroup of 256 threads before its last barrier) -> its experts.  D a multiple of 8.
template <typename T, int EC>
__device__ __forceinline__ void route_row(const RouteArgs& a, const RouteHead<T, EC>& head, size_t t, const T* row, int D, float (*part)[64], float* cs) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const float lane_bias = a.bias && lane < a.E ? ld((const T*)a.bias, lane) : 0.f, lane_corr = a.correction && lane < a.E ? a.correction[lane] : 0.f;
    float v[EC];
    auto add = [&](const typename Piece<T>::type (&rr)[EC], int c) __attribute__((always_inline)) {
        float x[8];
        load8(row + c, x);
#pragma unroll
        for (int e = 0; e < EC; ++e) {
            float r[8];
            load8((const T*)&rr[e], r);
#pragma unroll
            for (int q = 0; q < 8; ++q) v[e] += r[q] * x[q];
        }
    };
    auto more = [&](int e0, int c) __attribute__((always_inline)) {
        for (; c < D; c += 256 * 8) {
            typename Piece<T>::type rr[EC];
#pragma unroll
            for (int e = 0; e < EC; ++e) rr[e] = *(const typename Piece<T>::type*)((const T*)a.router + (size_t)min(e0 + e, a.E - 1) * D + c);
            add(rr, c);
        }
    };
    auto leave = [&](int e0) __attribute__((always_inline)) {
        wave_sum_scatter<EC>(v, lane);
        if (lane % (64 / EC) == 0) part[w][e0 + lane / (64 / EC)] = v[0];
    };
#pragma unroll
    for (int i = 0; i < EC; ++i) v[i] = 0.f;
    if ((int)threadIdx.x * 8 < D) add(head.r, threadIdx.x * 8);
    more(0, threadIdx.x * 8 + 256 * 8);
    leave(0);
    for (int e0 = EC; e0 < a.E; e0 += EC) {
#pragma unroll
        for (int i = 0; i < EC; ++i) v[i] = 0.f;
        more(e0, threadIdx.x * 8);
        leave(e0);
    }
    __syncthreads();
    if (w) return;
    float s = 0.f;
    if (lane < a.E) {
#pragma unroll
        for (int o = 0; o < 4; ++o) s += part[o][lane];
    }
    select_experts(s, lane_bias, lane_corr, a, t, cs, lane);
}
}  // namespace
