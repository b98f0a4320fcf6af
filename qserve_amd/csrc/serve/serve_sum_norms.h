// serve_sum_norms.h -- x += s0 a + s1 b + s2 c (element-wise scales); h0 = rms_norm(x) * g0, h1 = rms_norm(x) * g1: a row's work, for the kernel of its own
// (serve_rows.hip) and for a product of the normed rows (serve_linear.hip).
#pragma once
#include <type_traits>

#include "serve_common.h"
#include "serve_route.h"

namespace {
struct ScaledParts {
    const void *y[3], *s[3];
    const void* slot_scale;
};
struct NothingMore {
    __device__ __forceinline__ void operator()() const {}
};
// One trip to memory: the NP parts (and, Y other than void, what a mixture of experts left per slot, summed and rounded here as a tensor would hold it,
// scaled by slot_scale: added behind the first part) are requested before the first is used.  Rows of more than 4096 columns with two parts and more take two trips:
// in one their registers leave two waves to a SIMD (three parts of 8192, 1024 / 2048 rows 29.1 / 53.6 -> 23.9 / 43.6 us).
// THREADS: 64 or 128 for rows of up to 256 and 512 columns (idle waves repeat the row's last column: three parts of 256, 8192 rows 13.7 -> 7.4 us); VPT: groups
// of four columns a thread, the least that holds the row (three parts of 2304, 2048 rows: three groups 15.3 us, four 18.1).
// EC other than 0: the rows of the second norm go through a router on their way out (serve_route.h).
// PRODUCT: h0 alone goes into LDS, pieces of 16 bytes of every 128 permuted by the row's number, and nothing else is stored; behind(): called once every operand that
// the sums need is requested.
template <typename T, int VPT, int NP, typename Y, int EC, int THREADS, bool PRODUCT, class Behind>
__device__ __forceinline__ void scaled_sum_row(size_t t, float* x, const float* in, T* h0, T* h1, const ScaledParts& p,
                                               const float* __restrict__ g0, const float* __restrict__ g1, const int32_t* __restrict__ tokens, const T* __restrict__ table,
                                               float eps, int D, const SlotRows& slots, const RouteArgs& route, unsigned char* lds, Behind behind) {
    constexpr bool SLOTS = !std::is_void<Y>::value;
    constexpr int CH = VPT > 4 && NP >= 2 ? VPT / 2 : VPT, PARTS = NP ? NP : 1;
    static_assert(VPT % CH == 0 && (CH == VPT || (!SLOTS && EC == 0)) && (EC == 0 || THREADS == 256) && (!PRODUCT || (VPT <= 2 && EC == 0)), "");
    __shared__ float red[THREADS / 64 + 1];
    __shared__ __attribute__((aligned(16))) RouteRoom<T, VPT, EC> room;
    RouteHead<T, EC ? EC : 1> head;
    float v[VPT][4], ysum[CH][4], yf[CH][4];
    raw4f rg0[VPT], rg1[VPT];
    const bool norms = PRODUCT || h0 != nullptr, two = !PRODUCT && norms && h1 != nullptr;
    const T* sf[PARTS];
#pragma unroll
    for (int j = 0; j < NP; ++j) sf[j] = p.s[j] ? (const T*)p.s[j] : (const T*)p.y[j];      // (no scale: a row that there is)
    const T* sy = SLOTS ? (p.slot_scale ? (const T*)p.slot_scale : (const T*)p.y[0]) : nullptr;
    const float *first = norms ? g0 : in, *second = two ? g1 : first;
    const size_t row = tokens ? (size_t)tokens[t] * D : 0;
    float s = 0.f;
    auto gains = [&]() __attribute__((always_inline)) {
        if constexpr (VPT <= 2) {                                    // (wider rows would hold too much)
#pragma unroll
            for (int k = 0; k < VPT; ++k) {
                const int at = min(((int)threadIdx.x + k * THREADS) * 4, D - 4);
                rg0[k] = raw4(first, at);
                rg1[k] = raw4(second, at);
            }
        }
    };
#pragma unroll
    for (int k0 = 0; k0 < VPT; k0 += CH) {
        typename Raw4<T>::type rz[CH][PARTS], rf[CH][PARTS], ryf[CH], rt[CH];
        raw4f rx[CH];
        float z[CH][PARTS][4], f[CH][PARTS][4];
        if (tokens) {
#pragma unroll
            for (int k = 0; k < CH; ++k) rt[k] = raw4(table, row + min(((int)threadIdx.x + (k0 + k) * THREADS) * 4, D - 4));
        }
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int at = min(((int)threadIdx.x + (k0 + k) * THREADS) * 4, D - 4);
            if (!tokens) rx[k] = raw4(in, t * D + at);
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                rz[k][j] = raw4((const T*)p.y[j], t * D + at);
                rf[k][j] = raw4(sf[j], at);
            }
            if constexpr (SLOTS) ryf[k] = raw4(sy, at);
        }
        if constexpr (EC > 0) head.request(route, D);
        if constexpr (PRODUCT) gains();
        if constexpr (SLOTS) {
            slot_sum4<Y>(slots, t, D, threadIdx.x * 4, THREADS * 4, ysum, behind);
            round_stored<T>(ysum);
        } else {
            behind();
        }
        if constexpr (!PRODUCT) gains();
        requested();
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            if (tokens) widen4(rt[k], v[k0 + k]);
            else widen4(rx[k], v[k0 + k]);
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                widen4(rz[k][j], z[k][j]);
                widen4(rf[k][j], f[k][j]);
                if (!p.s[j]) f[k][j][0] = f[k][j][1] = f[k][j][2] = f[k][j][3] = 1.f;
            }
            if constexpr (SLOTS) {
                widen4(ryf[k], yf[k]);
                if (!p.slot_scale) yf[k][0] = yf[k][1] = yf[k][2] = yf[k][3] = 1.f;
            }
        }
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int i = (threadIdx.x + (k0 + k) * THREADS) * 4;
            if (i >= D) continue;
            float(&u)[4] = v[k0 + k];
            float y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                if (SLOTS && j == 1)
#pragma unroll
                    for (int e = 0; e < 4; ++e) y[e] += yf[k][e] * ysum[k][e];
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] += f[k][j][e] * z[k][j][e];
            }
            if (SLOTS && NP < 2)
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] += yf[k][e] * ysum[k][e];
#pragma unroll
            for (int e = 0; e < 4; ++e) u[e] += y[e];
            if constexpr (!PRODUCT) st4t(x, t * D + i, u);
            s += fmaf(u[3], u[3], fmaf(u[2], u[2], fmaf(u[0], u[0], u[1] * u[1])));   // (which product of two is rounded is not left to each form's compilation)
        }
    }
    if (!norms) return;
    const float inv = 1.0f / sqrtf(block_sum<THREADS>(s, red) / (float)D + eps);
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int i = (threadIdx.x + k * THREADS) * 4;
        if (i >= D) continue;
        float a[4], n[4];
        if constexpr (VPT <= 2) widen4(rg0[k], a);
        else ld4t(g0, i, a);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[k][e] *= inv;
            n[e] = v[k][e] * a[e];
        }
        if constexpr (PRODUCT) {
            *(uint2*)(lds + t * D * 2 + (i / 64) * 128 + ((((i & 63) >> 3) ^ ((int)t & 7)) << 4) + (i & 4) * 2) = make_uint2(pack_bf2(n[0], n[1]), pack_bf2(n[2], n[3]));
            continue;
        }
        st4t(h0, t * D + i, n);
        if (h1) {
            if constexpr (VPT <= 2) widen4(rg1[k], a);
            else ld4t(g1, i, a);
#pragma unroll
            for (int e = 0; e < 4; ++e) n[e] = v[k][e] * a[e];
            st4t(h1, t * D + i, n);
            if constexpr (EC > 0) st4t(room.row, i, n);
        }
    }
    if constexpr (EC > 0) {
        __syncthreads();
        route_row<T, EC>(route, head, t, room.row, D, room.part, room.cs);
    }
}
}  // namespace
