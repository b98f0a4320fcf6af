// serve_common.h -- helpers shared by the kernels of libqserve_serve.so (gfx950, 64-wide wavefronts)
#pragma once
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include "../../../include/qserve_serve.h"

void qsv_set_error(const char* fmt, ...);

#define QSV_REQUIRE(cond, ...)          \
    do {                                \
        if (!(cond)) {                  \
            qsv_set_error(__VA_ARGS__); \
            return QSV_EINVAL;          \
        }                               \
    } while (0)

static inline int qsv_launch_status(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        qsv_set_error("%s: launch failed: %s", what, hipGetErrorString(e));
        return (int)e;
    }
    return QSV_OK;
}

typedef uint16_t bf16_t;   // storage only: arithmetic is float

__device__ __forceinline__ float bf2f(bf16_t v) { return __uint_as_float((uint32_t)v << 16); }
// Round to nearest even; NaN stays NaN.  v_cvt_pk_bf16_f32: one instruction for two values, where bit arithmetic takes eight for each: a grouped product's epilogue
// (128 values a lane) 4.1 -> 3.5 us, a model's step of 64 tokens 2 % (64 sequences of Vekalorn 12.98 -> 12.68 ms).  Both forms were compared once over all 2^32 floats: the same
// bits but for a NaN's sign and payload (the tests hold ties, overflows, subnormals and NaN).
typedef float pair_f32 __attribute__((ext_vector_type(2)));
typedef __bf16 pair_bf16 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ bf16_t f2bf(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }
__device__ __forceinline__ uint32_t pack_bf2(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((pair_f32{a, b}), pair_bf16)); }
__device__ __forceinline__ float ld(const float* p, size_t i) { return p[i]; }
__device__ __forceinline__ float ld(const bf16_t* p, size_t i) { return bf2f(p[i]); }
__device__ __forceinline__ void st(float* p, size_t i, float v) { p[i] = v; }
__device__ __forceinline__ void st(bf16_t* p, size_t i, float v) { p[i] = f2bf(v); }

// Reductions over a wave, all 64 lanes active: the xor butterfly (offsets 32, 16, 8, 4, 2, 1; the same pairs in the same order as a
// __shfl_xor loop, so sums round alike) in register moves - permlane swaps for 32 and 16, DPP row rotations by 8 and by 4 (after the
// step before, the row is 8-periodic) and quad permutations - instead of six round trips through the LDS crossbar, which were most of
// a short row kernel's chain.
#define QSV_DPP(v, ctrl) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, true))
template <class Op>
__device__ __forceinline__ float wave_reduce(float v, Op op) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(b[0]), __uint_as_float(b[1]));
    v = op(v, QSV_DPP(v, 0x128));   // row_ror:8
    v = op(v, QSV_DPP(v, 0x124));   // row_ror:4
    v = op(v, QSV_DPP(v, 0x4E));    // quad_perm [2, 3, 0, 1]
    return op(v, QSV_DPP(v, 0xB1)); // quad_perm [1, 0, 3, 2]
}
__device__ __forceinline__ float wave_sum(float v) {
    return wave_reduce(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
    return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}
// NV values per lane (a power of two, at most 64) summed over the wave and scattered: v[0] of lane l ends up with the sum of value
// l / (64 / NV).  Half of the values left are exchanged with the lane across the next bit.
template <int NV, int O = 32, int M = NV>
__device__ __forceinline__ void wave_sum_scatter(float (&v)[NV], int lane) {
    if constexpr (O >= 1) {
        if constexpr (M > 1) {
#pragma unroll
            for (int i = 0; i < M / 2; ++i) {
                if constexpr (O == 32) {
                    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + M / 2]), false, false);
                    v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
                } else if constexpr (O == 16) {
                    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + M / 2]), false, false);
                    v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
                } else {
                    const bool up = lane & O;
                    const float give = up ? v[i] : v[i + M / 2], keep = up ? v[i + M / 2] : v[i];
                    v[i] = keep + (O == 8 ? QSV_DPP(give, 0x128) : O == 4 ? QSV_DPP(give, 0x141) : O == 2 ? QSV_DPP(give, 0x4E) : QSV_DPP(give, 0xB1));
                }
            }
            wave_sum_scatter<NV, O / 2, M / 2>(v, lane);
        } else {
            static_assert(O <= 4, "at least 8 values");
            v[0] += O == 4 ? QSV_DPP(v[0], 0x141) : O == 2 ? QSV_DPP(v[0], 0x4E) : QSV_DPP(v[0], 0xB1);   // (half mirror, quad permutations)
            wave_sum_scatter<NV, O / 2, 1>(v, lane);
        }
    }
}
// Sum over a workgroup of NT threads (a multiple of 64); every thread gets the result.  `red` holds NT / 64 + 1 floats.
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* red) {
    v = wave_sum(v);
    __syncthreads();   // (red may still be read from a previous call)
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) s += red[i];
    return s;
}

// four neighbouring elements at a multiple of four from an address that holds them whole
__device__ __forceinline__ void ld4t(const float* p, size_t i, float (&v)[4]) {
    const float4 a = *(const float4*)(p + i);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void ld4t(const bf16_t* p, size_t i, float (&v)[4]) {
    const uint2 u = *(const uint2*)(p + i);
    v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xffff0000u);
    v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xffff0000u);
}
__device__ __forceinline__ void st4t(float* p, size_t i, const float (&v)[4]) { *(float4*)(p + i) = make_float4(v[0], v[1], v[2], v[3]); }
__device__ __forceinline__ void st4t(bf16_t* p, size_t i, const float (&v)[4]) {
    *(uint2*)(p + i) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
}
// The same in two steps, request and use.  A row kernel requests every operand as it lies in memory, at a column inside the row (a lane behind its end repeats
// the last), and converts behind `requested()`: a conversion beside its load, or in a branch that not every lane takes, makes the wave wait there, and a row
// of a step would make one trip to memory after another.
typedef unsigned raw2u __attribute__((ext_vector_type(2)));
typedef float raw4f __attribute__((ext_vector_type(4)));
template <typename T>
struct Raw4;
template <>
struct Raw4<bf16_t> {
    typedef raw2u type;
};
template <>
struct Raw4<float> {
    typedef raw4f type;
};
template <typename T>
__device__ __forceinline__ typename Raw4<T>::type raw4(const T* p, size_t i) { return *(const typename Raw4<T>::type*)(p + i); }
__device__ __forceinline__ void widen4(raw4f r, float (&v)[4]) { v[0] = r[0]; v[1] = r[1]; v[2] = r[2]; v[3] = r[3]; }
__device__ __forceinline__ void widen4(raw2u r, float (&v)[4]) {
    v[0] = __uint_as_float(r[0] << 16); v[1] = __uint_as_float(r[0] & 0xffff0000u);
    v[2] = __uint_as_float(r[1] << 16); v[3] = __uint_as_float(r[1] & 0xffff0000u);
}
__device__ __forceinline__ void requested() { __builtin_amdgcn_sched_barrier(0); }
// token of a workgroup where each has `chunks` of them, neighbours (one: no division, which a kernel of 3 us would notice)
__device__ __forceinline__ unsigned token_of(unsigned block, int chunks) { return chunks == 1 ? block : block / (unsigned)chunks; }
// an address that 4 elements of its type may be read from at once
inline bool fits4(const void* p, int dtype) { return (uintptr_t)p % (dtype == QSV_BF16 ? 8 : 16) == 0; }

// What a mixture of experts leaves, a row per slot (t, k), to be summed by the kernel that uses it: y[t] = sum_k weight[t, k] ys[place ? place[t top + k] :
// t top + k] (weight NULL: ones; slots whose index names none of the experts add nothing).
struct SlotRows {
    const void* ys;
    const int32_t* place;
    const float* weight;
    const int32_t* idx;
    int top, n_experts;
};
// a[p] = four columns of y[t] from c + p * step on, p < P (zeros behind D).  The rows of four slots are requested together, beside their weights and indices
// where a slot's row is its number (a row without an expert holds anything: it is taken out by value).
// behind(): called once the first four are requested.
template <typename Y, int P, bool PLACED, class Behind>
__device__ __forceinline__ void slot_sum4_as(const SlotRows& s, size_t t, int D, int c, int step, float (&a)[P][4], Behind behind) {
    const float* weight = s.weight ? s.weight : (const float*)s.idx;           // (none: something that can be read)
    auto four = [&](int k0) __attribute__((always_inline)) {
        typename Raw4<Y>::type r[4][P];
        float w[4];
        int e[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const size_t slot = t * s.top + min(k0 + q, s.top - 1);
            e[q] = s.idx[slot];
            w[q] = weight[slot];
            const size_t row = !PLACED ? slot : (unsigned)e[q] < (unsigned)s.n_experts ? (size_t)s.place[slot] : 0;      // (no slot's row, but a row)
#pragma unroll
            for (int p = 0; p < P; ++p) r[q][p] = raw4((const Y*)s.ys, row * D + min(c + p * step, D - 4));
        }
        if (k0 == 0) behind();
        requested();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bool none = k0 + q >= s.top || (unsigned)e[q] >= (unsigned)s.n_experts;
            const float wq = s.weight ? w[q] : 1.0f;
#pragma unroll
            for (int p = 0; p < P; ++p) {
                float v[4];
                widen4(r[q][p], v);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float sum = a[p][j] + wq * v[j];
                    a[p][j] = none || c + p * step >= D ? a[p][j] : sum;
                }
            }
        }
    };
    four(0);                                                                   // (outside the loop, whose head waits for what the caller has requested)
    for (int k0 = 4; k0 < s.top; k0 += 4) four(k0);
}
template <typename Y, int P, class Behind>
__device__ __forceinline__ void slot_sum4(const SlotRows& s, size_t t, int D, int c, int step, float (&a)[P][4], Behind behind) {
#pragma unroll
    for (int p = 0; p < P; ++p) a[p][0] = a[p][1] = a[p][2] = a[p][3] = 0.f;
    if (s.place) slot_sum4_as<Y, P, true>(s, t, D, c, step, a, behind);
    else slot_sum4_as<Y, P, false>(s, t, D, c, step, a, behind);
}
template <typename Y, int P>
__device__ __forceinline__ void slot_sum4(const SlotRows& s, size_t t, int D, int c, int step, float (&a)[P][4]) {
    slot_sum4<Y>(s, t, D, c, step, a, [] __device__() {});
}

// A recurrence's decay from its gate z: sigmoid(z)^(1 / tau) = exp(-softplus(-z) / tau), or, with a log rate, exp(-exp(a) softplus(z))
__device__ __forceinline__ float softplusf(float z) { return z > 20.f ? z : log1pf(expf(z)); }
__device__ __forceinline__ float gate_decay(float z, bool with_rate, float a, float inv_tau) {
    return with_rate ? expf(-expf(a) * softplusf(z)) : expf(-softplusf(-z) * inv_tau);
}

// ... as a tensor of the storage type would hold it
__device__ __forceinline__ float stored(const float*, float v) { return v; }
__device__ __forceinline__ float stored(const bf16_t*, float v) { return bf2f(f2bf(v)); }
template <typename T, int P>
__device__ __forceinline__ void round_stored(float (&a)[P][4]) {
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int j = 0; j < 4; ++j) a[p][j] = stored((const T*)nullptr, a[p][j]);
}

// dtype dispatch of a templated launcher: F<bf16_t>() or F<float>()
#define QSV_DISPATCH(dtype, what, CALL)                                  \
    do {                                                                 \
        if ((dtype) == QSV_BF16) {                                       \
            typedef bf16_t T;                                            \
            CALL;                                                        \
        } else if ((dtype) == QSV_F32) {                                 \
            typedef float T;                                             \
            CALL;                                                        \
        } else {                                                         \
            qsv_set_error("%s: unknown dtype code %d", what, (dtype));   \
            return QSV_EINVAL;                                           \
        }                                                                \
    } while (0)
