// gemm_w4a8_rows.hip -- W4A8 products of one to four tokens, with the row operation in front of them as their prologue.
//
// A step of few tokens is a chain of launches whose row kernels (residual add + norm + quantiser, quantiser) take 3 - 4 us each while the weights' stream
// waits.  Here every workgroup does that row operation itself - one token's row is 10 - 80 KB from the caches - while its weights, all of them requested
// before the first value of the row is used, are on their way to registers: no ring, no hand-over between workgroups, a launch less per product.
//
// Workgroup = 4 waves x one row (or a gate / up pair of rows) of 32-channel weight tiles, the waves each a quarter of the reduction (of its K slice).  A stage
// is 64 k: 1 KiB of packed weights, 16 bytes a lane - lane l holds nibbles of channels 8 cl + (l >> 2 & 7), cl < 4, and of k 32 (l >> 5) + 16 gp + 4 (l & 3) ..
// + 3, gp < 2 -, multiplied by the token's int8 row (in LDS) with v_dot4_i32_i8.  Few tokens leave the matrix cores fifteen columns empty; four dot products a dword
// of weights and token cost less than the stream.  Sums are int32, so every split of the reduction gives the same bits; the row operations and the epilogues
// are the shared ones (row_ops.h, common.h).
//
// Bound by HBM (gate_up of one token: 58.7 MB in 14.5 us with its norm, 12.9 in the ring kernel behind a norm of 3.2) and, below some 15 MB, by the launch and the
// row's chain of trips.  Measured for one token, launches replaced -> this, us: norm + qkv 6144 x 4096 9.9 -> 6.9, norm + gate_up 28672 x 4096 16.1 -> 14.5, o 4096 x
// 4096 4.7 -> 3.5 (one slice 3.9, four 3.7), quantiser + down 4096 x 14336 10.2 -> 9.1, of 11008 9.6 -> 7.9; groups of 128 12.2 -> 8.6, 19.6 -> 19.2, 5.7 -> 4.0, 12.4 ->
// 10.4; a step of four layers 216.9 -> 191.5.  Every workgroup does every row, so it loses from two rows on wherever there are many of them (gate_up 16.2 -> 19.4,
// down 10.3 -> 12.7; three rows of qkv 10.0 -> 12.6); without a row operation (`o`) four rows take 4.7 -> 4.3.  The entries take those too; the decode engine asks for the forms that
// gain.  Registers: gate_up of one row with groups of 128 behind two planes holds 253 of 256, behind four (not asked for) 16 - 34 spill.  The norm is compiled for rows of 4096, the width
// of everything measured.
#include "common.h"
#include "row_ops.h"

namespace {
constexpr int TPB = 256, WAVES = TPB / 64;
constexpr int ROWS_MOST = 4;
enum { FROM_INT8, FROM_NORM, FROM_ACT, FROM_WIDE_ACT };   // what the token rows are made of (activations of up to 4096 and of 8193 .. 16384 values)
enum { TO_HALF, TO_SILU, TO_PLANES };

struct RowsArgs {
    const uint8_t* W;
    const int8_t *zeros, *scales8;                   // per group
    const _Float16 *wscales, *wszs;
    void* out;
    int M, N, K, ks, epi_fma;
    // FROM_INT8
    const int8_t* A;
    const __half *ascales, *asums;
    // FROM_NORM: hidden + the planes of the product in front, normed with gamma; the sum goes to hidden_out
    const _Float16 *hidden, *gamma, *pws, *pwz;
    _Float16* hidden_out;
    const int* planes;
    size_t pstride;
    const __half *psa, *pss;
    float eps;
    // FROM_ACT, FROM_WIDE_ACT
    const _Float16* act;
    __half *scale_out, *sum_out;
};

template <int MODE, int TR, int S, int MR, int FROM, int TO, int PKS>
__global__ __launch_bounds__(TPB, 2) void rows_kernel(RowsArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ float sm[3 * 16];
    __shared__ float s_scale[MR], s_sum[MR];
    static_assert(TO != TO_SILU || TR == 2, "");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = (int)blockIdx.x / a.ks, kq = (int)blockIdx.x - tile * a.ks;
    const int nst = (a.K >> 6) / a.ks;                                   // 64-k stages of the slice
    const int per = MODE == 1 ? ((nst + 7) >> 3) * 2 : (nst + 3) >> 2;  // of a wave (per group: whole groups of 128)
    const int u0 = wave * per, n = min(max(nst - u0, 0), per);          // (a wave may have fewer, or none)
    const int first = kq * nst;                                          // global stage of the slice's first
    uint8_t* const rows = lds;                                           // int8 [MR][64 nst]
    const int rstride = 64 * nst;
    auto trow = [&](int t) { return TO == TO_SILU && t ? (a.N >> 6) + tile : tile; };       // 32-channel tile row
    const int ch = tid & 31;
    float ws[TR], wz[TR];
#pragma unroll
    for (int t = 0; t < TR; ++t) {
        ws[t] = (float)a.wscales[trow(t) * 32 + ch];
        wz[t] = MODE == 0 ? (float)a.wszs[trow(t) * 32 + ch] : 0.f;
    }

    // ---- the weights: everything this wave multiplies, requested in one go ----------------------------------------------
    constexpr int G = S / 2;                                             // groups of 128 k of a wave
    v4u w[TR][S];
    u32 sd[MODE == 1 ? TR : 1][MODE == 1 ? G : 1], zd[MODE == 1 ? TR : 1][MODE == 1 ? G : 1];
    auto request = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TR; ++t) {
            const uint8_t* const base = a.W + (size_t)trow(t) * (size_t)(a.K >> 5) * 512 + (size_t)first * 1024 + lane * 16;
            if (MODE == 1) {
                const size_t at = (size_t)trow(t) * 32 + ((lane >> 2) & 7) * 4;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const size_t row = (size_t)((first + min(u0 + 2 * g, nst - 1)) >> 1) * a.N;
                    sd[t][g] = *reinterpret_cast<const u32*>(a.scales8 + row + at);
                    zd[t][g] = *reinterpret_cast<const u32*>(a.zeros + row + at);
                }
            }
#pragma unroll
            for (int i = 0; i < S; ++i)
                w[t][i] = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(base + (size_t)min(u0 + i, nst - 1) * 1024));
        }
    };

    // ---- the token rows ----------------------------------------------------------------------------------------------------
    if constexpr (FROM == FROM_INT8) {
        v4u x[MR];                                                       // (at most 256 chunks of 16 a row)
#pragma unroll
        for (int m = 0; m < MR; ++m)
            x[m] = *reinterpret_cast<const v4u*>(a.A + (size_t)min(m, a.M - 1) * a.K + (size_t)first * 64 + min(tid * 16, rstride - 16));
        float sa = 0.f, ss = 0.f;
        if (tid < MR) {
            if (TO != TO_PLANES) sa = __half2float(a.ascales[min(tid, a.M - 1)]);
            if (TO != TO_PLANES && MODE == 0) ss = __half2float(a.asums[min(tid, a.M - 1)]);
        }
        __builtin_amdgcn_sched_barrier(0);
        request();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < MR; ++m)
            if (tid * 16 < rstride) *reinterpret_cast<v4u*>(rows + m * rstride + tid * 16) = x[m];
        if (tid < MR) {
            s_scale[tid] = sa;
            s_sum[tid] = ss;
        }
    } else if constexpr (FROM == FROM_NORM) {
        struct Sink {
            const RowsArgs& a;
            uint8_t* row;
            _Float16* hidden;
            float *scale, *sum;
            int tid;
            __device__ __forceinline__ bool want_sum() const { return MODE == 0; }
            __device__ __forceinline__ void chunk(int i, const float (&f)[8], float mul, h8 v) const {
                qs_store_q8(reinterpret_cast<int8_t*>(row) + i, f, mul);
                if (hidden) *reinterpret_cast<h8*>(hidden + i) = v;
            }
            __device__ __forceinline__ void row_done(float mx, float s) const {
                if (tid == 0) {                                          // as a tensor would hold them
                    *scale = __half2float(__float2half_rn(mx / 127.f));
                    *sum = __half2float(__float2half_rn(s));
                }
            }
        };
        struct SinkOf : Sink {
            __device__ __forceinline__ void row(float mx, float s) const { Sink::row_done(mx, s); }
        };
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            if (m >= a.M) break;
            qs_row::FromPlanes<PKS, MODE> dfn;
            const size_t base = (size_t)m * a.K;
            dfn.fma = a.epi_fma;
            dfn.row0 = a.planes + base;
            dfn.pstride = a.pstride;
            dfn.ws = a.pws;
            dfn.wz = a.pwz;
            dfn.sa = __half2float(a.psa[m]);
            dfn.ss = MODE == 0 ? __half2float(a.pss[m]) : 0.f;
            SinkOf sink{{a, rows + m * rstride, blockIdx.x == 0 ? a.hidden_out + base : nullptr, &s_scale[m], &s_sum[m], tid}};
            auto after = [&]() __attribute__((always_inline)) {
                if (m == 0) request();
            };
            qs_row::norm_quant_row<2, 4, 4, true, false, qs_row::NoHook, qs_row::FromPlanes<PKS, MODE>, true, false>(
                nullptr, const_cast<_Float16*>(a.hidden) + base, nullptr, a.gamma, nullptr, nullptr, a.eps, a.K, sm, tid, qs_row::NoHook(), dfn, nullptr, after, sink);
        }
    } else {
        struct Sink {
            uint8_t* row;                                                // of the slice: values [k0, k1)
            int k0, k1;
            __device__ __forceinline__ void chunk(int i, const float (&f)[8], float mul) const {
                if (i >= k0 && i < k1) qs_store_q8(reinterpret_cast<int8_t*>(row) + (i - k0), f, mul);
            }
        };
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            if (m >= a.M) break;
            const bool tell = blockIdx.x == 0;
            auto after = [&]() __attribute__((always_inline)) {
                if (m == 0) request();
            };
            if (m) __syncthreads();                                      // (the statistics' room is free again)
            __half* none = nullptr;
            // (the sum is made by every workgroup: it decides nothing here but the code is one)
            qs_row::quant_row<2, FROM == FROM_WIDE_ACT ? 16 : 4, 4, false>(nullptr, a.act + (size_t)m * a.K, MODE == 0 ? (tell ? a.sum_out + m : reinterpret_cast<__half*>(&s_sum[m])) : none,
                                               tell ? a.scale_out + m : none, a.K, sm, tid, qs_row::NoHook(), after,
                                               Sink{rows + m * rstride, first * 64, (first + nst) * 64});
        }
    }
    __syncthreads();

    // ---- dot products --------------------------------------------------------------------------------------------------------
    int acc[TR][4][MR];
#pragma unroll
    for (int t = 0; t < TR; ++t)
#pragma unroll
        for (int cl = 0; cl < 4; ++cl)
#pragma unroll
            for (int m = 0; m < MR; ++m) acc[t][cl][m] = 0;
    const u32* const row32 = reinterpret_cast<const u32*>(rows) + u0 * 16 + 8 * (lane >> 5) + (lane & 3);
    bool carries = false;
    if (MODE == 1) {
        u32 any = 0;
#pragma unroll
        for (int t = 0; t < TR; ++t)
#pragma unroll
            for (int g = 0; g < G; ++g) any |= level2_carries(sd[t][g]) ? 1u : 0u;
        carries = __builtin_amdgcn_ballot_w64(any != 0) != 0;
    }
    auto stages = [&](auto exact_) __attribute__((always_inline)) {
        constexpr bool EXACT = decltype(exact_)::value;
#pragma unroll
        for (int i = 0; i < S; ++i) {
            if (i >= n) break;
            u32 x[MR][2];
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                x[m][0] = row32[m * (rstride >> 2) + 16 * i];
                x[m][1] = row32[m * (rstride >> 2) + 16 * i + 4];
            }
#pragma unroll
            for (int t = 0; t < TR; ++t) {
                Level2 l2[MODE == 1 && !EXACT ? 4 : 1];
                if constexpr (MODE == 1 && !EXACT) {
#pragma unroll
                    for (int cl = 0; cl < 4; ++cl) l2[cl] = level2_of(sd[t][i >> 1], zd[t][i >> 1], cl);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {                            // dword q: k half q >> 1, channels cl = q & 1 and 2 + (q & 1)
                    const u32 raw = w[t][i][q];
#pragma unroll
                    for (int hi = 0; hi < 2; ++hi) {
                        const int cl = (q & 1) + 2 * hi;
                        u32 b;
                        if constexpr (MODE == 1 && !EXACT) b = unpack_level2(raw, hi, l2[cl]);
                        else {
                            u32 s = 0, zb = 0;
                            if (MODE == 1) {
                                s = (sd[t][i >> 1] >> (8 * cl)) & 0xFFu;
                                zb = ((zd[t][i >> 1] >> (8 * cl)) & 0xFFu) * 0x01010101u;
                            }
                            b = hi ? unpack_hi<MODE>(raw, s, zb) : unpack_lo<MODE>(raw, s, zb);
                        }
#pragma unroll
                        for (int m = 0; m < MR; ++m) acc[t][cl][m] = __builtin_amdgcn_sdot4((int)b, (int)x[m][q >> 1], acc[t][cl][m], false);
                    }
                }
            }
        }
    };
    if (MODE == 0) stages(std::true_type());
    else if (carries) stages(std::true_type());
    else stages(std::false_type());

    // ---- sums over the lanes of a channel (l & 3, l >> 5) and the waves; epilogue ---------------------------------------------
    __shared__ int red[WAVES][TR][MR][32];
#pragma unroll
    for (int t = 0; t < TR; ++t)
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int cl = 0; cl < 4; ++cl) {
                int v = acc[t][cl][m];
                v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);       // quad_perm [1, 0, 3, 2]
                v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);       // quad_perm [2, 3, 0, 1]
                const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
                v = (int)r[0] + (int)r[1];
                if ((lane & 35) == 0) red[wave][t][m][8 * cl + ((lane >> 2) & 7)] = v;
            }
    __syncthreads();
    const int m = tid >> 5;
    if (m >= a.M || m >= MR) return;
    _Float16 o[TR];
#pragma unroll
    for (int t = 0; t < TR; ++t) {
        int v = red[0][t][m][ch];
#pragma unroll
        for (int x = 1; x < WAVES; ++x) v += red[x][t][m][ch];
        if constexpr (TO == TO_PLANES) {
            reinterpret_cast<int*>(a.out)[((size_t)kq * a.M + m) * a.N + trow(t) * 32 + ch] = v;
        } else {
            float r = MODE == 0 ? epi_per_chn(v, ws[t], s_scale[m], wz[t], s_sum[m], a.epi_fma) : epi_per_group(v, ws[t], s_scale[m]);
            asm("" : "+v"(r));                                           // (a float of its own: the cast fused with the product would round only once)
            o[t] = (_Float16)r;
            if constexpr (TO == TO_HALF) reinterpret_cast<_Float16*>(a.out)[(size_t)m * a.N + trow(t) * 32 + ch] = o[t];
        }
    }
    if constexpr (TO == TO_SILU)
        reinterpret_cast<_Float16*>(a.out)[(size_t)m * (a.N >> 1) + tile * 32 + ch] = (_Float16)((float)qs_silu_h((float)o[0]) * (float)o[1]);
}

// ---- launches -----------------------------------------------------------------------------------------------------------------
bool rows_fit(int per_group, int M, int N, int K, int ks, bool pair) {
    if (M < 1 || M > ROWS_MOST || N <= 0 || N % 64 || K <= 0 || ks < 1 || K % (64 * ks)) return false;
    if (per_group && K % (128 * ks)) return false;
    const int nst = (K >> 6) / ks, per = per_group ? ((nst + 7) >> 3) * 2 : (nst + 3) >> 2;
    return per <= 16 && (int64_t)(N >> (pair ? 6 : 5)) * ks < (1 << 24);
}
template <int MODE, int FROM, int TO, int PKS>
void launch_rows(const RowsArgs& a, hipStream_t stream) {
    constexpr int TR = TO == TO_SILU ? 2 : 1;
    const int nst = (a.K >> 6) / a.ks, per = MODE == 1 ? ((nst + 7) >> 3) * 2 : (nst + 3) >> 2;
    const dim3 grid((unsigned)((a.N >> (TR == 2 ? 6 : 5)) * a.ks)), block(TPB);
#define QS_ROWS(S, MR) hipLaunchKernelGGL((rows_kernel<MODE, TR, S, MR, FROM, TO, PKS>), grid, block, (size_t)MR * 64 * nst, stream, a)
#define QS_ROWS_M(S)                 \
    do {                             \
        if (a.M == 1) QS_ROWS(S, 1); \
        else if (a.M == 2) QS_ROWS(S, 2); \
        else QS_ROWS(S, 4);          \
    } while (0)
    // (the loads of a wave are as many as its template says, those behind its last stage again the last line: the next of four sizes)
    if constexpr (FROM == FROM_INT8 || FROM == FROM_ACT) {
        if (per <= 4) {
            QS_ROWS_M(4);
            return;
        }
        if (per <= 8) {
            QS_ROWS_M(8);
            return;
        }
    }
    if constexpr (FROM != FROM_NORM) {
        if (per <= 12) {
            QS_ROWS_M(12);
            return;
        }
    }
    QS_ROWS_M(16);
#undef QS_ROWS_M
#undef QS_ROWS
}
bool on16(const void* p) { return ((uintptr_t)p & 15) == 0; }
}  // namespace

extern "C" int qs_w4a8_rows_ok(int per_group, int M, int N, int K, int k_slices) { return rows_fit(per_group != 0, M, N, K, k_slices, false); }

extern "C" int qs_w4a8_rows_planes(const int8_t* in_feats, const int8_t* kernel, const int8_t* zeros, const int8_t* scales_i8, int32_t* planes, int M, int N, int K,
                                   int k_slices, qs_stream_t stream) {
    QS_REQUIRE(in_feats && kernel && planes && (zeros == nullptr) == (scales_i8 == nullptr), "w4a8_rows_planes: null pointer");
    QS_REQUIRE(rows_fit(zeros != nullptr, M, N, K, k_slices, false) && K / k_slices <= 4096, "w4a8_rows_planes: %d x %d x %d in %d slices", M, N, K, k_slices);
    QS_REQUIRE(on16(in_feats) && on16(kernel) && on16(planes) && ((uintptr_t)zeros & 3) == 0 && ((uintptr_t)scales_i8 & 3) == 0, "w4a8_rows_planes: unaligned");
    RowsArgs a = {};
    a.W = (const uint8_t*)kernel, a.zeros = zeros, a.scales8 = scales_i8, a.out = planes, a.M = M, a.N = N, a.K = K, a.ks = k_slices, a.A = in_feats;
    a.wscales = a.wszs = (const _Float16*)kernel;                        // (read, not used)
    if (zeros) launch_rows<1, FROM_INT8, TO_PLANES, 1>(a, (hipStream_t)stream);
    else launch_rows<0, FROM_INT8, TO_PLANES, 1>(a, (hipStream_t)stream);
    return qs_launch_status("w4a8_rows_planes");
}

extern "C" int qs_norm_w4a8_rows(void* out, int silu_mul, const void* hidden, void* hidden_out, const int32_t* planes, int plane_slices, int64_t plane_stride,
                                 const void* plane_wscales, const void* plane_wszs, const void* plane_ascales, const void* plane_asums, const void* weight, float epsilon,
                                 const int8_t* kernel, const int8_t* zeros, const int8_t* scales_i8, const void* wscales, const void* wszs, int M, int N, int K,
                                 qs_stream_t stream) {
    const bool group = zeros != nullptr;
    QS_REQUIRE(out && hidden && hidden_out && hidden != hidden_out && planes && plane_wscales && plane_ascales && weight && kernel && wscales &&
                   group == (scales_i8 != nullptr) && group == (wszs == nullptr) && group == (plane_wszs == nullptr) && group == (plane_asums == nullptr),
               "norm_w4a8_rows: null pointer");
    QS_REQUIRE(K == 4096 && rows_fit(group, M, N, K, 1, silu_mul != 0) && (plane_slices == 2 || plane_slices == 4) && plane_stride >= (int64_t)M * K && plane_stride % 4 == 0,
               "norm_w4a8_rows: %d x %d x %d behind %d planes", M, N, K, plane_slices);
    QS_REQUIRE(on16(hidden) && on16(hidden_out) && on16(planes) && on16(plane_wscales) && on16(plane_wszs) && on16(weight) && on16(kernel) && ((uintptr_t)zeros & 3) == 0 &&
                   ((uintptr_t)scales_i8 & 3) == 0, "norm_w4a8_rows: unaligned");
    RowsArgs a = {};
    a.W = (const uint8_t*)kernel, a.zeros = zeros, a.scales8 = scales_i8, a.wscales = (const _Float16*)wscales, a.wszs = (const _Float16*)wszs, a.out = out;
    a.M = M, a.N = N, a.K = K, a.ks = 1, a.epi_fma = g_epi_fma;
    a.hidden = (const _Float16*)hidden, a.hidden_out = (_Float16*)hidden_out, a.gamma = (const _Float16*)weight, a.pws = (const _Float16*)plane_wscales;
    a.pwz = (const _Float16*)plane_wszs, a.planes = planes, a.pstride = (size_t)plane_stride, a.psa = (const __half*)plane_ascales, a.pss = (const __half*)plane_asums;
    a.eps = epsilon;
    const hipStream_t s = (hipStream_t)stream;
#define QS_NORM_ROWS(MODE, TO)                                                   \
    do {                                                                         \
        if (plane_slices == 2) launch_rows<MODE, FROM_NORM, TO, 2>(a, s);        \
        else launch_rows<MODE, FROM_NORM, TO, 4>(a, s);                          \
    } while (0)
    if (group && silu_mul) QS_NORM_ROWS(1, TO_SILU);
    else if (group) QS_NORM_ROWS(1, TO_HALF);
    else if (silu_mul) QS_NORM_ROWS(0, TO_SILU);
    else QS_NORM_ROWS(0, TO_HALF);
#undef QS_NORM_ROWS
    return qs_launch_status("norm_w4a8_rows");
}

extern "C" int qs_quant_w4a8_rows_planes(int32_t* planes, const void* act, void* scale, void* input_sum, const int8_t* kernel, const int8_t* zeros, const int8_t* scales_i8,
                                         int M, int N, int K, int k_slices, qs_stream_t stream) {
    const bool group = zeros != nullptr;
    QS_REQUIRE(planes && act && scale && kernel && group == (scales_i8 != nullptr) && group == (input_sum == nullptr), "quant_w4a8_rows_planes: null pointer");
    const bool wide = K > 8192;                                          // (invoke_quant's two layouts of these widths, row_ops.h)
    QS_REQUIRE((wide || (K > 2048 && K <= 4096)) && K <= 16384 && rows_fit(group, M, N, K, k_slices, false), "quant_w4a8_rows_planes: %d x %d x %d in %d slices", M, N, K, k_slices);
    QS_REQUIRE(on16(planes) && on16(act) && on16(kernel) && ((uintptr_t)zeros & 3) == 0 && ((uintptr_t)scales_i8 & 3) == 0, "quant_w4a8_rows_planes: unaligned");
    RowsArgs a = {};
    a.W = (const uint8_t*)kernel, a.zeros = zeros, a.scales8 = scales_i8, a.out = planes, a.M = M, a.N = N, a.K = K, a.ks = k_slices;
    a.act = (const _Float16*)act, a.scale_out = (__half*)scale, a.sum_out = (__half*)input_sum;
    a.wscales = a.wszs = (const _Float16*)kernel;                        // (read, not used)
    const hipStream_t st = (hipStream_t)stream;
    if (group && wide) launch_rows<1, FROM_WIDE_ACT, TO_PLANES, 1>(a, st);
    else if (group) launch_rows<1, FROM_ACT, TO_PLANES, 1>(a, st);
    else if (wide) launch_rows<0, FROM_WIDE_ACT, TO_PLANES, 1>(a, st);
    else launch_rows<0, FROM_ACT, TO_PLANES, 1>(a, st);
    return qs_launch_status("quant_w4a8_rows_planes");
}
