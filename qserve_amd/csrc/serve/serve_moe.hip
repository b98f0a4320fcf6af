// serve_moe.hip -- mixture of experts: grouped top-k router and the per-token expert products (wave-per-output-row form).
//
// Router scores are float from the first product to the chosen weights.  The expert kernels keep one token's input in LDS
// and let every wave walk output rows with its lanes spread along the reduction (coalesced weight rows).
#include "serve_common.h"
#include "serve_expert_rows.h"
#include "serve_route.h"

namespace {
constexpr int NT = 256;
constexpr int NW = NT / 64;
constexpr int MAX_EXPERTS = 1024;

__device__ __forceinline__ void loadv(const bf16_t* p, float (&v)[4]) {
    const uint2 u = *(const uint2*)p;
    v[0] = __uint_as_float(u.x << 16);
    v[1] = __uint_as_float(u.x & 0xffff0000u);
    v[2] = __uint_as_float(u.y << 16);
    v[3] = __uint_as_float(u.y & 0xffff0000u);
}
__device__ __forceinline__ void loadv(const float* p, float (&v)[4]) {
    const float4 a = *(const float4*)p;
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
template <typename T>
__device__ __forceinline__ void loadv(const T* p, float (&v)[1]) { v[0] = ld(p, 0); }
__device__ __forceinline__ void storev(bf16_t* p, const float (&v)[4]) {
    *(uint2*)p = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
}
__device__ __forceinline__ void storev(float* p, const float (&v)[4]) { *(float4*)p = make_float4(v[0], v[1], v[2], v[3]); }
template <typename T>
__device__ __forceinline__ void storev(T* p, const float (&v)[1]) { st(p, 0, v[0]); }
// (value, index) of the largest value over a wave; ties go to the lower index.  Lanes without a candidate pass index -1.
__device__ __forceinline__ void wave_argmax(float& v, int& i) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(v, o, 64);
        const int oi = __shfl_xor(i, o, 64);
        if (oi >= 0 && (i < 0 || ov > v || (ov == v && oi < i))) {
            v = ov;
            i = oi;
        }
    }
}

// One workgroup per token.  z = router . h by the four waves (16-byte loads where the width allows), then wave 0 selects by
// repeated wave-wide argmax.  Scores s = softmax(z) over all experts (score_fn 0) or sigmoid(z) (1); the CHOICE goes by c = s +
// correction (correction may be NULL), the WEIGHTS are the chosen experts' s times `scale` (divided by their sum first if renorm).
// A group's score is its largest c (group_top 1) or the sum of its two largest (2); experts outside the `keep` best groups cannot
// be chosen, however low the others' c.  Ties go to the lower index, for groups and for experts.
template <typename T>
__global__ __launch_bounds__(NT) void moe_route_kernel(int32_t* __restrict__ idx, float* __restrict__ weight,
                                                       const T* __restrict__ h, const T* __restrict__ router,
                                                       const T* __restrict__ bias, int renorm, int D, int E, int top_k, int G,
                                                       int keep, int score_fn, const float* __restrict__ correction,
                                                       int group_top, float scale) {
    __shared__ float s[MAX_EXPERTS];
    __shared__ float c[MAX_EXPERTS];
    __shared__ float gs[MAX_EXPERTS];
    __shared__ unsigned char ok[MAX_EXPERTS];
    __shared__ unsigned char gtaken[MAX_EXPERTS];
    const size_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const T* x = h + t * D;
    for (int e = w; e < E; e += NW) {
        const T* r = router + (size_t)e * D;
        float d = 0.f;
        if (D % 8 == 0) {
            for (int cc = lane * 8; cc < D; cc += 64 * 8) {
                float a[8], b[8];
                load8(r + cc, a);
                load8(x + cc, b);
#pragma unroll
                for (int q = 0; q < 8; ++q) d += a[q] * b[q];
            }
        } else {
            for (int i = lane; i < D; i += 64) d += ld(r, i) * ld(x, i);
        }
        d = wave_sum(d);
        if (lane == 0) s[e] = bias ? d + ld(bias, e) : d;
    }
    __syncthreads();
    // (the other three waves only keep the barriers company from here on: the selection is a few hundred steps of one wave)
    const bool sel = w == 0;
    if (sel) {
        if (score_fn == 0) {                                // softmax over all experts
            float mx = -INFINITY;
            for (int e = lane; e < E; e += 64) mx = fmaxf(mx, s[e]);
            mx = wave_max(mx);
            float sum = 0.f;
            for (int e = lane; e < E; e += 64) {
                const float p = expf(s[e] - mx);
                s[e] = p;
                sum += p;
            }
            const float inv = 1.0f / wave_sum(sum);
            for (int e = lane; e < E; e += 64) s[e] *= inv;
        } else {
            for (int e = lane; e < E; e += 64) s[e] = 1.0f / (1.0f + expf(-s[e]));
        }
        for (int e = lane; e < E; e += 64) {
            c[e] = correction ? s[e] + correction[e] : s[e];
            ok[e] = 0;
        }
    }
    __syncthreads();
    const int per = E / G;
    if (sel) {                                              // group scores
        for (int g = lane; g < G; g += 64) {
            float v1 = c[g * per], v2 = -INFINITY;          // the two largest
            for (int e = 1; e < per; ++e) {
                const float v = c[g * per + e];
                if (v > v1) {
                    v2 = v1;
                    v1 = v;
                } else if (v > v2) {
                    v2 = v;
                }
            }
            gs[g] = (group_top == 2 && per > 1) ? v1 + v2 : v1;
            gtaken[g] = 0;
        }
    }
    __syncthreads();
    for (int k = 0; k < keep; ++k) {                        // the `keep` best groups
        if (sel) {
            float bv = 0.f;
            int bi = -1;
            for (int g = lane; g < G; g += 64)
                if (!gtaken[g] && (bi < 0 || gs[g] > bv)) {
                    bv = gs[g];
                    bi = g;
                }
            wave_argmax(bv, bi);
            if (lane == 0) gtaken[bi] = 1;
            for (int e = lane; e < per; e += 64) ok[bi * per + e] = 1;
        }
        __syncthreads();
    }
    float chosen = 0.f;                                     // (lane 0 of the selecting wave: sum of the chosen scores)
    for (int k = 0; k < top_k; ++k) {                       // the top_k eligible experts
        if (sel) {
            float bv = 0.f;
            int bi = -1;
            for (int e = lane; e < E; e += 64)
                if (ok[e] && (bi < 0 || c[e] > bv)) {
                    bv = c[e];
                    bi = e;
                }
            wave_argmax(bv, bi);
            if (lane == 0) {
                ok[bi] = 0;
                idx[t * top_k + k] = bi;
                weight[t * top_k + k] = s[bi];
                chosen += s[bi];
            }
        }
        __syncthreads();
    }
    // weights over the chosen only: p_i / sum of the chosen p = the softmax over the chosen logits
    if (sel && lane == 0 && (renorm || scale != 1.0f))
        for (int k = 0; k < top_k; ++k) {
            float v = weight[t * top_k + k];
            if (renorm) v /= chosen;
            weight[t * top_k + k] = v * scale;
        }
}

// The same for at most 64 experts and widths that are multiples of 8 (one expert per lane in the selection).  The wide form's time went
// into serial steps: a wave took its experts one by one, six shuffles each, and the selection was (keep + top_k) wave-wide argmax searches
// with a barrier each.  Here the four waves split the width and hold EC experts' sums for TT tokens side by side, the sums are reduced and
// scattered over the lanes in one butterfly, and a lane finds its expert's place by counting the better ones (broadcasts, no search).
// TT = 4 tokens share the router's rows in prompts; in steps one token per workgroup keeps more workgroups busy.
template <typename T, int TT, int EC>
__global__ __launch_bounds__(NT, 2) void moe_route_wave_kernel(int32_t* __restrict__ idx, float* __restrict__ weight, const T* __restrict__ h,
                                                            const T* __restrict__ router, const T* __restrict__ bias, int renorm, int n, int D, int E,
                                                            int top_k, int G, int keep, int score_fn, const float* __restrict__ correction,
                                                            int group_top, float scale) {
    constexpr int NV = TT * EC;
    __shared__ float part[NW][TT][64];
    __shared__ float cs[NW][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const size_t t0 = (size_t)blockIdx.x * TT;
    const float lane_bias = bias && lane < E ? ld(bias, lane) : 0.f, lane_corr = correction && lane < E ? correction[lane] : 0.f;
    for (int e0 = 0; e0 < E; e0 += EC) {
        float v[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = 0.f;
        for (int c = threadIdx.x * 8; c < D; c += NT * 8) {
            typename Piece<T>::type xr[TT], rr[EC];                // every load in flight before the first is used
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) xr[tt] = *(const typename Piece<T>::type*)(h + min(t0 + tt, (size_t)n - 1) * D + c);
#pragma unroll
            for (int e = 0; e < EC; ++e) rr[e] = *(const typename Piece<T>::type*)(router + (size_t)min(e0 + e, E - 1) * D + c);
            __builtin_amdgcn_sched_barrier(0);
            float x[TT][8];
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) load8((const T*)&xr[tt], x[tt]);
#pragma unroll
            for (int e = 0; e < EC; ++e) {
                float r[8];
                load8((const T*)&rr[e], r);
#pragma unroll
                for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                    for (int q = 0; q < 8; ++q) v[tt * EC + e] += r[q] * x[tt][q];
            }
        }
        wave_sum_scatter<NV>(v, lane);
        const int id = lane / (64 / NV);
        if (lane % (64 / NV) == 0) part[w][id / EC][e0 + id % EC] = v[0];
    }
    __syncthreads();
    if (w >= TT || t0 + w >= (size_t)n) return;                  // wave w selects for token w (no barrier follows)
    const size_t t = t0 + w;
    float s = 0.f;
    if (lane < E) {
#pragma unroll
        for (int o = 0; o < NW; ++o) s += part[o][w][lane];
    }
    select_experts(s, lane_bias, lane_corr, {idx, weight, router, bias, correction, renorm, E, top_k, G, keep, score_fn, group_top, scale}, t, cs[w], lane);
}

// One workgroup per (token, chosen expert): act = relu(up_e . h)^2 (or the gated unit).  Dynamic LDS: D floats.  ff: weight rows.
template <typename T, int ACT>
__global__ __launch_bounds__(NT) void moe_up_kernel(T* __restrict__ act, const T* __restrict__ h, const T* __restrict__ up,
                                                    const int32_t* __restrict__ idx, int top_k, int D, int ff, float limit, int n_experts,
                                                        const float* __restrict__ in_weight) {
    extern __shared__ float xs[];
    const size_t slot = blockIdx.x;
    if ((unsigned)idx[slot] >= (unsigned)n_experts) return;  // an identity expert: the down kernel adds the input itself (below 0: none)
    const size_t t = slot / top_k;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < D; i += NT) xs[i] = ld(h, t * D + i);
    __syncthreads();
    const T* W = up + (size_t)idx[slot] * ff * D;
    const float iw = in_weight ? in_weight[slot] : 1.0f;     // the expert works on iw * h
    if (ACT == ACT_GLU) {
        for (int f = w; f < ff / 2; f += NW) {
            const T* r = W + (size_t)(2 * f) * D;
            float d = 0.f, e = 0.f;
            for (int i = lane; i < D; i += 64) {
                d += ld(r, i) * xs[i];
                e += ld(r, D + i) * xs[i];
            }
            d = wave_sum(d);
            e = wave_sum(e);
            if (lane == 0) st(act, slot * (ff / 2) + f, glu(iw * d, iw * e, limit));
        }
        return;
    }
    for (int f = w; f < ff; f += NW) {
        const T* r = W + (size_t)f * D;
        float d = 0.f;
        for (int i = lane; i < D; i += 64) d += ld(r, i) * xs[i];
        d = wave_sum(d);
        if (lane == 0) st(act, slot * ff + f, relu_sq(iw * d));
    }
}

// One workgroup per token: y = sum_k weight_k * down_{e_k} . act_k.  Dynamic LDS: top_k * ff floats.
template <typename T>
__global__ __launch_bounds__(NT) void moe_down_kernel(T* __restrict__ y, const T* __restrict__ act, const T* __restrict__ down,
                                                      const int32_t* __restrict__ idx, const float* __restrict__ weight,
                                                      int top_k, int D, int ff, const T* __restrict__ h, int n_experts) {
    extern __shared__ float as[];
    const size_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < top_k * ff; i += NT) as[i] = ld(act, t * top_k * ff + i);
    __syncthreads();
    for (int d = w; d < D; d += NW) {
        float total = 0.f;
        for (int k = 0; k < top_k; ++k) {
            if (idx[t * top_k + k] < 0) continue;            // no expert
            if (idx[t * top_k + k] >= n_experts) {           // identity expert
                total += (weight ? weight[t * top_k + k] : 1.0f) * ld(h, t * D + d);
                continue;
            }
            const T* r = down + ((size_t)idx[t * top_k + k] * D + d) * ff;
            float v = 0.f;
            for (int i = lane; i < ff; i += 64) v += ld(r, i) * as[k * ff + i];
            total += (weight ? weight[t * top_k + k] : 1.0f) * wave_sum(v);
        }
        if (lane == 0) st(y, t * D + d, total);
    }
}

// The same two kernels for widths that are multiples of 8: 16-byte weight loads and four output rows per wave in flight at once
// (the scalar forms above wait for one row's loads before they issue the next row's: latency-bound at real layer sizes).
constexpr int ROWS = 4;      // output rows a wave works on at once

template <typename T, int ACT>
__global__ __launch_bounds__(NT) void moe_up_vec_kernel(T* __restrict__ act, const T* __restrict__ h, const T* __restrict__ up,
                                                        const int32_t* __restrict__ idx, int top_k, int D, int ff, float limit, int n_experts,
                                                        const float* __restrict__ in_weight) {
    extern __shared__ float xs[];
    const size_t slot = blockIdx.x;
    if ((unsigned)idx[slot] >= (unsigned)n_experts) return;  // an identity expert: the down kernel adds the input itself (below 0: none)
    const size_t t = slot / top_k;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < D; i += NT) xs[i] = ld(h, t * D + i);
    __syncthreads();
    const T* W = up + (size_t)idx[slot] * ff * D;
    const float iw = in_weight ? in_weight[slot] : 1.0f;     // the expert works on iw * h
    for (int f0 = w * ROWS; f0 < ff; f0 += NW * ROWS) {
        float acc[ROWS] = {0.f, 0.f, 0.f, 0.f};
        for (int c = lane * 8; c < D; c += 64 * 8) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = xs[c + e];
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                if (f0 + r < ff) {
                    float v[8];
                    load8(W + (size_t)(f0 + r) * D + c, v);
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[r] += v[e] * x[e];
                }
            }
        }
        float d[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) d[r] = iw * wave_sum(acc[r]);
        if (lane == 0) {
            if (ACT == ACT_GLU) {                               // (ROWS and ff are even: a pair never straddles two waves)
#pragma unroll
                for (int r = 0; r < ROWS; r += 2)
                    if (f0 + r < ff) st(act, slot * (ff / 2) + (f0 + r) / 2, glu(d[r], d[r + 1], limit));
            } else {
#pragma unroll
                for (int r = 0; r < ROWS; ++r)
                    if (f0 + r < ff) st(act, slot * ff + f0 + r, relu_sq(d[r]));
            }
        }
    }
}

template <typename T>
__global__ __launch_bounds__(NT) void moe_down_vec_kernel(T* __restrict__ y, const T* __restrict__ act, const T* __restrict__ down,
                                                          const int32_t* __restrict__ idx, const float* __restrict__ weight,
                                                          int top_k, int D, int ff, const T* __restrict__ h, int n_experts) {
    extern __shared__ float as[];
    const size_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < top_k * ff; i += NT) as[i] = ld(act, t * top_k * ff + i);
    __syncthreads();
    for (int d0 = w * ROWS; d0 < D; d0 += NW * ROWS) {
        float acc[ROWS] = {0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < top_k; ++k) {
            const float wk = weight ? weight[t * top_k + k] : 1.0f;
            if (idx[t * top_k + k] < 0) continue;            // no expert
            if (idx[t * top_k + k] >= n_experts) {           // identity expert: lane 0's share carries the input (the rest add zero)
                if (lane == 0) {
#pragma unroll
                    for (int r = 0; r < ROWS; ++r)
                        if (d0 + r < D) acc[r] += wk * ld(h, t * D + d0 + r);
                }
                continue;
            }
            const T* Wk = down + (size_t)idx[t * top_k + k] * D * ff;
            float part[ROWS] = {0.f, 0.f, 0.f, 0.f};
            for (int c = lane * 8; c < ff; c += 64 * 8) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = as[k * ff + c + e];
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    if (d0 + r < D) {
                        float v[8];
                        load8(Wk + (size_t)(d0 + r) * ff + c, v);
#pragma unroll
                        for (int e = 0; e < 8; ++e) part[r] += v[e] * x[e];
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < ROWS; ++r) acc[r] += wk * part[r];
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const float v = wave_sum(acc[r]);
            if (lane == 0 && d0 + r < D) st(y, t * D + d0 + r, v);
        }
    }
}

// expert_rows_block (serve_expert_rows.h) as a launch of its own
template <int ACT, bool FOUT, int FORM>
__global__ __launch_bounds__(NT, 2) void expert_rows_kernel(ExpertArgs a, SharedArgs sh) {
    __shared__ __attribute__((aligned(128))) unsigned char lds[EXPERT_LDS];
    expert_rows_block<ACT, FOUT, FORM>(a, sh, blockIdx.x, blockIdx.y, lds);
}

// ---- expert-sorted form (many tokens): the products are the vendor's, per expert over contiguous runs of sorted slots; these
// kernels do the permutation in, the activation, and the weighted permutation out -----------------------------------------------
template <typename T>
__global__ __launch_bounds__(NT) void gather_rows_kernel(T* __restrict__ out, const T* __restrict__ src,
                                                         const int64_t* __restrict__ order, int div, int width) {
    const size_t i = blockIdx.x;
    const T* s = src + (size_t)(order[i] / div) * width;
    for (int c = threadIdx.x; c < width; c += NT) out[i * width + c] = s[c];
}
template <typename T>
__global__ __launch_bounds__(NT) void relu_sq_kernel(T* __restrict__ a, size_t n) {
    const size_t i = (size_t)blockIdx.x * NT + threadIdx.x;
    if (i < n) {
        const float v = fmaxf(ld(a, i), 0.f);
        st(a, i, v * v);
    }
}
// y[t] = sum_k weight[t, k] * ys[inv ? inv[t top_k + k] : t top_k + k]   (weight NULL: ones).  VEC coordinates per thread.
template <typename T, typename Y, int VEC, typename I>
__global__ __launch_bounds__(NT) void moe_combine_kernel(T* __restrict__ y, const Y* __restrict__ ys, const I* __restrict__ inv,
                                                         const float* __restrict__ weight, int top_k, int D,
                                                         const int32_t* __restrict__ idx, const T* __restrict__ h, int n_experts) {
    const size_t t = blockIdx.x;
    for (int c = (blockIdx.y * NT + threadIdx.x) * VEC; c < D; c += gridDim.y * NT * VEC) {
        float a[VEC] = {};
#pragma unroll 4
        for (int k = 0; k < top_k; ++k) {
            const size_t slot = t * top_k + k;
            const int e = idx ? idx[slot] : 0;
            const bool none = e < 0;                                        // no expert: the slot has neither a row nor a place
            const bool same = idx && (unsigned)e >= (unsigned)n_experts;    // an identity expert's slot has no row of its own
            const float wk = weight ? weight[slot] : 1.0f;
            float v[VEC];
            if (same) loadv(h + t * D + c, v);
            else loadv(ys + (inv ? (size_t)inv[slot] : slot) * D + c, v);
            // (taken out by value: behind a jump the slots' rows are requested one after another: 8192 tokens of 2048, top 4, 29 us against 40)
#pragma unroll
            for (int q = 0; q < VEC; ++q) {
                const float sum = a[q] + wk * v[q];
                a[q] = none ? a[q] : sum;
            }
        }
        storev(y + t * D + c, a);
    }
}
}  // namespace

extern "C" int qsv_gather_rows(void* out, const void* src, const int64_t* order, int div, int n_rows, int width, int dtype,
                               void* stream) {
    QSV_REQUIRE(out && src && order && div > 0 && n_rows >= 0 && width > 0, "qsv_gather_rows: bad arguments");
    if (n_rows == 0) return QSV_OK;
    QSV_DISPATCH(dtype, "qsv_gather_rows",
                 hipLaunchKernelGGL(gather_rows_kernel<T>, dim3(n_rows), dim3(NT), 0, (hipStream_t)stream, (T*)out, (const T*)src,
                                    order, div, width));
    return qsv_launch_status("qsv_gather_rows");
}
static int launch_expert_rows(const char* what, ExpertArgs a, int n_experts, int act, bool float_out, void* stream, SharedArgs sh = {}, bool kept = false) {
    dim3 grid;
    const int rc = plan_expert_rows(what, a, sh, n_experts, act, kept, grid);
    if (rc != QSV_OK) return rc;
    const dim3 block(NT);
    const bool early = early_experts(a, n_experts);
#define QSV_EXPERTS(ACT, FOUT)                                                                                                                          \
    do {                                                                                                                                                \
        auto kernel = early ? expert_rows_kernel<ACT, FOUT, SLOTS_EARLY> : few_slots(a, sh) ? expert_rows_kernel<ACT, FOUT, SLOTS_FEW> : expert_rows_kernel<ACT, FOUT, SLOTS>; \
        if constexpr (!FOUT) kernel = a.offsets ? expert_rows_kernel<ACT, FOUT, SORTED_RUNS> : kernel;                                                  \
        hipLaunchKernelGGL(kernel, grid, block, 0, (hipStream_t)stream, a, sh);                                                                         \
    } while (0)
    if (float_out) QSV_EXPERTS(ACT_NONE, true);                                    // (never sorted runs)
    else if (act == ACT_RELU_SQ) QSV_EXPERTS(ACT_RELU_SQ, false);
    else if (act == ACT_GLU) QSV_EXPERTS(ACT_GLU, false);
    else QSV_EXPERTS(ACT_NONE, false);
#undef QSV_EXPERTS
    return qsv_launch_status(what);
}
extern "C" int qsv_expert_rows(void* out, const void* X, const int64_t* x_index, int div, const void* W, const int64_t* offsets,
                               int n_experts, int rows, int K, int act, float limit, const float* in_weight, void* stream) {
    QSV_REQUIRE(offsets, "qsv_expert_rows: bad arguments");
    const ExpertArgs a = {out, (const bf16_t*)X, (const bf16_t*)W, nullptr, x_index, offsets, in_weight, 0, div, rows, K, limit, false, false, false, 0};
    return launch_expert_rows("qsv_expert_rows", a, n_experts, act, false, stream);
}
extern "C" int qsv_expert_slots(void* out, int float_out, const void* X, int div, const void* W, const int32_t* idx, int n, int n_experts, int rows,
                                int K, int act, float limit, const float* in_weight, void* stream) {
    QSV_REQUIRE(idx && n >= 0 && (!float_out || act == ACT_NONE), "qsv_expert_slots: bad arguments");
    if (n == 0) return QSV_OK;
    const ExpertArgs a = {out, (const bf16_t*)X, (const bf16_t*)W, idx, nullptr, nullptr, in_weight, n, div, rows, K, limit, false, false, false, 0};
    return launch_expert_rows("qsv_expert_slots", a, n_experts, act, float_out != 0, stream);
}
// ... and, with sh_W, every token's row of X through a shared expert of sh_rows x sh_K in the same launch: sh_out [n / div, sh_rows (/ 2 for gated units)]
static int launch_expert_slots(const char* what, const qsv_expert_job& j, void* stream) {
    QSV_REQUIRE(j.n_experts < 65535, "%s: bad arguments", what);
    ExpertArgs a;
    SharedArgs sh;
    const int rc = expert_slots_args(what, j, a, sh);
    return rc != QSV_OK || j.n == 0 ? rc : launch_expert_rows(what, a, j.n_experts, j.act, j.float_out != 0, stream, sh, j.kept != 0);
}
extern "C" int qsv_expert_slots_shared(void* out, int float_out, const void* X, int div, const void* W, const int32_t* idx, int n, int n_experts, int rows, int K,
                                       int act, float limit, const float* in_weight, void* sh_out, const void* sh_X, const void* sh_W, int sh_n, int sh_rows, int sh_K,
                                       void* stream) {
    QSV_REQUIRE(sh_W, "qsv_expert_slots_shared: bad arguments");
    return launch_expert_slots("qsv_expert_slots_shared", {out, X, W, idx, in_weight, sh_out, sh_X, sh_W, float_out, div, n, n_experts, rows, K, act, sh_n, sh_rows, sh_K, 0,
                                                           limit}, stream);
}
// either of them (sh_W NULL: no shared expert) with weights that are to stay in the caches
extern "C" int qsv_expert_slots_kept(void* out, int float_out, const void* X, int div, const void* W, const int32_t* idx, int n, int n_experts, int rows, int K, int act,
                                     float limit, const float* in_weight, void* sh_out, const void* sh_X, const void* sh_W, int sh_n, int sh_rows, int sh_K, void* stream) {
    return launch_expert_slots("qsv_expert_slots_kept", {out, X, W, idx, in_weight, sh_out, sh_X, sh_W, float_out, div, n, n_experts, rows, K, act, sh_n, sh_rows, sh_K, 1,
                                                         limit}, stream);
}
extern "C" int qsv_relu_sq(void* a, int64_t n, int dtype, void* stream) {
    QSV_REQUIRE(a && n >= 0 && n < (1ll << 31) * NT, "qsv_relu_sq: bad arguments");
    if (n == 0) return QSV_OK;
    QSV_DISPATCH(dtype, "qsv_relu_sq",
                 hipLaunchKernelGGL(relu_sq_kernel<T>, dim3((unsigned)((n + NT - 1) / NT)), dim3(NT), 0, (hipStream_t)stream, (T*)a,
                                    (size_t)n));
    return qsv_launch_status("qsv_relu_sq");
}
// (four coordinates per thread where the rows' starts allow it; few tokens: a token's row over several workgroups)
template <typename T, typename Y, typename I>
static void launch_combine(void* y, const void* ys, const I* inv, const float* weight, int n, int top_k, int D, const int32_t* idx,
                           const void* h, int n_experts, void* stream) {
    const bool vec = D % 4 == 0 && ((uintptr_t)ys % (4 * sizeof(Y)) == 0) && ((uintptr_t)y % (4 * sizeof(T)) == 0) && (!h || (uintptr_t)h % (4 * sizeof(T)) == 0);
    const int per = NT * (vec ? 4 : 1), need = (D + per - 1) / per;
    const dim3 grid(n, n < 1024 ? need : 1);
    if (vec)
        hipLaunchKernelGGL((moe_combine_kernel<T, Y, 4, I>), grid, dim3(NT), 0, (hipStream_t)stream, (T*)y, (const Y*)ys, inv, weight, top_k, D, idx,
                           (const T*)h, n_experts);
    else
        hipLaunchKernelGGL((moe_combine_kernel<T, Y, 1, I>), grid, dim3(NT), 0, (hipStream_t)stream, (T*)y, (const Y*)ys, inv, weight, top_k, D, idx,
                           (const T*)h, n_experts);
}
extern "C" int qsv_moe_combine(void* y, const void* ys, const int64_t* inv, const float* weight, int n, int top_k, int D,
                               const int32_t* idx, const void* h, int n_experts, int dtype, void* stream) {
    QSV_REQUIRE(y && ys && inv && n >= 0 && top_k > 0 && D > 0 && (!idx || h), "qsv_moe_combine: bad arguments");
    if (n == 0) return QSV_OK;
    QSV_DISPATCH(dtype, "qsv_moe_combine", (launch_combine<T, T, int64_t>(y, ys, inv, weight, n, top_k, D, idx, h, n_experts, stream)));
    return qsv_launch_status("qsv_moe_combine");
}
extern "C" int qsv_moe_combine_sorted(void* y, const void* ys, const int32_t* place, const float* weight, int n, int top_k, int D, const int32_t* idx,
                                      const void* h, int n_experts, int dtype, void* stream) {
    QSV_REQUIRE(y && ys && place && n >= 0 && top_k > 0 && D > 0 && (!idx || h), "qsv_moe_combine_sorted: bad arguments");
    if (n == 0) return QSV_OK;
    QSV_DISPATCH(dtype, "qsv_moe_combine_sorted", (launch_combine<T, T, int32_t>(y, ys, place, weight, n, top_k, D, idx, h, n_experts, stream)));
    return qsv_launch_status("qsv_moe_combine_sorted");
}
extern "C" int qsv_moe_combine_slots(void* y, const float* ys, const float* weight, int n, int top_k, int D, const int32_t* idx, const void* h,
                                     int n_experts, int dtype, void* stream) {
    QSV_REQUIRE(y && ys && n >= 0 && top_k > 0 && D > 0 && (!idx || h), "qsv_moe_combine_slots: bad arguments");
    if (n == 0) return QSV_OK;
    QSV_DISPATCH(dtype, "qsv_moe_combine_slots", (launch_combine<T, float, int32_t>(y, ys, nullptr, weight, n, top_k, D, idx, h, n_experts, stream)));
    return qsv_launch_status("qsv_moe_combine_slots");
}

extern "C" int qsv_moe_route(int32_t* idx, float* weight, const void* h, const void* router, const void* bias, int renorm, int n,
                             int D, int E, int top_k, int G, int keep, int score_fn, const float* correction, int group_top,
                             float scale, int dtype, void* stream) {
    QSV_REQUIRE((score_fn == 0 || score_fn == 1) && (group_top == 1 || group_top == 2), "qsv_moe_route: score function %d, group score %d",
                score_fn, group_top);
    QSV_REQUIRE(idx && weight && h && router && n >= 0 && D > 0, "qsv_moe_route: bad arguments");
    QSV_REQUIRE(E > 0 && E <= MAX_EXPERTS && G > 0 && E % G == 0 && keep > 0 && keep <= G && top_k > 0 &&
                    top_k <= keep * (E / G),
                "qsv_moe_route: %d experts in %d groups, %d groups kept, top %d", E, G, keep, top_k);
    if (n == 0) return QSV_OK;
    if (E <= 64 && D % 8 == 0) {
#define QSV_ROUTE(TT, EC)                                                                                                         \
    QSV_DISPATCH(dtype, "qsv_moe_route",                                                                                         \
                 hipLaunchKernelGGL((moe_route_wave_kernel<T, TT, EC>), dim3((n + TT - 1) / TT), dim3(NT), 0, (hipStream_t)stream, idx, weight, \
                                    (const T*)h, (const T*)router, (const T*)bias, renorm, n, D, E, top_k, G, keep, score_fn, correction, \
                                    group_top, scale))
        // four tokens a workgroup where the router's rows are long or the tokens fill the chip all the same (1024 tokens, 64 experts of 64, one token /
        // four: 14.9 / 19.1 us; 8 of 8192 13.8 / 11.9); eight sums side by side for at most eight experts (1000 tokens, 2 of 8192: 13.6 -> 8.5 us)
        const bool four = n >= 1024 && (D >= 1024 || n >= 2048);
        if (E <= 8 && four) QSV_ROUTE(4, 8);
        else if (E <= 8) QSV_ROUTE(1, 8);
        else if (four) QSV_ROUTE(4, 16);
        else QSV_ROUTE(1, 16);
#undef QSV_ROUTE
        return qsv_launch_status("qsv_moe_route");
    }
    QSV_DISPATCH(dtype, "qsv_moe_route",
                 hipLaunchKernelGGL(moe_route_kernel<T>, dim3(n), dim3(NT), 0, (hipStream_t)stream, idx, weight, (const T*)h,
                                    (const T*)router, (const T*)bias, renorm, D, E, top_k, G, keep, score_fn, correction,
                                    group_top, scale));
    return qsv_launch_status("qsv_moe_route");
}

extern "C" int qsv_moe_up(void* act, const void* h, const void* up, const int32_t* idx, int n, int top_k, int D, int ff,
                          int activation, float limit, int n_experts, const float* in_weight, int dtype, void* stream) {
    QSV_REQUIRE(act && h && up && idx && n >= 0 && top_k > 0 && D > 0 && ff > 0 && n_experts > 0, "qsv_moe_up: bad arguments");
    QSV_REQUIRE(activation == ACT_RELU_SQ || ((activation == ACT_GLU || activation == QSV_ACT_CLAMPED_GLU) && ff % 2 == 0),
                "qsv_moe_up: activation %d over %d rows", activation, ff);
    QSV_REQUIRE(activation != QSV_ACT_CLAMPED_GLU || limit > 0.f, "qsv_moe_up: clamped units need a positive limit");
    if (activation == QSV_ACT_CLAMPED_GLU) activation = ACT_GLU;
    else limit = 0.f;
    QSV_REQUIRE((size_t)D * 4 <= 64 * 1024, "qsv_moe_up: width %d does not fit the workgroup's LDS", D);
    if (n == 0) return QSV_OK;
#define QSV_UP(KERNEL, ACT)                                                                                                  \
    QSV_DISPATCH(dtype, "qsv_moe_up",                                                                                        \
                 hipLaunchKernelGGL((KERNEL<T, ACT>), dim3(n * top_k), dim3(NT), (size_t)D * 4, (hipStream_t)stream, (T*)act,   \
                                    (const T*)h, (const T*)up, idx, top_k, D, ff, limit, n_experts, in_weight))
    if (D % 8 == 0) {
        if (activation == ACT_GLU) QSV_UP(moe_up_vec_kernel, ACT_GLU);
        else QSV_UP(moe_up_vec_kernel, ACT_RELU_SQ);
    } else {
        if (activation == ACT_GLU) QSV_UP(moe_up_kernel, ACT_GLU);
        else QSV_UP(moe_up_kernel, ACT_RELU_SQ);
    }
#undef QSV_UP
    return qsv_launch_status("qsv_moe_up");
}

extern "C" int qsv_moe_down(void* y, const void* act, const void* down, const int32_t* idx, const float* weight, int n,
                            int top_k, int D, int ff, const void* h, int n_experts, int dtype, void* stream) {
    QSV_REQUIRE(y && act && down && idx && h && n >= 0 && top_k > 0 && D > 0 && ff > 0 && n_experts > 0,
                "qsv_moe_down: bad arguments");
    QSV_REQUIRE((size_t)top_k * ff * 4 <= 64 * 1024, "qsv_moe_down: %d x %d activations do not fit the workgroup's LDS", top_k, ff);
    if (n == 0) return QSV_OK;
    if (ff % 8 == 0)
        QSV_DISPATCH(dtype, "qsv_moe_down",
                     hipLaunchKernelGGL(moe_down_vec_kernel<T>, dim3(n), dim3(NT), (size_t)top_k * ff * 4, (hipStream_t)stream, (T*)y,
                                        (const T*)act, (const T*)down, idx, weight, top_k, D, ff, (const T*)h, n_experts));
    else
        QSV_DISPATCH(dtype, "qsv_moe_down",
                     hipLaunchKernelGGL(moe_down_kernel<T>, dim3(n), dim3(NT), (size_t)top_k * ff * 4, (hipStream_t)stream, (T*)y,
                                        (const T*)act, (const T*)down, idx, weight, top_k, D, ff, (const T*)h, n_experts));
    return qsv_launch_status("qsv_moe_down");
}
