// serve_streams.hip -- one-workgroup-per-token kernels for models that keep several residual streams: the scaled embedding
// into all streams, the read of a sublayer's input (weighted sum of the streams, the statistics-free tanh norm, the token
// shift with its per-sequence state), the rewrite of all streams from a sublayer's output, the final norm over the streams'
// sum; and two small row kernels of the same models (RMS-normed mean of two branches, gated-unit activation).
// Streams, sums and norms are float; only what leaves for a matrix product is in the storage type.
#include "serve_common.h"
#include "serve_route.h"

#include <type_traits>

namespace {
constexpr int NT = 256;
constexpr int MAX_STREAMS = 16;

template <typename T>
__global__ __launch_bounds__(NT) void embed_streams_kernel(float* __restrict__ x, const T* __restrict__ table,
                                                           const int32_t* __restrict__ tokens, float scale, int S, int D) {
    const size_t t = blockIdx.x;
    const T* row = table + (size_t)tokens[t] * D;
    for (int i = threadIdx.x; i < D; i += NT) {
        const float v = ld(row, i) * scale;
        for (int s = 0; s < S; ++s) x[(t * S + s) * D + i] = v;
    }
}

// The same, four columns per thread, `chunks` workgroups per token.
template <typename T>
__global__ __launch_bounds__(NT) void embed_streams_vec_kernel(float* __restrict__ x, const T* __restrict__ table, const int32_t* __restrict__ tokens, float scale, int S,
                                                               int D, int chunks) {
    const size_t t = token_of(blockIdx.x, chunks);
    const int i = ((blockIdx.x - (unsigned)t * chunks) * NT + threadIdx.x) * 4;
    if (i >= D) return;
    float v[4];
    ld4t(table, (size_t)tokens[t] * D + i, v);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] *= scale;
    for (int s = 0; s < S; ++s) st4t(x, (t * S + s) * D + i, v);
}

__device__ __forceinline__ float stream_sum(const float* __restrict__ x, const float* __restrict__ w_in, size_t t, int S, int D,
                                            int i) {
    float u = 0.f;
    for (int s = 0; s < S; ++s) u += w_in[s] * x[(t * S + s) * D + i];
    return u;
}

// h[t] = n + (before - n) * shift,  n = tanh(alpha * sum_s w_in[s] x[t, s]) * w + b, `before` = the same n of the previous
// token of the sequence: recomputed from the previous row of the batch inside a run, read from the sequence's state at a run's
// start (zeros when the run starts the sequence).  The last token of a run leaves its n in the state's other copy.
template <typename T>
__global__ __launch_bounds__(NT) void hc_read_kernel(T* __restrict__ h, const float* __restrict__ x, const float* __restrict__ w_in,
                                                     const T* __restrict__ nw, const T* __restrict__ nb, float alpha,
                                                     const T* __restrict__ shift, float* __restrict__ prev,
                                                     const int32_t* __restrict__ run_off, const int32_t* __restrict__ state_rd,
                                                     const int32_t* __restrict__ state_wr, int S, int D) {
    const size_t t = blockIdx.x;
    const bool shifted = shift != nullptr;
    const int off = shifted ? run_off[t] : 0, rd = shifted ? state_rd[t] : -1, wr = shifted ? state_wr[t] : -1;
    for (int i = threadIdx.x; i < D; i += NT) {
        const float w = ld(nw, i), b = ld(nb, i);
        float n = tanhf(alpha * stream_sum(x, w_in, t, S, D, i)) * w + b;
        if (shifted) {
            float before = 0.f;
            if (off > 0) before = tanhf(alpha * stream_sum(x, w_in, t - 1, S, D, i)) * w + b;
            else if (rd >= 0) before = prev[(size_t)rd * D + i];
            if (wr >= 0) prev[(size_t)wr * D + i] = n;
            n += (before - n) * ld(shift, i);
        }
        st(h, t * D + i, n);
    }
}

// x[t, r] <- sum_s mix[s, r] x[t, s] + out[r] * y[t], all streams from the old ones; and, if asked for, the next sublayer's
// input from the new streams in the same pass (no token shift there: that needs the previous token's NEW streams)
template <typename T>
__global__ __launch_bounds__(NT) void hc_write_kernel(float* __restrict__ x, const T* __restrict__ y, const float* __restrict__ mix,
                                                      const float* __restrict__ w_out, int S, int D, T* __restrict__ h_next,
                                                      const float* __restrict__ w_in_next, const T* __restrict__ nw,
                                                      const T* __restrict__ nb, float alpha) {
    const size_t t = blockIdx.x;
    for (int i = threadIdx.x; i < D; i += NT) {
        float old[MAX_STREAMS];
#pragma unroll
        for (int s = 0; s < MAX_STREAMS; ++s) old[s] = s < S ? x[(t * S + s) * D + i] : 0.f;
        const float yv = ld(y, t * D + i);
        float u = 0.f;
        for (int r = 0; r < S; ++r) {
            float a = w_out[r] * yv;
#pragma unroll
            for (int s = 0; s < MAX_STREAMS; ++s)
                if (s < S) a += mix[s * S + r] * old[s];
            x[(t * S + r) * D + i] = a;
            if (h_next) u += w_in_next[r] * a;
        }
        if (h_next) st(h_next, t * D + i, tanhf(alpha * u) * ld(nw, i) + ld(nb, i));
    }
}

// ---- the same two kernels for widths that are multiples of four: 16-byte stream accesses, four elements per thread and pass, `chunks` workgroups
// per token ----
// A step's few tokens are spread over as many workgroups as their width fills: one pass each (read / written, 16 tokens of 2 x 2048: 3.2 -> 2.5 /
// 5.4 -> 3.4 us, 64 of 2 x 4096: 4.6 -> 2.6 / 9.1 -> 3.6).  Enough tokens to fill the chip keep one, with fewer workgroups to start: from 1024 for the
// reading kernel (8192 of 2 x 2048, shifted: 47 us against 51; 1023 of 4 x 2048 spread: 6.9 against 7.9), above 512 for the writing one, which keeps more
// in registers (1023 of 2 x 4096: 17.6 us against 19.4).
inline int stream_chunks(int n, int most, int D) { return n > most ? 1 : (int)(((int64_t)D + 4 * NT - 1) / (4 * NT)); }
template <int MS, class More>
__device__ __forceinline__ void stream_sum4(const float* __restrict__ x, const float* __restrict__ w_in, size_t t, int S, int D, int i,
                                            float (&u)[4], More more) {
    u[0] = u[1] = u[2] = u[3] = 0.f;
    if constexpr (MS <= 4) {                                               // all at once (a stream that there is not repeats the last)
        raw4f r[MS];
        float w[MS];
#pragma unroll
        for (int s = 0; s < MS; ++s) {
            r[s] = raw4(x, (t * S + min(s, S - 1)) * D + i);
            w[s] = w_in[min(s, S - 1)];
        }
        more();
        requested();
#pragma unroll
        for (int s = 0; s < MS; ++s)
            if (s < S) {
                float v[4];
                widen4(r[s], v);
#pragma unroll
                for (int j = 0; j < 4; ++j) u[j] += w[s] * v[j];
            }
        return;
    }
    more();
    for (int s = 0; s < S; ++s) {
        float v[4];
        ld4t(x, (t * S + s) * D + i, v);
        const float w = w_in[s];
#pragma unroll
        for (int j = 0; j < 4; ++j) u[j] += w * v[j];
    }
}

template <typename T, int MS = MAX_STREAMS>
__global__ __launch_bounds__(NT) void hc_read_vec_kernel(T* __restrict__ h, const float* __restrict__ x, const float* __restrict__ w_in,
                                                         const T* __restrict__ nw, const T* __restrict__ nb, float alpha,
                                                         const T* __restrict__ shift, float* __restrict__ prev,
                                                         const int32_t* __restrict__ run_off, const int32_t* __restrict__ state_rd,
                                                         const int32_t* __restrict__ state_wr, int S, int D, int chunks) {
    const size_t t = token_of(blockIdx.x, chunks);
    const bool shifted = shift != nullptr;
    const int off = shifted ? run_off[t] : 0, rd = shifted ? state_rd[t] : -1, wr = shifted ? state_wr[t] : -1;
    const T* mus = shifted ? shift : nw;
    for (int i = ((blockIdx.x - (unsigned)t * chunks) * NT + threadIdx.x) * 4; i < D; i += chunks * NT * 4) {
        float w[4], b[4], u[4], n[4];
        raw4f rp;
        const auto rw = raw4(nw, i), rb = raw4(nb, i), rm = raw4(mus, i);
        stream_sum4<MS>(x, w_in, t, S, D, i, u, [&] {                       // (behind the streams' requests)
            if (off == 0 && rd >= 0) rp = raw4(prev, (size_t)rd * D + i);
        });
        widen4(rw, w);
        widen4(rb, b);
#pragma unroll
        for (int j = 0; j < 4; ++j) n[j] = tanhf(alpha * u[j]) * w[j] + b[j];
        if (shifted) {
            float before[4] = {0.f, 0.f, 0.f, 0.f}, mu[4];
            if (off > 0) {
                stream_sum4<MS>(x, w_in, t - 1, S, D, i, u, [] {});
#pragma unroll
                for (int j = 0; j < 4; ++j) before[j] = tanhf(alpha * u[j]) * w[j] + b[j];
            } else if (rd >= 0) {
                widen4(rp, before);
            }
            if (wr >= 0) st4t(prev, (size_t)wr * D + i, n);
            widen4(rm, mu);
#pragma unroll
            for (int j = 0; j < 4; ++j) n[j] += (before[j] - n[j]) * mu[j];
        }
        st4t(h, t * D + i, n);
    }
}

// The next sublayer's input where that reads with a token shift and every run is one token: what hc_read_vec_kernel makes of the streams just written.
template <typename T>
struct ShiftedRead {
    T* h;
    const float* w_in;
    const T *nw, *nb, *shift;
    float* prev;
    const int32_t *rd, *wr;
    float alpha;
};

// (Y other than void: y is what a mixture of experts left per slot, float or the storage type; it is summed here, and rounded as a tensor would hold it)
// MS: streams at most; up to four of them are requested at once, with the mix beside them (a stream that there is not repeats the last).
// STEP (up to four streams, rows of experts): with the next sublayer's shifted input, a launch less between two layers of a step.
template <typename T, typename Y = void, int MS = MAX_STREAMS, bool STEP = false>
__global__ __launch_bounds__(NT) void hc_write_vec_kernel(float* __restrict__ x, const T* __restrict__ y, const float* __restrict__ mix,
                                                          const float* __restrict__ w_out, int S, int D, T* __restrict__ h_next,
                                                          const float* __restrict__ w_in_next, const T* __restrict__ nw,
                                                          const T* __restrict__ nb, float alpha, int chunks, SlotRows slots, ShiftedRead<T> next) {
    const size_t t = token_of(blockIdx.x, chunks);
    const int rd = STEP ? next.rd[t] : -1, wr = STEP ? next.wr[t] : -1;
    const float* w_in = STEP ? next.w_in : h_next ? w_in_next : w_out;
    const T *pw = h_next ? nw : y, *pb = h_next ? nb : y;              // (no next input: nothing of these is used)
    float m[MS <= 4 ? MS : 1][MS <= 4 ? MS : 1], wo[MS <= 4 ? MS : 1], wi[MS <= 4 ? MS : 1];
    if constexpr (MS <= 4) {
#pragma unroll
        for (int r = 0; r < MS; ++r) {
            wo[r] = w_out[min(r, S - 1)];
            wi[r] = w_in[min(r, S - 1)];
#pragma unroll
            for (int a = 0; a < MS; ++a) m[a][r] = mix[min(a, S - 1) * S + min(r, S - 1)];
        }
    }
    for (int i = ((blockIdx.x - (unsigned)t * chunks) * NT + threadIdx.x) * 4; i < D; i += chunks * NT * 4) {
        raw4f rx[MS], rp;
        typename Raw4<T>::type ry, rw, rb, rm;
        float old[MS][4], yv[1][4], u[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < MS; ++q)
            if (MS <= 4 || q < S) rx[q] = raw4(x, (t * S + min(q, S - 1)) * D + i);
        if constexpr (std::is_void<Y>::value) {
            ry = raw4(y, t * D + i);
            rw = raw4(pw, i);
            rb = raw4(pb, i);
        } else {
            if constexpr (STEP) {
                rw = raw4(next.nw, i);
                rb = raw4(next.nb, i);
                rm = raw4(next.shift, i);
                rp = raw4(next.prev, (size_t)max(rd, 0) * D + i);
            }
            slot_sum4<Y>(slots, t, D, i, 0, yv);
            round_stored<T>(yv);
        }
        requested();
        if constexpr (std::is_void<Y>::value) widen4(ry, yv[0]);
#pragma unroll
        for (int q = 0; q < MS; ++q) widen4(rx[q], old[q]);
        auto stream = [&](int r, auto mix_of, float wor, float wir) __attribute__((always_inline)) {
            float a[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = wor * yv[0][j];
#pragma unroll
            for (int q = 0; q < MS; ++q)
                if (q < S) {
                    const float mq = mix_of(q);
#pragma unroll
                    for (int j = 0; j < 4; ++j) a[j] += mq * old[q][j];
                }
            st4t(x, (t * S + r) * D + i, a);
            if (STEP || h_next) {
#pragma unroll
                for (int j = 0; j < 4; ++j) u[j] += wir * a[j];
            }
        };
        if constexpr (MS <= 4) {
#pragma unroll
            for (int r = 0; r < MS; ++r)
                if (r < S) stream(r, [&](int q) { return m[q][r]; }, wo[r], wi[r]);
        } else {
            for (int r = 0; r < S; ++r) stream(r, [&](int q) { return mix[q * S + r]; }, w_out[r], h_next ? w_in_next[r] : 0.f);
        }
        if constexpr (std::is_void<Y>::value)
            if (h_next) {
                float w[4], b[4], n[4];
                widen4(rw, w);
                widen4(rb, b);
#pragma unroll
                for (int j = 0; j < 4; ++j) n[j] = tanhf(alpha * u[j]) * w[j] + b[j];
                st4t(h_next, t * D + i, n);
            }
        if constexpr (STEP) {
            float w[4], b[4], n[4], mu[4], before[4];
            widen4(rw, w);
            widen4(rb, b);
            widen4(rm, mu);
            widen4(rp, before);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                n[j] = tanhf(next.alpha * u[j]) * w[j] + b[j];
                if (rd < 0) before[j] = 0.f;
            }
            if (wr >= 0) st4t(next.prev, (size_t)wr * D + i, n);
#pragma unroll
            for (int j = 0; j < 4; ++j) n[j] += (before[j] - n[j]) * mu[j];
            st4t(next.h, t * D + i, n);
        }
    }
}

// The same for a step (bfloat16, up to four streams, a workgroup per token), the next sublayer's input routed on its way out (serve_route.h).  P: groups of four
// columns a thread holds, all requested before the first is used.
// PAIR: y is half the sum of two normed rows, made here (rms_pair_mean_kernel's bits, a launch less).
struct NormedPair {
    const bf16_t *b, *wa, *wb;
    float eps;
};
template <int P, int MS, int EC, bool PAIR>
__global__ __launch_bounds__(NT) void hc_write_route_kernel(float* __restrict__ x, const bf16_t* __restrict__ y, const float* __restrict__ mix,
                                                            const float* __restrict__ w_out, int S, int D, bf16_t* __restrict__ h_next,
                                                            const float* __restrict__ w_in_next, const bf16_t* __restrict__ nw,
                                                            const bf16_t* __restrict__ nb, float alpha, RouteArgs route, NormedPair pair) {
    __shared__ __attribute__((aligned(16))) RouteRoom<bf16_t, P, EC> room;
    __shared__ float red[NT / 64 + 1];
    RouteHead<bf16_t, EC> head;
    const size_t t = blockIdx.x;
    raw4f rx[P][MS];
    raw2u ry[P], rw[P], rb[P], ry2[P], rwa[P], rwb[P];
    float m[MS][MS], wo[MS], wi[MS];
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int at = min((k * NT + (int)threadIdx.x) * 4, D - 4);
        if constexpr (PAIR) {
            ry2[k] = raw4(pair.b, t * D + at);
            rwa[k] = raw4(pair.wa, at);
            rwb[k] = raw4(pair.wb, at);
        }
#pragma unroll
        for (int q = 0; q < MS; ++q) rx[k][q] = raw4(x, (t * S + min(q, S - 1)) * D + at);
        ry[k] = raw4(y, t * D + at);
        rw[k] = raw4(nw, at);
        rb[k] = raw4(nb, at);
    }
#pragma unroll
    for (int r = 0; r < MS; ++r) {
        wo[r] = w_out[min(r, S - 1)];
        wi[r] = w_in_next[min(r, S - 1)];
#pragma unroll
        for (int q = 0; q < MS; ++q) m[q][r] = mix[min(q, S - 1) * S + min(r, S - 1)];
    }
    head.request(route, D);
    requested();
    float ia = 0.f, ib = 0.f;
    if constexpr (PAIR) {
        float sa = 0.f, sb = 0.f;
#pragma unroll
        for (int k = 0; k < P; ++k) {
            float u[4], v[4];
            widen4(ry[k], u);
            widen4(ry2[k], v);
            if ((k * NT + (int)threadIdx.x) * 4 >= D) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sa += u[j] * u[j];
                sb += v[j] * v[j];
            }
        }
        ia = 1.0f / sqrtf(block_sum<NT>(sa, red) / (float)D + pair.eps);
        ib = 1.0f / sqrtf(block_sum<NT>(sb, red) / (float)D + pair.eps);
    }
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int i = (k * NT + threadIdx.x) * 4;
        if (i >= D) continue;
        float old[MS][4], yv[4], w[4], b[4], u[4] = {0.f, 0.f, 0.f, 0.f}, n[4];
#pragma unroll
        for (int q = 0; q < MS; ++q) widen4(rx[k][q], old[q]);
        widen4(ry[k], yv);
        if constexpr (PAIR) {
            float v[4], wu[4], wv[4];
            widen4(ry2[k], v);
            widen4(rwa[k], wu);
            widen4(rwb[k], wv);
#pragma unroll
            for (int j = 0; j < 4; ++j) yv[j] = bf2f(f2bf(0.5f * (yv[j] * ia * wu[j] + v[j] * ib * wv[j])));
        }
        widen4(rw[k], w);
        widen4(rb[k], b);
#pragma unroll
        for (int r = 0; r < MS; ++r) {
            if (r >= S) continue;
            float a[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = wo[r] * yv[j];
#pragma unroll
            for (int q = 0; q < MS; ++q)
                if (q < S) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) a[j] += m[q][r] * old[q][j];
                }
            st4t(x, (t * S + r) * D + i, a);
#pragma unroll
            for (int j = 0; j < 4; ++j) u[j] += wi[r] * a[j];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) n[j] = tanhf(alpha * u[j]) * w[j] + b[j];
        st4t(h_next, t * D + i, n);
        st4t(room.row, i, n);
    }
    __syncthreads();
    route_row<bf16_t, EC>(route, head, t, room.row, D, room.part, room.cs);
}
template <typename T>
__global__ __launch_bounds__(NT) void dyt_sum_rows_kernel(T* __restrict__ out, const float* __restrict__ x,
                                                          const int32_t* __restrict__ rows, const T* __restrict__ nw,
                                                          const T* __restrict__ nb, float alpha, int S, int D) {
    const size_t r = blockIdx.x;
    const size_t t = rows ? (size_t)rows[r] : r;
    for (int i = threadIdx.x; i < D; i += NT) {
        float u = 0.f;
        for (int s = 0; s < S; ++s) u += x[(t * S + s) * D + i];
        st(out, r * D + i, tanhf(alpha * u) * ld(nw, i) + ld(nb, i));
    }
}
// The same for widths that are multiples of four and up to four streams: a thread's four columns in one trip to memory, `chunks` workgroups per row.
template <typename T, int MS>
__global__ __launch_bounds__(NT) void dyt_sum_rows_vec_kernel(T* __restrict__ out, const float* __restrict__ x, const int32_t* __restrict__ rows,
                                                              const T* __restrict__ nw, const T* __restrict__ nb, float alpha, int S, int D, int chunks) {
    const size_t r = token_of(blockIdx.x, chunks);
    const int i = ((blockIdx.x - (unsigned)r * chunks) * NT + threadIdx.x) * 4;
    if (i >= D) return;
    const auto rw = raw4(nw, i), rb = raw4(nb, i);
    const size_t t = rows ? (size_t)rows[r] : r;
    raw4f rx[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) rx[s] = raw4(x, (t * S + min(s, S - 1)) * D + i);
    requested();
    float u[4] = {0.f, 0.f, 0.f, 0.f}, w[4], b[4], n[4];
#pragma unroll
    for (int s = 0; s < MS; ++s)
        if (s < S) {
#pragma unroll
            for (int j = 0; j < 4; ++j) u[j] += rx[s][j];
        }
    widen4(rw, w);
    widen4(rb, b);
#pragma unroll
    for (int j = 0; j < 4; ++j) n[j] = tanhf(alpha * u[j]) * w[j] + b[j];
    st4t(out, r * D + i, n);
}

// out[t] = (a[t] / rms(a[t]) * wa + b[t] / rms(b[t]) * wb) / 2
// P other than 0: rows of up to 1024 P elements, a multiple of four, read once.
template <typename T, bool VEC, int P>
__global__ __launch_bounds__(NT) void rms_pair_mean_kernel(T* __restrict__ out, const T* __restrict__ a, const T* __restrict__ wa,
                                                           const T* __restrict__ b, const T* __restrict__ wb, float eps, int D) {
    __shared__ float red[NT / 64 + 1];
    const size_t t = blockIdx.x;
    float sa = 0.f, sb = 0.f;
    if constexpr (P > 0) {
        typename Raw4<T>::type ra[P], rb[P], rwa[P], rwb[P];
#pragma unroll
        for (int k = 0; k < P; ++k) {
            const int at = min((k * NT + (int)threadIdx.x) * 4, D - 4);
            ra[k] = raw4(a, t * D + at);
            rb[k] = raw4(b, t * D + at);
            rwa[k] = raw4(wa, at);
            rwb[k] = raw4(wb, at);
        }
        requested();
        float u[P][4], v[P][4], wu[4], wv[4], y[4];
#pragma unroll
        for (int k = 0; k < P; ++k) {
            widen4(ra[k], u[k]);
            widen4(rb[k], v[k]);
            if ((k * NT + (int)threadIdx.x) * 4 >= D) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sa += u[k][j] * u[k][j];
                sb += v[k][j] * v[k][j];
            }
        }
        const float ia = 1.0f / sqrtf(block_sum<NT>(sa, red) / (float)D + eps);
        const float ib = 1.0f / sqrtf(block_sum<NT>(sb, red) / (float)D + eps);
#pragma unroll
        for (int k = 0; k < P; ++k) {
            const int i = (k * NT + (int)threadIdx.x) * 4;
            if (i >= D) continue;
            widen4(rwa[k], wu);
            widen4(rwb[k], wv);
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = 0.5f * (u[k][j] * ia * wu[j] + v[k][j] * ib * wv[j]);
            st4t(out, t * D + i, y);
        }
        return;
    }
    if (VEC) {                                                           // D % 4 == 0
        for (int i = threadIdx.x * 4; i < D; i += NT * 4) {
            float u[4], v[4];
            ld4t(a, t * D + i, u);
            ld4t(b, t * D + i, v);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sa += u[j] * u[j];
                sb += v[j] * v[j];
            }
        }
    } else {
        for (int i = threadIdx.x; i < D; i += NT) {
            const float u = ld(a, t * D + i), v = ld(b, t * D + i);
            sa += u * u;
            sb += v * v;
        }
    }
    const float ia = 1.0f / sqrtf(block_sum<NT>(sa, red) / (float)D + eps);
    const float ib = 1.0f / sqrtf(block_sum<NT>(sb, red) / (float)D + eps);
    if (VEC) {
        for (int i = threadIdx.x * 4; i < D; i += NT * 4) {
            float u[4], v[4], wu[4], wv[4], y[4];
            ld4t(a, t * D + i, u);
            ld4t(b, t * D + i, v);
            ld4t(wa, i, wu);
            ld4t(wb, i, wv);
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = 0.5f * (u[j] * ia * wu[j] + v[j] * ib * wv[j]);
            st4t(out, t * D + i, y);
        }
        return;
    }
    for (int i = threadIdx.x; i < D; i += NT)
        st(out, t * D + i, 0.5f * (ld(a, t * D + i) * ia * ld(wa, i) + ld(b, t * D + i) * ib * ld(wb, i)));
}

// out[r, f] = act(s a[r, 2f]) * s a[r, 2f + 1] with s = row_scale[scale_index ? scale_index[r] : r] (row_scale NULL: 1);  act 0: silu, 1: gelu in its tanh form, 0.5 z (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3)));
// act 2: g = min(gate, limit), u = clamp(up, -limit, limit) -> g sigmoid(1.702 g) (u + 1)
__device__ __forceinline__ float glu_unit(float g, float u, int act, float limit) {
    if (act == 2) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
    }
    const float ag = act == 0 ? g / (1.0f + expf(-g)) : 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
    return ag * u;
}
template <typename T, bool VEC>
__global__ __launch_bounds__(NT) void glu_kernel(T* __restrict__ out, const T* __restrict__ a, int ff, int act, float limit,
                                                 const float* __restrict__ row_scale, const int64_t* __restrict__ scale_index) {
    const size_t r = blockIdx.x;
    const float rs = row_scale ? row_scale[scale_index ? (size_t)scale_index[r] : r] : 1.0f;
    if (VEC) {                                                           // ff % 4 == 0: four units per thread and pass
        for (int f = threadIdx.x * 4; f < ff; f += NT * 4) {
            float p[4], q[4];
            ld4t(a, (r * ff + f) * 2, p);
            ld4t(a, (r * ff + f) * 2 + 4, q);
            const float y[4] = {glu_unit(rs * p[0], rs * p[1], act, limit), glu_unit(rs * p[2], rs * p[3], act, limit),
                                glu_unit(rs * q[0], rs * q[1], act, limit), glu_unit(rs * q[2], rs * q[3], act, limit)};
            st4t(out, r * ff + f, y);
        }
        return;
    }
    for (int f = threadIdx.x; f < ff; f += NT)
        st(out, r * ff + f, glu_unit(rs * ld(a, (r * ff + f) * 2), rs * ld(a, (r * ff + f) * 2 + 1), act, limit));
}
}  // namespace

extern "C" int qsv_embed_streams(float* x, const void* table, const int32_t* tokens, float scale, int n, int streams, int D,
                                 int dtype, void* stream) {
    QSV_REQUIRE(x && table && tokens && n >= 0 && D > 0 && streams > 0, "qsv_embed_streams: bad arguments");
    if (n == 0) return QSV_OK;
    const int64_t chunks = ((int64_t)D / 4 + NT - 1) / NT;
    if (D % 4 == 0 && fits4(x, QSV_F32) && fits4(table, dtype) && chunks * n < (1ll << 31)) {
        QSV_DISPATCH(dtype, "qsv_embed_streams",
                     hipLaunchKernelGGL(embed_streams_vec_kernel<T>, dim3((unsigned)(chunks * n)), dim3(NT), 0, (hipStream_t)stream, x, (const T*)table, tokens, scale,
                                        streams, D, (int)chunks));
        return qsv_launch_status("qsv_embed_streams");
    }
    QSV_DISPATCH(dtype, "qsv_embed_streams",
                 hipLaunchKernelGGL(embed_streams_kernel<T>, dim3(n), dim3(NT), 0, (hipStream_t)stream, x, (const T*)table, tokens,
                                    scale, streams, D));
    return qsv_launch_status("qsv_embed_streams");
}

extern "C" int qsv_hc_read(void* h, const float* x, const float* w_in, const void* norm_w, const void* norm_b, float alpha,
                           const void* shift, float* prev, const int32_t* run_off, const int32_t* state_rd,
                           const int32_t* state_wr, int n, int streams, int D, int dtype, void* stream) {
    QSV_REQUIRE(h && x && w_in && norm_w && norm_b && n >= 0 && D > 0 && streams > 0, "qsv_hc_read: bad arguments");
    QSV_REQUIRE(!shift || (prev && run_off && state_rd && state_wr), "qsv_hc_read: token shift without its state");
    if (n == 0) return QSV_OK;
    const int chunks = stream_chunks(n, 1023, D);
    if (D % 4 == 0) {
#define QSV_HCRD(MS)                                                                                                                           \
    QSV_DISPATCH(dtype, "qsv_hc_read",                                                                                                        \
                 hipLaunchKernelGGL((hc_read_vec_kernel<T, MS>), dim3((unsigned)(chunks * n)), dim3(NT), 0, (hipStream_t)stream, (T*)h, x, w_in,       \
                                    (const T*)norm_w, (const T*)norm_b, alpha, (const T*)shift, prev, run_off, state_rd, state_wr, streams, D, chunks))
        // (without a shift, streams one after another are the faster ones between the steps, where latency counts, and the prompts, where memory does: 512 rows of
        // 4 x 4096 / 2 x 4096 7.7 / 6.3 us at once, 7.0 / 5.9 so)
        if (!shift && n > 128 && n <= 1023) QSV_HCRD(MAX_STREAMS);
        else if (streams <= 2) QSV_HCRD(2);
        else if (streams <= 4) QSV_HCRD(4);
        else QSV_HCRD(MAX_STREAMS);
#undef QSV_HCRD
    } else {
        QSV_DISPATCH(dtype, "qsv_hc_read",
                     hipLaunchKernelGGL(hc_read_kernel<T>, dim3(n), dim3(NT), 0, (hipStream_t)stream, (T*)h, x, w_in, (const T*)norm_w,
                                        (const T*)norm_b, alpha, (const T*)shift, prev, run_off, state_rd, state_wr, streams, D));
    }
    return qsv_launch_status("qsv_hc_read");
}

extern "C" int qsv_hc_write(float* x, const void* y, const float* mix, const float* w_out, int n, int streams, int D, void* h_next,
                            const float* w_in_next, const void* norm_w, const void* norm_b, float alpha, int dtype, void* stream) {
    QSV_REQUIRE(x && y && mix && w_out && n >= 0 && D > 0, "qsv_hc_write: bad arguments");
    QSV_REQUIRE(!h_next || (w_in_next && norm_w && norm_b), "qsv_hc_write: the next sublayer's input without its weights");
    QSV_REQUIRE(streams > 0 && streams <= MAX_STREAMS, "qsv_hc_write: %d streams (at most %d)", streams, MAX_STREAMS);
    if (n == 0) return QSV_OK;
    const int chunks = stream_chunks(n, 512, D);
    if (D % 4 == 0) {
#define QSV_HCV(MS)                                                                                                                            \
    QSV_DISPATCH(dtype, "qsv_hc_write",                                                                                                       \
                 hipLaunchKernelGGL((hc_write_vec_kernel<T, void, MS>), dim3((unsigned)(chunks * n)), dim3(NT), 0, (hipStream_t)stream, x, (const T*)y, mix, w_out, \
                                    streams, D, (T*)h_next, w_in_next, (const T*)norm_w, (const T*)norm_b, alpha, chunks, SlotRows{}, ShiftedRead<T>{}))
        if (streams <= 2) QSV_HCV(2);
        else if (streams <= 4) QSV_HCV(4);
        else QSV_HCV(MAX_STREAMS);
#undef QSV_HCV
    } else {
        QSV_DISPATCH(dtype, "qsv_hc_write",
                     hipLaunchKernelGGL(hc_write_kernel<T>, dim3(n), dim3(NT), 0, (hipStream_t)stream, x, (const T*)y, mix, w_out,
                                        streams, D, (T*)h_next, w_in_next, (const T*)norm_w, (const T*)norm_b, alpha));
    }
    return qsv_launch_status("qsv_hc_write");
}

// the same for a step, h_next's rows routed in the same launch (bfloat16, up to four streams)
static int hc_write_route(const char* what, float* x, const void* y, const float* mix, const float* w_out, int n, int streams, int D, void* h_next, const float* w_in_next,
                                  const void* norm_w, const void* norm_b, float alpha, int32_t* idx, float* weight, const void* router, const void* bias, int renorm, int E,
                                  int top_k, int G, int keep, int score_fn, const float* correction, int group_top, float scale, void* stream, const NormedPair* pair) {
    QSV_REQUIRE(x && y && mix && w_out && h_next && w_in_next && norm_w && norm_b && n >= 0 && D > 0 && D % 8 == 0 && D <= NT * 16 && streams > 0 && streams <= 4,
                "%s: bad arguments", what);
    QSV_REQUIRE(fits4(x, QSV_F32) && fits4(y, QSV_BF16) && fits4(h_next, QSV_BF16) && fits4(norm_w, QSV_BF16) && fits4(norm_b, QSV_BF16), "%s: rows on four elements", what);
    const RouteArgs r = {idx, weight, router, bias, correction, renorm, E, top_k, G, keep, score_fn, group_top, scale};
    QSV_REQUIRE(route_ok(r), "%s: %d experts in %d groups, %d groups kept, top %d", what, E, G, keep, top_k);
    if (n == 0) return QSV_OK;
#define QSV_HCR(P, MS, EC)                                                                                                                     \
    hipLaunchKernelGGL((pair ? hc_write_route_kernel<P, MS, EC, true> : hc_write_route_kernel<P, MS, EC, false>), dim3(n), dim3(NT), 0, (hipStream_t)stream, x, (const bf16_t*)y, mix, w_out, streams, D, (bf16_t*)h_next, \
                       w_in_next, (const bf16_t*)norm_w, (const bf16_t*)norm_b, alpha, r, pair ? *pair : NormedPair{})
#define QSV_HCR_P(MS, EC)                         \
    do {                                          \
        if (D <= NT * 4) QSV_HCR(1, MS, EC);      \
        else if (D <= NT * 8) QSV_HCR(2, MS, EC); \
        else QSV_HCR(4, MS, EC);                  \
    } while (0)
    if (streams <= 2 && E <= 8) QSV_HCR_P(2, 8);
    else if (streams <= 2) QSV_HCR_P(2, 16);
    else if (E <= 8) QSV_HCR_P(4, 8);
    else QSV_HCR_P(4, 16);
#undef QSV_HCR
#undef QSV_HCR_P
    return qsv_launch_status(what);
}

extern "C" int qsv_hc_write_route(float* x, const void* y, const float* mix, const float* w_out, int n, int streams, int D, void* h_next, const float* w_in_next,
                                  const void* norm_w, const void* norm_b, float alpha, int32_t* idx, float* weight, const void* router, const void* bias, int renorm, int E,
                                  int top_k, int G, int keep, int score_fn, const float* correction, int group_top, float scale, void* stream) {
    return hc_write_route("qsv_hc_write_route", x, y, mix, w_out, n, streams, D, h_next, w_in_next, norm_w, norm_b, alpha, idx, weight, router, bias, renorm, E, top_k, G,
                          keep, score_fn, correction, group_top, scale, stream, nullptr);
}
// ... with y the mean of two normed rows (qsv_rms_pair_mean's)
extern "C" int qsv_hc_write_pair_route(float* x, const void* a, const void* wa, const void* b, const void* wb, float eps, const float* mix, const float* w_out, int n,
                                       int streams, int D, void* h_next, const float* w_in_next, const void* norm_w, const void* norm_b, float alpha, int32_t* idx,
                                       float* weight, const void* router, const void* bias, int renorm, int E, int top_k, int G, int keep, int score_fn,
                                       const float* correction, int group_top, float scale, void* stream) {
    QSV_REQUIRE(b && wa && wb && fits4(b, QSV_BF16) && fits4(wa, QSV_BF16) && fits4(wb, QSV_BF16), "qsv_hc_write_pair_route: bad arguments");
    const NormedPair pair = {(const bf16_t*)b, (const bf16_t*)wa, (const bf16_t*)wb, eps};
    return hc_write_route("qsv_hc_write_pair_route", x, a, mix, w_out, n, streams, D, h_next, w_in_next, norm_w, norm_b, alpha, idx, weight, router, bias, renorm, E, top_k,
                          G, keep, score_fn, correction, group_top, scale, stream, &pair);
}

extern "C" int qsv_hc_write_slots(float* x, const void* ys, int float_rows, const int32_t* place, const float* weight, const int32_t* idx, int top_k, int n_experts,
                                  const float* mix, const float* w_out, int n, int streams, int D, int dtype, void* stream) {
    QSV_REQUIRE(x && ys && idx && mix && w_out && n >= 0 && D > 0 && top_k > 0 && n_experts > 0, "qsv_hc_write_slots: bad arguments");
    QSV_REQUIRE(streams > 0 && streams <= MAX_STREAMS, "qsv_hc_write_slots: %d streams (at most %d)", streams, MAX_STREAMS);
    QSV_REQUIRE(D % 4 == 0 && fits4(ys, float_rows ? QSV_F32 : dtype), "qsv_hc_write_slots: width %d (a multiple of 4), rows on four elements", D);
    if (n == 0) return QSV_OK;
    const int chunks = stream_chunks(n, 512, D);
    const SlotRows slots = {ys, place, weight, idx, top_k, n_experts};
#define QSV_HCW(Y, MS)                                                                                                                          \
    QSV_DISPATCH(dtype, "qsv_hc_write_slots",                                                                                                   \
                 hipLaunchKernelGGL((hc_write_vec_kernel<T, Y, MS>), dim3((unsigned)(chunks * n)), dim3(NT), 0, (hipStream_t)stream, x, (const T*)nullptr, mix, w_out, \
                                    streams, D, (T*)nullptr, (const float*)nullptr, (const T*)nullptr, (const T*)nullptr, 0.f, chunks, slots, ShiftedRead<T>{}))
#define QSV_HCW_S(Y)                          \
    do {                                      \
        if (streams <= 2) QSV_HCW(Y, 2);      \
        else if (streams <= 4) QSV_HCW(Y, 4); \
        else QSV_HCW(Y, MAX_STREAMS);         \
    } while (0)
    if (float_rows) QSV_HCW_S(float);
    else QSV_HCW_S(T);
#undef QSV_HCW
#undef QSV_HCW_S
    return qsv_launch_status("qsv_hc_write_slots");
}

// ... of a step, with the next sublayer's shifted input (one token a run, up to four streams)
extern "C" int qsv_hc_write_slots_read(float* x, const float* ys, const float* weight, const int32_t* idx, int top_k, int n_experts, const float* mix, const float* w_out,
                                       int n, int streams, int D, void* h_next, const float* w_in, const void* norm_w, const void* norm_b, float alpha, const void* shift,
                                       float* prev, const int32_t* state_rd, const int32_t* state_wr, int dtype, void* stream) {
    QSV_REQUIRE(x && ys && idx && mix && w_out && h_next && w_in && norm_w && norm_b && shift && prev && state_rd && state_wr && n >= 0 && D > 0 && top_k > 0 &&
                    n_experts > 0 && streams > 0 && streams <= 4, "qsv_hc_write_slots_read: bad arguments");
    QSV_REQUIRE(D % 4 == 0 && fits4(ys, QSV_F32) && fits4(x, QSV_F32) && fits4(prev, QSV_F32) && fits4(h_next, dtype) && fits4(norm_w, dtype) && fits4(norm_b, dtype) &&
                    fits4(shift, dtype), "qsv_hc_write_slots_read: width %d (a multiple of 4), rows on four elements", D);
    if (n == 0) return QSV_OK;
    const int chunks = stream_chunks(n, 512, D);
    const SlotRows slots = {ys, nullptr, weight, idx, top_k, n_experts};
#define QSV_HCWR(MS)                                                                                                                          \
    QSV_DISPATCH(dtype, "qsv_hc_write_slots_read",                                                                                            \
                 hipLaunchKernelGGL((hc_write_vec_kernel<T, float, MS, true>), dim3((unsigned)(chunks * n)), dim3(NT), 0, (hipStream_t)stream, x, (const T*)nullptr, \
                                    mix, w_out, streams, D, (T*)nullptr, (const float*)nullptr, (const T*)nullptr, (const T*)nullptr, 0.f, chunks, slots,            \
                                    ShiftedRead<T>{(T*)h_next, w_in, (const T*)norm_w, (const T*)norm_b, (const T*)shift, prev, state_rd, state_wr, alpha}))
    if (streams <= 2) QSV_HCWR(2);
    else QSV_HCWR(4);
#undef QSV_HCWR
    return qsv_launch_status("qsv_hc_write_slots_read");
}

extern "C" int qsv_dyt_sum_rows(void* out, const float* x, const int32_t* rows, const void* norm_w, const void* norm_b,
                                float alpha, int n_rows, int streams, int D, int dtype, void* stream) {
    QSV_REQUIRE(out && x && norm_w && norm_b && n_rows >= 0 && D > 0 && streams > 0, "qsv_dyt_sum_rows: bad arguments");
    if (n_rows == 0) return QSV_OK;
    const int64_t chunks = ((int64_t)D / 4 + NT - 1) / NT;
    if (D % 4 == 0 && streams <= 4 && fits4(out, dtype) && fits4(x, QSV_F32) && fits4(norm_w, dtype) && fits4(norm_b, dtype) && chunks * n_rows < (1ll << 31)) {
#define QSV_DSR(MS)                                                                                                                           \
    QSV_DISPATCH(dtype, "qsv_dyt_sum_rows",                                                                                                   \
                 hipLaunchKernelGGL((dyt_sum_rows_vec_kernel<T, MS>), dim3((unsigned)(chunks * n_rows)), dim3(NT), 0, (hipStream_t)stream, (T*)out, x, rows, \
                                    (const T*)norm_w, (const T*)norm_b, alpha, streams, D, (int)chunks))
        if (streams <= 2) QSV_DSR(2);
        else QSV_DSR(4);
#undef QSV_DSR
        return qsv_launch_status("qsv_dyt_sum_rows");
    }
    QSV_DISPATCH(dtype, "qsv_dyt_sum_rows",
                 hipLaunchKernelGGL(dyt_sum_rows_kernel<T>, dim3(n_rows), dim3(NT), 0, (hipStream_t)stream, (T*)out, x, rows,
                                    (const T*)norm_w, (const T*)norm_b, alpha, streams, D));
    return qsv_launch_status("qsv_dyt_sum_rows");
}

extern "C" int qsv_rms_pair_mean(void* out, const void* a, const void* wa, const void* b, const void* wb, float eps, int n, int D,
                                 int dtype, void* stream) {
    QSV_REQUIRE(out && a && wa && b && wb && n >= 0 && D > 0, "qsv_rms_pair_mean: bad arguments");
    if (n == 0) return QSV_OK;
#define QSV_RPM(VEC, P)                                                                                                                       \
    QSV_DISPATCH(dtype, "qsv_rms_pair_mean",                                                                                                  \
                 hipLaunchKernelGGL((rms_pair_mean_kernel<T, VEC, P>), dim3(n), dim3(NT), 0, (hipStream_t)stream, (T*)out, (const T*)a, (const T*)wa, (const T*)b, \
                                    (const T*)wb, eps, D))
    if (D % 4) QSV_RPM(false, 0);
    else if (D <= NT * 4) QSV_RPM(true, 1);
    else if (D <= NT * 8) QSV_RPM(true, 2);
    else if (D <= NT * 16) QSV_RPM(true, 4);
    else QSV_RPM(true, 0);
#undef QSV_RPM
    return qsv_launch_status("qsv_rms_pair_mean");
}

extern "C" int qsv_glu(void* out, const void* a, int n_rows, int ff, int act, float limit, const float* row_scale,
                       const int64_t* scale_index, int dtype, void* stream) {
    QSV_REQUIRE(out && a && n_rows >= 0 && ff > 0 && (act == 0 || act == 1 || (act == 2 && limit > 0.f)), "qsv_glu: bad arguments");
    if (n_rows == 0) return QSV_OK;
    if (ff % 4 == 0)
        QSV_DISPATCH(dtype, "qsv_glu",
                     hipLaunchKernelGGL((glu_kernel<T, true>), dim3(n_rows), dim3(NT), 0, (hipStream_t)stream, (T*)out, (const T*)a, ff, act,
                                        limit, row_scale, scale_index));
    else
        QSV_DISPATCH(dtype, "qsv_glu",
                     hipLaunchKernelGGL((glu_kernel<T, false>), dim3(n_rows), dim3(NT), 0, (hipStream_t)stream, (T*)out, (const T*)a, ff, act,
                                        limit, row_scale, scale_index));
    return qsv_launch_status("qsv_glu");
}
