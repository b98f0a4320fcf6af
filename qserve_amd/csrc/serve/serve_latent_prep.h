// serve_latent_prep.h -- the row that a latent attention layer's first product leaves, [query latent | key-value latent | rotated key]: both latents normed, the key
// part turned and written to the cache.  Used by the kernel of its own (serve_rows.hip) and beside the queries' product (serve_linear.hip).
#pragma once
#include "serve_common.h"

namespace {
template <typename T>
struct LatentPrep {
    const T* down;
    int64_t down_stride;
    int q_off, q_rank;
    const T* q_w;
    T* cq;                           // [n, q_rank]
    int kv_off, kv_rank;
    const T* kv_w;
    int rot_dim, rot_n;
    const float* rope;
    T* pool;
    const int64_t* slot;
    const int32_t* pos;
    float eps;
};
__device__ __forceinline__ float square_sum4(const float (&v)[4]) { return v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3]; }
// A workgroup of NT threads per row: a thread owns groups of four columns, all requested before the first sum; the two sums meet in one exchange.  Bound by the
// row's latency in a step, by memory in a prompt.  QUERY: the query latent is stored too.
template <typename T, int P, int NT, bool QUERY>
__device__ __forceinline__ void latent_prep_row(const LatentPrep<T>& a, size_t t) {
    __shared__ float red[2][NT / 64];
    const T* row = a.down + t * a.down_stride;
    const int q_rank = a.q_rank, kv_rank = a.kv_rank, rot_n = a.rot_n, width = q_rank + kv_rank + a.rot_dim, half = rot_n / 2;
    typename Raw4<T>::type rx[P], rw[P];
    float co[P][2], sn[P][2];
    const float* cs = a.rope ? a.rope + (size_t)a.pos[t] * (size_t)rot_n : nullptr;
    T* dst = a.pool + (size_t)a.slot[t] * (size_t)(kv_rank + a.rot_dim);
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int c = min((k * NT + (int)threadIdx.x) * 4, width - 4);
        rx[k] = raw4(row, c < q_rank ? a.q_off + c : a.kv_off + c - q_rank);
        rw[k] = raw4(c < q_rank ? a.q_w : a.kv_w, c < q_rank ? c : min(c - q_rank, kv_rank - 4));     // (no weight on the rotated part)
    }
    if (a.rope) {
#pragma unroll
        for (int k = 0; k < P; ++k) {                               // (a group's first pair may be rotated and its second not)
            const int d = (k * NT + (int)threadIdx.x) * 4 - q_rank - kv_rank, p = max(0, min(d, rot_n - 2)) / 2, q = max(0, min(d + 2, rot_n - 2)) / 2;
            co[k][0] = cs[p];
            sn[k][0] = cs[half + p];
            co[k][1] = cs[q];
            sn[k][1] = cs[half + q];
        }
    }
    requested();
    float v[P][4], sq = 0.f, sk = 0.f;
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int c = (k * NT + (int)threadIdx.x) * 4;
        widen4(rx[k], v[k]);
        const float s = square_sum4(v[k]);
        if (c < q_rank) sq += s;
        else if (c < q_rank + kv_rank) sk += s;
    }
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = sq;
        red[1][threadIdx.x >> 6] = sk;
    }
    __syncthreads();
    sq = sk = 0.f;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) {
        sq += red[0][i];
        sk += red[1][i];
    }
    const float qinv = 1.0f / sqrtf(sq / (float)q_rank + a.eps), kinv = 1.0f / sqrtf(sk / (float)kv_rank + a.eps);
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int c = (k * NT + (int)threadIdx.x) * 4, d = c - q_rank - kv_rank;
        if (c >= width) continue;
        float w[4];
        widen4(rw[k], w);
        if (d < 0) {
            const float inv = c < q_rank ? qinv : kinv;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[k][j] = v[k][j] * inv * w[j];
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j)
                if (d + 2 * j < rot_n) {
                    const float x = v[k][2 * j], y = v[k][2 * j + 1];
                    v[k][2 * j] = x * co[k][j] - y * sn[k][j];
                    v[k][2 * j + 1] = y * co[k][j] + x * sn[k][j];
                }
        }
        if (c >= q_rank) st4t(dst, c - q_rank, v[k]);
        else if (QUERY) st4t(a.cq, t * q_rank + c, v[k]);
    }
}
}  // namespace
