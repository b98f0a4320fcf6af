// serve_linear.hip -- products of the few rows of a decoding step (bfloat16, float accumulation): x [T, K] @ w [N, K]^T, and one product per head.
//
// Bound by HBM (the weight, read once) and below about 20 MB by the launch.  Workgroup = 16 or 32 weight rows and up to 32 inputs, the
// weight streamed through LDS rings (serve_stream.h), the four waves' shares of the reduction added in LDS.
// Measured against the vendor's product (MI355X, weights from HBM, 1 / 16 / 32 / 64 rows, us): 2048 x 2048 4.5 / 4.7 / 5.5 / 5.6 against 8.1 / 8.2 / 8.4 /
// 8.8; 6144 x 2048 7.4 / 7.6 / 8.4 / 10.9 against 12.7 / 12.5 / 12.4 / 13.0; 32000 x 2048 27 / 28 / 30 / 47 against 34 / 34 / 35 / 35.
// (Weights that pass once stream past the caches since: 32000 x 2048 of one or 16 rows 25 - 26 us, 4096 x 4096 8.9 -> 8.5.)
#include "serve_common.h"
#include "serve_expert_rows.h"
#include "serve_latent_prep.h"
#include "serve_stream.h"
#include "serve_sum_norms.h"

namespace {
// What becomes of a product x [T, K] @ w [N, K]^T: rounded to bfloat16 it is stored, stored as float (a caller that would widen it), or, as a decay's gate, turned
// into the decay (float) with bias [N] and the log rate of its head, a_log [N / dim] or NULL.
enum { AS_IS, WIDENED, DECAY };
struct SkinnyJob {
    void* out;
    const bf16_t* X;
    int64_t x_stride;
    const bf16_t* W;
    int T, N, K, wide;
    const bf16_t* bias;
    const float* a_log;
    float inv_tau;
    int dim;
};
template <int RB, int SG, int HOW, bool ONCE>
__device__ __forceinline__ void skinny_product(const SkinnyJob& a, int block, int inputs, unsigned char* rings) {
    constexpr int TILES = RB * SG;
    static_assert(STREAM_WAVES * TILES * 1024 <= STREAM_WAVES * XRING, "");
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = block * 16 * RB, t0 = inputs * 16 * SG, count = min(16 * SG, a.T - t0);
    v4f acc[RB][SG];
    stream_products<RB, SG, ONCE>(a.W + (size_t)r0 * a.K, a.K, min(16 * RB, a.N - r0), rings + w * XRING, w, lane,
                            [&](int i) { return a.X + (size_t)(t0 + min(i, count - 1)) * (size_t)a.x_stride; }, acc);
    v4f* red = (v4f*)rings;                                         // [wave][tile][lane]
    __syncthreads();                                                // every wave is done with its ring
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int g = 0; g < SG; ++g) red[(w * TILES + r * SG + g) * 64 + lane] = acc[r][g];
    __syncthreads();
    if constexpr (HOW == DECAY) {                                   // (some hundred instructions a value: every wave takes one of a lane's four)
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const int c = 16 * (t % SG) + (lane & 15), n = r0 + 16 * (t / SG) + 4 * (lane >> 4) + w;
            if (c >= count || n >= a.N) continue;
            const float* p = (const float*)(red + t * 64 + lane) + w;
            float v = p[0];
#pragma unroll
            for (int o = 1; o < STREAM_WAVES; ++o) v += p[o * TILES * 256];
            v = gate_decay(bf2f(f2bf(v)) + bf2f(a.bias[n]), a.a_log != nullptr, a.a_log ? a.a_log[n / a.dim] : 0.f, a.inv_tau);
            ((float*)a.out)[(size_t)(t0 + c) * a.N + n] = v;
        }
        return;
    }
    for (int t = w; t < TILES; t += STREAM_WAVES) {
        const int c = 16 * (t % SG) + (lane & 15), n = r0 + 16 * (t / SG) + 4 * (lane >> 4);
        if (c >= count) continue;
        v4f v = red[t * 64 + lane];
#pragma unroll
        for (int o = 1; o < STREAM_WAVES; ++o) v += red[(o * TILES + t) * 64 + lane];
        const size_t at = (size_t)(t0 + c) * a.N + n;
        const bool whole = a.wide && n + 4 <= a.N;
        if constexpr (HOW == AS_IS) {
            bf16_t* p = (bf16_t*)a.out + at;
            if (whole) {
                *(uint2*)p = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
            } else {
                for (int q = 0; q < 4; ++q)
                    if (n + q < a.N) p[q] = f2bf(v[q]);
            }
        } else {
            float* p = (float*)a.out + at;
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = bf2f(f2bf(v[q]));
            if (whole) *(v4f*)p = v;
            else
                for (int q = 0; q < 4; ++q)
                    if (n + q < a.N) p[q] = v[q];
        }
    }
}
template <int RB, int SG, int HOW, bool ONCE>
__global__ __launch_bounds__(64 * STREAM_WAVES, 2) void skinny_linear_kernel(SkinnyJob a) {
    __shared__ __attribute__((aligned(128))) unsigned char rings[STREAM_WAVES * XRING];
    skinny_product<RB, SG, HOW, ONCE>(a, blockIdx.x, blockIdx.y, rings);
}
// A recurrence's two second stages in one launch: the decay's product (its first `blocks` workgroups) and the output gate's (N 0: none)
template <int SG>
__global__ __launch_bounds__(64 * STREAM_WAVES, 2) void decay_products_kernel(SkinnyJob decay, SkinnyJob gate, int blocks) {
    __shared__ __attribute__((aligned(128))) unsigned char rings[STREAM_WAVES * XRING];
    if ((int)blockIdx.x < blocks) skinny_product<1, SG, DECAY, false>(decay, blockIdx.x, blockIdx.y, rings);
    else skinny_product<1, SG, AS_IS, false>(gate, blockIdx.x - blocks, blockIdx.y, rings);
}
// A product (its first `blocks` workgroups, `columns` of them for the same inputs) beside the second products of a mixture's experts, which read nothing of it: a
// launch and its start less (2048 x 2048 beside 4 of 16 experts of 2048 x 1408 and a shared one, 1 / 16 / 64 tokens 3.9 / 5.6 / 4.5 us; figures of a whole layer at
// maps_beside_experts_kernel).
template <int RB, int SG, bool ONCE, int FORM>
__global__ __launch_bounds__(64 * STREAM_WAVES, 2) void skinny_beside_experts_kernel(SkinnyJob a, ExpertArgs e, SharedArgs sh, int blocks, int columns, int tiles) {
    __shared__ __attribute__((aligned(128))) unsigned char lds[EXPERT_LDS];
    const int b = blockIdx.x;
    if (b < blocks) skinny_product<RB, SG, AS_IS, ONCE>(a, b % columns, b / columns, lds);
    else expert_rows_block<ACT_NONE, true, FORM>(e, sh, (b - blocks) % tiles, (b - blocks) / tiles, lds);
}

// ---- one product per head: y[t, h] = x[t, h] @ W[h], W [H, K, N] with N contiguous -------------------------------------------------------
// Up to 64 tokens.  Bound by latency (16 heads of 128 x 512: 2 MB), so everything a wave needs is requested at once: a workgroup owns 32
// columns of one head, its four waves take the 32-deep steps of the reduction in turn (S of them at a time), and the B operands - eight
// consecutive k of a column - are put together in registers from eight rows' pairs of columns, so the weight needs neither LDS nor a second
// layout.  The waves' sums meet in LDS.
// QUERY: the result is the absorbed part of the latent query, scaled, in float rows of N + rot_dim; workgroups behind the N / 32 of the
// product turn and scale the rest of the row.
struct HeadProductArgs {
    void* out;
    const bf16_t *x, *w;
    int64_t x_tok, x_head;
    int T, K, N, H;
    const float* rope;
    const int32_t* pos;
    float scale;
    int dim, rot_dim, rot_n;
    const bf16_t* gate;              // (not QUERY) the result is multiplied by sigmoid(gate[t, h]) before it is rounded
    int64_t gate_stride;
};
template <int RT, int S, bool QUERY>
__global__ __launch_bounds__(256) void head_product_kernel(HeadProductArgs a) {
    __shared__ __attribute__((aligned(16))) float red[4][RT * 16][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = blockIdx.y;
    if (QUERY && (int)blockIdx.x * 32 >= a.N) {
        const int i = ((int)blockIdx.x - a.N / 32) * 256 + tid, t = i / a.rot_dim, c = i - t * a.rot_dim;
        if (t >= a.T) return;
        const bf16_t* qr = a.x + t * a.x_tok + h * a.x_head + a.dim;
        float v = ld(qr, c);
        if (c < a.rot_n) {
            const int half = a.rot_n / 2, p = c >> 1;
            const float* cs = a.rope + (size_t)a.pos[t] * (size_t)a.rot_n;
            const float co = cs[p], sn = cs[half + p], u = ld(qr, 2 * p), w2 = ld(qr, 2 * p + 1);
            v = (c & 1) ? (w2 * co + u * sn) : (u * co - w2 * sn);
        }
        ((float*)a.out)[((size_t)t * a.H + h) * (a.N + a.rot_dim) + a.N + c] = v * a.scale;
        return;
    }
    const int n0 = blockIdx.x * 32, kq = (lane >> 4) * 8;
    const bf16_t* W = a.w + (size_t)h * a.K * a.N + n0 + 2 * (lane & 15);
    const bf16_t* X = a.x + h * a.x_head;
    unsigned gate[RT] = {};                                                     // (first: asked for behind the sum, each row's waits for the row before)
    if (!QUERY && a.gate) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
            gate[r] = *(const unsigned*)(a.gate + min(16 * r + (tid >> 4), a.T - 1) * a.gate_stride + (size_t)h * a.N + n0 + 2 * (tid & 15));
    }
    v4f acc[RT][2];
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][0] = acc[r][1] = (v4f){0.f, 0.f, 0.f, 0.f};
    for (int k0 = wave * 32 * S; k0 < a.K; k0 += 4 * 32 * S) {                  // (K is a multiple of 32 S)
        unsigned b[S][8];
        v4u x[S][RT];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int k = k0 + 32 * s + kq;
#pragma unroll
            for (int i = 0; i < 8; ++i) b[s][i] = *(const unsigned*)(W + (size_t)(k + i) * a.N);
#pragma unroll
            for (int r = 0; r < RT; ++r) x[s][r] = *(const v4u*)(X + min(16 * r + (lane & 15), a.T - 1) * a.x_tok + k);
        }
        __builtin_amdgcn_sched_barrier(0);                                     // every request before the first use
#pragma unroll
        for (int s = 0; s < S; ++s) {
            v4u lo, hi;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                lo[i] = __builtin_amdgcn_perm(b[s][2 * i + 1], b[s][2 * i], 0x05040100u);
                hi[i] = __builtin_amdgcn_perm(b[s][2 * i + 1], b[s][2 * i], 0x07060302u);
            }
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, x[s][r]), __builtin_bit_cast(bf8, lo), acc[r][0], 0, 0, 0);
                acc[r][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, x[s][r]), __builtin_bit_cast(bf8, hi), acc[r][1], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j) *(float2*)&red[wave][16 * r + 4 * (lane >> 4) + j][2 * (lane & 15)] = make_float2(acc[r][0][j], acc[r][1][j]);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int t = 16 * r + (tid >> 4), c = 2 * (tid & 15);
        if (t >= a.T) continue;
        float2 v = make_float2(0.f, 0.f);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float2 p = *(const float2*)&red[w][t][c];
            v.x += p.x;
            v.y += p.y;
        }
        if (QUERY) *(float2*)((float*)a.out + ((size_t)t * a.H + h) * (a.N + a.rot_dim) + n0 + c) = make_float2(v.x * a.scale, v.y * a.scale);
        else {
            if (a.gate) {
                v.x *= 1.0f / (1.0f + expf(-__uint_as_float(gate[r] << 16)));
                v.y *= 1.0f / (1.0f + expf(-__uint_as_float(gate[r] & 0xffff0000u)));
            }
            *(unsigned*)((bf16_t*)a.out + ((size_t)t * a.H + h) * a.N + n0 + c) = pack_bf2(v.x, v.y);
        }
    }
}
template <int RT, bool QUERY>
void launch_head_product(const HeadProductArgs& a, int steps, int tail, hipStream_t stream) {
    const dim3 grid(a.N / 32 + tail, a.H), block(256);
    if (steps == 4) hipLaunchKernelGGL((head_product_kernel<RT, 4, QUERY>), grid, block, 0, stream, a);
    else if (steps == 2) hipLaunchKernelGGL((head_product_kernel<RT, 2, QUERY>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((head_product_kernel<RT, 1, QUERY>), grid, block, 0, stream, a);
}
bool head_product_ok(int T, int64_t x_tok, int64_t x_head, const void* x, const void* w, int K, int N, int H) {
    return T > 0 && T <= 64 && H > 0 && H <= 65535 && K > 0 && N > 0 && K % 32 == 0 && N % 32 == 0 && (int64_t)K * N < (1ll << 31) && x_tok >= 0 &&
           x_head >= 0 && x_tok % 8 == 0 && x_head % 8 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 4 == 0;
}
template <bool QUERY>
int run_head_product(const HeadProductArgs& a, hipStream_t stream, const char* what) {
    const int tail = QUERY ? (a.T * a.rot_dim + 255) / 256 : 0;
    const int steps = a.K % 512 == 0 ? 4 : a.K % 256 == 0 ? 2 : 1;            // per wave at once: the four waves share K evenly
    if (a.T <= 16) launch_head_product<1, QUERY>(a, steps, tail, stream);
    else if (a.T <= 32) launch_head_product<2, QUERY>(a, steps, tail, stream);
    else launch_head_product<4, QUERY>(a, steps, tail, stream);
    return qsv_launch_status(what);
}
// ---- products of few rows that their workgroups make themselves: 16 weight rows a workgroup, its weights in registers ---------------------
// The stages of a wave, w + 4 s as in stream_products (stages behind the row's end repeat the last)
template <int S, bool ONCE>
__device__ __forceinline__ void request_stages(const bf16_t* W, int N, int K, int block, v4u (&A)[S][2]) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), stages = K / XK;
    const bf16_t* row = W + (size_t)min(16 * block + (lane & 15), N - 1) * K + 8 * (lane >> 4);
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const v4u* from = (const v4u*)(row + min(w + STREAM_WAVES * s, stages - 1) * XK + 32 * ks);
            A[s][ks] = ONCE ? __builtin_nontemporal_load(from) : *from;
        }
}
// out [T, N] from them and `held` rows of K elements in LDS (of every 128 bytes piece p at p ^ (row & 7)), T <= held; red: 4 KiB of LDS.  The order of the sums is that
// of skinny_product.  N a multiple of four.
template <int S>
__device__ __forceinline__ void register_product(const v4u (&A)[S][2], const unsigned char* rows, int held, int K, unsigned char* red_, bf16_t* out, int T, int N, int block) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), stages = K / XK;
    __syncthreads();                                                 // the rows are there
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    const int in = min(lane & 15, held - 1);                         // (columns behind T are not stored)
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int stage = w + STREAM_WAVES * s;
        if (stage >= stages) break;                                  // (wave-uniform)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const v4u B = *(const v4u*)(rows + in * K * 2 + stage * 128 + (((4 * ks + (lane >> 4)) ^ (in & 7)) << 4));
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, A[s][ks]), __builtin_bit_cast(bf8, B), acc, 0, 0, 0);
        }
    }
    v4f* red = (v4f*)red_;                                           // [wave][lane]
    red[w * 64 + lane] = acc;
    __syncthreads();
    const int c = lane & 15, n = 16 * block + 4 * (lane >> 4);
    if (w || c >= T) return;
    v4f v = red[lane];
#pragma unroll
    for (int o = 1; o < STREAM_WAVES; ++o) v += red[o * 64 + lane];
    if (n < N) *(uint2*)(out + (size_t)c * N + n) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
}

// ---- a step's latent queries: out [T, N] = rms_norm(row's query latent) @ w [N, q_rank]^T, the rows' key-value halves beside it ------------
// Up to 16 tokens.  The norm and the product were two launches, each a trip to memory behind the other.  Here a product's workgroup (16 weight rows) requests its
// inputs' rows and then all of its weights, norms the rows into LDS while those are on their way (R rows a wave) and multiplies what it has in registers: one
// trip.  Every workgroup norms every row, which is what bounds it; the first T workgroups write the cache rows.  The sums, roundings and the order of the
// products are the two kernels': the same bits.
// Measured, the two launches -> this one, weights from memory, 1 / 8 / 16 tokens, us: 768 to 3072 5.7 -> 3.4, 6.0 -> 3.6, 6.3 -> 4.6, to 2048 5.4 -> 3.3, 5.6 -> 3.6, 6.1 -> 4.4,
// 512 to 3072 5.4 -> 3.0, 5.6 -> 3.3, 5.9 -> 3.9, 256 to 1536 4.5 -> 2.5, 4.7 -> 2.7, 4.8 -> 3.5.  The rows' norms grow with the tokens: 32 rows a workgroup lost at 48 and 64 tokens
// (7.5 -> 9.0), and so do large products of more than 8 (1024 to 6144, 16 tokens 7.5 -> 7.5, left in the caches 6.9 -> 7.1; 768 to 6144 7.0 -> 6.4), which is latent_up_sizes' line;
// beyond the sizes measured the two launches stay.
template <int R, int S, bool ONCE>
__device__ __forceinline__ void latent_up_product(const LatentPrep<bf16_t>& a, const bf16_t* W, bf16_t* out, int T, int N, int block, unsigned char* lds) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), K = a.q_rank;
    raw2u rx[R][S], rw[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int c = min(4 * (64 * s + lane), K - 4);
        rw[s] = raw4(a.q_w, c);
#pragma unroll
        for (int r = 0; r < R; ++r) rx[r][s] = raw4(a.down + (size_t)min(w * R + r, T - 1) * a.down_stride + a.q_off, c);
    }
    v4u A[S][2];
    request_stages<S, ONCE>(W, N, K, block, A);
    requested();
    float g[S][4];
#pragma unroll
    for (int s = 0; s < S; ++s) widen4(rw[s], g[s]);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = w * R + r;
        float v[S][4], sum = 0.f;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            widen4(rx[r][s], v[s]);
            float q = 0.f;
            const float s4 = square_sum4(v[s]);
            if (4 * (64 * s + lane) < K) q += s4;
            sum += wave_sum(q);
        }
        const float inv = 1.0f / sqrtf(sum / (float)K + a.eps);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int c = 4 * (64 * s + lane);
            if (c >= K) continue;
            *(uint2*)(lds + row * K * 2 + (c / XK) * 128 + ((((c & 63) >> 3) ^ (row & 7)) << 4) + (c & 4) * 2) =
                make_uint2(pack_bf2(v[s][0] * inv * g[s][0], v[s][1] * inv * g[s][1]), pack_bf2(v[s][2] * inv * g[s][2], v[s][3] * inv * g[s][3]));
        }
    }
    register_product<S>(A, lds, 4 * R, K, lds + 4 * R * S * 512, out, T, N, block);
}
template <int R, int S, int P, bool ONCE>
__global__ __launch_bounds__(64 * STREAM_WAVES, 2) void latent_up_kernel(LatentPrep<bf16_t> a, const bf16_t* W, bf16_t* out, int T, int N) {
    __shared__ __attribute__((aligned(128))) unsigned char lds[4 * R * S * 512 + STREAM_WAVES * 1024];
    const int b = (int)blockIdx.x - T;
    if (b < 0) latent_prep_row<bf16_t, P, 64 * STREAM_WAVES, false>(a, blockIdx.x);
    else latent_up_product<R, S, ONCE>(a, W, out, T, N, b, lds);
}

// ---- a parallel layer's norms with the mixer's product of the first one: scaled_sum_row and out [T, N] = h0 @ w [N, D]^T --------------------
// One or two tokens.  The norms' kernel is one workgroup a token, a chain from the parts' rows to the router's choice, and the product waited for it.  Here its
// workgroups make the first norm's rows themselves, while their weights are on the way; the first T do the norms' kernel's work as before, the router's included, which
// nothing waits for before the next launch.  x is read by every workgroup, so the sum goes to rows of its own (x_out).  The same bits.
// Measured, the two launches -> this one, weights from memory, 4 of 16 experts' rows and a shared one's, rows of 2048, one / two tokens, us: to 2560 10.0 -> 6.5, 10.3 -> 8.2, 4096
// 11.0 -> 8.6, 10.9 -> 9.9, 5120 12.0 -> 10.7, 11.8 -> 12.8, 8192 14.0 -> 14.0, 13.9 -> 15.4; of 1024 to 2560 8.4 -> 5.2, 8.6 -> 5.5, 512 to 1536 6.6 -> 4.1, 6.7 -> 5.1; 64 experts,
// 4096 18.3 -> 16.3, 18.5 -> 16.3.  A workgroup reads as many bytes of parts as of weights, so wide products lose: the line is at 6144 for one token, 4096 for two.
struct SumProduct {
    float* x_out;
    const float* x;
    bf16_t *h0, *h1;
    ScaledParts parts;
    const float *g0, *g1;
    const int32_t* tokens;
    const bf16_t* table;
    float eps;
    int D;
    SlotRows slots;
    RouteArgs route;
    bf16_t* out;
    const bf16_t* W;
    int T, N;
};
template <int VPT, int NP, typename Y, int EC, bool ONCE>
__global__ __launch_bounds__(256, 2) void sum_norms_product_kernel(SumProduct a) {
    __shared__ __attribute__((aligned(128))) unsigned char lds[2 * VPT * 2048 + STREAM_WAVES * 1024];
    const int block = (int)blockIdx.x - a.T;
    if (block < 0) {
        scaled_sum_row<bf16_t, VPT, NP, Y, EC, 256, false>(blockIdx.x, a.x_out, a.x, a.h0, a.h1, a.parts, a.g0, a.g1, a.tokens, a.table, a.eps, a.D, a.slots, a.route, nullptr,
                                                          NothingMore());
        return;
    }
    constexpr int S = 4 * VPT;
    v4u A[S][2];
    scaled_sum_row<bf16_t, VPT, NP, Y, 0, 256, true>(0, nullptr, a.x, nullptr, nullptr, a.parts, a.g0, a.g1, a.tokens, a.table, a.eps, a.D, a.slots, a.route, lds,
                                                     [&]() __attribute__((always_inline)) { request_stages<S, ONCE>(a.W, a.N, a.D, block, A); });
    if (a.T > 1)
        scaled_sum_row<bf16_t, VPT, NP, Y, 0, 256, true>(1, nullptr, a.x, nullptr, nullptr, a.parts, a.g0, a.g1, a.tokens, a.table, a.eps, a.D, a.slots, a.route, lds, NothingMore());
    register_product<S>(A, lds, a.T, a.D, lds + 2 * VPT * 2048, a.out, a.T, a.N, block);
}
}  // namespace

// out [T, H, N] = x[t, h] @ w[h], x rows x_tok / x_head elements apart, w [H, K, N]
extern "C" int qsv_head_product(void* out, const void* x, int64_t x_tok, int64_t x_head, const void* w, int T, int H, int K, int N, void* stream) {
    QSV_REQUIRE(out && x && w && head_product_ok(T, x_tok, x_head, x, w, K, N, H) && (uintptr_t)out % 4 == 0, "qsv_head_product: bad arguments");
    return run_head_product<false>({out, (const bf16_t*)x, (const bf16_t*)w, x_tok, x_head, T, K, N, H, nullptr, nullptr, 1.0f, 0, 0, 0, nullptr, 0},
                                   (hipStream_t)stream, "qsv_head_product");
}
// ... times sigmoid(gate[t, h]), rows of gate gate_stride apart
extern "C" int qsv_head_product_gated(void* out, const void* x, int64_t x_tok, int64_t x_head, const void* w, int T, int H, int K, int N, const void* gate,
                                      int64_t gate_stride, void* stream) {
    QSV_REQUIRE(out && x && w && gate && head_product_ok(T, x_tok, x_head, x, w, K, N, H) && (uintptr_t)out % 4 == 0 && (uintptr_t)gate % 4 == 0 && gate_stride % 2 == 0 &&
                    gate_stride >= (int64_t)H * N, "qsv_head_product_gated: bad arguments");
    return run_head_product<false>({out, (const bf16_t*)x, (const bf16_t*)w, x_tok, x_head, T, K, N, H, nullptr, nullptr, 1.0f, 0, 0, 0, (const bf16_t*)gate, gate_stride},
                                   (hipStream_t)stream, "qsv_head_product_gated");
}

// qf [T, H, rank + rot_dim] (float) = scale * [q[t, h, :dim] @ w_uk[h] | rotated q[t, h, dim:]], q [T, H, dim + rot_dim], w_uk [H, dim, rank]
extern "C" int qsv_latent_query_product(float* qf, const void* q, const void* w_uk, const float* rope, const int32_t* pos, float scale, int T, int H,
                                        int dim, int rot_dim, int rot_n, int rank, void* stream) {
    QSV_REQUIRE(qf && q && w_uk && pos && dim > 0 && rot_dim >= 0 && rot_n >= 0 && rot_n <= rot_dim && rot_n % 2 == 0 && (rot_n == 0 || rope) &&
                    rot_dim <= (1 << 20) && rot_dim % 2 == 0 && (uintptr_t)qf % 8 == 0, "qsv_latent_query_product: bad arguments");
    const int64_t row = dim + rot_dim;
    QSV_REQUIRE(head_product_ok(T, row * H, row, q, w_uk, dim, rank, H), "qsv_latent_query_product: sizes or addresses it does not take");
    return run_head_product<true>({qf, (const bf16_t*)q, (const bf16_t*)w_uk, row * H, row, T, dim, rank, H, rope, pos, scale, dim, rot_dim, rot_n, nullptr, 0},
                                  (hipStream_t)stream, "qsv_latent_query_product");
}

static int skinny_fits(const char* what, const void* out, const void* x, int64_t x_stride, const void* w, int n_rows, int N, int K) {
    QSV_REQUIRE(out && x && w && n_rows >= 0 && N > 0 && K > 0 && K % 8 == 0 && x_stride % 8 == 0 && x_stride >= 0, "%s: bad arguments", what);
    QSV_REQUIRE(((uintptr_t)x | (uintptr_t)w) % 16 == 0, "%s: inputs and weights start on 16 bytes", what);
    QSV_REQUIRE(K <= (1 << 25) && n_rows <= 65535 * 16, "%s: %d inputs of %d", what, n_rows, K);
    return QSV_OK;
}
template <int HOW>
static int launch_skinny(const char* what, void* out, const void* x, int64_t x_stride, const void* w, int n_rows, int N, int K, void* stream, bool kept = false, const qsv_expert_job* beside = nullptr) {
    const int rc = skinny_fits(what, out, x, x_stride, w, n_rows, N, K);
    if (rc != QSV_OK || n_rows == 0) return rc;
    ExpertArgs e = {};
    SharedArgs sh = {};
    dim3 experts;
    if (beside) {
        int act = beside->act, rc2 = expert_slots_args(what, *beside, e, sh);
        if (rc2 == QSV_OK) rc2 = plan_expert_rows(what, e, sh, beside->n_experts, act, beside->kept != 0, experts);
        if (rc2 != QSV_OK) return rc2;
        QSV_REQUIRE(beside->float_out && beside->n > 0 && (int64_t)experts.x * experts.y < (1ll << 30), "%s: not these experts", what);
    }
    const SkinnyJob a = {out, (const bf16_t*)x, x_stride, (const bf16_t*)w, n_rows, N, K, N % 4 == 0 && (uintptr_t)out % (HOW == AS_IS ? 8 : 16) == 0, nullptr, nullptr, 0.f, 1};
    // 16 weight rows per workgroup where 32 would leave CUs without one, or need a second round for a few (8256 x 2048: 11.4 -> 10.5 us); else 32,
    // which reads the inputs half as often (6144 x 2048: 8.2 -> 7.4 us)
    const bool few = n_rows <= 16, small = N < 5120 || (N > 8192 && N <= 16384 && n_rows <= 32);
    // every weight is read once, or twice at the same time
    const bool once = !kept && streams_once(w, N, K);
#define QSV_SKINNY(RB, SG)                                                                                                                    \
    do {                                                                                                                                      \
        const dim3 grid((N + 16 * RB - 1) / (16 * RB), (n_rows + 16 * SG - 1) / (16 * SG)), block(64 * STREAM_WAVES);                         \
        const bool past = once && (grid.y == 1 || (int64_t)grid.x * grid.y <= 256);                                                          \
        if (beside) {                                                                                                                         \
            if constexpr (HOW == AS_IS) {                                                                                                     \
                const int64_t blocks = (int64_t)grid.x * grid.y, all = blocks + (int64_t)experts.x * experts.y;                               \
                QSV_REQUIRE(all < (1ll << 31), "%s: too many workgroups", what);                                                              \
                auto kernel = past ? skinny_beside_experts_kernel<RB, SG, true, SLOTS> : skinny_beside_experts_kernel<RB, SG, false, SLOTS>;  \
                if (early_experts(e, beside->n_experts))                                                                                      \
                    kernel = past ? skinny_beside_experts_kernel<RB, SG, true, SLOTS_EARLY> : skinny_beside_experts_kernel<RB, SG, false, SLOTS_EARLY>; \
                else if (SG == 1 && few_slots(e, sh))                                                                                              \
                    kernel = past ? skinny_beside_experts_kernel<RB, 1, true, SLOTS_FEW> : skinny_beside_experts_kernel<RB, 1, false, SLOTS_FEW>; \
                hipLaunchKernelGGL(kernel, dim3((unsigned)all), block, 0, (hipStream_t)stream, a, e, sh, (int)blocks, (int)grid.x, (int)experts.x); \
            }                                                                                                                                 \
        } else if (past)                                                                                                                      \
            hipLaunchKernelGGL((skinny_linear_kernel<RB, SG, HOW, true>), grid, block, 0, (hipStream_t)stream, a);                            \
        else hipLaunchKernelGGL((skinny_linear_kernel<RB, SG, HOW, false>), grid, block, 0, (hipStream_t)stream, a);                          \
    } while (0)
    if (few && small) QSV_SKINNY(1, 1);
    else if (few) QSV_SKINNY(2, 1);
    else if (small) QSV_SKINNY(1, 2);
    else QSV_SKINNY(2, 2);
#undef QSV_SKINNY
    return qsv_launch_status(what);
}
extern "C" int qsv_skinny_linear(void* out, const void* x, int64_t x_stride, const void* w, int n_rows, int N, int K, void* stream) {
    return launch_skinny<AS_IS>("qsv_skinny_linear", out, x, x_stride, w, n_rows, N, K, stream);
}
// ... beside expert products into float (kept: w is to stay in the caches)
extern "C" int qsv_skinny_linear_beside(void* out, int kept, const void* x, int64_t x_stride, const void* w, int n_rows, int N, int K, const qsv_expert_job* experts,
                                        void* stream) {
    QSV_REQUIRE(experts && n_rows > 0, "qsv_skinny_linear_beside: bad arguments");
    return launch_skinny<AS_IS>("qsv_skinny_linear_beside", out, x, x_stride, w, n_rows, N, K, stream, kept != 0, experts);
}
// the same values in float
extern "C" int qsv_skinny_linear_widened(float* out, const void* x, int64_t x_stride, const void* w, int n_rows, int N, int K, void* stream) {
    return launch_skinny<WIDENED>("qsv_skinny_linear_widened", out, x, x_stride, w, n_rows, N, K, stream);
}
// either of them with weights that are to stay in the caches
extern "C" int qsv_skinny_linear_kept(void* out, int widened, const void* x, int64_t x_stride, const void* w, int n_rows, int N, int K, void* stream) {
    return widened ? launch_skinny<WIDENED>("qsv_skinny_linear_kept", out, x, x_stride, w, n_rows, N, K, stream, true)
                   : launch_skinny<AS_IS>("qsv_skinny_linear_kept", out, x, x_stride, w, n_rows, N, K, stream, true);
}
// decay [n_rows, N] (float) of z = x @ w^T as qsv_decay makes it, and, with gate_N > 0, gate [n_rows, gate_N] = gate_x @ gate_w^T
extern "C" int qsv_decay_products(float* decay, const void* x, int64_t x_stride, const void* w, int N, int K, const void* bias, const float* a_log, float tau, int dim,
                                  void* gate, const void* gate_x, int64_t gate_x_stride, const void* gate_w, int gate_N, int gate_K, int n_rows, void* stream) {
    int rc = skinny_fits("qsv_decay_products", decay, x, x_stride, w, n_rows, N, K);
    if (rc == QSV_OK && gate_N) rc = skinny_fits("qsv_decay_products (gate)", gate, gate_x, gate_x_stride, gate_w, n_rows, gate_N, gate_K);
    if (rc != QSV_OK) return rc;
    QSV_REQUIRE(bias && dim > 0 && N % dim == 0 && gate_N >= 0 && (a_log || tau > 0.f), "qsv_decay_products: %d decays of heads of %d", N, dim);
    if (n_rows == 0) return QSV_OK;
    const SkinnyJob a = {decay, (const bf16_t*)x, x_stride, (const bf16_t*)w, n_rows, N, K, N % 4 == 0 && (uintptr_t)decay % 16 == 0, (const bf16_t*)bias, a_log,
                         a_log ? 0.f : 1.0f / tau, dim};
    const SkinnyJob g = {gate, (const bf16_t*)gate_x, gate_x_stride, (const bf16_t*)gate_w, n_rows, gate_N, gate_N ? gate_K : 8, gate_N % 4 == 0 && (uintptr_t)gate % 8 == 0,
                         nullptr, nullptr, 0.f, 1};
    const int blocks = (N + 15) / 16, more = (gate_N + 15) / 16;
    if (n_rows <= 16) hipLaunchKernelGGL(decay_products_kernel<1>, dim3(blocks + more, 1), dim3(64 * STREAM_WAVES), 0, (hipStream_t)stream, a, g, blocks);
    else hipLaunchKernelGGL(decay_products_kernel<2>, dim3(blocks + more, (n_rows + 31) / 32), dim3(64 * STREAM_WAVES), 0, (hipStream_t)stream, a, g, blocks);
    return qsv_launch_status("qsv_decay_products");
}

// Whether qsv_latent_up takes a row's parts: the latents in groups of four columns, the query's in stages of the product
static bool latent_up_sizes(int n, int q_off, int q_rank, int kv_off, int kv_rank, int rot_dim, int64_t down_stride, int N) {
    return q_rank > 0 && n <= (N <= 4800000 / q_rank ? 16 : 8) && q_rank % XK == 0 && q_rank <= 1024 && kv_rank > 0 && kv_rank % 4 == 0 && rot_dim >= 0 && rot_dim % 4 == 0 && q_off % 4 == 0 && kv_off % 4 == 0 &&
           down_stride % 4 == 0 && q_rank + kv_rank + rot_dim <= 4096 && N > 0 && N % 4 == 0 && N <= 6144;
}
extern "C" int qsv_latent_up_ok(int n, int q_off, int q_rank, int kv_off, int kv_rank, int rot_dim, int64_t down_stride, int N) {
    return latent_up_sizes(n, q_off, q_rank, kv_off, kv_rank, rot_dim, down_stride, N);
}
// qsv_latent_prep of up to 16 tokens (bfloat16) with its query latents multiplied in the same launch: q [n, N] = cq @ w_uq [N, q_rank]^T
extern "C" int qsv_latent_up(void* q, const void* w_uq, int N, int kept, const void* down, int64_t down_stride, int q_off, int q_rank, const void* q_w, int kv_off, int kv_rank,
                             const void* kv_w, int rot_dim, int rot_n, const float* rope, void* pool, const int64_t* slot, const int32_t* pos, float eps, int n, void* stream) {
    QSV_REQUIRE(q && w_uq && down && q_w && kv_w && pool && slot && pos && n >= 0, "qsv_latent_up: bad arguments");
    QSV_REQUIRE(latent_up_sizes(n, q_off, q_rank, kv_off, kv_rank, rot_dim, down_stride, N) && rot_n >= 0 && rot_n <= rot_dim && rot_n % 2 == 0 && (rot_n == 0 || rope),
                "qsv_latent_up: sizes it does not take");
    QSV_REQUIRE(q_off >= 0 && kv_off >= 0 && q_off + q_rank <= down_stride && kv_off + kv_rank + rot_dim <= down_stride,
                "qsv_latent_up: the slices do not fit a row of %lld elements", (long long)down_stride);
    QSV_REQUIRE(((uintptr_t)w_uq % 16 | ((uintptr_t)q | (uintptr_t)down | (uintptr_t)q_w | (uintptr_t)kv_w | (uintptr_t)pool) % 8) == 0, "qsv_latent_up: addresses it does not take");
    if (n == 0) return QSV_OK;
    const LatentPrep<bf16_t> a = {(const bf16_t*)down, down_stride, q_off, q_rank, (const bf16_t*)q_w, nullptr, kv_off, kv_rank, (const bf16_t*)kv_w, rot_dim, rot_n,
                                  rot_n ? rope : nullptr, (bf16_t*)pool, slot, pos, eps};
    const int columns = (N + 15) / 16, width = q_rank + kv_rank + rot_dim;
    const bool once = !kept && streams_once(w_uq, N, q_rank);
    const dim3 grid(n + columns), block(64 * STREAM_WAVES);
#define QSV_UP(R, S, P)                                                                                                                       \
    do {                                                                                                                                      \
        auto kernel = once ? latent_up_kernel<R, S, P, true> : latent_up_kernel<R, S, P, false>;                                              \
        hipLaunchKernelGGL(kernel, grid, block, 0, (hipStream_t)stream, a, (const bf16_t*)w_uq, (bf16_t*)q, n, N);                            \
    } while (0)
#define QSV_UP_P(R, S)                                                                                                                        \
    do {                                                                                                                                      \
        if (width <= 2048) QSV_UP(R, S, 2);                                                                                                   \
        else QSV_UP(R, S, 4);                                                                                                                 \
    } while (0)
#define QSV_UP_S(R)                                                                                                                           \
    do {                                                                                                                                      \
        if (q_rank <= 512) QSV_UP_P(R, 2);                                                                                                    \
        else if (q_rank <= 768) QSV_UP_P(R, 3);                                                                                               \
        else QSV_UP_P(R, 4);                                                                                                                  \
    } while (0)
    if (n <= 4) QSV_UP_S(1);
    else if (n <= 8) QSV_UP_S(2);
    else QSV_UP_S(4);
#undef QSV_UP_S
#undef QSV_UP_P
#undef QSV_UP
    return qsv_launch_status("qsv_latent_up");
}

extern "C" int qsv_sum_norms_product(void* out, const void* w, int N, int kept, float* x_out, const float* x, void* h0, void* h1, const void* a, const void* sa, const float* ys,
                                     const int32_t* slot_idx, const float* slot_weight, int slot_top, int n_experts, const void* slot_scale, const void* c, const void* sc,
                                     const float* g0, const float* g1, const int32_t* tokens, const void* table, float eps, int n, int D, int32_t* idx, float* weight,
                                     const void* router, const void* bias, int renorm, int E, int top_k, int G, int keep, int score_fn, const float* correction, int group_top,
                                     float scale, void* stream) {
    QSV_REQUIRE(out && w && x_out && h0 && h1 && g0 && g1 && n >= 0 && n <= 2 && D > 0 && D % XK == 0 && D <= 2048 && N > 0 && N % 4 == 0 && N <= 1 << 24 &&
                    (tokens ? table && !a && !ys && !c : x && x != x_out && a && ys && slot_idx && slot_top > 0 && n_experts > 0), "qsv_sum_norms_product: bad arguments");
    const RouteArgs r = {idx, weight, router, bias, correction, renorm, E, top_k, G, keep, score_fn, group_top, scale};
    QSV_REQUIRE(route_ok(r), "qsv_sum_norms_product: %d experts in %d groups, %d groups kept, top %d", E, G, keep, top_k);
    QSV_REQUIRE(((uintptr_t)w % 16 | ((uintptr_t)x | (uintptr_t)x_out | (uintptr_t)ys | (uintptr_t)g0 | (uintptr_t)g1) % 16 |
                 ((uintptr_t)out | (uintptr_t)h0 | (uintptr_t)h1 | (uintptr_t)a | (uintptr_t)sa | (uintptr_t)slot_scale | (uintptr_t)c | (uintptr_t)sc | (uintptr_t)table) % 8) == 0,
                "qsv_sum_norms_product: addresses it does not take");
    if (n == 0) return QSV_OK;
    const SumProduct p = {x_out, x, (bf16_t*)h0, (bf16_t*)h1, {{a, c, nullptr}, {sa, sc, nullptr}, slot_scale}, g0, g1, tokens, (const bf16_t*)table, eps, D,
                          {ys, nullptr, slot_weight, slot_idx, slot_top, n_experts}, r, (bf16_t*)out, (const bf16_t*)w, n, N};
    const bool once = !kept && streams_once(w, N, D);
#define QSV_SNP(V, NP, Y, EC)                                                                                                                 \
    do {                                                                                                                                      \
        auto kernel = once ? sum_norms_product_kernel<V, NP, Y, EC, true> : sum_norms_product_kernel<V, NP, Y, EC, false>;                    \
        hipLaunchKernelGGL(kernel, dim3(n + (N + 15) / 16), dim3(256), 0, (hipStream_t)stream, p);                                            \
    } while (0)
#define QSV_SNP_V(NP, Y, EC)                   \
    do {                                       \
        if (D <= 1024) QSV_SNP(1, NP, Y, EC);  \
        else QSV_SNP(2, NP, Y, EC);            \
    } while (0)
#define QSV_SNP_P(EC)                          \
    do {                                       \
        if (tokens) QSV_SNP_V(0, void, EC);    \
        else if (c) QSV_SNP_V(2, float, EC);   \
        else QSV_SNP_V(1, float, EC);          \
    } while (0)
    if (E <= 8) QSV_SNP_P(8);
    else QSV_SNP_P(16);
#undef QSV_SNP
#undef QSV_SNP_V
#undef QSV_SNP_P
    return qsv_launch_status("qsv_sum_norms_product");
}
