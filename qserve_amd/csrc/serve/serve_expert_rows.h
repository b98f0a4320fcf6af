// serve_expert_rows.h -- a mixture's expert products of a decoding step (expert-major form): the work of one workgroup and the launch's checks and grid,
// for the kernel of its own (serve_moe.hip) and for kernels that run it beside a mixer's (serve_differential.hip, serve_linear.hip).
#pragma once
#include <type_traits>

#include "serve_common.h"
#include "serve_stream.h"

namespace {
// Activation of the first expert product.  ACT_GLU: the weight rows come in pairs (2f = gate, 2f + 1 = up) and output f is
// silu(gate) * up, so the output is half as wide as the product.
constexpr int ACT_NONE = 0, ACT_RELU_SQ = 1, ACT_GLU = 2;
// (QSV_ACT_CLAMPED_GLU runs the ACT_GLU kernels with limit > 0: g = min(gate, limit), u = clamp(up, -limit, limit), g sigmoid(1.702 g) (u + 1))
__device__ __forceinline__ float relu_sq(float d) {
    const float a = fmaxf(d, 0.f);
    return a * a;
}
__device__ __forceinline__ float glu(float g, float u, float limit) {
    if (limit > 0.f) {                                       // (uniform over the launch)
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
    }
    return g / (1.0f + expf(-g)) * u;
}

// ---- expert-major form (decoding and short portions, bfloat16): workgroup = (32 weight rows, expert), every weight read once per step
// however many tokens share the expert.  Bound by HBM (the chosen experts' weights) and, below that, by launch latency.
// * The slots (token t's k-th choice: slot t top_k + k) of an expert are found by the workgroup itself from the router's indices - no
//   sort, no counts on the host - or given as sorted runs (`offsets`).
// * The weights stream through per-wave LDS rings (serve_stream.h); the expert's inputs are read once per workgroup.
// * The partial sums of the four waves meet in LDS; more than 32 slots per expert are walked in chunks (the weights then come from L2).
// Two workgroups per CU keep up to 96 KiB of weights in flight.
// Measured per launch in a step (MI355X): 64 tokens, 4 of 16 experts of 2048 x 1408 (92 MB a product) 55.6 / 62.4 us -> 23.8 / 21.1 us (up /
// down) against the form it replaces, which kept weight rows in registers and paid a wave-wide sum per token and row; 16 tokens with
// gated units (184 + 92 MB) 42.6 / 26.1 -> 36.5 / 19.3 us (5.0 TB/s); one token 1446 / 3117 us (the per-token kernels) -> 14.0 / 8.8 us.
// The sort, search and permutation launches in front of it (60 us a layer) are gone.  Streamed past the caches, the shared expert in the same
// launch: 64 tokens 22.7 / 19.4 us (98 MB), 16 tokens gated 33.8 / 17.6 (196 / 98 MB, 5.7 TB/s), one token 15.3 / 9.5 (before its workgroups were the slots').
// 32 rows: 16, more evenly spread over the CUs, read the inputs twice as often and are slower everywhere (64 tokens 24.7 / 25.7, 16 tokens 36.3 / 21.4,
// one 18.7 / 11.7), and so are 64; rings twice as deep give no more.
constexpr int EXPERT_THREADS = 64 * STREAM_WAVES;
constexpr int XR = 32;               // weight rows per workgroup
constexpr int XLIST = 1024;          // router indices looked at in one go
constexpr int EXPERT_LDS = STREAM_WAVES * XRING + XLIST * 2 + STREAM_WAVES * 4;

struct ExpertArgs {
    void* out;                       // bf16, or float (no activation)
    const bf16_t* X;
    const bf16_t* W;
    const int32_t* idx;              // the router's indices [n] (or NULL)
    const int64_t* x_index;          // sorted runs: sorted slot -> slot (or NULL: itself)
    const int64_t* offsets;
    const float* in_weight;
    int n, div, rows, K;
    float limit;
    bool wide;                       // out starts on 16 bytes
    bool stored;                     // gated units are made from their halves as a tensor would hold them
    bool once;                       // weights that one reading may stream past the caches
    int by_slot;                     // workgroups by slot in place of expert (of this many experts; 0: by expert)
};
// An expert every token goes through, of sizes of its own: X row t, out row t in bfloat16, the bits that the products and the activation give one by one.
// W NULL: none.  Alone it took four launches, three of them at 4 - 5 us whatever they read (16 experts of 2048 x 1408 and one more, top 4, with the router,
// 1 / 16 / 64 tokens: 42 / 77 / 85 -> 32 / 63 / 71 us; of 4096 x 2752 106 / 387 / 432 -> 91 / 369 / 409).
struct SharedArgs {
    void* out;
    const bf16_t *X, *W;
    int n, rows, K;
    bool wide, once;
};

// The four waves' partial sums (through LDS), the weight on the input, the activation, the store: slot of column c by slot_of(c).
template <int ACT, bool FOUT, int SG, class Slot>
__device__ __forceinline__ void expert_finish(const ExpertArgs& a, int r0, int count, unsigned char* rings, int w, int lane, Slot slot_of,
                                              const v4f (&acc)[XR / 16][SG]) {
    constexpr int TILES = XR / 16 * SG;
    v4f* red = (v4f*)rings;                                                        // [wave][tile][lane]
    __syncthreads();                                                               // every wave is done with its ring
#pragma unroll
    for (int r = 0; r < XR / 16; ++r)
#pragma unroll
        for (int g = 0; g < SG; ++g) red[(w * TILES + r * SG + g) * 64 + lane] = acc[r][g];
    __syncthreads();
#pragma unroll
    for (int t0 = 0; t0 < TILES; t0 += STREAM_WAVES) {
        const int t = t0 + w, r = t / SG, c = 16 * (t % SG) + (lane & 15);
        if (t < TILES && c < count) {
            v4f v = red[t * 64 + lane];
#pragma unroll
            for (int o = 1; o < STREAM_WAVES; ++o) v += red[(o * TILES + t) * 64 + lane];
            const int n0 = r0 + 16 * r + 4 * (lane >> 4);
            int64_t slot;
            float iw = 1.0f;                                                       // the expert works on weight * input
            slot_of(c, slot, iw);
            v *= iw;
            float u[4] = {v[0], v[1], v[2], v[3]};
            int m = 4, stride = a.rows, at = n0;
            if (ACT == ACT_GLU) {
                if (a.stored) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) u[q] = bf2f(f2bf(u[q]));
                }
                u[0] = glu(u[0], u[1], a.limit);
                u[1] = glu(u[2], u[3], a.limit);
                m = 2;
                stride /= 2;
                at /= 2;
            } else if (ACT == ACT_RELU_SQ) {
#pragma unroll
                for (int q = 0; q < 4; ++q) u[q] = relu_sq(u[q]);
            }
            if (FOUT) {
                float* o = (float*)a.out + (size_t)slot * stride + at;
                if (a.wide && stride % 4 == 0 && at + 4 <= stride) *(v4f*)o = v4f{u[0], u[1], u[2], u[3]};
                else
                    for (int q = 0; q < m; ++q)
                        if (at + q < stride) o[q] = u[q];
            } else {
                bf16_t* o = (bf16_t*)a.out + (size_t)slot * stride + at;
                const unsigned lo = pack_bf2(u[0], u[1]);
                if (a.wide && stride % m == 0 && at + m <= stride) {
                    if (m == 2) *(unsigned*)o = lo;
                    else *(uint2*)o = make_uint2(lo, pack_bf2(u[2], u[3]));
                } else {
                    for (int q = 0; q < m; ++q)
                        if (at + q < stride) o[q] = f2bf(u[q]);
                }
            }
        }
    }
    __syncthreads();                                                               // (the rings are free again)
}

// The work of workgroup (bx, by) of the launch's grid; lds: EXPERT_LDS bytes.
// FORM: slots by the router's indices (SLOTS_EARLY, where early_experts says so: the indices and, behind them, the first weights are requested into LDS, where no load
// into registers waits for them, and the slots are looked for while they are on their way;
// SLOTS_FEW, where few_slots says so: one group of inputs and one policy) or sorted runs.  A form holds its own code only: a launch of a
// step fetches its instructions anew, and what it jumps over costs it too (in one kernel with the others the early form gave steps of 64 sequences 0.7 % and took 0.5 from those of one; apart it gives 2.8 and takes nothing).
enum { SLOTS, SLOTS_EARLY, SORTED_RUNS, SLOTS_FEW };
template <int ACT, bool FOUT, int FORM = SLOTS>
__device__ __forceinline__ void expert_rows_block(const ExpertArgs& a, const SharedArgs& sh, int bx, int by, unsigned char* lds) {
    unsigned char* rings = lds;
    unsigned short* list = (unsigned short*)(lds + STREAM_WAVES * XRING);
    int* listed = (int*)(list + XLIST);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r0 = bx * XR;
    constexpr bool FEW = FORM == SLOTS_FEW, GENERAL = FORM == SLOTS || FEW, SHARED = FORM != SORTED_RUNS;
    if (SHARED && sh.W && by == 0) {                                                 // (first: it has the most inputs)
        if (r0 >= sh.rows) return;
        const ExpertArgs b = {sh.out, sh.X, sh.W, nullptr, nullptr, nullptr, nullptr, sh.n, 1, sh.rows, sh.K, a.limit, sh.wide, true, false, 0};
        auto chunk = [&](int c0, auto once) __attribute__((always_inline)) {
            constexpr bool ONCE = decltype(once)::value;
            const int c = min(32, sh.n - c0);
            auto rows = [&](int i) { return sh.X + (size_t)(c0 + min(i, c - 1)) * (size_t)sh.K; };
            auto slots = [&](int i, int64_t& slot, float&) { slot = c0 + i; };
            if (FEW || c <= 16) {
                v4f acc[XR / 16][1];
                stream_products<XR / 16, 1, ONCE>(sh.W + (size_t)r0 * sh.K, sh.K, min(XR, sh.rows - r0), rings + w * XRING, w, lane, rows, acc);
                expert_finish<ACT, false, 1>(b, r0, c, rings, w, lane, slots, acc);
            } else {
                v4f acc[XR / 16][2];
                stream_products<XR / 16, 2, ONCE>(sh.W + (size_t)r0 * sh.K, sh.K, min(XR, sh.rows - r0), rings + w * XRING, w, lane, rows, acc);
                expert_finish<ACT, false, 2>(b, r0, c, rings, w, lane, slots, acc);
            }
        };
        if (FEW || (sh.n <= 32 && sh.once)) return chunk(0, std::true_type());
        for (int c0 = 0; c0 < sh.n; c0 += 32) chunk(c0, std::false_type());
        return;
    }
    if (r0 >= a.rows) return;
    const int which = by - (SHARED && sh.W ? 1 : 0), rows_here = min(XR, a.rows - r0);
    int e = which;
    if (GENERAL && a.by_slot) {                                              // the expert of slot `which`, by its first slot
        e = a.idx[which];
        if ((unsigned)e >= (unsigned)a.by_slot) return;
    }
    const bf16_t* W0 = a.W + ((size_t)e * a.rows + r0) * (size_t)a.K;
    unsigned char* ring = rings + w * XRING;
    // `count` inputs: X row by row_of(i), output row (and weight) by slot_of(i); pre_: the first chunk's weights are on their way
    auto walk = [&](int count, auto pre_, auto row_of, auto slot_of) __attribute__((always_inline)) {
        auto chunk = [&](int c0, auto once, auto pre) __attribute__((always_inline)) {
            constexpr bool ONCE = decltype(once)::value, PRE = decltype(pre)::value;
            const int c = min(32, count - c0);
            auto rows = [&](int i) { return a.X + (size_t)row_of(c0 + min(i, c - 1)) * (size_t)a.K; };
            auto slots = [&](int i, int64_t& slot, float& iw) { slot_of(c0 + i, slot, iw); };
            if (FEW || c <= 16) {
                v4f acc[XR / 16][1];
                stream_products<XR / 16, 1, ONCE, PRE>(W0, a.K, rows_here, ring, w, lane, rows, acc);
                expert_finish<ACT, FOUT, 1>(a, r0, c, rings, w, lane, slots, acc);
            } else {
                v4f acc[XR / 16][2];
                stream_products<XR / 16, 2, ONCE, PRE>(W0, a.K, rows_here, ring, w, lane, rows, acc);
                expert_finish<ACT, FOUT, 2>(a, r0, c, rings, w, lane, slots, acc);
            }
        };
        if (count <= 0) {
            if (decltype(pre_)::value) wait_vm<0>();                               // (the workgroup's LDS is another's once it ends)
            return;
        }
        if (FEW || (count <= 32 && a.once)) return chunk(0, std::true_type(), pre_);
        int c0 = 0;
        if constexpr (decltype(pre_)::value) {
            chunk(0, std::false_type(), pre_);
            c0 = 32;
        }
        for (; c0 < count; c0 += 32) chunk(c0, std::false_type(), std::false_type());
    };
    if constexpr (FORM == SORTED_RUNS) {
        const int64_t s0 = a.offsets[e];
        walk((int)(a.offsets[e + 1] - s0), std::false_type(),
             [&](int i) {
                 const int64_t s = s0 + i;
                 return a.x_index ? a.x_index[s] / a.div : s;
             },
             [&](int i, int64_t& slot, float& iw) {
                 slot = s0 + i;
                 if (a.in_weight) iw = a.in_weight[a.x_index ? a.x_index[slot] : slot];
             });
        return;
    }
    constexpr bool EARLY_W = FORM == SLOTS_EARLY;
    constexpr int PIECES = FEW ? 1 : XLIST / EXPERT_THREADS;
    const int* held = (const int*)(ring + XRING - 2048);                           // (an input's place: not requested before the search is done)
    if constexpr (EARLY_W) {
        const int span = (a.n + EXPERT_THREADS - 1) / EXPERT_THREADS * 64;
        const unsigned dst = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)held);
        wait_vm<0>();
#pragma unroll
        for (int q = 0; q < PIECES; ++q)
            if (64 * q < span) lds_copy4(dst + 256 * q, a.idx + min(w * span + 64 * q + lane, a.n - 1));
        if (a.once) request_early<XR / 16, true>(W0, a.K, rows_here, ring, w, lane);
        else request_early<XR / 16, false>(W0, a.K, rows_here, ring, w, lane);
        wait_vm<EARLY * 2 * (XR / 16)>();
    }
    for (int n0 = 0; n0 < a.n; n0 += XLIST) {                                      // (EARLY_W, FEW: once)
        // this expert's slots among the next XLIST, in order: wave w looks at a quarter of them
        const int len = min(XLIST, a.n - n0), span = (len + EXPERT_THREADS - 1) / EXPERT_THREADS * 64;
        int found = 0;
        unsigned long long hit[PIECES];
        if constexpr (EARLY_W) {
#pragma unroll
            for (int q = 0; q < PIECES; ++q) hit[q] = __ballot(64 * q < span && w * span + 64 * q + lane < len && held[64 * q + lane] == e);
        } else {
#pragma unroll
            for (int q = 0; q < PIECES; ++q) {
                const int i = w * span + 64 * q + lane;
                hit[q] = __ballot(64 * q < span && i < len && a.idx[n0 + i] == e);
            }
        }
#pragma unroll
        for (int q = 0; q < PIECES; ++q) found += __popcll(hit[q]);
        if (lane == 0) listed[w] = found;
        if constexpr (EARLY_W) barrier_in_flight();
        else __syncthreads();
        int at = 0, count = 0;
#pragma unroll
        for (int o = 0; o < STREAM_WAVES; ++o) {
            at += o < w ? listed[o] : 0;
            count += listed[o];
        }
#pragma unroll
        for (int q = 0; q < PIECES; ++q) {
            if (hit[q] >> lane & 1) list[at + __popcll(hit[q] & ((1ull << lane) - 1))] = (unsigned short)(w * span + 64 * q + lane);
            at += __popcll(hit[q]);
        }
        if constexpr (EARLY_W) barrier_in_flight();
        else __syncthreads();
        if (GENERAL && a.by_slot && list[0] != which) return;                     // (an earlier slot's workgroups do this expert)
        auto row_of = [&](int i) { return (int64_t)((n0 + list[i]) / a.div); };
        auto slot_of = [&](int i, int64_t& slot, float& iw) {
            slot = n0 + list[i];
            if (a.in_weight) iw = a.in_weight[slot];
        };
        walk(count, std::integral_constant<bool, EARLY_W>(), row_of, slot_of);
        if constexpr (EARLY_W || FEW) return;
        __syncthreads();
    }
}

// Whether the weights are requested before the slots are looked for, of a launch that plan_expert_rows has passed.  Measured, 16 experts, 16 / 24 slots each, out of memory, us: 1024 x
// 2048 16.7 -> 15.4, 17.7 -> 16.7, 1408 x 2048 21.6 -> 19.9, 23.1 -> 21.6, 2048 x 1408 19.4 -> 18.1, 21.3 -> 20.1, 2816 x 2048 37.9 -> 35.7, 40.1 -> 38.2, 5632 x 2048 69.3 -> 67.8,
// 73.8 -> 72.7; steps of 32 and 64 sequences (Vekalorn, 20 and their prompts) 9202 -> 8924, 10741 -> 10446.  The first requests of an expert that no slot has are for nothing (a
// quarter of its weights): steps of 4 tokens, top 4 of 16, took 4 % longer, so four slots an expert on average, of which one expert in 50 has none.
inline bool early_experts(const ExpertArgs& a, int n_experts) {
    return a.idx && !a.by_slot && a.n <= XLIST && a.n >= 4 * n_experts && a.K >= EARLY_MIN;
}
// Whether one group of inputs and the weights' one reading are all that a launch has: steps of 4 sequences 6600 -> 6440 us (Rivolix, 20 of them and their prompts), 8420 -> 8260
// (Mumelix), 7270 -> 7100 (Vekalorn), of two 6460 -> 6350
inline bool few_slots(const ExpertArgs& a, const SharedArgs& sh) { return a.idx && a.n <= 16 && a.once && (!sh.W || (sh.n <= 16 && sh.once)); }
// Checks of a launch (a, sh as its caller filled them in), what it derives from them, and its grid; act: clamped units become ACT_GLU.
inline int plan_expert_rows(const char* what, ExpertArgs& a, SharedArgs& sh, int n_experts, int& act, bool kept, dim3& grid) {
    QSV_REQUIRE(a.out && a.X && a.W && n_experts > 0 && a.rows > 0 && a.div > 0, "%s: bad arguments", what);
    QSV_REQUIRE(act == ACT_NONE || act == ACT_RELU_SQ || ((act == ACT_GLU || act == QSV_ACT_CLAMPED_GLU) && a.rows % 2 == 0), "%s: activation %d", what,
                act);
    QSV_REQUIRE(act != QSV_ACT_CLAMPED_GLU || a.limit > 0.f, "%s: clamped units need a positive limit", what);
    if (act == QSV_ACT_CLAMPED_GLU) act = ACT_GLU;
    else a.limit = 0.f;
    // (a workgroup's rows within 32-bit byte offsets)
    QSV_REQUIRE(a.K > 0 && a.K % 8 == 0 && a.K <= 1 << 25, "%s: inner width %d (a multiple of 8, at most 2^25)", what, a.K);
    QSV_REQUIRE(n_experts <= 65535, "%s: too many experts", what);
    QSV_REQUIRE(((uintptr_t)a.X | (uintptr_t)a.W) % 16 == 0, "%s: inputs and weights start on 16 bytes", what);
    a.wide = (uintptr_t)a.out % 16 == 0;
    a.once = !kept && streams_once(a.W, (int64_t)n_experts * a.rows, a.K);
    sh.once = !kept && streams_once(sh.W, sh.rows, sh.K);
    // Few slots: workgroups by slot, so that those of experts without one are not there.  Measured for both products of a token, us before and after: 1 token of 4 of
    // 16 experts of 2048 x 1408 gated with a shared one 24.2 -> 20.3 (1496 and 1088 workgroups, of which 440 and 320 have rows), 2 tokens 29.2 -> 27.5, 1 token of
    // 8 of 64 of 2048 x 768 35.0 -> 21.1.  The line: slots past half of the experts gain little and lose up to 4 % (3 tokens of the first: 37.3 -> 38.8, the empty
    // workgroups between the others' are then few), and a grid that fits the chip at once loses .2 us to the load of the slot's expert.
    const int tiles = ((sh.W && sh.rows > a.rows ? sh.rows : a.rows) + XR - 1) / XR;
    a.by_slot = a.idx && a.n <= XLIST && 2 * a.n <= n_experts && (int64_t)n_experts * tiles > 512 ? n_experts : 0;
    grid = dim3(tiles, (a.by_slot ? a.n : n_experts) + (sh.W ? 1 : 0));
    return QSV_OK;
}
// The checks in front of plan_expert_rows for experts by the router's indices
inline int expert_slots_args(const char* what, const qsv_expert_job& j, ExpertArgs& a, SharedArgs& sh) {
    QSV_REQUIRE(j.idx && j.n >= 0 && (!j.float_out || j.act == ACT_NONE), "%s: bad arguments", what);
    if (j.sh_W) {
        QSV_REQUIRE(j.n_experts < 65535 && j.sh_out && j.sh_X && j.sh_n > 0 && j.sh_rows > 0, "%s: bad arguments", what);
        QSV_REQUIRE(j.sh_K > 0 && j.sh_K % 8 == 0 && j.sh_K <= 1 << 25 && ((uintptr_t)j.sh_X | (uintptr_t)j.sh_W) % 16 == 0, "%s: inner width %d, rows on 16 bytes", what,
                    j.sh_K);
        QSV_REQUIRE(j.act == ACT_NONE || j.act == ACT_RELU_SQ || j.sh_rows % 2 == 0, "%s: %d rows of gated units", what, j.sh_rows);
        sh = {j.sh_out, (const bf16_t*)j.sh_X, (const bf16_t*)j.sh_W, j.sh_n, j.sh_rows, j.sh_K, (uintptr_t)j.sh_out % 16 == 0, false};
    } else {
        sh = {};
    }
    a = {j.out, (const bf16_t*)j.X, (const bf16_t*)j.W, j.idx, nullptr, nullptr, j.in_weight, j.n, j.div, j.rows, j.K, j.limit, false, false, false, 0};
    return QSV_OK;
}
}  // namespace
