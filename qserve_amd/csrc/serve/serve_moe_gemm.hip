// serve_moe_gemm.hip -- grouped expert products on the bf16 matrix cores for the prompt phase (many tokens per expert): the slots sorted
// by expert on the device, out[s, n] = act(W[e][n, :] . x(s)).
//
// Both operands are contiguous along the reduction, so with the weight rows as the A operand and the slots' inputs as the B operand
// (v_mfma_f32_16x16x32_bf16) a lane ends up with 4 consecutive n of one slot - an 8-byte store.  The input row of a slot is fetched
// through an index (the gather into sorted order is part of the copy), relu(.)^2 or the gated unit (gate and up rows interleaved in
// the weight: rows 2f and 2f + 1 are neighbours, so a lane's four rows are two whole units) is the epilogue of the first product.
#include "serve_common.h"

#include <type_traits>

namespace {
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

constexpr int KS = 64;       // reduction elements per step

__device__ __forceinline__ unsigned pack_bf2(float a, float b) { return (unsigned)f2bf(a) | ((unsigned)f2bf(b) << 16); }

// Tiles of 256 weight rows x 256 slots (128 or 64 where an expert has no more left).  Bound by the matrix cores.  Eight waves (64 rows x 128
// slots each, two per SIMD) multiply while the next K step of 64 is copied straight into the other half of a 128 KiB LDS buffer
// (global_load_lds, one 128-byte line per row; pieces permuted by the row's number: 16-byte reads without bank conflicts); one barrier
// per step.  Workgroups are persistent (one per CU): each finds its tiles from the experts' offsets - no tile list, no count reaches
// the host -, an XCD's workgroups walk neighbouring tiles (shared weight and input panels in its L2), and the last step of a tile copies the
// first one of the next, so the epilogue's stores have something to hide behind.  A tile with few slots gives each wave fewer columns
// instead of multiplying padding, and no copies of inputs it does not have; an XCD cuts the tiles of its last, part-empty round by slots into
// halves where at most half of its 32 workgroups have one, into quarters where at most a quarter have: with more than half nothing is cut, and
// fewer than eight tiles leave workgroups idle.  The XCDs' shares are ceil(tiles / 8) each, so the last of them can be short or empty.
// Measured (MI355X, both products with sort and combine): 8192 tokens, 4 of 16 experts of 2048 x 1408: 1010 us (the form before: 256 x 128 tiles staged
// through registers, tile list from the host, torch's sort) -> 485 -> 463 (with the cut of the last round, in turn; 815 TFLOP/s), gated
// 647 -> 620 us (915), 600 tokens 121 -> 106 us; 32 gated experts of 4096 x 2752: 3.5 ms -> 2547 -> 2494 us (888).
constexpr int PR = 256, PS = 256, PWAVES = 8, PT = 64 * PWAVES;
constexpr int PBUF = (PR + PS) * 128;               // bytes of one K step
constexpr int MAX_K = 1 << 23;                      // (a tile's weight rows within 32-bit byte offsets)
constexpr int LISTED_SLOTS = 128;                   // slots of a tile in a caller's list, at most
constexpr int MAX_GROUPS = 8064;                   // (what is left of 160 KiB of LDS holds a count for each)

typedef __attribute__((address_space(3))) void* lds_ptr;
__device__ __forceinline__ void lds_copy16(unsigned dst, const void* base, unsigned off) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst) : "memory");
}
__device__ __forceinline__ void lds_copy16(unsigned dst, const void* from) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(dst) : "memory");
}

struct GroupedArgs {
    bf16_t* out;
    const bf16_t* X;
    const bf16_t* W;
    const int32_t* order;            // sorted slot -> slot (NULL: itself); the input row is slot / div
    const int32_t* offsets;          // [E + 1] first sorted slot of every expert
    const float* in_weight;
    int div, E, N, K;
    float limit;
    // the caller's own tiles in place of offsets (LISTED): [n_tiles][3] expert, first sorted slot, slots; x_index for order
    const int32_t* tiles;
    const int64_t* x_index;
    int n_tiles;
};
struct GroupedTile {
    int e, n0, first, ns;            // expert, first weight row, first sorted slot, slots
};

template <int ACT, bool LISTED, int NTS>
__device__ __forceinline__ void grouped_store(const GroupedArgs& a, const GroupedTile& t, int n_wave, int s_wave, int lane, const v4f (&acc)[4][NTS]) {
    const int col = lane & 15, g4 = lane >> 4;
#pragma unroll
    for (int nt = 0; nt < NTS; ++nt) {
        const int sl = s_wave + 16 * nt + col;
        if (sl >= t.ns) continue;
        float iw = 1.0f;                                            // the expert works on iw * input
        if (a.in_weight) iw = a.in_weight[LISTED ? (a.x_index ? a.x_index[t.first + sl] : t.first + sl) : (a.order ? a.order[t.first + sl] : t.first + sl)];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const int n = t.n0 + n_wave + 16 * mt + 4 * g4;
            if (n >= a.N) continue;                                 // N % 4 == 0: the four rows are inside together
            v4f v = acc[mt][nt] * iw;
            if (ACT == 2) {
                float u0, u1;
                if (a.limit > 0.f) {                                // clamped units: g sigmoid(1.702 g) (u + 1) (uniform over the launch)
                    const float ga = fminf(v[0], a.limit), gb = fminf(v[2], a.limit);
                    u0 = ga / (1.0f + expf(-1.702f * ga)) * (fminf(fmaxf(v[1], -a.limit), a.limit) + 1.0f);
                    u1 = gb / (1.0f + expf(-1.702f * gb)) * (fminf(fmaxf(v[3], -a.limit), a.limit) + 1.0f);
                } else {
                    u0 = v[0] / (1.0f + expf(-v[0])) * v[1];
                    u1 = v[2] / (1.0f + expf(-v[2])) * v[3];
                }
                *(unsigned*)(a.out + (size_t)(t.first + sl) * (a.N / 2) + n / 2) = pack_bf2(u0, u1);
                continue;
            }
            if (ACT == 1) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float x = fmaxf(v[r], 0.f);
                    v[r] = x * x;
                }
            }
            const v2u pk = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
            *(v2u*)(a.out + (size_t)(t.first + sl) * a.N + n) = pk;
        }
    }
}

template <int ACT, bool LISTED>
__global__ __launch_bounds__(PT, 2) void grouped_gemm_persistent_kernel(GroupedArgs a) {
    __shared__ __attribute__((aligned(128))) unsigned char buf[2 * PBUF];
    __shared__ int tiles_before[MAX_GROUPS + 1];                    // slot tiles of the experts before e
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (!LISTED && w == 0) {
        int carry = 0;
        for (int e0 = 0; e0 < a.E; e0 += 64) {
            const int e = e0 + lane;
            int x = e < a.E ? (a.offsets[e + 1] - a.offsets[e] + PS - 1) / PS : 0;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(x, o, 64);
                if (lane >= o) x += y;
            }
            if (e < a.E) tiles_before[e + 1] = carry + x;
            carry += __shfl(x, 63, 64);
        }
        if (lane == 0) tiles_before[0] = 0;
    }
    __syncthreads();
    const int row_tiles = (a.N + PR - 1) / PR, total = (LISTED ? a.n_tiles : __builtin_amdgcn_readfirstlane(tiles_before[a.E])) * row_tiles;
    // An XCD's share of the tiles: whole rounds of its workgroups, then what is left - fewer tiles than workgroups - cut by slots into as many
    // parts (two or four) as there are workgroups for.  Place p: tile (p) of the share, or a part of one.
    const int xcd = blockIdx.x & 7, per_xcd = gridDim.x >> 3, chunk = (total + 7) >> 3;
    const int begin = xcd * chunk, here = max(0, min(chunk, total - begin));
    const int whole = here / per_xcd * per_xcd, rest = here - whole, cut = LISTED ? 0 : rest * 4 <= per_xcd ? 2 : rest * 2 <= per_xcd ? 1 : 0;   // log2 of the parts
    const int last = whole + (rest << cut);
    int at = blockIdx.x >> 3;
    if (at >= last) return;

    auto tile_at = [&](int place) __attribute__((always_inline)) {
        const int over = place - whole, part = over >= 0 ? over & ((1 << cut) - 1) : 0, size = over >= 0 ? PS >> cut : PS;
        const int L = begin + (over >= 0 ? whole + (over >> cut) : place), s = L / row_tiles;   // which slot tile
        GroupedTile t;
        t.n0 = (L % row_tiles) * PR;
        if (LISTED) {
            t.e = __builtin_amdgcn_readfirstlane(a.tiles[3 * s]);
            t.first = __builtin_amdgcn_readfirstlane(a.tiles[3 * s + 1]);
            t.ns = __builtin_amdgcn_readfirstlane(min(max(a.tiles[3 * s + 2], 0), LISTED_SLOTS));
            return t;
        }
        int lo = 0, hi = a.E;                                       // tiles_before[lo] <= s < tiles_before[hi]
        while (hi - lo > 1) {
            const int m = (lo + hi) >> 1;
            if (__builtin_amdgcn_readfirstlane(tiles_before[m]) <= s) lo = m;
            else hi = m;
        }
        const int skip = __builtin_amdgcn_readfirstlane(tiles_before[lo]), first = a.offsets[lo] + (s - skip) * PS + part * size;
        t.e = lo;
        t.first = __builtin_amdgcn_readfirstlane(first);
        t.ns = __builtin_amdgcn_readfirstlane(min(size, a.offsets[lo + 1] - first));   // (none or less: a part behind the expert's last slot)
        return t;
    };
    // copies: wave w brings rows 32 w .. 32 w + 31 of the weights and of the inputs, eight rows (of 128 bytes) per instruction
    const int piece = ((lane & 7) ^ (lane >> 3)) * 16;
    auto x_slot = [&](const GroupedTile& t, int j) __attribute__((always_inline)) {
        if (LISTED && t.ns <= 0) return 0;                          // (an empty tile of the list: nothing is read or stored)
        const int s = t.first + min(32 * w + 8 * j + (lane >> 3), t.ns - 1);
        if (LISTED) return a.x_index ? (int)a.x_index[s] : s;
        return a.order ? a.order[s] : s;
    };
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)buf) + (unsigned)w * 4096u;
    GroupedTile t = tile_at(at);
    if (!LISTED && t.ns <= 0) return;                                        // (parts are the last places: nothing follows)
    const bf16_t* W0 = a.W + ((size_t)t.e * a.N + t.n0) * (size_t)a.K;
    unsigned woff[4];
    const unsigned char* xrow[4];
    int rows_here = 0;                                              // inputs of the tile that is being copied, from this wave's first on
    auto point = [&](const GroupedTile& g, const int (&slot)[4]) __attribute__((always_inline)) {
        W0 = a.W + ((size_t)g.e * a.N + g.n0) * (size_t)a.K;
        rows_here = g.ns - 32 * w;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            woff[j] = (unsigned)min(32 * w + 8 * j + (lane >> 3), a.N - 1 - g.n0) * (unsigned)a.K * 2u + piece;
            xrow[j] = (const unsigned char*)(a.X + (size_t)(slot[j] / a.div) * (size_t)a.K) + piece;
        }
    };
    auto copy = [&](int j, int which, int k0) __attribute__((always_inline)) {   // one of the wave's eight copies of a step
        if (j < 4) lds_copy16(lds0 + which * PBUF + 1024 * j, W0 + k0, woff[j]);
        else if (8 * (j - 4) < rows_here) lds_copy16(lds0 + which * PBUF + PR * 128 + 1024 * (j - 4), xrow[j - 4] + (size_t)k0 * 2);
    };
    {
        int slot[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) slot[j] = x_slot(t, j);
        point(t, slot);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) copy(j, 0, 0);
    const int col = lane & 15, g4 = lane >> 4, wr = w & 3, ws = w >> 2;
    const int steps = a.K / KS;
    int which = 0;

    auto run_tile = [&](auto nts) __attribute__((always_inline)) {
        constexpr int NTS = decltype(nts)::value;
        const int next = at + per_xcd;
        const GroupedTile u = next < last ? tile_at(next) : t;
        const bool more = next < last && (LISTED || u.ns > 0);
        int slot[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) slot[j] = x_slot(more ? u : t, j);
        v4f acc[4][NTS];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
            for (int nt = 0; nt < NTS; ++nt) acc[mt][nt] = v4f{0.f, 0.f, 0.f, 0.f};
        const int s_wave = ws * 16 * NTS;
        for (int i = 0; i < steps; ++i) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();                           // this step has landed; the other half has been read by everyone
            asm volatile("" ::: "memory");
            const unsigned char* A = buf + which * PBUF + (64 * wr + col) * 128;
            const unsigned char* B = buf + which * PBUF + (PR + s_wave + col) * 128;
            const int p0 = (g4 ^ (col & 7)) << 4, p1 = ((4 + g4) ^ (col & 7)) << 4;
            int k_next = (i + 1) * KS;
            bool bring = true;
            if (i + 1 == steps) {                                   // the next tile's first step
                k_next = 0;
                bring = more;
                if (more) point(u, slot);
            }
            which ^= 1;
            // 2 NTS groups of four products; group g's inputs are requested three groups ahead, the weights' second half and the copies
            // of the next step in between (the order is the source's: left alone, the compiler reads each operand just before its use)
            v4u av[2][4], bv[4];
            auto read_b = [&](int g) __attribute__((always_inline)) { bv[g & 3] = *(const v4u*)(B + 2048 * (g % NTS) + (g < NTS ? p0 : p1)); };
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) av[0][mt] = *(const v4u*)(A + 2048 * mt + p0);
            read_b(0), read_b(1), read_b(2);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < 2 * NTS; ++g) {
                if (g + 3 < 2 * NTS) read_b(g + 3);
#pragma unroll
                for (int mt = 0; mt < 4; ++mt)
                    if (mt * NTS / 4 == g) av[1][mt] = *(const v4u*)(A + 2048 * mt + p1);
                if (bring) {
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (j * (NTS < 4 ? 2 * NTS : 8) / 8 == g) copy(j, which, k_next);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int mt = 0; mt < 4; ++mt)
                    acc[mt][g % NTS] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, av[g / NTS][mt]), __builtin_bit_cast(bf8, bv[g & 3]),
                                                                               acc[mt][g % NTS], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        grouped_store<ACT, LISTED, NTS>(a, t, 64 * wr, s_wave, lane, acc);
        asm volatile("" ::: "memory");                              // (the stores' branches join here: what follows stays uniform)
        if (more) t = u;
        at = next;
        return more;
    };
    for (;;) {
        const bool more = t.ns > PS / 2   ? run_tile(std::integral_constant<int, 8>())
                          : t.ns > PS / 4 ? run_tile(std::integral_constant<int, 4>())
                                          : run_tile(std::integral_constant<int, 2>());
        if (!more) break;
    }
}

// ---- slots sorted by expert, in order --------------------------------------------------------------------------------------------------
// Workgroup e gathers the slots of expert e: every wave counts its share of the indices (those of smaller experts give the first place, its
// own the place within), then writes them.  Indices from E on and below 0 are left out.
constexpr int ST = 1024;
__global__ __launch_bounds__(ST) void sort_slots_kernel(int32_t* __restrict__ order, int32_t* __restrict__ place, int32_t* __restrict__ offsets,
                                                        const int32_t* __restrict__ idx, int n, int E) {
    __shared__ int same_w[ST / 64], less_w[ST / 64];
    const int e = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int per = ((n + ST - 1) / ST) * 64, i0 = min(n, w * per), i1 = min(n, i0 + per);   // wave w looks at indices [i0, i1)
    constexpr int Q = 16;
    int same = 0, less = 0;
    for (int i = i0; i < i1; i += 64 * Q) {
        int v[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) v[q] = i + 64 * q + lane < i1 ? idx[i + 64 * q + lane] : 0x7fffffff;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            same += __popcll(__ballot(v[q] == e));
            less += __popcll(__ballot((unsigned)v[q] < (unsigned)e));   // (below 0: no expert, left out)
        }
    }
    if (lane == 0) {
        same_w[w] = same;
        less_w[w] = less;
    }
    __syncthreads();
    int at = 0, all = 0;
#pragma unroll
    for (int o = 0; o < ST / 64; ++o) {
        at += less_w[o] + (o < w ? same_w[o] : 0);
        all += less_w[o] + same_w[o];
    }
    if (threadIdx.x == 0) {
        if (e == 0) offsets[0] = 0;
        offsets[e + 1] = all;
    }
    if (same == 0) return;
    for (int i = i0; i < i1; i += 64 * Q) {
        int v[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) v[q] = i + 64 * q + lane < i1 ? idx[i + 64 * q + lane] : 0x7fffffff;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const unsigned long long hit = __ballot(v[q] == e);
            if (v[q] == e) {
                const int s = at + __popcll(hit & ((1ull << lane) - 1));
                order[s] = i + 64 * q + lane;
                place[i + 64 * q + lane] = s;
            }
            at += __popcll(hit);
        }
    }
}
}  // namespace

extern "C" int qsv_moe_sort(int32_t* order, int32_t* place, int32_t* offsets, const int32_t* idx, int n, int n_experts, void* stream) {
    QSV_REQUIRE(order && place && offsets && idx && n > 0 && n_experts > 0, "qsv_moe_sort: bad arguments");
    hipLaunchKernelGGL(sort_slots_kernel, dim3(n_experts), dim3(ST), 0, (hipStream_t)stream, order, place, offsets, idx, n, n_experts);
    return qsv_launch_status("qsv_moe_sort");
}
template <bool LISTED>
static int launch_grouped(const char* what, GroupedArgs a, int act, void* stream) {
    QSV_REQUIRE(act == QSV_ACT_NONE || act == QSV_ACT_RELU_SQ || act == QSV_ACT_GLU || (act == QSV_ACT_CLAMPED_GLU && a.limit > 0.f),
                "%s: activation %d (limit %g)", what, act, (double)a.limit);
    QSV_REQUIRE(((uintptr_t)a.X | (uintptr_t)a.W) % 16 == 0 && (uintptr_t)a.out % 8 == 0, "%s: inputs and weights start on 16 bytes", what);
    if (act == QSV_ACT_CLAMPED_GLU) act = QSV_ACT_GLU;
    else a.limit = 0.f;
    const dim3 grid(256), block(PT);                                // one workgroup per CU, 32 per XCD
    if (act == QSV_ACT_RELU_SQ) hipLaunchKernelGGL((grouped_gemm_persistent_kernel<1, LISTED>), grid, block, 0, (hipStream_t)stream, a);
    else if (act == QSV_ACT_GLU) hipLaunchKernelGGL((grouped_gemm_persistent_kernel<2, LISTED>), grid, block, 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL((grouped_gemm_persistent_kernel<0, LISTED>), grid, block, 0, (hipStream_t)stream, a);
    return qsv_launch_status(what);
}
extern "C" int qsv_grouped_gemm_sorted_ok(int n_experts, int N, int K) { return n_experts > 0 && n_experts <= MAX_GROUPS && N > 0 && N % 4 == 0 && K > 0 && K % KS == 0 && K <= MAX_K; }
extern "C" int qsv_grouped_gemm_sorted(void* out, const void* X, const int32_t* order, int div, const void* W, const int32_t* offsets, int n_experts,
                                       int N, int K, int act, float limit, const float* in_weight, void* stream) {
    QSV_REQUIRE(out && X && W && offsets && div > 0, "qsv_grouped_gemm_sorted: bad arguments");
    QSV_REQUIRE(qsv_grouped_gemm_sorted_ok(n_experts, N, K), "qsv_grouped_gemm_sorted: %d experts (at most %d), N %d (a multiple of 4), K %d (a multiple of %d, at most %d)",
                n_experts, MAX_GROUPS, N, K, KS, MAX_K);
    return launch_grouped<false>("qsv_grouped_gemm_sorted", {(bf16_t*)out, (const bf16_t*)X, (const bf16_t*)W, order, offsets, in_weight, div, n_experts, N, K,
                                                             limit, nullptr, nullptr, 0}, act, stream);
}
// The same over the caller's own tiles.
extern "C" int qsv_grouped_gemm_tile_slots(void) { return LISTED_SLOTS; }
extern "C" int qsv_grouped_gemm_k_step(void) { return KS; }
extern "C" int qsv_grouped_gemm(void* out, const void* X, const int64_t* x_index, int div, const void* W, const int32_t* tiles, int n_tiles, int N, int K,
                                int act, float limit, const float* in_weight, void* stream) {
    QSV_REQUIRE(out && X && W && tiles && div > 0 && n_tiles >= 0, "qsv_grouped_gemm: bad arguments");
    QSV_REQUIRE(N > 0 && N % 4 == 0 && K > 0 && K % KS == 0 && K <= MAX_K, "qsv_grouped_gemm: N %d (a multiple of 4), K %d (a multiple of %d, at most %d)", N,
                K, KS, MAX_K);
    QSV_REQUIRE(n_tiles <= 65535, "qsv_grouped_gemm: %d tiles (at most 65535 per launch)", n_tiles);
    QSV_REQUIRE((int64_t)n_tiles * ((N + PR - 1) / PR) < (1ll << 30), "qsv_grouped_gemm: %d tiles of %d rows", n_tiles, N);
    if (n_tiles == 0) return QSV_OK;
    return launch_grouped<true>("qsv_grouped_gemm", {(bf16_t*)out, (const bf16_t*)X, (const bf16_t*)W, nullptr, nullptr, in_weight, x_index ? div : 1, 0, N, K,
                                                     limit, tiles, x_index, n_tiles}, act, stream);
}
