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


// Tiles of 256 weight rows x 256 slots (128 or 64 where an expert has no more left).  Bound by the matrix cores.
//
// Eight waves, two per SIMD: waves 0 - 3 and 4 - 7 are half a phase apart, so that one of a SIMD's two always multiplies while the other reads its next
// operands.  A K step of 64 has two phases, one per half of the tile's rows; in each a wave has 64 rows x 64 slots: 32 instructions.  The first reads a weight half
// and both input halves (16 reads of 16 bytes a lane), the second the other weight half (8).  What every wave has read is requested anew for the step after
// the next (global_load_lds, whole 128-byte lines of a row; pieces permuted by the row's number: 16-byte reads without bank conflicts), and a phase waits
// for what the next one reads, which was requested three phases before: 64 - 112 KiB in flight a CU, no wait for the youngest requests.  Every wave issues the
// same requests in every phase - of rows that a tile does not have with one lane active - so that the counted waits hold whatever the tile's size.
//
// Workgroups are persistent (one per CU): each finds its tiles from the experts' offsets - no tile list, no count reaches the host -, the last
// two steps of a tile request the first two of the next one, so the epilogue's stores have something to hide behind.  An XCD's workgroups walk
// bands of 8 row tiles and through an expert's slots inside a band: 8 weight and 4 input panels are in its L2 at a time, where rows first meant 22
// and 2.  A tile with few slots multiplies and requests those only; an XCD cuts the tiles of its last, part-empty round by slots into
// halves where at most half of its 32 workgroups have one, into quarters where at most a quarter have: with more than half nothing is cut, and
// fewer than eight tiles leave workgroups idle.  The XCDs' shares are ceil(tiles / 8) each, so the last of them can be short or empty.
//
// Measured (MI355X, one product out of memory, us, the form before -> now in one call; before: four phases of a quarter each, conditions in every step): 32768 slots of one
// expert of 4096 x 4096 835 -> 745 (1480 TFLOP/s; hipBLASLt's dense product of that size 700), 890 slots for each of 32 experts of 5504 x 4096 1200 -> 1114 (1155),
// 2048 of 16 of 1408 x 2048 171 -> 159, of 2048 x 1408 172 -> 164, 550 of 16 of 2816 x 2048 138 -> 124, 512 107 -> 101, 300 94 -> 84; of 64 - 128 slots the same (the weights out
// of memory).  12 000 random shapes: in median 1.10 times as fast, gated 1.08; slower where few tiles wait for long reductions (up to 64 tiles and more than 3500 elements, by up to
// 13 %; experts of up to 128 rows and more than 2500, 22 %: less is in flight).  The card's power bounds it: it holds 1.5 GHz over random numbers and 2.1 over ones (745 -> 620 us).  What counts there is cycles, not bytes: the branches
// that a step held for the first and the last ones alone took 8 % (they are the forms with EDGE now), halving the barriers 2 %; operands that never miss L2
// give 4 %, requests and reads left out altogether 18 and 8 %.  Eight waves without the half phase between them 785, four waves of 128 x 128 970 (one wave a SIMD has nothing
// beside its own barriers and requests); tiles of 192 rows cost 0.89 of 256 (a step's time is its requests and reads as much as its products); another order of the
// matrix instructions, a raised priority and requests without masks: no difference.
// Small layers, both products with sort and sum, weights out of memory / left in the caches by the call before: 4 gated of 2048 x 1408, 1024 slots 75 / 75 us, 8 of
// them, 1200 83 / 81, 8 of 1024 x 512 46 / 45, 4 of 512 x 2048 57 / 56 (before this set of forms).
constexpr int PR = 256, PS = 256, PWAVES = 8, PT = 64 * PWAVES;
constexpr int PBUF = (PR + PS) * 128;               // bytes of one K step
constexpr int HALF = 128 * 128;                     // of an operand half of it
constexpr int BAND = 8;                             // row tiles of a band
constexpr int MAX_K = 1 << 23;                      // (a tile's weight rows within 32-bit byte offsets)
constexpr int LISTED_SLOTS = 128;                   // slots of a tile in a caller's list, at most
constexpr int SIDE = (160 * 1024 - 2 * PBUF) / 4;   // what is left of LDS, in words: a count for each expert,
constexpr int AHEAD = SIDE - PWAVES * 64;           // and where they leave room the next tile's input rows
constexpr int MAX_GROUPS = 8064;

typedef __attribute__((address_space(3))) void* lds_ptr;
// A request into LDS by all lanes (left < 0: 1 KiB) or by the first one alone, for the counted waits' sake: an instruction without a lane need not count.
__device__ __forceinline__ void lds_copy16(unsigned dst, const void* base, unsigned off, int left) {
    asm volatile("s_mov_b32 m0, %2\n\ts_ashr_i32 exec_hi, %3, 31\n\ts_or_b32 exec_lo, exec_hi, 1\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(base), "s"(dst), "s"(left) : "memory", "scc");
}
__device__ __forceinline__ void lds_copy16(unsigned dst, const void* from, int left) {
    asm volatile("s_mov_b32 m0, %1\n\ts_ashr_i32 exec_hi, %2, 31\n\ts_or_b32 exec_lo, exec_hi, 1\n\tglobal_load_lds_dwordx4 %0, off\n\ts_mov_b64 exec, -1" ::"v"(from), "s"(dst), "s"(left) : "memory", "scc");
}
__device__ __forceinline__ void lds_copy4(unsigned dst, const void* from) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(from), "s"(dst) : "memory");
}
// two neighbouring words through the scalar path: the wave's requests in flight are not waited for
__device__ __forceinline__ int2 scalar_pair(const int32_t* p) {
    unsigned long long v;
    asm volatile("s_load_dwordx2 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(p) : "memory");
    return make_int2((int)v, (int)(v >> 32));
}
__device__ __forceinline__ int scalar_word(const int32_t* p) {
    int v;
    asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(p) : "memory");
    return v;
}
template <int N>
__device__ __forceinline__ void wait_copies() {     // all but the wave's N youngest, and every read of LDS
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void step_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
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

// v[0 .. 3] of one slot's neighbouring rows -> what is stored of them: two words, for gated units the lower one
template <int ACT>
__device__ __forceinline__ v2u grouped_result(v4f v, float limit) {
    if (ACT == 2) {
        // (the arithmetic of the steps' kernel and of the activation by itself, bit for bit.  It is 4.2 us of vector work a tile, three steps of its loop: with the hardware's
        // exp2 and reciprocal 512 slots for each of 16 experts gated 2816 x 2048 take 97 us in place of 104 and 890 for each of 32 of 5504 x 4096 1133 in place of 1157, but
        // exp2 of a rounded product loses a bit for every doubling of |x|, the reciprocal is 0 for gates below -87.3, and a prompt's units differ from a step's)
        float u0, u1;
        if (limit > 0.f) {                                          // clamped units: g sigmoid(1.702 g) (u + 1) (uniform over the launch)
            const float ga = fminf(v[0], limit), gb = fminf(v[2], limit);
            u0 = ga / (1.0f + expf(-1.702f * ga)) * (fminf(fmaxf(v[1], -limit), limit) + 1.0f);
            u1 = gb / (1.0f + expf(-1.702f * gb)) * (fminf(fmaxf(v[3], -limit), limit) + 1.0f);
        } else {
            u0 = v[0] / (1.0f + expf(-v[0])) * v[1];
            u1 = v[2] / (1.0f + expf(-v[2])) * v[3];
        }
        return v2u{pack_bf2(u0, u1), 0u};
    }
    if (ACT == 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float x = fmaxf(v[r], 0.f);
            v[r] = x * x;
        }
    }
    return v2u{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
}
// A quarter of a tile: 16 mt + .. of the 64 rows from n0 on, 16 nt + .. of the slots from sl0 on.  The wide form (N a multiple of 16): the four lanes of
// a slot exchange what they have, so that each ends up with 16 neighbouring rows; returns how many stores the wave has issued.
__device__ __forceinline__ void swap_rows32(unsigned& a, unsigned& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0], b = r[1];
}
__device__ __forceinline__ void swap_rows16(unsigned& a, unsigned& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
}
__device__ __forceinline__ void store16(void* to, v4u v, unsigned long long lanes) {
    asm volatile("s_mov_b64 exec, %2\n\tglobal_store_dwordx4 %0, %1, off\n\ts_mov_b64 exec, -1\n\ts_nop 0" ::"v"(to), "v"(v), "s"(lanes) : "memory");
}
template <int ACT, int NT>
__device__ __forceinline__ int grouped_store_wide(const GroupedArgs& a, const GroupedTile& t, int n0, int sl0, int lane, const float (&iw)[NT], const v4f (&acc)[4][NT]) {
    constexpr int W = ACT == 2 ? 1 : 2;
    const int n = n0 + 16 * (lane >> 4);
    int issued = 0;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int sl = sl0 + 16 * nt + (lane & 15);
        unsigned d[4][2];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const v2u r = grouped_result<ACT>(acc[mt][nt] * iw[nt], a.limit);
            d[mt][0] = r[0], d[mt][1] = r[1];
        }
#pragma unroll
        for (int x = 0; x < W; ++x) {                               // d[mt] of lanes 16 g + .. <-> d[g] of lanes 16 mt + ..
            swap_rows32(d[0][x], d[2][x]), swap_rows32(d[1][x], d[3][x]);
            swap_rows16(d[0][x], d[1][x]), swap_rows16(d[2][x], d[3][x]);
        }
        const unsigned long long lanes = __ballot(sl < t.ns && n < a.N);
        bf16_t* to = a.out + (ACT == 2 ? ((size_t)(t.first + sl) * a.N + n) / 2 : (size_t)(t.first + sl) * a.N + n);
        if (lanes) {
            if (ACT == 2) {
                store16(to, v4u{d[0][0], d[1][0], d[2][0], d[3][0]}, lanes);
            } else {
                store16(to, v4u{d[0][0], d[0][1], d[1][0], d[1][1]}, lanes);
                store16(to + 8, v4u{d[2][0], d[2][1], d[3][0], d[3][1]}, lanes);
            }
            issued += W;
        }
    }
    return issued;
}
template <int ACT, int NT>
__device__ __forceinline__ void grouped_store(const GroupedArgs& a, const GroupedTile& t, int n0, int sl0, int lane, const float (&iw)[NT], const v4f (&acc)[4][NT]) {
    const int col = lane & 15, g4 = lane >> 4;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int sl = sl0 + 16 * nt + col;
        if (sl >= t.ns) continue;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const int n = n0 + 16 * mt + 4 * g4;
            if (n >= a.N) continue;                                 // N % 4 == 0: the four rows are inside together
            const v2u r = grouped_result<ACT>(acc[mt][nt] * iw[nt], a.limit);
            if (ACT == 2) *(unsigned*)(a.out + ((size_t)(t.first + sl) * a.N + n) / 2) = r[0];
            else *(v2u*)(a.out + (size_t)(t.first + sl) * a.N + n) = r;
        }
    }
}

template <int ACT, bool LISTED>
__global__ __launch_bounds__(PT, 2) void grouped_gemm_persistent_kernel(GroupedArgs a) {
    __shared__ __attribute__((aligned(128))) unsigned char buf[2 * PBUF];
    __shared__ int side[SIDE];                                      // slot tiles of the experts before e | from AHEAD on the next tile's input rows
    static_assert(MAX_GROUPS < SIDE, "");
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
            if (e < a.E) side[e + 1] = carry + x;
            carry += __shfl(x, 63, 64);
        }
        if (lane == 0) side[0] = 0;
    }
    __syncthreads();
    const int row_tiles = (a.N + PR - 1) / PR, total = (LISTED ? a.n_tiles : __builtin_amdgcn_readfirstlane(side[a.E])) * row_tiles;
    // An XCD's share of the tiles: whole rounds of its workgroups, then what is left - fewer tiles than workgroups - cut by slots into as many
    // parts (two or four) as there are workgroups for.  Place p: tile (p) of the share, or a part of one.
    const int xcd = blockIdx.x & 7, per_xcd = gridDim.x >> 3, chunk = (total + 7) >> 3;
    const int begin = xcd * chunk, here = max(0, min(chunk, total - begin));
    const int whole = here / per_xcd * per_xcd, rest = here - whole, cut = LISTED ? 0 : rest * 4 <= per_xcd ? 2 : rest * 2 <= per_xcd ? 1 : 0;   // log2 of the parts
    const int last = whole + (rest << cut);
    int at = blockIdx.x >> 3;
    if (at >= last) return;

    auto tile_at = [&](int place, int from) __attribute__((always_inline)) {   // from: the expert of an earlier place
        const int over = place - whole, part = over >= 0 ? over & ((1 << cut) - 1) : 0, size = over >= 0 ? PS >> cut : PS;
        const int L = begin + (over >= 0 ? whole + (over >> cut) : place);
        GroupedTile t;
        if (LISTED) {
            const int s = __builtin_amdgcn_readfirstlane(L / row_tiles);       // which slot tile
            t.n0 = (L - s * row_tiles) * PR;
            const int2 ef = scalar_pair(a.tiles + 3 * (size_t)s);
            t.e = ef.x;
            t.first = ef.y;
            t.ns = min(max(scalar_word(a.tiles + 3 * (size_t)s + 2), 0), LISTED_SLOTS);
            return t;
        }
        int e = from & ~63;                                         // side[e] row_tiles <= L < side[e + 1] row_tiles, 64 experts at a time
        for (;;) {
            const int before = __popcll(__ballot(e + lane < a.E && side[min(e + lane, a.E - 1) + 1] * row_tiles <= L));
            e += before;
            if (before < 64) break;
        }
        e = __builtin_amdgcn_readfirstlane(e);
        const int skip = __builtin_amdgcn_readfirstlane(side[e]), slots = __builtin_amdgcn_readfirstlane(side[e + 1]) - skip;
        const int2 off = scalar_pair(a.offsets + e);
        const int l = L - skip * row_tiles, band = l / (BAND * slots), high = min(BAND, row_tiles - BAND * band), in = l - band * BAND * slots;
        const int s = __builtin_amdgcn_readfirstlane(in / high);
        t.e = e;
        t.n0 = __builtin_amdgcn_readfirstlane((BAND * band + in - s * high) * PR);
        t.first = __builtin_amdgcn_readfirstlane(off.x + s * PS + part * size);
        t.ns = __builtin_amdgcn_readfirstlane(min(size, off.y - t.first));   // (none or less: a part behind the expert's last slot)
        return t;
    };
    // Copies: of an operand half wave w brings rows 16 w .. 16 w + 15, eight (of 128 bytes) per instruction.  Request (h, j): half h, j of 2.
    auto x_row = [&](const GroupedTile& t, int r) __attribute__((always_inline)) { return t.first + min(r, max(t.ns, 1) - 1); };
    // (the lane's number is taken anew where a tile ends, so that nothing made of it is kept through the steps)
    auto fresh_lane = [&]() __attribute__((always_inline)) {
        int l = threadIdx.x & 63;
        asm volatile("" : "+v"(l));
        return l;
    };
    auto x_slot = [&](const GroupedTile& t, int h, int j, int lane) __attribute__((always_inline)) {
        if (LISTED && t.ns <= 0) return 0;                          // (an empty tile of the list: nothing is read or stored)
        const int s = x_row(t, 128 * h + 16 * w + 8 * j + (lane >> 3));
        if (LISTED) return a.x_index ? (int)a.x_index[s] : s;
        return a.order ? a.order[s] : s;
    };
    const bool indexed = LISTED ? a.x_index != nullptr : a.order != nullptr;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)buf) + (unsigned)w * 2048u;
    const unsigned ahead0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)side) + (unsigned)(AHEAD + 64 * w) * 4u;
    const int steps = a.K / KS, V = max(steps, 2);                  // (one step: a second one that copies and multiplies nothing)
    // the next tile's input rows come through LDS where there is room and time for it: nothing that is in flight is waited for
    const bool early = V >= 6 && indexed && (LISTED || a.E < AHEAD);
    GroupedTile t = tile_at(at, 0);
    if (!LISTED && t.ns <= 0) return;                               // (parts are the last places: nothing follows)
    const bf16_t* W0;
    unsigned woff[4];
    const unsigned char* xrow[4];
    int rows_here, steps_here;                                      // of the tile that is being copied: inputs from this wave's first on, steps (none: 0)
    auto point = [&](const GroupedTile& g, bool more, bool staged) __attribute__((always_inline)) {
        steps_here = __builtin_amdgcn_readfirstlane(more ? steps : 0);
        if (!more) return;                                          // (the requests that only count go to the last tile's addresses)
        const int lane = fresh_lane(), piece = ((lane & 7) ^ (lane >> 3)) * 16;
        W0 = a.W + ((size_t)g.e * a.N + g.n0) * (size_t)a.K;
        rows_here = __builtin_amdgcn_readfirstlane(g.ns - 16 * w);
        int slot[4];                                                // (all four asked for before the first is divided)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            slot[i] = staged ? side[AHEAD + 64 * w + 16 * (i >> 1) + 8 * (i & 1) + (lane >> 3)] : x_slot(g, i >> 1, i & 1, lane);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            woff[i] = (unsigned)min(128 * (i >> 1) + 16 * w + 8 * (i & 1) + (lane >> 3), a.N - 1 - g.n0) * (unsigned)a.K * 2u + piece;
            xrow[i] = (const unsigned char*)(a.X + (size_t)(a.div == 1 ? slot[i] : slot[i] / a.div) * (size_t)a.K) + piece;
            if (LISTED && g.ns <= 0) xrow[i] = (const unsigned char*)W0 + woff[i];   // (no input need exist)
        }
    };
    auto copy_w = [&](int h, unsigned to, int step) __attribute__((always_inline)) {
        const int k0 = step < steps ? step * KS : 0;
#pragma unroll
        for (int j = 0; j < 2; ++j) lds_copy16(lds0 + to + h * HALF + 1024 * j, W0 + k0, woff[2 * h + j], step - steps_here);
    };
    auto copy_x = [&](int h, unsigned to, int step) __attribute__((always_inline)) {
        const int k0 = step < steps ? step * KS : 0;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int left = (step - steps_here) & (128 * h + 8 * j - rows_here);
            lds_copy16(lds0 + to + (2 + h) * HALF + 1024 * j, xrow[2 * h + j] + (size_t)k0 * 2, left);
        }
    };
    point(t, true, false);
#pragma unroll
    for (int i = 0; i < 8; ++i) {                              // (in the order of the phases that read them)
        const int to = i / 4 * PBUF;
        if (i % 4 == 0) copy_x(0, to, i / 4);
        if (i % 4 == 1) copy_w(0, to, i / 4);
        if (i % 4 == 2) copy_x(1, to, i / 4);
        if (i % 4 == 3) copy_w(1, to, i / 4);
    }
    wait_copies<8>();                 // (as in front of every tile's epilogue)
    const int col = lane & 15, g4 = lane >> 4, group = w >> 2, q = w & 3;
    const bool wide = a.N % 16 == 0;
    int stored = 0;                                                 // stores behind the last tile, at least
    unsigned which = 0;                                             // the half of buf that holds the step
    const int p0 = (g4 ^ (col & 7)) << 4, p1 = ((4 + g4) ^ (col & 7)) << 4;

    auto run_tile = [&](auto na_, auto nb_, auto nt_) __attribute__((always_inline)) {
        constexpr int NA = decltype(na_)::value, NB = decltype(nb_)::value, NT = decltype(nt_)::value;   // row halves, slot halves, slots / 16 of a wave
        const int next = at + per_xcd;
        GroupedTile u = t;
        bool more = false;
        auto look = [&]() __attribute__((always_inline)) {
            if (next < last) {
                u = tile_at(next, t.e);
                more = LISTED || u.ns > 0;
            }
        };
        if (!early) look();
        v4f acc[NA][NB][4][NT];
#pragma unroll
        for (int i = 0; i < NA * NB * 4 * NT; ++i) (&acc[0][0][0][0])[i] = v4f{0.f, 0.f, 0.f, 0.f};
        const unsigned char* A = buf + (64 * group + col) * 128;
        const unsigned char* B = buf + 2 * HALF + (16 * NT * q + col) * 128;
        v4u av[2][4], b[NB][2][NT];
        auto read_a = [&](int h) __attribute__((always_inline)) {
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                av[0][mt] = *(const v4u*)(A + which + h * HALF + 2048 * mt + p0);
                av[1][mt] = *(const v4u*)(A + which + h * HALF + 2048 * mt + p1);
            }
        };
        auto read_b = [&](int h) __attribute__((always_inline)) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                b[h][0][nt] = *(const v4u*)(B + which + h * HALF + 2048 * nt + p0);
                b[h][1][nt] = *(const v4u*)(B + which + h * HALF + 2048 * nt + p1);
            }
        };
        auto multiply = [&](v4f(&c)[NB][4][NT]) __attribute__((always_inline)) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int h = 0; h < NB; ++h)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                        for (int mt = 0; mt < 4; ++mt)
                            c[h][mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, av[ks][mt]), __builtin_bit_cast(bf8, b[h][ks][nt]), c[h][mt][nt], 0, 0, 0);
        };
        // Requests come in the order x0 w0 x1 w1 (halves of a step), a phase's as soon as every wave has read what they replace; eight are younger than what the
        // next phase reads.  `late`: what the phase reads was requested before the last tile's stores, which may be under way still.
        auto settle = [&](bool late) __attribute__((always_inline)) {
            if (late && stored) {
                if (stored >= 16) wait_copies<8 + 16>();
                else if (stored >= 8) wait_copies<8 + 8>();
                else if (stored >= 4) wait_copies<8 + 4>();
                else wait_copies<8>();
            } else wait_copies<8>();
            step_barrier();
        };
        auto step = [&](auto edge_, int i) __attribute__((always_inline)) {
            constexpr bool EDGE = decltype(edge_)::value;              // (the first two steps and the last two: the others hold no branch)
            const bool live = !EDGE || V == steps || i < steps;
            const int k = !EDGE || i + 2 < V ? i + 2 : i + 2 - V;
            read_a(0);
#pragma unroll
            for (int h = 0; h < NB; ++h) read_b(h);
            if (!EDGE || i) copy_w(1, which ^ PBUF, !EDGE || i + 1 < V ? i + 1 : i + 1 - V);
            if (EDGE && i == 0) {                                           // (all of the first step has landed)
                wait_copies<63>();
                step_barrier();
            } else settle(EDGE && i == 1);
            if (live) multiply(acc[0]);
            step_barrier();

            if (NA == 2) read_a(1);
            if (EDGE && i == V - 2) point(u, more, early);
            copy_x(0, which, k);
            copy_w(0, which, k);
            copy_x(1, which, k);
            if (EDGE && early && i == 0) look();
            if (EDGE && early && i == 1 && more && u.ns > 0) {
                const int lane = fresh_lane();
                const int s = x_row(u, 128 * ((lane >> 4) & 1) + 16 * w + (lane & 15));
                lds_copy4(ahead0, LISTED ? (const void*)(a.x_index + s) : (const void*)(a.order + s));
            }
            settle(EDGE && i == 0);
            if (NA == 2 && live) multiply(acc[NA - 1]);
            step_barrier();
            which ^= PBUF;
        };
        step_barrier();                                             // every wave's requests for the first phases have landed
        if (group) step_barrier();
        typedef std::integral_constant<bool, true> Edge;
        typedef std::integral_constant<bool, false> Inner;
        int i = 0;
        do {
            if (i == 2)
                for (; i + 2 < V; ++i) step(Inner(), i);
            step(Edge(), i++);
        } while (i < V);
        if (!group) step_barrier();
        copy_w(1, which ^ PBUF, 1);
        // (what the next tile's first step reads; the stores below are younger)
        wait_copies<8>();
        const int lane = fresh_lane(), col = lane & 15;
        const int n0 = t.n0 + 64 * group, sl0 = 16 * NT * q;
        stored = 0;
        float iw[NB][NT];                                           // the expert works on iw * input
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                iw[b][nt] = 1.0f;
                const int sl = 128 * b + sl0 + 16 * nt + col;
                if (a.in_weight && sl < t.ns) {
                    const int s = t.first + sl;
                    iw[b][nt] = a.in_weight[LISTED ? (a.x_index ? a.x_index[s] : s) : (a.order ? a.order[s] : s)];
                }
            }
#pragma unroll
        for (int h = 0; h < NA; ++h)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (wide) stored += grouped_store_wide<ACT, NT>(a, t, n0 + 128 * h, 128 * b + sl0, lane, iw[b], acc[h][b]);
                else grouped_store<ACT, NT>(a, t, n0 + 128 * h, 128 * b + sl0, lane, iw[b], acc[h][b]);
            }
        asm volatile("" ::: "memory");                              // (the stores' branches join here: what follows stays uniform)
        if (more) t = u;
        at = next;
        return more;
    };
    typedef std::integral_constant<int, 1> One;
    typedef std::integral_constant<int, 2> Two;
    for (;;) {
        bool more;
        if (t.n0 + PR / 2 < a.N) more = t.ns > PS / 2 ? run_tile(Two(), Two(), Two()) : t.ns > PS / 4 ? run_tile(Two(), One(), Two()) : run_tile(Two(), One(), One());
        else more = t.ns > PS / 2 ? run_tile(One(), Two(), Two()) : t.ns > PS / 4 ? run_tile(One(), One(), Two()) : run_tile(One(), One(), One());
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
