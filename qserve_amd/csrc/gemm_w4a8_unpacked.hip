// gemm_w4a8_unpacked.hip -- W4A8 products of prompts in two launches: the weights widened to int8 once, in scratch that the caller hands in,
// then an int8 x int8 product whose loop holds nothing but copies and matrix instructions.
//
// For per-group weights, whose level-2 dequant is vector work beside the matrix instructions wherever it is done in the loop: once a weight here, in the four-wave
// tile (gemm_w4a8_wide.hip) once a weight and 256 tokens.  Both are bound by the card's power under matrix load: 8192 tokens x 28672 x 4096 + silu 880 -> 769 us
// (2.19 -> 2.50 POP/s; of the 769 30 are the widening, 178 MB at 5.9 TB/s), 5331 x 12288 x 4096 253 -> 224, 5331 x 4096 x 11008 274 -> 218 (the last round of tiles cut),
// 1100 x 4096 x 14336 228 -> 117.  Per-channel weights gain nothing (8192 x 28672 x 4096 670 -> 700: the nibbles need no arithmetic, and packed they halve what LDS
// delivers), 32 x 32 x 32 instructions lose (769 -> 791 with random data).  Where it is taken: qs_w4a8_per_group_scratch_bytes in gemm_w4a8.hip.
//
// Same integers as the other kernels (gemm_w4a8.hip: packed layout, level-2 dequant; reference kernels w4a8_per_group/gemm_cuda.cu:328-628 and
// w4a8_per_chn/gemm_cuda.cu:303-594), so the accumulators are the same and so are the outputs, bit for bit.
#include "common.h"
#include <type_traits>

namespace {
typedef __attribute__((address_space(3))) void* lds_ptr;

// ---- weights -> int8 rows ---------------------------------------------------------------------------------------------------------------
// A workgroup widens 32 channels x 256 k.  Bound by HBM (1.5 bytes a weight).  A packed 16-byte chunk (c, e) of a (32 channels, 32 k) tile
// holds channels 8 b + c (low nibbles) and 8 b + c + 16 (high), k = 16 d + 4 e .. + 3 in dword 2 d + b; through LDS whole 256-byte runs of a row
// are stored.  ACT: channel f of the lower half of N goes to row 2 f, of the upper half to 2 f + 1, so that a lane of the product ends up with both.
__global__ __launch_bounds__(128) void unpack_kernel(int8_t* __restrict__ out, const uint8_t* __restrict__ W, const int8_t* __restrict__ zeros,
                                                     const int8_t* __restrict__ scales8, int N, int K, int act) {
    constexpr int RS = 256 + 16;
    __shared__ __attribute__((aligned(16))) uint8_t rows[32 * RS];
    const int n32 = blockIdx.y, k0 = blockIdx.x * 256, kt = min(8, (K - k0) >> 5);      // tiles of 32 k here (K % 128 == 0: 4 or 8)
    const v4u* src = (const v4u*)(W + ((size_t)n32 * (K >> 5) + (k0 >> 5)) * 512);
    const int tid = threadIdx.x;
    v4u raw[2];
    u32 s[2], z[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int chunk = tid + 128 * i, t = chunk >> 5, c = (chunk >> 2) & 7;
        if (t >= kt) continue;
        raw[i] = __builtin_nontemporal_load(src + chunk);
        const size_t at = (size_t)((k0 >> 7) + (t >> 2)) * N + n32 * 32 + c * 4;   // stored in the order (c, j) of channel 8 j + c in every 32
        s[i] = *(const u32*)(scales8 + at);
        z[i] = *(const u32*)(zeros + at);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int chunk = tid + 128 * i, t = chunk >> 5, c = (chunk >> 2) & 7, e = chunk & 3;
        if (t >= kt) continue;
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const u32 r = raw[i][2 * d + b];
                uint8_t* to = rows + (8 * b + c) * RS + 32 * t + 16 * d + 4 * e;
                *(u32*)to = unpack_lo<1>(r, (s[i] >> (8 * b)) & 0xFFu, ((z[i] >> (8 * b)) & 0xFFu) * 0x01010101u);
                *(u32*)(to + 16 * RS) = unpack_hi<1>(r, (s[i] >> (8 * b + 16)) & 0xFFu, ((z[i] >> (8 * b + 16)) & 0xFFu) * 0x01010101u);
            }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int piece = tid + 128 * i, r = piece >> 4, at = (piece & 15) * 16, n = n32 * 32 + r;
        if (at >= 32 * kt) continue;
        const int row = act ? (n < N / 2 ? 2 * n : 2 * (n - N / 2) + 1) : n;
        *(v4u*)(out + (size_t)row * K + k0 + at) = *(const v4u*)(rows + r * RS + at);
    }
}

// ---- int8 x int8 ------------------------------------------------------------------------------------------------------------------------
// Tiles of 256 channels x 256 tokens (128 or 64 where no more are left).  Bound by the matrix cores.
//
// Eight waves, two per SIMD: waves 0 - 3 and 4 - 7 are half a phase apart, so that one of a SIMD's two always multiplies while the other reads its next
// operands.  A K step of 128 has two phases, one per half of the tile's channels; in each a wave has 64 channels x 64 tokens: 32 instructions.  The first reads a
// weight half and both token halves (16 reads of 16 bytes a lane), the second the other weight half (8).  What every wave has read is requested anew for the
// step after the next (global_load_lds, whole 128-byte lines of a row; pieces permuted by the row's number: reads without bank conflicts), and a phase waits
// for what the next one reads, requested three phases before: 64 - 112 KiB in flight a CU.  Of tokens that a tile does not have every wave issues the same
// requests with one lane, so that the counted waits hold whatever the tile's size.
//
// Workgroups are persistent, one per CU; the last two steps of a tile request the first two of the next.  An XCD walks bands of 8 channel tiles and through
// the tokens inside a band; the tiles of its last, part-empty round are cut by tokens into as many parts (two or four) as it has workgroups for.
constexpr int PR = 256, PS = 256, PWAVES = 8, PT = 64 * PWAVES;
constexpr int KS = 128;                             // k of a step: one line of a row
constexpr int PBUF = (PR + PS) * KS, HALF = 128 * KS, BAND = 8;

// A request into LDS by all lanes (left < 0: 1 KiB) or by the first one alone, for the counted waits' sake: an instruction without a lane need not count.
__device__ __forceinline__ void lds_copy16(unsigned dst, const void* base, unsigned off, int left) {
    asm volatile("s_mov_b32 m0, %2\n\ts_ashr_i32 exec_hi, %3, 31\n\ts_or_b32 exec_lo, exec_hi, 1\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(base), "s"(dst), "s"(left) : "memory", "scc");
}
__device__ __forceinline__ void lds_copy2(unsigned dst, const void* from) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_ushort %0, off" ::"v"(from), "s"(dst) : "memory");
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
__device__ __forceinline__ void store16(void* to, v4u v, unsigned long long lanes) {
    asm volatile("s_mov_b64 exec, %2\n\tglobal_store_dwordx4 %0, %1, off\n\ts_mov_b64 exec, -1\n\ts_nop 0" ::"v"(to), "v"(v), "s"(lanes) : "memory");
}

struct I8Args {
    _Float16* out;
    const int8_t* X;                 // [M, K]
    const int8_t* W;                 // [N, K] widened
    const _Float16 *ws, *sa;         // [N], [M]
    int M, N, K;
    unsigned long long* clk;         // qs_debug_gemm_clock_probe
};
struct I8Tile {
    int n0, first, ns;               // first channel row, first token, tokens
};

template <bool ACT>
__global__ __launch_bounds__(PT, 2) void gemm_i8_kernel(I8Args a) {
    __shared__ __attribute__((aligned(128))) unsigned char buf[2 * PBUF];
    __shared__ __attribute__((aligned(16))) u32 side[2 * 256];      // of the tile: channel scales | token scales
    unsigned long long ck0 = 0, rt0 = 0;
    if (a.clk) {
        ck0 = __builtin_amdgcn_s_memtime();
        rt0 = __builtin_amdgcn_s_memrealtime();
    }
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row_tiles = a.N / PR, slots = (a.M + PS - 1) / PS, total = row_tiles * slots;
    const int xcd = blockIdx.x & 7, per_xcd = gridDim.x >> 3, chunk = (total + 7) >> 3;
    const int begin = xcd * chunk, here = max(0, min(chunk, total - begin));
    const int whole = here / per_xcd * per_xcd, rest = here - whole, cut = rest * 4 <= per_xcd ? 2 : rest * 2 <= per_xcd ? 1 : 0;
    const int last = whole + (rest << cut);
    int at = blockIdx.x >> 3;
    if (at >= last) return;
    auto tile_at = [&](int place) __attribute__((always_inline)) {
        const int over = place - whole, part = over >= 0 ? over & ((1 << cut) - 1) : 0, size = over >= 0 ? PS >> cut : PS;
        const int l = begin + (over >= 0 ? whole + (over >> cut) : place);
        const int band = l / (BAND * slots), high = min(BAND, row_tiles - BAND * band), in = l - band * BAND * slots;
        const int s = in / high;
        I8Tile t;
        t.n0 = __builtin_amdgcn_readfirstlane((BAND * band + in - s * high) * PR);
        t.first = __builtin_amdgcn_readfirstlane(s * PS + part * size);
        t.ns = __builtin_amdgcn_readfirstlane(min(size, a.M - t.first));    // (none or less: a part behind the last token)
        return t;
    };
    auto fresh_lane = [&]() __attribute__((always_inline)) {
        int l = threadIdx.x & 63;
        asm volatile("" : "+v"(l));
        return l;
    };
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)buf) + (unsigned)w * 2048u;
    const unsigned side0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)side);
    const int steps = a.K / KS, V = max(steps, 2);                  // (one step: a second one that copies and multiplies nothing)
    I8Tile t = tile_at(at);
    if (t.ns <= 0) return;                                          // (parts are the last places: nothing follows)
    // Copies: of an operand half wave w brings rows 16 w .. 16 w + 15, eight (of 128 bytes) per instruction.
    unsigned woff[4], xoff[4];
    const int8_t *W0, *X0;
    int rows_here, steps_here;
    {
        const int piece = ((lane & 7) ^ (lane >> 3)) * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i) woff[i] = (unsigned)(128 * (i >> 1) + 16 * w + 8 * (i & 1) + (lane >> 3)) * (unsigned)a.K + piece;
    }
    auto point = [&](const I8Tile& g, bool more) __attribute__((always_inline)) {
        steps_here = __builtin_amdgcn_readfirstlane(more ? steps : 0);
        if (!more) return;                                          // (the requests that only count go to the last tile's addresses)
        W0 = a.W + (size_t)g.n0 * (size_t)a.K;
        X0 = a.X + (size_t)g.first * (size_t)a.K;
        rows_here = __builtin_amdgcn_readfirstlane(g.ns - 16 * w);
        const int lane = fresh_lane(), piece = ((lane & 7) ^ (lane >> 3)) * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i) xoff[i] = (unsigned)min(128 * (i >> 1) + 16 * w + 8 * (i & 1) + (lane >> 3), g.ns - 1) * (unsigned)a.K + piece;
    };
    auto copy_w = [&](int h, unsigned to, int step) __attribute__((always_inline)) {
        const int k0 = step < steps ? step * KS : 0;
#pragma unroll
        for (int j = 0; j < 2; ++j) lds_copy16(lds0 + to + h * HALF + 1024 * j, W0 + k0, woff[2 * h + j], step - steps_here);
    };
    auto copy_x = [&](int h, unsigned to, int step) __attribute__((always_inline)) {
        const int k0 = step < steps ? step * KS : 0;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            lds_copy16(lds0 + to + (2 + h) * HALF + 1024 * j, X0 + k0, xoff[2 * h + j], (step - steps_here) & (128 * h + 8 * j - rows_here));
    };
    // what the tile's epilogue multiplies with, a 16-bit value a word: waves 0 - 3 the channels', 4 - 7 the tokens'
    auto copy_side = [&](const I8Tile& g) __attribute__((always_inline)) {
        const int i = 64 * (w & 3) + fresh_lane();
        if (w < 4) {
            const int n = g.n0 + i;
            lds_copy2(side0 + 256u * w, a.ws + (ACT ? (n >> 1) + (n & 1) * (a.N >> 1) : n));
        } else {
            lds_copy2(side0 + 256u * w, a.sa + g.first + min(i, g.ns - 1));
        }
    };
    point(t, true);
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
    int stored = 0;                                                 // stores behind the last tile
    unsigned which = 0;                                             // the half of buf that holds the step
    const int p0 = (g4 ^ (col & 7)) << 4, p1 = ((4 + g4) ^ (col & 7)) << 4;

    auto run_tile = [&](auto nb_, auto nt_) __attribute__((always_inline)) {
        constexpr int NB = decltype(nb_)::value, NT = decltype(nt_)::value;   // token halves, tokens / 16 of a wave
        const int next = at + per_xcd;
        I8Tile u = t;
        bool more = false;
        if (next < last) {
            u = tile_at(next);
            more = u.ns > 0;
        }
        v4i acc[2][NB][4][NT];
#pragma unroll
        for (int i = 0; i < 2 * NB * 4 * NT; ++i) (&acc[0][0][0][0])[i] = v4i{0, 0, 0, 0};
        const unsigned char* A = buf + (64 * group + col) * KS;
        const unsigned char* B = buf + 2 * HALF + (16 * NT * q + col) * KS;
        v4i av[2][4], b[NB][2][NT];
        auto read_a = [&](int h) __attribute__((always_inline)) {
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                av[0][mt] = *(const v4i*)(A + which + h * HALF + 2048 * mt + p0);
                av[1][mt] = *(const v4i*)(A + which + h * HALF + 2048 * mt + p1);
            }
        };
        auto read_b = [&](int h) __attribute__((always_inline)) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                b[h][0][nt] = *(const v4i*)(B + which + h * HALF + 2048 * nt + p0);
                b[h][1][nt] = *(const v4i*)(B + which + h * HALF + 2048 * nt + p1);
            }
        };
        auto multiply = [&](v4i(&c)[NB][4][NT]) __attribute__((always_inline)) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int h = 0; h < NB; ++h)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                        for (int mt = 0; mt < 4; ++mt) c[h][mt][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[ks][mt], b[h][ks][nt], c[h][mt][nt], 0, 0, 0);
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
            if (EDGE && i == 0) {                                   // (all of the first step has landed)
                wait_copies<63>();
                step_barrier();
            } else settle(EDGE && i == 1);
            if (live) multiply(acc[0]);
            step_barrier();

            read_a(1);
            if (EDGE && i == 0) copy_side(t);                       // (every wave is past the last tile's epilogue)
            if (EDGE && i == V - 2) point(u, more);
            copy_x(0, which, k);
            copy_w(0, which, k);
            copy_x(1, which, k);
            settle(EDGE && i == 0);
            if (live) multiply(acc[1]);
            step_barrier();
            which ^= PBUF;
        };
        typedef std::integral_constant<bool, true> Edge;
        typedef std::integral_constant<bool, false> Inner;
        step_barrier();                                             // every wave's requests for the first step have landed
        if (group) step_barrier();
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
        const int lane = fresh_lane(), col = lane & 15, g = lane >> 4;
        stored = 0;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float sa[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) sa[nt] = (float)__builtin_bit_cast(_Float16, (unsigned short)side[256 + 128 * b + 16 * NT * q + 16 * nt + col]);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float ws[4][4];
#pragma unroll
                for (int mt = 0; mt < 4; ++mt) {
                    const v4u four = *(const v4u*)(side + 128 * h + 64 * group + 16 * mt + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) ws[mt][r] = (float)__builtin_bit_cast(_Float16, (unsigned short)four[r]);
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    constexpr int D = ACT ? 1 : 2;
                    u32 d[4][2];
#pragma unroll
                    for (int mt = 0; mt < 4; ++mt) {
                        const v4i c = acc[h][b][mt][nt];
                        _Float16 o[4];
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            float y = epi_per_group(c[r], ws[mt][r], sa[nt]);
                            asm("" : "+v"(y));                      // (a float of its own, then rounded to 16 bits: not both in one rounding)
                            o[r] = (_Float16)y;
                        }
                        if (ACT) {                                  // gate, up of two units -> silu_and_mul's arithmetic
                            const h2 u2 = {(_Float16)((float)qs_silu_h((float)o[0]) * (float)o[1]), (_Float16)((float)qs_silu_h((float)o[2]) * (float)o[3])};
                            d[mt][0] = __builtin_bit_cast(u32, u2), d[mt][1] = 0;
                        } else {
                            d[mt][0] = __builtin_bit_cast(u32, (h2){o[0], o[1]}), d[mt][1] = __builtin_bit_cast(u32, (h2){o[2], o[3]});
                        }
                    }
#pragma unroll
                    for (int x = 0; x < D; ++x) {                   // d[mt] of lanes 16 g + .. <-> d[g] of lanes 16 mt + ..
                        auto swap32 = [](u32& p, u32& q) { const auto r = __builtin_amdgcn_permlane32_swap(p, q, false, false); p = r[0], q = r[1]; };
                        auto swap16 = [](u32& p, u32& q) { const auto r = __builtin_amdgcn_permlane16_swap(p, q, false, false); p = r[0], q = r[1]; };
                        swap32(d[0][x], d[2][x]), swap32(d[1][x], d[3][x]);
                        swap16(d[0][x], d[1][x]), swap16(d[2][x], d[3][x]);
                    }
                    const int m = 128 * b + 16 * NT * q + 16 * nt + col, n = t.n0 + 128 * h + 64 * group + 16 * g;
                    const unsigned long long lanes = __ballot(m < t.ns);
                    if (lanes) {
                        if (ACT) {
                            store16(a.out + ((size_t)(t.first + m) * a.N + n) / 2, v4u{d[0][0], d[1][0], d[2][0], d[3][0]}, lanes);
                        } else {
                            _Float16* to = a.out + (size_t)(t.first + m) * a.N + n;
                            store16(to, v4u{d[0][0], d[0][1], d[1][0], d[1][1]}, lanes);
                            store16(to + 8, v4u{d[2][0], d[2][1], d[3][0], d[3][1]}, lanes);
                        }
                        stored += D;
                    }
                }
            }
        }
        asm volatile("" ::: "memory");                              // (the stores' branches join here: what follows stays uniform)
        if (more) t = u;
        at = next;
        return more;
    };
    typedef std::integral_constant<int, 1> One;
    typedef std::integral_constant<int, 2> Two;
    for (;;) {
        const bool more = t.ns > PS / 2 ? run_tile(Two(), Two()) : t.ns > PS / 4 ? run_tile(One(), Two()) : run_tile(One(), One());
        if (!more) break;
    }
    if (a.clk && threadIdx.x == 0) {
        a.clk[2 * blockIdx.x] = __builtin_amdgcn_s_memtime() - ck0;
        a.clk[2 * blockIdx.x + 1] = __builtin_amdgcn_s_memrealtime() - rt0;
    }
}
}  // namespace

// Entry used by the dispatcher in gemm_w4a8.hip; preconditions (checked there): N % 256 == 0, K % 128 == 0, M K and N K below 2^32, `scratch` holds N K bytes.
int qs_launch_gemm_unpacked(bool act, const int8_t* A, const uint8_t* W, const int8_t* zeros, const int8_t* scales8, const void* wscales, const void* ascales,
                            void* out, int M, int N, int K, void* scratch, hipStream_t stream) {
    hipLaunchKernelGGL(unpack_kernel, dim3((K + 255) / 256, N / 32), dim3(128), 0, stream, (int8_t*)scratch, W, zeros, scales8, N, K, act ? 1 : 0);
    const int rc = qs_launch_status("w4a8 gemm (weights widened)");
    if (rc != QS_OK) return rc;
    const I8Args a = {(_Float16*)out, A, (const int8_t*)scratch, (const _Float16*)wscales, (const _Float16*)ascales, M, N, K, g_gemm_clk_cap >= 256 ? g_gemm_clk : nullptr};
    const dim3 grid(256), block(PT);                                // one workgroup per CU, 32 per XCD
    if (act) hipLaunchKernelGGL(gemm_i8_kernel<true>, grid, block, 0, stream, a);
    else hipLaunchKernelGGL(gemm_i8_kernel<false>, grid, block, 0, stream, a);
    return qs_launch_status("w4a8 gemm (widened weights)");
}
