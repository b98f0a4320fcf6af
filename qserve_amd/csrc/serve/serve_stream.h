// serve_stream.h -- products of many weight rows with few inputs (bfloat16): every weight read once, streamed through LDS.
//
// The four waves of a workgroup split the reduction (stage i of 64 elements belongs to wave i % 4).  Each streams its stages - one 128-byte
// line of 16 RB weight rows and of 16 SG inputs - through a ring of its own in LDS (global_load_lds, whole lines; the wave waits for its
// own oldest stage only, no barrier in the loop) and multiplies them with v_mfma_f32_16x16x32_bf16, weights as the A operand.  Pieces of
// a row are permuted by its number: 16-byte reads without bank conflicts.
#pragma once
#include "serve_common.h"

namespace {
constexpr int STREAM_WAVES = 4;
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr;
constexpr int XK = 64;               // reduction elements per stage
constexpr int XRING = 18 * 1024;     // ring of one wave: two workgroups fit a CU

// A ring of DEPTH stages, each weights and then inputs; APART: all stages' weights and then all inputs, so that the weights' places don't depend on SG
template <int RB, int SG, bool APART>
struct StreamRing {
    static constexpr int STAGE = 16 * (RB + SG) * 128, INSTR = STAGE / 1024, DEPTH = XRING / STAGE;
    static constexpr int WEIGHTS = APART ? 2048 * RB : STAGE, INPUTS = APART ? 2048 * SG : STAGE, INPUTS_AT = APART ? DEPTH * WEIGHTS : 2048 * RB;
    static_assert(DEPTH >= 2 && DEPTH <= 4, "");
};
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// ONCE: nothing reads these lines again (non-temporal: they leave the caches to what is read again)
template <bool ONCE>
__device__ __forceinline__ void lds_copy16(unsigned dst, const void* base, unsigned off) {
    if constexpr (ONCE) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(off), "s"(base), "s"(dst) : "memory");
    else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst) : "memory");
}
__device__ __forceinline__ void lds_copy4(unsigned dst, const void* from) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(from), "s"(dst) : "memory");
}
// a workgroup's barrier that leaves requests into LDS in flight
__device__ __forceinline__ void barrier_in_flight() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void lds_copy16(unsigned dst, const void* from) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(dst) : "memory");
}

// ONCE: the launch reads every weight once, so non-temporally: a large stream gets 4 - 10 % faster (92 / 185 MB of experts 21.5 / 39.1 -> 19.5 / 36.8 us, 4096 x 4096
// 8.9 -> 8.5).  Where workgroups read the same rows one after another, or rows start inside a line of 128 bytes, whose halves two requests would fetch, it loses
// (2560 x 5120 read twice 16.1 -> 20.7).  Under 1 MB, which a cache keeps beside anything, it loses too (64 x 2048 of 64 inputs 5.0 -> 5.6).
// A model whose weights the caches hold from step to step loses by it with many rows (the forms *_kept, which the engine asks for): whole steps of four layers, 74 /
// 116 / 187 / 194 / 234 MB of weights, non-temporally -> kept, us: 8 rows 234 -> 246, 204 -> 208, 223 -> 225, 227 -> 226, 224 -> 228, 24 rows 250 -> 255, 222 -> 218,
// 240 -> 235, 245 -> 240, 243 -> 244, 32 rows 258 -> 257, 227 -> 220, 243 -> 238, 253 -> 243, 248 -> 247, 64 rows 290 -> 287, 260 -> 255, 268 -> 266, 287 -> 284, 270 ->
// 270.  So up to 200 MB they are kept in steps of more than 24 rows.  Larger ones lose by that at any number (24 layers of 43 MB: 17 / 32 rows 1340 -> 1446, 1377 -> 1477).
inline bool streams_once(const void* w, int64_t rows, int K) { return K % 64 == 0 && (uintptr_t)w % 128 == 0 && rows * K >= 1 << 19; }
// The weights of a wave's first EARLY stages, requested before it knows its inputs (EARLY_MIN: elements from which every wave has three stages)
constexpr int EARLY = 2, EARLY_MIN = 3 * STREAM_WAVES * XK;
template <int RB, bool ONCE>
__device__ __forceinline__ void request_early(const bf16_t* W0, int K, int rows_here, unsigned char* ring, int w, int lane) {
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)ring), piece = (unsigned)((lane & 7) ^ (lane >> 3)) * 16u;
#pragma unroll
    for (int i = 0; i < EARLY; ++i) {                                              // (every one of these stages is whole: the row's last one is a third or later)
        const bf16_t* from = W0 + (w + STREAM_WAVES * i) * XK;
#pragma unroll
        for (int j = 0; j < 2 * RB; ++j) lds_copy16<ONCE>(lds0 + 2048 * RB * i + 1024 * j, from, (unsigned)min(8 * j + (lane >> 3), rows_here - 1) * (unsigned)K * 2u + piece);
    }
}
// acc[r][g]: this wave's share of the products of weight rows W0 + 16 r + .. (rows_here of them, K elements each) with inputs 16 g + ..;
// input(i): where input i starts.  w (the wave) is wave-uniform; `ring`: its XRING bytes of LDS.  PRE: request_early has been called and nothing else is in flight.
template <int RB, int SG, bool ONCE, bool PRE = false, class Input>
__device__ __forceinline__ void stream_products(const bf16_t* W0, int K, int rows_here, unsigned char* ring, int w, int lane, Input input,
                                                v4f (&acc)[RB][SG]) {
    typedef StreamRing<RB, SG, PRE> R;
    const int stages = (K + XK - 1) / XK, mine = stages > w ? (stages - w + STREAM_WAVES - 1) / STREAM_WAVES : 0;
    const int piece = (lane & 7) ^ (lane >> 3);
    unsigned woff[2 * RB];
    const bf16_t* xrow[2 * SG];
#pragma unroll
    for (int j = 0; j < 2 * RB; ++j) woff[j] = (unsigned)min(8 * j + (lane >> 3), rows_here - 1) * (unsigned)K * 2u;
#pragma unroll
    for (int j = 0; j < 2 * SG; ++j) xrow[j] = input(8 * j + (lane >> 3));
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int g = 0; g < SG; ++g) acc[r][g] = v4f{0.f, 0.f, 0.f, 0.f};
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)ring);
    auto issue = [&](int i, bool weights) __attribute__((always_inline)) {
        const int k0 = (w + STREAM_WAVES * i) * XK;
        const unsigned po = k0 + piece * 8 < K ? (unsigned)piece * 16u : 0u;       // (beyond the row: any valid piece, masked below)
        const unsigned at = i % R::DEPTH, wdst = lds0 + at * R::WEIGHTS, xdst = lds0 + R::INPUTS_AT + at * R::INPUTS;
        if (weights) {
#pragma unroll
            for (int j = 0; j < 2 * RB; ++j) lds_copy16<ONCE>(wdst + 1024 * j, W0 + k0, woff[j] + po);
        }
#pragma unroll
        for (int j = 0; j < 2 * SG; ++j) lds_copy16(xdst + 1024 * j, (const unsigned char*)(xrow[j] + k0) + po);
    };
    const int row = lane & 15, quad = lane >> 4;
    if constexpr (PRE) {
        static_assert(R::DEPTH >= EARLY && R::DEPTH <= 3, "");
        for (int i = 0; i < R::DEPTH; ++i) issue(i, i >= EARLY);                   // (three stages at least)
    } else {
        wait_vm<0>();
        for (int i = 0; i < min(R::DEPTH, mine); ++i) issue(i, true);
    }
    for (int i = 0; i < mine; ++i) {
        const int ahead = min(R::DEPTH - 1, mine - 1 - i);                         // stages requested behind this one
        if (PRE && i == 0) wait_vm<(R::DEPTH - 1) * 2 * SG + (R::DEPTH - EARLY) * 2 * RB>();   // (whose first weights are older)
        else if (R::DEPTH > 3 && ahead == 3) wait_vm<3 * R::INSTR>();
        else if (R::DEPTH > 2 && ahead == 2) wait_vm<2 * R::INSTR>();
        else if (ahead == 1) wait_vm<R::INSTR>();
        else wait_vm<0>();
        const unsigned char *ws = ring + (i % R::DEPTH) * R::WEIGHTS, *xs = ring + R::INPUTS_AT + (i % R::DEPTH) * R::INPUTS;
        const int left = K - (w + STREAM_WAVES * i) * XK;                          // elements of this stage inside the row
#pragma unroll
        for (int ks = 0; ks < XK / 32; ++ks) {
            const int p = 4 * ks + quad;
            v4u A[RB], B[SG];
#pragma unroll
            for (int r = 0; r < RB; ++r) A[r] = *(const v4u*)(ws + (16 * r + row) * 128 + ((p ^ (row & 7)) << 4));
#pragma unroll
            for (int g = 0; g < SG; ++g) B[g] = *(const v4u*)(xs + (16 * g + row) * 128 + ((p ^ (row & 7)) << 4));
            if (left < XK && p * 8 >= left) {
#pragma unroll
                for (int r = 0; r < RB; ++r) A[r] = v4u{0u, 0u, 0u, 0u};
#pragma unroll
                for (int g = 0; g < SG; ++g) B[g] = v4u{0u, 0u, 0u, 0u};
            }
#pragma unroll
            for (int r = 0; r < RB; ++r)
#pragma unroll
                for (int g = 0; g < SG; ++g)
                    acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, A[r]), __builtin_bit_cast(bf8, B[g]), acc[r][g], 0, 0, 0);
        }
        if (i + R::DEPTH < mine) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                     // the slot has been read
            issue(i + R::DEPTH, true);
        }
    }
}
}  // namespace
