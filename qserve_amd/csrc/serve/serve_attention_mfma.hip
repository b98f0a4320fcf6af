// serve_attention_mfma.hip -- latent attention on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16), prompts and decoding.
//
// Work unit ("tile", made by the host): up to TPB consecutive tokens of ONE sequence in this step.  A workgroup of four waves
// serves a tile; a wave owns 16 query rows = TQ tokens x HP head slots (HP = heads rounded up to a power of two, at most 16;
// more than 16 heads: blockIdx.y walks head groups of 16).  Sixteen rows, not 32: a row of 576 query values and 512 output
// columns then costs a lane 72 + 128 registers and nothing spills (the 32-row form needed 144 + 256).  Keys arrive in tiles
// of 32 cache rows, staged once per workgroup in LDS in two forms: row-major (A operand of S^T = K Q^T, plain 16-byte
// reads) and transposed (A operand of O^T = C^T P^T, 8-byte reads).  With the products swapped like this a lane holds 8 of
// the 32 scores of ITS query row, so the softmax needs two exchanges (lanes ^ 16, ^ 32) and the probabilities already sit in
// B-operand order (the k-slot <-> key mapping of the second product is chosen to match the accumulator layout of the first).
// A tile with few tokens (decoding: one) does not fill four waves with rows; then the waves split the KEY tiles among them and
// merge their partial softmax results through LDS at the end.
// Scores, running maxima and sums are float; q and the probabilities enter the matrix cores as bfloat16.
//
// Keys behind the window: a workgroup's key tiles are numbered, first nA tiles of such keys, then the tiles from the window's start.
// With `keep_first` these are the tiles of the sequence's first positions that lie wholly below the window's first tile (a kept
// position inside a window tile is simply visible there); with `pooled` they are tiles of 32 consecutive BLOCKS, one row per block of
// `pool_block` positions from a second pool, each row addressed through the page of the block's first position.  A sink starts the
// softmax state of the rows' first key split at (maximum = sink, sum = 1).
#include "serve_common.h"

namespace {
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

constexpr int NWV = 4;
constexpr int BN = 32;          // keys per tile
constexpr int VS = BN + 4;      // row stride (elements) of the transposed tile: 18 dwords, 8-byte reads of 32 lanes hit 64 banks


// RT: 32-element steps along a cache row (R <= 32 RT); CT: 16-column tiles of the output (rank <= 16 CT).
template <int RT, int CT>
__global__ __launch_bounds__(64 * NWV, (RT > 10 ? 1 : 2)) void latent_attention_mfma_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ qf, const bf16_t* __restrict__ pool_base,
    const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ pos, const int32_t* __restrict__ tiles,
    int window, int H, int rank, int R, int page, int HP, int TQ, float* __restrict__ part_o, float* __restrict__ part_ml,
    int n_tokens, int s_lo, int s_hi, int per, int64_t pool_stride, int chunk, const float* __restrict__ bias, int bias_len,
    int keep_first, const float* __restrict__ sink, const bf16_t* __restrict__ pooled_base, int64_t pooled_stride, int pool_block,
    int block_rows, const float* __restrict__ slopes) {
    constexpr int RS = 32 * RT + 8;                      // row stride (elements) of the row-major tile
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    bf16_t* Ks = (bf16_t*)smem;                          // [BN][RS]
    bf16_t* Vt = Ks + BN * RS;                           // [16 CT][VS]
    float* scratch = (float*)smem;                       // merge phase (after the key loop)

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int col = lane & 15, g4 = lane >> 4;           // query row of this lane; k-group / accumulator row block
    const int slot = tiles[3 * blockIdx.x], t0 = tiles[3 * blockIdx.x + 1], ntok = tiles[3 * blockIdx.x + 2];
    // heads [g per, (g + 1) per) read pool g (pool_stride elements apart): blockIdx.y walks the pools' head groups of 16
    const int gpp = (per + 15) / 16, pool_id = blockIdx.y / gpp;
    const int h0 = pool_id * per + (blockIdx.y % gpp) * 16, h_end = pool_id * per + per;
    const bf16_t* __restrict__ pool = pool_base + (size_t)pool_id * (size_t)pool_stride;
    const bf16_t* __restrict__ pooled = pooled_base ? pooled_base + (size_t)pool_id * (size_t)pooled_stride : nullptr;
    const int32_t* bt = block_table + (size_t)slot * table_stride;

    // rows of this wave: group grp of TQ tokens, key split sp
    const int G = (ntok + TQ - 1) / TQ;                  // 1 .. 4
    const int S = NWV / G;
    const bool active = w < G * S;
    const int grp = active ? w % G : 0, sp = active ? w / G : 0;
    const int tok_in = grp * TQ + col / HP;              // token of this lane's query row within the tile
    const int head = h0 + col % HP;
    const bool row_ok = active && tok_in < ntok && head < h_end;
    const int t = t0 + (tok_in < ntok ? tok_in : 0);
    const int p_row = pos[t];
    int lo_row = window > 0 ? max(0, p_row - window + 1) : 0;
    if (chunk > 0) lo_row = max(lo_row, p_row - p_row % chunk);   // chunks are counted from position 0 of the sequence
    const float* brow = bias ? bias + (size_t)(row_ok ? head : 0) * bias_len : nullptr;

    const float slope = slopes ? slopes[row_ok ? head : 0] : 0.f;

    // block key range (tokens of a tile are consecutive positions; read both ends)
    const int p_first = pos[t0], p_last = pos[t0 + ntok - 1];
    int lo_first = window > 0 ? max(0, p_first - window + 1) : 0;
    if (chunk > 0) lo_first = max(lo_first, p_first - p_first % chunk);   // (the first token's bound is the tile's lowest)
    const int kstart = (lo_first / BN) * BN;
    // tiles of keys behind the window, and each row's count of such keys
    const int nb_last = pooled ? max(0, p_last - window + 1) / pool_block : 0;      // blocks the tile's last token sees
    const int nb_row = pooled ? max(0, p_row - window + 1) / pool_block : 0;
    const int nA = pooled ? (nb_last + BN - 1) / BN : (keep_first > 0 ? min((keep_first + BN - 1) / BN, kstart / BN) : 0);
    const int nT = nA + (p_last - kstart) / BN + 1;
    // wave key range: rows of this wave's group
    const int gt_first = min(grp * TQ, ntok - 1), gt_last = min(grp * TQ + TQ - 1, ntok - 1);
    const int wp_last = p_first + gt_last;
    int wlo = window > 0 ? max(0, p_first + gt_first - window + 1) : 0;
    if (chunk > 0) wlo = max(wlo, (p_first + gt_first) - (p_first + gt_first) % chunk);

    // Q fragments (B operand of S^T): the 8 consecutive elements 32 s + 8 g4 of this lane's row
    v4u qfrag[RT];
    {
        const float* qrow = qf + ((size_t)t * H + (row_ok ? head : 0)) * (size_t)R;
#pragma unroll
        for (int s = 0; s < RT; ++s) {
            const int e0 = 32 * s + 8 * g4;
            float4 lo4 = make_float4(0.f, 0.f, 0.f, 0.f), hi4 = lo4;
            if (row_ok && e0 < R) {                      // R % 8 == 0: a piece of 8 is inside or outside as a whole
                lo4 = *(const float4*)(qrow + e0);
                hi4 = *(const float4*)(qrow + e0 + 4);
            }
            qfrag[s] = v4u{pack_bf2(lo4.x, lo4.y), pack_bf2(lo4.z, lo4.w), pack_bf2(hi4.x, hi4.y), pack_bf2(hi4.z, hi4.w)};
        }
    }
    v4f oacc[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) oacc[c] = v4f{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    if (sink && row_ok && sp == 0 && blockIdx.z == 0) {  // the sink's term: once per row, in its first key split
        m = sink[head];
        l = g4 == 0 ? 1.f : 0.f;                         // (l is a lane's share of the row's sum)
    }

    const int chunks_per_row = R / 8;                    // 16-byte pieces of a cache row (R % 8 == 0)
    // gridDim.z > 1 (decoding with few sequences): workgroup z takes every gridDim.z-th key tile and leaves an unnormalised
    // partial result; a second launch merges them
    const int Z = gridDim.z, z = blockIdx.z;
    // One tile = 32 consecutive positions inside ONE page (page % 32 == 0): a single block-table entry per tile.  The 16-byte
    // pieces of the NEXT tile are in flight (registers) while this tile is computed from LDS.
    constexpr int NCH = (BN * 4 * RT + 64 * NWV - 1) / (64 * NWV);
    v4u stage[NCH];
    auto issue = [&](int tile) {
        if (pooled && tile < nA) {                       // 32 blocks: every row through the page of its block's first position
#pragma unroll
            for (int i = 0; i < NCH; ++i) {
                const int q = tid + 64 * NWV * i, row = q % BN, cc = q / BN;
                stage[i] = v4u{0u, 0u, 0u, 0u};
                const int b = tile * BN + row;
                if (b < nb_last && cc < chunks_per_row) {
                    const int first = b * pool_block;
                    stage[i] = *(const v4u*)(pooled + ((size_t)bt[first / page] * block_rows + (size_t)((first % page) / pool_block)) * (size_t)R + cc * 8);
                }
            }
            return;
        }
        const int k0 = tile < nA ? tile * BN : kstart + (tile - nA) * BN;
        const bf16_t* base = pool + ((size_t)bt[k0 / page] * page + (size_t)(k0 % page)) * (size_t)R;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int q = tid + 64 * NWV * i, row = q % BN, cc = q / BN;
            stage[i] = v4u{0u, 0u, 0u, 0u};
            if (k0 + row <= p_last && cc < chunks_per_row) stage[i] = *(const v4u*)(base + (size_t)row * R + cc * 8);
        }
    };
    int ti = 0;
    if (z < nT) issue(z);
    for (int tile = z; tile < nT; tile += Z, ++ti) {
        const bool pre = tile < nA;                      // (block-uniform) a tile of keys behind the window
        const int k0 = pre ? tile * BN : kstart + (tile - nA) * BN;
        __syncthreads();                                 // the previous tile has been read
        // ---- the staged rows into LDS: row-major and transposed (lanes walk the rows: the 2-byte transposed writes of a
        //      wave fall into 32 different banks) ----
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int q = tid + 64 * NWV * i, row = q % BN, cc = q / BN;
            if (cc < 4 * RT) {
                const v4u d = stage[i];
                *(v4u*)(Ks + row * RS + cc * 8) = d;
                if (cc * 8 < 16 * CT) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        Vt[(cc * 8 + 2 * e) * VS + row] = (bf16_t)(d[e] & 0xffffu);
                        Vt[(cc * 8 + 2 * e + 1) * VS + row] = (bf16_t)(d[e] >> 16);
                    }
                }
            }
        }
        __syncthreads();
        if (tile + Z < nT) issue(tile + Z);
        // (wave-uniform; a tile below the wave's window may still hold kept first positions)
        if (!active || (ti % S) != sp || (!pre && (k0 > wp_last || (k0 + BN - 1 < wlo && k0 >= keep_first)))) continue;
        // the bias of this lane's eight (query, key) pairs: requested before the score product, added after it
        float bv[2][4];
        if (brow) {
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                for (int r = 0; r < 4; ++r) bv[mt][r] = brow[min(max(p_row - (k0 + 16 * mt + 4 * g4 + r), 0), bias_len - 1)];
        }
        // ---- S^T = K Q^T: two blocks of 16 keys; this lane gets keys 16 mt + 4 g4 + r of its own query row ----
        v4f sacc[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s = 0; s < RT; ++s) {
            if (s < s_lo || s >= s_hi) continue;         // (uniform) steps where every query is zero: a leading zero part, padding
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
                const v4u a = *(const v4u*)(Ks + (16 * mt + col) * RS + 32 * s + 8 * g4);
                sacc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, qfrag[s]),
                                                                   sacc[mt], 0, 0, 0);
            }
        }
        // ---- mask + online softmax (this lane: 8 keys of its query row; the other 24 sit in lanes ^16, ^32, ^48) ----
        float tmax = -INFINITY;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = k0 + 16 * mt + 4 * g4 + r;
                const bool vis = (pooled && pre) ? key < nb_row : (key <= p_row && (key >= lo_row || key < keep_first));
                if (brow) sacc[mt][r] += bv[mt][r];
                if (slopes) sacc[mt][r] -= slope * (float)(p_row - key);
                sacc[mt][r] = vis ? sacc[mt][r] : -INFINITY;
                tmax = fmaxf(tmax, sacc[mt][r]);
            }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
        const float mnew = fmaxf(m, tmax);
        const float msafe = mnew == -INFINITY ? 0.f : mnew;
        const float alpha = __expf(m - msafe);           // m = -inf: 0
        float psum = 0.f;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sacc[mt][r] = __expf(sacc[mt][r] - msafe);
                psum += sacc[mt][r];
            }
        l = l * alpha + psum;                            // (this lane's share; the four shares are added after the loop)
        m = mnew;
        if (__any(alpha != 1.0f)) {                      // (wave-uniform: the running maxima seldom move after the first tiles)
#pragma unroll
            for (int c = 0; c < CT; ++c) oacc[c] *= alpha;
        }
        // probabilities as B operand: k-slot (g4, e) <-> key 16 (e / 4) + 4 g4 + e % 4, i.e. exactly this lane's eight scores
        const v4u pb = {pack_bf2(sacc[0][0], sacc[0][1]), pack_bf2(sacc[0][2], sacc[0][3]),
                        pack_bf2(sacc[1][0], sacc[1][1]), pack_bf2(sacc[1][2], sacc[1][3])};
        // ---- O^T += C^T P^T ----
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const bf16_t* vrow = Vt + (16 * c + col) * VS + 4 * g4;
            const v2u a0 = *(const v2u*)vrow, a1 = *(const v2u*)(vrow + 16);
            const v4u a = {a0[0], a0[1], a1[0], a1[1]};
            oacc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, pb), oacc[c], 0, 0, 0);
        }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);

    // ---- merge the key splits (waves grp + G s, s = 1 .. S - 1, into wave grp) ----
    if (S > 1) {                                         // (block-uniform)
        __syncthreads();                                 // the last tile has been read: LDS becomes scratch
        float* ml = scratch + NWV * 8 * 64 * 4;          // [NWV][64][2], behind the accumulator exchange area
        if (active && sp > 0) {
            ml[(w * 64 + lane) * 2] = m;
            ml[(w * 64 + lane) * 2 + 1] = l;
        }
        __syncthreads();
        float f[NWV];
#pragma unroll
        for (int s = 0; s < NWV; ++s) f[s] = 0.f;
        if (active && sp == 0) {
            float M = m;
            for (int s = 1; s < S; ++s) M = fmaxf(M, ml[((grp + G * s) * 64 + lane) * 2]);
            const float Ms = M == -INFINITY ? 0.f : M;
            f[0] = __expf(m - Ms);
            float L = f[0] * l;
            for (int s = 1; s < S; ++s) {
                f[s] = __expf(ml[((grp + G * s) * 64 + lane) * 2] - Ms);
                L += f[s] * ml[((grp + G * s) * 64 + lane) * 2 + 1];
            }
            l = L;
            m = M;                                       // (what a cross-workgroup merge reads)
        }
        // accumulators through LDS, MB column tiles per exchange (two barriers each)
        constexpr int MB = CT < 8 ? CT : 8;
#pragma unroll
        for (int c0 = 0; c0 < CT; c0 += MB) {
            __syncthreads();
            if (active && sp > 0) {
#pragma unroll
                for (int j = 0; j < MB; ++j)
                    if (c0 + j < CT) *(v4f*)(scratch + ((w * MB + j) * 64 + lane) * 4) = oacc[c0 + j];
            }
            __syncthreads();
            if (active && sp == 0) {
#pragma unroll
                for (int j = 0; j < MB; ++j)
                    if (c0 + j < CT) {
                        v4f a = oacc[c0 + j] * f[0];
                        for (int s = 1; s < S; ++s) a += *(const v4f*)(scratch + (((grp + G * s) * MB + j) * 64 + lane) * 4) * f[s];
                        oacc[c0 + j] = a;
                    }
            }
        }
    }
    if (!row_ok || sp != 0) return;
    if (Z > 1) {                                         // partial result of this key split: [z][t][h][rank] and (m, l)
        const size_t rowi = ((size_t)z * n_tokens + t) * H + head;
        if (g4 == 0) {
            part_ml[rowi * 2] = m;
            part_ml[rowi * 2 + 1] = l;
        }
        float* po = part_o + rowi * (size_t)rank;
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int c0 = 16 * c + 4 * g4;
            if (c0 < rank) *(v4f*)(po + c0) = oacc[c];
        }
        return;
    }
    const float inv = 1.0f / l;
    bf16_t* o = out + ((size_t)t * H + head) * (size_t)rank;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int c0 = 16 * c + 4 * g4;
        if (c0 < rank) {                                 // rank % 8 == 0: the four values are all inside
            const v2u v = {pack_bf2(oacc[c][0] * inv, oacc[c][1] * inv), pack_bf2(oacc[c][2] * inv, oacc[c][3] * inv)};
            *(v2u*)(o + c0) = v;
        }
    }
}

// ---- plain rows (causal or windowed, nothing else on the scores) of exact sizes: R = 32 RT a multiple of 64, rank = 16 CT a multiple of 64 ----
// The kernel above stages a key tile through registers and writes it twice, the second time transposed in 2-byte pieces; at 576-wide rows
// that and 74 KB of code were its time (143 TFLOP/s in a prompt, 47 us for a step of 100 positions).  Here a tile is copied straight into
// LDS as it lies in memory (32 rows of one page are contiguous), once, the 16-byte pieces of a row permuted by the row's number, two
// tiles in turn with one barrier each; K is read from it row by row and V through the transposing read (ds_read_b64_tr_b16).  Eight waves
// of 16 query rows (one token of 16 heads, or several of fewer).  Bound by the LDS reads: a wave reads the whole tile for its 16 rows.
// Measured (MI355X): 8 prompts of 1024, 16 heads, 576 / 512: 1004 -> 335 us; 512 / 512: 973 -> 315 us; 256 / 128, 32 heads on 8 pools: 484 -> 242 us; steps
// of 64 sequences at 100 / 1000 / 4000 positions, 576 / 512: 41 / 69 / 200 -> 15 / 31 / 71 us, 256 / 128, 16 heads on 4 pools: 15 / 45 / 135 -> 13 / 26 / 95 us.
constexpr int RW = 8;
typedef short s4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4* lds_s4;
typedef __attribute__((address_space(3))) void* lds_ptr;

// (eight neighbouring rows: eight different pieces for the key reads; four: four different pairs for the transposing value reads)
__device__ __forceinline__ int row_turn(int row) { return ((row & 3) << 1) | ((row >> 2) & 1); }

// S0: every query is zero before element 32 S0
template <int RT, int CT, int S0>
__global__ __launch_bounds__(64 * RW, RT + CT > 24 ? 2 : 4) void latent_rows_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ qf, const bf16_t* __restrict__ pool_base, const int32_t* __restrict__ block_table,
    int table_stride, const int32_t* __restrict__ pos, const int32_t* __restrict__ tiles, int n_tiles, int window, int H, int page, int HP, int TQ,
    float* __restrict__ part_o, float* __restrict__ part_ml, int n_tokens, int per, int64_t pool_stride) {
    constexpr int R = 32 * RT, RANK = 16 * CT, PPR = R / 8, TILE = BN * R * 2, NJ = (BN * PPR / 64 + RW - 1) / RW;
    static_assert(R % 64 == 0 && RANK % 64 == 0, "");
    __shared__ __attribute__((aligned(128))) unsigned char buf[2 * TILE];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6) & (RW - 1);
    const int col = lane & 15, g4 = lane >> 4;
    const int32_t* tl = tiles + 3 * (n_tiles - 1 - (int)blockIdx.x);            // (a sequence's longest first)
    const int slot = __builtin_amdgcn_readfirstlane(tl[0]), t0 = __builtin_amdgcn_readfirstlane(tl[1]), ntok = __builtin_amdgcn_readfirstlane(tl[2]);
    const int gpp = (per + 15) / 16, pool_id = blockIdx.y / gpp;
    const int h0 = pool_id * per + (blockIdx.y % gpp) * 16, h_end = pool_id * per + per;
    const bf16_t* __restrict__ pool = pool_base + (size_t)pool_id * (size_t)pool_stride;
    const int32_t* bt = block_table + (size_t)slot * table_stride;
    const bool active = w * TQ < ntok;                                          // this wave has tokens
    const int tok_in = w * TQ + col / HP, head = h0 + col % HP;
    const bool row_ok = tok_in < ntok && head < h_end;
    const int t = t0 + min(tok_in, ntok - 1);
    // (tokens of a tile are consecutive positions)
    const int p_first = __builtin_amdgcn_readfirstlane(pos[t0]), p_last = p_first + ntok - 1, p_row = p_first + (t - t0);
    const int lo_row = window > 0 ? max(0, p_row - window + 1) : 0;
    const int kstart = window > 0 ? max(0, p_first - window + 1) / BN * BN : 0;
    const int nT = (p_last - kstart) / BN + 1;
    const int wp_last = p_first + min(w * TQ + TQ - 1, ntok - 1), wlo = window > 0 ? max(0, p_first + w * TQ - window + 1) : 0;

    // copies: piece i = 64 (w + RW j) + lane of the tile's BN x PPR, to where it lies; it carries piece (i % PPR) ^ row_turn(row) of its row
    // (worked out anew for every tile: kept across the loop, the offsets would be spilled)
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)buf);
    auto copy = [&](int k0, int page_id, int which) __attribute__((always_inline)) {
        const bf16_t* base = pool + ((size_t)page_id * page + (size_t)(k0 % page)) * (size_t)R;
        const int left = p_last - k0;                                           // rows past the last position repeat it
        int me = lane;
        asm volatile("" : "+v"(me));
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            if (w + RW * j < BN * PPR / 64) {
                const int i = 64 * (w + RW * j) + me, row = i / PPR;
                const unsigned off = (unsigned)(min(row, left) * PPR + ((i - row * PPR) ^ row_turn(row))) * 16u;
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base),
                             "s"(lds0 + which * TILE + (w + RW * j) * 1024)
                             : "memory");
            }
    };
    // the query row, whole before anything is rounded: rounded under its condition, every piece waited for the one before
    float4 q[RT][2];
    {
        const float* qrow = qf + ((size_t)t * H + (row_ok ? head : h0)) * (size_t)R + 8 * g4;
#pragma unroll
        for (int s = S0; s < RT; ++s) {
            q[s][0] = *(const float4*)(qrow + 32 * s);
            q[s][1] = *(const float4*)(qrow + 32 * s + 4);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    const int Z = gridDim.z, z = blockIdx.z;
    auto page_of = [&](int tile) __attribute__((always_inline)) { return bt[(kstart + min(tile, nT - 1) * BN) / page]; };
    int next_page = 0;
    if (z < nT) {
        copy(kstart + z * BN, __builtin_amdgcn_readfirstlane(page_of(z)), 0);
        next_page = page_of(z + Z);
    }
    v4u qfrag[RT];
    const unsigned kept = row_ok ? ~0u : 0u;
#pragma unroll
    for (int s = S0; s < RT; ++s)
        qfrag[s] = v4u{pack_bf2(q[s][0].x, q[s][0].y), pack_bf2(q[s][0].z, q[s][0].w), pack_bf2(q[s][1].x, q[s][1].y), pack_bf2(q[s][1].z, q[s][1].w)} & kept;
    v4f oacc[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) oacc[c] = v4f{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    // K: key 16 mt + col, pieces 4 s + g4;  V: keys 4 g4 + col / 4 (+ 16), pieces 2 c + (col & 3) / 2, half col & 1
    const int k_at = col * (R * 2), k_odd[2] = {(g4 ^ row_turn(col)) << 4, ((4 + g4) ^ row_turn(col)) << 4};
    const int vk = 4 * g4 + (col >> 2), v_at = vk * (R * 2) + (col & 1) * 8;
    int v_turn[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) v_turn[c] = ((2 * c + ((col & 3) >> 1)) ^ row_turn(vk)) << 4;
    int which = 0;
    for (int tile = z; tile < nT; tile += Z) {
        const int k0 = kstart + tile * BN;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                                           // this tile has landed; the other half has been read by everyone
        asm volatile("" ::: "memory");
        const unsigned char* T = buf + which * TILE;
        which ^= 1;
        if (tile + Z < nT) {
            copy(k0 + Z * BN, __builtin_amdgcn_readfirstlane(next_page), which);
            next_page = page_of(tile + 2 * Z);
        }
        if (!active || k0 > wp_last || k0 + BN - 1 < wlo) continue;             // (wave-uniform)
        // operands are requested a few products ahead (the order is the source's: left alone, the compiler reads each one just before use)
        v4f sacc[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
        constexpr int KN = 2 * (RT - S0), RING = RT + CT >= 50 ? 4 : RT + CT > 24 ? 5 : 6;
        v4u ring[RING];
        auto read = [&](int u) __attribute__((always_inline)) {                 // operand u: the KN of the keys, then the CT of the values
            if (u < KN) {
                const int s = S0 + (u >> 1);
                ring[u % RING] = *(const v4u*)(T + k_at + 16 * (u & 1) * (R * 2) + (s >> 1) * 128 + k_odd[s & 1]);
            } else if (u < KN + CT) {
                const int c = u - KN;
                const unsigned char* v = T + v_at + (c >> 2) * 128 + v_turn[c & 3];
                const v2u a0 = __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)v));
                const v2u a1 = __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(v + 16 * (R * 2))));
                ring[u % RING] = v4u{a0[0], a0[1], a1[0], a1[1]};
            }
        };
#pragma unroll
        for (int u = 0; u < RING - 1; ++u) read(u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < KN; ++u) {
            read(u + RING - 1);
            __builtin_amdgcn_sched_barrier(0);
            sacc[u & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, ring[u % RING]), __builtin_bit_cast(bf8, qfrag[S0 + (u >> 1)]),
                                                                  sacc[u & 1], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        // this lane: keys k0 + 16 mt + 4 g4 + r of its query row (the other 24 sit in lanes ^16, ^32, ^48)
        float tmax = -INFINITY;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = k0 + 16 * mt + 4 * g4 + r;
                sacc[mt][r] = key <= p_row && key >= lo_row ? sacc[mt][r] : -INFINITY;
                tmax = fmaxf(tmax, sacc[mt][r]);
            }
        const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
        tmax = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
        const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
        tmax = fmaxf(__uint_as_float(y[0]), __uint_as_float(y[1]));
        const float mnew = fmaxf(m, tmax);
        const float msafe = mnew == -INFINITY ? 0.f : mnew;
        const float alpha = __expf(m - msafe);                                  // m = -inf: 0
        float psum = 0.f;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sacc[mt][r] = __expf(sacc[mt][r] - msafe);
                psum += sacc[mt][r];
            }
        l = l * alpha + psum;                                                   // (this lane's share; the four shares are added after the loop)
        m = mnew;
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int c = 0; c < CT; ++c) oacc[c] *= alpha;
        }
        // probabilities as B operand: k-slot (g4, e) <-> key 16 (e / 4) + 4 g4 + e % 4, i.e. exactly this lane's eight scores
        const v4u pb = {pack_bf2(sacc[0][0], sacc[0][1]), pack_bf2(sacc[0][2], sacc[0][3]), pack_bf2(sacc[1][0], sacc[1][1]),
                        pack_bf2(sacc[1][2], sacc[1][3])};
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            read(KN + c + RING - 1);
            __builtin_amdgcn_sched_barrier(0);
            oacc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, ring[(KN + c) % RING]), __builtin_bit_cast(bf8, pb), oacc[c], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    int me = lane;                                                              // (as above: the row's place is worked out again)
    asm volatile("" : "+v"(me));
    const int my_tok = w * TQ + (me & 15) / HP, my_head = h0 + (me & 15) % HP;
    if (my_tok >= ntok || my_head >= h_end) return;
    const size_t my_row = (size_t)(t0 + my_tok) * H + my_head;
    const int c4 = 4 * (me >> 4);
    if (Z > 1) {                                                                // partial result of this key split: [z][t][h][rank] and (m, l)
        const size_t rowi = (size_t)z * n_tokens * H + my_row;
        if (c4 == 0) {
            part_ml[rowi * 2] = m;
            part_ml[rowi * 2 + 1] = l;
        }
        float* po = part_o + rowi * RANK + c4;
#pragma unroll
        for (int c = 0; c < CT; ++c) *(v4f*)(po + 16 * c) = oacc[c];
        return;
    }
    const float inv = 1.0f / l;
    bf16_t* o = out + my_row * RANK + c4;
#pragma unroll
    for (int c = 0; c < CT; ++c)
        *(v2u*)(o + 16 * c) = v2u{pack_bf2(oacc[c][0] * inv, oacc[c][1] * inv), pack_bf2(oacc[c][2] * inv, oacc[c][3] * inv)};
}

// ---- the same rows for steps: one token per tile ----------------------------------------------------------------------------------------------
// With one token a single wave of the kernel above has queries, and a step waits for it: 64 keys took 4 us.  Here four waves share the token:
// rounds of 64 keys, copied as above (two rounds in turn); a wave scores 16 of the keys (its rows of K only), the maximum and the
// probabilities of a round meet in LDS, and a wave multiplies them with its quarter of the value columns.  Bound by latency at short contexts, by
// HBM at long ones.
// Its chain is the launch: tiles, positions and pages, the queries, the first keys.  The queries are requested first, all of them, and rounded
// before the keys' copies are (rounded under their condition, each of the 18 pairs waited for the one before; rounded behind the copies, the wait
// is for those too); then two rounds are in flight, the next two pages with them: in a step of 64 sequences at 50 - 150 positions 576 / 512 16.5 ->
// 13.4 us and 512 / 512 15.1 -> 12.3 (13.7 and 12.4 with one round ahead), 16 sequences at 100 - 220 of 256 / 128 8.7 -> 7.2.
// Measured alone, its queries in the caches (16 heads, 576 / 512, best split each, kernel above -> this one and the merge below): 64 sequences at 128 / 1000 /
// 2000 positions 15 -> 12.5 / 31 -> 26 / 44 -> 36 us, 16 at 1000 25 -> 18, one at 300 / 2000 17 -> 14.5 / 28 -> 17.5; 256 / 128, 16 heads on 4 pools, 16
// sequences at 1000: 15 -> 10.8 us.  The queries' early requests are for a step, whose queries come from memory: alone, short contexts lose 0.5 us by them (64 at 128
// 12 -> 12.5, one at 300 / 2000 14 -> 14.5 / 17 -> 17.5), inside a step of one sequence at 300 / 2000 positions 576 / 512 takes 16.4 -> 12.7 / 16.5 -> 13.1 us and
// 512 / 512 14.8 -> 11.8 / 15.2 -> 12.1.
constexpr int SW = 4, SN = 64;       // waves, keys of a round
template <int RT, int CT, int S0>
__global__ __launch_bounds__(64 * SW, 1) void latent_step_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ qf, const bf16_t* __restrict__ pool_base, const int32_t* __restrict__ block_table,
    int table_stride, const int32_t* __restrict__ pos, const int32_t* __restrict__ tiles, int window, int H, int page, int HP,
    float* __restrict__ part_o, float* __restrict__ part_ml, int n_tokens, int per, int64_t pool_stride) {
    constexpr int R = 32 * RT, RANK = 16 * CT, PPR = R / 8, TILE = SN * R * 2, NJ = 32 * PPR / 64 / SW, WC = CT / SW;
    static_assert(32 * PPR % (64 * SW) == 0 && CT % SW == 0 && 2 * TILE + 4096 <= 160 * 1024, "");
    __shared__ __attribute__((aligned(128))) unsigned char buf[2 * TILE];
    __shared__ float tops[SW][16], sums[SW][16];
    __shared__ uint2 probs[SW][64];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6) & (SW - 1);
    const int col = lane & 15, g4 = lane >> 4;
    const int32_t* tl = tiles + 3 * (int)blockIdx.x;
    const int slot = __builtin_amdgcn_readfirstlane(tl[0]), t = __builtin_amdgcn_readfirstlane(tl[1]);
    const int gpp = (per + 15) / 16, pool_id = blockIdx.y / gpp;
    const int h0 = pool_id * per + (blockIdx.y % gpp) * 16, h_end = pool_id * per + per;
    const bf16_t* __restrict__ pool = pool_base + (size_t)pool_id * (size_t)pool_stride;
    const int32_t* bt = block_table + (size_t)slot * table_stride;
    const int head = h0 + col;
    const bool row_ok = col < HP && head < h_end;
    // the query row, whole before anything is rounded: rounded under its condition, every piece waited for the one before
    float4 q[RT][2];
    {
        const float* qrow = qf + ((size_t)t * H + (row_ok ? head : h0)) * (size_t)R + 8 * g4;
#pragma unroll
        for (int s = S0; s < RT; ++s) {
            q[s][0] = *(const float4*)(qrow + 32 * s);
            q[s][1] = *(const float4*)(qrow + 32 * s + 4);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    const int p_row = __builtin_amdgcn_readfirstlane(pos[t]), lo_row = window > 0 ? max(0, p_row - window + 1) : 0;
    const int kstart = lo_row / BN * BN, nT = (p_row - kstart) / SN + 1, last_half = (p_row - kstart) / BN;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)buf);
    // piece i = 64 (w + SW j) + lane of a half round's BN x PPR, permuted by the row's number; halves behind the last position repeat its half,
    // rows behind it its row
    auto copy_half = [&](int half, int page_id, int at) __attribute__((always_inline)) {
        const int k0 = kstart + min(half, last_half) * BN;
        const bf16_t* base = pool + ((size_t)page_id * page + (size_t)(k0 % page)) * (size_t)R;
        const int left = p_row - k0;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int i = 64 * (w + SW * j) + lane, row = i / PPR;
            const unsigned off = (unsigned)(min(row, left) * PPR + ((i - row * PPR) ^ row_turn(row))) * 16u;
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base),
                         "s"(lds0 + at + (w + SW * j) * 1024)
                         : "memory");
        }
    };
    const int Z = gridDim.z, z = blockIdx.z;
    auto page_of = [&](int half) __attribute__((always_inline)) { return bt[(kstart + min(half, last_half) * BN) / page]; };
    auto copy = [&](int round, int which, int page_a, int page_b) __attribute__((always_inline)) {
        copy_half(2 * round, __builtin_amdgcn_readfirstlane(page_a), which * TILE);
        copy_half(2 * round + 1, __builtin_amdgcn_readfirstlane(page_b), which * TILE + TILE / 2);
    };
    const int a0 = page_of(2 * z), b0 = page_of(2 * z + 1), a1 = page_of(2 * (z + Z)), b1 = page_of(2 * (z + Z) + 1);
    int next_a = page_of(2 * (z + 2 * Z)), next_b = page_of(2 * (z + 2 * Z) + 1);
    __builtin_amdgcn_sched_barrier(0);
    v4u qfrag[RT];
    const unsigned kept = row_ok ? ~0u : 0u;
#pragma unroll
    for (int s = S0; s < RT; ++s)
        qfrag[s] = v4u{pack_bf2(q[s][0].x, q[s][0].y), pack_bf2(q[s][0].z, q[s][0].w), pack_bf2(q[s][1].x, q[s][1].y), pack_bf2(q[s][1].z, q[s][1].w)} & kept;
#pragma unroll
    for (int s = S0; s < RT; ++s) asm volatile("" : "+v"(qfrag[s]));               // (before the copies: behind them its wait would be for them too)
    if (z < nT) copy(z, 0, a0, b0);
    if (z + Z < nT) copy(z + Z, 1, a1, b1);
    v4f oacc[WC];
#pragma unroll
    for (int c = 0; c < WC; ++c) oacc[c] = v4f{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    // K: key 16 w + col of the round, pieces 4 s + g4;  V: keys 4 g4 + col / 4 (+ 16, + 32, + 48), column tile WC w + c
    const int k_at = (16 * w + col) * (R * 2), k_odd[2] = {(g4 ^ row_turn(col)) << 4, ((4 + g4) ^ row_turn(col)) << 4};
    const int vk = 4 * g4 + (col >> 2);
    int v_at[WC];
#pragma unroll
    for (int c = 0; c < WC; ++c) {
        const int ct = WC * w + c;
        v_at[c] = vk * (R * 2) + (col & 1) * 8 + (ct >> 2) * 128 + (((2 * (ct & 3) + ((col & 3) >> 1)) ^ row_turn(vk)) << 4);
    }
    int which = 0;
    for (int round = z; round < nT; round += Z) {
        if (round + Z < nT) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NJ) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                                           // these keys have landed
        asm volatile("" ::: "memory");
        const unsigned char* T = buf + which * TILE;
        v4f sacc[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
        v4u kf[RT];
#pragma unroll
        for (int s = S0; s < RT; ++s) kf[s] = *(const v4u*)(T + k_at + (s >> 1) * 128 + k_odd[s & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = S0; s < RT; ++s)
            sacc[s & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, kf[s]), __builtin_bit_cast(bf8, qfrag[s]), sacc[s & 1], 0, 0, 0);
        float p[4], tmax = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {                                           // this lane: keys 16 w + 4 g4 + r of the round
            const int key = kstart + round * SN + 16 * w + 4 * g4 + r;
            p[r] = key <= p_row && key >= lo_row ? sacc[0][r] + sacc[1][r] : -INFINITY;
            tmax = fmaxf(tmax, p[r]);
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
        if (g4 == 0) tops[w][col] = tmax;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        // the value operands do not wait for the probabilities
        v4u vf[WC][2];
#pragma unroll
        for (int c = 0; c < WC; ++c)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const unsigned char* v = T + v_at[c] + b * 32 * (R * 2);
                const v2u a0 = __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)v));
                const v2u a1 = __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(v + 16 * (R * 2))));
                vf[c][b] = v4u{a0[0], a0[1], a1[0], a1[1]};
            }
        float mnew = m;
#pragma unroll
        for (int o = 0; o < SW; ++o) mnew = fmaxf(mnew, tops[o][col]);
        const float msafe = mnew == -INFINITY ? 0.f : mnew;
        const float alpha = __expf(m - msafe);                                  // m = -inf: 0
        float psum = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[r] = __expf(p[r] - msafe);
            psum += p[r];
        }
        l = l * alpha + psum;                                                   // (this lane's share)
        m = mnew;
        probs[w][lane] = make_uint2(pack_bf2(p[0], p[1]), pack_bf2(p[2], p[3]));
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int c = 0; c < WC; ++c) oacc[c] *= alpha;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (round + 2 * Z < nT) {                                               // (everyone has read these)
            copy(round + 2 * Z, which, next_a, next_b);
            next_a = page_of(2 * (round + 3 * Z));
            next_b = page_of(2 * (round + 3 * Z) + 1);
        }
        which ^= 1;
#pragma unroll
        for (int b = 0; b < 2; ++b) {                                           // 32 keys: k-slot (g4, e) <-> key 16 (e / 4) + 4 g4 + e % 4
            const uint2 p0 = probs[2 * b][lane], p1 = probs[2 * b + 1][lane];
            const v4u pb = {p0.x, p0.y, p1.x, p1.y};
#pragma unroll
            for (int c = 0; c < WC; ++c)
                oacc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, vf[c][b]), __builtin_bit_cast(bf8, pb), oacc[c], 0, 0, 0);
        }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (g4 == 0) sums[w][col] = l;
    __syncthreads();
    l = (sums[0][col] + sums[1][col]) + (sums[2][col] + sums[3][col]);
    if (!row_ok) return;
    const size_t my_row = (size_t)t * H + head;
    const int c0 = 16 * WC * w + 4 * g4;
    if (Z > 1) {
        const size_t rowi = (size_t)z * n_tokens * H + my_row;
        if (w == 0 && g4 == 0) {
            part_ml[rowi * 2] = m;
            part_ml[rowi * 2 + 1] = l;
        }
        float* po = part_o + rowi * RANK + c0;
#pragma unroll
        for (int c = 0; c < WC; ++c) *(v4f*)(po + 16 * c) = oacc[c];
        return;
    }
    const float inv = 1.0f / l;
    bf16_t* o = out + my_row * RANK + c0;
#pragma unroll
    for (int c = 0; c < WC; ++c)
        *(v2u*)(o + 16 * c) = v2u{pack_bf2(oacc[c][0] * inv, oacc[c][1] * inv), pack_bf2(oacc[c][2] * inv, oacc[c][3] * inv)};
}

// out[t, h] = sum_z e^(m_z - M) o_z / sum_z e^(m_z - M) l_z   (one workgroup per (token, head); rank a multiple of 4, at most 64 splits: lane z of
// every wave weighs split z, a thread adds four columns, four splits requested at a time)
__global__ __launch_bounds__(128) void latent_attention_merge_kernel(bf16_t* __restrict__ out, const float* __restrict__ part_o,
                                                                     const float* __restrict__ part_ml, int Z, int rows, int rank) {
    const size_t r = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const float2 ml = lane < Z ? *(const float2*)(part_ml + ((size_t)lane * rows + r) * 2) : make_float2(-INFINITY, 0.f);
    const float M = wave_max(ml.x), e = lane < Z ? __expf(ml.x - M) : 0.f;
    const float inv = 1.0f / wave_sum(e * ml.y);
    for (int c = threadIdx.x * 4; c < rank; c += 128 * 4) {
        const float* po = part_o + r * (size_t)rank + c;
        const size_t step = (size_t)rows * rank;
        v4f a = v4f{0.f, 0.f, 0.f, 0.f};
        for (int z = 0; z < Z; z += 4) {
            v4f v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = *(const v4f*)(po + (size_t)min(z + i, Z - 1) * step);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (z + i < Z) a += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(e), z + i)) * v[i];
        }
        *(v2u*)(out + r * (size_t)rank + c) = v2u{pack_bf2(a[0] * inv, a[1] * inv), pack_bf2(a[2] * inv, a[3] * inv)};
    }
}

struct Geometry {
    int HP, TQ;
};
Geometry geometry(int H) {
    int hp = 1;
    while (hp < H && hp < 16) hp <<= 1;
    return {hp, 16 / hp};
}
}  // namespace

// Tokens of one sequence a work tile may hold, for `heads` heads (the host cuts a step's portions into tiles of this size).
extern "C" int qsv_latent_attention_tile_tokens(int heads) {
    if (heads <= 0) return 0;
    return NWV * geometry(heads).TQ;
}

// 1 if the matrix-core kernel takes these sizes (bfloat16 storage only), else 0 and the caller uses the wave kernel.
extern "C" int qsv_latent_attention_mfma_ok(int rank, int row_width, int dtype) {
    return dtype == QSV_BF16 && rank % 8 == 0 && row_width % 8 == 0 && row_width <= 576 && rank <= 512 && rank >= 8;   // (and page % 32 == 0)
}

// tiles: int32 [n_tiles, 3] = (sequence slot, first flat token index, tokens <= qsv_latent_attention_tile_tokens(heads)).
// key_splits > 1: every tile's keys are cut over that many workgroups (for steps with few tiles: decoding); then part_o
// (float [key_splits, n_tokens, H, rank]) and part_ml (float [key_splits, n_tokens, H, 2]) are workspace.
extern "C" int qsv_latent_attention_mfma(void* out, const float* qf, const void* pool, const int32_t* block_table,
                                         int table_stride, const int32_t* pos, const int32_t* tiles, int n_tiles, int window,
                                         int H, int rank, int R, int page, int key_splits, float* part_o, float* part_ml,
                                         int n_tokens, int q_first, int heads_per_pool, int64_t pool_stride, int chunk,
                                         const float* bias, int bias_len, int keep_first, const float* sink, const void* pooled,
                                         int64_t pooled_stride, int pool_block, int block_rows, const float* slopes, void* stream) {
    QSV_REQUIRE(keep_first >= 0 && (!keep_first || (window > 0 && !chunk)),
                "qsv_latent_attention_mfma: %d kept first positions need a window and no chunks", keep_first);
    QSV_REQUIRE(!pooled || (window > 0 && !chunk && !bias && !keep_first && pool_block > 0 && block_rows > 0 && pooled_stride >= 0 &&
                            (int64_t)block_rows * pool_block >= page),
                "qsv_latent_attention_mfma: pooled blocks of %d positions, %d rows per page of %d", pool_block, block_rows, page);
    QSV_REQUIRE(chunk >= 0 && (!bias || bias_len > 0), "qsv_latent_attention_mfma: chunk %d, bias table of %d distances", chunk, bias_len);
    QSV_REQUIRE(out && qf && pool && block_table && pos && tiles, "qsv_latent_attention_mfma: null argument");
    QSV_REQUIRE(qsv_latent_attention_mfma_ok(rank, R, QSV_BF16) && R >= rank && H > 0 && page > 0 && page % BN == 0 && window >= 0 && n_tiles >= 0,
                "qsv_latent_attention_mfma: sizes not supported (rank %d, row %d)", rank, R);
    QSV_REQUIRE(!slopes || !pooled, "qsv_latent_attention_mfma: distance slopes with pooled blocks");
    if (n_tiles == 0) return QSV_OK;
    QSV_REQUIRE(heads_per_pool > 0 && H % heads_per_pool == 0 && pool_stride >= 0,
                "qsv_latent_attention_mfma: %d heads over pools of %d", H, heads_per_pool);
    const Geometry g = geometry(heads_per_pool);
    QSV_REQUIRE(key_splits >= 1 && key_splits <= 64 && (key_splits == 1 || (part_o && part_ml && n_tokens > 0)),
                "qsv_latent_attention_mfma: key splits without workspace");
    const dim3 grid(n_tiles, (H / heads_per_pool) * ((heads_per_pool + 15) / 16), key_splits), block(64 * NWV);
    QSV_REQUIRE(q_first >= 0 && q_first < R, "qsv_latent_attention_mfma: first query element %d of %d", q_first, R);
    const int rt = (R + 31) / 32, ct = (rank + 15) / 16;
    const int s_lo = q_first / 32, s_hi = rt;
#define QSV_MFMA(RT, CT)                                                                                                     \
    do {                                                                                                                     \
        size_t lds = (size_t)(BN * (32 * RT + 8) + 16 * CT * VS) * 2;                                                        \
        const size_t need = (size_t)NWV * 64 * (8 * 4 + 2) * 4;       /* merge scratch */                                                                       \
        if (lds < need) lds = need;                                                                                          \
        if (lds > 64 * 1024) {   /* above the default limit of dynamic LDS: raise it for this kernel */                        \
            const hipError_t e = hipFuncSetAttribute((const void*)latent_attention_mfma_kernel<RT, CT>,                      \
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                  \
            QSV_REQUIRE(e == hipSuccess, "qsv_latent_attention_mfma: %s", hipGetErrorString(e));                             \
        }                                                                                                                    \
        hipLaunchKernelGGL((latent_attention_mfma_kernel<RT, CT>), grid, block, lds, (hipStream_t)stream, (bf16_t*)out, qf,  \
                           (const bf16_t*)pool, block_table, table_stride, pos, tiles, window, H, rank, R, page, g.HP, g.TQ, \
                           part_o, part_ml, n_tokens, s_lo, s_hi, heads_per_pool, pool_stride, chunk, bias, bias_len,         \
                           keep_first, sink, (const bf16_t*)pooled, pooled_stride, pool_block, block_rows, slopes);                       \
    } while (0)
    if (rt <= 4 && ct <= 8) QSV_MFMA(4, 8);
    else if (rt <= 6 && ct <= 12) QSV_MFMA(6, 12);
    else if (rt <= 8 && ct <= 8) QSV_MFMA(8, 8);
    else if (rt <= 10 && ct <= 16) QSV_MFMA(10, 16);
    else QSV_MFMA(18, 32);
#undef QSV_MFMA
    if (key_splits > 1) {
        const int rc = qsv_launch_status("qsv_latent_attention_mfma");
        if (rc != QSV_OK) return rc;
        hipLaunchKernelGGL(latent_attention_merge_kernel, dim3(n_tokens * H), dim3(128), 0, (hipStream_t)stream, (bf16_t*)out,
                           part_o, part_ml, key_splits, n_tokens * H, rank);
    }
    return qsv_launch_status("qsv_latent_attention_mfma");
}

// The plain-rows kernel: 1 if it takes these sizes, tokens per tile, and the launch (arguments as above; no option changes the scores).
extern "C" int qsv_latent_rows_ok(int rank, int row_width, int page, int dtype) {
    return dtype == QSV_BF16 && page > 0 && page % BN == 0 &&
           ((row_width == 576 && rank == 512) || (row_width == 512 && rank == 512) || (row_width == 256 && rank == 128));
}
extern "C" int qsv_latent_rows_tile_tokens(int heads) { return heads <= 0 ? 0 : RW * geometry(heads).TQ; }
extern "C" int qsv_latent_rows(void* out, const float* qf, const void* pool, const int32_t* block_table, int table_stride, const int32_t* pos,
                               const int32_t* tiles, int n_tiles, int window, int H, int rank, int R, int page, int key_splits, float* part_o,
                               float* part_ml, int n_tokens, int q_first, int heads_per_pool, int64_t pool_stride, void* stream) {
    QSV_REQUIRE(out && qf && pool && block_table && pos && tiles && n_tiles >= 0 && H > 0 && window >= 0, "qsv_latent_rows: bad arguments");
    QSV_REQUIRE(qsv_latent_rows_ok(rank, R, page, QSV_BF16), "qsv_latent_rows: sizes not supported (rank %d, row %d, page %d)", rank, R, page);
    QSV_REQUIRE(((uintptr_t)pool | (uintptr_t)qf) % 16 == 0 && pool_stride % 8 == 0, "qsv_latent_rows: rows start on 16 bytes");
    if (n_tiles == 0) return QSV_OK;
    QSV_REQUIRE(heads_per_pool > 0 && H % heads_per_pool == 0 && pool_stride >= 0, "qsv_latent_rows: %d heads over pools of %d", H, heads_per_pool);
    QSV_REQUIRE(key_splits >= 1 && key_splits <= 64 && (key_splits == 1 || (part_o && part_ml && n_tokens > 0)),
                "qsv_latent_rows: key splits without workspace");
    QSV_REQUIRE(q_first >= 0 && q_first < R, "qsv_latent_rows: first query element %d of %d", q_first, R);
    const Geometry g = geometry(heads_per_pool);
    const dim3 grid(n_tiles, (H / heads_per_pool) * ((heads_per_pool + 15) / 16), key_splits), block(64 * RW);
#define QSV_ROWS(RT, CT, S0)                                                                                                                   \
    hipLaunchKernelGGL((latent_rows_kernel<RT, CT, S0>), grid, block, 0, (hipStream_t)stream, (bf16_t*)out, qf, (const bf16_t*)pool,             \
                       block_table, table_stride, pos, tiles, n_tiles, window, H, page, g.HP, g.TQ, part_o, part_ml, n_tokens, heads_per_pool,   \
                       pool_stride)
#define QSV_STEP_ROWS(RT, CT, S0)                                                                                                              \
    hipLaunchKernelGGL((latent_step_kernel<RT, CT, S0>), grid, dim3(64 * SW), 0, (hipStream_t)stream, (bf16_t*)out, qf, (const bf16_t*)pool,   \
                       block_table, table_stride, pos, tiles, window, H, page, g.HP, part_o, part_ml, n_tokens, heads_per_pool, pool_stride)
    if (n_tiles == n_tokens) {                                                 // (every tile holds a token, so each holds one)
        if (R == 576) QSV_STEP_ROWS(18, 32, 0);
        else if (R == 512) QSV_STEP_ROWS(16, 32, 0);
        else if (q_first >= 128) QSV_STEP_ROWS(8, 8, 4);
        else QSV_STEP_ROWS(8, 8, 0);
    } else if (R == 576) QSV_ROWS(18, 32, 0);
    else if (R == 512) QSV_ROWS(16, 32, 0);
    else if (q_first >= 128) QSV_ROWS(8, 8, 4);
    else QSV_ROWS(8, 8, 0);
#undef QSV_ROWS
#undef QSV_STEP_ROWS
    if (key_splits > 1) {
        const int rc = qsv_launch_status("qsv_latent_rows");
        if (rc != QSV_OK) return rc;
        hipLaunchKernelGGL(latent_attention_merge_kernel, dim3(n_tokens * H), dim3(128), 0, (hipStream_t)stream, (bf16_t*)out, part_o, part_ml,
                           key_splits, n_tokens * H, rank);
    }
    return qsv_launch_status("qsv_latent_rows");
}
