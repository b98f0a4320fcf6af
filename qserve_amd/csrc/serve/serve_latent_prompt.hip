// serve_latent_prompt.hip -- attention of prompts through low-rank latents, keys and values of the heads written out (bfloat16, gfx950).
//
// On the latent rows themselves (serve_attention_mfma.hip) a query and key cost rank + rot_dim + rank products a head, here dim + rot_dim + vdim: 320 in
// place of 1088 at 128 + 64 of 512.  The rows' products with w_uk and w_uv take the place of the queries' and the results', so a prompt that brings its
// own keys pays nothing for it.
//
//   qsv_latent_gather   the cached rows of a step's runs, one behind another (what the two products read)
//   qsv_latent_prompt   causal or windowed attention of 128 tokens of a run and one head per workgroup
#include "serve_common.h"

namespace {
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void* lds_ptr;

// ---- rows of the runs: run (slot, first position, keys, first row); keys are padded to a multiple of 8 with zeros -----------------------------
// Bound by memory: a row of 16-byte pieces per group of threads.
constexpr int GATHER_ROWS = 32;
__global__ __launch_bounds__(256) void latent_gather_kernel(bf16_t* __restrict__ rows, const bf16_t* __restrict__ pool, const int32_t* __restrict__ block_table,
                                                            int table_stride, const int32_t* __restrict__ runs, int n_rows, int R, int page) {
    const int32_t* run = runs + 4 * blockIdx.y;
    const int slot = run[0], lo = run[1], keys = run[2], base = run[3], padded = (keys + 7) & ~7, ppr = R / 8;
    const int r0 = blockIdx.x * GATHER_ROWS, r1 = min(min(r0 + GATHER_ROWS, padded), n_rows - base);
    if (r0 >= r1) return;
    const int32_t* bt = block_table + (size_t)slot * table_stride;
    for (int i = threadIdx.x; i < (r1 - r0) * ppr; i += 256) {
        const int d = i / ppr, r = r0 + d, p = i - d * ppr, at = lo + r;
        v4u v = {0u, 0u, 0u, 0u};
        if (r < keys) v = *(const v4u*)(pool + ((size_t)bt[at / page] * page + (size_t)(at % page)) * R + 8 * p);
        *(v4u*)(rows + (size_t)(base + r) * R + 8 * p) = v;
    }
}

// ---- attention ----------------------------------------------------------------------------------------------------------------------------------
struct PromptArgs {
    bf16_t* out;                     // [T, H, 128]
    const bf16_t *q, *k, *vt, *rows; // [T, H, 128 + ROT], [n_rows, H, 128], [H, 128, n_rows], [n_rows, R] (rotated key part from column rank on)
    const int32_t* tiles;            // [n, 8] = (first token, tokens <= 128, its position, position of the run's first key, its row, keys of the run, -, -)
    const float* rope;
    const bf16_t* gate;              // the result is multiplied by sigmoid(gate[t, h]) before it is rounded
    int64_t gate_stride;
    float scale2;                    // scale * log2(e)
    int H, R, rank, rot_n, window, n_rows;
};
constexpr int PW = 4, PQ = 32 * PW, PK = 64;      // waves, query rows, keys of a tile

__device__ __forceinline__ unsigned pack2(float a, float b) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const b2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(unsigned, v);
}

// A wave owns 32 query rows (S^T = K Q^T, O^T = V^T P^T on 32 x 32 x 16 products, so a lane holds one query row's scores and the probabilities are
// B operands where they were made).  Tiles of 64 keys lie in LDS as [64][128] K | [64][ROT] rotated K | [128][64] V^T, 16-byte pieces permuted by the
// row's number, two tiles in turn with one barrier each; 80 KB, so two workgroups share a CU and one's matrix products run under the other's softmax.
// The key of score row 8 j + 4 g + r is 16 (j / 2) + 8 g + 4 (j % 2) + r: then a lane's eight neighbouring scores are eight neighbouring keys, and V^T is
// read in whole pieces.  Bound by the matrix cores, LDS reads (one per product) and the exponentials about evenly.
// Measured (MI355X, 128 + 64 / 128 dimensions): 8 prompts of 1024, 16 heads 78 / 53 us (550 / 650 TFLOP/s; on the latent rows 350 / 331 us and
// 99 us for their float queries), one of 4100, 32 heads 204 / 163 us (845 TFLOP/s).  Eight waves that share a tile's copy, one workgroup a CU: 82 /
// 56 us, 64 prompts of 50 - 100 tokens 34 / 23 -> 46 / 31.
// In a model, gated, 8 prompts of 1024: 110 -> 94 us with 64 rotated dimensions since their cosines and the gate are requested whole (58 without either).
template <int ROT>
__global__ __launch_bounds__(64 * PW, 2) void latent_prompt_kernel(PromptArgs a) {
    constexpr int D = 128 + ROT, NS = D / 16, KB = PK * 256, RB = PK * ROT * 2, TILE = KB + RB + 128 * PK * 2;
    __shared__ __attribute__((aligned(128))) unsigned char buf[2 * TILE];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, g = lane >> 5;
    const int tile_id = blockIdx.x / a.H, h = blockIdx.x - tile_id * a.H;
    const int32_t* tl = a.tiles + 8 * tile_id;
    const int t0 = __builtin_amdgcn_readfirstlane(tl[0]), ntok = __builtin_amdgcn_readfirstlane(tl[1]), p0 = __builtin_amdgcn_readfirstlane(tl[2]),
              lo = __builtin_amdgcn_readfirstlane(tl[3]), base = __builtin_amdgcn_readfirstlane(tl[4]), keys = __builtin_amdgcn_readfirstlane(tl[5]);
    const int p_last = p0 + ntok - 1;
    const int kstart = a.window > 0 ? lo + max(0, p0 - a.window + 1 - lo) / PK * PK : lo;      // position of the first tile's first key
    const int nT = (p_last - kstart) / PK + 1;
    const int wq = w * 32, mine = min(wq + col, ntok - 1), p_row = p0 + mine;
    const int lo_row = a.window > 0 ? p_row - a.window + 1 : lo;
    const bool active = wq < ntok;
    const int wp_first = p0 + wq, wp_last = p0 + min(wq + 31, ntok - 1);                       // this wave's positions
    const int wlo_first = a.window > 0 ? wp_first - a.window + 1 : lo, wlo_last = a.window > 0 ? wp_last - a.window + 1 : lo;

    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr)buf);
    auto fetch = [&](const bf16_t* from, unsigned off, unsigned to) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(from), "s"(to) : "memory");
    };
    auto copy = [&](int k0, int which) __attribute__((always_inline)) {
        const int row0 = base + (k0 - lo), left = min(p_last, lo + keys - 1) - k0;              // rows past the last position repeat it
        const int pieces = ((lo + keys - k0 + 7) >> 3) - 1;                                   // (the run's columns of V^T end on a whole piece)
        const unsigned to = lds0 + which * TILE;
        int me = lane;
        asm volatile("" : "+v"(me));                                                          // (offsets kept across the loop would be spilled)
        const bf16_t* kb = a.k + ((size_t)row0 * a.H + h) * 128;
#pragma unroll
        for (int j = 0; j < KB / 1024 / PW; ++j) {
            const int n = w + PW * j, row = 4 * n + (me >> 4);
            fetch(kb, (unsigned)min(row, left) * (unsigned)(a.H * 256) + (unsigned)(((me & 15) ^ (row & 15)) << 4), to + n * 1024);
        }
        if constexpr (ROT > 0) {
            const bf16_t* rb = a.rows + (size_t)row0 * a.R + a.rank;
#pragma unroll
            for (int j = 0; j < RB / 1024 / PW; ++j) {
                const int n = w + PW * j, row = 8 * n + (me >> 3);
                fetch(rb, (unsigned)min(row, left) * (unsigned)(a.R * 2) + (unsigned)(((me & 7) ^ (row & 7)) << 4), to + KB + n * 1024);
            }
        }
        const bf16_t* vb = a.vt + (size_t)h * 128 * a.n_rows + row0;
#pragma unroll
        for (int j = 0; j < 16 / PW; ++j) {
            const int n = w + PW * j, row = 8 * n + (me >> 3);
            fetch(vb, (unsigned)row * (unsigned)(a.n_rows * 2) + (unsigned)(min((me & 7) ^ (row & 7), pieces) << 4), to + KB + RB + n * 1024);
        }
    };
    copy(kstart, 0);
    bf8 qf[NS];
    {
        const bf16_t* qr = a.q + ((size_t)(t0 + mine) * a.H + h) * D + 8 * g;
#pragma unroll
        for (int s = 0; s < NS; ++s) qf[s] = __builtin_bit_cast(bf8, *(const v4u*)(qr + 16 * s));
        if constexpr (ROT > 0)
        if (a.rot_n > 0) {                                                      // (nothing turned: there need be no table)
            // cosines and sines, all requested before the first turn (behind its condition, every pair waited for the one before)
            const float* cs = a.rope + (size_t)p_row * a.rot_n;
            float co[NS - 8][4], sn[NS - 8][4];
#pragma unroll
            for (int s = 0; s < NS - 8; ++s)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = min(8 * s + 4 * g + e, (a.rot_n >> 1) - 1);
                    co[s][e] = cs[c];
                    sn[s][e] = cs[(a.rot_n >> 1) + c];
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 8; s < NS; ++s) {
                v4u x = __builtin_bit_cast(v4u, qf[s]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float u = __uint_as_float(x[e] << 16), v = __uint_as_float(x[e] & 0xffff0000u), c = co[s - 8][e], i = sn[s - 8][e];
                    const unsigned turned = pack2(u * c - v * i, v * c + u * i);
                    x[e] = 16 * (s - 8) + 8 * g + 2 * e < a.rot_n ? turned : x[e];
                }
                qf[s] = __builtin_bit_cast(bf8, x);
            }
        }
    }
    v16f o[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[c][i] = 0.f;
    float m = -INFINITY, l = 0.f;
    // K row of score row col: 16 (col / 16) + 8 (col / 4 % 2) + 4 (col / 8 % 2) + col % 4, piece 2 s + g;  V^T: row 32 c + col, piece 2 st + g
    const int krow = (col & 16) | ((col & 4) << 1) | ((col & 8) >> 1) | (col & 3);
    const int k_at = krow * 256, k_turn = (krow & 15) ^ g, r_at = KB + krow * (ROT * 2), r_turn = (krow & 7) ^ g, v_at = KB + RB + col * 128, v_turn = (col & 7) ^ g;
    int which = 0;
    for (int it = 0; it < nT; ++it) {
        const int k0 = kstart + it * PK;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                                           // this tile has landed; the other half has been read by everyone
        asm volatile("" ::: "memory");
        const unsigned char* T = buf + which * TILE;
        which ^= 1;
        if (it + 1 < nT) copy(k0 + PK, which);
        if (!active || k0 > wp_last || k0 + PK - 1 < wlo_first) continue;       // (wave-uniform)
        constexpr int KN = 2 * NS, RING = 6;
        v4u ring[RING];
        auto read = [&](int u) __attribute__((always_inline)) {                 // operand u: the KN of the keys, then the 16 of the values
            if (u < KN) {
                const int s = u >> 1, half = u & 1;
                if (s < 8) ring[u % RING] = *(const v4u*)(T + k_at + half * 32 * 256 + ((2 * s ^ k_turn) << 4));
                else ring[u % RING] = *(const v4u*)(T + r_at + half * 32 * (ROT * 2) + ((2 * (s - 8) ^ r_turn) << 4));
            } else if (u < KN + 16) {
                const int st = (u - KN) >> 2, c = (u - KN) & 3;
                ring[u % RING] = *(const v4u*)(T + v_at + c * 32 * 128 + ((2 * st ^ v_turn) << 4));
            }
        };
#pragma unroll
        for (int u = 0; u < RING - 1; ++u) read(u);
        __builtin_amdgcn_sched_barrier(0);
        v16f s[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) s[0][i] = s[1][i] = 0.f;
#pragma unroll
        for (int u = 0; u < KN; ++u) {
            read(u + RING - 1);
            __builtin_amdgcn_sched_barrier(0);
            s[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, ring[u % RING]), qf[u >> 1], s[u & 1], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        // this lane: keys k0 + 32 half + 16 (v / 8) + 8 g + v % 8 of its query row (the others sit in lane ^ 32)
        if (k0 + PK - 1 > wp_first || k0 < wlo_last) {                          // (wave-uniform)
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int key = k0 + 32 * x + 16 * (v >> 3) + 8 * g + (v & 7);
                    s[x][v] = key <= p_row && key >= lo_row ? s[x][v] : -INFINITY;
                }
        }
        float tmax = fmaxf(s[0][0], s[1][0]);
#pragma unroll
        for (int v = 1; v < 16; ++v) tmax = fmaxf(fmaxf(tmax, s[0][v]), s[1][v]);
        const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
        tmax = fmaxf(__uint_as_float(y[0]), __uint_as_float(y[1]));
        // the row's reference moves only when a score exceeds it by more than 2^8 (the sums stay far inside their range, the roundings are relative)
        if (__any(tmax * a.scale2 > m * a.scale2 + 8.0f)) {
            const float mnew = fmaxf(m, tmax), alpha = mnew == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f((m - mnew) * a.scale2);
            m = mnew;
            l *= alpha;
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[c][i] *= alpha;
        }
        const float mm = m == -INFINITY ? 0.f : m * a.scale2;
        float psum = 0.f;
#pragma unroll
        for (int st = 0; st < 4; ++st) {                                        // (the next eight exponentials run under these products)
            float p[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[st >> 1][8 * (st & 1) + e], a.scale2, -mm));
                psum += p[e];
            }
            const v4u pb = {pack2(p[0], p[1]), pack2(p[2], p[3]), pack2(p[4], p[5]), pack2(p[6], p[7])};
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int u = KN + 4 * st + c;
                read(u + RING - 1);
                __builtin_amdgcn_sched_barrier(0);
                o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, ring[u % RING]), __builtin_bit_cast(bf8, pb), o[c], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        l += psum;
    }
    l += __shfl_xor(l, 32, 64);
    if (wq + col >= ntok) return;
    const float inv = 1.0f / l;
    const size_t t = (size_t)(t0 + wq + col);
    bf16_t* out = a.out + (t * a.H + h) * 128 + 4 * g;
    const bf16_t* gate = a.gate ? a.gate + t * a.gate_stride + (size_t)h * 128 + 4 * g : nullptr;
    raw2u rg[4][4] = {};                                            // (whole before the first store: each would wait for the store before it)
    if (gate) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j) rg[c][j] = raw4(gate, 32 * c + 8 * j);
    }
    requested();
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = o[c][4 * j + r] * inv;
            if (gate) {
                float x[4];
                widen4(rg[c][j], x);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] *= 1.0f / (1.0f + expf(-x[r]));
            }
            st4t(out, 32 * c + 8 * j, v);
        }
}
}  // namespace

extern "C" int qsv_latent_prompt_tile_tokens(void) { return PQ; }
extern "C" int qsv_latent_prompt_ok(int dim, int rot_dim, int vdim, int rank, int dtype) {
    return dtype == QSV_BF16 && dim == 128 && vdim == 128 && (rot_dim == 0 || rot_dim == 64) && rank > 0 && rank % 8 == 0;
}

extern "C" int qsv_latent_gather(void* rows, const void* pool, const int32_t* block_table, int table_stride, const int32_t* runs, int n_runs, int longest,
                                 int n_rows, int R, int page, void* stream) {
    QSV_REQUIRE(rows && pool && block_table && runs && n_runs >= 0 && n_runs <= 65535 && longest >= 0 && n_rows >= 0 && R > 0 && R % 8 == 0 && page > 0,
                "qsv_latent_gather: bad arguments");
    QSV_REQUIRE(((uintptr_t)rows | (uintptr_t)pool) % 16 == 0, "qsv_latent_gather: rows start on 16 bytes");
    if (n_runs == 0 || longest == 0 || n_rows == 0) return QSV_OK;
    hipLaunchKernelGGL(latent_gather_kernel, dim3((longest + 7 + GATHER_ROWS - 1) / GATHER_ROWS, n_runs), dim3(256), 0, (hipStream_t)stream, (bf16_t*)rows,
                       (const bf16_t*)pool, block_table, table_stride, runs, n_rows, R, page);
    return qsv_launch_status("qsv_latent_gather");
}

extern "C" int qsv_latent_prompt(void* out, const void* q, const void* k, const void* vt, const void* rows, const int32_t* tiles, int n_tiles, const float* rope,
                                 float scale, int H, int rot_dim, int rot_n, int rank, int window, int n_rows, const void* gate, int64_t gate_stride, void* stream) {
    QSV_REQUIRE(out && q && k && vt && rows && tiles && n_tiles >= 0 && H > 0 && window >= 0 && scale > 0.0f, "qsv_latent_prompt: bad arguments");
    QSV_REQUIRE(qsv_latent_prompt_ok(128, rot_dim, 128, rank, QSV_BF16) && rot_n >= 0 && rot_n <= rot_dim && rot_n % 2 == 0 && (rot_n == 0 || rope),
                "qsv_latent_prompt: %d rotated of %d dimensions, rank %d", rot_n, rot_dim, rank);
    QSV_REQUIRE(n_rows > 0 && n_rows % 8 == 0 && n_rows <= (1 << 23) && H <= (1 << 16) && (int64_t)n_tiles * H <= 0x7fffffff, "qsv_latent_prompt: %d keys, %d heads", n_rows, H);
    QSV_REQUIRE(((uintptr_t)out | (uintptr_t)q | (uintptr_t)k | (uintptr_t)vt | (uintptr_t)rows) % 16 == 0, "qsv_latent_prompt: operands start on 16 bytes");
    QSV_REQUIRE(!gate || ((uintptr_t)gate % 8 == 0 && gate_stride % 4 == 0 && gate_stride >= (int64_t)H * 128), "qsv_latent_prompt: gate rows of %lld", (long long)gate_stride);
    if (n_tiles == 0) return QSV_OK;
    const PromptArgs a = {(bf16_t*)out, (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)vt, (const bf16_t*)rows, tiles, rope, (const bf16_t*)gate, gate_stride,
                          scale * 1.44269504088896340736f, H, rank + rot_dim, rank, rot_n, window, n_rows};
    if (rot_dim) hipLaunchKernelGGL(latent_prompt_kernel<64>, dim3(n_tiles * H), dim3(64 * PW), 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL(latent_prompt_kernel<0>, dim3(n_tiles * H), dim3(64 * PW), 0, (hipStream_t)stream, a);
    return qsv_launch_status("qsv_latent_prompt");
}
