// serve_recurrent.hip -- matrix-state recurrences (gated linear attention, gated delta rule) and what feeds them: decays,
// the short causal convolution with its history state, unit norms, the per-head output norm with its gate; and the rotations of
// the attention that runs beside them (queries, keys and values in the halves layout, cache rows written in the same pass).
// Everything that enters a recurrence is float; the state is float in memory and in registers.
#include "serve_common.h"

namespace {
constexpr int NT = 256;
constexpr int NW = NT / 64;

// ---- decays (gate_decay) ---------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(NT) void decay_kernel(float* __restrict__ out, const T* __restrict__ z, int64_t z_stride,
                                                   const T* __restrict__ bias, const float* __restrict__ a_log, float inv_tau,
                                                   int dim, int n) {
    const size_t t = blockIdx.x;
    for (int c = threadIdx.x; c < n; c += NT) {
        const float v = ld(z, t * z_stride + c) + ld(bias, c);
        out[t * n + c] = gate_decay(v, a_log != nullptr, a_log ? a_log[c / dim] : 0.f, inv_tau);
    }
}

// The same, four channels per thread, `chunks` workgroups per token.
template <typename T>
__global__ __launch_bounds__(NT) void decay_vec_kernel(float* __restrict__ out, const T* __restrict__ z, int64_t z_stride, const T* __restrict__ bias,
                                                       const float* __restrict__ a_log, float inv_tau, int dim, int n, int chunks) {
    const size_t t = token_of(blockIdx.x, chunks);
    const int c = ((blockIdx.x - (unsigned)t * chunks) * NT + threadIdx.x) * 4;
    if (c >= n) return;
    const auto rz = raw4(z, t * z_stride + c), rb = raw4(bias, c);
    float a[4] = {0.f, 0.f, 0.f, 0.f}, v[4], b[4];
    if (a_log) {
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = a_log[(c + j) / dim];
    }
    requested();
    widen4(rz, v);
    widen4(rb, b);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = gate_decay(v[j] + b[j], a_log != nullptr, a[j], inv_tau);
    }
    st4t(out, t * n + c, v);
}

// ---- causal convolution over time + silu (act 0: no activation), unit norm of the leading groups -----------------------------------------------------
// Workgroup = token.  Tap j (last column = the current token) reads the input taps - 1 - j tokens back: a row of this batch
// inside the run, the sequence's history state before the run's start, zero before the sequence's start.  The last token of a
// run writes the new history (the last taps - 1 inputs) into the state's other copy.  Dynamic LDS: C floats.
template <typename T>
__global__ __launch_bounds__(NT) void conv_silu_unit_kernel(float* __restrict__ out, const T* __restrict__ proj, int64_t stride,
                                                            int off, int C, int taps, const float* __restrict__ w,
                                                            float* __restrict__ hist, const int32_t* __restrict__ run_off,
                                                            const int32_t* __restrict__ state_rd,
                                                            const int32_t* __restrict__ state_wr, int n_unit, int unit_dim, int act) {
    extern __shared__ float ys[];
    const size_t t = blockIdx.x;
    const int i = run_off[t], rd = state_rd[t], wr = state_wr[t];
    const int past = taps - 1;
    for (int c = threadIdx.x; c < C; c += NT) {
        float acc = 0.f;
        for (int j = 0; j < taps; ++j) {
            const int d = past - j;
            float xv = 0.f;
            if (d <= i) xv = ld(proj, (t - d) * stride + off + c);
            else if (rd >= 0) xv = hist[((size_t)rd * past + (past + i - d)) * C + c];
            acc += w[(size_t)c * taps + j] * xv;
        }
        ys[c] = act ? acc / (1.0f + expf(-acc)) : acc;
        if (wr >= 0) {
            for (int jj = 0; jj < past; ++jj) {
                const int e = i + 1 - past + jj;            // index within the run of the input that becomes history entry jj
                float xv = 0.f;
                if (e >= 0) xv = ld(proj, (t - (i - e)) * stride + off + c);
                else if (rd >= 0) xv = hist[((size_t)rd * past + (jj + i + 1)) * C + c];
                hist[((size_t)wr * past + jj) * C + c] = xv;
            }
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int g = wv; g < n_unit; g += NW) {
        float s = 0.f;
        for (int e = lane; e < unit_dim; e += 64) s += ys[g * unit_dim + e] * ys[g * unit_dim + e];
        const float inv = 1.0f / sqrtf(wave_sum(s) + 1e-6f);
        for (int e = lane; e < unit_dim; e += 64) out[t * C + g * unit_dim + e] = ys[g * unit_dim + e] * inv;
    }
    for (int c = n_unit * unit_dim + threadIdx.x; c < C; c += NT) out[t * C + c] = ys[c];
}

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// sum over the lpc neighbouring lanes of a column (lpc a power of two); every one of them gets it
__device__ __forceinline__ float column_sum(float v, int lpc) {
    if (lpc >= 2) v = dpp_add<0xB1>(v);          // quad_perm [1, 0, 3, 2]
    if (lpc >= 4) v = dpp_add<0x4E>(v);          // quad_perm [2, 3, 0, 1]
    if (lpc >= 8) v = dpp_add<0x141>(v);         // row_half_mirror: the other quad of eight lanes
    if (lpc >= 16) v = dpp_add<0x140>(v);        // row_mirror: the other half of sixteen lanes
    if (lpc >= 32) v += __shfl_xor(v, 16, 64);
    if (lpc >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

// The same for channels in fours (TAPS taps; whole groups of 4 to 256 channels, a power of two): a thread owns four channels of a token, so every
// tap of theirs is requested before the first is used, a group is 1 - 64 neighbouring lanes, and a token is `chunks` workgroups.  The entries of
// the new history are the taps behind the first, already in registers.  Bound by latency in a step, by HBM in a prompt (2560 channels: 16 tokens
// 15.7 -> 2.7 us, 8192 tokens 137 -> 55 us).
template <typename T, int TAPS>
__global__ __launch_bounds__(NT) void conv_silu_unit_vec_kernel(float* __restrict__ out, const T* __restrict__ proj, int64_t stride, int off, int C,
                                                                const float* __restrict__ w, float* __restrict__ hist,
                                                                const int32_t* __restrict__ run_off, const int32_t* __restrict__ state_rd,
                                                                const int32_t* __restrict__ state_wr, int unit_channels, int group_lanes, int act,
                                                                int chunks) {
    constexpr int PAST = TAPS - 1;
    const unsigned t = token_of(blockIdx.x, chunks);
    const int c = ((blockIdx.x - t * chunks) * NT + threadIdx.x) * 4;
    const bool in = c < C;
    const int from = in ? c : 0;                                   // (lanes behind the end stay for the sums below)
    const int i = run_off[t], rd = state_rd[t], wr = state_wr[t];
    float x[TAPS][4], wt[TAPS][4];
    typename Raw4<T>::type rx[TAPS];
    raw4f rh[PAST];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) ld4t(w, (size_t)from * TAPS + 4 * j, wt[j]);
#pragma unroll
    for (int j = 0; j < TAPS; ++j) rx[j] = raw4(proj, (size_t)(t - min(PAST - j, min(i, PAST))) * stride + off + from);
    if (i < PAST && rd >= 0) {                                      // (the same for the whole workgroup)
#pragma unroll
        for (int j = 0; j < PAST; ++j) rh[j] = raw4(hist, ((size_t)rd * PAST + min(i + j, PAST - 1)) * C + from);
    }
    requested();
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
        const int d = PAST - j;
        float a[4], b[4];
        widen4(rx[j], a);
        widen4(rh[min(j, PAST - 1)], b);
#pragma unroll
        for (int q = 0; q < 4; ++q) x[j][q] = d <= i ? a[q] : rd >= 0 ? b[q] : 0.f;
    }
    float y[4], s = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < TAPS; ++j) acc += wt[(q * TAPS + j) / 4][(q * TAPS + j) % 4] * x[j][q];
        y[q] = act ? acc / (1.0f + expf(-acc)) : acc;
        s += y[q] * y[q];
    }
    const float inv = 1.0f / sqrtf(column_sum(s, group_lanes) + 1e-6f);
    if (!in) return;
    if (wr >= 0) {
#pragma unroll
        for (int jj = 0; jj < PAST; ++jj) st4t(hist, ((size_t)wr * PAST + jj) * C + c, x[jj + 1]);
    }
    if (c < unit_channels) {
#pragma unroll
        for (int q = 0; q < 4; ++q) y[q] *= inv;
    }
    st4t(out, (size_t)t * C + c, y);
}

// ---- the recurrence ---------------------------------------------------------------------------------------------------------
// Columns of S (value channels) never meet: column j of head h needs k, q and the decay of the token and its own v_j.  A
// workgroup owns a block of columns of one (run, head): a wave 64 / LPC groups of NC of them, a lane R rows of its NC columns;
// the LPC lanes of a column are neighbours and add their partial dot products through DPP moves.  The run's tokens are walked in order, CT at
// a time: the workgroup stages k, q, the decay (float, zero-padded to LPC * R rows), its v columns and sigmoid(beta) of CT
// tokens in LDS - the next CT tokens' values are already in registers while these are computed - so a token's step reads
// LDS only, and the only exchange on the state's dependency chain is the delta rule's S^T k; the read-outs' partial sums wait
// in registers until the chunk's end and are exchanged together.  The state is read once before and written once after (a run
// that starts its sequence starts from zeros).
constexpr int SCAN_CT = 16;       // tokens per staged chunk, at most
constexpr int SCAN_PFK = 24;      // staged k / q / decay values per thread and chunk, at most
constexpr int SCAN_PFV = 16;      // staged v values per thread and chunk, at most

__device__ __forceinline__ float4 ld4(const float* p, size_t i) { return *(const float4*)(p + i); }
__device__ __forceinline__ float4 ld4(const bf16_t* p, size_t i) {
    const uint2 u = *(const uint2*)(p + i);
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                       __uint_as_float(u.y & 0xffff0000u));
}

// VEC: dim, vdim, the row strides and the operands' addresses are multiples of four elements - staged four at a time.
// R rows and NC columns of the state per lane (with NC > 1 the token's k, q and decay rows are read from LDS once for NC columns).
// OCC: waves per SIMD the register allocation must leave room for (1: no demand - the compiler takes about 230 registers, two waves).
template <typename TQ, typename TB, bool DELTA, bool VEC, int R, int NC, int OCC>
__global__ __launch_bounds__(256, OCC) void recurrent_scan_kernel(float* __restrict__ o, const TQ* __restrict__ q, int64_t q_stride,
                                                             const TQ* __restrict__ k, int64_t k_stride, const TQ* __restrict__ v,
                                                             int64_t v_stride, const float* __restrict__ decay,
                                                             const TB* __restrict__ beta, int64_t beta_stride,
                                                             float* __restrict__ state, const int32_t* __restrict__ runs, int H,
                                                             int QH, int dim, int vdim, int lpc_log, int CT, float q_scale,
                                                             const float* __restrict__ kscale, int head_decay, int v_cols) {
    static_assert(R == 4 || R == 8 || R == 16, "rows per lane");
    // (the three-wave variant stages half as many tokens per chunk: fewer prefetch registers and deferred read-outs, no spills)
    constexpr int MAX_CT = OCC >= 3 ? SCAN_CT / 2 : SCAN_CT, PFK = OCC >= 3 ? SCAN_PFK / 2 : SCAN_PFK, PFV = OCC >= 3 ? SCAN_PFV / 2 : SCAN_PFV;
    extern __shared__ __attribute__((aligned(16))) float sm[];
    const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, wave = tid >> 6, nw = nthr >> 6;
    const int lpc = 1 << lpc_log, cols = 64 >> lpc_log;                           // cols: column groups (of NC) per wave
    const int dimp_log = lpc_log + (R == 16 ? 4 : R == 8 ? 3 : 2), DIMP = 1 << dimp_log, VB = nw * cols * NC;   // (all powers of two)
    const int vb_log = 31 - __clz(VB);
    const int row_len = 3 * DIMP + ((VB + 4) & ~3);              // floats of one staged token: k | q | decay | v | beta, 16-byte rows
    const int part = lane & (lpc - 1), cb = (wave * cols + (lane >> lpc_log)) * NC;
    const int j = blockIdx.z * VB + cb;                          // first of this lane's NC columns
    const int r0 = part * R;
    const int slot = runs[4 * blockIdx.x], first = runs[4 * blockIdx.x + 1], n = runs[4 * blockIdx.x + 2];
    const bool fresh = runs[4 * blockIdx.x + 3] == 0;
    const int h = blockIdx.y, qh = h / (H / QH);
    float* Sg = state + (((size_t)slot * H + h) * dim) * (size_t)vdim;
    float S[NC][R];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < R; ++i) S[c][i] = (!fresh && j + c < vdim && r0 + i < dim) ? Sg[(size_t)(r0 + i) * vdim + j + c] : 0.f;

    float pk[PFK], pv[PFV], pb = 0.f;
    // requests the operands of tokens [c0, c0 + ct) of the run into registers
    auto fetch = [&](int c0, int ct) {
        const int nk = ct * 3 * DIMP, nv = ct * VB;
        if (VEC) {
#pragma unroll
            for (int i = 0; i < PFK / 4; ++i) {
                const int idx = (tid + i * nthr) * 4;
                float4 val = make_float4(0.f, 0.f, 0.f, 0.f);
                if (idx < nk) {
                    const int seg = idx >> dimp_log, r = idx & (DIMP - 1), tt = seg / 3, which = seg - 3 * tt;
                    const size_t t = (size_t)(first + c0 + tt);
                    if (r < dim) {
                        if (which == 2 && head_decay) {
                            const float g = head_decay == 2 ? decay[h] : decay[t * H + h];
                            val = make_float4(g, g, g, g);
                        } else {
                            val = which == 0 ? ld4(k, t * k_stride + (size_t)qh * dim + r)
                                : which == 1 ? ld4(q, t * q_stride + (size_t)qh * dim + r)
                                             : ld4(decay, (t * H + h) * (size_t)dim + r);
                            if (which == 0 && kscale) {
                                const float b = kscale[t * H + h];
                                val.x *= b; val.y *= b; val.z *= b; val.w *= b;
                            }
                        }
                    }
                }
                pk[4 * i] = val.x; pk[4 * i + 1] = val.y; pk[4 * i + 2] = val.z; pk[4 * i + 3] = val.w;
            }
#pragma unroll
            for (int i = 0; i < PFV / 4; ++i) {
                const int idx = (tid + i * nthr) * 4;
                float4 val = make_float4(0.f, 0.f, 0.f, 0.f);
                if (idx < nv) {
                    const int tt = idx >> vb_log, c = idx & (VB - 1), jj = blockIdx.z * VB + c;
                    if (jj < v_cols) val = ld4(v, (size_t)(first + c0 + tt) * v_stride + (size_t)h * v_cols + jj);
                    else if (jj == v_cols && jj < vdim) val.x = 1.0f;        // the state's column of ones (a state wider than v)
                }
                pv[4 * i] = val.x; pv[4 * i + 1] = val.y; pv[4 * i + 2] = val.z; pv[4 * i + 3] = val.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < PFK; ++i) {
                const int idx = tid + i * nthr;
                float val = 0.f;
                if (idx < nk) {
                    const int seg = idx >> dimp_log, r = idx & (DIMP - 1), tt = seg / 3, which = seg - 3 * tt;
                    const size_t t = (size_t)(first + c0 + tt);
                    if (r < dim)
                        val = which == 0 ? ld(k, t * k_stride + (size_t)qh * dim + r) * (kscale ? kscale[t * H + h] : 1.0f)
                            : which == 1 ? ld(q, t * q_stride + (size_t)qh * dim + r)
                                         : (head_decay == 2 ? decay[h] : head_decay ? decay[t * H + h] : decay[(t * H + h) * (size_t)dim + r]);
                }
                pk[i] = val;
            }
#pragma unroll
            for (int i = 0; i < PFV; ++i) {
                const int idx = tid + i * nthr;
                float val = 0.f;
                if (idx < nv) {
                    const int tt = idx >> vb_log, c = idx & (VB - 1), jj = blockIdx.z * VB + c;
                    if (jj < v_cols) val = ld(v, (size_t)(first + c0 + tt) * v_stride + (size_t)h * v_cols + jj);
                    else if (jj == v_cols && jj < vdim) val = 1.0f;
                }
                pv[i] = val;
            }
        }
        if (DELTA && tid < ct) pb = ld(beta, (size_t)(first + c0 + tid) * beta_stride + h);
    };
    auto stage = [&](int ct) {
        const int nk = ct * 3 * DIMP, nv = ct * VB;
        if (VEC) {
#pragma unroll
            for (int i = 0; i < PFK / 4; ++i) {
                const int idx = (tid + i * nthr) * 4;
                if (idx < nk) {
                    const int tt = (idx >> dimp_log) / 3;
                    *(float4*)(sm + tt * row_len + (idx - tt * 3 * DIMP)) = make_float4(pk[4 * i], pk[4 * i + 1], pk[4 * i + 2], pk[4 * i + 3]);
                }
            }
#pragma unroll
            for (int i = 0; i < PFV / 4; ++i) {
                const int idx = (tid + i * nthr) * 4;
                if (idx < nv) {
                    const int tt = idx >> vb_log;
                    *(float4*)(sm + tt * row_len + 3 * DIMP + (idx & (VB - 1))) = make_float4(pv[4 * i], pv[4 * i + 1], pv[4 * i + 2], pv[4 * i + 3]);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < PFK; ++i) {
                const int idx = tid + i * nthr;
                if (idx < nk) {
                    const int tt = (idx >> dimp_log) / 3;
                    sm[tt * row_len + (idx - tt * 3 * DIMP)] = pk[i];
                }
            }
#pragma unroll
            for (int i = 0; i < PFV; ++i) {
                const int idx = tid + i * nthr;
                if (idx < nv) {
                    const int tt = idx >> vb_log;
                    sm[tt * row_len + 3 * DIMP + (idx & (VB - 1))] = pv[i];
                }
            }
        }
        if (DELTA && tid < ct) sm[tid * row_len + 3 * DIMP + VB] = 1.0f / (1.0f + expf(-pb));
    };

    fetch(0, min(CT, n));
    for (int c0 = 0; c0 < n; c0 += CT) {
        const int ct = min(CT, n - c0);
        __syncthreads();                                         // the previous chunk has been read by every wave
        stage(ct);
        __syncthreads();
        if (c0 + CT < n) fetch(c0 + CT, min(CT, n - c0 - CT));   // in flight while this chunk is computed
        float oacc[MAX_CT][NC];
#pragma unroll
        for (int tt = 0; tt < MAX_CT; ++tt) {
#pragma unroll
            for (int c = 0; c < NC; ++c) oacc[tt][c] = 0.f;
            if (tt >= ct) continue;                              // (uniform)
            const float* row = sm + tt * row_len;
            float kc[R], qc[R], gc[R], vc[NC];
#pragma unroll
            for (int i = 0; i < R; i += 4) {
                const float4 a = *(const float4*)(row + r0 + i), b = *(const float4*)(row + DIMP + r0 + i),
                             c = *(const float4*)(row + 2 * DIMP + r0 + i);
                kc[i] = a.x; kc[i + 1] = a.y; kc[i + 2] = a.z; kc[i + 3] = a.w;
                qc[i] = b.x; qc[i + 1] = b.y; qc[i + 2] = b.z; qc[i + 3] = b.w;
                gc[i] = c.x; gc[i + 1] = c.y; gc[i + 2] = c.z; gc[i + 3] = c.w;
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) vc[c] = row[3 * DIMP + cb + c];
            if (DELTA) {
                const float bt = row[3 * DIMP + VB];
                float acc[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    acc[c] = 0.f;
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        S[c][i] *= gc[i];
                        acc[c] += S[c][i] * kc[i];
                    }
                }
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const float u = (vc[c] - column_sum(acc[c], lpc)) * bt;
                    float a2 = 0.f;
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        S[c][i] += kc[i] * u;
                        a2 += S[c][i] * qc[i];
                    }
                    oacc[tt][c] = a2;
                }
            } else {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    float a2 = 0.f;
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        S[c][i] = gc[i] * S[c][i] + kc[i] * vc[c];
                        a2 += S[c][i] * qc[i];
                    }
                    oacc[tt][c] = a2;
                }
            }
        }
#pragma unroll
        for (int tt = 0; tt < MAX_CT; ++tt)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const float sum = column_sum(oacc[tt][c], lpc);
                if (tt < ct && part == 0 && j + c < vdim) o[((size_t)(first + c0 + tt) * H + h) * (size_t)vdim + j + c] = sum * q_scale;
            }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (j + c < vdim && r0 + i < dim) Sg[(size_t)(r0 + i) * vdim + j + c] = S[c][i];
}

// ---- the same recurrence for 33 - 128 rows, operands in fours -------------------------------------------------------------------------------
// A token's step is three or four multiply-adds per element of the state and lane, behind twelve 16-byte LDS reads of its k, q and decay: what
// bounds it is the wait for those reads and the issue of both.  So a lane holds 16 rows of NC columns (two: every read serves twice as many
// multiply-adds; one where two would leave CUs without a workgroup), LPC lanes a column; a chunk of 16 tokens is straight-line code in which the
// next token's operands are requested before the current one is computed; the chunks alternate between two LDS buffers (one barrier each), the
// chunk after in registers meanwhile.  A run's last tokens, fewer than a chunk, go one by one.  Rows of the parts 4 .. 7 are taken in another
// order, so that their reads fall on other banks than those of 0 .. 3.
// Measured (8 runs of 1024 tokens, delta rule / plain; before: the form above): 32 heads of 64 x 128 1102 -> 428 / 1000 -> 365 us, 16 heads 477 -> 253 /
// 431 -> 220, 32 heads of 128 x 128 2424 -> 617 / 1971 -> 456; 64 runs of 4 tokens 63 -> 21 / 31 -> 18, one of 2 6.8 -> 5.3 / 6.5 -> 4.1.
// (Reads laid between the rows of the token before, instead of ahead of them: the same time, and spills.)
constexpr int ROWS_CT = 16;
template <int NC>
struct TokenRows {
    float k[16], q[16], g[16], v[NC], b;
};
template <typename TQ, typename TB, bool DELTA, int LPC, int NC>
__global__ __launch_bounds__(256, 2) void recurrent_rows_kernel(float* __restrict__ o, const TQ* __restrict__ q, int64_t q_stride,
                                                                const TQ* __restrict__ k, int64_t k_stride, const TQ* __restrict__ v,
                                                                int64_t v_stride, const float* __restrict__ decay, const TB* __restrict__ beta,
                                                                int64_t beta_stride, float* __restrict__ state, const int32_t* __restrict__ runs,
                                                                int H, int QH, int dim, int vdim, float q_scale, const float* __restrict__ kscale,
                                                                int head_decay, int v_cols) {
    constexpr int CT = ROWS_CT, D = 16 * LPC, COLS = 64 / LPC, VB = 4 * COLS * NC;
    constexpr int KP = CT * D / 4 / 256, VPIECES = CT * VB / 4, VP = (VPIECES + 255) / 256;
    static_assert(CT * D % 1024 == 0, "");
    __shared__ __attribute__((aligned(16))) float rows[2][3][CT][D];     // k, q, decay
    __shared__ __attribute__((aligned(16))) float vs[2][CT][VB];
    __shared__ float rates[2][CT];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, part = lane & (LPC - 1), turn = part >> 2;
    const int cb = (wave * COLS + lane / LPC) * NC, j = blockIdx.z * VB + cb;
    const int slot = runs[4 * blockIdx.x], first = runs[4 * blockIdx.x + 1], n = runs[4 * blockIdx.x + 2];
    const bool fresh = runs[4 * blockIdx.x + 3] == 0;
    const int h = blockIdx.y, qh = h / (H / QH);
    const bool col_ok = j < vdim;                                  // (vdim is a multiple of 4: both columns or none)
    float* Sg = state + (((size_t)slot * H + h) * dim) * (size_t)vdim + (col_ok ? j : 0);
    float S[NC][16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = part * 16 + 4 * ((i >> 2) ^ turn) + (i & 3);
#pragma unroll
        for (int c = 0; c < NC; ++c) S[c][i] = (!fresh && col_ok && r < dim) ? Sg[(size_t)r * vdim + c] : 0.f;
    }
    float4 pk[KP], pq[KP], pg[KP], pv[VP];
    float pb = 0.f;
    auto fetch = [&](int c0, int ct) __attribute__((always_inline)) {                 // requests the operands of tokens c0 .. c0 + ct of the run
#pragma unroll
        for (int i = 0; i < KP; ++i) {
            const int piece = tid + 256 * i, tt = piece / (D / 4), r = (piece % (D / 4)) * 4;
            pk[i] = pq[i] = pg[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (tt < ct && r < dim) {
                const size_t t = (size_t)(first + c0 + tt);
                pk[i] = ld4(k, t * k_stride + (size_t)qh * dim + r);
                pq[i] = ld4(q, t * q_stride + (size_t)qh * dim + r);
                if (head_decay) {
                    const float g = head_decay == 2 ? decay[h] : decay[t * H + h];
                    pg[i] = make_float4(g, g, g, g);
                } else {
                    pg[i] = ld4(decay, (t * H + h) * (size_t)dim + r);
                }
                if (kscale) {
                    const float b = kscale[t * H + h];
                    pk[i].x *= b; pk[i].y *= b; pk[i].z *= b; pk[i].w *= b;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int piece = tid + 256 * i, tt = piece / (VB / 4), jj = blockIdx.z * VB + (piece % (VB / 4)) * 4;
            pv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (tt < ct) {
                if (jj < v_cols) pv[i] = ld4(v, (size_t)(first + c0 + tt) * v_stride + (size_t)h * v_cols + jj);
                else if (jj == v_cols && jj < vdim) pv[i].x = 1.0f;       // the state's column of ones (a state wider than v)
            }
        }
        if (DELTA && tid < ct) pb = ld(beta, (size_t)(first + c0 + tid) * beta_stride + h);
    };
    auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KP; ++i) {
            const int piece = tid + 256 * i, tt = piece / (D / 4), r = (piece % (D / 4)) * 4;
            *(float4*)&rows[buf][0][tt][r] = pk[i];
            *(float4*)&rows[buf][1][tt][r] = pq[i];
            *(float4*)&rows[buf][2][tt][r] = pg[i];
        }
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int piece = tid + 256 * i;
            if (VPIECES % 256 == 0 || piece < VPIECES) *(float4*)&vs[buf][piece / (VB / 4)][(piece % (VB / 4)) * 4] = pv[i];
        }
        if (DELTA && tid < CT) rates[buf][tid] = 1.0f / (1.0f + expf(-pb));
    };
    auto request = [&](TokenRows<NC>& x, int buf, int tt) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = part * 16 + 4 * (i ^ turn);
            const float4 a = *(const float4*)&rows[buf][0][tt][r], b = *(const float4*)&rows[buf][1][tt][r], c = *(const float4*)&rows[buf][2][tt][r];
            x.k[4 * i] = a.x, x.k[4 * i + 1] = a.y, x.k[4 * i + 2] = a.z, x.k[4 * i + 3] = a.w;
            x.q[4 * i] = b.x, x.q[4 * i + 1] = b.y, x.q[4 * i + 2] = b.z, x.q[4 * i + 3] = b.w;
            x.g[4 * i] = c.x, x.g[4 * i + 1] = c.y, x.g[4 * i + 2] = c.z, x.g[4 * i + 3] = c.w;
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) x.v[c] = vs[buf][tt][cb + c];
        x.b = DELTA ? rates[buf][tt] : 0.f;
    };
    auto step = [&](const TokenRows<NC>& x, float (&out)[NC]) __attribute__((always_inline)) {   // out: this lane's share of the read-out
        float u[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            u[c] = x.v[c];
            if (DELTA) {
                float a = 0.f, b = 0.f;
#pragma unroll
                for (int i = 0; i < 16; i += 2) {
                    S[c][i] *= x.g[i];
                    S[c][i + 1] *= x.g[i + 1];
                    a += S[c][i] * x.k[i];
                    b += S[c][i + 1] * x.k[i + 1];
                }
                u[c] = a + b;
            }
        }
        if (DELTA) {
#pragma unroll
            for (int c = 0; c < NC; ++c) u[c] = (x.v[c] - column_sum(u[c], LPC)) * x.b;
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            float a = 0.f, b = 0.f;
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                S[c][i] = (DELTA ? S[c][i] : x.g[i] * S[c][i]) + x.k[i] * u[c];
                S[c][i + 1] = (DELTA ? S[c][i + 1] : x.g[i + 1] * S[c][i + 1]) + x.k[i + 1] * u[c];
                a += S[c][i] * x.q[i];
                b += S[c][i + 1] * x.q[i + 1];
            }
            out[c] = a + b;
        }
    };
    fetch(0, min(CT, n));
    int buf = 0;
    for (int c0 = 0; c0 < n; c0 += CT, buf ^= 1) {
        const int ct = min(CT, n - c0);
        stage(buf);
        __syncthreads();                                           // (the other buffer: every wave is behind the chunk that read it)
        if (c0 + CT < n) fetch(c0 + CT, min(CT, n - c0 - CT));     // in flight while this chunk is computed
        float* og = o + ((size_t)(first + c0) * H + h) * (size_t)vdim + j;
        if (ct == CT) {
            float out[8][NC];
            TokenRows<NC> x[2];
            request(x[0], buf, 0);
#pragma unroll
            for (int tt = 0; tt < CT; ++tt) {
                if (tt + 1 < CT) request(x[(tt + 1) & 1], buf, tt + 1);
                __builtin_amdgcn_sched_barrier(0);
                step(x[tt & 1], out[tt & 7]);
                __builtin_amdgcn_sched_barrier(0);
                if ((tt & 7) != 7) continue;
#pragma unroll
                for (int s = 0; s < 8; ++s)
#pragma unroll
                    for (int c = 0; c < NC; ++c) out[s][c] = column_sum(out[s][c], LPC);
#pragma unroll
                for (int t0 = 0; t0 < 8; t0 += LPC) {              // lane `part` of a column writes token t0 + part of the eight
                    float w[NC];
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        w[c] = out[t0][c];
#pragma unroll
                        for (int p = 1; p < LPC; ++p) w[c] = part == p ? out[t0 + p][c] : w[c];
                        w[c] *= q_scale;
                    }
                    if (col_ok) {
                        float* d = og + (size_t)(tt - 7 + t0 + part) * H * vdim;
                        if (NC == 2) *(float2*)d = make_float2(w[0], w[NC - 1]);
                        else *d = w[0];
                    }
                }
            }
        } else {
            for (int tt = 0; tt < ct; ++tt) {
                TokenRows<NC> x;
                float out[NC];
                request(x, buf, tt);
                step(x, out);
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const float w = column_sum(out[c], LPC) * q_scale;
                    if (col_ok && part == 0) og[(size_t)tt * H * vdim + c] = w;
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = part * 16 + 4 * ((i >> 2) ^ turn) + (i & 3);
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (col_ok && r < dim) Sg[(size_t)r * vdim + c] = S[c][i];
    }
}

// ---- one token per run (decoding): no staging, no barriers - every lane fetches its 8 rows of k, q and the decay itself, the
// state makes one round trip -----------------------------------------------------------------------------------------------------
template <typename TQ, typename TB, bool DELTA>
__global__ __launch_bounds__(256) void recurrent_step_kernel(float* __restrict__ o, const TQ* __restrict__ q, int64_t q_stride,
                                                             const TQ* __restrict__ k, int64_t k_stride, const TQ* __restrict__ v,
                                                             int64_t v_stride, const float* __restrict__ decay,
                                                             const TB* __restrict__ beta, int64_t beta_stride,
                                                             float* __restrict__ state, const int32_t* __restrict__ runs, int H,
                                                             int QH, int dim, int vdim, int lpc_log, float q_scale,
                                                             const float* __restrict__ kscale, int head_decay, int v_cols) {
    constexpr int R = 8;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lpc = 1 << lpc_log, cols = 64 >> lpc_log;
    const int part = lane & (lpc - 1), j = (blockIdx.z * 4 + wave) * cols + (lane >> lpc_log);
    const bool col_ok = j < vdim;
    const int r0 = part * R;
    const int slot = runs[4 * blockIdx.x];
    const size_t t = (size_t)runs[4 * blockIdx.x + 1];
    const bool fresh = runs[4 * blockIdx.x + 3] == 0;
    const int h = blockIdx.y, qh = h / (H / QH);
    float* Sg = state + (((size_t)slot * H + h) * dim) * (size_t)vdim + (col_ok ? j : 0);
    float S[R], kc[R], qc[R], gc[R];
    const float kb = kscale ? kscale[t * H + h] : 1.0f;
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const bool ok = r0 + i < dim;
        S[i] = (!fresh && col_ok && ok) ? Sg[(size_t)(r0 + i) * vdim] : 0.f;
        kc[i] = ok ? ld(k, t * k_stride + (size_t)qh * dim + r0 + i) * kb : 0.f;
        qc[i] = ok ? ld(q, t * q_stride + (size_t)qh * dim + r0 + i) : 0.f;
        gc[i] = ok ? (head_decay == 2 ? decay[h] : head_decay ? decay[t * H + h] : decay[(t * H + h) * (size_t)dim + r0 + i]) : 0.f;
    }
    const float vc = !col_ok ? 0.f : j < v_cols ? ld(v, t * v_stride + (size_t)h * v_cols + j) : j == v_cols ? 1.0f : 0.f;
    float acc = 0.f;
    if (DELTA) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            S[i] *= gc[i];
            acc += S[i] * kc[i];
        }
        const float u = (vc - column_sum(acc, lpc)) / (1.0f + expf(-ld(beta, t * beta_stride + h)));
        acc = 0.f;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            S[i] += kc[i] * u;
            acc += S[i] * qc[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            S[i] = gc[i] * S[i] + kc[i] * vc;
            acc += S[i] * qc[i];
        }
    }
    acc = column_sum(acc, lpc);
    if (!col_ok) return;
    if (part == 0) o[(t * H + h) * (size_t)vdim + j] = acc * q_scale;
#pragma unroll
    for (int i = 0; i < R; ++i)
        if (r0 + i < dim) Sg[(size_t)(r0 + i) * vdim] = S[i];
}

// The same for states whose columns come in fours: a workgroup owns 128 columns of one (run, head), a thread four of them (16-byte accesses, a
// row's 512 bytes together) and 8 rows of every 64.  Row sums meet across two half waves and, through LDS, four waves.  Bound by the state's two
// trips to memory (16 sequences of 16 heads, 64 x 128: 17 MB; 11.9 -> 4.9 us
// with the delta rule; 64 sequences of 128 x 128 132 -> 25 us: the form above reads 32 bytes of a row at a time).
// GATED (a head's columns in one workgroup, vdim a power of two): the head's norm, weight and gate (head_rms_gate_vec_kernel's, the same bits) on the way out, a
// launch less and no read-out in memory.  With the streams' two fused passes (serve_streams.hip) nine launches of 46 less in a step of four layers: 16 sequences of
// Mumelix 451 -> 434 us.
struct GateTail {
    bf16_t* out;                    // [T, H * vdim]
    const bf16_t *w, *gate;
    int64_t gate_stride;
    int kind;
    float eps;
};
template <typename TQ, typename TB, bool DELTA, int P, bool GATED>
__global__ __launch_bounds__(256) void recurrent_step_wide_kernel(float* __restrict__ o, const TQ* __restrict__ q, int64_t q_stride,
                                                                  const TQ* __restrict__ k, int64_t k_stride, const TQ* __restrict__ v,
                                                                  int64_t v_stride, const float* __restrict__ decay, const TB* __restrict__ beta,
                                                                  int64_t beta_stride, float* __restrict__ state,
                                                                  const int32_t* __restrict__ runs, int H, int QH, int dim, int vdim, float q_scale,
                                                                  const float* __restrict__ kscale, int head_decay, int v_cols, GateTail tail) {
    __shared__ float4 sums[2][4][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, cg = tid & 31, rg = tid >> 5;
    const int j = blockIdx.z * 128 + cg * 4;
    const bool col_ok = j < vdim;
    const int slot = runs[4 * blockIdx.x];
    const size_t t = (size_t)runs[4 * blockIdx.x + 1];
    const bool fresh = runs[4 * blockIdx.x + 3] == 0;
    const int h = blockIdx.y, qh = h / (H / QH);
    float* Sg = state + (((size_t)slot * H + h) * dim) * (size_t)vdim + (col_ok ? j : 0);
    float S[P][8][4], kc[P][8], qc[P][8], gc[P][8], vc[4];
    const float kb = kscale ? kscale[t * H + h] : 1.0f;
    const float hd = head_decay == 2 ? decay[h] : head_decay ? decay[t * H + h] : 0.f;
    // every operand as it lies in memory, rows and columns clamped into the state: one trip
    typename Raw4<TQ>::type rk[P][2], rq[P][2];
    raw4f rg4[P][2];
    TQ rv[4];
    TB rb = TB();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int r0 = min(p * 64 + rg * 8, dim - 8);               // (dim is a multiple of 8)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            rk[p][x] = raw4(k, t * k_stride + (size_t)qh * dim + r0 + 4 * x);
            rq[p][x] = raw4(q, t * q_stride + (size_t)qh * dim + r0 + 4 * x);
            if (!head_decay) rg4[p][x] = raw4(decay, (t * H + h) * (size_t)dim + r0 + 4 * x);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            S[p][i][0] = S[p][i][1] = S[p][i][2] = S[p][i][3] = 0.f;
            if (p * 64 + rg * 8 < dim && col_ok && !fresh) ld4t(Sg, (size_t)(r0 + i) * vdim, S[p][i]);
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) rv[c] = v[t * v_stride + (size_t)h * v_cols + min(j + c, v_cols - 1)];
    if (DELTA) rb = beta[t * beta_stride + h];
    raw2u rgate = {}, rw = {};
    if (GATED && tid < 32) {
        rgate = raw4(tail.gate, t * tail.gate_stride + (size_t)h * vdim + (col_ok ? j : 0));
        rw = raw4(tail.w, col_ok ? j : 0);
    }
    requested();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const bool ok = p * 64 + rg * 8 < dim;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            float a[4], b[4], g[4];
            widen4(rk[p][x], a);
            widen4(rq[p][x], b);
            widen4(rg4[p][x], g);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                kc[p][4 * x + e] = ok ? a[e] : 0.f;
                qc[p][4 * x + e] = ok ? b[e] : 0.f;
                gc[p][4 * x + e] = head_decay || !ok ? hd : g[e];
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) vc[c] = j + c < v_cols ? ld(&rv[c], 0) : j + c == v_cols ? 1.0f : 0.f;
    const float rate = DELTA ? 1.0f / (1.0f + expf(-ld(&rb, 0))) : 0.f;
    // sum over the workgroup's rows; every thread gets its columns'
    auto row_sum = [&](float (&a)[4], int buffer) {
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] += __shfl_xor(a[c], 32, 64);
        if (lane < 32) sums[buffer][wave][cg] = make_float4(a[0], a[1], a[2], a[3]);
        __syncthreads();
        const float4 s0 = sums[buffer][0][cg], s1 = sums[buffer][1][cg], s2 = sums[buffer][2][cg], s3 = sums[buffer][3][cg];
        a[0] = (s0.x + s1.x) + (s2.x + s3.x);
        a[1] = (s0.y + s1.y) + (s2.y + s3.y);
        a[2] = (s0.z + s1.z) + (s2.z + s3.z);
        a[3] = (s0.w + s1.w) + (s2.w + s3.w);
    };
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    if (DELTA) {
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float kk = kc[p][i] * kb;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    S[p][i][c] *= gc[p][i];
                    acc[c] += S[p][i][c] * kk;
                }
            }
        row_sum(acc, 0);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            vc[c] = (vc[c] - acc[c]) * rate;
            acc[c] = 0.f;
        }
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float kk = kc[p][i] * kb;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                S[p][i][c] = (DELTA ? S[p][i][c] : gc[p][i] * S[p][i][c]) + kk * vc[c];
                acc[c] += S[p][i][c] * qc[p][i];
            }
        }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (col_ok && p * 64 + rg * 8 < dim) st4t(Sg, (size_t)(p * 64 + rg * 8 + i) * vdim, S[p][i]);
    row_sum(acc, 1);
    if (tid < 32 && col_ok) {
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] *= q_scale;
        if constexpr (GATED) {
            float s = 0.f, g[4], ww[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) s += acc[c] * acc[c];
            const float inv = 1.0f / sqrtf(column_sum(s, vdim / 4) / (float)vdim + tail.eps);
            widen4(rgate, g);
            widen4(rw, ww);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float sg = 1.0f / (1.0f + expf(-g[c]));
                acc[c] = acc[c] * inv * ww[c] * (tail.kind == 0 ? g[c] * sg : sg);
            }
            st4t(tail.out, (t * H + h) * (size_t)vdim + j, acc);
        } else {
            st4t(o, (t * H + h) * (size_t)vdim + j, acc);
        }
    }
}

// ---- per-head RMS norm of the read-out, times a weight, times a gate ------------------------------------------------------------
// gate_kind 0: silu(g), 1: sigmoid(g).  o rows are o_stride floats apart per head (>= vdim); w_stride 0: one weight row shared by
// the heads, vdim: a row per head.  den_m != NULL: before the norm the read-out is divided by max(|o[vdim]|, exp(-den_m[t, h])) +
// 1e-6, o[vdim] being the head's extra column (the normaliser's dot product with the query).
template <typename T>
__global__ __launch_bounds__(NT) void head_rms_gate_kernel(T* __restrict__ out, const float* __restrict__ o, const T* __restrict__ w,
                                                           const T* __restrict__ gate, int64_t gate_stride, int gate_kind, float eps,
                                                           int H, int vdim, int o_stride, int w_stride,
                                                           const float* __restrict__ den_m) {
    const size_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int h = wv; h < H; h += NW) {
        const float* oh = o + (t * H + h) * (size_t)o_stride;
        const float sc = den_m ? 1.0f / (fmaxf(fabsf(oh[vdim]), expf(-den_m[t * H + h])) + 1e-6f) : 1.0f;
        float s = 0.f;
        for (int e = lane; e < vdim; e += 64) s += (oh[e] * sc) * (oh[e] * sc);
        const float inv = 1.0f / sqrtf(wave_sum(s) / (float)vdim + eps);
        for (int e = lane; e < vdim; e += 64) {
            const float g = ld(gate, t * gate_stride + (size_t)h * vdim + e);
            const float sg = 1.0f / (1.0f + expf(-g));
            st(out, (t * H + h) * (size_t)vdim + e, oh[e] * sc * inv * ld(w, (size_t)h * w_stride + e) * (gate_kind == 0 ? g * sg : sg));
        }
    }
}

// The same for heads of 4 to 256 values, a power of two: a thread owns four values of a head, a head is 1 - 64 neighbouring lanes, and the
// heads of all tokens follow one another; everything is read once, before the sum.  (16 heads of 128: 16 tokens 5.6 -> 2.3 us, 8192 tokens 44 -> 31 us;
// one head of 64, 8192 tokens: 3.4 us, with a workgroup per token 8.1.)
template <typename T>
__global__ __launch_bounds__(NT) void head_rms_gate_vec_kernel(T* __restrict__ out, const float* __restrict__ o, const T* __restrict__ w,
                                                               const T* __restrict__ gate, int64_t gate_stride, int gate_kind, float eps, int H,
                                                               int vdim, int lanes_log, int o_stride, int w_stride,
                                                               const float* __restrict__ den_m, unsigned n_heads) {
    const unsigned idx = blockIdx.x * NT + threadIdx.x;
    const bool in = idx >> lanes_log < n_heads;
    const unsigned row = in ? idx >> lanes_log : 0, t = row / (unsigned)H;
    const int h = row - t * H, e = (idx & ((1 << lanes_log) - 1)) * 4;
    const size_t th = row;
    float x[4], g[4], ww[4];
    ld4t(o, th * (size_t)o_stride + e, x);
    ld4t(gate, t * gate_stride + (size_t)h * vdim + e, g);
    ld4t(w, (size_t)h * w_stride + e, ww);
    const float sc = den_m ? 1.0f / (fmaxf(fabsf(o[th * (size_t)o_stride + vdim]), expf(-den_m[th])) + 1e-6f) : 1.0f;
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        x[j] *= sc;
        s += x[j] * x[j];
    }
    const float inv = 1.0f / sqrtf(column_sum(s, 1 << lanes_log) / (float)vdim + eps);
    if (!in) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float sg = 1.0f / (1.0f + expf(-g[j]));
        x[j] = x[j] * inv * ww[j] * (gate_kind == 0 ? g[j] * sg : sg);
    }
    st4t(out, th * (size_t)vdim + e, x);
}

// ---- exponential gates kept in range by a running maximum (mLSTM) ----------------------------------------------------------------
// Per (run, head) one wave; a lane takes one token of 64 at a time.  li = cap tanh((z_i + b_i) / cap), lf = logsigmoid(cap tanh((z_f
// + b_f) / cap)); m_t = max(lf_t + m_(t-1), li_t) is a scan over the maps x -> max(x + A, B), which compose to (A1 + A2, max(B1 + A2,
// B2)); decay a_t = exp(lf_t + m_(t-1) - m_t), input scale b_t = exp(li_t - m_t).  m of a run's last token goes back to the state
// (a run that starts its sequence starts from m = 0).
__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }
template <typename T>
__global__ __launch_bounds__(64) void max_gates_kernel(float* __restrict__ a_out, float* __restrict__ b_out, float* __restrict__ m_out,
                                                       const T* __restrict__ zi, const T* __restrict__ zf, int64_t z_stride,
                                                       const float* __restrict__ bias_i, const float* __restrict__ bias_f, float cap,
                                                       float* __restrict__ m_state, const int32_t* __restrict__ runs, int H) {
    const int lane = threadIdx.x;
    const int slot = runs[4 * blockIdx.x], first = runs[4 * blockIdx.x + 1], n = runs[4 * blockIdx.x + 2];
    const int h = blockIdx.y;
    float carry = runs[4 * blockIdx.x + 3] == 0 ? 0.f : m_state[(size_t)slot * H + h];
    const float inv_cap = 1.0f / cap;
    for (int c0 = 0; c0 < n; c0 += 64) {
        const bool ok = c0 + lane < n;
        const size_t t = (size_t)first + c0 + (ok ? lane : 0);
        const float li = cap * tanhf((ld(zi, t * z_stride + h) + bias_i[h]) * inv_cap);
        const float lf = log_sigmoid(cap * tanhf((ld(zf, t * z_stride + h) + bias_f[h]) * inv_cap));
        float A = ok ? lf : 0.f, B = ok ? li : -INFINITY;       // (a lane past the end is the identity map)
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const float pA = __shfl_up(A, o, 64), pB = __shfl_up(B, o, 64);
            if (lane >= o) {
                B = fmaxf(pB + A, B);
                A = pA + A;
            }
        }
        const float m = fmaxf(carry + A, B);
        float prev = __shfl_up(m, 1, 64);
        if (lane == 0) prev = carry;
        if (ok) {
            a_out[t * H + h] = expf(lf + (prev - m));            // (prev - m is exact; lf + prev would round lf away)
            b_out[t * H + h] = expf(li - m);
            m_out[t * H + h] = m;
        }
        carry = __shfl(m, min(63, n - c0 - 1), 64);
    }
    if (lane == 0) m_state[(size_t)slot * H + h] = carry;
}

// ---- rotations, halves layout: pair p of n rotated dimensions = (p, p + n / 2); rope [positions, 2, n / 2] -------------------
__device__ __forceinline__ float rot_halves(float u_lo, float u_hi, bool upper, float c, float s) {
    return upper ? u_hi * c + u_lo * s : u_lo * c - u_hi * s;
}
template <typename T>
__device__ __forceinline__ float rotated(const T* vec, int d, int n, const float* cs) {   // element d of the rotated vector
    if (d >= n) return ld(vec, d);
    const int half = n >> 1, p = d < half ? d : d - half;
    return rot_halves(ld(vec, p), ld(vec, p + half), d >= half, cs[p], cs[half + p]);
}

// qf[t, h] = [0 (vdim) | rot(q[t, h]) * scale]; pool[g, slot[t]] = [rot_v(v[t, g]) | rot(k[t, g])]
template <typename T>
__global__ __launch_bounds__(NT) void attention_prep_kernel(float* __restrict__ qf, T* __restrict__ pool, int64_t pool_rows,
                                                            const T* __restrict__ proj, int64_t stride, int q_off, int k_off,
                                                            int v_off, int H, int G, int dim, int vdim, int rot_n,
                                                            const float* __restrict__ rope_k, const float* __restrict__ rope_v,
                                                            float scale, const int64_t* __restrict__ slot,
                                                            const int32_t* __restrict__ pos) {
    const size_t t = blockIdx.x;
    const int R = vdim + dim, p = pos[t];
    const T* row = proj + t * stride;
    const float* ck = rope_k + (size_t)p * rot_n;
    const float* cv = rope_v + (size_t)p * vdim;
    for (int idx = threadIdx.x; idx < H * R; idx += NT) {
        const int h = idx / R, c = idx - h * R;
        qf[t * H * (size_t)R + idx] = c < vdim ? 0.f : rotated(row + q_off + h * dim, c - vdim, rot_n, ck) * scale;
    }
    for (int idx = threadIdx.x; idx < G * R; idx += NT) {
        const int g = idx / R, c = idx - g * R;
        const float val = c < vdim ? rotated(row + v_off + g * vdim, c, vdim, cv) : rotated(row + k_off + g * dim, c - vdim, rot_n, ck);
        st(pool, ((size_t)g * pool_rows + (size_t)slot[t]) * R + c, val);
    }
}

// The same, four columns per thread (sizes, halves and offsets that are multiples of four), `chunks` workgroups per token.  Bound by latency in a
// step, by HBM in a prompt (16 + 4 heads of 128 + 128: 16 tokens 7.3 -> 2.6 us, 8192 tokens 53 -> 47 us).
template <typename T>
__device__ __forceinline__ void rotated4(const T* vec, int d, int n, const float* cs, float (&out)[4]) {
    if (d >= n) return ld4t(vec, d, out);
    const int half = n >> 1, p = d < half ? d : d - half;
    float lo[4], hi[4], c[4], s[4];
    ld4t(vec, p, lo);
    ld4t(vec, p + half, hi);
    ld4t(cs, p, c);
    ld4t(cs, half + p, s);
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = rot_halves(lo[j], hi[j], d >= half, c[j], s[j]);
}
template <typename T>
__global__ __launch_bounds__(NT) void attention_prep_vec_kernel(float* __restrict__ qf, T* __restrict__ pool, int64_t pool_rows,
                                                                const T* __restrict__ proj, int64_t stride, int q_off, int k_off, int v_off, int H,
                                                                int G, int dim, int vdim, int rot_n, const float* __restrict__ rope_k,
                                                                const float* __restrict__ rope_v, float scale, const int64_t* __restrict__ slot,
                                                                const int32_t* __restrict__ pos, int chunks) {
    const unsigned t = token_of(blockIdx.x, chunks), idx = (blockIdx.x - t * chunks) * NT + threadIdx.x;
    const unsigned R = vdim + dim;
    const int u = idx / (R / 4), c = (idx - u * (R / 4)) * 4, p = pos[t];
    if (u >= H + G) return;
    const T* row = proj + (size_t)t * stride;
    const float* ck = rope_k + (size_t)p * rot_n;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (u < H) {
        if (c >= vdim) {
            rotated4(row + q_off + u * dim, c - vdim, rot_n, ck, v);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] *= scale;
        }
        st4t(qf, ((size_t)t * H + u) * R + c, v);
    } else {
        const int g = u - H;
        if (c < vdim) rotated4(row + v_off + g * vdim, c, vdim, rope_v + (size_t)p * vdim, v);
        else rotated4(row + k_off + g * dim, c - vdim, rot_n, ck, v);
        st4t(pool, ((size_t)g * pool_rows + (size_t)slot[t]) * R + c, v);
    }
}

// o[t, h, :n] turned by sign * pos[t] in place
template <typename T, bool V4>
__global__ __launch_bounds__(NT) void rotate_heads_kernel(T* __restrict__ o, const float* __restrict__ rope,
                                                          const int32_t* __restrict__ pos, float sign, int H, int n) {
    const size_t t = blockIdx.x;
    const int half = n >> 1;
    const float* cs = rope + (size_t)pos[t] * n;
    if (V4) {
        for (int idx = threadIdx.x * 4; idx < H * half; idx += NT * 4) {
            const int h = idx / half, p = idx - h * half;
            T* vec = o + (t * H + h) * (size_t)n;
            const auto ra = raw4((const T*)vec, p), rb = raw4((const T*)vec, p + half);
            const auto rc = raw4(cs, p), rs = raw4(cs, half + p);
            requested();
            float a[4], b[4], x[4], y[4];
            widen4(ra, a);
            widen4(rb, b);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float c = rc[j], s = rs[j] * sign;
                x[j] = a[j] * c - b[j] * s;
                y[j] = b[j] * c + a[j] * s;
            }
            st4t(vec, p, x);
            st4t(vec, p + half, y);
        }
        return;
    }
    for (int idx = threadIdx.x; idx < H * half; idx += NT) {
        const int h = idx / half, p = idx - h * half;
        T* vec = o + (t * H + h) * (size_t)n;
        const float a = ld(vec, p), b = ld(vec, p + half), c = cs[p], s = cs[half + p] * sign;
        st(vec, p, a * c - b * s);
        st(vec, p + half, b * c + a * s);
    }
}
}  // namespace

extern "C" int qsv_decay(float* out, const void* z, int64_t z_stride, const void* bias, const float* a_log, float tau, int n_tokens,
                         int heads, int dim, int dtype, void* stream) {
    QSV_REQUIRE(out && z && bias && n_tokens >= 0 && heads > 0 && dim > 0 && z_stride >= (int64_t)heads * dim,
                "qsv_decay: bad arguments");
    QSV_REQUIRE(a_log || tau > 0.f, "qsv_decay: a power-sigmoid decay needs tau > 0");
    if (n_tokens == 0) return QSV_OK;
    const int width = heads * dim;
    const int64_t chunks = ((int64_t)width / 4 + NT - 1) / NT;
    // (below 1024 channels the general kernel has a thread for each, and a thread's four would come one after another: 256 channels, 1 - 512 tokens 3.3 against 4.3 us)
    if (width >= 4 * NT && width % 4 == 0 && z_stride % 4 == 0 && fits4(out, QSV_F32) && fits4(z, dtype) && fits4(bias, dtype) && chunks * n_tokens < (1ll << 31)) {
        QSV_DISPATCH(dtype, "qsv_decay",
                     hipLaunchKernelGGL(decay_vec_kernel<T>, dim3((unsigned)(chunks * n_tokens)), dim3(NT), 0, (hipStream_t)stream, out, (const T*)z, z_stride,
                                        (const T*)bias, a_log, a_log ? 0.f : 1.0f / tau, dim, width, (int)chunks));
        return qsv_launch_status("qsv_decay");
    }
    QSV_DISPATCH(dtype, "qsv_decay",
                 hipLaunchKernelGGL(decay_kernel<T>, dim3(n_tokens), dim3(NT), 0, (hipStream_t)stream, out, (const T*)z, z_stride,
                                    (const T*)bias, a_log, a_log ? 0.f : 1.0f / tau, dim, heads * dim));
    return qsv_launch_status("qsv_decay");
}

extern "C" int qsv_conv_silu_unit(float* out, const void* proj, int64_t stride, int off, int channels, int taps, const float* w,
                                  float* hist, const int32_t* run_off, const int32_t* state_rd, const int32_t* state_wr,
                                  int n_unit, int unit_dim, int act, int n_tokens, int dtype, void* stream) {
    QSV_REQUIRE(out && proj && w && hist && run_off && state_rd && state_wr, "qsv_conv_silu_unit: null argument");
    QSV_REQUIRE(channels > 0 && taps >= 1 && off >= 0 && off + channels <= stride && n_unit >= 0 && unit_dim > 0 &&
                    (int64_t)n_unit * unit_dim <= channels && n_tokens >= 0 && (act == 0 || act == 1),
                "qsv_conv_silu_unit: bad sizes");
    QSV_REQUIRE((size_t)channels * 4 <= 64 * 1024, "qsv_conv_silu_unit: %d channels do not fit the workgroup's LDS", channels);
    if (n_tokens == 0) return QSV_OK;
    const int64_t chunks = ((int64_t)channels / 4 + NT - 1) / NT;
    // (a prompt of few channels: one lane in eight has any, 8192 tokens of 96: 11.3 -> 13.1 us)
    if ((channels >= 256 || n_tokens < 1024) && taps >= 2 && taps <= 4 && channels % 4 == 0 && off % 4 == 0 && stride % 4 == 0 && fits4(proj, dtype) && fits4(out, QSV_F32) &&
        fits4(w, QSV_F32) && fits4(hist, QSV_F32) && chunks * n_tokens < (1ll << 31) &&
        (n_unit == 0 || (unit_dim >= 4 && unit_dim <= 256 && (unit_dim & (unit_dim - 1)) == 0))) {
        const dim3 grid((unsigned)(chunks * n_tokens));
        const int lanes = n_unit ? unit_dim / 4 : 1;
#define QSV_CONV(TAPS)                                                                                                                        \
    QSV_DISPATCH(dtype, "qsv_conv_silu_unit",                                                                                                 \
                 hipLaunchKernelGGL((conv_silu_unit_vec_kernel<T, TAPS>), grid, dim3(NT), 0, (hipStream_t)stream, out, (const T*)proj, stride, \
                                    off, channels, w, hist, run_off, state_rd, state_wr, n_unit* unit_dim, lanes, act, (int)chunks))
        if (taps == 4) QSV_CONV(4);
        else if (taps == 3) QSV_CONV(3);
        else QSV_CONV(2);
#undef QSV_CONV
        return qsv_launch_status("qsv_conv_silu_unit");
    }
    QSV_DISPATCH(dtype, "qsv_conv_silu_unit",
                 hipLaunchKernelGGL(conv_silu_unit_kernel<T>, dim3(n_tokens), dim3(NT), (size_t)channels * 4, (hipStream_t)stream, out,
                                    (const T*)proj, stride, off, channels, taps, w, hist, run_off, state_rd, state_wr, n_unit,
                                    unit_dim, act));
    return qsv_launch_status("qsv_conv_silu_unit");
}

// the operand types a step's launch is made for
#define QSV_STEP_TYPES                                                                                     \
    if (beta) {                                                                                            \
        if (qkv_dtype == QSV_F32 && beta_dtype == QSV_F32) QSV_STEP(float, float, true);                   \
        else if (qkv_dtype == QSV_F32 && beta_dtype == QSV_BF16) QSV_STEP(float, bf16_t, true);            \
        else if (qkv_dtype == QSV_BF16 && beta_dtype == QSV_BF16) QSV_STEP(bf16_t, bf16_t, true);          \
        else QSV_REQUIRE(false, "qsv_recurrent_scan: operand types %d / %d", qkv_dtype, beta_dtype);       \
    } else {                                                                                               \
        if (qkv_dtype == QSV_F32) QSV_STEP(float, float, false);                                           \
        else if (qkv_dtype == QSV_BF16) QSV_STEP(bf16_t, bf16_t, false);                                   \
        else QSV_REQUIRE(false, "qsv_recurrent_scan: operand type %d", qkv_dtype);                         \
    }
extern "C" int qsv_recurrent_scan(float* o, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                                  int64_t v_stride, int qkv_dtype, const float* decay, const void* beta, int64_t beta_stride,
                                  int beta_dtype, float* state, const int32_t* runs, int n_runs, int max_run, int heads, int qk_heads,
                                  int dim, int vdim, float q_scale, const float* kscale, int head_decay, int v_cols, void* stream) {
    QSV_REQUIRE(o && q && k && v && decay && state && runs, "qsv_recurrent_scan: null argument");
    if (v_cols <= 0) v_cols = vdim;
    QSV_REQUIRE(v_cols <= vdim, "qsv_recurrent_scan: %d value columns for a state of %d", v_cols, vdim);
    if (max_run == 1 && n_runs > 0 && dim <= 64 * 8 && heads > 0 && qk_heads > 0 && heads % qk_heads == 0 && vdim > 0 && heads <= 65535) {
        const int qkv = qkv_dtype == QSV_F32 ? QSV_F32 : QSV_BF16;
        if (dim % 8 == 0 && dim <= 256 && vdim % 4 == 0 && q_stride % 4 == 0 && k_stride % 4 == 0 && fits4(q, qkv) && fits4(k, qkv) &&
            fits4(decay, QSV_F32) && fits4(state, QSV_F32) && fits4(o, QSV_F32) && (vdim + 127) / 128 <= 65535) {
            const dim3 grid(n_runs, heads, (vdim + 127) / 128), block(256);   // (heads and vdim are checked above)
#define QSV_STEP_P(TQ, TB, DELTA, P)                                                                                            \
    hipLaunchKernelGGL((recurrent_step_wide_kernel<TQ, TB, DELTA, P, false>), grid, block, 0, (hipStream_t)stream, o, (const TQ*)q, q_stride, \
                       (const TQ*)k, k_stride, (const TQ*)v, v_stride, decay, (const TB*)beta, beta_stride, state, runs, heads,  \
                       qk_heads, dim, vdim, q_scale, kscale, head_decay, v_cols, GateTail{})
#define QSV_STEP(TQ, TB, DELTA)                            \
    do {                                                   \
        if (dim <= 64) QSV_STEP_P(TQ, TB, DELTA, 1);       \
        else if (dim <= 128) QSV_STEP_P(TQ, TB, DELTA, 2); \
        else QSV_STEP_P(TQ, TB, DELTA, 4);                 \
    } while (0)
            QSV_STEP_TYPES
#undef QSV_STEP
#undef QSV_STEP_P
            return qsv_launch_status("qsv_recurrent_scan");
        }
        int lpc = 1, lpc_log = 0;
        while (lpc * 8 < dim) lpc <<= 1, ++lpc_log;
        const int per_block = 4 * (64 / lpc);
        const dim3 grid(n_runs, heads, (vdim + per_block - 1) / per_block), block(256);
        QSV_REQUIRE(grid.z <= 65535, "qsv_recurrent_scan: too many column blocks");
#define QSV_STEP(TQ, TB, DELTA)                                                                                              \
    hipLaunchKernelGGL((recurrent_step_kernel<TQ, TB, DELTA>), grid, block, 0, (hipStream_t)stream, o, (const TQ*)q, q_stride,    \
                       (const TQ*)k, k_stride, (const TQ*)v, v_stride, decay, (const TB*)beta, beta_stride, state, runs, heads,  \
                       qk_heads, dim, vdim, lpc_log, q_scale, kscale, head_decay, v_cols)
        QSV_STEP_TYPES
#undef QSV_STEP
        return qsv_launch_status("qsv_recurrent_scan");
    }
    QSV_REQUIRE(heads > 0 && qk_heads > 0 && heads % qk_heads == 0 && dim > 0 && dim <= 64 * 16 && vdim > 0 && n_runs >= 0 &&
                    heads <= 65535,
                "qsv_recurrent_scan: bad sizes (%d heads over %d, state %d x %d)", heads, qk_heads, dim, vdim);
    if (n_runs == 0) return QSV_OK;
    const int qkv = qkv_dtype == QSV_F32 ? QSV_F32 : QSV_BF16;
    // Short runs of narrow states leave its lanes without columns and its chunks without tokens, which counts once the CUs have no workgroup left over (64 runs
    // of 2 tokens, 64 heads of 64 x 4: 13.6 us with the general kernel, 28 here; 64 heads of 64 x 24: 32 and 30; 64 runs of 64 tokens 0.9 of its time).
    const bool narrow = vdim <= (dim <= 64 ? 16 : 8) && max_run <= 8 && (int64_t)n_runs * heads >= 1024;
    if (!narrow && dim > 32 && dim <= 128 && dim % 4 == 0 && vdim % 4 == 0 && v_cols % 4 == 0 && q_stride % 4 == 0 && k_stride % 4 == 0 && v_stride % 4 == 0 &&
        fits4(q, qkv) && fits4(k, qkv) && fits4(v, qkv) && fits4(decay, QSV_F32) && fits4(o, QSV_F32) && vdim <= 65535 * 32) {
        const int lpc = dim <= 64 ? 4 : 8, cols = 4 * 64 / lpc;
        // two columns per lane while that gives every CU a workgroup (half as many CUs: a token costs them as much as it would cost all) and the
        // state has more columns than one per lane serves (16 runs of 64 tokens, 32 heads of 64 x 32, delta rule: 46 -> 29 us)
        const bool two = vdim > cols && (int64_t)n_runs * heads * ((vdim + 2 * cols - 1) / (2 * cols)) >= 256;
        const dim3 grid(n_runs, heads, two ? (vdim + 2 * cols - 1) / (2 * cols) : (vdim + cols - 1) / cols), block(256);
#define QSV_STEP_P(TQ, TB, DELTA, LPC, NC)                                                                                      \
    hipLaunchKernelGGL((recurrent_rows_kernel<TQ, TB, DELTA, LPC, NC>), grid, block, 0, (hipStream_t)stream, o, (const TQ*)q, q_stride, \
                       (const TQ*)k, k_stride, (const TQ*)v, v_stride, decay, (const TB*)beta, beta_stride, state, runs, heads,  \
                       qk_heads, dim, vdim, q_scale, kscale, head_decay, v_cols)
#define QSV_STEP(TQ, TB, DELTA)                                      \
    do {                                                             \
        if (lpc == 4 && two) QSV_STEP_P(TQ, TB, DELTA, 4, 2);        \
        else if (lpc == 4) QSV_STEP_P(TQ, TB, DELTA, 4, 1);          \
        else if (two) QSV_STEP_P(TQ, TB, DELTA, 8, 2);               \
        else QSV_STEP_P(TQ, TB, DELTA, 8, 1);                        \
    } while (0)
        QSV_STEP_TYPES
#undef QSV_STEP
#undef QSV_STEP_P
        return qsv_launch_status("qsv_recurrent_scan");
    }
    // States of other heights (up to 32 rows, 129 and more), and operands that are not in fours.
    // Rows of one column per lane: 8 while that leaves the launch at no more than ~2.5 waves per SIMD, else 16 (and for the tallest
    // states).  The figures here are of 16 heads of 64 x 128, which come here only where their operands are not in fours: 8 x 1024 tokens
    // (2048 / 1024 waves) 0.46 / 0.51 ms plain, 0.50 / 0.55 ms delta rule; 64 runs of a token (16384 / 8192 waves) 56 / 43 us; two columns per lane
    // 0.60 / 0.75 ms.  A token's step is a short chain of dependent instructions: up to the chip's fill, more and lighter waves win; beyond
    // it, fewer and heavier ones.
    int lpc8 = 1;
    while (lpc8 * 8 < dim) lpc8 <<= 1;
    const int64_t waves8 = (int64_t)n_runs * heads * (((int64_t)vdim * lpc8 + 63) / 64);
    int R = dim <= 64 * 8 && waves8 <= 2560 ? 8 : 16;
    const int NC = 1;
    // Both forms take about 230 registers: two four-wave workgroups of the 8-row form (one of the 16-row form) per CU, and a launch
    // of more workgroups than that runs in rounds, each as long as a full one (132 columns instead of 128 at 8 x 16 (run, head)
    // pairs: 0.94 ms instead of 0.49).  A third form - 8 rows, compiled for three waves per SIMD, half the staging - holds three
    // workgroups per CU at 1.23 times the round's length; it is taken where that saves rounds (costs in rounds of the 8-row form).
    bool three = false;
    if (!beta && dim <= 64 * 8) {
        const int cols8 = 64 / lpc8, wpb8 = (vdim + cols8 - 1) / cols8 >= 4 ? 4 : (vdim + cols8 - 1) / cols8 > 1 ? 2 : 1;
        const int64_t pairs = (int64_t)n_runs * heads;
        const int64_t groups8 = pairs * ((vdim + wpb8 * cols8 - 1) / (wpb8 * cols8)) * wpb8 / 4;
        const int cols16 = cols8 * 2 > 64 ? 64 : cols8 * 2;
        const int64_t groups16 = pairs * ((vdim + 4 * cols16 - 1) / (4 * cols16));
        const double legacy = R == 8 ? (double)((groups8 + 511) / 512) : 1.12 * (double)((groups16 + 255) / 256);
        const double lean = 1.23 * (double)((groups8 + 767) / 768);
        const size_t el8 = qkv_dtype == QSV_F32 ? 4 : 2;         // (the third form has 16-byte staging only)
        const bool vec8 = dim % 4 == 0 && vdim % 4 == 0 && v_cols % 4 == 0 && (wpb8 * cols8) % 4 == 0 && q_stride % 4 == 0 &&
                          k_stride % 4 == 0 && v_stride % 4 == 0 && (uintptr_t)q % (4 * el8) == 0 && (uintptr_t)k % (4 * el8) == 0 &&
                          (uintptr_t)v % (4 * el8) == 0 && (uintptr_t)decay % 16 == 0;
        if (vec8 && lean < legacy) {
            three = true;
            R = 8;
        }
    }
    int lpc = 1, lpc_log = 0;
    while (lpc * R < dim) lpc <<= 1, ++lpc_log;
    QSV_REQUIRE(lpc <= 64, "qsv_recurrent_scan: %d rows per lane for a state of %d rows", R, dim);
    const int cols = 64 / lpc, DIMP = lpc * R;
    const int waves_needed = (vdim + cols * NC - 1) / (cols * NC);
    // waves per workgroup: they share the staged k, q and decay (fewer: the staging loads multiply; more: the launch's waves
    // stack up on the CUs of a few large workgroups while a token's step is bound by instruction issue)
    int nw = 1;
    while (nw < 4 && nw < waves_needed) nw <<= 1;
    const int VB = nw * cols * NC, nthr = nw * 64;
    const size_t el = qkv_dtype == QSV_F32 ? 4 : 2;
    const bool vec = dim % 4 == 0 && vdim % 4 == 0 && v_cols % 4 == 0 && VB % 4 == 0 && q_stride % 4 == 0 && k_stride % 4 == 0 && v_stride % 4 == 0 &&
                     (uintptr_t)q % (4 * el) == 0 && (uintptr_t)k % (4 * el) == 0 && (uintptr_t)v % (4 * el) == 0 &&
                     (uintptr_t)decay % 16 == 0;
    const bool lean = three && vec;                              // (the variant for three waves per SIMD: half the staging)
    const int max_ct = lean ? SCAN_CT / 2 : SCAN_CT, pfk = lean ? SCAN_PFK / 2 : SCAN_PFK, pfv = lean ? SCAN_PFV / 2 : SCAN_PFV;
    int CT = max_ct;                                             // tokens per staged chunk: what the prefetch registers and 48 KiB hold
    while (CT > 1 && ((CT * 3 * DIMP + nthr - 1) / nthr > pfk || (CT * VB + nthr - 1) / nthr > pfv ||
                      (size_t)CT * (3 * DIMP + ((VB + 4) & ~3)) * 4 > 48 * 1024))
        CT >>= 1;
    QSV_REQUIRE((CT * 3 * DIMP + nthr - 1) / nthr <= pfk && (CT * VB + nthr - 1) / nthr <= pfv,
                "qsv_recurrent_scan: a state of %d rows does not fit the staging registers", dim);
    const size_t lds = (size_t)CT * (3 * DIMP + ((VB + 4) & ~3)) * 4;
    const dim3 grid(n_runs, heads, (vdim + VB - 1) / VB), block(nthr);
    QSV_REQUIRE(grid.z <= 65535, "qsv_recurrent_scan: too many column blocks");
#define QSV_SCAN_V(TQ, TB, DELTA, VEC, RR, CC, OC)                                                                              \
    hipLaunchKernelGGL((recurrent_scan_kernel<TQ, TB, DELTA, VEC, RR, CC, OC>), grid, block, lds, (hipStream_t)stream, o,        \
                       (const TQ*)q, q_stride, (const TQ*)k, k_stride, (const TQ*)v, v_stride, decay, (const TB*)beta,         \
                       beta_stride, state, runs, heads, qk_heads, dim, vdim, lpc_log, CT, q_scale, kscale, head_decay, v_cols)
#define QSV_SCAN(TQ, TB, DELTA)                                \
    do {                                                       \
        if (lean && !DELTA) QSV_SCAN_V(TQ, TB, false, true, 8, 1, 3);   \
        else if (vec && R == 8) QSV_SCAN_V(TQ, TB, DELTA, true, 8, 1, 1);   \
        else if (R == 8) QSV_SCAN_V(TQ, TB, DELTA, false, 8, 1, 1);    \
        else if (vec) QSV_SCAN_V(TQ, TB, DELTA, true, 16, 1, 1);       \
        else QSV_SCAN_V(TQ, TB, DELTA, false, 16, 1, 1);               \
    } while (0)
    if (beta) {
        if (qkv_dtype == QSV_F32 && beta_dtype == QSV_F32) QSV_SCAN(float, float, true);
        else if (qkv_dtype == QSV_F32 && beta_dtype == QSV_BF16) QSV_SCAN(float, bf16_t, true);
        else if (qkv_dtype == QSV_BF16 && beta_dtype == QSV_BF16) QSV_SCAN(bf16_t, bf16_t, true);
        else QSV_REQUIRE(false, "qsv_recurrent_scan: operand types %d / %d", qkv_dtype, beta_dtype);
    } else {
        if (qkv_dtype == QSV_F32) QSV_SCAN(float, float, false);
        else if (qkv_dtype == QSV_BF16) QSV_SCAN(bf16_t, bf16_t, false);
        else QSV_REQUIRE(false, "qsv_recurrent_scan: operand type %d", qkv_dtype);
    }
#undef QSV_SCAN
#undef QSV_SCAN_V
    return qsv_launch_status("qsv_recurrent_scan");
}

// One token per run and what qsv_head_rms_gate makes of its read-out, in one launch
extern "C" int qsv_recurrent_step_gated(void* out, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride, int qkv_dtype,
                                        const float* decay, const void* beta, int64_t beta_stride, int beta_dtype, float* state, const int32_t* runs, int n_runs,
                                        int heads, int qk_heads, int dim, int vdim, float q_scale, int head_decay, const void* w, const void* gate,
                                        int64_t gate_stride, int gate_kind, float eps, void* stream) {
    QSV_REQUIRE(out && q && k && v && decay && state && runs && w && gate && n_runs > 0 && (gate_kind == 0 || gate_kind == 1), "qsv_recurrent_step_gated: bad arguments");
    const int qkv = qkv_dtype == QSV_F32 ? QSV_F32 : QSV_BF16;
    QSV_REQUIRE(heads > 0 && qk_heads > 0 && heads % qk_heads == 0 && heads <= 65535 && dim > 0 && dim % 8 == 0 && dim <= 256 && vdim >= 4 && vdim <= 128 &&
                    (vdim & (vdim - 1)) == 0 && gate_stride >= (int64_t)heads * vdim,
                "qsv_recurrent_step_gated: %d heads over %d of %d x %d", heads, qk_heads, dim, vdim);
    QSV_REQUIRE(q_stride % 4 == 0 && k_stride % 4 == 0 && gate_stride % 4 == 0 && fits4(q, qkv) && fits4(k, qkv) && fits4(decay, QSV_F32) && fits4(state, QSV_F32) &&
                    fits4(out, QSV_BF16) && fits4(w, QSV_BF16) && fits4(gate, QSV_BF16), "qsv_recurrent_step_gated: operands of four start inside four");
    const GateTail tail = {(bf16_t*)out, (const bf16_t*)w, (const bf16_t*)gate, gate_stride, gate_kind, eps};
    const dim3 grid(n_runs, heads), block(256);
    float* o = nullptr;
    const float* kscale = nullptr;
    const int v_cols = vdim;
#define QSV_STEP_P(TQ, TB, DELTA, P)                                                                                                  \
    hipLaunchKernelGGL((recurrent_step_wide_kernel<TQ, TB, DELTA, P, true>), grid, block, 0, (hipStream_t)stream, o, (const TQ*)q, q_stride, \
                       (const TQ*)k, k_stride, (const TQ*)v, v_stride, decay, (const TB*)beta, beta_stride, state, runs, heads,        \
                       qk_heads, dim, vdim, q_scale, kscale, head_decay, v_cols, tail)
#define QSV_STEP(TQ, TB, DELTA)                            \
    do {                                                   \
        if (dim <= 64) QSV_STEP_P(TQ, TB, DELTA, 1);       \
        else if (dim <= 128) QSV_STEP_P(TQ, TB, DELTA, 2); \
        else QSV_STEP_P(TQ, TB, DELTA, 4);                 \
    } while (0)
    QSV_STEP_TYPES
#undef QSV_STEP
#undef QSV_STEP_P
    return qsv_launch_status("qsv_recurrent_step_gated");
}

extern "C" int qsv_head_rms_gate(void* out, const float* o, const void* w, const void* gate, int64_t gate_stride, int gate_kind,
                                 float eps, int n_tokens, int heads, int vdim, int o_stride, int w_per_head, const float* den_m,
                                 int dtype, void* stream) {
    QSV_REQUIRE(out && o && w && gate && n_tokens >= 0 && heads > 0 && vdim > 0 && gate_stride >= (int64_t)heads * vdim &&
                    (gate_kind == 0 || gate_kind == 1),
                "qsv_head_rms_gate: bad arguments");
    if (o_stride <= 0) o_stride = vdim;
    QSV_REQUIRE(o_stride >= vdim && (!den_m || o_stride > vdim), "qsv_head_rms_gate: read-out rows of %d floats for %d values%s",
                o_stride, vdim, den_m ? " and the normaliser's column" : "");
    if (n_tokens == 0) return QSV_OK;
    if (vdim >= 4 && vdim <= 256 && (vdim & (vdim - 1)) == 0 && o_stride % 4 == 0 && gate_stride % 4 == 0 && fits4(out, dtype) &&
        fits4(o, QSV_F32) && fits4(w, dtype) && fits4(gate, dtype) && heads <= (1 << 20)) {
        int lanes_log = 0;
        while ((4 << lanes_log) < vdim) ++lanes_log;
        const int64_t n_heads = (int64_t)n_tokens * heads, lanes = n_heads << lanes_log;
        if (lanes < (1ll << 32) - NT) {
            QSV_DISPATCH(dtype, "qsv_head_rms_gate",
                         hipLaunchKernelGGL(head_rms_gate_vec_kernel<T>, dim3((unsigned)((lanes + NT - 1) / NT)), dim3(NT), 0, (hipStream_t)stream,
                                            (T*)out, o, (const T*)w, (const T*)gate, gate_stride, gate_kind, eps, heads, vdim, lanes_log, o_stride,
                                            w_per_head ? vdim : 0, den_m, (unsigned)n_heads));
            return qsv_launch_status("qsv_head_rms_gate");
        }
    }
    QSV_DISPATCH(dtype, "qsv_head_rms_gate",
                 hipLaunchKernelGGL(head_rms_gate_kernel<T>, dim3(n_tokens), dim3(NT), 0, (hipStream_t)stream, (T*)out, o, (const T*)w,
                                    (const T*)gate, gate_stride, gate_kind, eps, heads, vdim, o_stride, w_per_head ? vdim : 0, den_m));
    return qsv_launch_status("qsv_head_rms_gate");
}

extern "C" int qsv_max_gates(float* a, float* b, float* m, const void* zi, const void* zf, int64_t z_stride, const float* bias_i,
                             const float* bias_f, float cap, float* m_state, const int32_t* runs, int n_runs, int heads, int dtype,
                             void* stream) {
    QSV_REQUIRE(a && b && m && zi && zf && bias_i && bias_f && m_state && runs, "qsv_max_gates: null argument");
    QSV_REQUIRE(cap > 0.f && heads > 0 && heads <= 65535 && n_runs >= 0 && z_stride >= heads, "qsv_max_gates: bad sizes");
    if (n_runs == 0) return QSV_OK;
    QSV_DISPATCH(dtype, "qsv_max_gates",
                 hipLaunchKernelGGL(max_gates_kernel<T>, dim3(n_runs, heads), dim3(64), 0, (hipStream_t)stream, a, b, m, (const T*)zi,
                                    (const T*)zf, z_stride, bias_i, bias_f, cap, m_state, runs, heads));
    return qsv_launch_status("qsv_max_gates");
}

extern "C" int qsv_attention_prep(float* qf, void* pool, int64_t pool_rows, const void* proj, int64_t stride, int q_off, int k_off,
                                  int v_off, int heads, int kv_heads, int dim, int vdim, int rot_n, const float* rope_k,
                                  const float* rope_v, float scale, const int64_t* slot, const int32_t* pos, int n_tokens,
                                  int dtype, void* stream) {
    QSV_REQUIRE(qf && pool && proj && (rope_k || rot_n == 0) && rope_v && slot && pos, "qsv_attention_prep: null argument");
    QSV_REQUIRE(heads > 0 && kv_heads > 0 && dim > 0 && vdim > 0 && vdim % 2 == 0 && rot_n >= 0 && rot_n % 2 == 0 && rot_n <= dim &&
                    q_off >= 0 && k_off >= 0 && v_off >= 0 && q_off + (int64_t)heads * dim <= stride &&
                    k_off + (int64_t)kv_heads * dim <= stride && v_off + (int64_t)kv_heads * vdim <= stride && n_tokens >= 0,
                "qsv_attention_prep: bad sizes");
    if (n_tokens == 0) return QSV_OK;
    const int64_t chunks = (((int64_t)heads + kv_heads) * ((vdim + dim) / 4) + NT - 1) / NT;
    if (dim % 4 == 0 && vdim % 8 == 0 && rot_n % 8 == 0 && stride % 4 == 0 && q_off % 4 == 0 && k_off % 4 == 0 && v_off % 4 == 0 &&
        fits4(qf, QSV_F32) && fits4(pool, dtype) && fits4(proj, dtype) && fits4(rope_k, QSV_F32) && fits4(rope_v, QSV_F32) &&
        chunks * n_tokens < (1ll << 31) && chunks < (1 << 22)) {
        QSV_DISPATCH(dtype, "qsv_attention_prep",
                     hipLaunchKernelGGL(attention_prep_vec_kernel<T>, dim3((unsigned)(chunks * n_tokens)), dim3(NT), 0, (hipStream_t)stream, qf,
                                        (T*)pool, pool_rows, (const T*)proj, stride, q_off, k_off, v_off, heads, kv_heads, dim, vdim, rot_n, rope_k,
                                        rope_v, scale, slot, pos, (int)chunks));
        return qsv_launch_status("qsv_attention_prep");
    }
    QSV_DISPATCH(dtype, "qsv_attention_prep",
                 hipLaunchKernelGGL(attention_prep_kernel<T>, dim3(n_tokens), dim3(NT), 0, (hipStream_t)stream, qf, (T*)pool, pool_rows,
                                    (const T*)proj, stride, q_off, k_off, v_off, heads, kv_heads, dim, vdim, rot_n, rope_k, rope_v,
                                    scale, slot, pos));
    return qsv_launch_status("qsv_attention_prep");
}

extern "C" int qsv_rotate_heads(void* o, const float* rope, const int32_t* pos, float sign, int n_tokens, int heads, int n,
                                int dtype, void* stream) {
    QSV_REQUIRE(o && rope && pos && n_tokens >= 0 && heads > 0 && n > 0 && n % 2 == 0, "qsv_rotate_heads: bad arguments");
    if (n_tokens == 0) return QSV_OK;
    if (n % 8 == 0 && fits4(o, dtype) && fits4(rope, QSV_F32))
        QSV_DISPATCH(dtype, "qsv_rotate_heads",
                     hipLaunchKernelGGL((rotate_heads_kernel<T, true>), dim3(n_tokens), dim3(NT), 0, (hipStream_t)stream, (T*)o, rope, pos, sign, heads, n));
    else
        QSV_DISPATCH(dtype, "qsv_rotate_heads",
                 hipLaunchKernelGGL((rotate_heads_kernel<T, false>), dim3(n_tokens), dim3(NT), 0, (hipStream_t)stream, (T*)o, rope, pos, sign,
                                    heads, n));
    return qsv_launch_status("qsv_rotate_heads");
}


// ---- element-wise gated recurrence (minGRU) ---------------------------------------------------------------------------------------
// Thread = one channel of one run; the run's tokens are walked in order, UN at a time: the UN tokens' three pre-activations are
// requested together (rows of the batch, coalesced over the channels), the gates are computed, then the UN dependent steps run.
// Gates, candidate and state are float.
template <typename T>
__global__ __launch_bounds__(NT) void min_gru_scan_kernel(T* __restrict__ out, const T* __restrict__ proj, int64_t stride, int z_off,
                                                          int x_off, int g_off, const T* __restrict__ b_z, const T* __restrict__ b_x,
                                                          float* __restrict__ state, const int32_t* __restrict__ runs, int width) {
    constexpr int UN = 8;
    const int i = blockIdx.x * NT + threadIdx.x;
    if (i >= width) return;
    const int32_t* r = runs + 4 * blockIdx.y;
    const int slot = r[0], first = r[1], n = r[2], p0 = r[3];
    float S = p0 > 0 ? state[(size_t)slot * width + i] : 0.f;
    const float bz = ld(b_z, i), bx = ld(b_x, i);
    for (int t0 = 0; t0 < n; t0 += UN) {
        float z[UN], u[UN], g[UN];
#pragma unroll
        for (int j = 0; j < UN; ++j) {
            const size_t row = (size_t)(first + min(t0 + j, n - 1)) * stride;
            z[j] = ld(proj, row + z_off + i);
            u[j] = ld(proj, row + x_off + i);
            g[j] = ld(proj, row + g_off + i);
        }
#pragma unroll
        for (int j = 0; j < UN; ++j) {
            z[j] = 1.0f / (1.0f + expf(-(z[j] + bz)));
            const float uu = u[j] + bx;
            u[j] = uu >= 0.f ? uu + 0.5f : 1.0f / (1.0f + expf(-uu));
            g[j] = g[j] / (1.0f + expf(-g[j]));
        }
#pragma unroll
        for (int j = 0; j < UN; ++j) {
            if (t0 + j < n) {
                S = (1.0f - z[j]) * S + z[j] * u[j];
                st(out, (size_t)(first + t0 + j) * width + i, S * g[j]);
            }
        }
    }
    state[(size_t)slot * width + i] = S;
}
// Long runs (prompt portions): a workgroup of SEG waves owns 64 channels of one run and cuts the run's tokens into SEG segments, one
// a wave.  The recurrence S <- a S + b (a = 1 - z, b = z c) composes: a segment as a whole maps S to A S + B with A the product of
// its a and B its own scan from zero.  Pass 1: every wave walks its segment for (A, B); the waves exchange them through LDS and each
// folds its predecessors' into the state its segment starts from; pass 2: the segment again (from L2), now with outputs.
template <typename T>
__global__ __launch_bounds__(64 * 8) void min_gru_scan_segments_kernel(T* __restrict__ out, const T* __restrict__ proj, int64_t stride,
                                                                       int z_off, int x_off, int g_off, const T* __restrict__ b_z,
                                                                       const T* __restrict__ b_x, float* __restrict__ state,
                                                                       const int32_t* __restrict__ runs, int width) {
    constexpr int SEG = 8, UN = 8;
    __shared__ float sA[SEG][64], sB[SEG][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ch = blockIdx.x * 64 + lane;
    const bool valid = ch < width;
    const int i = valid ? ch : width - 1;
    const int32_t* r = runs + 4 * blockIdx.y;
    const int slot = r[0], first = r[1], n = r[2], p0 = r[3];
    const int per = (n + SEG - 1) / SEG;
    const int t_lo = min(n, w * per), t_hi = min(n, t_lo + per);
    const float bz = ld(b_z, i), bx = ld(b_x, i);
    float A = 1.f, B = 0.f;
    for (int t0 = t_lo; t0 < t_hi; t0 += UN) {
        float z[UN], u[UN];
#pragma unroll
        for (int j = 0; j < UN; ++j) {
            const size_t row = (size_t)(first + min(t0 + j, t_hi - 1)) * stride;
            z[j] = ld(proj, row + z_off + i);
            u[j] = ld(proj, row + x_off + i);
        }
#pragma unroll
        for (int j = 0; j < UN; ++j) {
            const float zz = 1.0f / (1.0f + expf(-(z[j] + bz)));
            const float uu = u[j] + bx;
            const float c = uu >= 0.f ? uu + 0.5f : 1.0f / (1.0f + expf(-uu));
            if (t0 + j < t_hi) {
                A *= 1.0f - zz;
                B = (1.0f - zz) * B + zz * c;
            }
        }
    }
    sA[w][lane] = A;
    sB[w][lane] = B;
    __syncthreads();
    float S = p0 > 0 ? state[(size_t)slot * width + i] : 0.f;
    for (int k = 0; k < w; ++k) S = sA[k][lane] * S + sB[k][lane];
    for (int t0 = t_lo; t0 < t_hi; t0 += UN) {
        float z[UN], u[UN], g[UN];
#pragma unroll
        for (int j = 0; j < UN; ++j) {
            const size_t row = (size_t)(first + min(t0 + j, t_hi - 1)) * stride;
            z[j] = ld(proj, row + z_off + i);
            u[j] = ld(proj, row + x_off + i);
            g[j] = ld(proj, row + g_off + i);
        }
#pragma unroll
        for (int j = 0; j < UN; ++j) {
            z[j] = 1.0f / (1.0f + expf(-(z[j] + bz)));
            const float uu = u[j] + bx;
            u[j] = uu >= 0.f ? uu + 0.5f : 1.0f / (1.0f + expf(-uu));
            g[j] = g[j] / (1.0f + expf(-g[j]));
        }
#pragma unroll
        for (int j = 0; j < UN; ++j) {
            if (t0 + j < t_hi) {
                S = (1.0f - z[j]) * S + z[j] * u[j];
                if (valid) st(out, (size_t)(first + t0 + j) * width + i, S * g[j]);
            }
        }
    }
    if (w == SEG - 1 && valid) state[(size_t)slot * width + i] = S;     // (the last wave ends with the run's last state, also if its segment is empty)
}
extern "C" int qsv_min_gru_scan(void* out, const void* proj, int64_t stride, int z_off, int x_off, int g_off, const void* b_z,
                                const void* b_x, float* state, const int32_t* runs, int n_runs, int max_run, int width, int dtype,
                                void* stream) {
    QSV_REQUIRE(out && proj && b_z && b_x && state && runs, "qsv_min_gru_scan: null argument");
    QSV_REQUIRE(width > 0 && n_runs >= 0 && n_runs <= 65535 && z_off >= 0 && x_off >= 0 && g_off >= 0 &&
                    (int64_t)z_off + width <= stride && (int64_t)x_off + width <= stride && (int64_t)g_off + width <= stride,
                "qsv_min_gru_scan: bad sizes");
    if (n_runs == 0) return QSV_OK;
    if (max_run <= 0 || max_run > 32) {          // (0: unknown) long runs: segments of the run side by side
        QSV_DISPATCH(dtype, "qsv_min_gru_scan",
                     hipLaunchKernelGGL(min_gru_scan_segments_kernel<T>, dim3((width + 63) / 64, n_runs), dim3(64 * 8), 0,
                                        (hipStream_t)stream, (T*)out, (const T*)proj, stride, z_off, x_off, g_off, (const T*)b_z,
                                        (const T*)b_x, state, runs, width));
        return qsv_launch_status("qsv_min_gru_scan");
    }
    QSV_DISPATCH(dtype, "qsv_min_gru_scan",
                 hipLaunchKernelGGL(min_gru_scan_kernel<T>, dim3((width + NT - 1) / NT, n_runs), dim3(NT), 0, (hipStream_t)stream,
                                    (T*)out, (const T*)proj, stride, z_off, x_off, g_off, (const T*)b_z, (const T*)b_x, state, runs,
                                    width));
    return qsv_launch_status("qsv_min_gru_scan");
}
