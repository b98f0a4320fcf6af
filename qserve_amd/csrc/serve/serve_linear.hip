// serve_linear.hip -- x [T, K] @ w [N, K]^T for the few rows of a decoding step (bfloat16, float accumulation).
//
// Bound by HBM (the weight, read once) and below about 20 MB by the launch.  Workgroup = 16 or 32 weight rows and up to 32 inputs, the
// weight streamed through LDS rings (serve_stream.h), the four waves' shares of the reduction added in LDS.
// Measured against the vendor's product (MI355X, weights from HBM, 1 / 16 / 32 / 64 rows, us): 2048 x 2048 4.5 / 4.7 / 5.5 / 5.6 against 8.1 / 8.2 / 8.4 /
// 8.8; 6144 x 2048 7.4 / 7.6 / 8.4 / 10.9 against 12.7 / 12.5 / 12.4 / 13.0; 32000 x 2048 27 / 28 / 30 / 47 against 34 / 34 / 35 / 35.
#include "serve_common.h"
#include "serve_stream.h"

namespace {
template <int RB, int SG>
__global__ __launch_bounds__(64 * STREAM_WAVES, 2) void skinny_linear_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ X, int64_t x_stride,
                                                                            const bf16_t* __restrict__ W, int T, int N, int K, int wide) {
    __shared__ __attribute__((aligned(128))) unsigned char rings[STREAM_WAVES * XRING];
    constexpr int TILES = RB * SG;
    static_assert(STREAM_WAVES * TILES * 1024 <= STREAM_WAVES * XRING, "");
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = blockIdx.x * 16 * RB, t0 = blockIdx.y * 16 * SG, count = min(16 * SG, T - t0);
    v4f acc[RB][SG];
    stream_products<RB, SG>(W + (size_t)r0 * K, K, min(16 * RB, N - r0), rings + w * XRING, w, lane,
                            [&](int i) { return X + (size_t)(t0 + min(i, count - 1)) * (size_t)x_stride; }, acc);
    v4f* red = (v4f*)rings;                                         // [wave][tile][lane]
    __syncthreads();                                                // every wave is done with its ring
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int g = 0; g < SG; ++g) red[(w * TILES + r * SG + g) * 64 + lane] = acc[r][g];
    __syncthreads();
    for (int t = w; t < TILES; t += STREAM_WAVES) {
        const int c = 16 * (t % SG) + (lane & 15), n = r0 + 16 * (t / SG) + 4 * (lane >> 4);
        if (c >= count) continue;
        v4f v = red[t * 64 + lane];
#pragma unroll
        for (int o = 1; o < STREAM_WAVES; ++o) v += red[(o * TILES + t) * 64 + lane];
        bf16_t* p = out + (size_t)(t0 + c) * N + n;
        if (wide && n + 4 <= N) {
            *(uint2*)p = make_uint2((unsigned)f2bf(v[0]) | ((unsigned)f2bf(v[1]) << 16), (unsigned)f2bf(v[2]) | ((unsigned)f2bf(v[3]) << 16));
        } else {
            for (int q = 0; q < 4; ++q)
                if (n + q < N) p[q] = f2bf(v[q]);
        }
    }
}
}  // namespace

extern "C" int qsv_skinny_linear(void* out, const void* x, int64_t x_stride, const void* w, int n_rows, int N, int K, void* stream) {
    QSV_REQUIRE(out && x && w && n_rows >= 0 && N > 0 && K > 0 && K % 8 == 0 && x_stride % 8 == 0 && x_stride >= 0, "qsv_skinny_linear: bad arguments");
    QSV_REQUIRE(((uintptr_t)x | (uintptr_t)w) % 16 == 0, "qsv_skinny_linear: inputs and weights start on 16 bytes");
    QSV_REQUIRE(K <= (1 << 25) && n_rows <= 65535 * 16, "qsv_skinny_linear: %d inputs of %d", n_rows, K);
    if (n_rows == 0) return QSV_OK;
    const int wide = N % 4 == 0 && (uintptr_t)out % 8 == 0;
    // 16 weight rows per workgroup where 32 would leave CUs without one, or need a second round for a few (8256 x 2048: 11.4 -> 10.5 us); else 32,
    // which reads the inputs half as often (6144 x 2048: 8.2 -> 7.4 us)
    const bool few = n_rows <= 16, small = N < 5120 || (N > 8192 && N <= 16384 && n_rows <= 32);
#define QSV_SKINNY(RB, SG)                                                                                                                    \
    hipLaunchKernelGGL((skinny_linear_kernel<RB, SG>), dim3((N + 16 * RB - 1) / (16 * RB), (n_rows + 16 * SG - 1) / (16 * SG)),               \
                       dim3(64 * STREAM_WAVES), 0, (hipStream_t)stream, (bf16_t*)out, (const bf16_t*)x, x_stride, (const bf16_t*)w, n_rows, N, K, wide)
    if (few && small) QSV_SKINNY(1, 1);
    else if (few) QSV_SKINNY(2, 1);
    else if (small) QSV_SKINNY(1, 2);
    else QSV_SKINNY(2, 2);
#undef QSV_SKINNY
    return qsv_launch_status("qsv_skinny_linear");
}
