// dW [K, N] = dY [M, K]^T * X0 [M, N] for a narrow N (64 or 128) and many rows M, bf16 in, fp32 accumulation, bf16 out.
//
// This is the weight gradient of the second half of the HDLA layer's low-rank projections (f_proj and output_gate:
// Linear(embed_dim -> head_dim) followed by Linear(head_dim -> embed_dim), HRDPLR/hdla_custom.py:117-121,151-155; in the
// reference a BLAS call inside autograd).  The output is tiny (K x N) and the contraction runs over all rows, so a
// BLAS kernel tiled over the output has 16 workgroups to work with; here the rows are split as well: a workgroup owns
// 32 columns of dY and one range of rows, its four wavefronts take every fourth 16-row tile of that range (16 bytes a
// lane from dY and from X0), add their sums through LDS, and leave a fp32 partial result; a second small kernel adds
// the partial results of the row ranges in a fixed order.
//
// The contraction index (the row) must be the inner index of both MFMA operands, and both are stored with the row
// outermost, so each 16 x 16 tile is transposed on its way in by one product with the identity (exact in bf16).
#include "hdla_common.cuh"
#include "../../include/hdla_hip.h"

namespace hdla {

// Two 16 x 16 tiles from one 16-byte load per lane: lane (g, c) reads elements 8g .. 8g+7 of row c of a 16 x 32 block;
// the first four are the fragment of tile A, the last four of tile B, where tile A holds the block's columns
// 8j + 0..3 and tile B the columns 8j + 4..7 (j = 0..3).  Element e = 0..15 of a tile's column index is therefore
// column 8 (e / 4) + e % 4 (+ 4 for tile B) of the block.
__device__ __forceinline__ void ld_two_tiles(const bf16* p, bool ok, Frag<bf16>& a, Frag<bf16>& b) {
    s16x8 x = *reinterpret_cast<const s16x8*>(p);
    const s16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    x = ok ? x : z;
    a.v = __builtin_shufflevector(x, x, 0, 1, 2, 3);
    b.v = __builtin_shufflevector(x, x, 4, 5, 6, 7);
}

// One product, or the two of the layer (blockIdx.z).  With F given the gradient is that of logsigmoid(F): dY sigmoid(-F),
// rounded to bf16 as a stored gradient would be (forming it here saves a pass over it: 10.7 us of 8192 x 1024).
struct WgradArgs {
    const bf16 *dY[2], *F[2], *X0[2];
    float* part[2];
    long long ldy, ldx;
    int M, K, rows_per;
};
template <int N>
__global__ __launch_bounds__(256) void skinny_wgrad_kernel(WgradArgs p) {
    const int which = blockIdx.z;
    const bf16* __restrict__ dY = p.dY[which];
    const bf16* __restrict__ F = p.F[which];
    const bf16* __restrict__ X0 = p.X0[which];
    float* __restrict__ part = p.part[which];
    const long long ldy = p.ldy, ldx = p.ldx;
    const int M = p.M, K = p.K, rows_per = p.rows_per;
    constexpr int ZP = N / 32;                                 // 32-column blocks of X0
    __shared__ f32x4 red[3][2 * 2 * ZP][64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const int k0 = blockIdx.x * 32, s = blockIdx.y;
    const long long rbeg = (long long)s * rows_per;
    const long long rend = rbeg + rows_per < M ? rbeg + rows_per : M;
    const Frag<bf16> id = ident_frag<bf16>();
    f32x4 acc[2][2 * ZP];                                      // [tile of dY's 32 columns][tile of X0's columns]
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2 * ZP; ++b) acc[a][b] = zero4();
    // the four wavefronts take every fourth 16-row tile of the range
#pragma unroll 4
    for (long long r0 = rbeg + 16 * w; r0 < rend; r0 += 64) {
        const bool ok = r0 + c < rend;
        const long long row = ok ? r0 + c : rbeg;              // a readable row on every lane
        Frag<bf16> x[2], z[2 * ZP];
        ld_two_tiles(dY + row * ldy + k0 + 8 * g, ok, x[0], x[1]);
#pragma unroll
        for (int b = 0; b < ZP; ++b) ld_two_tiles(X0 + row * ldx + 32 * b + 8 * g, ok, z[2 * b], z[2 * b + 1]);
        if (F) {
            Frag<bf16> f[2];
            ld_two_tiles(F + row * ldy + k0 + 8 * g, ok, f[0], f[1]);
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                f32x4 d = to_f32(x[a]);
                const f32x4 t = to_f32(f[a]);
                float e[4], s[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) e[i] = __expf(t[i]);
                sigmoid_of_exp<4>(e, s);
#pragma unroll
                for (int i = 0; i < 4; ++i) d[i] *= s[i];
                x[a] = to_frag<bf16>(d);
            }
        }
        // transposed tiles: rows = columns of the block, inner index = row of the range
        x[0] = transpose(x[0], id);
        x[1] = transpose(x[1], id);
#pragma unroll
        for (int b = 0; b < 2 * ZP; ++b) {
            const Frag<bf16> zt = transpose(z[b], id);
            acc[0][b] = mm(x[0], zt, acc[0][b]);
            acc[1][b] = mm(x[1], zt, acc[1][b]);
        }
    }
    if (w) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2 * ZP; ++b) red[w - 1][a * 2 * ZP + b][lane] = acc[a][b];
    }
    __syncthreads();
    if (w) return;
    // lane (g, c) register i of acc[a][b]: dY column k0 + 8 (c / 4) + c % 4 + 4 a,
    //                                      X0 column 32 (b / 2) + 8 g + 4 (b % 2) + i
    const int krow = k0 + 8 * (c >> 2) + (c & 3);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2 * ZP; ++b) {
            const f32x4 v = acc[a][b] + red[0][a * 2 * ZP + b][lane] + red[1][a * 2 * ZP + b][lane] + red[2][a * 2 * ZP + b][lane];
            *reinterpret_cast<f32x4*>(part + ((long long)s * K + krow + 4 * a) * N + 32 * (b >> 1) + 8 * g + 4 * (b & 1)) = v;
        }
}

// dW = sum over the row ranges of their partial results, eight outputs a thread
__global__ __launch_bounds__(256) void skinny_wgrad_sum_kernel(const float* __restrict__ part0, const float* __restrict__ part1,
                                                               bf16* __restrict__ dW0, bf16* __restrict__ dW1, long long kn, int S) {
    const float* const part = blockIdx.y ? part1 : part0;
    bf16* const dW = blockIdx.y ? dW1 : dW0;
    const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i >= kn) return;
    f32x4 a = zero4(), b = zero4();
    for (int s = 0; s < S; ++s) {
        a += *reinterpret_cast<const f32x4*>(part + s * kn + i);
        b += *reinterpret_cast<const f32x4*>(part + s * kn + i + 4);
    }
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    u32x4 o;
    o[0] = (uint32_t)f2bf(a[0]) | ((uint32_t)f2bf(a[1]) << 16);
    o[1] = (uint32_t)f2bf(a[2]) | ((uint32_t)f2bf(a[3]) << 16);
    o[2] = (uint32_t)f2bf(b[0]) | ((uint32_t)f2bf(b[1]) << 16);
    o[3] = (uint32_t)f2bf(b[2]) | ((uint32_t)f2bf(b[3]) << 16);
    *reinterpret_cast<u32x4*>(dW + i) = o;
}

// row ranges: enough workgroups for the chip (and, when there are many rows, several per CU, about 1024 rows each, so
// that enough loads are in flight to cover the latency of HBM), whole 16-row tiles each
static int wgrad_split(long long M, int K, int& rows_per) {
    const int kb = K / 32;
    long long S = (256 + kb - 1) / kb;
    const long long by_rows = M / 1024, most = (2048 + kb - 1) / kb;
    if (by_rows > S) S = by_rows < most ? by_rows : most;
    const long long tiles = (M + 15) / 16;
    if (S > tiles) S = tiles;
    if (S < 1) S = 1;
    rows_per = (int)(((tiles + S - 1) / S) * 16);
    return (int)((M + rows_per - 1) / rows_per);
}

}  // namespace hdla

using namespace hdla;

// `count` products (1 or 2), then the sums of their partial results
static int wgrad_launch(const WgradArgs& a, int N, int S, int count, bf16* dW0, bf16* dW1, hipStream_t s) {
    const dim3 grid(a.K / 32, S, count), block(256);
    if (N == 64) hipLaunchKernelGGL((skinny_wgrad_kernel<64>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((skinny_wgrad_kernel<128>), grid, block, 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    const long long kn = (long long)a.K * N;
    hipLaunchKernelGGL(skinny_wgrad_sum_kernel, dim3((unsigned)((kn / 8 + 255) / 256), count), block, 0, s, a.part[0], a.part[1], dW0, dW1, kn, S);
    e = hipGetLastError();
    return e == hipSuccess ? HDLA_OK : (int)e;
}

static int wgrad_check(int dtype, int64_t M, int32_t N, int32_t K) {
    if (dtype != HDLA_BF16) return HDLA_ERR_DTYPE;
    if (M <= 0 || M > 0x7fffffffLL || (N != 64 && N != 128) || K <= 0 || K % 64) return HDLA_ERR_SHAPE;
    return HDLA_OK;
}

extern "C" size_t hdla_skinny_wgrad_workspace_bytes(int dtype, int64_t M, int32_t N, int32_t K) {
    if (wgrad_check(dtype, M, N, K)) return 0;
    int rows_per;
    const int S = wgrad_split(M, K, rows_per);
    return (size_t)S * K * N * sizeof(float);
}

extern "C" int hdla_skinny_wgrad(int dtype, int64_t M, int32_t N, int32_t K, const void* dY, int64_t ldy,
                                 const void* X0, int64_t ldx, void* dW, void* workspace, size_t workspace_bytes,
                                 void* stream) {
    const int rc = wgrad_check(dtype, M, N, K);
    if (rc) return rc;
    if (ldy < K || ldx < N) return HDLA_ERR_SHAPE;
    if (!dY || !X0 || !dW) return HDLA_ERR_NULL;
    const auto al = [](const void* p, int a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
    if (!al(dY, 16) || !al(X0, 16) || !al(dW, 16) || ldy % 8 || ldx % 8) return HDLA_ERR_ALIGN;
    int rows_per;
    const int S = wgrad_split(M, K, rows_per);
    const size_t need = (size_t)S * K * N * sizeof(float);
    if (!workspace || !al(workspace, 16) || workspace_bytes < need) return HDLA_ERR_WORKSPACE;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    WgradArgs a{};
    a.dY[0] = static_cast<const bf16*>(dY); a.X0[0] = static_cast<const bf16*>(X0); a.part[0] = static_cast<float*>(workspace);
    a.ldy = ldy; a.ldx = ldx; a.M = (int)M; a.K = K; a.rows_per = rows_per;
    return wgrad_launch(a, N, S, 1, static_cast<bf16*>(dW), nullptr, static_cast<hipStream_t>(stream));
}

static int up_wgrad_check(const hdla_up_dims* q) {
    if (!q) return HDLA_ERR_NULL;
    const int rc = wgrad_check(HDLA_BF16, q->rows, q->D, q->d);
    if (rc) return rc;
    if (q->ld < q->D || q->ld % 8 || q->col_f < 0 || q->col_g < 0 || q->col_f % 8 || q->col_g % 8) return HDLA_ERR_ALIGN;
    return q->col_f + q->D > q->ld || q->col_g + q->D > q->ld ? HDLA_ERR_SHAPE : HDLA_OK;
}

extern "C" size_t hdla_layer_up_wgrad_workspace_bytes(const hdla_up_dims* dims) {
    if (up_wgrad_check(dims)) return 0;
    int rows_per;
    return (size_t)wgrad_split(dims->rows, dims->d, rows_per) * dims->d * dims->D * sizeof(float) * 2;
}

extern "C" int hdla_layer_up_wgrad(const hdla_up_dims* dims, const void* y, const void* f, const void* dlog_f, const void* dgate, void* dwf,
                                   void* dwg, void* workspace, size_t workspace_bytes, void* stream) {
    const int rc = up_wgrad_check(dims);
    if (rc) return rc;
    if (!y || !f || !dlog_f || !dgate || !dwf || !dwg) return HDLA_ERR_NULL;
    for (const void* p : {y, f, dlog_f, dgate, (const void*)dwf, (const void*)dwg})
        if (reinterpret_cast<uintptr_t>(p) & 15) return HDLA_ERR_ALIGN;
    int rows_per;
    const int S = wgrad_split(dims->rows, dims->d, rows_per);
    const size_t one = (size_t)S * dims->d * dims->D;
    if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 15) || workspace_bytes < 2 * one * sizeof(float)) return HDLA_ERR_WORKSPACE;
    WgradArgs a{};
    a.dY[0] = static_cast<const bf16*>(dlog_f); a.dY[1] = static_cast<const bf16*>(dgate);
    a.F[0] = static_cast<const bf16*>(f);
    a.X0[0] = static_cast<const bf16*>(y) + dims->col_f; a.X0[1] = static_cast<const bf16*>(y) + dims->col_g;
    a.part[0] = static_cast<float*>(workspace); a.part[1] = a.part[0] + one;
    a.ldy = dims->d; a.ldx = dims->ld; a.M = (int)dims->rows; a.K = dims->d; a.rows_per = rows_per;
    return wgrad_launch(a, dims->D, S, 2, static_cast<bf16*>(dwf), static_cast<bf16*>(dwg), static_cast<hipStream_t>(stream));
}

extern "C" int hdla_sum_partials(const float* part, int32_t count, int64_t n, void* out, void* stream) {
    if (count < 1 || n < 0 || n % 8) return HDLA_ERR_SHAPE;
    if (n == 0) return HDLA_OK;
    if (!part || !out) return HDLA_ERR_NULL;
    if (((reinterpret_cast<uintptr_t>(part) | reinterpret_cast<uintptr_t>(out)) & 15) != 0) return HDLA_ERR_ALIGN;
    if ((n / 8 + 255) / 256 > 0x7fffffffLL) return HDLA_ERR_SHAPE;
    hipLaunchKernelGGL(skinny_wgrad_sum_kernel, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), part,
                       part, static_cast<bf16*>(out), static_cast<bf16*>(out), (long long)n, (int)count);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? HDLA_OK : (int)e;
}
