// dW [K, N] = dY [M, K]^T * X0 [M, N] for a narrow N (64 or 128) and many rows M, bf16 in, fp32 accumulation, bf16 out.
//
// This is the weight gradient of the second half of the HDLA layer's low-rank projections (f_proj and output_gate:
// Linear(embed_dim -> head_dim) followed by Linear(head_dim -> embed_dim), HRDPLR/hdla_custom.py:117-121,151-155; in the
// reference a BLAS call inside autograd).  The output is tiny (K x N) and the contraction runs over all rows, so a
// BLAS kernel tiled over the output has 16 workgroups to work with; here the rows are split as well: a workgroup owns
// 16 KA columns of dY and one range of rows, its WW wavefronts take every WW'th 32-row tile of that range, add their sums through
// LDS, and leave a fp32 partial result; a second small kernel adds the partial results of the row ranges in a fixed order.
//
// The contraction index (the row) must be the inner index of both MFMA operands, and both are stored with the row outermost: tiles of
// 32 rows go through LDS as they come (RowTile) and the transposing LDS read takes them from there.
#include "row_tile.cuh"
#include "sums.cuh"
#include "../../include/hdla_hip.h"

namespace hdla {

// One product, or the two of the layer (blockIdx.z).  With F given the gradient is that of logsigmoid(F): dY sigmoid(-F),
// rounded to bf16 as a stored gradient would be (forming it here saves a pass over it: 10.7 us of 8192 x 1024).
struct WgradArgs {
    const bf16 *dY[2], *F[2], *X0[2];
    float* part[2];
    long long ldy, ldx;
    int M, K, rows_per;
};
// Measured, both products of the layer, 8192 rows, K = 1024, N = 64 (three 16.8 MB tensors read: 10.2 us at copy rate), without the sums of
// the partial results: 25.2 us with the lanes of a request in fragment order (row_tile.cuh), tiles turned by products with the identity and
// 32 columns a workgroup; 17.5 like this.
template <int N, int KA, int WW>
__global__ __launch_bounds__(64 * WW) void skinny_wgrad_kernel(WgradArgs p) {
    const int which = blockIdx.z;
    const bf16* __restrict__ dY = p.dY[which];
    const bf16* __restrict__ F = p.F[which];
    const bf16* __restrict__ X0 = p.X0[which];
    constexpr int NB = N / 16;
    typedef RowTile<16 * KA> TY;
    typedef RowTile<N> TX;
    constexpr int RY = 32 / TY::RPR, RX = 32 / TX::RPR;        // requests of a tile of 32 rows
    constexpr int TILES = 32 * (TY::ROW + TX::ROW), SUMS = KA * NB * 1024;   // bytes a wave
    constexpr int BYTES = WW * (TILES > SUMS ? TILES : SUMS);
    static_assert(KA * NB % WW == 0, "whole tiles a wavefront");
    __shared__ __attribute__((aligned(16))) char sm[BYTES];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id(), g = l >> 4, c = l & 15;
    char* const ty = sm + wv * TILES;
    char* const tx = ty + 32 * TY::ROW;
    const int k0 = blockIdx.x * (16 * KA), s = blockIdx.y;
    const long long rbeg = (long long)s * p.rows_per;
    const long long rend = rbeg + p.rows_per < p.M ? rbeg + p.rows_per : p.M;
    f32x4 acc[KA][NB];                                         // [tile of dY's columns][tile of X0's columns]
#pragma unroll
    for (int a = 0; a < KA; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = zero4();
    // a tile's rows as they come; rows past the range: its last one again, zeros where used
    struct In { s16x8 y[RY], f[RY], x[RX]; };
    auto request = [&](long long r0) __attribute__((always_inline)) {
        In in;
#pragma unroll
        for (int j = 0; j < RY; ++j) {
            const long long at = min(r0 + TY::row(j, l), rend - 1) * p.ldy + k0 + TY::col(l);
            in.y[j] = *reinterpret_cast<const s16x8*>(dY + at);
            if (F) in.f[j] = *reinterpret_cast<const s16x8*>(F + at);
        }
#pragma unroll
        for (int j = 0; j < RX; ++j) in.x[j] = *reinterpret_cast<const s16x8*>(X0 + min(r0 + TX::row(j, l), rend - 1) * p.ldx + TX::col(l));
        return in;
    };
    long long r0 = rbeg + 32 * wv;
    In next;
    if (r0 < rend) next = request(r0);
    for (; r0 < rend; r0 += 32 * WW) {
        In in = next;
        if (r0 + 32 * WW < rend) next = request(r0 + 32 * WW);   // (the next tile's on their way while this one is worked on)
        const s16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
        const int live = (int)(rend - r0 < 32 ? rend - r0 : 32);
        if (F) {
#pragma unroll
            for (int j = 0; j < RY; ++j) in.y[j] = times_sigmoid_neg(in.y[j], in.f[j]);
        }
        wave_lds_fence();                                      // (the reads of the tile before)
#pragma unroll
        for (int j = 0; j < RY; ++j) TY::put(ty, j, l, TY::row(j, l) < live ? in.y[j] : zero);
#pragma unroll
        for (int j = 0; j < RX; ++j) TX::put(tx, j, l, TX::row(j, l) < live ? in.x[j] : zero);
        wave_lds_fence();
        Frag<bf16> y[KA][2];
#pragma unroll
        for (int a = 0; a < KA; ++a)
#pragma unroll
            for (int h = 0; h < 2; ++h) y[a][h] = TY::columns(ty, 16 * h, 4, a, l);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const Frag<bf16> x0 = TX::columns(tx, 0, 4, b, l), x1 = TX::columns(tx, 16, 4, b, l);
#pragma unroll
            for (int a = 0; a < KA; ++a) acc[a][b] = mm2(y[a][0], y[a][1], x0, x1, acc[a][b]);
        }
    }
    // the wavefronts' sums: each adds up its share of the tiles
    f32x4* const red = reinterpret_cast<f32x4*>(sm);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KA * NB; ++i) red[(wv * KA * NB + i) * 64 + l] = acc[i / NB][i % NB];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < KA * NB / WW; ++j) {
        const int i = wv * (KA * NB / WW) + j, a = i / NB, b = i % NB;
        f32x4 sum = red[i * 64 + l];
#pragma unroll
        for (int w = 1; w < WW; ++w) sum += red[(w * KA * NB + i) * 64 + l];
        // lane (g, c) register e: dY column k0 + 16 a + c, X0 column 16 b + 4 g + e
        *reinterpret_cast<f32x4*>(p.part[which] + ((long long)s * p.K + k0 + 16 * a + c) * N + 16 * b + 4 * g) = sum;
    }
}

// row ranges: enough workgroups for the chip (and, when there are many rows, several per CU, about 1024 rows each, so
// that enough loads are in flight to cover the latency of HBM), whole 32-row tiles each
static int wgrad_split(long long M, int K, int& rows_per) {
    const int kb = K / 32;
    long long S = (256 + kb - 1) / kb;
    const long long by_rows = M / 1024, most = (2048 + kb - 1) / kb;
    if (by_rows > S) S = by_rows < most ? by_rows : most;
    const long long tiles = (M + 31) / 32;
    if (S > tiles) S = tiles;
    if (S < 1) S = 1;
    rows_per = (int)(((tiles + S - 1) / S) * 32);
    return (int)((M + rows_per - 1) / rows_per);
}

}  // namespace hdla

using namespace hdla;

// `count` products (1 or 2), then the sums of their partial results
static int wgrad_launch(const WgradArgs& a, int N, int S, int count, bf16* dW0, bf16* dW1, hdla_sum* later, hipStream_t s) {
    const dim3 block(256);
    // Columns of dY and wavefronts a workgroup.  Many rows, N = 64: whole cache lines of dY and half of the reads of X0; few rows leave
    // some of eight wavefronts without any.  Both products and their sums, us, 32 columns and 4 wavefronts / 64 and 8: 8192 x 1024
    // 26.9 / 22.8, 3000 x 1024 14.7 / 14.7, 1000 x 512 9.1 / 13.8.  N = 128 has no registers for 64 columns; with 8 wavefronts, so one
    // workgroup a compute unit, 8192 x 2048 takes 61.8, with 4 52.0.
    if (N == 64 && a.M >= 2048) hipLaunchKernelGGL((skinny_wgrad_kernel<64, 4, 8>), dim3(a.K / 64, S, count), dim3(512), 0, s, a);
    else if (N == 64) hipLaunchKernelGGL((skinny_wgrad_kernel<64, 2, 4>), dim3(a.K / 32, S, count), block, 0, s, a);
    else hipLaunchKernelGGL((skinny_wgrad_kernel<128, 2, 4>), dim3(a.K / 32, S, count), block, 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    SumJob job{};
    job.kind = SUM_PARTS; job.count = S; job.n = (long long)a.K * N;
    job.blocks = (int)((job.n / 8 + 255) / 256);
    hdla_sum own[2];
    for (int i = 0; i < count; ++i) {
        job.part = a.part[i];
        job.out[0] = i ? dW1 : dW0;
        sum_now_or_later(job, (later ? later : own) + i, s);
    }
    return later ? HDLA_OK : hdla_run_sums(own, count, s);
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
    return wgrad_launch(a, N, S, 1, static_cast<bf16*>(dW), nullptr, nullptr, static_cast<hipStream_t>(stream));
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

static int layer_up_wgrad(const hdla_up_dims* dims, const void* y, const void* f, const void* dlog_f, const void* dgate, void* dwf, void* dwg, void* workspace,
                          size_t workspace_bytes, hdla_sum* later, void* stream) {
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
    return wgrad_launch(a, dims->D, S, 2, static_cast<bf16*>(dwf), static_cast<bf16*>(dwg), later, static_cast<hipStream_t>(stream));
}
extern "C" int hdla_layer_up_wgrad(const hdla_up_dims* dims, const void* y, const void* f, const void* dlog_f, const void* dgate, void* dwf,
                                   void* dwg, void* workspace, size_t workspace_bytes, void* stream) {
    return layer_up_wgrad(dims, y, f, dlog_f, dgate, dwf, dwg, workspace, workspace_bytes, nullptr, stream);
}
extern "C" int hdla_layer_up_wgrad_later(const hdla_up_dims* dims, const void* y, const void* f, const void* dlog_f, const void* dgate, void* dwf,
                                         void* dwg, void* workspace, size_t workspace_bytes, hdla_sum* sums, void* stream) {
    if (!sums) return HDLA_ERR_NULL;
    return layer_up_wgrad(dims, y, f, dlog_f, dgate, dwf, dwg, workspace, workspace_bytes, sums, stream);
}

extern "C" int hdla_sum_partials(const float* part, int32_t count, int64_t n, void* out, void* stream) {
    if (count < 1 || n < 0 || n % 8) return HDLA_ERR_SHAPE;
    if (n == 0) return HDLA_OK;
    if (!part || !out) return HDLA_ERR_NULL;
    if (((reinterpret_cast<uintptr_t>(part) | reinterpret_cast<uintptr_t>(out)) & 15) != 0) return HDLA_ERR_ALIGN;
    if ((n / 8 + 255) / 256 > 0x7fffffffLL) return HDLA_ERR_SHAPE;
    SumJob job{};
    job.kind = SUM_PARTS; job.count = (int)count; job.n = (long long)n; job.part = part; job.out[0] = out;
    job.blocks = (int)((n / 8 + 255) / 256);
    return sum_now_or_later(job, nullptr, static_cast<hipStream_t>(stream));
}
