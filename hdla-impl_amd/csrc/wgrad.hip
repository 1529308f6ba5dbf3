// weight_grad: dW [N, K] = dY [M, N]^T X [M, K], bf16 in and out, fp32 sums: the weight gradients of the layer's projections, whose contraction runs over
// the rows of both operands (M tokens) and is far longer than the result is wide.
//
// A workgroup per 128 x 128 tile of dW (and share of the rows, where the tiles alone leave compute units without work).  Four waves bring 64 rows of
// both operands at a time straight to LDS, up to four stages ahead; eight waves, two on a SIMD, multiply: four of them a 64 x 64 quarter of the
// tile each over the stage's first 32 rows, the other four over its last, one set of sums added to the other at the end.  The contraction index is outermost in
// memory, so fragments come by the transposing LDS read, a stage ahead of their products.
//
// LDS: rows of 256 bytes; piece p (16 bytes) of row r lies at p ^ f(r), which the loading lanes see to by what they ask for.  A fragment's 16 columns
// are halves of four neighbouring pieces, so that a lane of the result has eight consecutive columns of dW (a 16-byte store) from two fragments; f puts the
// four rows of such a read into four different quarters of the banks.
//
// What bounds it: a workgroup makes 4.1 TFLOP/s on its compute unit, 88 % of what a large library product makes on one, where the operands come from
// the last-level cache; the rest is the compute units without a workgroup (208 tiles on 256).  us, one call behind the other, the BLAS product (the rows
// in parts, with a sum, where it had few tiles) -> this: 8192 rows, 3328 x 1024 89 -> 65 (856 TFLOP/s), 2048 x 2048 95 -> 74, 1792 x 512 43 -> 28, 1024 x 1024
// 35.0 -> 34.6; 4096 rows, 3328 x 1024 44 -> 34; 1500 rows 27 -> 16.  (Within a training step, operands from HBM: native.cpp, weight_grad.)  Four
// computing waves with 128 x 64 each, three quarters of the LDS reads but one wave a SIMD: 74 for the first.
#include "hdla_common.cuh"
#include "../../include/hdla_hip.h"

#include <algorithm>

namespace hdla {

struct WeightGradArgs {
    const bf16 *dy, *x;                   // rows ldy and ldx apart
    bf16* dw;                             // [N, K], or (several shares)
    float* part;                          // [shares][N, K]
    long long ldy, ldx;
    int M, N, K, per;                     // per: rows of a share, a multiple of a stage's
};

constexpr int WG_TILE = 128, WG_ROWS = 64, WG_SLOTS = 5, WG_LOADERS = 4, WG_COMPUTE = 8;
constexpr int WG_OPERAND = WG_ROWS * WG_TILE * 2, WG_STAGE = 2 * WG_OPERAND;
// loads of a loading wave per stage, and of all stages but the one that is waited for
constexpr int WG_LOADS = WG_STAGE / 1024 / WG_LOADERS;
static_assert(WG_SLOTS * WG_STAGE <= 160 * 1024 && (WG_SLOTS - 1) * WG_LOADS < 63, "what LDS holds; the memory counter's range");

__device__ __forceinline__ int wg_turn(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

__global__ __launch_bounds__(64 * (WG_LOADERS + WG_COMPUTE)) void weight_grad_kernel(WeightGradArgs p) {
    __shared__ __attribute__((aligned(16))) char smem[WG_SLOTS * WG_STAGE];
    const int l = lane_id(), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroups go round the eight XCDs: neighbouring tiles, which read the same rows of dY, on one of them
    const int tiles = gridDim.x, kts = p.K / WG_TILE;
    const int tile = tiles % 8 == 0 ? (int)(blockIdx.x % 8) * (tiles / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    const int n0 = tile / kts * WG_TILE, k0 = tile % kts * WG_TILE;
    const int m0 = (int)blockIdx.y * p.per, m1 = min(p.M, m0 + p.per);
    const int stages = (m1 - m0 + 2 * WG_ROWS - 1) / (2 * WG_ROWS) * 2, whole = (m1 - m0) / WG_ROWS;   // (an even number, which needs one loop only)

    if (wv >= WG_COMPUTE) {
        // ---- loading waves: wave w has requests w, w + 4, ... of each operand, four rows each.  The lanes of a row side by side
        const int w = wv - WG_COMPUTE, r0 = 4 * w + (l >> 4);     // (a request 16 rows further on is turned the same way)
        const int col = 8 * ((l & 15) ^ wg_turn(r0));
        const bf16 *const dy = p.dy + n0 + col, *const x = p.x + k0 + col;
        int slot = 0;
        auto load = [&](int t) __attribute__((always_inline)) {
            char* const to = smem + slot * WG_STAGE;
#pragma unroll
            for (int j = 0; j < WG_ROWS / 16; ++j) {
                const long long row = min(m0 + t * WG_ROWS + r0 + 16 * j, p.M - 1);   // rows past the end: cleared or never looked at
                const bf16* const from[2] = {dy + row * p.ldy, x + row * p.ldx};
#pragma unroll
                for (int o = 0; o < 2; ++o)
                    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from[o],
                                                     (__attribute__((address_space(3))) void*)(to + o * WG_OPERAND + (4 * j + w) * 1024), 16, 0, 0);
            }
            slot = slot + 1 == WG_SLOTS ? 0 : slot + 1;
        };
        // before stage t is handed over: its rows that are not this share's become zeros, each by the wave that asked for them
        auto clear = [&](int t) __attribute__((always_inline)) {
            char* const to = smem + t % WG_SLOTS * WG_STAGE;
#pragma unroll
            for (int j = 0; j < WG_ROWS / 16; ++j)
                if (m0 + t * WG_ROWS + r0 + 16 * j >= m1)
#pragma unroll
                    for (int o = 0; o < 2; ++o) *reinterpret_cast<i32x4*>(to + o * WG_OPERAND + (4 * j + w) * 1024 + 16 * l) = i32x4{0, 0, 0, 0};
        };
#pragma unroll
        for (int t = 0; t < WG_SLOTS; ++t) load(min(t, stages - 1));
        wait_loads<(WG_SLOTS - 1) * WG_LOADS>();
        if (whole == 0) clear(0);
        lds_barrier();
        for (int t = 0; t + 1 < stages; ++t) {
            wait_loads<(WG_SLOTS - 2) * WG_LOADS>();          // stage t + 1
            if (t + 1 >= whole) clear(t + 1);
            lds_barrier();
            load(min(t + WG_SLOTS, stages - 1));                  // where stage t was
        }
        wait_loads<0>();                                      // nothing may arrive where the sums go
        lds_barrier();
        return;
    }

    // ---- computing waves: rows 32 half .. of a stage, rows 64 (quarter & 1) .. and columns 64 (quarter >> 1) .. of the tile
    const int half = wv >> 2, nq = wv & 1, kq = (wv >> 1) & 1, g = l >> 4, s = l & 15, c = s;
    struct Frags { Frag<bf16> n[4][2], k[4][2]; };                // by 32-column block and half of its pieces: [2 block + h][rows 0..3, 4..7 of a lane group's]
    int at[2][2][2];                                              // operand, block, rows: this lane's piece
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int row = 32 * half + 8 * g + 4 * r + (s >> 2), piece = 4 * (2 * (o ? kq : nq) + b) + (s & 3);
                at[o][b][r] = o * WG_OPERAND + row * 256 + ((piece ^ wg_turn(row)) << 4);
            }
    auto read = [&](int slot, Frags& f) __attribute__((always_inline)) {
        const char* const from = smem + slot * WG_STAGE;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    f.n[2 * b + h][r] = ld_turned(from + at[0][b][r] + 8 * h);
                    f.k[2 * b + h][r] = ld_turned(from + at[1][b][r] + 8 * h);
                }
    };
    f32x4 acc[4][4];                                              // [n][k]: lane (g, c) row c, columns 4 g .. + 3 of the fragments
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = zero4();
    auto multiply = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = mm2(f.n[i][0], f.n[i][1], f.k[j][0], f.k[j][1], acc[i][j]);
    };
    Frags f[2];
    lds_barrier();
    read(0, f[0]);
    int slot = 0;
    auto stage = [&](const Frags& now, Frags& next) __attribute__((always_inline)) {
        slot = slot + 1 == WG_SLOTS ? 0 : slot + 1;
        lds_barrier();                                             // the next stage is there; this one has been read by all
        read(slot, next);
        __builtin_amdgcn_sched_barrier(0);
        multiply(now);
    };
#pragma unroll 1
    for (int t = 2; t < stages; t += 2) {
        stage(f[0], f[1]);
        stage(f[1], f[0]);
    }
    stage(f[0], f[1]);
    multiply(f[1]);
    lds_barrier();
    f32x4* const sums = reinterpret_cast<f32x4*>(smem) + (wv & 3) * 1024 + l;
    if (half) {
#pragma unroll
        for (int i = 0; i < 16; ++i) sums[i * 64] = acc[i / 4][i % 4];
    }
    lds_barrier();
    if (half) return;
    const long long first = (long long)(n0 + 64 * nq) * p.K + k0 + 64 * kq;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const f32x4 lo = acc[i][2 * b] + sums[(4 * i + 2 * b) * 64], hi = acc[i][2 * b + 1] + sums[(4 * i + 2 * b + 1) * 64];
            const long long to = first + (long long)(32 * (i >> 1) + 8 * (c >> 2) + 4 * (i & 1) + (c & 3)) * p.K + 32 * b + 8 * g;
            if (gridDim.y > 1) {
                float* const out = p.part + (long long)blockIdx.y * p.N * p.K + to;
                *reinterpret_cast<f32x4*>(out) = lo;
                *reinterpret_cast<f32x4*>(out + 4) = hi;
            } else {
                *reinterpret_cast<s16x8*>(p.dw + to) = __builtin_shufflevector(to_frag<bf16>(lo).v, to_frag<bf16>(hi).v, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        }
}

// Shares of the rows: as many as give each compute unit a workgroup, of at least eight stages.
static int weight_grad_shares(long long M, int N, int K, int& per) {
    const long long tiles = (long long)(N / WG_TILE) * (K / WG_TILE);
    const long long want = std::max(1LL, std::min(256 / tiles, M / (8 * WG_ROWS)));
    const long long pairs = (M + 2 * WG_ROWS - 1) / (2 * WG_ROWS);
    per = (int)((pairs + want - 1) / want) * 2 * WG_ROWS;
    return (int)((M + per - 1) / per);
}

}  // namespace hdla

using namespace hdla;

static bool weight_grad_shape(int64_t M, int32_t N, int32_t K) {
    return M >= 1 && M <= 0x7fff0000LL && N >= WG_TILE && K >= WG_TILE && N % WG_TILE == 0 && K % WG_TILE == 0 &&
           (int64_t)(N / WG_TILE) * (K / WG_TILE) <= 0x7fffffffLL;
}
extern "C" size_t hdla_weight_grad_workspace_bytes(int64_t M, int32_t N, int32_t K) {
    if (!weight_grad_shape(M, N, K)) return 0;
    int per;
    const int shares = weight_grad_shares(M, N, K, per);
    return shares > 1 ? (size_t)shares * N * K * sizeof(float) : 0;
}
extern "C" int hdla_weight_grad(int64_t M, int32_t N, int32_t K, const void* dY, int64_t ldy, const void* X, int64_t ldx, void* dW, void* workspace,
                                size_t workspace_bytes, void* stream) {
    if (!weight_grad_shape(M, N, K) || ldy < N || ldx < K || ldy % 8 || ldx % 8) return HDLA_ERR_SHAPE;
    if (!dY || !X || !dW) return HDLA_ERR_NULL;
    auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    if (!al16(dY) || !al16(X) || !al16(dW)) return HDLA_ERR_ALIGN;
    const size_t need = hdla_weight_grad_workspace_bytes(M, N, K);
    if (need && (!workspace || !al16(workspace) || workspace_bytes < need)) return HDLA_ERR_WORKSPACE;
    WeightGradArgs a{};
    a.dy = static_cast<const bf16*>(dY); a.x = static_cast<const bf16*>(X); a.dw = static_cast<bf16*>(dW); a.part = static_cast<float*>(workspace);
    a.ldy = ldy; a.ldx = ldx; a.M = (int)M; a.N = N; a.K = K;
    const int shares = weight_grad_shares(M, N, K, a.per);
    hipLaunchKernelGGL(weight_grad_kernel, dim3((unsigned)((N / WG_TILE) * (K / WG_TILE)), (unsigned)shares), dim3(64 * (WG_LOADERS + WG_COMPUTE)), 0,
                       static_cast<hipStream_t>(stream), a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    return shares > 1 ? hdla_sum_partials(a.part, shares, (int64_t)N * K, dW, stream) : HDLA_OK;
}
