// weight_grad: dW [N, K] = dY [M, N]^T X [M, K], bf16 in and out, fp32 sums: the weight gradients of the layer's projections, whose contraction runs over
// the rows of both operands (M tokens) and is far longer than the result is wide.
//
// One product or two of the same rows.  A workgroup per 128 x 128 tile of dW (and share of the rows, where the tiles alone leave compute units without
// work).  Of two products with more tiles than there are compute units each workgroup has a share of one of the tiles that are too many, and then a tile of
// its own: the loading waves begin it while the share's sums leave.  Four waves bring 64 rows of
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
// A pair, in a training step of the layer: 208 and 64 tiles over 8192 rows, the second in four shares in a launch of its own 82 + 30 us -> 94 together (256 whole
// tiles, 16 in 16 shares) and 5 for their sums; the step 714 -> 693, with 4096 rows 442 -> 417; 56 and 16 tiles, 8192 rows 408 -> 395.
#include "sums.cuh"

#include <algorithm>

namespace hdla {

struct WeightGradProduct {
    const bf16 *dy, *x;                   // rows ldy and ldx apart
    bf16* dw;                             // [N, K]
    long long ldy, ldx;
    int K;
};
struct WeightGradArgs {
    WeightGradProduct of[2];
    float* part;                          // [shares][rest][128, 128], where there are several shares
    int first;                            // tiles of of[0]; numbers from there on are of[1]'s
    int whole, rest, shares, per;         // tiles by whole workgroups (0, or as many as there are workgroups), tiles behind them in shares; rows of a share
    int M;
};

constexpr int WG_TILE = SUM_TILE, WG_ROWS = 64, WG_SLOTS = 5, WG_LOADERS = 4, WG_COMPUTE = 8;
constexpr int WG_OPERAND = WG_ROWS * WG_TILE * 2, WG_STAGE = 2 * WG_OPERAND;
// loads of a loading wave per stage, and of all stages but the one that is waited for
constexpr int WG_LOADS = WG_STAGE / 1024 / WG_LOADERS;
static_assert(WG_SLOTS * WG_STAGE <= 160 * 1024 && (WG_SLOTS - 1) * WG_LOADS < 63, "what LDS holds; the memory counter's range");

// what a workgroup does: a tile, the rows of a share of it, and where that share's sums go (null: it is all of them)
struct WgItem {
    WeightGradProduct of;
    int n0, k0, m0, m1;
    float* part;
};
// (neighbouring tiles, which read the same rows of dY, on one XCD: workgroups go round the eight of them)
__device__ __forceinline__ int wg_swizzle(int tile, int tiles) { return tiles % 8 == 0 ? tile % 8 * (tiles / 8) + tile / 8 : tile; }
__device__ __forceinline__ WgItem wg_item(const WeightGradArgs& p, int which) {
    WgItem w;
    int tile = wg_swizzle((int)blockIdx.x, p.whole);
    w.m0 = 0;
    w.m1 = p.M;
    w.part = nullptr;
    if (which == 0) {
        const int r = wg_swizzle((int)blockIdx.x % p.rest, p.rest), share = (int)blockIdx.x / p.rest;
        tile = p.whole + r;
        w.m0 = share * p.per;
        w.m1 = min(p.M, w.m0 + p.per);
        if (p.shares > 1) w.part = p.part + ((long long)share * p.rest + r) * (WG_TILE * WG_TILE);
    }
    const bool second = tile >= p.first;
    w.of = p.of[second ? 1 : 0];
    if (second) tile -= p.first;
    const int kts = w.of.K / WG_TILE;
    w.n0 = tile / kts * WG_TILE;
    w.k0 = tile % kts * WG_TILE;
    return w;
}

__device__ __forceinline__ int wg_turn(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

__global__ __launch_bounds__(64 * (WG_LOADERS + WG_COMPUTE)) void weight_grad_kernel(WeightGradArgs p) {
    __shared__ __attribute__((aligned(16))) char smem[WG_SLOTS * WG_STAGE];
    const int l = lane_id(), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // items 0 (a share) and 1 (a tile), as far as the workgroup has them.  The second one's stages begin behind the slots that the first one's sums go through
    const int item0 = (int)blockIdx.x < p.rest * p.shares ? 0 : 1, items = p.whole ? 2 : 1;
    constexpr int SUM_SLOTS = 2;
    static_assert(SUM_SLOTS * WG_STAGE >= 4 * 16 * 1024 && SUM_SLOTS < WG_SLOTS, "four waves' sums");

    if (wv >= WG_COMPUTE) {
        // ---- loading waves: wave w4 has requests w4, w4 + 4, ... of each operand, four rows each.  The lanes of a row side by side
        const int w4 = wv - WG_COMPUTE, r0 = 4 * w4 + (l >> 4);     // (a request 16 rows further on is turned the same way)
        const int col = 8 * ((l & 15) ^ wg_turn(r0));
        int asked = 0;                                        // stages of the next item that are on their way
#pragma unroll 1
        for (int it = item0; it < items; ++it) {
            const WgItem of = wg_item(p, it);
            const int stages = (of.m1 - of.m0 + 2 * WG_ROWS - 1) / (2 * WG_ROWS) * 2, whole = (of.m1 - of.m0) / WG_ROWS;   // (an even number, which needs one loop only)
            const int base = it == item0 ? 0 : SUM_SLOTS;
            auto load = [&](const WgItem& w, int t, int slot) __attribute__((always_inline)) {
                char* const to = smem + slot * WG_STAGE;
#pragma unroll
                for (int j = 0; j < WG_ROWS / 16; ++j) {
                    const long long row = min(w.m0 + t * WG_ROWS + r0 + 16 * j, p.M - 1);   // rows past the end: cleared or never looked at
                    const bf16* const from[2] = {w.of.dy + w.n0 + col + row * w.of.ldy, w.of.x + w.k0 + col + row * w.of.ldx};
#pragma unroll
                    for (int o = 0; o < 2; ++o)
                        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from[o],
                                                         (__attribute__((address_space(3))) void*)(to + o * WG_OPERAND + (4 * j + w4) * 1024), 16, 0, 0);
                }
            };
            // before stage t is handed over: its rows that are not this share's become zeros, each by the wave that asked for them
            auto clear = [&](int t) __attribute__((always_inline)) {
                char* const to = smem + (base + t) % WG_SLOTS * WG_STAGE;
#pragma unroll
                for (int j = 0; j < WG_ROWS / 16; ++j)
                    if (of.m0 + t * WG_ROWS + r0 + 16 * j >= of.m1)
#pragma unroll
                        for (int o = 0; o < 2; ++o) *reinterpret_cast<i32x4*>(to + o * WG_OPERAND + (4 * j + w4) * 1024 + 16 * l) = i32x4{0, 0, 0, 0};
            };
#pragma unroll 1
            for (int t = asked; t < WG_SLOTS; ++t) load(of, min(t, stages - 1), (base + t) % WG_SLOTS);
            int slot = base;
            wait_loads<(WG_SLOTS - 1) * WG_LOADS>();
            if (whole == 0) clear(0);
            lds_barrier();
            for (int t = 0; t + 1 < stages; ++t) {
                wait_loads<(WG_SLOTS - 2) * WG_LOADS>();          // stage t + 1
                if (t + 1 >= whole) clear(t + 1);
                lds_barrier();
                load(of, min(t + WG_SLOTS, stages - 1), slot);    // where stage t was
                slot = slot + 1 == WG_SLOTS ? 0 : slot + 1;
            }
            wait_loads<0>();                                      // nothing may arrive where the sums go
            lds_barrier();
            if (it + 1 == items) break;
            const WgItem next = wg_item(p, it + 1);
            const int last = (next.m1 - next.m0 + 2 * WG_ROWS - 1) / (2 * WG_ROWS) * 2 - 1;
#pragma unroll 1
            for (asked = 0; asked < WG_SLOTS - SUM_SLOTS; ++asked) load(next, min(asked, last), SUM_SLOTS + asked);
            lds_barrier();                                        // the sums are there
            lds_barrier();                                        // and have been read
        }
        return;
    }

    // ---- computing waves: rows 32 half .. of a stage, rows 64 (quarter & 1) .. and columns 64 (quarter >> 1) .. of the tile
    const int half = wv >> 2, nq = wv & 1, kq = (wv >> 1) & 1, g = l >> 4, s = l & 15;
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
#pragma unroll 1
    for (int it = item0; it < items; ++it) {
        const WgItem of = wg_item(p, it);
        const int stages = (of.m1 - of.m0 + 2 * WG_ROWS - 1) / (2 * WG_ROWS) * 2;
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
        int slot = it == item0 ? 0 : SUM_SLOTS;
        lds_barrier();
        read(slot, f[0]);
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
        int e = l;
        asm volatile("" : "+v"(e));                                // (what follows is formed here: kept over the products it would be spilled)
        const int ge = e >> 4, c = e & 15;
        f32x4* const sums = reinterpret_cast<f32x4*>(smem) + (wv & 3) * 1024 + e;
        if (half) {
#pragma unroll
            for (int i = 0; i < 16; ++i) sums[i * 64] = acc[i / 4][i % 4];
        }
        lds_barrier();
        if (!half) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const f32x4 lo = acc[i][2 * b] + sums[(4 * i + 2 * b) * 64], hi = acc[i][2 * b + 1] + sums[(4 * i + 2 * b + 1) * 64];
                    const int row = 64 * nq + 32 * (i >> 1) + 8 * (c >> 2) + 4 * (i & 1) + (c & 3), column = 64 * kq + 32 * b + 8 * ge;
                    if (of.part) {
                        float* const out = of.part + row * WG_TILE + column;
                        *reinterpret_cast<f32x4*>(out) = lo;
                        *reinterpret_cast<f32x4*>(out + 4) = hi;
                    } else {
                        *reinterpret_cast<s16x8*>(of.of.dw + (long long)(of.n0 + row) * of.of.K + of.k0 + column) =
                            __builtin_shufflevector(to_frag<bf16>(lo).v, to_frag<bf16>(hi).v, 0, 1, 2, 3, 4, 5, 6, 7);
                    }
                }
        }
        if (it + 1 < items) lds_barrier();                            // (the loading waves go on where the sums were)
    }
}

// Tiles and shares of the rows.  Shares: as many as give each compute unit a workgroup, of at least eight stages.  One product has them of all its tiles
// (none, where they fill the device).
constexpr int WG_UNITS = 256;                                     // compute units, a workgroup each
static void weight_grad_plan(long long M, const int* N, const int* K, int count, WeightGradArgs& a) {
    long long tiles = 0;
    for (int i = 0; i < count; ++i) {
        tiles += (long long)(N[i] / WG_TILE) * (K[i] / WG_TILE);
        if (i == 0) a.first = (int)tiles;
    }
    a.whole = count > 1 && tiles > WG_UNITS ? WG_UNITS : 0;
    a.rest = (int)tiles - a.whole;
    const long long want = std::max(1LL, std::min<long long>(WG_UNITS / a.rest, M / (8 * WG_ROWS)));
    const long long pairs = (M + 2 * WG_ROWS - 1) / (2 * WG_ROWS);
    a.per = (int)((pairs + want - 1) / want) * 2 * WG_ROWS;
    a.shares = (int)((M + a.per - 1) / a.per);
    a.M = (int)M;
}
static size_t weight_grad_room(const WeightGradArgs& a) { return a.shares > 1 ? (size_t)a.shares * a.rest * WG_TILE * WG_TILE * sizeof(float) : 0; }

}  // namespace hdla

using namespace hdla;

static bool weight_grad_shape(int64_t M, int32_t N, int32_t K) {
    return M >= 1 && M <= 0x7fff0000LL && N >= WG_TILE && K >= WG_TILE && N % WG_TILE == 0 && K % WG_TILE == 0 &&
           (int64_t)(N / WG_TILE) * (K / WG_TILE) <= 0x7fffffffLL;
}
static bool weight_grad_pair(int64_t M, const int32_t* N, const int32_t* K) {
    if (!N || !K) return false;
    for (int i = 0; i < 2; ++i)
        if (!weight_grad_shape(M, N[i], K[i]) || (int64_t)(N[i] / WG_TILE) * (K[i] / WG_TILE) > WG_UNITS) return false;
    return true;
}
static int weight_grad_run(int64_t M, int count, const int32_t* N, const int32_t* K, const void* const* dY, const int64_t* ldy, const void* const* X,
                           const int64_t* ldx, void* const* dW, void* workspace, size_t workspace_bytes, hdla_sum* later, void* stream) {
    WeightGradArgs a{};
    auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    for (int i = 0; i < count; ++i) if (ldy[i] < N[i] || ldx[i] < K[i] || ldy[i] % 8 || ldx[i] % 8) return HDLA_ERR_SHAPE;
    for (int i = 0; i < count; ++i) if (!dY[i] || !X[i] || !dW[i]) return HDLA_ERR_NULL;
    for (int i = 0; i < count; ++i) {
        if (!al16(dY[i]) || !al16(X[i]) || !al16(dW[i])) return HDLA_ERR_ALIGN;
        a.of[i] = WeightGradProduct{static_cast<const bf16*>(dY[i]), static_cast<const bf16*>(X[i]), static_cast<bf16*>(dW[i]), ldy[i], ldx[i], K[i]};
    }
    weight_grad_plan(M, N, K, count, a);
    const size_t need = weight_grad_room(a);
    if (need && (!workspace || !al16(workspace) || workspace_bytes < need)) return HDLA_ERR_WORKSPACE;
    a.part = static_cast<float*>(workspace);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(weight_grad_kernel, dim3((unsigned)(a.whole ? a.whole : a.rest * a.shares)), dim3(64 * (WG_LOADERS + WG_COMPUTE)), 0, s, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    SumJob job{};
    if (a.shares > 1) {
        job.kind = SUM_TILES; job.blocks = 8 * a.rest; job.count = a.shares;
        job.first = a.first; job.whole = a.whole; job.rest = a.rest;
        for (int i = 0; i < count; ++i) { job.K[i] = K[i]; job.out[i] = dW[i]; }
        job.part = a.part;
    }
    return sum_now_or_later(job, later, s);
}

extern "C" size_t hdla_weight_grad_workspace_bytes(int64_t M, int32_t N, int32_t K) {
    if (!weight_grad_shape(M, N, K)) return 0;
    WeightGradArgs a{};
    weight_grad_plan(M, &N, &K, 1, a);
    return weight_grad_room(a);
}
extern "C" int hdla_weight_grad(int64_t M, int32_t N, int32_t K, const void* dY, int64_t ldy, const void* X, int64_t ldx, void* dW, void* workspace,
                                size_t workspace_bytes, void* stream) {
    if (!weight_grad_shape(M, N, K)) return HDLA_ERR_SHAPE;
    return weight_grad_run(M, 1, &N, &K, &dY, &ldy, &X, &ldx, &dW, workspace, workspace_bytes, nullptr, stream);
}
extern "C" size_t hdla_weight_grad_pair_workspace_bytes(int64_t M, const int32_t* N, const int32_t* K) {
    if (!weight_grad_pair(M, N, K)) return 0;
    WeightGradArgs a{};
    weight_grad_plan(M, N, K, 2, a);
    return weight_grad_room(a);
}
extern "C" int hdla_weight_grad_pair(int64_t M, const int32_t* N, const int32_t* K, const void* const* dY, const int64_t* ldy, const void* const* X,
                                     const int64_t* ldx, void* const* dW, void* workspace, size_t workspace_bytes, hdla_sum* sum, void* stream) {
    if (!dY || !ldy || !X || !ldx || !dW) return HDLA_ERR_NULL;
    if (!weight_grad_pair(M, N, K)) return HDLA_ERR_SHAPE;
    return weight_grad_run(M, 2, N, K, dY, ldy, X, ldx, dW, workspace, workspace_bytes, sum, stream);
}
