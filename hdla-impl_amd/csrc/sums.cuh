// Sums over partial results that several kernels of the layer's backward pass leave: each as a launch of its own behind its kernel, or as a job of
// one launch for all of them (sums.hip).
#pragma once
#include "hdla_common.cuh"
#include "../../include/hdla_hip.h"

namespace hdla {

enum SumKind { SUM_NONE, SUM_PARTS, SUM_ROWS, SUM_TILES };
struct SumJob {
    int kind, blocks;             // workgroups of 256 threads
    int count;                    // PARTS: partial results; TILES: shares
    int G, E;                     // ROWS
    int f32;                      // ROWS: out in 32 bits
    int first, whole, rest;       // TILES: as in WeightGradArgs (wgrad.hip)
    int K[2];                     // TILES
    long long n;                  // PARTS: elements, a multiple of 8; ROWS: rows
    const float* part;
    void* out[2];                 // (the second: TILES)
};
static_assert(sizeof(SumJob) <= sizeof(hdla_sum), "what callers keep it in");

__device__ __forceinline__ void st_sum(bf16* to, f32x4 lo, f32x4 hi) {
    *reinterpret_cast<s16x8*>(to) = __builtin_shufflevector(to_frag<bf16>(lo).v, to_frag<bf16>(hi).v, 0, 1, 2, 3, 4, 5, 6, 7);
}
// `count` partial results `apart` elements apart, in their order: eight elements a thread
__device__ __forceinline__ void sum_eight(const float* from, int count, long long apart, bf16* to) {
    f32x4 lo = zero4(), hi = zero4();
#pragma unroll 8
    for (int s = 0; s < count; ++s, from += apart) {
        lo += *reinterpret_cast<const f32x4*>(from);
        hi += *reinterpret_cast<const f32x4*>(from + 4);
    }
    st_sum(to, lo, hi);
}
__device__ __forceinline__ void sum_parts(const SumJob& j, int block) {
    const long long i = ((long long)block * 256 + threadIdx.x) * 8;
    if (i < j.n) sum_eight(j.part + i, j.count, j.n, static_cast<bf16*>(j.out[0]) + i);
}
// The weight gradient of the norm, [G E]: the rows of `part` [n][E], row r of group r % G.  A workgroup owns 16 columns: four threads of four
// columns each, 64 row phases, summed through LDS in a fixed order.
__device__ __forceinline__ void sum_rows_of_groups(const float* part, void* out, bool f32, long long n, int G, int E, int block) {
    __shared__ f32x4 red[64][4];
    const int cq = threadIdx.x & 3, rl = threadIdx.x >> 2;
    const long long col = (long long)block * 16 + cq * 4;
    const long long D = (long long)G * E;
    f32x4 acc = zero4();
    if (col < D) {
        const int g = (int)(col / E), e = (int)(col % E);
#pragma unroll 8
        for (long long idx = g + (long long)rl * G; idx < n; idx += 64LL * G) acc += *reinterpret_cast<const f32x4*>(part + idx * E + e);
    }
    red[rl][cq] = acc;
    __syncthreads();
    if (rl == 0 && col < D) {
        f32x4 s = red[0][cq];
#pragma unroll
        for (int r = 1; r < 64; ++r) s += red[r][cq];
        if (f32) *reinterpret_cast<f32x4*>(static_cast<float*>(out) + col) = s;
        else st_frag(static_cast<bf16*>(out) + col, to_frag<bf16>(s));
    }
}
// Tiles of weight gradients that were worked on in shares of the rows, [shares][rest][128, 128]: eight workgroups a tile
constexpr int SUM_TILE = 128;
__device__ __forceinline__ void sum_tiles(const SumJob& j, int block) {
    const int r = block / 8, e = (block % 8 * 256 + (int)threadIdx.x) * 8;
    int tile = j.whole + r;
    const bool second = tile >= j.first;
    if (second) tile -= j.first;
    const int K = second ? j.K[1] : j.K[0], kts = K / SUM_TILE;
    bf16* const to = static_cast<bf16*>(second ? j.out[1] : j.out[0]) + (long long)(tile / kts * SUM_TILE + e / SUM_TILE) * K + tile % kts * SUM_TILE + e % SUM_TILE;
    sum_eight(j.part + (long long)r * (SUM_TILE * SUM_TILE) + e, j.count, (long long)j.rest * (SUM_TILE * SUM_TILE), to);
}

// runs a job by itself, or (later != nullptr) leaves it there
int sum_now_or_later(const SumJob& job, hdla_sum* later, hipStream_t stream);

}  // namespace hdla
