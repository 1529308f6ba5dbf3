// 16-bit tiles that come from memory row by row and are taken by the matrix units as fragments: a wave's own piece of LDS between the two.
//
// A fragment's lane order (16 rows, 16 bytes of each) puts the four lanes that the address unit takes at a time into four cache lines, at
// a quarter of the rate.  So a request has the lanes of a row side by side, and the lanes change here.
#pragma once
#include "hdla_common.cuh"

namespace hdla {

// a wave's LDS writes before its reads of what its other lanes wrote, and the other way round: the hardware keeps the order
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// d sigmoid(-f), rounded to bf16 as the stored gradient of logsigmoid(f) would be
__device__ __forceinline__ s16x8 times_sigmoid_neg(s16x8 d, s16x8 f) {
    Frag<bf16> x[2], y[2];
    x[0].v = __builtin_shufflevector(d, d, 0, 1, 2, 3);
    x[1].v = __builtin_shufflevector(d, d, 4, 5, 6, 7);
    y[0].v = __builtin_shufflevector(f, f, 0, 1, 2, 3);
    y[1].v = __builtin_shufflevector(f, f, 4, 5, 6, 7);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        f32x4 v = to_f32(x[h]);
        const f32x4 z = to_f32(y[h]);
        float e[4], s[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = __expf(z[i]);
        sigmoid_of_exp<4>(e, s);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] *= s[i];
        x[h] = to_frag<bf16>(v);
    }
    return __builtin_shufflevector(x[0].v, x[1].v, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Rows of W (32, 64 or 128) elements.  Piece p (16 bytes) of row r lies at place p ^ f(r), f the bits of the row above those that the banks
// tell apart, turned by one: 16 lanes meet each bank once when they write or read rows side by side, when they read one piece of 16 rows
// (rows), and when they read 16 columns of four rows with the transposing read (columns).
template <int W> struct RowTile {
    static constexpr int P = W / 8, RPR = 64 / P, ROW = 2 * W;   // pieces a row, rows a request, bytes a row
    static_assert(W == 32 || W == 64 || W == 128, "a row fills a quarter of the banks, half of them or all");
    static __device__ __forceinline__ int place(int r, int p) {
        const int f = W == 32 ? (r >> 2) & 3 : W == 64 ? ((r & 6) | ((r >> 3) & 1)) : (((r << 1) & 14) | ((r >> 3) & 1));
        return r * ROW + ((p ^ f) << 4);
    }
    // request j of a tile: this lane's row and first element
    static __device__ __forceinline__ int row(int j, int l) { return j * RPR + l / P; }
    static __device__ __forceinline__ int col(int l) { return l % P * 8; }
    static __device__ __forceinline__ void put(char* tile, int j, int l, s16x8 x) { *reinterpret_cast<s16x8*>(tile + place(row(j, l), l % P)) = x; }
    static __device__ __forceinline__ s16x8 get(const char* tile, int j, int l) { return *reinterpret_cast<const s16x8*>(tile + place(row(j, l), l % P)); }
    // row r (the lane's) of columns 32 k .. + 31: lane (g, c) elements 8 g .. 8 g + 7, as two fragments
    static __device__ __forceinline__ void rows(const char* tile, int r, int k, int l, Frag<bf16>& a, Frag<bf16>& b) {
        const s16x8 x = *reinterpret_cast<const s16x8*>(tile + place(r, 4 * k + (l >> 4)));
        a.v = __builtin_shufflevector(x, x, 0, 1, 2, 3);
        b.v = __builtin_shufflevector(x, x, 4, 5, 6, 7);
    }
    // columns 16 b .. + 15 as rows of a fragment whose inner index is the rows r0 + step g .. + 3 for lane group g: lane (g, c) has column c
    static __device__ __forceinline__ Frag<bf16> columns(const char* tile, int r0, int step, int b, int l) {
        const int s = l & 15, r = r0 + step * (l >> 4) + (s >> 2);
        Frag<bf16> f;
        f.v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(tile + place(r, 2 * b + ((s & 2) >> 1)) + 8 * (s & 1)));
        return f;
    }
};

}  // namespace hdla
