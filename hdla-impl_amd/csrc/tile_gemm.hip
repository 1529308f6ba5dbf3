// y [M, N] = x [M, K] W with W [N, K]^T, or (TURNED) W [K, N] as it is: the layer's large projections and their input gradients for some hundred rows, where
// a BLAS call is 15 to 20 us of host time, most of what the step in it takes.  bf16 in and out, fp32 sums.
//
// A workgroup per tile of 16 MT rows x 32 NP columns.  Its four waves take a quarter of K each, 64 at a time straight to LDS of their own (global_load_lds,
// SLOTS blocks ahead, whole cache lines of each row), and add up through LDS at the end: no barrier in between, and a wave uses each fragment 2 NP or MT times.  W's rows
// are taken in the order that leaves a lane eight consecutive columns of y.  TURNED: W's contraction index is outermost; the transposing LDS read takes its tiles.
//
// What bounds it: what a compute unit takes in.  128 KiB are on their way into it at a time, and a workgroup of 64 x 64 reads 256 bytes for each column of K (with
// eight waves, 32 columns of K and half lines at a time, 7.0 took 10.6).  So tiles are as small as give every workgroup a compute unit of its own, and where those of 64 x 64
// are more than there are compute units the BLAS kernels' larger tiles win.  us on the device, operands from HBM, BLAS / 32 x 32 / 64 x 32 / 64 x 64 (* the choice):
// 100 x 3216 x 1024 9.0 / 9.3 / 6.2* / 7.0, 100 x 1024 x 1024 7.8 / 4.6* / 5.4 / 6.4, 256 x 3216 x 1024 9.5 / 17.0 / 11.2 / 8.8*, 484 x 904 x 256 5.3 / 6.3 / 4.6* / 5.0,
// 512 x 1024 x 3216 17.1 / 19.8 / 14.8* / 17.2, 256 x 4096 x 4096 21.7 / 37 / 27 / 18.9*, 1024 x 1024 x 1024 9.2 / 14.3 / 9.9 / 7.6*; turned 484 x 256 x 904 9.6 / 6.3* / 7.4 / 8.1,
// 512 x 1024 x 3216 19.0 / 23.9 / 16.2* / 18.8, 1024 x 1024 x 3328 19.2 / 44 / 28 / 18.9*.  Beyond the line 256 x 6416 x 2048 23.8 / 41 / 29 / 24.5, 512 x 3216 x 1024 11.6 / 28 / 20 / 15.6.
// Over all products of the layer at 128 to 4096 channels and 65 to 8000 rows within the line (432 of them, one shape behind the other) the time is 0.77 of the BLAS library's, geometric mean.  By themselves some
// are slower: turned, many rows over long sums (1500 x 512 x 1792 13.1 / 14.0, 2000 x 512 x 1792 13.3 / 15.5, 4000 x 256 x 1024 10.4 / 11.0) and weights of 32 MB and more (160 x 3072 x 9496 49.1 / 53.0,
// 256 x 4096 x 4096 24.9 / 26.5); 65 to 80 x 4880 x 1536 8.8 / 9.7.  Within a step, where their operands come from the launch before, they are not: as a graph's replay, which has no host to
// gain by, training steps with these two kinds by BLAS / by this took 1 x 1500 tokens of 512 channels 197.5 / 197.1, 4 x 500 186.1 / 186.4, 4 x 1000 of 256 197.3 / 196.7, 1 x 200 of
// 4096 423.0 / 421.9, 1 x 256 438.3 / 439.4.  So one line serves both, and calls and replays have the same bits.
#include "row_tile.cuh"
#include "host_path.h"

namespace hdla {

constexpr int TG_WAVES = 4, TG_K = 64, TG_UNITS = 256;                 // TG_UNITS: compute units
template <int MT, int NP> struct TileCfg {
    static constexpr int A = 2 * MT, B = 4 * NP, REQ = A + B;          // requests of 1 KiB a block: of x, of W
    static constexpr int SLOT = REQ * 1024, MOST = 160 * 1024 / (TG_WAVES * SLOT), SLOTS = MOST < 4 ? MOST : 4;
    static constexpr int SUMS = MT * 2 * NP * 1024;                    // bytes a wave
    static constexpr int BYTES = TG_WAVES * (SLOT * SLOTS > SUMS ? SLOT * SLOTS : SUMS);
    static_assert(SLOTS >= 2 && (SLOTS - 1) * REQ < 63, "LDS; the memory counter's range");
};

template <int MT, int NP, bool TURNED>
__global__ __launch_bounds__(64 * TG_WAVES) void tile_gemm_kernel(const bf16* __restrict__ x, long long ldx, const bf16* __restrict__ w, long long ldw,
                                                                  bf16* __restrict__ y, long long ldy, int M, int N, int K) {
    typedef TileCfg<MT, NP> C;
    typedef RowTile<TG_K> TR;                                         // rows of x and of W
    typedef RowTile<32 * NP> TW;                                      // TURNED: rows of K of W
    __shared__ __attribute__((aligned(16))) char sm[C::BYTES];
    const int l = lane_id(), g = l >> 4, c = l & 15;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * (32 * NP), m0 = blockIdx.y * (16 * MT);
    const int nb = (K + TG_K - 1) / TG_K, per = (nb + TG_WAVES - 1) / TG_WAVES, b0 = wv * per, blocks = min(nb - b0, per);
    char* const mine = sm + wv * (C::SLOT * C::SLOTS);

    // What a lane asks for: its 16 bytes arrive at 16 l of the request's KiB, where RowTile has the piece that is asked for.  Rows past the end: the last one
    // again, not stored
    auto spot = [&](auto tile, int i) __attribute__((always_inline)) {
        typedef decltype(tile) R;
        return l % R::P ^ ((R::place(R::row(i, l), 0) - R::row(i, l) * R::ROW) >> 4);
    };
    const bf16* from[C::REQ];
    int at_k[C::A + (TURNED ? 0 : C::B)];
#pragma unroll
    for (int i = 0; i < C::A; ++i) {
        at_k[i] = 8 * spot(TR(), i);
        from[i] = x + (long long)min(m0 + TR::row(i, l), M - 1) * ldx;
    }
#pragma unroll
    for (int i = 0; i < C::B; ++i) {
        if constexpr (TURNED) {
            from[C::A + i] = w + n0 + 8 * spot(TW(), i);
        } else {
            const int r = TR::row(i, l), n = r >> 4, j = r & 15;      // rows of fragment n, in its order
            at_k[C::A + i] = 8 * spot(TR(), i);
            from[C::A + i] = w + (long long)min(n0 + 32 * (n >> 1) + 8 * (j >> 2) + (j & 3) + 4 * (n & 1), N - 1) * ldw;
        }
    }
    auto load = [&](int b, int slot) __attribute__((always_inline)) {
        // (a block past the wave's last, and past K the row's last piece: asked for again, never looked at)
        const int k0 = TG_K * (b0 + min(b, blocks - 1));
        char* const to = mine + slot * C::SLOT;
#pragma unroll
        for (int i = 0; i < C::REQ; ++i) {
            const bf16* src;
            if constexpr (TURNED) src = i < C::A ? from[i] + min(k0 + at_k[i < C::A ? i : 0], K - 8) : from[i] + (long long)min(k0 + TW::row(i - C::A, l), K - 1) * ldw;
            else src = from[i] + min(k0 + at_k[i], K - 8);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)(to + i * 1024), 16, 0, 0);
        }
    };
    f32x4 acc[MT][2 * NP];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < 2 * NP; ++n) acc[m][n] = zero4();
    if (blocks > 0) {
#pragma unroll
        for (int s = 0; s < C::SLOTS; ++s) load(s, s);
        int slot = 0;
#pragma unroll 1
        for (int b = 0; b < blocks; ++b) {
            wait_loads<(C::SLOTS - 1) * C::REQ>();
            const char* const at = mine + slot * C::SLOT;
            const char* const tw = at + C::A * 1024;
            Frag<bf16> xa[2][MT], xb[2][MT], wa[2][2 * NP], wb[2][2 * NP];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
#pragma unroll
                for (int m = 0; m < MT; ++m) TR::rows(at, 16 * m + c, k, l, xa[k][m], xb[k][m]);
#pragma unroll
                for (int n = 0; n < 2 * NP; ++n) {
                    if constexpr (!TURNED) {
                        TR::rows(tw, 16 * n + c, k, l, wa[k][n], wb[k][n]);
                    } else {
                        // rows 8 g + 0 .. 3 and + 4 .. 7; columns 32 (n / 2) + 8 q + 4 (n % 2) + 0 .. 3 for the four lanes q (as W's rows above)
                        const int r = 32 * k + 8 * g + (c >> 2), p = 4 * (n >> 1) + (c & 3);
                        wa[k][n] = ld_turned(tw + TW::place(r, p) + 8 * (n & 1));
                        wb[k][n] = ld_turned(tw + TW::place(r + 4, p) + 8 * (n & 1));
                    }
                }
                if (TG_K * (b0 + b) + 32 * k + 32 > K && TG_K * (b0 + b) + 32 * k + 8 * g >= K) {
                    // columns of no row, in both operands
#pragma unroll
                    for (int m = 0; m < MT; ++m) { xa[k][m] = zero_frag<bf16>(); xb[k][m] = zero_frag<bf16>(); }
#pragma unroll
                    for (int n = 0; n < 2 * NP; ++n) { wa[k][n] = zero_frag<bf16>(); wb[k][n] = zero_frag<bf16>(); }
                }
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xc07f);                       // the fragments are there (no LDS access is on its way)
            asm volatile("" ::: "memory");
            load(b + C::SLOTS, slot);
            slot = slot + 1 == C::SLOTS ? 0 : slot + 1;
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < 2 * NP; ++n)
#pragma unroll
                    for (int k = 0; k < 2; ++k) acc[m][n] = mm2(xa[k][m], xb[k][m], wa[k][n], wb[k][n], acc[m][n]);
        }
        wait_loads<0>();                                              // nothing may arrive where the sums go
    }
    __syncthreads();
    // lane (g, c) of tile (m, n): row 16 m + c of y, columns 32 (n / 2) + 8 g + 4 (n % 2) + 0 .. 3
    f32x4* const red = reinterpret_cast<f32x4*>(sm);
    constexpr int TILES = MT * 2 * NP;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < 2 * NP; ++n) red[(wv * TILES + m * 2 * NP + n) * 64 + l] = acc[m][n];
    __syncthreads();
#pragma unroll
    for (int u = wv; u < MT * NP; u += TG_WAVES) {
        const int m = u / NP, t = u % NP;
        f32x4 lo = red[(2 * u) * 64 + l], hi = red[(2 * u + 1) * 64 + l];
#pragma unroll
        for (int i = 1; i < TG_WAVES; ++i) {
            lo += red[(i * TILES + 2 * u) * 64 + l];
            hi += red[(i * TILES + 2 * u + 1) * 64 + l];
        }
        const int at_m = m0 + 16 * m + c, at_n = n0 + 32 * t + 8 * g;
        if (at_m < M && at_n < N)
            *reinterpret_cast<s16x8*>(y + (long long)at_m * ldy + at_n) = __builtin_shufflevector(to_frag<bf16>(lo).v, to_frag<bf16>(hi).v, 0, 1, 2, 3, 4, 5, 6, 7);
    }
}

template <int MT, int NP, bool TURNED>
static hipError_t launch_tile_gemm(int M, int N, int K, const bf16* x, long long ldx, const bf16* w, long long ldw, bf16* y, long long ldy, hipStream_t s) {
    const dim3 grid((N + 32 * NP - 1) / (32 * NP), (M + 16 * MT - 1) / (16 * MT));
    hipLaunchKernelGGL((tile_gemm_kernel<MT, NP, TURNED>), grid, dim3(64 * TG_WAVES), 0, s, x, ldx, w, ldw, y, ldy, M, N, K);
    return hipGetLastError();
}

}  // namespace hdla

using namespace hdla;

extern "C" int hdla_tile_gemm(int32_t M, int32_t N, int32_t K, const void* x, int64_t ldx, const void* w, int64_t ldw, int32_t turned, void* y, int64_t ldy,
                              void* stream) {
    if (M < 0 || N < 8 || N % 8 || K < 8 || K % 8 || (turned && N % 64)) return HDLA_ERR_SHAPE;
    if (M == 0) return HDLA_OK;
    if (ldx < K || ldw < (turned ? N : K) || ldy < N || (M + 31) / 32 > 65535) return HDLA_ERR_SHAPE;
    if (!x || !w || !y) return HDLA_ERR_NULL;
    for (const void* p : {x, w, (const void*)y})
        if (reinterpret_cast<uintptr_t>(p) & 15) return HDLA_ERR_ALIGN;
    if (ldx % 8 || ldw % 8 || ldy % 8) return HDLA_ERR_ALIGN;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16 *xp = static_cast<const bf16*>(x), *wp = static_cast<const bf16*>(w);
    bf16* const yp = static_cast<bf16*>(y);
    const auto units = [&](int m, int n) { return (long long)((M + m - 1) / m) * ((N + n - 1) / n); };
#define HDLA_TILE(MT, NP)                                                                               \
    (turned ? launch_tile_gemm<MT, NP, true>(M, N, K, xp, ldx, wp, ldw, yp, ldy, s)                     \
            : launch_tile_gemm<MT, NP, false>(M, N, K, xp, ldx, wp, ldw, yp, ldy, s))
    return (int)(units(32, 32) <= TG_UNITS ? HDLA_TILE(2, 1) : units(64, 32) <= TG_UNITS ? HDLA_TILE(4, 1) : HDLA_TILE(4, 2));
#undef HDLA_TILE
}
