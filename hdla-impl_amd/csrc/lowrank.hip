// Matrix products of the HDLA layer for which a BLAS call is the wrong tool.
//
// layer_up: the second halves of the layer's two low-rank projections (f_proj and output_gate, HRDPLR/hdla_custom.py:117-121,
// 151-155: Linear(head_dim -> embed_dim)) and log_f = logsigmoid(f) (:219), in one launch.  x0 [M, D] -> [M, d] with D = 64
// or 128 is bound by what it writes (M x d, three times).  As two BLAS calls and an elementwise kernel it took
// 14.6 + 9.1 + 10.1 us at M = 8192, d = 1024, and in a decode step three launches of 4.5 us and 40 us of host time.
// layer_down: their input gradients, dx0 [M, D] = dY [M, d] W [d, D], with dY = dlog_f sigmoid(-f) formed on the way in for
// the first (as BLAS calls 12 + 12 us and a pass of its own for dY, 10.7 us).
// rows_gemm: y [M, N] = x [M, K] W [N, K]^T for at most 64 rows, i.e. the large projections of a decode step: a stream of W,
// all of the chip's workgroups on it, where the BLAS call costs 20 us of host time and 6 to 13 us (16 x 6416 x 2048; here 5 to 9).
//
// bf16 in and out, fp32 accumulation.  Operands are read 16 bytes a lane; the eight elements are two fragments whose inner
// index is permuted the same way on both sides (elements 8j..8j+3 and 8j+4..8j+7), which a
// sum over that index does not notice.
#include "row_tile.cuh"
#include "../../include/hdla_hip.h"

namespace hdla {

struct TwoTiles { Frag<bf16> a, b; };
__device__ __forceinline__ TwoTiles ld16(const bf16* p) {
    const s16x8 x = *reinterpret_cast<const s16x8*>(p);
    TwoTiles t;
    t.a.v = __builtin_shufflevector(x, x, 0, 1, 2, 3);
    t.b.v = __builtin_shufflevector(x, x, 4, 5, 6, 7);
    return t;
}
// column 8g + i (tile a) and 8g + 4 + i (tile b) of a 32-column block, row c: eight consecutive elements of a row
__device__ __forceinline__ s16x8 pack16(f32x4 a, f32x4 b) {
    return __builtin_shufflevector(to_frag<bf16>(a).v, to_frag<bf16>(b).v, 0, 1, 2, 3, 4, 5, 6, 7);
}
// row of a 32-row block that lane c of a fragment holds, for tile a (+ 4 for tile b)
__device__ __forceinline__ int row8(int c) { return 8 * (c >> 2) + (c & 3); }

// log(sigmoid(x)) as logsigmoid_kernel<bf16> forms it (layer_pre.hip)
__device__ __forceinline__ float logsig(float x) {
    const float e = __expf(-fabsf(x));
    return fminf(x, 0.f) - (e < 1e-4f ? e : __logf(1.f + e));
}

struct UpArgs {
    const bf16 *x0[2], *w[2];             // inner activations [M, D] (rows ldx apart), weights [d, D]: decay, gate
    bf16 *f, *log_f, *gate;               // [M, d]; f may be null (nothing but log_f is asked for)
    long long ldx;
    int M, d;
};
// A wave per 16 MT rows and 32 NB columns; blockIdx.y: decay or gate.  Every wave reads its rows of W (8 or 16 KiB) from L2:
// with one row tile a wave that was 134 MB next to 50 MB of results, 28 us (8192 x 1024), with four 21.  x0, W and (NB = 2) the results
// change lanes in LDS (row_tile.cuh), one after the other in the same place: 21 -> 16.
template <int D, int MT, int NB>
__global__ __launch_bounds__(256) void layer_up_kernel(UpArgs p) {
    constexpr int KB = D / 32;
    typedef RowTile<D> TI;
    typedef RowTile<64> TO;
    constexpr int XR = 16 * MT / TI::RPR, WR = 32 * NB / TI::RPR, BYTES = (MT > 2 * NB ? 16 * MT : 32 * NB) * TI::ROW;
    static_assert(BYTES >= 16 * TO::ROW, "a row tile's results fit as well");
    __shared__ __attribute__((aligned(16))) char sm[4 * BYTES];
    const int l = lane_id(), g = l >> 4, c = l & 15, which = blockIdx.y;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long unit = (long long)blockIdx.x * (blockDim.x >> 6) + wv;
    const int cbs = p.d / (32 * NB);
    const long long r0 = unit / cbs * (16 * MT);
    const int n0 = (int)(unit % cbs) * (32 * NB);
    if (r0 >= p.M) return;
    char* const tile = sm + wv * BYTES;
    s16x8 x[XR], w[WR];
#pragma unroll
    for (int j = 0; j < XR; ++j) x[j] = *reinterpret_cast<const s16x8*>(p.x0[which] + min(r0 + TI::row(j, l), (long long)p.M - 1) * p.ldx + TI::col(l));
#pragma unroll
    for (int j = 0; j < WR; ++j) w[j] = *reinterpret_cast<const s16x8*>(p.w[which] + (long long)(n0 + TI::row(j, l)) * D + TI::col(l));
    TwoTiles xf[MT][KB], wf[NB][2][KB];
#pragma unroll
    for (int j = 0; j < XR; ++j) TI::put(tile, j, l, x[j]);
    wave_lds_fence();
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int k = 0; k < KB; ++k) TI::rows(tile, 16 * m + c, k, l, xf[m][k].a, xf[m][k].b);
    wave_lds_fence();
#pragma unroll
    for (int j = 0; j < WR; ++j) TI::put(tile, j, l, w[j]);
    wave_lds_fence();
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int k = 0; k < KB; ++k) TI::rows(tile, 32 * b + row8(c) + 4 * h, k, l, wf[b][h][k].a, wf[b][h][k].b);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const long long m0 = r0 + 16 * m;
        f32x4 acc[NB][2];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                acc[b][h] = zero4();
#pragma unroll
                for (int k = 0; k < KB; ++k) acc[b][h] = mm2(xf[m][k].a, xf[m][k].b, wf[b][h][k].a, wf[b][h][k].b, acc[b][h]);
            }
        // lane (g, c): row c, columns 32 b + 8 g + 0..7
        auto store = [&](bf16* out) __attribute__((always_inline)) {
            if constexpr (NB == 2) {
                wave_lds_fence();
#pragma unroll
                for (int b = 0; b < NB; ++b) *reinterpret_cast<s16x8*>(tile + TO::place(c, 4 * b + g)) = pack16(acc[b][0], acc[b][1]);
                wave_lds_fence();
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    if (m0 + TO::row(j, l) < p.M) *reinterpret_cast<s16x8*>(out + (m0 + TO::row(j, l)) * p.d + n0 + TO::col(l)) = TO::get(tile, j, l);
            } else if (m0 + c < p.M) {
                *reinterpret_cast<s16x8*>(out + (m0 + c) * p.d + n0 + 8 * g) = pack16(acc[0][0], acc[0][1]);
            }
        };
        if (which == 1) {
            store(p.gate);
        } else {
            if (p.f) store(p.f);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const f32x4 r = to_f32(to_frag<bf16>(acc[b][h]));      // f as the stored tensor has it
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[b][h][i] = logsig(r[i]);
                }
            store(p.log_f);
        }
    }
}

struct DownArgs {
    const bf16 *dy[2], *f, *w[2];         // dlog_f, dgate [M, d]; f [M, d]; weights [d, D]
    bf16* dx[2];                          // [M, D], rows ldx apart
    long long ldx;
    int M, d;
};
// A workgroup per 16 MT rows; its four waves share out the columns of dY, 64 (a cache line of each row) at a time, and add up through
// LDS; blockIdx.y: decay or gate.  W has the contraction index outermost: its rows go to LDS as they come and the transposing LDS read
// takes its tiles from there; dY changes lanes in LDS as well (row_tile.cuh).  8192 x 1024, D = 64: lanes of a request in fragment order
// and products with the identity for W's tiles 18.3 us, this 16.3.
template <int D, int MT>
__global__ __launch_bounds__(256) void layer_down_kernel(DownArgs p) {
    constexpr int NT = D / 16;
    typedef RowTile<64> TY;
    typedef RowTile<D> TW;
    constexpr int YR = 16 * MT / TY::RPR, WR = 64 / TW::RPR, BYTES = 16 * MT * TY::ROW + 64 * TW::ROW;
    static_assert(BYTES >= MT * NT * 1024, "a wave's sums fit where its tiles were");
    __shared__ __attribute__((aligned(16))) char sm[4 * BYTES];
    const int l = lane_id(), g = l >> 4, c = l & 15, which = blockIdx.y;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long r0 = (long long)blockIdx.x * (16 * MT);
    char* const ty = sm + wv * BYTES;
    char* const tw = ty + 16 * MT * TY::ROW;
    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[m][b] = zero4();
    struct In { s16x8 y[YR], f[YR], w[WR]; };
    long long yo[YR];                                     // rows past the end: the last one again, computed and not stored
#pragma unroll
    for (int j = 0; j < YR; ++j) yo[j] = min(r0 + TY::row(j, l), (long long)p.M - 1) * p.d + TY::col(l);
    auto request = [&](int n0) __attribute__((always_inline)) {
        In in;
        const bf16 *const y0 = p.dy[which] + n0, *const f0 = p.f + n0, *const w0 = p.w[which] + (long long)n0 * D;
#pragma unroll
        for (int j = 0; j < YR; ++j) {
            in.y[j] = *reinterpret_cast<const s16x8*>(y0 + yo[j]);
            if (which == 0) in.f[j] = *reinterpret_cast<const s16x8*>(f0 + yo[j]);
        }
#pragma unroll
        for (int j = 0; j < WR; ++j) in.w[j] = *reinterpret_cast<const s16x8*>(w0 + TW::row(j, l) * D + TW::col(l));
        return in;
    };
    // the next columns on their way while some are worked on (D = 64: the other's registers are all taken)
    constexpr bool AHEAD = D == 64;
    int n0 = 64 * wv;
    In next;
    if (AHEAD && n0 < p.d) next = request(n0);
    for (; n0 < p.d; n0 += 256) {
        In in;
        if constexpr (AHEAD) in = next;
        else in = request(n0);
        if (AHEAD && n0 + 256 < p.d) next = request(n0 + 256);
        if (which == 0) {
#pragma unroll
            for (int j = 0; j < YR; ++j) in.y[j] = times_sigmoid_neg(in.y[j], in.f[j]);
        }
        wave_lds_fence();                                 // (the reads of the columns before)
#pragma unroll
        for (int j = 0; j < YR; ++j) TY::put(ty, j, l, in.y[j]);
#pragma unroll
        for (int j = 0; j < WR; ++j) TW::put(tw, j, l, in.w[j]);
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            TwoTiles y[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) TY::rows(ty, 16 * m + c, k, l, y[m].a, y[m].b);
#pragma unroll
            for (int b = 0; b < NT; ++b) {
                const Frag<bf16> wa = TW::columns(tw, 32 * k, 8, b, l), wb = TW::columns(tw, 32 * k + 4, 8, b, l);
#pragma unroll
                for (int m = 0; m < MT; ++m) acc[m][b] = mm2(y[m].a, y[m].b, wa, wb, acc[m][b]);
            }
        }
    }
    __syncthreads();                                      // the sums lie where the waves' tiles were
    f32x4* const red = reinterpret_cast<f32x4*>(sm);
    if (wv) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int b = 0; b < NT; ++b) red[((wv - 1) * MT * NT + m * NT + b) * 64 + l] = acc[m][b];
    }
    __syncthreads();
    if (wv) return;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        if (r0 + 16 * m + c >= p.M) continue;
#pragma unroll
        for (int b = 0; b < NT; ++b) {
            f32x4 s = acc[m][b];
#pragma unroll
            for (int i = 0; i < 3; ++i) s += red[(i * MT * NT + m * NT + b) * 64 + l];
            st_frag(p.dx[which] + (r0 + 16 * m + c) * p.ldx + 16 * b + 4 * g, to_frag<bf16>(s));
        }
    }
}

// y [M, N] = x [M, K] W [N, K]^T, M <= 16 MT.  A workgroup per 16 RT rows of W; its RW waves (eight) take as many parts of K and
// add up through LDS.
//
// What bounds it is the path from memory into the compute unit, and on that the order of the lanes: a fragment's lane order
// (16 rows, 16 bytes of each) puts the four lanes that the address unit takes at a time into four cache lines, at a quarter of the
// rate.  So a request is 64 bytes of 16 rows with the four lanes of a row side by side, and the pieces change lanes through
// 1 KiB of LDS that only their wave uses; what a wave asks for is one stretch of a row (a whole cache line in two requests),
// UNR blocks of it at a time.  Measured (us; every fourth block, lanes in fragment order -> this; weights in the last-level
// cache, then from HBM): 16 x 6416 x 2048 9.1 -> 5.0, 12.0 -> 9.0; 16 x 2048 x 2048 5.2 -> 3.2, 6.9 -> 5.3; 64 x 2048 x 2048
// 11.0 -> 5.6, 13.8 -> 8.3; 16 x 512 x 512, one launch's time, 2.65 -> 2.3.  (The 26 MB of the first at copy rate: 5.4.)
// UNR: a wave's whole share of K up to 2048 (16 rows) in one or two goes; twice as many is no faster (16 x 6416 x 2048 5.0,
// 64 x 6416 x 2048 7.6 -> 8.7) and asks twice for K = 512 what is there once (1 -> 2 blocks a wave too many, 2.5 -> 3.0 for 32 rows).
constexpr int ROW_WAVES = 8;
// NORM (one row tile): x is formed on the way in, x = gated c / sqrt(K) / sqrt(sum of the row's parts / K + eps) weight, rounded to bf16
// as the norm's output is: one launch less, and no pass over a few rows that is all latency (16 x 2048 x 2048: norm 4.1 and product 4.4
// -> 7.6 us).
struct NormIn {
    const float *gated, *sums;            // [M, K], [M, parts]
    const void* weight;                   // [K] or null
    int parts, w_f32;
    float cn, inv_e, eps;
};
template <int MT, int RT, int UNR, bool NORM, int RW = 8>
__global__ __launch_bounds__(64 * RW) void rows_gemm_kernel(const bf16* __restrict__ x, long long ldx, const bf16* __restrict__ w, long long ldw,
                                                            bf16* __restrict__ y, long long ldy, int M, int N, int K, NormIn nrm) {
    static_assert(!NORM || MT == 1, "one row tile");
    constexpr int TURN = RT + MT, SUMS = RT * MT;         // KiB a wave: to change lanes in, of sums
    static_assert(SUMS <= RW, "a wave per tile of the result");
    __shared__ __attribute__((aligned(16))) char sm[RW * (TURN > SUMS ? TURN : SUMS) * 1024];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id(), g = l >> 4, c = l & 15;
    const int n0 = blockIdx.x * (16 * RT), row = l >> 2, piece = l & 3;
    // row r's pieces p lie at 4 r + (p ^ r / 4): 16 lanes of either order meet each bank once
    char* const put = sm + wv * (TURN * 1024) + ((4 * row + (piece ^ (row >> 2))) << 4);
    char* const put_half = sm + wv * (TURN * 1024) + 64 * row + 8 * (piece & 1);
    const char* const get = sm + wv * (TURN * 1024) + ((4 * c + (g ^ (c >> 2))) << 4);
    const bf16* from[TURN];                               // rows past the end: read again, not stored
#pragma unroll
    for (int i = 0; i < TURN; ++i)
        from[i] = (i < RT ? w + (long long)min(n0 + 16 * i + row, N - 1) * ldw : x + (long long)min(16 * (i - RT) + row, M - 1) * ldx) + 8 * piece;
    float rs = 0.f;
    // (of gated, twice the bytes, a lane has four columns in each half of the block: requests of 64 bytes a row here too)
    const float* const gated = NORM ? nrm.gated + (long long)min(row, M - 1) * K + 4 * piece : nullptr;
    bool scaled = false;
    // the row's scale, four lanes a row as everywhere here; behind the first blocks' requests, and all of its own at once
    auto scale_row = [&]() __attribute__((always_inline)) {
        const float* const sums = nrm.sums + (long long)min(row, M - 1) * nrm.parts;
        float ss = 0.f;
        for (int h0 = 0; h0 < nrm.parts; h0 += 32) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = sums[min(h0 + 4 * i + piece, nrm.parts - 1)];
#pragma unroll
            for (int i = 0; i < 8; ++i) ss += h0 + 4 * i + piece < nrm.parts ? v[i] : 0.f;
        }
        ss = sum_lanes(ss, 4);
        rs = nrm.cn / sqrtf(ss * nrm.inv_e + nrm.eps);
        scaled = true;
    };
    const int nb = K / 32, per = (nb + RW - 1) / RW, end = min(nb, (wv + 1) * per);
    f32x4 acc[RT][MT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[r][m] = zero4();
    // (no branch around a block's products: its requests would be moved behind it)
    auto blocks = [&](int b0, bool whole) __attribute__((always_inline)) {
        s16x8 in[UNR][TURN];
        f32x4 gx[NORM ? UNR : 1][2], wx[NORM ? UNR : 1][2];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int at = 32 * (whole ? b0 + u : min(b0 + u, end - 1));
#pragma unroll
            for (int i = 0; i < (NORM ? RT : TURN); ++i) in[u][i] = *reinterpret_cast<const s16x8*>(from[i] + at);
            if constexpr (NORM) {
#pragma unroll
                for (int i = 0; i < 2; ++i) gx[u][i] = *reinterpret_cast<const f32x4*>(gated + at + 16 * i);
                if (!nrm.weight) {
                    wx[u][0] = wx[u][1] = f32x4{1.f, 1.f, 1.f, 1.f};
                } else if (nrm.w_f32) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) wx[u][i] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(nrm.weight) + at + 16 * i + 4 * piece);
                } else {
#pragma unroll
                    for (int i = 0; i < 2; ++i) wx[u][i] = to_f32(ld_frag(static_cast<const bf16*>(nrm.weight) + at + 16 * i + 4 * piece));
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);                // all of them requested before the first is waited for
        if (NORM && !scaled) scale_row();
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const s16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
            wave_lds_fence();                             // (the reads of the block before)
#pragma unroll
            for (int i = 0; i < (NORM ? RT : TURN); ++i) *reinterpret_cast<s16x8*>(put + 1024 * i) = whole || b0 + u < end ? in[u][i] : zero;
            if constexpr (NORM) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    *reinterpret_cast<s16x4*>(put_half + 1024 * RT + (((piece >> 1) + 2 * i) ^ (row >> 2)) * 16) = to_frag<bf16>(gx[u][i] * rs * wx[u][i]).v;
            }
            wave_lds_fence();
            TwoTiles t[TURN];
#pragma unroll
            for (int i = 0; i < TURN; ++i) t[i] = ld16(reinterpret_cast<const bf16*>(get + 1024 * i));
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int m = 0; m < MT; ++m) acc[r][m] = mm2(t[RT + m].a, t[RT + m].b, t[r].a, t[r].b, acc[r][m]);
        }
    };
    int b0 = wv * per;
    for (; b0 + UNR <= end; b0 += UNR) blocks(b0, true);
    if (b0 < end) blocks(b0, false);
    __syncthreads();                                      // the sums lie where the others changed lanes
    f32x4* const red = reinterpret_cast<f32x4*>(sm);
#pragma unroll
    for (int i = 0; i < SUMS; ++i) red[(wv * SUMS + i) * 64 + l] = acc[i / MT][i % MT];
    __syncthreads();
    if (wv >= SUMS) return;
    f32x4 s = red[wv * 64 + l];
#pragma unroll
    for (int i = 1; i < RW; ++i) s += red[(i * SUMS + wv) * 64 + l];
    const int m = 16 * (wv % MT) + c, n = n0 + 16 * (wv / MT) + 4 * g;
    if (m >= M) return;
    bf16* o = y + (long long)m * ldy + n;
    if (n + 3 < N) st_frag(o, to_frag<bf16>(s));
    else {
#pragma unroll
        for (int i = 0; i < 4; ++i) if (n + i < N) st_elem(o + i, s[i]);
    }
}

static bool lr_al(const void* p, int a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }
static int lr_check(const hdla_up_dims* q) {
    if (!q) return HDLA_ERR_NULL;
    if (q->rows < 0 || q->rows > 0x7fffffff || (q->D != 64 && q->D != 128) || q->d <= 0 || q->d % 128) return HDLA_ERR_SHAPE;
    if (q->ld < q->D || q->ld % 8 || q->col_f < 0 || q->col_g < 0 || q->col_f % 8 || q->col_g % 8) return HDLA_ERR_ALIGN;
    if (q->col_f + q->D > q->ld || q->col_g + q->D > q->ld) return HDLA_ERR_SHAPE;
    return HDLA_OK;
}

}  // namespace hdla

using namespace hdla;

extern "C" int hdla_layer_up_fwd(const hdla_up_dims* dims, const void* y, const void* wf, const void* wg, void* f, void* log_f, void* gate,
                                 void* stream) {
    const int rc = lr_check(dims);
    if (rc) return rc;
    if (dims->rows == 0) return HDLA_OK;
    if (!y || !wf || !wg || !log_f || !gate) return HDLA_ERR_NULL;
    for (const void* p : {y, wf, wg, (const void*)f, (const void*)log_f, (const void*)gate}) if (!lr_al(p, 16)) return HDLA_ERR_ALIGN;
    // four row tiles a wave where that leaves enough waves for the device; few rows: half the columns a wave, a compute unit each
    const int mt = (dims->rows + 63) / 64 * (dims->d / 64) >= 1024 ? 4 : 1;
    const bool few = (dims->rows + 15) / 16 * (dims->d / 64) <= 256;
    const long long units = (dims->rows + 16 * mt - 1) / (16 * mt) * (dims->d / (few ? 32 : 64)), each = few ? 1 : 4;
    if ((units + each - 1) / each > 0x7fffffffLL) return HDLA_ERR_SHAPE;
    UpArgs a{};
    a.x0[0] = static_cast<const bf16*>(y) + dims->col_f; a.x0[1] = static_cast<const bf16*>(y) + dims->col_g;
    a.w[0] = static_cast<const bf16*>(wf); a.w[1] = static_cast<const bf16*>(wg);
    a.f = static_cast<bf16*>(f); a.log_f = static_cast<bf16*>(log_f); a.gate = static_cast<bf16*>(gate);
    a.ldx = dims->ld; a.M = (int)dims->rows; a.d = dims->d;
    const dim3 grid((unsigned)((units + each - 1) / each), 2), block((unsigned)(64 * each));
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (dims->D == 64) {
        if (mt == 4) hipLaunchKernelGGL((layer_up_kernel<64, 4, 2>), grid, block, 0, s, a);
        else if (few) hipLaunchKernelGGL((layer_up_kernel<64, 1, 1>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((layer_up_kernel<64, 1, 2>), grid, block, 0, s, a);
    } else {
        if (mt == 4) hipLaunchKernelGGL((layer_up_kernel<128, 4, 2>), grid, block, 0, s, a);
        else if (few) hipLaunchKernelGGL((layer_up_kernel<128, 1, 1>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((layer_up_kernel<128, 1, 2>), grid, block, 0, s, a);
    }
    return (int)hipGetLastError();
}

extern "C" int hdla_layer_down(const hdla_up_dims* dims, const void* wf, const void* wg, const void* f, const void* dlog_f, const void* dgate,
                               void* dy, void* stream) {
    const int rc = lr_check(dims);
    if (rc) return rc;
    if (dims->rows == 0) return HDLA_OK;
    if (!wf || !wg || !f || !dlog_f || !dgate || !dy) return HDLA_ERR_NULL;
    for (const void* p : {wf, wg, f, dlog_f, dgate, (const void*)dy}) if (!lr_al(p, 16)) return HDLA_ERR_ALIGN;
    DownArgs a{};
    a.dy[0] = static_cast<const bf16*>(dlog_f); a.dy[1] = static_cast<const bf16*>(dgate); a.f = static_cast<const bf16*>(f);
    a.w[0] = static_cast<const bf16*>(wf); a.w[1] = static_cast<const bf16*>(wg);
    a.dx[0] = static_cast<bf16*>(dy) + dims->col_f; a.dx[1] = static_cast<bf16*>(dy) + dims->col_g;
    a.ldx = dims->ld; a.M = (int)dims->rows; a.d = dims->d;
    const dim3 block(256);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    // row tiles a workgroup: what the registers hold; few rows are spread over more workgroups
    const bool wide = dims->rows >= 4096;
    const auto grid = [&](int mt) { return dim3((unsigned)((dims->rows + 16 * mt - 1) / (16 * mt)), 2); };
    if (dims->D == 64) {
        if (wide) hipLaunchKernelGGL((layer_down_kernel<64, 2>), grid(2), block, 0, s, a);
        else hipLaunchKernelGGL((layer_down_kernel<64, 1>), grid(1), block, 0, s, a);
    } else {
        if (wide) hipLaunchKernelGGL((layer_down_kernel<128, 2>), grid(2), block, 0, s, a);
        else hipLaunchKernelGGL((layer_down_kernel<128, 1>), grid(1), block, 0, s, a);
    }
    return (int)hipGetLastError();
}

// ---- the weights of the projections that share an input, one behind the other, zeros behind them ---------------------------
// A copy that runs as long as its launch and one trip through memory: torch's cat and the zeros of the padding were two launches and
// 12 us for 3328 x 1024 (7 MB each way); every thread here has four pieces of 16 bytes on their way at once.
// Measured: layer training step 770.8 -> 766.8 us (4 x 2048 tokens, d = 1024), a small one bound by the host 360 -> 345.
namespace hdla {
constexpr int STACK_MAX = 8, STACK_PIECES = 4;
struct StackArgs { const i32x4* p[STACK_MAX]; long long end[STACK_MAX]; };   // end: of each part in the output, in 16-byte pieces
__global__ __launch_bounds__(256) void stack_rows_kernel(StackArgs a, i32x4* out, long long n) {
    const long long i0 = (long long)blockIdx.x * (256 * STACK_PIECES) + threadIdx.x;
    i32x4 x[STACK_PIECES];
#pragma unroll
    for (int j = 0; j < STACK_PIECES; ++j) {
        const long long i = i0 + 256 * j;
        const i32x4* src = nullptr;
        long long start = 0;
#pragma unroll
        for (int m = 0; m < STACK_MAX; ++m) {             // the parts' ends never decrease; those past `count` equal the last
            if (src == nullptr && i < a.end[m]) src = a.p[m] + (i - start);
            start = a.end[m];
        }
        x[j] = i32x4{0, 0, 0, 0};
        if (src) x[j] = *src;
    }
#pragma unroll
    for (int j = 0; j < STACK_PIECES; ++j)
        if (i0 + 256 * j < n) out[i0 + 256 * j] = x[j];
}
}  // namespace hdla

extern "C" int hdla_stack_rows(const void* const* parts, const int64_t* rows, int32_t count, int64_t width, void* out, int64_t total_rows,
                               void* stream) {
    if (count < 1 || count > STACK_MAX || width < 8 || width % 8 || total_rows < 0 || total_rows > INT32_MAX || width > INT32_MAX) return HDLA_ERR_SHAPE;
    if (!parts || !rows || (!out && total_rows)) return HDLA_ERR_NULL;
    StackArgs a{};
    long long end = 0;
    for (int m = 0; m < STACK_MAX; ++m) {
        if (m < count) {
            if (rows[m] < 0 || rows[m] > total_rows) return HDLA_ERR_SHAPE;
            if (rows[m] && !parts[m]) return HDLA_ERR_NULL;
            if (!lr_al(parts[m], 16)) return HDLA_ERR_ALIGN;
            a.p[m] = static_cast<const i32x4*>(parts[m]);
            end += rows[m] * (width / 8);
        }
        a.end[m] = end;
    }
    const long long n = (long long)total_rows * (width / 8);
    if (end > n) return HDLA_ERR_SHAPE;
    if (!lr_al(out, 16)) return HDLA_ERR_ALIGN;
    if (n == 0) return HDLA_OK;
    const long long blocks = (n + 256 * STACK_PIECES - 1) / (256 * STACK_PIECES);
    if (blocks > INT32_MAX) return HDLA_ERR_SHAPE;
    hipLaunchKernelGGL(stack_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), a, static_cast<i32x4*>(out), n);
    return (int)hipGetLastError();
}

extern "C" int hdla_rows_gemm(int32_t M, int32_t N, int32_t K, const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy,
                              void* stream) {
    if (M < 0 || M > 64 || N < 1 || K < 32 || K % 32) return HDLA_ERR_SHAPE;
    if (M == 0) return HDLA_OK;
    if (ldx < K || ldw < K || ldy < N) return HDLA_ERR_SHAPE;
    if (!x || !w || !y) return HDLA_ERR_NULL;
    if (!lr_al(x, 16) || !lr_al(w, 16) || !lr_al(y, 8) || ldx % 8 || ldw % 8 || ldy % 4) return HDLA_ERR_ALIGN;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16 *xp = static_cast<const bf16*>(x), *wp = static_cast<const bf16*>(w);
    bf16* yp = static_cast<bf16*>(y);
    // Two tiles of W's rows a workgroup where the x that every workgroup reads is as much as that (more than 16 rows of it), once
    // one tile each is more than a workgroup a compute unit.  One tile / two, weights in the last-level cache, us: K = 2048, 64 rows,
    // 4096 columns 6.5 / 7.3, 5120 9.2 / 7.4, 6416 9.4 / 7.5; 32 rows 4.4 / 5.9, 6.6 / 6.1, 6.5 / 6.25.
    const bool two = M > 16 && N > 16 * 256;
    const dim3 grid((N + (two ? 31 : 15)) / (two ? 32 : 16)), block(64 * ROW_WAVES);
#define HDLA_ROWS(MT, RT, UNR) \
    hipLaunchKernelGGL((rows_gemm_kernel<MT, RT, UNR, false>), grid, block, 0, s, xp, (long long)ldx, wp, (long long)ldw, yp, (long long)ldy, M, N, K, NormIn{})
    if (M <= 16 && K <= 64 * ROW_WAVES) HDLA_ROWS(1, 1, 2);
    else if (M <= 16) HDLA_ROWS(1, 1, 4);
    else if (M <= 32 && !two && K <= 64 * ROW_WAVES) HDLA_ROWS(2, 1, 2);
    else if (M <= 32 && !two) HDLA_ROWS(2, 1, 4);
    else if (M <= 32) HDLA_ROWS(2, 2, 4);
    else if (!two) HDLA_ROWS(4, 1, 2);
    else HDLA_ROWS(4, 2, 2);
#undef HDLA_ROWS
    return (int)hipGetLastError();
}

extern "C" int hdla_rows_gemm_norm(int32_t M, int32_t N, int32_t K, const float* gated, int32_t parts, const hdla_norm_dims* norm, const void* weight,
                                   const void* w, int64_t ldw, void* y, int64_t ldy, void* stream) {
    if (!norm) return HDLA_ERR_NULL;
    if (norm->dtype != HDLA_BF16 || (weight && norm->weight_dtype != HDLA_BF16 && norm->weight_dtype != HDLA_FP32)) return HDLA_ERR_DTYPE;
    if (M < 0 || M > 16 || N < 1 || K < 32 || K % 32 || parts < 1 || norm->rows != M || norm->G != 1 || norm->E != K || !(norm->eps >= 0.f)) return HDLA_ERR_SHAPE;
    if (M == 0) return HDLA_OK;
    if (ldw < K || ldy < N) return HDLA_ERR_SHAPE;
    if (!gated || !w || !y) return HDLA_ERR_NULL;
    if (!lr_al(gated, 16) || !lr_al(weight, 16) || !lr_al(w, 16) || !lr_al(y, 8) || ldw % 8 || ldy % 4) return HDLA_ERR_ALIGN;
    const NormIn nrm{gated, gated + (int64_t)M * K, weight, parts, norm->weight_dtype == HDLA_FP32, norm->c / sqrtf((float)K), 1.f / (float)K, norm->eps};
    const dim3 grid((N + 15) / 16);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16* wp = static_cast<const bf16*>(w);
    bf16* yp = static_cast<bf16*>(y);
    // Waves and blocks a go as ask for all of K at once, as far as the registers reach: sixteen waves for K = 2048, where eight asked twice.  us a decode step of
    // the layer, as a graph's replay, eight / sixteen: 16 sequences, 2048 channels 24.4 / 23.4, 4 21.4 / 20.5, 1 20.9 / 19.8; 16, 1152 channels 22.5 / 21.3, 1536 22.9 / 22.1, 1792 23.9 / 23.5; 16, 1024
    // channels, whose K eight have in one go, 13.9 / 14.6.
#define HDLA_ROWS(UNR, WAVES)                                                                                                                       \
    hipLaunchKernelGGL((rows_gemm_kernel<1, 1, UNR, true, WAVES>), grid, dim3(64 * WAVES), 0, s, nullptr, 0LL, wp, (long long)ldw, yp, (long long)ldy, M, N, K, nrm)
    if (K <= 64 * ROW_WAVES) HDLA_ROWS(2, ROW_WAVES);
    else if (K <= 128 * ROW_WAVES) HDLA_ROWS(4, ROW_WAVES);
    else HDLA_ROWS(4, 16);
#undef HDLA_ROWS
    return (int)hipGetLastError();
}
