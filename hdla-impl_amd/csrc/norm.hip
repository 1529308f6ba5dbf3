// Fused normalisation with an optional gate: the operator the HDLA layer applies right after the attention
// operator (gated RMSNorm, HRDPLR/hdla_custom.py:341-345) and to q, k, v right before it (l2_norm, :247-251).
//
// Replaces _normalize_fwd / _normalize_bwd, HRDPLR/normalizations/normalize/normalize/normalize_triton.py:21-253,
// for use_mean = False and no bias or residual.  Per (row, group) of E channels:
//     x' = x * sigmoid(gate)                      gate before the norm            (normalize_triton.py:84-89)
//     sigma = sqrt(sum x'^2 / E + eps)                                            (:103)
//     o = (c / sqrt(E)) * x' / sigma * weight  [ * sigmoid(gate), gate after ]    (:104-117)
// and the matching backward pass (:186-251), with sigma recomputed instead of stored.
//
// Both passes are streams through HBM (forward: read x, gate, write o; backward: read x, gate, do, write dx, dgate),
// so the layout is chosen for that: a row (or, for short groups, 64/LPR consecutive groups) per wavefront pass, 16
// bytes per lane and piece, LPR = a power of two lanes across one group, all pieces of a pass in flight before the
// first use, sums over a group as butterflies inside the wavefront (no LDS, no barrier).  Wavefronts stride over the
// groups such that a lane always meets the same weight columns: weights are loaded once, and the weight gradient
// accumulates in registers and leaves as one partial row per (wavefront, group position), summed by a second small
// kernel in a fixed order (results do not depend on timing).
#include "sums.cuh"
#include "../../include/hdla_hip.h"

namespace hdla {

struct NormArgs {
    const void *x, *gate, *weight, *d_o;
    void *o, *dx, *dgate;
    float* partial;            // [(workgroups or waves) * groups per pass][E], backward with a weight
    long long nslot;           // rows * G: groups to normalise, E consecutive elements each
    long long nsg;             // wavefront passes: ceil(nslot / (64 >> lpr_log2))
    int G, E, lpr_log2, w_f32, gate_pos;
    int wg_reduce;             // the four wavefronts of a workgroup meet the same weight columns: one partial row set
    int wg_row;                // long groups: the four wavefronts of a workgroup share one group, 256 lanes across it
    float cn, inv_e, eps;      // c / sqrt(E), 1 / E
};

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes of a row as floats
template <typename T> struct Piece;
template <> struct Piece<bf16> {
    static constexpr int N = 8;
    static __device__ __forceinline__ u32x4 raw(const void* base, long long elem) {
        return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(static_cast<const bf16*>(base) + elem));
    }
    static __device__ __forceinline__ void unpack(u32x4 r, float (&f)[8]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[2 * i] = __uint_as_float(r[i] << 16);
            f[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
        }
    }
    static __device__ __forceinline__ void st(void* base, long long elem, const float (&f)[8]) {
        const s16x4 lo = to_frag<bf16>(f32x4{f[0], f[1], f[2], f[3]}).v, hi = to_frag<bf16>(f32x4{f[4], f[5], f[6], f[7]}).v;
        __builtin_nontemporal_store(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), reinterpret_cast<s16x8*>(static_cast<bf16*>(base) + elem));
    }
};
template <> struct Piece<float> {
    static constexpr int N = 4;
    static __device__ __forceinline__ u32x4 raw(const void* base, long long elem) {
        return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(static_cast<const float*>(base) + elem));
    }
    static __device__ __forceinline__ void unpack(u32x4 r, float (&f)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(r[i]);
    }
    static __device__ __forceinline__ void st(void* base, long long elem, const float (&f)[4]) {
        f32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = f[i];
        __builtin_nontemporal_store(r, reinterpret_cast<f32x4*>(static_cast<float*>(base) + elem));
    }
};

// N consecutive weights, 16 bytes a load
template <int N> __device__ __forceinline__ void ld_weight(const void* w, int w_f32, int col, float (&f)[N]) {
    if (w_f32) {
#pragma unroll
        for (int i = 0; i < N; i += 4) {
            const f32x4 r = *reinterpret_cast<const f32x4*>(static_cast<const float*>(w) + col + i);
#pragma unroll
            for (int j = 0; j < 4; ++j) f[i + j] = r[j];
        }
    } else {
        // (fp32 data next to bf16 weights: N = 4, eight bytes)
#pragma unroll
        for (int i = 0; i < N; i += 4) {
            const f32x4 r = to_f32(ld_frag(static_cast<const bf16*>(w) + col + i));
#pragma unroll
            for (int j = 0; j < 4; ++j) f[i + j] = r[j];
        }
    }
}

// x = sigmoid(x)
template <int N> __device__ __forceinline__ void sigmoids(float (&x)[N]) {
    float e[N];
#pragma unroll
    for (int j = 0; j < N; ++j) e[j] = __expf(-x[j]);
    sigmoid_of_exp<N>(e, x);
}

// Where a lane stands: lane sl of the LPR lanes across one group, group position rw of the 64/LPR groups of a pass;
// `wave` counts passes' owners (wavefronts, or workgroups when a workgroup shares one long group).
struct NormLane {
    int lpr, rpw, sl, rw, wg_row;
    long long wave, nwave;
    __device__ __forceinline__ explicit NormLane(const NormArgs& p) {
        const int lane = threadIdx.x & 63;
        wg_row = p.wg_row;
        if (wg_row) {
            lpr = 256; rpw = 1; sl = threadIdx.x; rw = 0;
            nwave = gridDim.x;
            wave = blockIdx.x;
        } else {
            lpr = 1 << p.lpr_log2;
            rpw = 64 >> p.lpr_log2;
            sl = lane & (lpr - 1);
            rw = lane >> p.lpr_log2;
            nwave = (long long)gridDim.x * 4;
            wave = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
        }
    }
};

// Sums of a and b over the lanes of one group, on all of them.  Across the wavefronts of a workgroup the partial
// sums go through `sred` ([2][4][2] floats, alternating halves, so one barrier per call is enough); every thread of
// the workgroup makes the same calls.
__device__ __forceinline__ void group_sum(const NormLane& L, float& a, float& b, float* sred, int& buf) {
    const int width = L.wg_row ? 64 : L.lpr;
    // (us, by __shfl_xor -> this: 8192 x 1024 bf16 11.7 + 21.3 -> 11.2 + 20.4, 65536 x 4096 364 + 621 -> 350 + 605)
    float both[2] = {a, b};
    sum_lanes<2>(both, width);
    a = both[0];
    b = both[1];
    if (L.wg_row) {
        float* s = sred + buf * 8;
        if ((threadIdx.x & 63) == 0) { s[2 * (threadIdx.x >> 6)] = a; s[2 * (threadIdx.x >> 6) + 1] = b; }
        __syncthreads();
        a = (s[0] + s[2]) + (s[4] + s[6]);
        b = (s[1] + s[3]) + (s[5] + s[7]);
        buf ^= 1;
    }
}

template <typename T, int NV>
__global__ __launch_bounds__(256) void normalize_fwd_kernel(NormArgs p) {
    constexpr int N = Piece<T>::N;
    const NormLane L(p);
    __shared__ float sred[16];
    int buf = 0;
    const bool pre = p.gate_pos == 1, post = p.gate_pos == 2;
    const int E = p.E;
    // the launch makes nwave * rpw a multiple of G: the group index of a lane's slots never changes
    const int g = (int)((L.wave * L.rpw + L.rw) % p.G);
    // A pass's pieces are requested while the pass before it is worked on (the first one's before the weights): otherwise a
    // wavefront with two passes waits for HBM twice (8192 x 1024 bf16, with the weights loaded 16 bytes at a time: 19.2 -> 11.6 us
    // by itself, 17.3 -> 14.2 in a layer training step).  The largest rows have no registers for it.
    constexpr bool AHEAD = NV <= 4;
    u32x4 rx[NV], rg[NV];
    auto request = [&](long long sg) __attribute__((always_inline)) {
        const long long slot = sg * L.rpw + L.rw;
        const bool live = sg < p.nsg && slot < p.nslot;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int e = (i * L.lpr + L.sl) * N;
            rx[i] = u32x4{0, 0, 0, 0};
            rg[i] = u32x4{0, 0, 0, 0};
            if (live && e < E) {
                rx[i] = Piece<T>::raw(p.x, slot * E + e);
                if (p.gate_pos) rg[i] = Piece<T>::raw(p.gate, slot * E + e);
            }
        }
    };
    if (AHEAD) request(L.wave);
    float w[NV][N];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int e = (i * L.lpr + L.sl) * N;
        if (p.weight && e < E) ld_weight<N>(p.weight, p.w_f32, g * E + e, w[i]);
        else {
#pragma unroll
            for (int j = 0; j < N; ++j) w[i][j] = 1.f;
        }
    }
    for (long long sg = L.wave; sg < p.nsg; sg += L.nwave) {
        const long long slot = sg * L.rpw + L.rw;
        const bool live = slot < p.nslot;
        if (!AHEAD) request(sg);
        float x[NV][N], gs[NV][N];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            Piece<T>::unpack(rx[i], x[i]);
            Piece<T>::unpack(rg[i], gs[i]);
        }
        if (AHEAD) request(sg + L.nwave);
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            if (p.gate_pos) sigmoids<N>(gs[i]);
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (pre) x[i][j] *= gs[i][j];
                ss += x[i][j] * x[i][j];
            }
        }
        float unused = 0.f;
        group_sum(L, ss, unused, sred, buf);
        const float rs = p.cn / sqrtf(ss * p.inv_e + p.eps);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int e = (i * L.lpr + L.sl) * N;
            float o[N];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                o[j] = x[i][j] * rs * w[i][j];
                if (post) o[j] *= gs[i][j];
            }
            if (live && e < E) Piece<T>::st(p.o, slot * E + e, o);
        }
    }
}

template <typename T, int NV>
__global__ __launch_bounds__(256) void normalize_bwd_kernel(NormArgs p) {
    constexpr int N = Piece<T>::N;
    const NormLane L(p);
    __shared__ float sred[16];
    int buf = 0;
    const bool pre = p.gate_pos == 1, post = p.gate_pos == 2, has_w = p.weight != nullptr;
    const int E = p.E;
    const int g = (int)((L.wave * L.rpw + L.rw) % p.G);
    constexpr bool AHEAD = NV <= 2;                       // see the forward kernel
    u32x4 rx[NV], rg[NV], rd[NV];
    auto request = [&](long long sg) __attribute__((always_inline)) {
        const long long slot = sg * L.rpw + L.rw;
        const bool live = sg < p.nsg && slot < p.nslot;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int e = (i * L.lpr + L.sl) * N;
            rx[i] = u32x4{0, 0, 0, 0};
            rg[i] = u32x4{0, 0, 0, 0};
            rd[i] = u32x4{0, 0, 0, 0};
            if (live && e < E) {
                rx[i] = Piece<T>::raw(p.x, slot * E + e);
                rd[i] = Piece<T>::raw(p.d_o, slot * E + e);
                if (p.gate_pos) rg[i] = Piece<T>::raw(p.gate, slot * E + e);
            }
        }
    };
    if (AHEAD) request(L.wave);
    float w[NV][N], dw[NV][N];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int e = (i * L.lpr + L.sl) * N;
        if (has_w && e < E) ld_weight<N>(p.weight, p.w_f32, g * E + e, w[i]);
        else {
#pragma unroll
            for (int j = 0; j < N; ++j) w[i][j] = 1.f;
        }
#pragma unroll
        for (int j = 0; j < N; ++j) dw[i][j] = 0.f;
    }
    // A workgroup that shares its groups meets four times as many as a wavefront would: the weight gradient's sums of FOLD of them are added to those of
    // the ones before in the lane's own place in LDS, so that no sum is longer than it was (fp32 20000 x 1024, error 1.93e-7; one sum of 20: 2.06e-7).
    constexpr int FOLD = 4;
    __shared__ float sdw[NV * N * 256];
    int folded = 0, met = 0;
    for (long long sg = L.wave; sg < p.nsg; sg += L.nwave) {
        if (has_w && L.wg_row && met == FOLD) {
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    float* const at = sdw + (i * N + j) * 256 + threadIdx.x;
                    *at = folded ? *at + dw[i][j] : dw[i][j];
                    dw[i][j] = 0.f;
                }
            folded = 1;
            met = 0;
        }
        ++met;
        const long long slot = sg * L.rpw + L.rw;
        const bool live = slot < p.nslot;
        if (!AHEAD) request(sg);
        float x[NV][N], gs[NV][N], dr[NV][N];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            Piece<T>::unpack(rx[i], x[i]);
            Piece<T>::unpack(rd[i], dr[i]);
            Piece<T>::unpack(rg[i], gs[i]);
        }
        if (AHEAD) request(sg + L.nwave);
        // x: the normalised quantity (gated when the gate comes first); dr: gradient of x / sigma before the weight
        float ss = 0.f, sd = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            if (p.gate_pos) sigmoids<N>(gs[i]);
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (pre) x[i][j] *= gs[i][j];
                dr[i][j] *= p.cn;
                if (post) dr[i][j] *= gs[i][j];
                ss += x[i][j] * x[i][j];
                sd += x[i][j] * dr[i][j] * w[i][j];
            }
        }
        group_sum(L, ss, sd, sred, buf);
        const float inv = 1.f / sqrtf(ss * p.inv_e + p.eps);          // 1 / sigma
        const float proj = sd * inv * p.inv_e;                         // sum(r * dr * w) / E, r = x / sigma
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int e = (i * L.lpr + L.sl) * N;
            float dx[N], dg[N];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const float r = x[i][j] * inv;
                dw[i][j] += dr[i][j] * r;
                const float dxn = inv * (dr[i][j] * w[i][j] - r * proj);
                if (pre) {
                    // x = x_in * gs: d x_in = dxn * gs, d gate = dxn * x_in * gs (1 - gs) = dxn * x * (1 - gs)
                    dx[j] = dxn * gs[i][j];
                    dg[j] = dxn * x[i][j] * (1.f - gs[i][j]);
                } else if (post) {
                    // o = n * gs with n = cn * r * w; dr already carries gs, so d gate = do * n * gs (1 - gs)
                    dx[j] = dxn;
                    dg[j] = dr[i][j] * r * w[i][j] * (1.f - gs[i][j]);
                } else {
                    dx[j] = dxn;
                    dg[j] = 0.f;
                }
            }
            if (live && e < E) {
                Piece<T>::st(p.dx, slot * E + e, dx);
                if (p.gate_pos) Piece<T>::st(p.dgate, slot * E + e, dg);
            }
        }
    }
    if (has_w) {
        if (folded) {
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int j = 0; j < N; ++j) dw[i][j] += sdw[(i * N + j) * 256 + threadIdx.x];
        }
        long long prow = L.wave * L.rpw + L.rw;
        if (p.wg_reduce) {
            // lane by lane the four wavefronts hold the same columns: waves 2, 3 hand over to 0, 1, then 1 to 0
            float* const swg = sdw;                       // [2][NV * N][64]
            const int wl = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
            for (int round = 0; round < 2; ++round) {
                const int half = 2 >> round;                  // 2, then 1
                if (wl >= half && wl < 2 * half) {
#pragma unroll
                    for (int i = 0; i < NV; ++i)
#pragma unroll
                        for (int j = 0; j < N; ++j) swg[((wl - half) * NV * N + i * N + j) * 64 + lane] = dw[i][j];
                }
                __syncthreads();
                if (wl < half) {
#pragma unroll
                    for (int i = 0; i < NV; ++i)
#pragma unroll
                        for (int j = 0; j < N; ++j) dw[i][j] += swg[(wl * NV * N + i * N + j) * 64 + lane];
                }
                __syncthreads();
            }
            if (wl != 0) return;
            prow = (long long)blockIdx.x * L.rpw + L.rw;
        }
        float* row = p.partial + prow * E;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int e = (i * L.lpr + L.sl) * N;
            if (e < E) {
#pragma unroll
                for (int j = 0; j < N; j += 4) {
                    f32x4 v = {dw[i][j], dw[i][j + 1], dw[i][j + 2], dw[i][j + 3]};
                    *reinterpret_cast<f32x4*>(row + e + j) = v;
                }
            }
        }
    }
}

// Launch shape shared by both passes and by the workspace size.
struct NormCfg {
    int n, nv, lpr_log2, rpw, wg_reduce, wg_row;
    long long nslot, nsg, nwg;
    long long partial_rows() const { return wg_row ? nwg : nwg * (wg_reduce ? 1 : 4) * rpw; }
};

static long long gcd_ll(long long a, long long b) { while (b) { const long long t = a % b; a = b; b = t; } return a; }

// The backward kernel of 2-byte elements with two pieces a lane: its registers leave room for three workgroups a compute unit, and a fourth on all of them
// would come in a round of its own.  us, 1024 workgroups -> as many as are resident, evenly filled: 20000 x 1024 43.0 -> 38.8, 65536 x 4096 548 -> 516.
// (The forward kernel, and 4-byte elements, were the same or slower so.)
constexpr long long NORM_RESIDENT = 3 * 256;
// Workgroups after which a launch meets the same groups again, at the most
constexpr long long NORM_PERIOD = 65536;
static int norm_config(const hdla_norm_dims* d, bool bwd, NormCfg& c) {
    if (!d) return HDLA_ERR_NULL;
    if (d->dtype != HDLA_BF16 && d->dtype != HDLA_FP32) return HDLA_ERR_DTYPE;
    if (d->weight_dtype != HDLA_BF16 && d->weight_dtype != HDLA_FP32) return HDLA_ERR_DTYPE;
    if (d->gate_pos < 0 || d->gate_pos > 2) return HDLA_ERR_SHAPE;
    if (d->rows < 0 || d->G <= 0 || d->E <= 0 || !(d->eps >= 0.f)) return HDLA_ERR_SHAPE;
    c.n = d->dtype == HDLA_BF16 ? 8 : 4;
    if (d->E % c.n) return HDLA_ERR_SHAPE;                      // groups start on 16-byte boundaries
    const int pieces = d->E / c.n;
    if (pieces > 256 * 8) return HDLA_ERR_SHAPE;                // a group lives in one workgroup's registers
    if (d->rows > (1LL << 40) / d->G) return HDLA_ERR_SHAPE;
    c.nslot = d->rows * d->G;
    // groups of more than two pieces a lane, whose wavefronts would have the registers of few, and of two when there are too few of them
    // to fill the chip one wavefront each (a decode step: a few hundred rows).  us, both passes, one wavefront a group -> four: bf16 65536 x 4096 1000 -> 838,
    // 10000 x 4096 202 -> 135, 20000 x 2048 130 -> 122; fp32 5000 x 2048 81 -> 68, 20000 x 1024 124 -> 115, 30000 x 2048 362 both.
    // (Up to NORM_PERIOD groups: the grid is a multiple of their number then, and of a quarter of it where each wavefront has one.)
    c.wg_row = pieces > 64 * 8 || (pieces > 64 * 2 && d->G <= NORM_PERIOD) || (pieces >= 128 && c.nslot <= 2048);
    if (c.wg_row) {
        // one group per workgroup pass, 256 lanes across it
        c.nv = 1;
        while (c.nv * 256 < pieces) c.nv *= 2;
        c.lpr_log2 = 8; c.rpw = 1; c.wg_reduce = 0;
        c.nsg = c.nslot;
    } else {
        c.nv = 1;
        while (c.nv * 64 < pieces) c.nv *= 2;
        const int per = (pieces + c.nv - 1) / c.nv;
        c.lpr_log2 = 0;
        while ((1 << c.lpr_log2) < per) ++c.lpr_log2;
        c.rpw = 64 >> c.lpr_log2;
        c.nsg = (c.nslot + c.rpw - 1) / c.rpw;
        c.wg_reduce = c.rpw % d->G == 0;
    }
    // a few passes per wavefront to amortise the weight loads, enough workgroups to fill the chip, and, backward, a
    // bound on the partial rows of the weight gradient; then a multiple of what keeps a lane on one weight column
    const long long cap = bwd ? 1024 : 8192, owners = c.wg_row ? 1 : 4;
    const long long per_wave = c.nsg >= 4 * owners * 1024 ? 4 : (c.nsg >= 2 * owners * 1024 ? 2 : 1);
    long long nwg = (c.nsg + owners * per_wave - 1) / (owners * per_wave);
    if (nwg < 1) nwg = 1;
    if (nwg > cap) nwg = cap;
    if (bwd && d->dtype == HDLA_BF16 && c.nv == 2 && nwg > NORM_RESIDENT) {
        const long long passes = (c.nsg + owners * NORM_RESIDENT - 1) / (owners * NORM_RESIDENT);
        nwg = (c.nsg + owners * passes - 1) / (owners * passes);
    }
    const long long m = d->G / gcd_ll(d->G, owners * c.rpw);
    if (m > NORM_PERIOD) return HDLA_ERR_SHAPE;
    c.nwg = (nwg + m - 1) / m * m;
    return HDLA_OK;
}

template <typename T>
static hipError_t launch_norm(const NormArgs& a, const NormCfg& c, bool bwd, hipStream_t s) {
    const dim3 grid((unsigned)c.nwg), block(256);
#define HDLA_NORM_CASE(NVV)                                                                              \
    case NVV:                                                                                            \
        if (bwd) hipLaunchKernelGGL((normalize_bwd_kernel<T, NVV>), grid, block, 0, s, a);               \
        else hipLaunchKernelGGL((normalize_fwd_kernel<T, NVV>), grid, block, 0, s, a);                   \
        break;
    switch (c.nv) {
        HDLA_NORM_CASE(1)
        HDLA_NORM_CASE(2)
        HDLA_NORM_CASE(4)
        HDLA_NORM_CASE(8)
        default: return hipErrorInvalidValue;
    }
#undef HDLA_NORM_CASE
    return hipGetLastError();
}

static NormArgs norm_args(const hdla_norm_dims* d, const NormCfg& c) {
    NormArgs a{};
    a.nslot = c.nslot; a.nsg = c.nsg; a.G = d->G; a.E = d->E; a.lpr_log2 = c.lpr_log2;
    a.w_f32 = d->weight_dtype == HDLA_FP32; a.gate_pos = d->gate_pos; a.wg_reduce = c.wg_reduce; a.wg_row = c.wg_row;
    a.cn = d->c / sqrtf((float)d->E); a.inv_e = 1.f / (float)d->E; a.eps = d->eps;
    return a;
}

static bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace hdla

using namespace hdla;

extern "C" size_t hdla_normalize_workspace_bytes(const hdla_norm_dims* dims) {
    NormCfg c;
    if (norm_config(dims, true, c) != HDLA_OK) return 0;
    return (size_t)c.partial_rows() * dims->E * sizeof(float);
}

extern "C" int hdla_normalize_fwd(const hdla_norm_dims* dims, const void* x, const void* weight, const void* gate,
                                  void* o, void* stream) {
    NormCfg c;
    const int rc = norm_config(dims, false, c);
    if (rc) return rc;
    if (dims->rows == 0) return HDLA_OK;
    if (!x || !o || (dims->gate_pos && !gate)) return HDLA_ERR_NULL;
    if (!al16(x) || !al16(o) || !al16(gate) || !al16(weight)) return HDLA_ERR_ALIGN;
    NormArgs a = norm_args(dims, c);
    a.x = x; a.weight = weight; a.gate = gate; a.o = o;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const hipError_t e = dims->dtype == HDLA_BF16 ? launch_norm<bf16>(a, c, false, s) : launch_norm<float>(a, c, false, s);
    return e == hipSuccess ? HDLA_OK : (int)e;
}

static int normalize_bwd(const hdla_norm_dims* dims, const void* x, const void* weight, const void* gate, const void* d_o, void* dx, void* dgate, void* dw,
                         bool dw_f32, void* workspace, size_t workspace_bytes, hdla_sum* later, void* stream) {
    NormCfg c;
    const int rc = norm_config(dims, true, c);
    if (rc) return rc;
    if (weight && !dw) return HDLA_ERR_NULL;
    if (dims->rows > 0 && (!x || !d_o || !dx || (dims->gate_pos && (!gate || !dgate)))) return HDLA_ERR_NULL;
    if (!al16(x) || !al16(d_o) || !al16(dx) || !al16(gate) || !al16(dgate) || !al16(weight) || !al16(dw))
        return HDLA_ERR_ALIGN;
    const size_t need = weight ? (size_t)c.partial_rows() * dims->E * sizeof(float) : 0;
    if (need && (!workspace || !al16(workspace) || workspace_bytes < need)) return HDLA_ERR_WORKSPACE;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    NormArgs a = norm_args(dims, c);
    a.x = x; a.weight = weight; a.gate = gate; a.d_o = d_o; a.dx = dx; a.dgate = dgate;
    a.partial = static_cast<float*>(workspace);
    if (dims->rows > 0) {
        const hipError_t e = dims->dtype == HDLA_BF16 ? launch_norm<bf16>(a, c, true, s) : launch_norm<float>(a, c, true, s);
        if (e != hipSuccess) return (int)e;
    }
    if (!weight) return later ? sum_now_or_later(SumJob{}, later, s) : HDLA_OK;
    // (dw in 32 bits or in the weight's own 16, rounded once: as a launch of its own that was 4.8 us of a training step of the layer)
    SumJob job{};
    job.kind = SUM_ROWS;
    job.blocks = (int)(((long long)dims->G * dims->E + 15) / 16);
    job.part = a.partial; job.out[0] = dw; job.f32 = dw_f32; job.G = dims->G; job.E = dims->E;
    job.n = dims->rows > 0 ? c.partial_rows() : 0LL;
    return sum_now_or_later(job, later, s);
}
extern "C" int hdla_normalize_bwd(const hdla_norm_dims* dims, const void* x, const void* weight, const void* gate,
                                  const void* d_o, void* dx, void* dgate, float* dw, void* workspace,
                                  size_t workspace_bytes, void* stream) {
    return normalize_bwd(dims, x, weight, gate, d_o, dx, dgate, dw, true, workspace, workspace_bytes, nullptr, stream);
}
extern "C" int hdla_normalize_bwd_as(const hdla_norm_dims* dims, const void* x, const void* weight, const void* gate, const void* d_o, void* dx,
                                     void* dgate, void* dw, void* workspace, size_t workspace_bytes, void* stream) {
    return normalize_bwd(dims, x, weight, gate, d_o, dx, dgate, dw, !dims || dims->weight_dtype == HDLA_FP32, workspace, workspace_bytes, nullptr, stream);
}
extern "C" int hdla_normalize_bwd_later(const hdla_norm_dims* dims, const void* x, const void* weight, const void* gate, const void* d_o, void* dx,
                                        void* dgate, void* dw, void* workspace, size_t workspace_bytes, hdla_sum* sum, void* stream) {
    if (!sum) return HDLA_ERR_NULL;
    return normalize_bwd(dims, x, weight, gate, d_o, dx, dgate, dw, !dims || dims->weight_dtype == HDLA_FP32, workspace, workspace_bytes, sum, stream);
}
