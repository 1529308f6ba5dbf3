// Fused token-serial recurrent kernel (decode step and short prefills).
//
// Replaces HRDPLR/recurrent.py:26-119.  Per token
//     S <- Diag(exp(g)) S + sum_r b_r (a_r^T S) + k v^T ,   o = scale * S^T q
// with both rank terms reading the state before the decay (recurrent.py:93-100) and the output reading the
// updated state (recurrent.py:104).  For a decode step the kernel is a pure stream of the fp32 state through
// HBM (read K*V*4 bytes, write K*V*4 bytes per head), so the layout is chosen for that: one 256-thread
// workgroup owns a K x 64 column block of one head's state, every lane moves 16-byte pieces of whole 256-byte
// row segments, and all of a block's loads are in flight before the first use.  The two reductions over K
// (a^T S and q^T S) run as in-lane partial sums, two cross-lane butterfly steps and one LDS exchange between
// the four wavefronts: one barrier a token, since the next token's values are put in place and the last one's output is
// summed up beside the work of this one.
//
// What bounds it: the state's way from and to HBM (256 sequences of 32 heads, K = V = 128, one token: 1.09 GB), and where the state is
// in a cache the chain of a token: its values, the LDS fill, two reductions.
// Figures: us a call on the device, calls in a row in one process; the largest one's depends on where its two states of 0.5 GB lie
// (193 to 196 with one pair of buffers, 186 with fresh outputs from a graph's pool, 202 for a launch that waits for the last one).
//   - A token's values are requested before the previous token's arithmetic, the first token's before the state: requests complete in
//     order, so behind the state they would be waited for as long.
//   - The column blocks of a head are neighbours in launch order: they are in flight together and memory sees whole rows.  As the second
//     dimension of the grid they ran thousands of workgroups apart.  Below 256 workgroups that order is kept: there the blocks of a head meet
//     in the same L2 where the number of heads is a multiple of 8, and the token's values are what is waited for (4 sequences of 16 heads with
//     beta 5.2 against 5.5).
//     Both together, against values requested at the token's begin and blocks apart: 256 sequences of 32 heads, 128 x 128, one token 199.6 -> 193.2
//     (204 -> 186 with fresh outputs), 128 of 32 104.2 -> 91.7, 64 of 32 51.7 -> 46.0, 24 of 16 9.5 -> 8.2, 16 of 16 7.5 -> 7.0; 4 of 8, 16 tokens
//     34.1 -> 29.8; 8 of 16, 64 x 64, 8 tokens 15.1 -> 12.9; 4 of 16, 128 x 128, one token 4.9 -> 5.1 (a graph's replay).
//   - One barrier a token instead of four (five in HD mode), a thread's channels read 16 bytes at a time, sums over lanes without LDS: 64 of 16 with
//     beta, 64 x 64, 8 tokens 25.3 -> 21.3; 8 of 16, 128 x 128, 8 tokens 18.3 -> 14.9; 1 of 16, 64 x 64, 8 tokens 12.5 -> 10.7; 128 of 16, 128 x 128,
//     6 tokens 83 -> 77; one token: 51 of 16 with beta, 128 x 128, 19.2 -> 18.6, 256 of 32 as before.
//   - Tried, where this form took the 186: the blocks of a head on one XCD 195 to 199; no branch around the state's loads instead of one
//     (94 registers a lane at K = 128 and five waves a SIMD, not 110 and four) 192; all 128 columns in one workgroup 196.  Held to five waves it spills.
//
// HD mode (p.beta given) forms the rank terms of the HDLA layer per token from (beta, k, gk) instead of reading
// them (HRDPLR/hdla_custom.py:19-43): with f = exp(gk) and s = sum_c k_c^2 f_c,
//     a_1 = -beta k,  a_2 = beta k (beta s - f),  b_1 = f k,  b_2 = k,
// each rounded to the input type as the stored tensors would be.
#include "hdla_common.cuh"
#include "hdla_launch.h"

namespace hdla {

__device__ __forceinline__ float as_float(bf16 x) { return bf2f(x.x); }
__device__ __forceinline__ float as_float(float x) { return x; }
__device__ __forceinline__ float round_as(const bf16*, float x) { return bf2f(f2bf(x)); }
__device__ __forceinline__ float round_as(const float*, float x) { return x; }

// A token's values for one thread (channel tid; value column tid - 192) as they lie in memory: converted where they are used.  A conversion
// beside a load is a wait for it in the conditional block that the load stands in.
template <typename T, bool HD, int MORE>
struct TokenValues {
    T q, k, v, b0;       // b0: beta with HD
    T a0, a1, b1;        // without HD
    T km[MORE];          // with HD and K > 64: k and the decay of the other wavefronts' channels, tid's place in each
    uint32_t gk, gm[MORE];    // the bits, fp32's or in the low half bf16's
};

template <typename T, int K, int V, int BV, bool HD>
__global__ __launch_bounds__(256) void recurrent_kernel(RecurrentArgs<T> p) {
    constexpr int CG = BV / 4;        // lanes across a row segment (float4 each)
    constexpr int RG = 256 / CG;      // row groups
    constexpr int RPT = K / RG;       // state rows per thread
    constexpr int NF = K / 64;        // wavefronts that fill, one channel a lane
    static_assert(K % RG == 0 && RPT % 4 == 0 && BV == 64, "tile shape");
    static_assert(K <= 256, "one channel per thread in the per-token fill");
    // A token's channels in LDS lie so that the rows of a thread, rg + RG j, are neighbours: 16-byte reads
    enum { Q, KK, EG, A0, A1, B0, B1, NA };
    __shared__ __attribute__((aligned(16))) float st[3][NA][K];
    __shared__ __attribute__((aligned(16))) float sv[3][BV], red[2][4][2][BV], redo[2][4][BV];

    constexpr int NV = V / BV;
    const bool apart = NV > 1 && gridDim.y > 1;
    const int nh = apart ? blockIdx.x : blockIdx.x / NV, vb = apart ? blockIdx.y : blockIdx.x % NV;
    const int n = nh / p.H, h = nh - n * p.H;
    const int H = p.H;
    const int tid = threadIdx.x, cg = tid % CG, rg = tid / CG, wave = tid >> 6, lane = tid & 63;
    int64_t bos, eos;
    if (p.cu) packed_bounds(p.cu, n, p.T_, bos, eos);
    else { bos = (int64_t)n * p.T_; eos = bos + p.T_; }
    const int len = (int)(eos - bos);

    constexpr int MORE = HD && NF > 1 ? NF : 1;
    auto request = [&](int64_t t) __attribute__((always_inline)) {
        TokenValues<T, HD, MORE> x{};
        auto decay = [&](int64_t off) __attribute__((always_inline)) {
            return p.gk_f32 ? reinterpret_cast<const uint32_t*>(p.gk)[off] : (uint32_t)reinterpret_cast<const uint16_t*>(p.gk)[off];
        };
        if (tid < K) {
            const int64_t off = (t * H + h) * K + tid;
            x.q = p.q[off];
            x.k = p.k[off];
            x.gk = decay(off);
            if constexpr (HD) {
                x.b0 = p.beta[t * H + h];
                if constexpr (NF > 1) {
#pragma unroll
                    for (int i = 0; i < NF; ++i) {
                        x.km[i] = p.k[off - tid + 64 * i + lane];
                        x.gm[i] = decay(off - tid + 64 * i + lane);
                    }
                }
            } else {
                const int64_t off0 = ((t * RANK + 0) * H + h) * K + tid, off1 = ((t * RANK + 1) * H + h) * K + tid;
                x.a0 = p.a[off0];
                x.a1 = p.a[off1];
                x.b0 = p.b[off0];
                x.b1 = p.b[off1];
            }
        }
        if (tid >= 192) x.v = p.v[(t * H + h) * V + vb * BV + tid - 192];
        return x;
    };
    auto fill = [&](const TokenValues<T, HD, MORE>& x, int buf) __attribute__((always_inline)) {
        auto factor = [&](uint32_t g) __attribute__((always_inline)) { return exp_t<T>(p.gk_f32 ? __builtin_bit_cast(float, g) : bf2f((uint16_t)g)); };
        if (tid < K) {
            float (*to)[K] = st[buf];
            const int at = (tid % RG) * RPT + tid / RG;
            const float kk = as_float(x.k), f = factor(x.gk);
            to[Q][at] = as_float(x.q) * p.scale;
            to[KK][at] = kk;
            to[EG][at] = f;
            if constexpr (HD) {
                float s = 0.f;
                if constexpr (NF == 1) s = sum_lanes(kk * kk * f, 64);
                else {
                    // every wavefront that fills forms all the sums: no barrier between them
#pragma unroll
                    for (int i = 0; i < NF; ++i) {
                        const float ki = as_float(x.km[i]);
                        s += sum_lanes(ki * ki * factor(x.gm[i]), 64);
                    }
                }
                const float beta = as_float(x.b0);
                to[A0][at] = round_as(p.k, -beta * kk);
                to[A1][at] = round_as(p.k, (beta * s - f) * beta * kk);
                to[B0][at] = round_as(p.k, f * kk);
                to[B1][at] = kk;
            } else {
                to[A0][at] = as_float(x.a0);
                to[A1][at] = as_float(x.a1);
                to[B0][at] = as_float(x.b0);
                to[B1][at] = as_float(x.b1);
            }
        }
        if (tid >= 192) sv[buf][tid - 192] = as_float(x.v);
    };
    auto token = [&](int step) __attribute__((always_inline)) { return p.reverse ? eos - 1 - step : bos + step; };
    TokenValues<T, HD, MORE> raw{};
    if (len > 0) raw = request(token(0));
    const int64_t sbase = (int64_t)nh * K * V + vb * BV + 4 * cg;
    f32x4 S[RPT];
    if (p.h0) {
#pragma unroll
        for (int j = 0; j < RPT; ++j) S[j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.h0 + sbase + (int64_t)(rg + RG * j) * V));
    } else {
#pragma unroll
        for (int j = 0; j < RPT; ++j) S[j] = zero4();
    }
    // the output of a token is complete a barrier after its own: one wavefront's work
    auto output = [&](int step) __attribute__((always_inline)) {
        if (wave != 2) return;
        const float (*r)[BV] = redo[step & 1];
        st_elem(p.o + (token(step) * H + h) * V + vb * BV + lane, r[0][lane] + r[1][lane] + r[2][lane] + r[3][lane]);
    };
    if (len > 0) {
        fill(raw, 0);
        if (len > 1) raw = request(token(1));
    }
    __syncthreads();
    // One barrier a token.  In front of it the parts of a^T S are written and the next token's values: into the third place, since a wavefront may
    // still read the token before this one's in the second.  The parts have two places each.
    for (int step = 0, now = 0; step < len; ++step) {
        const int next = now == 2 ? 0 : now + 1;
        const float (*const x)[K] = st[now];
        auto rows = [&](int which, int j) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(&x[which][rg * RPT + j]); };

        // a_r^T S over the block's rows
        f32x4 p0 = zero4(), p1 = zero4();
#pragma unroll
        for (int j = 0; j < RPT; j += 4) {
            const f32x4 a0 = rows(A0, j), a1 = rows(A1, j);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p0 += S[j + i] * a0[i];
                p1 += S[j + i] * a1[i];
            }
        }
        sum_rows<CG>(p0);
        sum_rows<CG>(p1);
        float (*const r)[2][BV] = red[step & 1];
        if (lane < CG) {
            *reinterpret_cast<f32x4*>(&r[wave][0][4 * cg]) = p0;
            *reinterpret_cast<f32x4*>(&r[wave][1][4 * cg]) = p1;
        }
        if (step + 1 < len) {
            fill(raw, next);
            if (step + 2 < len) raw = request(token(step + 2));
        }
        __syncthreads();
        if (step > 0) output(step - 1);
        f32x4 u0 = zero4(), u1 = zero4();
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            u0 += *reinterpret_cast<const f32x4*>(&r[w][0][4 * cg]);
            u1 += *reinterpret_cast<const f32x4*>(&r[w][1][4 * cg]);
        }
        const f32x4 v4 = *reinterpret_cast<const f32x4*>(&sv[now][4 * cg]);
        f32x4 po = zero4();
#pragma unroll
        for (int j = 0; j < RPT; j += 4) {
            const f32x4 eg = rows(EG, j), b0 = rows(B0, j), b1 = rows(B1, j), kk = rows(KK, j), q = rows(Q, j);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                S[j + i] = S[j + i] * eg[i] + u0 * b0[i] + u1 * b1[i] + v4 * kk[i];
                po += S[j + i] * q[i];
            }
        }
        sum_rows<CG>(po);
        if (lane < CG) *reinterpret_cast<f32x4*>(&redo[step & 1][wave][4 * cg]) = po;
        now = next;
    }
    if (p.ht) {
#pragma unroll
        for (int j = 0; j < RPT; ++j)
            __builtin_nontemporal_store(S[j], reinterpret_cast<f32x4*>(p.ht + sbase + (int64_t)(rg + RG * j) * V));
    }
    if (len > 0) {
        __syncthreads();
        output(len - 1);
    }
}

template <typename T, int K, int V>
static hipError_t launch_recurrent_kv(const RecurrentArgs<T>& a, hipStream_t stream) {
    constexpr int BV = 64;
    // A head's column blocks next to each other in launch order, except on grids that do not give every CU a workgroup (and where
    // the grid would reach 2^32 threads).  See above.
    const int64_t blocks = (int64_t)a.N * a.H * (V / BV);
    const bool apart = blocks < 256 || blocks >= (1 << 24);
    dim3 grid = apart ? dim3(a.N * a.H, V / BV) : dim3((unsigned)blocks), block(256);
    if (a.beta) hipLaunchKernelGGL((recurrent_kernel<T, K, V, BV, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((recurrent_kernel<T, K, V, BV, false>), grid, block, 0, stream, a);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_recurrent(const RecurrentArgs<T>& a, int K, int V, hipStream_t stream) {
    if (K == 64 && V == 64) return launch_recurrent_kv<T, 64, 64>(a, stream);
    if (K == 128 && V == 128) return launch_recurrent_kv<T, 128, 128>(a, stream);
    if (K == 64 && V == 128) return launch_recurrent_kv<T, 64, 128>(a, stream);
    if (K == 128 && V == 64) return launch_recurrent_kv<T, 128, 64>(a, stream);
    // head sizes up to 256 (the reference's token-serial kernel takes any K, HRDPLR/recurrent.py:155-176): the state
    // block of a workgroup is K x 64 values in registers, 64 per lane at K = 256
    if (K == 256 && V == 256) return launch_recurrent_kv<T, 256, 256>(a, stream);
    if (K == 256 && V == 128) return launch_recurrent_kv<T, 256, 128>(a, stream);
    if (K == 128 && V == 256) return launch_recurrent_kv<T, 128, 256>(a, stream);
    if (K == 256 && V == 64) return launch_recurrent_kv<T, 256, 64>(a, stream);
    if (K == 64 && V == 256) return launch_recurrent_kv<T, 64, 256>(a, stream);
    return hipErrorInvalidValue;
}
template hipError_t launch_recurrent<bf16>(const RecurrentArgs<bf16>&, int, int, hipStream_t);
template hipError_t launch_recurrent<float>(const RecurrentArgs<float>&, int, int, hipStream_t);

}  // namespace hdla
