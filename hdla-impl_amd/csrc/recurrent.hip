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
// the four wavefronts.
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
//   - Tried, where this form took the 186: the blocks of a head on one XCD 195 to 199; no branch around the state's loads instead of one
//     (94 registers a lane at K = 128 and five waves a SIMD, not 108 and four) 192; all 128 columns in one workgroup 196.  Held to five waves it spills.
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

// A token's values for one thread (channel tid, value column tid) as they lie in memory: converted where they are used.  A conversion
// beside a load is a wait for it in the conditional block that the load stands in.
template <typename T, bool HD>
struct TokenValues {
    T q, k, v, b0;       // b0: beta with HD
    T a0, a1, b1;        // without HD
    uint32_t gk;         // the bits, fp32's or in the low half bf16's
};

template <typename T, int K, int V, int BV, bool HD>
__global__ __launch_bounds__(256) void recurrent_kernel(RecurrentArgs<T> p) {
    constexpr int CG = BV / 4;        // lanes across a row segment (float4 each)
    constexpr int RG = 256 / CG;      // row groups
    constexpr int RPT = K / RG;       // state rows per thread
    static_assert(K % RG == 0 && RPT >= 1, "tile shape");
    static_assert(K <= 256, "one channel per thread in the per-token fill");
    __shared__ float sq[K], sk[K], seg[K], sa[2][K], sb[2][K], sv[BV];
    __shared__ float red[4][3][BV];

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

    auto request = [&](int64_t t) __attribute__((always_inline)) {
        TokenValues<T, HD> x{};
        if (tid < K) {
            const int64_t off = (t * H + h) * K + tid;
            x.q = p.q[off];
            x.k = p.k[off];
            x.gk = p.gk_f32 ? reinterpret_cast<const uint32_t*>(p.gk)[off] : reinterpret_cast<const uint16_t*>(p.gk)[off];
            if constexpr (HD) {
                x.b0 = p.beta[t * H + h];
            } else {
                const int64_t off0 = ((t * RANK + 0) * H + h) * K + tid, off1 = ((t * RANK + 1) * H + h) * K + tid;
                x.a0 = p.a[off0];
                x.a1 = p.a[off1];
                x.b0 = p.b[off0];
                x.b1 = p.b[off1];
            }
        }
        if (tid < BV) x.v = p.v[(t * H + h) * V + vb * BV + tid];
        return x;
    };
    TokenValues<T, HD> raw{};
    if (len > 0) raw = request(p.reverse ? eos - 1 : bos);
    const int64_t sbase = (int64_t)nh * K * V + vb * BV + 4 * cg;
    f32x4 S[RPT];
    if (p.h0) {
#pragma unroll
        for (int j = 0; j < RPT; ++j) S[j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.h0 + sbase + (int64_t)(rg + RG * j) * V));
    } else {
#pragma unroll
        for (int j = 0; j < RPT; ++j) S[j] = zero4();
    }

    for (int step = 0; step < len; ++step) {
        const int64_t t = p.reverse ? (eos - 1 - step) : (bos + step);
        __syncthreads();
        const float kk = as_float(raw.k), f = exp_t<T>(p.gk_f32 ? __builtin_bit_cast(float, raw.gk) : bf2f((uint16_t)raw.gk));
        if constexpr (HD) {
            const float part = sum_lanes(tid < K ? kk * kk * f : 0.f, 64);
            if (lane == 0) red[wave][0][0] = part;
            __syncthreads();
        }
        if (tid < K) {
            sq[tid] = as_float(raw.q) * p.scale;
            sk[tid] = kk;
            seg[tid] = f;
            if constexpr (HD) {
                const float s = red[0][0][0] + red[1][0][0] + red[2][0][0] + red[3][0][0];
                const float beta = as_float(raw.b0);
                sa[0][tid] = round_as(p.k, -beta * kk);
                sa[1][tid] = round_as(p.k, (beta * s - f) * beta * kk);
                sb[0][tid] = round_as(p.k, f * kk);
                sb[1][tid] = kk;
            } else {
                sa[0][tid] = as_float(raw.a0);
                sa[1][tid] = as_float(raw.a1);
                sb[0][tid] = as_float(raw.b0);
                sb[1][tid] = as_float(raw.b1);
            }
        }
        if (tid < BV) sv[tid] = as_float(raw.v);
        __syncthreads();
        if (step + 1 < len) raw = request(p.reverse ? t - 1 : t + 1);

        // a_r^T S over the block's rows
        f32x4 p0 = zero4(), p1 = zero4();
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int row = rg + RG * j;
            p0 += S[j] * sa[0][row];
            p1 += S[j] * sa[1][row];
        }
        sum_rows<CG>(p0);
        sum_rows<CG>(p1);
        if (lane < CG) {
            *reinterpret_cast<f32x4*>(&red[wave][0][4 * cg]) = p0;
            *reinterpret_cast<f32x4*>(&red[wave][1][4 * cg]) = p1;
        }
        __syncthreads();
        f32x4 u0 = zero4(), u1 = zero4();
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            u0 += *reinterpret_cast<const f32x4*>(&red[w][0][4 * cg]);
            u1 += *reinterpret_cast<const f32x4*>(&red[w][1][4 * cg]);
        }
        const f32x4 v4 = *reinterpret_cast<const f32x4*>(&sv[4 * cg]);
        f32x4 po = zero4();
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int row = rg + RG * j;
            S[j] = S[j] * seg[row] + u0 * sb[0][row] + u1 * sb[1][row] + v4 * sk[row];
            po += S[j] * sq[row];
        }
        sum_rows<CG>(po);
        if (lane < CG) *reinterpret_cast<f32x4*>(&red[wave][2][4 * cg]) = po;
        __syncthreads();
        if (tid < BV) {
            const float o = red[0][2][tid] + red[1][2][tid] + red[2][2][tid] + red[3][2][tid];
            st_elem(p.o + (t * H + h) * V + vb * BV + tid, o);
        }
    }
    if (p.ht) {
#pragma unroll
        for (int j = 0; j < RPT; ++j)
            __builtin_nontemporal_store(S[j], reinterpret_cast<f32x4*>(p.ht + sbase + (int64_t)(rg + RG * j) * V));
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
