// A few tokens of the HDLA layer between its projections, states carried (HRDPLR/hdla_custom.py:221-251, 19-43 and 341-345 around
// HRDPLR/recurrent.py:26-119): what layer_pre_fwd_kernel, recurrent_kernel in its HD mode and, where the norm has a group a head,
// normalize_fwd_kernel do one after the other, in one launch; for one token (UP) layer_up_kernel's work too.  Every value that those
// kernels hand on through memory (q, k, v, beta, f, the decay, the gate, the rank terms, o) is rounded to bf16 where it was stored.
//
// A workgroup owns one (sequence, head): 4 D threads, a float4 of every 16th row of the state in registers.  For one token it
// is a stream of the state, 64 KiB each way at D = 128, so everything the token needs is requested first, the state behind it
// (requests complete in order: the other way round the token's values would wait for the state), and the state arrives while
// the values are formed.  Per token six barriers; q, k, v and the decay are formed side by side, a quarter of the threads each.
// The two D x D products of UP are 2 x 32 KiB of weights a workgroup, from L2, 16 lanes a row.
//
// What it is for: a decode step is bound by its launches, 3 to 4 us of host time each (figures at layer_step in native.cpp).
#include "hdla_common.cuh"
#include "../../include/hdla_hip.h"

#include <type_traits>

namespace hdla {

// what becomes of o: it is stored as it is, gated and normalised, or gated in fp32 with its head's part of the sum of squares
enum StepNorm { NORM_NOT, NORM_HERE, NORM_LATER };
struct StepArgs {
    const bf16 *y, *log_f;                // [rows, ldy]; [rows, H, D] (not UP)
    bf16* gate;                           // [rows, H, D]: read, or (UP, null if nobody wants it) written
    const bf16 *wf, *wg;                  // UP: [H D, D] x 2, of the decay and of the gate
    const void* weight;                   // [H, D] of the norm, or null
    const float* h0;                      // [N, H, D, D], or null
    bf16* o;                              // [rows, H, D] (not where the norm is left to the projection)
    float *gated, *sums;                  // NORM_LATER: [rows, H, D] o sigmoid(gate), [rows, H] sums of squares
    float* ht;                            // [N, H, D, D], or null
    int T, H, ldy, cq, ck, cv, cb, cf, cg;
    int norm_q, norm_k, norm_v, w_f32, norm, gate_pre;
    float beta_scale, eps_d, scale, cn, inv_e, eps;
};

__device__ __forceinline__ float step_sigmoid(float x) {
    float e[1] = {__expf(-x)}, s[1];
    sigmoid_of_exp<1>(e, s);
    return s[0];
}
__device__ __forceinline__ float as_bf16(float x) { return bf2f(f2bf(x)); }
__device__ __forceinline__ float wave_sum(float x) { return sum_lanes(x, 64); }

// the sum over 16 lanes side by side, on all of them
__device__ __forceinline__ float row_sum(float x) {
    auto ror = [](float v, auto n) __attribute__((always_inline)) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + decltype(n)::value, 0xf, 0xf, false));
    };
    x += ror(x, std::integral_constant<int, 8>{});
    x += ror(x, std::integral_constant<int, 4>{});
    x += ror(x, std::integral_constant<int, 2>{});
    x += ror(x, std::integral_constant<int, 1>{});
    return x;
}
// log(sigmoid(x)) as layer_up_kernel forms it
__device__ __forceinline__ float step_logsig(float x) {
    const float e = __expf(-fabsf(x));
    return fminf(x, 0.f) - (e < 1e-4f ? e : __logf(1.f + e));
}

template <int D, bool UP>
__global__ __launch_bounds__(4 * D, 4) void layer_step_kernel(StepArgs p) {
    constexpr int NW = D / 16;            // wavefronts
    constexpr int CG = D / 4;             // lanes across a row of the state
    constexpr int RG = 16, RPT = D / RG;  // row groups, rows a thread
    constexpr int WPR = D / 64;           // wavefronts of a quarter of the threads
    __shared__ float sq[D], sk[D], sf[D], sv[D], sa[2][D], sb[D], part[2][NW], up[2][D];
    __shared__ __attribute__((aligned(16))) float red[NW][3][D];
    const int n = blockIdx.x / p.H, h = blockIdx.x - n * p.H;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int role = wave / WPR, ch = tid & (D - 1);      // 0 q, 1 k, 2 v, 3 decay
    const int cg = tid & (CG - 1), rg = tid / CG;
    const int col = (role == 0 ? p.cq : role == 1 ? p.ck : p.cv) + h * D + ch;

    // a token's values as they come from memory
    struct Raw { bf16 x, beta; uint32_t gate; };
    auto request = [&](int64_t t) __attribute__((always_inline)) {
        Raw r;
        r.x = !UP && role == 3 ? p.log_f[(t * p.H + h) * D + ch] : p.y[t * p.ldy + col];
        r.beta = p.y[t * p.ldy + p.cb + h];
        r.gate = 0;
        if (!UP && p.norm) {
            const bf16* g = p.gate + (t * p.H + h) * D + WPR * lane;   // wave 0's: the channels whose o it forms
            if constexpr (WPR == 2) r.gate = *reinterpret_cast<const uint32_t*>(g);
            else r.gate = g->x;
        }
        return r;
    };
    const int64_t t0 = (int64_t)n * p.T;
    Raw next = request(t0);
    float w[WPR];
#pragma unroll
    for (int i = 0; i < WPR; ++i) {
        const int at = h * D + WPR * lane + i;
        w[i] = p.norm != NORM_HERE || !p.weight ? 1.f : p.w_f32 ? static_cast<const float*>(p.weight)[at] : bf2f(static_cast<const bf16*>(p.weight)[at].x);
    }
    // UP: 16 lanes a row of the weights, D / 16 elements a lane, D / 4 rows at a time
    constexpr int EL = D / 16;
    typedef short Row __attribute__((ext_vector_type(EL)));
    Row in[2], wr[2][4];
    const int sub = tid & 15, urow = tid >> 4;
    if constexpr (UP) {
        in[0] = *reinterpret_cast<const Row*>(p.y + t0 * p.ldy + p.cf + EL * sub);
        in[1] = *reinterpret_cast<const Row*>(p.y + t0 * p.ldy + p.cg + EL * sub);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t at = ((int64_t)h * D + urow + D / 4 * j) * D + EL * sub;
            wr[0][j] = *reinterpret_cast<const Row*>(p.wf + at);
            wr[1][j] = *reinterpret_cast<const Row*>(p.wg + at);
        }
    }
    const int64_t sbase = (int64_t)blockIdx.x * D * D + 4 * cg;
    f32x4 S[RPT];
#pragma unroll
    for (int j = 0; j < RPT; ++j)
        S[j] = p.h0 ? __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.h0 + sbase + (rg + RG * j) * D)) : zero4();

    for (int step = 0; step < p.T; ++step) {
        const int64_t t = t0 + step;
        const Raw now = next;
        if (step + 1 < p.T) next = request(t + 1);
        // q, k, v: silu and norm; the decay: exp
        float x = bf2f(now.x.x);
        if (role != 3) {
            x *= step_sigmoid(x);
            const float ss = wave_sum(x * x);
            if (lane == 0) part[0][wave] = ss;
        }
        if constexpr (UP) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    float s = 0.f;
#pragma unroll
                    for (int e = 0; e < EL; ++e) s += bf2f((uint16_t)in[i][e]) * bf2f((uint16_t)wr[i][j][e]);
                    s = as_bf16(row_sum(s));
                    if (i == 0) s = as_bf16(step_logsig(s));
                    if (sub == 0) up[i][urow + D / 4 * j] = s;
                }
        }
        __syncthreads();
        if (role == 3) {
            x = exp_t<bf16>(UP ? up[0][ch] : x);
            if (UP && p.gate) st_elem(p.gate + (t * p.H + h) * D + ch, up[1][ch]);
        } else {
            float s = part[0][role * WPR];
            if constexpr (WPR == 2) s += part[0][role * WPR + 1];
            if (role == 0 ? p.norm_q : role == 1 ? p.norm_k : p.norm_v) x *= 1.f / sqrtf(s + p.eps_d);
            x = as_bf16(x);
        }
        if (role == 0) sq[ch] = x * p.scale;
        else if (role == 1) sk[ch] = x;
        else if (role == 2) sv[ch] = x;
        else sf[ch] = x;
        __syncthreads();
        // the rank terms: a_1 = -beta k, a_2 = beta k (beta s - f), b_1 = f k, b_2 = k with s = sum k^2 f
        const float f = sf[ch];
        if (role == 1) {
            const float s = wave_sum(x * x * f);
            if (lane == 0) part[1][wave] = s;
        }
        __syncthreads();
        if (role == 1) {
            float s = part[1][WPR];
            if constexpr (WPR == 2) s += part[1][WPR + 1];
            const float beta = as_bf16(p.beta_scale * step_sigmoid(bf2f(now.beta.x)));
            sa[0][ch] = as_bf16(-beta * x);
            sa[1][ch] = as_bf16((beta * s - f) * beta * x);
            sb[ch] = as_bf16(f * x);
        }
        __syncthreads();

        // a_r^T S over the rows
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
        for (int i = 0; i < NW; ++i) {
            u0 += *reinterpret_cast<const f32x4*>(&red[i][0][4 * cg]);
            u1 += *reinterpret_cast<const f32x4*>(&red[i][1][4 * cg]);
        }
        const f32x4 v4 = *reinterpret_cast<const f32x4*>(&sv[4 * cg]);
        f32x4 po = zero4();
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int row = rg + RG * j;
            S[j] = S[j] * sf[row] + u0 * sb[row] + u1 * sk[row] + v4 * sk[row];
            po += S[j] * sq[row];
        }
        sum_rows<CG>(po);
        if (lane < CG) *reinterpret_cast<f32x4*>(&red[wave][2][4 * cg]) = po;
        __syncthreads();
        // o of the head, its gate and norm, by one wavefront (the others go on: what it reads here is written again behind the
        // barriers of the next token)
        if (wave == 0) {
            float o[WPR], gs[WPR], sum = 0.f;
#pragma unroll
            for (int i = 0; i < WPR; ++i) {
                o[i] = 0.f;
#pragma unroll
                for (int k = 0; k < NW; ++k) o[i] += red[k][2][WPR * lane + i];
                o[i] = as_bf16(o[i]);
                gs[i] = step_sigmoid(UP ? up[1][WPR * lane + i] : bf2f((uint16_t)(now.gate >> (16 * i))));
                if (p.norm == NORM_HERE && p.gate_pre) o[i] *= gs[i];
                const float x = p.norm == NORM_LATER && p.gate_pre ? o[i] * gs[i] : o[i];
                sum += x * x;
            }
            if (p.norm == NORM_LATER) {
                sum = wave_sum(sum);
                if (lane == 0) p.sums[t * p.H + h] = sum;
#pragma unroll
                for (int i = 0; i < WPR; ++i) p.gated[(t * p.H + h) * D + WPR * lane + i] = o[i] * gs[i];
                continue;
            }
            const float rs = p.cn / sqrtf(wave_sum(sum) * p.inv_e + p.eps);
#pragma unroll
            for (int i = 0; i < WPR; ++i) {
                if (p.norm == NORM_HERE) {
                    o[i] = o[i] * rs * w[i];
                    if (!p.gate_pre) o[i] *= gs[i];
                }
                st_elem(p.o + (t * p.H + h) * D + WPR * lane + i, o[i]);
            }
        }
    }
    if (p.ht) {
#pragma unroll
        for (int j = 0; j < RPT; ++j)
            __builtin_nontemporal_store(S[j], reinterpret_cast<f32x4*>(p.ht + sbase + (rg + RG * j) * D));
    }
}

static bool step_al(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace hdla

using namespace hdla;

extern "C" int hdla_layer_step(const hdla_pre_dims* pre, const hdla_up_dims* up, const hdla_norm_dims* norm, int32_t T, const void* y,
                               const void* wf, const void* wg, const void* log_f, void* gate, const void* weight, const float* h0, void* o,
                               float* gated, float* ht, void* stream) {
    if (!pre) return HDLA_ERR_NULL;
    if (pre->dtype != HDLA_BF16) return HDLA_ERR_DTYPE;
    const long long rows = pre->rows, H = pre->H, D = pre->D;
    if (rows < 0 || H <= 0 || (D != 64 && D != 128) || T < 1 || rows % T || !(pre->eps >= 0.f)) return HDLA_ERR_SHAPE;
    for (long long c : {pre->col_q, pre->col_k, pre->col_v}) if (c < 0 || c + H * D > pre->ldy) return HDLA_ERR_SHAPE;
    if (pre->col_beta < 0 || pre->col_beta + H > pre->ldy) return HDLA_ERR_SHAPE;
    if (rows / T > 0x7fffffffLL / H) return HDLA_ERR_SHAPE;
    if (up) {
        if (T != 1 || up->rows != rows || up->D != D || up->d != H * D || up->ld != pre->ldy) return HDLA_ERR_SHAPE;
        for (long long c : {up->col_f, up->col_g}) if (c < 0 || c + D > up->ld) return HDLA_ERR_SHAPE;
        if (up->col_f % 8 || up->col_g % 8 || up->ld % 8) return HDLA_ERR_ALIGN;
    }
    if (norm) {
        if (norm->dtype != HDLA_BF16 || (weight && norm->weight_dtype != HDLA_BF16 && norm->weight_dtype != HDLA_FP32)) return HDLA_ERR_DTYPE;
        if (norm->rows != rows || norm->G != (gated ? 1 : H) || norm->E != (gated ? H * D : D) || (norm->gate_pos != 1 && norm->gate_pos != 2) || !(norm->eps >= 0.f))
            return HDLA_ERR_SHAPE;
    }
    if (gated && !norm) return HDLA_ERR_NULL;
    if (rows == 0) return HDLA_OK;
    if (!y || (!o && !gated) || (up ? !wf || !wg : !log_f || (norm && !gate))) return HDLA_ERR_NULL;
    for (const void* p : {y, wf, wg, log_f, (const void*)gate, weight, (const void*)h0, (const void*)o, (const void*)gated, (const void*)ht})
        if (!step_al(p)) return HDLA_ERR_ALIGN;
    StepArgs a{};
    a.y = static_cast<const bf16*>(y); a.log_f = static_cast<const bf16*>(log_f); a.gate = static_cast<bf16*>(gate);
    a.wf = static_cast<const bf16*>(wf); a.wg = static_cast<const bf16*>(wg);
    a.weight = weight; a.h0 = h0; a.o = static_cast<bf16*>(o); a.ht = ht;
    a.T = T; a.H = (int)H; a.ldy = pre->ldy; a.cq = pre->col_q; a.ck = pre->col_k; a.cv = pre->col_v; a.cb = pre->col_beta;
    if (up) { a.cf = up->col_f; a.cg = up->col_g; }
    a.norm_q = pre->norm_q; a.norm_k = pre->norm_k; a.norm_v = pre->norm_v;
    a.beta_scale = pre->beta_scale; a.eps_d = pre->eps * (float)D; a.scale = 1.f;
    if (norm) {
        a.norm = gated ? NORM_LATER : NORM_HERE; a.gated = gated; a.sums = gated + rows * H * D;
        a.w_f32 = norm->weight_dtype == HDLA_FP32; a.gate_pre = norm->gate_pos == 1;
        a.cn = norm->c / sqrtf((float)norm->E); a.inv_e = 1.f / (float)norm->E; a.eps = norm->eps;
    }
    const dim3 grid((unsigned)(rows / T * H)), block((unsigned)(4 * D));
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (D == 64) {
        if (up) hipLaunchKernelGGL((layer_step_kernel<64, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((layer_step_kernel<64, false>), grid, block, 0, s, a);
    } else {
        if (up) hipLaunchKernelGGL((layer_step_kernel<128, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((layer_step_kernel<128, false>), grid, block, 0, s, a);
    }
    return (int)hipGetLastError();
}
