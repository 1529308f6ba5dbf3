// chunk_grad kernel: everything of the backward pass that is local to one 16-token chunk.
//
// One workgroup of four wavefronts per (chunk, head) fuses what the reference runs as five launches: the dA part of
// HRDPLR/bwd_triton.py:30-105, the dv kernel :239-290, the dqg/dkg/dbg/dw/dgk_last kernel :309-487, the WY
// backward :503-612, the score backward :627-883 and the log-decay gradient :899-948.  Its inputs are the
// original tensors, do, and per chunk the state entering it (h), the gradient of the state leaving it (dh) and
// the gradient of v_new, left in the workspace by the two scans, and (I - A_ab)^-1 and u from the prep kernel (w as
// well with the HDLA parameterisation; otherwise it is rebuilt here).  Nothing but the seven gradients is written back.
//
// Two differences from the reference's algebra, both exact:
//  * the WY backward never forms d(Tm): with X = [w | u] = Tm R, R = [ag | A_ak v] one has dR = Tm^T dX and
//    dA_ab = mask(dR X^T), which replaces the Tm^T dTm Tm^T chain of bwd_triton.py:577-612;
//  * the score backward covers the whole 16 x 16 (x2 ranks) tile with MFMA products against the same
//    factorised operands as the forward pass instead of a serial per-column loop.
//
// Division of the work: every product here contracts over channels or over value columns, so wave w owns the
// channel tiles kt = w*KT/4 .. and the value tiles vt = w*VT/4 ..; what is summed over the other dimension (the
// score tiles, their gradients, dv) is exchanged through LDS, with five workgroup barriers in all.  One wave per
// chunk would hold the whole chunk in registers, at one wave per SIMD, and nothing would overlap its arithmetic
// with the memory round trips of its neighbours; four waves on a quarter each leave room for two or three
// workgroups per compute unit.
//
// What bounds it: the chain of a chunk's dependent steps at the two or three workgroups a compute unit holds.  The time per
// (chunk, head) is the same whether its inputs are in the last-level cache or not (K = V = 64: 13.5 ns, 128: 32), and no unit
// is saturated (vector issue 56 %, address unit 56 %, LDS 36 %, matrix cores 26 % of the time).  So what shortens the chain
// counts, and what merely saves instructions gave nothing: products requested in the order of their use; three
// exponentials a channel tile instead of seven; do, v and the score gradients turned by the transposing LDS read instead
// of a product and a second store each; sum S dS as the diagonal of a product.  Together, bf16, a/b form, before -> after:
// K = V = 64: 1024 (chunk, head) 22.3 -> 21.4 us, 8192 118.6 -> 116.0, 16384 221.6 -> 214.9; K = V = 128: 1024 41.9 -> 39.8,
// 16384 537 -> 524.  A fixed grid whose workgroups loop over the pairs was slower (114.7 -> 118.7; 519 -> 552), and so were
// one 32-deep product in place of two 16-deep ones where tiles pair up (a few registers more, spilled).
#include "hdla_common.cuh"
#include "hdla_launch.h"

namespace hdla {

constexpr int NW = 4;     // wavefronts per (chunk, head)

// LDS of a workgroup (byte offsets)
template <typename T, int K, int V> struct CgLds {
    static constexpr int ES = sizeof(T);
    // do, v, v_new (2 ranks), dv_new (2 ranks) of the chunk, [matrix][token][value], rows padded by 16 bytes
    static constexpr int VP = V + 16 / ES;
    static constexpr int TOK = 0, TOK_B = 6 * CH * VP * ES;
    // first, per wave: its part of A_qk^T, A_ak^T (2 ranks), fp32 tiles in fragment order (read between barriers 1
    // and 2); later the nine score-gradient tiles, as fragments (4-byte elements: and as fragments of their transposes;
    // 2-byte ones are turned by the transposing LDS read), written between barriers 2 and 3
    static constexpr bool TURN = ES == 2;
    static constexpr int SCORE = TOK + TOK_B, SCORE_B = NW * 3 * 1024, FIN = SCORE, FIN_B = (TURN ? 9 : 18) * TILE * ES;
    // kg of every channel tile (fragments), for dv
    static constexpr int KG = SCORE + (SCORE_B > FIN_B ? SCORE_B : FIN_B), KG_B = (K / 16) * TILE * ES;
    // first: the parts of the nine tiles (fp32), summed in two rounds through NW/2 slots; later, for 2-byte elements: the rows of the seven
    // gradients, so that they leave as whole rows (a lane holds 8 bytes of a row; 8-byte stores of four lanes
    // would write 32-byte pieces, half of what HBM writes at once)
    static constexpr bool STAGE_OUT = ES == 2;
    static constexpr int OPK = K * ES + 16, OPV = V * ES + 16;       // padded rows
    static constexpr int PART_B = (NW / 2) * 9 * 1024, OUT_B = STAGE_OUT ? (7 * OPK + OPV) * CH : 0;
    // all tiles of w (2 ranks), rebuilt by the waves from (I - A_ab)^-1 and a instead of read from the workspace: behind
    // the sums above, in what is otherwise free until the staged rows are written
    static constexpr int WALL_B = 2 * (K / 16) * TILE * ES;
    // per wave and token: three partial sums over channels of the backward of the HDLA parameterisation
    static constexpr int RED = KG + KG_B, RED_B = NW * 3 * CH * 4;
    static constexpr int R1 = RED + RED_B, WALL = R1 + PART_B, R1_B = PART_B + WALL_B > OUT_B ? PART_B + WALL_B : OUT_B;
    // tiles of 4-byte elements that are turned from registers, per wave (K = V = 128 has no registers for it; what lies in LDS as rows is read by columns there too)
    static constexpr bool BY_LDS = ES == 4 && K * V < 128 * 128;
    static constexpr int TURNING = R1 + R1_B;
    static constexpr int BYTES = TURNING + (BY_LDS ? NW * TURN_SCRATCH : 0);
};

// waves per SIMD asked of the compiler (lowest, highest): three workgroups per compute unit for the smallest 2-byte
// shape, two for the other 2-byte shapes
template <typename T, bool GKF32, int K, int V, bool HD> constexpr int cg_waves(bool highest) {
    const bool small = sizeof(T) * K * V <= 2 * 64 * 64;
    if (sizeof(T) != 2) return highest ? 2 : 1;
    return small ? 3 : 2;
}

// x y + u v and x y - u v of the body's text.  Of the two products one is rounded by itself and the other added to it in one step: which, the compiler would decide by what stands
// around them, in each kernel that has the text by itself.  FIRST: x y is the rounded one.  (4-byte elements: one kernel a shape, as it is compiled.)
template <bool FIRST> __device__ __forceinline__ f32x4 sum_of_two(f32x4 x, f32x4 y, f32x4 u, f32x4 v) {
    return FIRST ? __builtin_elementwise_fma(u, v, x * y) : __builtin_elementwise_fma(x, y, u * v);
}
#define CG_SUM(FIRST, x, y, u, v) (sizeof(T) == 4 ? x * y + u * v : sum_of_two<FIRST>(x, y, u, v))
#define CG_DIFF(FIRST, x, y, u, v) (sizeof(T) == 4 ? x * y - u * v : sum_of_two<FIRST>(x, y, -(u), v))

template <typename T, bool GKF32, int K, int V, bool HD>
__device__ __forceinline__ void chunk_grad_strong_pair(const ChunkArgs<T>& p, int cid, int h, char* smem) {
#define CG_STRONG 1
#include "chunk_grad_body.inc"
#undef CG_STRONG
}
// a common pair; a flagged one is left alone, and said to be
template <typename T, bool GKF32, int K, int V, bool HD>
__device__ __forceinline__ void chunk_grad_common_pair(const ChunkArgs<T>& p, int cid, int h, char* smem, bool& was_flagged) {
#define CG_STRONG 0
#define CG_LEAVE do { was_flagged = true; return; } while (0)
#include "chunk_grad_body.inc"
#undef CG_LEAVE
#undef CG_STRONG
}

// The common pairs, one workgroup per (chunk, head), which leave the flagged ones alone; and behind them, or in a launch of their own, what looks for
// the flagged pairs and works them off.  They are rare (a channel must lose more than e^-70 within eight tokens), so this is a small number of
// workgroups that each look through their share of the flags (one read per thread and round) and work off what they find one pair after the other.
// CG_ALL: one launch, where the three passes of a flagged pair do with the registers that the common pairs' occupancy leaves a wave (4-byte elements).
// CG_COMMON and CG_FLAGGED: elsewhere (up to 138 registers too many) the flagged pairs have all registers of a wave per SIMD, the common ones, at the
// limit of their occupancy, pay nothing for them, and when nothing is flagged, which is the rule, their launch costs its start-up and one round of flag
// reads, 4 to 5 us.  fp32, training step of 2 x 1003 tokens, 8 heads, K = V = 64, two launches -> one: 185.6 -> 181.5 us;
// 838 tokens, 12 heads, K = V = 128 382 -> 377; beta form, 900 tokens, 8 heads 141.6 -> 138.6; 2 x 2000 tokens, 16 heads 547 both.
// CG_EACH (2-byte elements): one launch for no more pairs than the device holds at once, where occupancy is nothing and a workgroup may have more registers: each does its own pair,
// flagged or not.  us a training step as
// a graph's replay, two launches -> one: 32 pairs of K = V = 64 36.0 -> 34.2, 252 82.7 -> 80.4 (beta form), 480 54.4 -> 50.1 (beta form), 512 64.6 -> 61.9; K = V = 128, 14 37.7 -> 36.2,
// 256 (beta form, with less to store and read in the scans) 65.4 -> 62.7; 256, ab form, K = 64, V = 128 42.9 -> 40.4, K = 128, V = 64 44.9 -> 42.6, with fp32 decays 43.6 -> 41.2, 46.4 -> 44.3; of
// 82 shapes, forms and types of decays at 4 to 512 pairs all are 0.8 to 3.9 faster.  Beyond, with one workgroup a compute unit: 960 of K = V = 64 62.5 -> 68.4, K = V = 128 528 90 -> 96, 1552 159 -> 188.
enum CgPairs { CG_COMMON, CG_FLAGGED, CG_ALL, CG_EACH };
constexpr int CG_STRONG_GRID = 256;
// CG_EACH's waves per SIMD, and so workgroups a compute unit: what its registers allow
template <bool GKF32, int K, int V> constexpr int cg_each_waves() { return !GKF32 && K == 64 && V == 64 ? 2 : 1; }
template <typename T, bool GKF32, int K, int V, bool HD, CgPairs WHAT>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(WHAT == CG_EACH ? cg_each_waves<GKF32, K, V>() : WHAT == CG_FLAGGED ? 1 : cg_waves<T, GKF32, K, V, HD>(false),
                                                                         WHAT == CG_EACH ? cg_each_waves<GKF32, K, V>() : WHAT == CG_FLAGGED ? 1 : cg_waves<T, GKF32, K, V, HD>(true))))
void chunk_grad_kernel(ChunkArgs<T> p) {
    __shared__ __attribute__((aligned(16))) char smem[CgLds<T, K, V>::BYTES];
    const int total = p.H * p.st.nch;
    if (WHAT != CG_COMMON && WHAT != CG_EACH && (WHAT == CG_FLAGGED || (int)blockIdx.x >= total)) {
        __shared__ unsigned long long sMask[NW];
        constexpr int nth = 64 * NW;
        const int group = (int)blockIdx.x - (WHAT == CG_ALL ? total : 0), groups = (int)gridDim.x - (WHAT == CG_ALL ? total : 0);
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        for (int base = group; base < total; base += groups * nth) {               // uniform over the workgroup
            const int mine = base + (int)threadIdx.x * groups;
            const unsigned long long m = __ballot(mine < total && p.ws.STRONG[mine] != 0);
            if (lane_id() == 0) sMask[w] = m;
            __syncthreads();
            for (int ww = 0; ww < NW; ++ww) {
                unsigned long long todo = sMask[ww];                               // uniform: the same word for all
                while (todo) {
                    const int t = 64 * ww + __builtin_ctzll(todo);
                    todo &= todo - 1;
                    const int chw = base + t * groups;
                    chunk_grad_strong_pair<T, GKF32, K, V, HD>(p, chw % p.st.nch, chw / p.st.nch, smem);
                    __syncthreads();                                               // the next pair reuses the staging areas
                }
            }
            __syncthreads();
        }
        return;
    }
    // Which of the two indices runs fastest over the workgroups decides which rows of the [token][head][channel]
    // tensors the workgroups resident at one time touch.  Measured: with rows of 4 KiB and more, neighbouring
    // workgroups should be the heads of one chunk (together they read whole rows; chunk-fastest, all of them would
    // touch the same few hundred bytes of every row, a fraction of the HBM channels); with shorter rows the chunks
    // of one head, whose workspace records are contiguous.
    const bool head_fastest = (uint32_t)(p.H * K) * sizeof(T) >= 4096;
    const int cid = head_fastest ? blockIdx.x / p.H : blockIdx.x % p.st.nch;
    const int h = head_fastest ? blockIdx.x % p.H : blockIdx.x / p.st.nch;
    if constexpr (WHAT == CG_EACH) {
        bool flagged = false;                                 // (uniform over the workgroup)
        chunk_grad_common_pair<T, GKF32, K, V, HD>(p, cid, h, smem, flagged);
        if (flagged) chunk_grad_strong_pair<T, GKF32, K, V, HD>(p, cid, h, smem);
    } else {
#define CG_STRONG 0
#define CG_LEAVE return
#include "chunk_grad_body.inc"
#undef CG_LEAVE
#undef CG_STRONG
    }
}

template <typename T, bool GKF32, int K, int V, bool HD>
static hipError_t launch_chunk_grad_gk(const ChunkArgs<T>& a, hipStream_t stream) {
    const int total = a.st.nch * a.H, strong = total < CG_STRONG_GRID ? total : CG_STRONG_GRID;
    if constexpr (sizeof(T) == 4) {
        hipLaunchKernelGGL((chunk_grad_kernel<T, GKF32, K, V, HD, CG_ALL>), dim3(total + strong), dim3(64 * NW), 0, stream, a);
    } else if (total <= 256 * cg_each_waves<GKF32, K, V>()) {
        hipLaunchKernelGGL((chunk_grad_kernel<T, GKF32, K, V, HD, CG_EACH>), dim3(total), dim3(64 * NW), 0, stream, a);
    } else {
        hipLaunchKernelGGL((chunk_grad_kernel<T, GKF32, K, V, HD, CG_COMMON>), dim3(total), dim3(64 * NW), 0, stream, a);
        hipLaunchKernelGGL((chunk_grad_kernel<T, GKF32, K, V, HD, CG_FLAGGED>), dim3(strong), dim3(64 * NW), 0, stream, a);
    }
    return hipGetLastError();
}
template <typename T, int K, int V, bool HD>
static hipError_t launch_chunk_grad_kv(const ChunkArgs<T>& a, hipStream_t stream) {
    constexpr bool kAlwaysF32 = sizeof(T) == 4;
    return kAlwaysF32 || a.gk_f32 ? launch_chunk_grad_gk<T, true, K, V, HD>(a, stream) : launch_chunk_grad_gk<T, kAlwaysF32, K, V, HD>(a, stream);
}

template <typename T, bool HD>
static hipError_t launch_chunk_grad_hd(const ChunkArgs<T>& a, int K, int V, hipStream_t stream) {
    if (K == 64 && V == 64) return launch_chunk_grad_kv<T, 64, 64, HD>(a, stream);
    if (K == 128 && V == 128) return launch_chunk_grad_kv<T, 128, 128, HD>(a, stream);
    if (K == 64 && V == 128) return launch_chunk_grad_kv<T, 64, 128, HD>(a, stream);
    if (K == 128 && V == 64) return launch_chunk_grad_kv<T, 128, 64, HD>(a, stream);
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_chunk_grad(const ChunkArgs<T>& a, int K, int V, hipStream_t stream) {
    return a.beta ? launch_chunk_grad_hd<T, true>(a, K, V, stream) : launch_chunk_grad_hd<T, false>(a, K, V, stream);
}
template hipError_t launch_chunk_grad<bf16>(const ChunkArgs<bf16>&, int, int, hipStream_t);
template hipError_t launch_chunk_grad<float>(const ChunkArgs<float>&, int, int, hipStream_t);

}  // namespace hdla
