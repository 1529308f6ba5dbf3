// Fused chunk kernels: the per-chunk preparation (cumulative decays, score tiles, (I - A_ab)^-1, w, u, gated copies:
// HRDPLR/fwd_triton.py:22-790 and fla's chunk_rwkv6_fwd_cumsum) and the inter-chunk state scan that consumes it
// (HRDPLR/fwd_triton.py:808-1095, HRDPLR/bwd_triton.py:127-222) in ONE kernel, so that what the preparation produces
// for the scan -- 14 to 20 KB per (16-token chunk, head) -- goes through LDS and never through HBM.
//
// Work division.  A workgroup owns one (sequence, head, time segment): the chunks of a sequence are cut into `nseg`
// consecutive segments so that few (sequence, head) pairs still fill the device.  It has
//   * FNP = 4 pairs of producer waves.  Pair p prepares the chunks p, p+4, ... of the segment and leaves the operands in
//     LDS slot p.  The two waves of a pair take two of the four channel tiles each.  What comes after their parts of the
//     score tiles is shared out by what the longer chain leaves room for: one of them (the pair's lead) adds up A_ab and
//     solves for (I - A_ab)^-1; the other one adds up the other score tiles, has v to itself (A_ak v, then u) and copies out;
//   * V/16 consumer waves.  Consumer j owns column block j of the fp32 state for the whole segment, in registers, and
//     walks the chunks in order, exactly as the stand-alone scan kernels do.
// A segment other than the first does not know the state that enters it.  The state leaving a chunk is affine in the
// state entering it, so such a segment runs from zero and, beside it, carries the K x K transition matrix M (the same
// update applied to K more columns that start from the identity: consumer j also owns column block j of M).  What the
// chunk's output gains per unit of entering state, G = (qg + A_qb w) M (16 x K), comes out of the same products.
//   forward pass:   o_local and G go to the workspace; fixup_kernel chains the segments' (M, S_local) into the true
//                   entering states and adds G S_in.
//   backward pass:  the entering states are known (kept by the forward pass, or re-derived by a summary-only pass), so
//                   the state checkpoints are exact; M and R = sum_t G_t^T do_t give the gradient entering each
//                   segment from the right, d S_in(s) = M_s^T d S_in(s+1) + R_s, which the reverse kernel's consumers
//                   chain themselves before they start.
//
// What the backward pass's two kernels take over from the forward pass (or from the summary pass, which is the forward
// kernel without its outputs): the record.  Per (chunk, head), 2-byte elements: (I - A_ab)^-1, A_ak, A_qb (8 tiles of
// 16 x 16) and in segments > 0 G (16 x K); per segment M.  That is 6 KB beside the 16 KB of a chunk's inputs at K = V = 64,
// and it is all that takes a producer pair its time: the score products and the triangular solve were three quarters of
// each of the two kernels.  With the record a producer only forms the gated copies, w and
// u (fused_replay), and nothing of M is computed twice.  Measured (4 x 2048 tokens, 16 heads, K = V = 64):
// checkpoint kernel 76 -> 57 us, reverse kernel 69 -> 54 us (with the loads of rows_to_tiles), the forward kernel pays 2 us.
//
// Synchronisation.  Producers and consumers run at their own pace; a slot is handed over through two counters in LDS
// that only ever grow: ready[p] (+1 per wave of pair p and chunk completed) and consumed[p] (consumer-steps finished on
// slot p); the waves of a pair hand each other the parts and the inverse the same way (part[p], inv[p]).
// Waiting is polling with s_sleep; every wait is bounded (FUSED_SPIN_LIMIT polls), and a wave that runs into the bound
// raises an abort flag that ends every other wave's waits as well and is reported through FusedArgs::err, so the grid
// always drains.  There are no workgroup barriers after the first.
//
// What bounds the forward kernel: the producers' instructions.  A pair takes 13 k cycles a chunk, four pairs 3.3 k, the
// consumers 1.3 k; the two producer waves of a SIMD and its consumer issue vector instructions 70 to 80 % of the time, and
// requesting the inputs earlier gains nothing.  Two things had cost a tenth of it on top.  The lead did everything on its
// own while the other wave waited for the inverse: 4 of 15 k cycles.  And a SIMD prefers its older wave: pairs 0 and 1 ran a
// whole round ahead of pairs 2 and 3, whose chunks the consumers needed first, until they stood still for want of a slot;
// with the waves that are past the scores, so nearer to the hand-over, preferred (s_setprio), the pairs take turns.
// us for a forward pass, before -> the work shared out -> and the priority: 4 x 2048 tokens of 16 heads 76.2 -> 74.0 -> 71.6 (a
// and b formed here 77.6 -> 74.4 -> 70.6), 8 x 1024 70.6 -> 67.3 -> 64.1, 16 x 512 of 32 heads 116.5 -> 110.7 -> 101, 1 x 16384 154 ->
// 149 -> 140, 2 x 777 of 8 heads 33.8 -> 32.5 -> 30.6.  Priority for the consumers as well: 72.8; a third level for the solve: the
// same; and in fused_replay, which is bound by its traffic: the same or 5 % more.
#pragma once
#include "hdla_common.cuh"
#include "fused_shapes.h"

#include <type_traits>

namespace hdla {

constexpr int FNP = 4;                    // producer pairs = LDS slots
constexpr int FLDP = 36;                  // padded row length of the 32 x 32 matrices of the triangular solve
constexpr int FUSED_SPIN_LIMIT = 1 << 20; // polls of ~256 cycles: a tenth of a second, four orders above any real wait
// What a wave that gave up writes to FusedArgs::err (+1 producer, +2 forward consumer, +3 reverse consumer).  The word is
// never cleared (that would take a launch of its own): it is a diagnostic that reads as this pattern only after an
// abort, or by a one-in-a-billion coincidence with what the caller's memory held before.
constexpr int FUSED_ABORTED = 0x48444c00;

// chunk range [s0, s1) of time segment `seg` of sequence n
__device__ __forceinline__ void seg_range(const SeqTab& st, int n, int nseg, int seg, int& s0, int& s1) {
    int c0, c1;
    seq_chunks(st, n, c0, c1);
    seg_range(c0, c1, nseg, seg, s0, s1);
}

// Columns 16 j + 4 g .. + 3 of row c of a chunk's G, in elements from its start: pieces of eight columns, the 16 rows of a piece side by side
__device__ __forceinline__ int gw_at(int j, int g, int c) { return (j >> 1) * PAIR + ((2 * (j & 1) + (g >> 1)) * 16 + c) * 8 + 4 * (g & 1); }

// LDS of a fused workgroup (byte offsets): per producer pair one slot = [operands | outbox | solver scratch], then the flags
template <typename T, int K, int V, int MODE> struct FusedLds {
    static constexpr int ES = sizeof(T), TB = TILE * ES, KT = K / 16, VT = V / 16;
    static constexpr bool REV = MODE == FUSED_REV, FWD = MODE == FUSED_FWD, SOLVES = FWD || MODE == FUSED_SUM;
    static constexpr BlkF BF = blk_fwd(K, ES, SOLVES);
    static constexpr SlotB SB = slot_bwd(K, ES);
    // forward direction: the forward-scan block, then u^T (VT tile pairs), v^T (VT tiles); checkpoint kernel: do^T (VT
    // tiles); where the score tiles are solved: (I - A_ab)^-1 as chunk_grad reads it (2 tile pairs) and A_ak (a tile pair)
    static constexpr int UT = BF.SIZE, VTT = UT + 2 * VT * TB, FWD_END = VTT + VT * TB;
    static constexpr int TMB = FWD_END, AKB = TMB + 4 * TB;
    // reverse direction: the reverse-scan slot, then do^T
    static constexpr int DOT = REV ? SB.SIZE : FWD_END;
    static constexpr int OPER = SOLVES ? AKB + 2 * TB : DOT + VT * TB;
    // outbox of the forward pass: 16 rows of o (fp32 in segments > 0, element type in segment 0) and 16 rows of G
    static constexpr int OROW = V * 4 + 16, GROW = K * ES + 16;
    static constexpr int OBOX = OPER, GBOX = OBOX + (FWD ? CH * OROW : 0);
    static constexpr int SOLVE = GBOX + (FWD ? CH * GROW : 0);
    static constexpr int SLOT = SOLVE + (SOLVES ? 2 * 32 * FLDP * 4 : 0);
    // int ready[4], consumed[4], abort, -, -, -, part[4], inv[4], strong[4] (per producer pair; see fused_producer), then
    // two counters of the reverse kernel's consumers (words 24 and 25; records staged, records used: fused_consumer_rev), -, -, and rest[4]
    // (fused_producer): all 32 words
    static constexpr int FLAGS = FNP * SLOT;
    // reverse kernel: transition records of the segments to the right, as split operands, for the consumers' chain
    // (CHAIN_STAGE records of K x K at a time: every consumer wave needs them whole, each loads a quarter)
    static constexpr int CHAIN_STAGE = 2;
    // scratch of the producers for their loads (rows_to_tiles): one area a wave; where the waves of a pair solve, one a pair
    // for its lead, the other wave has the second half of the solver scratch, which is free until that wave itself fills it with its parts
    static constexpr int ROWS = FLAGS + 128, ROWS_B = (SOLVES ? FNP : 2 * FNP) * ROWS_SCRATCH;
    static constexpr int CHAIN = ROWS + ROWS_B;
    static constexpr int BYTES = CHAIN + (REV ? CHAIN_STAGE * 2 * KT * KT * TB : 0);
};

// ---- hand-over counters ------------------------------------------------------------------------------------------
__device__ __forceinline__ bool wait_ge(int* flag, int want, int* abort_flag) {
    int spins = 0;
    while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < want) {
        if (__hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0 || ++spins > FUSED_SPIN_LIMIT) {
            __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            return false;
        }
        __builtin_amdgcn_s_sleep(4);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    return true;
}
// all LDS accesses of the wave so far are complete before the counter moves
__device__ __forceinline__ void signal_set(int* flag, int value) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    if (lane_id() == 0) __hip_atomic_store(flag, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void signal_add(int* flag) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    if (lane_id() == 0) __hip_atomic_fetch_add(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// the log-decays of four channels as they sit in memory (element type or fp32), converted only where they are used, and of
// the wave's share of a chunk as loaded (a row's 32 channels: 64 bytes as one piece a lane, or 128 bytes as two)
template <typename T, bool GKF32> struct GkRaw {
    typedef Frag<T> type;
    typedef i32x4 rows;
    static __device__ __forceinline__ void load(const char* p, int l, uint32_t row_ch, rows& x) { x = *reinterpret_cast<const i32x4*>(at(p, 2 * row_ch + 16 * (l & 3))); }
    static __device__ __forceinline__ void tiles(char* scratch, int l, rows x, type (&f)[2]) { rows_to_tiles(scratch, l, x, f[0], f[1]); }
    static __device__ __forceinline__ void drop(rows& x) { forget(x); }
    static __device__ __forceinline__ f32x4 value(type x) { return to_f32(x); }
    static __device__ __forceinline__ void mask(type& x, bool ok) { x.v = ok ? x.v : zero_frag<T>().v; }
};
template <typename T> struct GkRaw<T, true> {
    typedef f32x4 type;
    struct rows { f32x4 x[2]; };
    static __device__ __forceinline__ void load(const char* p, int l, uint32_t row_ch, rows& x) {
#pragma unroll
        for (int j = 0; j < 2; ++j) x.x[j] = *reinterpret_cast<const f32x4*>(at(p, 4 * row_ch + 64 * j + 16 * (l & 3)));
    }
    static __device__ __forceinline__ void tiles(char* scratch, int l, const rows& x, type (&f)[2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) f[j] = rows_to_tile(scratch, l, x.x[j]);
    }
    static __device__ __forceinline__ void drop(rows& x) { forget(x.x[0]); forget(x.x[1]); }
    static __device__ __forceinline__ f32x4 value(type x) { return x; }
    static __device__ __forceinline__ void mask(type& x, bool ok) { x = ok ? x : zero4(); }
};

// F(I16) for lane (g, c), like ident_frag() but from the caller's lane coordinates
template <typename T> __device__ __forceinline__ Frag<T> ident_of(int g, int c) {
    f32x4 e;
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = (c == 4 * g + i) ? 1.f : 0.f;
    return to_frag<T>(e);
}

// ---- producers -----------------------------------------------------------------------------------------------------
// Everything of a chunk that does not depend on the state, by a PAIR of waves, into LDS slot `pp`.  Wave `half` of the
// pair takes the channel tiles 2 half, 2 half + 1 (one stored tile pair of every operand).  The score tiles are sums over
// all channels: each wave hands the other its parts of some through LDS.  The pair's `lead` wave finishes A_ab, solves the
// (small) triangular system and hands (I - A_ab)^-1 back; meanwhile the other wave finishes A_qk, A_qb and A_ak, forms A_ak v
// and copies out the chunk before; each forms w for its own tiles, the other wave u.  The formulas are the stand-alone prep kernel's (prep.hip); what differs from its one-wave form is the order
// in which the two halves of a score tile's sum over channels are added.
//
// One wave per chunk (the first form of this kernel) took 19,000 cycles a chunk, most of them waiting for its own
// previous instruction: alone on its SIMD nothing fills those gaps.  Two waves per chunk on three waves per SIMD do.
template <typename T, bool GKF32, int K, int V, int MODE, bool HD>
__device__ __forceinline__ void fused_producer(const FusedArgs<T>& a, char* smem, int n, int h, int seg, int s0, int s1, int pp, int half) {
    static_assert(K == 64 && sizeof(T) == 2 && V % 32 == 0, "a producer pair holds all channels of a chunk: K = 64, 2-byte elements");
    typedef FusedLds<T, K, V, MODE> L;
    constexpr bool FWD = MODE == FUSED_FWD;
    static_assert(L::SOLVES, "the backward pass's kernels read what this producer solves for (fused_replay)");
    constexpr int KT = K / 16, VT = V / 16, KT2 = KT / 2, KH = 2;
    constexpr BlkF BF = L::BF;
    const ChunkArgs<T>& p = a.c;
    char* slot = smem + pp * L::SLOT;
    // the pair's scratch: first the other wave's parts of A_ab's four tiles (fp32, 4 KiB); then, in the same bytes,
    // A_ab and its inverse for the solve; then the inverse as operand tiles for the other wave
    float *sP, *sN, *sT;
    T* sPub;
    int* const flags = reinterpret_cast<int*>(smem + L::FLAGS);
    int* const f_ready = flags + pp, * const f_consumed = flags + 4 + pp, * const f_abort = flags + 8;
    int* const f_part = flags + 12 + pp, * const f_inv = flags + 16 + pp, * const f_strong = flags + 20 + pp, * const f_rest = flags + 28 + pp;
    const bool lead = half == (pp >> 1);                  // spreads the leads over the SIMDs
    int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H;
    const float scale = p.scale;
    const int nst = s1 - s0;
    const int kt0 = half * KH;
    int64_t bos, eos;
    seq_bounds(p.st, n, bos, eos);
    int c0, c1;
    seq_chunks(p.st, n, c0, c1);

    // rows [rb, rb + NR) of the previous chunk's results, left in the outbox by the consumers, out to global memory
    // (forward pass)
    auto copy_out = [&](int cid, int rb, auto nr) __attribute__((always_inline)) {
        constexpr int NR = decltype(nr)::value;
        if constexpr (FWD) {
            // the lane's offsets below are formed afresh in every call: hoisted out of the chunk loop they would be held
            // in registers through all of it
            int l = lane_id();
            asm volatile("" : "+v"(l));
            const int64_t tok0 = bos + (int64_t)(cid - c0) * CH;
            const int len = (int)min((int64_t)CH, eos - tok0);
            const int64_t chw = (int64_t)h * p.st.nch + cid;
            if (seg == 0) {
                constexpr int LPR = V * (int)sizeof(T) / 16, RPI = 64 / LPR;
#pragma unroll
                for (int r0 = 0; r0 < NR; r0 += RPI) {
                    const int r = rb + r0 + l / LPR, e = (l % LPR) * 16;
                    const i32x4 x = *reinterpret_cast<const i32x4*>(slot + L::OBOX + r * L::OROW + e);
                    if (r < len) st_past(reinterpret_cast<i32x4*>(reinterpret_cast<char*>(p.o + ((tok0 + r) * H + h) * V) + e), x);
                }
            } else {
                // in the order in which fixup_kernel takes them: 1-KiB pieces, lane (g, c) has columns 16 j + 4 g .. + 3 of o's row c, and
                // columns 32 j + 8 g .. + 7 of G's
                const int g = l >> 4, c = l & 15;
                char* ol = reinterpret_cast<char*>(a.ol + chw * (CH * V)) + 16 * l;
#pragma unroll
                for (int i = 0; i < V / 16 * NR / CH; ++i) {
                    const int j = rb * (V / 16) / CH + i;
                    *reinterpret_cast<i32x4*>(ol + j * 1024) = *reinterpret_cast<const i32x4*>(slot + L::OBOX + c * L::OROW + 64 * j + 16 * g);
                }
                char* gw = reinterpret_cast<char*>(a.gw + chw * (CH * K)) + 16 * l;
#pragma unroll
                for (int i = 0; i < K / 32 * NR / CH; ++i) {
                    const int j = rb * (K / 32) / CH + i;
                    *reinterpret_cast<i32x4*>(gw + j * 1024) = *reinterpret_cast<const i32x4*>(slot + L::GBOX + c * L::GROW + 64 * j + 16 * g);
                }
            }
        }
    };

    // The wave's share of the chunk's inputs as loaded, 16 bytes a lane (rows_to_tiles): requested one chunk of this pair
    // ahead, as soon as the registers are free, so that the round trip to HBM runs behind the rest of the previous chunk.
    // With the HDLA parameterisation the sum over ALL channels of k^2 f is needed: the other half's k and gk come along.
    // In parts, by what three waves per SIMD have registers for: 0 beside the score tiles, 1 when those are done with; v (2)
    // only behind the scores of its own chunk; the decays once more (3) where the strong-decay passes want them.
    i32x4 xq, xk, xa[2], xb[2], xv[2], xok;
    typename GkRaw<T, GKF32>::rows xg, xog;
    T nbeta;
    char* const sX = lead ? smem + L::ROWS + pp * ROWS_SCRATCH : smem + pp * L::SLOT + L::SOLVE + 32 * FLDP * 4;
    static_assert(K / 2 == 32 && V / 2 == 32, "half a row of any operand is 64 bytes");
    auto request = [&](int t, int part) __attribute__((always_inline)) {
        const int cid = s0 + t;
        const int64_t tok0 = bos + (int64_t)(cid - c0) * CH;
        const int len = (int)min((int64_t)CH, eos - tok0);
        // uniform base of the chunk's first row + a 32-bit offset per lane, formed afresh in every call (see copy_out);
        // rows past the end alias the last valid row and are masked at use
        int ll = l;
        asm volatile("" : "+v"(ll));
        const uint32_t row = (uint32_t)min(ll >> 2, max(len, 1) - 1), last = (uint32_t)(max(len, 1) - 1), piece = 16 * (ll & 3);
        constexpr uint32_t ES = sizeof(T), GS = GKF32 ? 4 : 2;
        if (part == 2) {
#pragma unroll
            for (int j = 0; j < 2; ++j) xv[j] = *reinterpret_cast<const i32x4*>(at(p.v + (tok0 * H + h) * V, (row * (uint32_t)(H * V) + 32 * j) * ES + piece));
            return;
        }
        const uint32_t qo = (row * (uint32_t)(H * K) + 16 * kt0) * ES + piece, ao = (row * (uint32_t)(RANK * H * K) + 16 * kt0) * ES + piece;
        const int64_t qb = (tok0 * H + h) * K, ab = (tok0 * RANK * H + h) * K;
        const char* gkp = reinterpret_cast<const char*>(p.gk) + qb * GS;
        auto rows = [](const T* b, uint32_t off) __attribute__((always_inline)) { return *reinterpret_cast<const i32x4*>(at(b, off)); };
        if (part != 1) GkRaw<T, GKF32>::load(gkp, ll, row * (uint32_t)(H * K) + 16 * kt0, xg);
        if (part == 3) return;
        if (part == 0) {
            xk = rows(p.k + qb, qo);
            if (!HD) {
#pragma unroll
                for (int r = 0; r < 2; ++r) xb[r] = rows(p.b + ab, ao + r * (uint32_t)(H * K) * ES);
            }
            return;
        }
        if (HD) {
            const uint32_t other = 16 * (KH - kt0);
            nbeta = *at(p.beta + tok0 * H + h, min((uint32_t)(ll & 15), last) * (uint32_t)H * ES);
            GkRaw<T, GKF32>::load(gkp, ll, row * (uint32_t)(H * K) + other, xog);
            xok = rows(p.k + qb, qo + (other - 16 * kt0) * ES);
        }
        xq = rows(p.q + qb, qo);
        if (!HD) {
#pragma unroll
            for (int r = 0; r < 2; ++r) xa[r] = rows(p.a + ab, ao + r * (uint32_t)(H * K) * ES);
        }
    };
    // rows past the end of a ragged chunk become zeros, in place and only there (a uniform branch: whole chunks pay nothing)
    auto mask = [](Frag<T>& f, bool ok) __attribute__((always_inline)) { f.v = ok ? f.v : zero_frag<T>().v; };
    auto mask_gk = [](typename GkRaw<T, GKF32>::type& x, bool ok) __attribute__((always_inline)) { GkRaw<T, GKF32>::mask(x, ok); };
    if (pp < nst) { request(pp, 0); request(pp, 1); }
    // (the requested inputs are forgotten where the wave ends early, and where they may or may not be requested again: otherwise
    // their old values stay in registers through the whole chunk)
    auto forget_first = [&]() __attribute__((always_inline)) { GkRaw<T, GKF32>::drop(xg); forget(xk); forget(xb[0]); forget(xb[1]); };
    auto forget_rest = [&]() __attribute__((always_inline)) { GkRaw<T, GKF32>::drop(xog); forget(xok); forget(xq); forget(xa[0]); forget(xa[1]); };
    // A wait that gave up (see wait_ge) ends the loop, not the chunk: with the abort flag up no later wait takes time, what the chunk's steps
    // then make of LDS is thrown away, no address depends on it, and the steps stay one straight piece of code for the register allocation.
    bool alive = true;
    int it = 0, prev_cid = -1;
    for (int t = pp; t < nst && alive; t += FNP, ++it) {
        const int cid = s0 + t;
        const int64_t tok0 = bos + (int64_t)(cid - c0) * CH;
        const int len = (int)min((int64_t)CH, eos - tok0);
        const int64_t chw = (int64_t)h * p.st.nch + cid;
        // What depends on the lane only (offsets into the slot, masks, the identity tile) is formed afresh for every chunk:
        // hoisted out of the loop it would be held in registers, or spilled, through all of it.
        asm volatile("" : "+v"(l));
        g = l >> 4;
        c = l & 15;
        {
            int so = pp * L::SLOT;
            asm volatile("" : "+s"(so));
            slot = smem + so;
            sP = reinterpret_cast<float*>(slot + L::SOLVE);
            sN = sP;
            sT = sP + 32 * FLDP;
            sPub = reinterpret_cast<T*>(sP);
        }
        const Frag<T> ident = ident_of<T>(g, c);
        const bool rowok = c < len;

        Frag<T> nq[KH], nk[KH], na[2][KH], nb[2][KH], ok_[KH];
        typename GkRaw<T, GKF32>::type ng[KH], og[KH];
        GkRaw<T, GKF32>::tiles(sX, l, xg, ng);
        rows_to_tiles(sX, l, xk, nk[0], nk[1]);
        if (!HD) {
#pragma unroll
            for (int r = 0; r < 2; ++r) rows_to_tiles(sX, l, xb[r], nb[r][0], nb[r][1]);
        } else {
            GkRaw<T, GKF32>::tiles(sX, l, xog, og);
            rows_to_tiles(sX, l, xok, ok_[0], ok_[1]);
        }
        rows_to_tiles(sX, l, xq, nq[0], nq[1]);
        if (!HD) {
#pragma unroll
            for (int r = 0; r < 2; ++r) rows_to_tiles(sX, l, xa[r], na[r][0], na[r][1]);
        }
        __builtin_amdgcn_sched_barrier(0);
        // (ag^T waits in the slot where w will go: w = Tm ag is formed further down, when the inverse is there)
        T* const sWW = reinterpret_cast<T*>(slot + BF.W);

        // ---- own channel tiles: decays, parts of the score tiles (prep.hip, phase A) -------------------------------------
        // Nothing here needs the slot: the consumers are through with the chunk it held by the time the gated copies below
        // are to go there (waiting for them first left a pair idle for a fifth of its time).
        f32x4 egi[KH], edn[KH];
        f32x4 aqk = zero4(), aqb[2] = {zero4(), zero4()}, aak[2] = {zero4(), zero4()};
        f32x4 aab[2][2] = {{zero4(), zero4()}, {zero4(), zero4()}};
        bool strong = false;                              // a channel decays beyond the safe range (uniform over the wave)
        float beta_t = 0.f, s_t = 0.f;
        if (HD) {
            if (len < CH) {
#pragma unroll
                for (int j = 0; j < KH; ++j) { mask_gk(ng[j], rowok); mask_gk(og[j], rowok); mask(nk[j], rowok); mask(ok_[j], rowok); }
            }
            beta_t = rowok ? ld_elem(&nbeta) : 0.f;
#pragma unroll
            for (int j = 0; j < KH; ++j) {
                const f32x4 g4 = GkRaw<T, GKF32>::value(ng[j]), gx = GkRaw<T, GKF32>::value(og[j]);
                const f32x4 k4 = to_f32(nk[j]), kx = to_f32(ok_[j]);
                const f32x4 kf = k4 * k4 * exp4<T>(g4) + kx * kx * exp4<T>(gx);
                s_t += kf[0] + kf[1] + kf[2] + kf[3];
            }
            s_t = sum_groups(s_t);
        }
        // the operands of channel tile j as the products take them: as loaded, or (HDLA parameterisation) formed from k,
        // gk, beta and s
        auto operands = [&](int j, f32x4 g4, Frag<T>& rq, Frag<T>& rk, Frag<T> (&ra)[2], Frag<T> (&rb)[2]) __attribute__((always_inline)) {
            rq = nq[j];
            rk = nk[j];
            if (HD) {
                const f32x4 kk = to_f32(rk), f4 = exp4<T>(g4);
                ra[0] = to_frag<T>(kk * (-beta_t));
                ra[1] = to_frag<T>(kk * ((beta_t * s_t - f4) * beta_t));
                rb[0] = to_frag<T>(f4 * kk);
                rb[1] = rk;
            } else {
                ra[0] = na[0][j];
                ra[1] = na[1][j];
                rb[0] = nb[0][j];
                rb[1] = nb[1][j];
            }
        };
        auto decays = [&](int j, f32x4& gi, f32x4& ge) __attribute__((always_inline)) {
            const f32x4 g4 = GkRaw<T, GKF32>::value(ng[j]);
            gi = scan16_incl(g4);
            ge = gi - g4;
        };
#pragma unroll
        for (int j = 0; j < KH; ++j) {
            if (len < CH) {
                mask_gk(ng[j], rowok);
                mask(nq[j], rowok);
                mask(nk[j], rowok);
                if (!HD) { mask(na[0][j], rowok); mask(na[1][j], rowok); mask(nb[0][j], rowok); mask(nb[1][j], rowok); }
            }
            if (HD) pin(ng[j]);                           // e^{gk} formed again, not kept from the sum above
            const f32x4 g4 = GkRaw<T, GKF32>::value(ng[j]);
            Frag<T> rq, rk, ra[2], rb[2];
            operands(j, g4, rq, rk, ra, rb);
            if (HD) __builtin_amdgcn_sched_barrier(0);
            const TileDecay<T> e(g4, c);
            strong |= e.strong;
            egi[j] = e.egi;
            edn[j] = e.edn;
            // One row-side operand at a time against the three inner-side ones, the scheduler kept from interleaving the
            // groups (each tile still gets its products in the order of the channel tiles): all six split operands
            // at once are more registers than three waves per SIMD leave.
            {
                Split<T> kh, bh[2];
                split(to_f32(rk) * e.ek, kh);
                split(to_f32(rb[0]) * e.ek, bh[0]);
                split(to_f32(rb[1]) * e.ek, bh[1]);
                __builtin_amdgcn_sched_barrier(0);
                {
                    Split<T> qh;
                    split(to_f32(rq) * e.eq * scale, qh);
                    if constexpr (FWD) mm_split<3>(qh, {&kh, &bh[0], &bh[1]}, {&aqk, &aqb[0], &aqb[1]});
                    else mm_split<2>(qh, {&bh[0], &bh[1]}, {&aqb[0], &aqb[1]});
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    Split<T> ah;
                    split(to_f32(ra[r]) * e.ea, ah);
                    mm_split<3>(ah, {&kh, &bh[0], &bh[1]}, {&aak[r], &aab[r][0], &aab[r][1]});
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        // Each wave decides for its own channels (the parts of the score tiles add up whichever way they were formed).
        // Where a channel decays too strongly for the single centre, what was accumulated above may hold infinities: it
        // is thrown away and the parts are formed again by passes whose exponents cannot overflow (see DecayPass).
        if (strong) {
            if (!HD) {                                    // (not held through the common path)
                request(t, 3);
                GkRaw<T, GKF32>::tiles(sX, l, xg, ng);
                if (len < CH) { mask_gk(ng[0], rowok); mask_gk(ng[1], rowok); }
            }
            aqk = zero4();
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                aqb[s] = zero4(); aak[s] = zero4(); aab[0][s] = zero4(); aab[1][s] = zero4();
            }
#pragma unroll 1
            for (int ps = 0; ps < DecayPass::COUNT; ++ps) {
                const DecayPass dp(ps, c);
#pragma unroll
                for (int j = 0; j < KH; ++j) {
                    f32x4 gi, ge, eq, ek, ea;
                    decays(j, gi, ge);
                    dp.factors<T>(gi, ge, eq, ek, ea);
                    Frag<T> rq, rk, ra[2], rb[2];
                    operands(j, gi - ge, rq, rk, ra, rb);
                    pin(rk); pin(rq); pin(ra[0]); pin(ra[1]); pin(rb[0]); pin(rb[1]);
                    Split<T> qh, kh, bh[2];
                    split(to_f32(rk) * ek, kh);
                    split(to_f32(rq) * eq * scale, qh);
                    if (FWD) aqk = mm_split(qh, kh, aqk);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        split(to_f32(rb[s]) * ek, bh[s]);
                        aqb[s] = mm_split(qh, bh[s], aqb[s]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        Split<T> ah;
                        split(to_f32(ra[r]) * ea, ah);
                        aak[r] = mm_split(ah, kh, aak[r]);
                        aab[r][0] = mm_split(ah, bh[0], aab[r][0]);
                        aab[r][1] = mm_split(ah, bh[1], aab[r][1]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
        __builtin_amdgcn_s_setprio(1);                    // nearer to the hand-over than a wave that forms scores (see the top of the file)
        // ---- what both waves do with their own channel tiles ------------------------------------------------------------
        auto gated = [&]() __attribute__((always_inline)) {
            // gated copies (prep.hip, phase C), each to its half of the stored pair
#pragma unroll
            for (int j = 0; j < KH; ++j) {
                pin(nq[j]); pin(nk[j]);                       // converted again, not kept converted from above
                if (HD) pin(ng[j]);
                else { pin(na[0][j]); pin(na[1][j]); pin(nb[0][j]); pin(nb[1][j]); }
                Frag<T> rq, rk, ra[2], rb[2];
                operands(j, HD ? GkRaw<T, GKF32>::value(ng[j]) : zero4(), rq, rk, ra, rb);
                const f32x4 one = {1.f, 1.f, 1.f, 1.f}, ege = prev_token(egi[j], one), egl = bcast16<CH - 1>(egi[j]);
                st_pair2(sWW + (j * KT2 + half) * PAIR, transpose(to_frag<T>(to_f32(ra[0]) * ege), ident),
                         transpose(to_frag<T>(to_f32(ra[1]) * ege), ident));
                const Frag<T> fqg = to_frag<T>(to_f32(rq) * egi[j] * scale);
                const Frag<T> fbg[2] = {to_frag<T>(to_f32(rb[0]) * edn[j]), to_frag<T>(to_f32(rb[1]) * edn[j])};
                st_pair(reinterpret_cast<T*>(slot + BF.KGT) + half * PAIR, j, transpose(to_frag<T>(to_f32(rk) * edn[j]), ident));
                st_pair2(reinterpret_cast<T*>(slot + BF.BGT) + (kt0 + j) * PAIR, transpose(fbg[0], ident), transpose(fbg[1], ident));
                st_pair(reinterpret_cast<T*>(slot + BF.QG) + half * PAIR, j, fqg);
                if (c == 0) *reinterpret_cast<f32x4*>(slot + BF.EGL + (16 * (kt0 + j) + 4 * g) * 4) = egl;
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // the inputs are used up: the next chunk's may come
        auto next_first = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            forget_first();
            if (t + FNP < nst) request(t + FNP, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto next_rest = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            forget_rest();
            if (t + FNP < nst) request(t + FNP, 1);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto form_w = [&](const Frag<T> (&tm)[2][2]) __attribute__((always_inline)) {
            // w = Tm ag, in place of ag^T
            {
                Frag<T> agT[2][2], fw[2][2];
                ld_pair(sWW + half * PAIR, agT[0][0], agT[1][0]);
                ld_pair(sWW + (KT2 + half) * PAIR, agT[0][1], agT[1][1]);
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        fw[s][e] = to_frag<T>(mm2(tm[s][0], tm[s][1], agT[0][e], agT[1][e], zero4()));
                    }
#pragma unroll
                for (int s = 0; s < 2; ++s) st_pair2(sWW + (s * KT2 + half) * PAIR, fw[s][0], fw[s][1]);
            }
        };
        // causal masks: lane (g,c) reg i is entry (row c, inner 4g+i)
        auto below = [&](f32x4& x, bool diag) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = 4 * g + i;
                if (!(diag ? j <= c : j < c)) x[i] = 0.f;
            }
        };
        // Each wave leaves the other its parts of the score tiles that the other one finishes: the lead has A_ab, the other wave the
        // rest, whose parts lie in the slot where that wave itself writes later (u's place and, the fifth, A_ak's).
        constexpr int NPART = FWD ? 5 : 4;
        static_assert(VT == 4, "four tiles in u's place");
        auto part_at = [&](int i) __attribute__((always_inline)) { return reinterpret_cast<f32x4*>(slot + (i < 4 ? L::UT + i * 1024 : L::AKB) + 16 * l); };
        f32x4* const rest[5] = {&aak[0], &aak[1], &aqb[0], &aqb[1], &aqk};
        if (lead) {
            // the slot: wait until the consumers have left the chunk it held
            __builtin_amdgcn_sched_barrier(0);
            alive &= wait_ge(f_consumed, VT * it, f_abort);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NPART; ++i) *part_at(i) = *rest[i];
            signal_set(f_rest, it + 1);
            __builtin_amdgcn_sched_barrier(0);
            gated();
            next_first();
            // ---- whole A_ab, (I - A_ab)^-1 by forward substitution (prep.hip, phase B) -----------------------------------
            Frag<T> tm[2][2];
            alive &= wait_ge(f_part, it + 1, f_abort);
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    aab[r][s] += *reinterpret_cast<const f32x4*>(sP + ((2 * r + s) * 64 + l) * 4);
                    below(aab[r][s], false);
                }
            if (p.ws.TM && l == 0) p.ws.STRONG[chw] = (strong || *f_strong != 0) ? 1 : 0;
            // (all of the other wave's parts have been read: the scratch may be written)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    *reinterpret_cast<f32x4*>(&sN[(16 * r + c) * FLDP + 16 * s + 4 * g]) = aab[r][s];
            __builtin_amdgcn_sched_barrier(0);
            // The system in token halves, L = tokens 0..7 and H = 8..15 (both ranks: 16 rows each):
            //   (I - A)^-1 = [[T_LL, 0], [T_HL, T_HH]],  T_LL = (I - A_LL)^-1,  T_HH = (I - A_HH)^-1,  T_HL = T_HH A_HL T_LL.
            // The two diagonal blocks are independent eight-step substitutions that run side by side on the lanes (a
            // quarter of the dependent multiply-adds of one sixteen-step substitution); the block below the diagonal is
            // two 16 x 16 x 16 products, in split operands like the score products (the error of fp32 products).
            {
                int lb = l;                               // formed afresh per chunk (see copy_out)
                asm volatile("" : "+v"(lb));
                // lane: rank of the rows r, token half hf, column (rank sc, token jc of the same half)
                const int r = lb >> 5, hf = (lb >> 4) & 1, sc = (lb >> 3) & 1, jc = lb & 7;
                const int col = 16 * sc + 8 * hf + jc;
                float x[8], y[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float* nrow = &sN[(16 * r + 8 * hf + i) * FLDP + 8 * hf];
                    float acc0 = (sc == r && jc == i) ? 1.f : 0.f, acc1 = 0.f;
#pragma unroll
                    for (int j4 = 0; j4 < (i + 3) / 4; ++j4) {
                        const f32x4 co = *reinterpret_cast<const f32x4*>(nrow + 16 * r + 4 * j4);
                        const f32x4 cx = *reinterpret_cast<const f32x4*>(nrow + 16 * (1 - r) + 4 * j4);
#pragma unroll
                        for (int jj = 0; jj < 4; ++jj) {
                            const int j = 4 * j4 + jj;
                            if (j < i) { acc0 = fmaf(co[jj], x[j], acc0); acc1 = fmaf(cx[jj], y[j], acc1); }
                        }
                    }
                    x[i] = acc0 + acc1;
                    y[i] = xor32(x[i]);
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    sT[(16 * r + 8 * hf + i) * FLDP + col] = x[i];
                    // the block above the diagonal (rows of L, columns of H) is zero: the lanes of L write it
                    if (hf == 0) sT[(16 * r + i) * FLDP + col + 8] = 0.f;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            {
                // 16 x 16 matrices in (rank, token of the half) order: row c = 8 rank + token, inner 4g .. 4g+3 likewise
                const int rr = c >> 3, ii = c & 7, ss = g >> 1, j0 = 4 * (g & 1);
                const f32x4 ahl = *reinterpret_cast<const f32x4*>(&sN[(16 * rr + 8 + ii) * FLDP + 16 * ss + j0]);
                const f32x4 thh = *reinterpret_cast<const f32x4*>(&sT[(16 * rr + 8 + ii) * FLDP + 16 * ss + 8 + j0]);
                f32x4 tllT;                               // T_LL^T: row c is column c of T_LL
#pragma unroll
                for (int e = 0; e < 4; ++e) tllT[e] = sT[(16 * ss + j0 + e) * FLDP + 16 * rr + ii];
                Split<T> pa, pb;
                split(tllT, pa);
                split(ahl, pb);
                const f32x4 xT = mm_split(pa, pb, zero4());    // (A_HL T_LL)^T = T_LL^T A_HL^T
                split(thh, pa);
                split(xT, pb);
                const f32x4 thl = mm_split(pa, pb, zero4());   // T_HH (A_HL T_LL)
                *reinterpret_cast<f32x4*>(&sT[(16 * rr + 8 + ii) * FLDP + 16 * ss + j0]) = thl;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int s2 = 0; s2 < 2; ++s2)
                    tm[s][s2] = to_frag<T>(*reinterpret_cast<const f32x4*>(&sT[(16 * s + c) * FLDP + 16 * s2 + 4 * g]));
            // for the other wave: the inverse's four blocks as operand tiles (in A_ab's bytes, which are used up)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s) st_pair2(sPub + s * PAIR, tm[s][0], tm[s][1]);
            if (p.ws.TM) {
                // the record goes out from the consumers, which have no loads to wait for: a store issued here would stand
                // behind the next chunk's loads in this wave's in-order memory counter
                T* tmw = reinterpret_cast<T*>(slot + L::TMB);
#pragma unroll
                for (int s = 0; s < 2; ++s) st_pair2(tmw + s * PAIR, transpose(tm[s][0], ident), transpose(tm[s][1], ident));
            }
            signal_set(f_inv, it + 1);
            next_rest();
            form_w(tm);
        } else {
            f32x4* const parts[4] = {&aab[0][0], &aab[0][1], &aab[1][0], &aab[1][1]};
#pragma unroll
            for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4*>(sP + (i * 64 + l) * 4) = *parts[i];
            if (l == 0) *f_strong = strong;
            signal_set(f_part, it + 1);
            request(t, 2);
            __builtin_amdgcn_sched_barrier(0);
            alive &= wait_ge(f_consumed, VT * it, f_abort);
            __builtin_amdgcn_sched_barrier(0);
            // the other score tiles, whole
            alive &= wait_ge(f_rest, it + 1, f_abort);
#pragma unroll
            for (int i = 0; i < NPART; ++i) {
                *rest[i] += *part_at(i);
                below(*rest[i], i >= 2);
            }
            if (FWD) st_frag(reinterpret_cast<T*>(slot + BF.AQK) + 4 * l, to_frag<T>(aqk));
            st_pair2(reinterpret_cast<T*>(slot + BF.AQB), to_frag<T>(aqb[0]), to_frag<T>(aqb[1]));
            const Frag<T> aakf[2] = {to_frag<T>(aak[0]), to_frag<T>(aak[1])};
            if (p.ws.TM) st_pair2(reinterpret_cast<T*>(slot + L::AKB), aakf[0], aakf[1]);
            __builtin_amdgcn_sched_barrier(0);
            gated();
            // v, turned, of all value tiles
            char* const sV = slot + L::VTT;
            static_assert(ROWS_SCRATCH <= VT * TILE * (int)sizeof(T), "");
            Frag<T> vT[VT];
#pragma unroll
            for (int j = 0; j < 2; ++j) rows_to_tiles(sV, l, xv[j], vT[2 * j], vT[2 * j + 1]);
#pragma unroll
            for (int j = 0; j < VT; ++j) {
                if (len < CH) mask(vT[j], rowok);
                vT[j] = transpose(vT[j], ident);
                st_frag(reinterpret_cast<T*>(sV) + j * TILE + 4 * l, vT[j]);
            }
            next_first();
            // ---- while the lead solves: A_ak v, and the rows the consumers left in the outbox for the chunk the slot held (they write the
            // outbox again only after both signals at the end)
            Frag<T> mT[VT][2];
#pragma unroll
            for (int j = 0; j < VT; ++j)
#pragma unroll
                for (int r = 0; r < 2; ++r) mT[j][r] = to_frag<T>(mm(vT[j], aakf[r], zero4()));
            __builtin_amdgcn_sched_barrier(0);
            if (it > 0) copy_out(prev_cid, 0, std::integral_constant<int, CH>());
            alive &= wait_ge(f_inv, it + 1, f_abort);
            Frag<T> tm[2][2];
#pragma unroll
            for (int s = 0; s < 2; ++s) ld_pair(sPub + s * PAIR, tm[s][0], tm[s][1]);
            next_rest();
            form_w(tm);
            // ---- u = Tm (A_ak v), transposed (prep.hip, phase D) ---------------------------------------------------------
#pragma unroll
            for (int j = 0; j < VT; ++j) {
                Frag<T> fu[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) fu[s] = to_frag<T>(mm2(mT[j][0], mT[j][1], tm[s][0], tm[s][1], zero4()));
                st_pair2(reinterpret_cast<T*>(slot + L::UT) + j * PAIR, fu[0], fu[1]);
            }
        }
        signal_add(f_ready);
        __builtin_amdgcn_s_setprio(0);
        prev_cid = cid;
    }
    if (!alive) {
        if (l == 0) *a.err = FUSED_ABORTED + 1;
        return;
    }
    // the last chunk's rows, half by each wave
    if (FWD && it > 0) {
        if (!wait_ge(f_consumed, VT * it, f_abort)) { if (l == 0) *a.err = FUSED_ABORTED + 1; return; }
        copy_out(prev_cid, half * (CH / 2), std::integral_constant<int, CH / 2>());
    }
}

// ---- producers of the backward pass's kernels ----------------------------------------------------------------------
// The same pairs, slots and shares of a chunk, with the score tiles' results read from the record: nothing is exchanged
// between the waves of a pair and nothing is solved, a wave forms the gated copies, w and (checkpoint kernel) u of its own
// tiles.  What is left is mostly traffic (29 KB a chunk and head each, at K = V = 64): a wave requests the whole of its next
// chunk as soon as this one's is unpacked, long before it waits for the slot, and holds its results in registers until then.
template <typename T, bool GKF32, int K, int V, int MODE, bool HD>
__device__ __forceinline__ void fused_replay(const FusedArgs<T>& a, char* smem, int n, int h, int seg, int s0, int s1, int pp, int half) {
    static_assert(K == 64 && sizeof(T) == 2 && V % 32 == 0, "a producer pair holds all channels of a chunk: K = 64, 2-byte elements");
    typedef FusedLds<T, K, V, MODE> L;
    constexpr bool REV = MODE == FUSED_REV;
    static_assert(REV || MODE == FUSED_CKPT, "the backward pass's kernels");
    constexpr int VT = V / 16, KT2 = K / 32, KH = 2, VH = VT / 2;
    constexpr BlkF BF = L::BF;
    constexpr SlotB SB = L::SB;
    const ChunkArgs<T>& p = a.c;
    int* const flags = reinterpret_cast<int*>(smem + L::FLAGS);
    int* const f_ready = flags + pp, * const f_consumed = flags + 4 + pp, * const f_abort = flags + 8;
    int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H;
    // (The read-first-lane keeps the optimiser from turning "load, splat" into a vector load of the kernel argument: that
    // ties it to its neighbour st.cu in one memory object, which then goes to LDS, and what depends on st.cu becomes
    // per-lane control flow that reads the absent table of an unpacked batch.)
    const float scale = __int_as_float(uniform(__float_as_int(p.scale)));
    const int nst = s1 - s0;
    const int kt0 = half * KH, vt0 = half * VH;
    int64_t bos, eos;
    seq_bounds(p.st, n, bos, eos);
    int c0, c1;
    seq_chunks(p.st, n, c0, c1);

    // the wave's share of a chunk's inputs as loaded (see fused_producer), and the record's tiles
    i32x4 xq, xk, xa[2], xb[2], xv, xdo, xok, xtm[2], xaq;
    typename GkRaw<T, GKF32>::rows xg, xog;
    T nbeta;
    char* const sX = smem + L::ROWS + (2 * pp + half) * ROWS_SCRATCH;
    static_assert(K / 2 == 32 && V / 2 == 32, "half a row of any operand is 64 bytes");
    constexpr bool WITH_K = HD || !REV;                   // the reverse kernel needs k only to form a and b from it
    auto request = [&](int t) __attribute__((always_inline)) {
        const int cid = REV ? s1 - 1 - t : s0 + t;
        const int64_t tok0 = bos + (int64_t)(cid - c0) * CH;
        const int len = (int)min((int64_t)CH, eos - tok0);
        const int64_t chw = (int64_t)h * p.st.nch + cid;
        // uniform base + a 32-bit byte offset per lane, formed afresh in every call (hoisted out of the chunk loop they would
        // be held in registers through all of it); rows past the end alias the last valid row and are masked at use
        int ll = l;
        asm volatile("" : "+v"(ll));
        const uint32_t row = (uint32_t)min(ll >> 2, max(len, 1) - 1), last = (uint32_t)(max(len, 1) - 1), piece = 16 * (ll & 3);
        constexpr uint32_t ES = sizeof(T), GS = GKF32 ? 4 : 2;
        const uint32_t qo = (row * (uint32_t)(H * K) + 16 * kt0) * ES + piece, ao = (row * (uint32_t)(RANK * H * K) + 16 * kt0) * ES + piece;
        const uint32_t vo = (row * (uint32_t)(H * V) + 16 * vt0) * ES + piece, lo = (uint32_t)ll * 16;
        const int64_t qb = (tok0 * H + h) * K, ab = (tok0 * RANK * H + h) * K, vb = (tok0 * H + h) * V;
        const char* gkp = reinterpret_cast<const char*>(p.gk) + qb * GS;
        auto rows = [](const T* b, uint32_t off) __attribute__((always_inline)) { return *reinterpret_cast<const i32x4*>(at(b, off)); };
        GkRaw<T, GKF32>::load(gkp, ll, row * (uint32_t)(H * K) + 16 * kt0, xg);
        if (WITH_K) xk = rows(p.k + qb, qo);
        if (HD) {
            const uint32_t other = 16 * (KH - kt0);
            nbeta = *at(p.beta + tok0 * H + h, min((uint32_t)(ll & 15), last) * (uint32_t)H * ES);
            GkRaw<T, GKF32>::load(gkp, ll, row * (uint32_t)(H * K) + other, xog);
            xok = rows(p.k + qb, qo + (other - 16 * kt0) * ES);
        } else {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                xa[r] = rows(p.a + ab, ao + r * (uint32_t)(H * K) * ES);
                xb[r] = rows(p.b + ab, ao + r * (uint32_t)(H * K) * ES);
            }
        }
        if (REV) xq = rows(p.q + qb, qo);
        else xv = rows(p.v + vb, vo);
        xdo = rows(p.dout + vb, vo);
        const T* tm = p.ws.TM + chw * 1024;
        xtm[0] = rows(tm, lo);
        xtm[1] = rows(tm + PAIR, lo);
        xaq = rows(a.aq + chw * 1024 + (REV ? PAIR : 0), lo);
    };
    auto mask = [](Frag<T>& f, bool ok) __attribute__((always_inline)) { f.v = ok ? f.v : zero_frag<T>().v; };
    auto mask_gk = [](typename GkRaw<T, GKF32>::type& x, bool ok) __attribute__((always_inline)) { GkRaw<T, GKF32>::mask(x, ok); };
    if (pp < nst) request(pp);

    int it = 0;
    for (int t = pp; t < nst; t += FNP, ++it) {
        const int cid = REV ? s1 - 1 - t : s0 + t;
        const int64_t tok0 = bos + (int64_t)(cid - c0) * CH;
        const int len = (int)min((int64_t)CH, eos - tok0);
        asm volatile("" : "+v"(l));                       // lane-only values formed afresh for every chunk (see fused_producer)
        g = l >> 4;
        c = l & 15;
        char* slot;
        {
            int so = pp * L::SLOT;
            asm volatile("" : "+s"(so));
            slot = smem + so;
        }
        const Frag<T> ident = ident_of<T>(g, c);
        const bool rowok = c < len;
        Frag<T> nq[KH], nk[KH], na[2][KH], nb[2][KH], nv[VH], ndo[VH], ok_[KH], ntm[2][2], naq[2];
        typename GkRaw<T, GKF32>::type ng[KH], og[KH];
        GkRaw<T, GKF32>::tiles(sX, l, xg, ng);
        if (WITH_K) rows_to_tiles(sX, l, xk, nk[0], nk[1]);
        if (HD) {
            GkRaw<T, GKF32>::tiles(sX, l, xog, og);
            rows_to_tiles(sX, l, xok, ok_[0], ok_[1]);
        } else {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                rows_to_tiles(sX, l, xa[r], na[r][0], na[r][1]);
                rows_to_tiles(sX, l, xb[r], nb[r][0], nb[r][1]);
            }
        }
        if (REV) rows_to_tiles(sX, l, xq, nq[0], nq[1]);
        else rows_to_tiles(sX, l, xv, nv[0], nv[1]);
        rows_to_tiles(sX, l, xdo, ndo[0], ndo[1]);
        auto pair = [](i32x4 x, Frag<T>& f0, Frag<T>& f1) __attribute__((always_inline)) {
            const s16x8 y = __builtin_bit_cast(s16x8, x);
            f0.v = __builtin_shufflevector(y, y, 0, 1, 2, 3);
            f1.v = __builtin_shufflevector(y, y, 4, 5, 6, 7);
        };
        pair(xtm[0], ntm[0][0], ntm[0][1]);
        pair(xtm[1], ntm[1][0], ntm[1][1]);
        pair(xaq, naq[0], naq[1]);
        const T bt = nbeta;
        // (everything requested has arrived: the next chunk's inputs may be)
        __builtin_amdgcn_sched_barrier(0);
        if (t + FNP < nst) request(t + FNP);
        __builtin_amdgcn_sched_barrier(0);
        if (len < CH) {
#pragma unroll
            for (int j = 0; j < KH; ++j) {
                mask_gk(ng[j], rowok);
                if (WITH_K) mask(nk[j], rowok);
                if (HD) { mask_gk(og[j], rowok); mask(ok_[j], rowok); }
                else { mask(na[0][j], rowok); mask(na[1][j], rowok); mask(nb[0][j], rowok); mask(nb[1][j], rowok); }
                if (REV) mask(nq[j], rowok);
            }
#pragma unroll
            for (int j = 0; j < VH; ++j) {
                if (!REV) mask(nv[j], rowok);
                mask(ndo[j], rowok);
            }
        }
        float beta_t = 0.f, s_t = 0.f;
        if (HD) {
            beta_t = rowok ? ld_elem(&bt) : 0.f;
#pragma unroll
            for (int j = 0; j < KH; ++j) {
                const f32x4 g4 = GkRaw<T, GKF32>::value(ng[j]), gx = GkRaw<T, GKF32>::value(og[j]);
                const f32x4 k4 = to_f32(nk[j]), kx = to_f32(ok_[j]);
                const f32x4 kf = k4 * k4 * exp4<T>(g4) + kx * kx * exp4<T>(gx);
                s_t += kf[0] + kf[1] + kf[2] + kf[3];
            }
            s_t = sum_groups(s_t);
            if (!REV && half == 0 && g == 0) p.ws.SUM[((int64_t)h * p.st.nch + cid) * CH + c] = s_t;
        }
        // ---- gated copies of the own channel tiles (prep.hip, phase C) ---------------------------------------------------
        Frag<T> agT[2][KH], fb[2][KH], fx[KH];            // fb, fx: bg^T, kg^T (checkpoint kernel); bg, qg^T (reverse kernel)
        f32x4 egl[KH];
#pragma unroll
        for (int j = 0; j < KH; ++j) {
            const f32x4 g4 = GkRaw<T, GKF32>::value(ng[j]), one = {1.f, 1.f, 1.f, 1.f};
            const f32x4 gi = scan16_incl(g4), egi = exp4<T>(gi), edn = exp4<T>(bcast16<CH - 1>(gi) - gi);
            const f32x4 ege = prev_token(egi, one);
            egl[j] = bcast16<CH - 1>(egi);
            Frag<T> ra[2], rb[2];
            if (HD) {
                const f32x4 kk = to_f32(nk[j]), f4 = exp4<T>(g4);
                ra[0] = to_frag<T>(kk * (-beta_t));
                ra[1] = to_frag<T>(kk * ((beta_t * s_t - f4) * beta_t));
                rb[0] = to_frag<T>(f4 * kk);
                rb[1] = nk[j];
            } else {
#pragma unroll
                for (int r = 0; r < 2; ++r) { ra[r] = na[r][j]; rb[r] = nb[r][j]; }
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                agT[r][j] = transpose(to_frag<T>(to_f32(ra[r]) * ege), ident);
                fb[r][j] = to_frag<T>(to_f32(rb[r]) * edn);
                if (!REV) fb[r][j] = transpose(fb[r][j], ident);
            }
            if constexpr (REV) fx[j] = transpose(to_frag<T>(to_f32(nq[j]) * egi * scale), ident);
            else fx[j] = transpose(to_frag<T>(to_f32(nk[j]) * edn), ident);
        }
        // ---- w = Tm ag for the own channel tiles (reverse kernel: w^T), u = Tm (A_ak v) for the own value tiles -----------
        Frag<T> tm[2][2], fw[2][KH], vT[VH], doT[VH], fu[VH][2], aq[2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int r = 0; r < 2; ++r) tm[s][r] = transpose(ntm[s][r], ident);
#pragma unroll
        for (int s = 0; s < 2; ++s) aq[s] = REV ? transpose(naq[s], ident) : naq[s];
#pragma unroll
        for (int j = 0; j < VH; ++j) {
            doT[j] = transpose(ndo[j], ident);
            if (!REV) vT[j] = transpose(nv[j], ident);
        }
#pragma unroll
        for (int j = 0; j < KH; ++j)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                fw[s][j] = to_frag<T>(REV ? mm2(agT[0][j], agT[1][j], tm[s][0], tm[s][1], zero4()) : mm2(tm[s][0], tm[s][1], agT[0][j], agT[1][j], zero4()));
            }
        if (!REV) {
#pragma unroll
            for (int j = 0; j < VH; ++j) {
                const Frag<T> mT[2] = {to_frag<T>(mm(vT[j], aq[0], zero4())), to_frag<T>(mm(vT[j], aq[1], zero4()))};
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    fu[j][s] = to_frag<T>(mm2(mT[0], mT[1], tm[s][0], tm[s][1], zero4()));
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // ---- the slot --------------------------------------------------------------------------------------------------------
        if (!wait_ge(f_consumed, VT * it, f_abort)) { if (l == 0) *a.err = FUSED_ABORTED + 1; return; }
        T* const sW = reinterpret_cast<T*>(slot + (REV ? SB.W : BF.W)), * const sB = reinterpret_cast<T*>(slot + (REV ? SB.BGT : BF.BGT));
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            // the operand of the v_new products pairs two channel tiles, that of the state update the two ranks of a channel tile
            if (REV) {
                st_pair2(sW + (kt0 + s) * PAIR, fw[0][s], fw[1][s]);
                st_pair2(sB + (s * KT2 + half) * PAIR, fb[s][0], fb[s][1]);
            } else {
                st_pair2(sW + (s * KT2 + half) * PAIR, fw[s][0], fw[s][1]);
                st_pair2(sB + (kt0 + s) * PAIR, fb[0][s], fb[1][s]);
            }
        }
        st_pair2(reinterpret_cast<T*>(slot + (REV ? SB.QGT : BF.KGT)) + half * PAIR, fx[0], fx[1]);
        if (REV && half == 0) st_pair2(reinterpret_cast<T*>(slot + SB.AQBT), aq[0], aq[1]);
        if (c == 0) {
#pragma unroll
            for (int j = 0; j < KH; ++j) *reinterpret_cast<f32x4*>(slot + (REV ? SB.EGL : BF.EGL) + (16 * (kt0 + j) + 4 * g) * 4) = egl[j];
        }
#pragma unroll
        for (int j = 0; j < VH; ++j) {
            st_frag(reinterpret_cast<T*>(slot + L::DOT) + (vt0 + j) * TILE + 4 * l, doT[j]);
            if (!REV) {
                st_frag(reinterpret_cast<T*>(slot + L::VTT) + (vt0 + j) * TILE + 4 * l, vT[j]);
                st_pair2(reinterpret_cast<T*>(slot + L::UT) + (vt0 + j) * PAIR, fu[j][0], fu[j][1]);
            }
        }
        signal_add(f_ready);
    }
}

// ---- consumers, forward direction ----------------------------------------------------------------------------------
// Fragment-order records in the workspace (256 fp32 per tile, lane l owns elements 4l..4l+3), per (sequence, head,
// segment):
//   sloc  [V/16][K/16] tiles  F(S^T): the state leaving the segment (started from h0 in segment 0, from zero otherwise)
//   mseg  [K/16][K/16] tiles  the segment's transition M (segments > 0): tile (kt, k't) = F(M block), rows k, inner k'
//   mt    [K/16][K/16] tiles  the same with the blocks transposed, rows k', inner k (part of the record)
//   rseg  [V/16][K/16] tiles  F(R^T), R = sum_t G_t^T do_t (checkpoint kernel, segments > 0)
//   sin   [V/16][K/16] tiles  F(S_in^T): the state entering the segment (segments > 0)
template <typename T, int K, int V, int MODE>
__device__ __forceinline__ void fused_consumer_fwd(const FusedArgs<T>& a, char* smem, int n, int h, int seg, int s0, int s1, int wv) {
    typedef FusedLds<T, K, V, MODE> L;
    constexpr bool FWD = MODE == FUSED_FWD;
    constexpr int KT = K / 16, VT = V / 16, KT2 = KT / 2;
    static_assert(KT == VT, "consumer j owns column block j of the state and of the transition matrix");
    constexpr BlkF BF = L::BF;
    const ChunkArgs<T>& p = a.c;
    int* const flags = reinterpret_cast<int*>(smem + L::FLAGS);
    const int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H, vt = wv;
    const int nst = s1 - s0;
    const bool pblk = seg > 0;                            // uniform over the workgroup
    const int64_t rec = ((int64_t)n * H + h) * a.nseg + seg;
    const int64_t soff = ((int64_t)n * H + h) * K * V + 16 * vt + c;

    // state block: lane (g,c) reg i of tile kt = S[16kt + 4g + i][16vt + c]; likewise M with column 16vt + c
    f32x4 S[KT], M[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
        S[kt] = zero4();
#pragma unroll
        for (int i = 0; i < 4; ++i) M[kt][i] = (16 * kt + 4 * g + i == 16 * vt + c) ? 1.f : 0.f;
    }
    if (seg == 0 && p.h0) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) S[kt][i] = p.h0[soff + (int64_t)(16 * kt + 4 * g + i) * V];
    }

    for (int t = 0; t < nst; ++t) {
        const int pp = t & (FNP - 1), it = t / FNP;
        if (!wait_ge(&flags[pp], 2 * (it + 1), &flags[8])) { if (l == 0) *a.err = FUSED_ABORTED + 2; return; }
        const char* slot = smem + pp * L::SLOT;
        const int cid = s0 + t;
        const int64_t chw = (int64_t)h * p.st.nch + cid;
        const T* sW = reinterpret_cast<const T*>(slot + BF.W);
        const T* sBGT = reinterpret_cast<const T*>(slot + BF.BGT);
        const T* sKGT = reinterpret_cast<const T*>(slot + BF.KGT);
        const float* sEGL = reinterpret_cast<const float*>(slot + BF.EGL);
        Frag<T> w[2][KT], qg[KT], aqb[2], aqk, kgt[KT], bgt[2][KT], ut[2], vtt;
        f32x4 egl[KT];
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) {
            ld_pair(sW + (0 * KT2 + kp) * PAIR, w[0][2 * kp], w[0][2 * kp + 1]);
            ld_pair(sW + (1 * KT2 + kp) * PAIR, w[1][2 * kp], w[1][2 * kp + 1]);
        }
        ld_pair(reinterpret_cast<const T*>(slot + L::UT) + wv * PAIR, ut[0], ut[1]);
        vtt = ld_tile(reinterpret_cast<const T*>(slot + L::VTT) + wv * TILE);
        if (FWD || pblk) {
#pragma unroll
            for (int kp = 0; kp < KT2; ++kp) ld_pair(reinterpret_cast<const T*>(slot + BF.QG) + kp * PAIR, qg[2 * kp], qg[2 * kp + 1]);
            ld_pair(reinterpret_cast<const T*>(slot + BF.AQB), aqb[0], aqb[1]);
        }
        if (FWD) aqk = ld_tile(reinterpret_cast<const T*>(slot + BF.AQK));
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) {
            ld_pair(sKGT + kp * PAIR, kgt[2 * kp], kgt[2 * kp + 1]);
            ld_pair(sBGT + (2 * kp) * PAIR, bgt[0][2 * kp], bgt[1][2 * kp]);
            ld_pair(sBGT + (2 * kp + 1) * PAIR, bgt[0][2 * kp + 1], bgt[1][2 * kp + 1]);
            egl[2 * kp] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (2 * kp) + 4 * g);
            egl[2 * kp + 1] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (2 * kp + 1) + 4 * g);
        }

        // ---- the state's column block: the stand-alone scan's step (scan_impl.cuh), operation for operation ---------
        Frag<T> sb[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) sb[kt] = to_frag<T>(S[kt]);
        // first what is one product a sum, then the rest in twos: one change of instruction for all accumulators (see mm2)
        f32x4 x[KT + 1];
        x[KT] = FWD ? mm(aqk, vtt, zero4()) : zero4();
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) x[kt] = mm(vtt, kgt[kt], S[kt] * egl[kt]);
        settle<T>(x);
        f32x4 vn[2] = {to_f32(ut[0]), to_f32(ut[1])}, o = x[KT];
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) {
            vn[0] = mm2(sb[2 * kp], sb[2 * kp + 1], w[0][2 * kp], w[0][2 * kp + 1], vn[0]);
            vn[1] = mm2(sb[2 * kp], sb[2 * kp + 1], w[1][2 * kp], w[1][2 * kp + 1], vn[1]);
        }
        if (FWD) {
#pragma unroll
            for (int kp = 0; kp < KT2; ++kp) o = mm2(qg[2 * kp], qg[2 * kp + 1], sb[2 * kp], sb[2 * kp + 1], o);
        }
        const Frag<T> vnb[2] = {to_frag<T>(vn[0]), to_frag<T>(vn[1])};
        if (p.ws.TM) {
            // the record, a tile pair by each wave: (I - A_ab)^-1, A_ak, A_qb
            static_assert(VT == 4, "four tile pairs");
            const int src = wv < 2 ? L::TMB + wv * PAIR * (int)sizeof(T) : wv == 2 ? L::AKB : BF.AQB;
            T* dst = (wv < 2 ? p.ws.TM : a.aq) + chw * 1024 + (wv & 1) * PAIR;
            Frag<T> t0, t1;
            ld_pair(reinterpret_cast<const T*>(slot + src), t0, t1);
            st_pair2(dst, t0, t1);
        }
        if (FWD) {
            o = mm2(aqb[0], aqb[1], vnb[0], vnb[1], o);
            char* ob = smem + pp * L::SLOT + L::OBOX + c * L::OROW;
            if (seg == 0) st_frag(reinterpret_cast<T*>(ob) + 16 * wv + 4 * g, to_frag<T>(o));
            else *reinterpret_cast<f32x4*>(ob + (16 * wv + 4 * g) * 4) = o;
        }
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) S[kt] = mm2(vnb[0], vnb[1], bgt[0][kt], bgt[1][kt], x[kt]);
        // ---- the transition matrix's column block: the same update without the chunk's own input --------------------
        if (pblk) {
            Frag<T> mb[KT];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) mb[kt] = to_frag<T>(M[kt]);
            f32x4 vp[2] = {zero4(), zero4()};
#pragma unroll
            for (int kp = 0; kp < KT2; ++kp) {
                vp[0] = mm2(mb[2 * kp], mb[2 * kp + 1], w[0][2 * kp], w[0][2 * kp + 1], vp[0]);
                vp[1] = mm2(mb[2 * kp], mb[2 * kp + 1], w[1][2 * kp], w[1][2 * kp + 1], vp[1]);
            }
            f32x4 G = zero4();
#pragma unroll
            for (int kp = 0; kp < KT2; ++kp) G = mm2(qg[2 * kp], qg[2 * kp + 1], mb[2 * kp], mb[2 * kp + 1], G);
            const Frag<T> vpb[2] = {to_frag<T>(vp[0]), to_frag<T>(vp[1])};
            G = mm2(aqb[0], aqb[1], vpb[0], vpb[1], G);
            const Frag<T> Gf = to_frag<T>(G);             // rows token, inner k' (the block's columns)
            if (FWD) st_frag(reinterpret_cast<T*>(smem + pp * L::SLOT + L::GBOX + c * L::GROW) + 16 * wv + 4 * g, Gf);
            else st_frag(a.gw + chw * (CH * K) + gw_at(wv, g, c), Gf);
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) M[kt] = mm2(vpb[0], vpb[1], bgt[0][kt], bgt[1][kt], M[kt] * egl[kt]);
        }
        signal_add(&flags[4 + pp]);
    }

    // ---- what the segment leaves behind ------------------------------------------------------------------------------
    if (a.nseg == 1) {
        if (FWD && p.ht) {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) p.ht[soff + (int64_t)(16 * kt + 4 * g + i) * V] = S[kt][i];
        }
        return;
    }
    float* sloc = a.sloc + rec * (K * V);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) *reinterpret_cast<f32x4*>(sloc + (vt * KT + kt) * TILE + 4 * l) = S[kt];
    if (pblk) {
        float* mseg = a.mseg + rec * (K * K);
        const Frag<float> identf = ident_frag<float>();
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            Frag<float> f;
            f.v = M[kt];
            if (a.mt) *reinterpret_cast<f32x4*>(a.mt + rec * (K * K) + (kt * KT + wv) * TILE + 4 * l) = f.v;
            f = transpose(f, identf);                     // exact: fp32 products with ones and zeros
            *reinterpret_cast<f32x4*>(mseg + (kt * KT + wv) * TILE + 4 * l) = f.v;
        }
    }
}

// ---- consumers, checkpoint kernel ------------------------------------------------------------------------------------
// The state walk of the forward direction from the true entering state, leaving the state entering every chunk for
// chunk_grad, and R from the record's G.
// W_GLOBAL: chunk_grad reads u and w from the workspace where it cannot rebuild them (chunk_grad_body.inc: REBUILD_W).  (With the HDLA
// parameterisation it rebuilds them too, from the sums over channels that the producers leave.)
template <typename T, int K, int V, bool W_GLOBAL>
__device__ __forceinline__ void fused_consumer_ckpt(const FusedArgs<T>& a, char* smem, int n, int h, int seg, int s0, int s1, int wv) {
    typedef FusedLds<T, K, V, FUSED_CKPT> L;
    constexpr int KT = K / 16, VT = V / 16, KT2 = KT / 2;
    static_assert(KT == VT, "consumer j owns column block j of the state and of G");
    constexpr BlkF BF = L::BF;
    const ChunkArgs<T>& p = a.c;
    int* const flags = reinterpret_cast<int*>(smem + L::FLAGS);
    const int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H, vt = wv;
    const int nst = s1 - s0;
    const bool later = seg > 0;                           // uniform over the workgroup
    const int64_t rec = ((int64_t)n * H + h) * a.nseg + seg;
    const int64_t soff = ((int64_t)n * H + h) * K * V + 16 * vt + c;

    f32x4 S[KT], R[VT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) S[kt] = zero4();
#pragma unroll
    for (int j = 0; j < VT; ++j) R[j] = zero4();
    if (later) {
        const float* sin = a.sin + rec * (K * V);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) S[kt] = *reinterpret_cast<const f32x4*>(sin + (vt * KT + kt) * TILE + 4 * l);
    } else if (p.h0) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) S[kt][i] = p.h0[soff + (int64_t)(16 * kt + 4 * g + i) * V];
    }
    const Frag<T> ident = ident_frag<T>();
    // rows token, inner k' (the block's columns), requested a chunk ahead
    const T* gw = a.gw + ((int64_t)h * p.st.nch + s0) * (CH * K) + gw_at(wv, g, c);
    Frag<T> gn = zero_frag<T>();
    if (later) gn = ld_frag(gw);

    for (int t = 0; t < nst; ++t) {
        const int pp = t & (FNP - 1), it = t / FNP;
        if (!wait_ge(&flags[pp], 2 * (it + 1), &flags[8])) { if (l == 0) *a.err = FUSED_ABORTED + 2; return; }
        const char* slot = smem + pp * L::SLOT;
        const int cid = s0 + t;
        const int64_t chw = (int64_t)h * p.st.nch + cid;
        const T* sW = reinterpret_cast<const T*>(slot + BF.W);
        const T* sBGT = reinterpret_cast<const T*>(slot + BF.BGT);
        const T* sKGT = reinterpret_cast<const T*>(slot + BF.KGT);
        const float* sEGL = reinterpret_cast<const float*>(slot + BF.EGL);
        Frag<T> w[2][KT], kgt[KT], bgt[2][KT], ut[2], vtt, dot[VT];
        f32x4 egl[KT];
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) {
            ld_pair(sW + (0 * KT2 + kp) * PAIR, w[0][2 * kp], w[0][2 * kp + 1]);
            ld_pair(sW + (1 * KT2 + kp) * PAIR, w[1][2 * kp], w[1][2 * kp + 1]);
        }
        ld_pair(reinterpret_cast<const T*>(slot + L::UT) + wv * PAIR, ut[0], ut[1]);
        vtt = ld_tile(reinterpret_cast<const T*>(slot + L::VTT) + wv * TILE);
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) {
            ld_pair(sKGT + kp * PAIR, kgt[2 * kp], kgt[2 * kp + 1]);
            ld_pair(sBGT + (2 * kp) * PAIR, bgt[0][2 * kp], bgt[1][2 * kp]);
            ld_pair(sBGT + (2 * kp + 1) * PAIR, bgt[0][2 * kp + 1], bgt[1][2 * kp + 1]);
            egl[2 * kp] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (2 * kp) + 4 * g);
            egl[2 * kp + 1] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (2 * kp + 1) + 4 * g);
        }
        Frag<T> gt = gn;
        if (later) {
#pragma unroll
            for (int j = 0; j < VT; ++j) dot[j] = ld_tile(reinterpret_cast<const T*>(slot + L::DOT) + j * TILE);
            gt = transpose(gn, ident);
            if (t + 1 < nst) gn = ld_frag(gw + (int64_t)(t + 1) * (CH * K));
        }
        // the stand-alone scan's step (scan_impl.cuh), operation for operation
        Frag<T> sb[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) sb[kt] = to_frag<T>(S[kt]);
        f32x4 x[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) x[kt] = mm(vtt, kgt[kt], S[kt] * egl[kt]);
        settle<T>(x);
        f32x4 vn[2] = {to_f32(ut[0]), to_f32(ut[1])};
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) {
            vn[0] = mm2(sb[2 * kp], sb[2 * kp + 1], w[0][2 * kp], w[0][2 * kp + 1], vn[0]);
            vn[1] = mm2(sb[2 * kp], sb[2 * kp + 1], w[1][2 * kp], w[1][2 * kp + 1], vn[1]);
        }
        const Frag<T> vnb[2] = {to_frag<T>(vn[0]), to_frag<T>(vn[1])};
        T* hc = p.ws.HC + chw * (K * V) + vt * PAIR;
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) st_pair2_past(hc + kp * (VT * PAIR), sb[2 * kp], sb[2 * kp + 1]);
        if (W_GLOBAL) {
            static_assert(2 * KT2 == VT, "one pair of w per consumer");
            st_pair2(p.ws.UT + (chw * VT + vt) * PAIR, ut[0], ut[1]);
            T* wg = p.ws.W + chw * (p.ws.sa_stride / (int)sizeof(T));
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int kp = 0; kp < KT2; ++kp)
                    if (wv == s * KT2 + kp) st_pair2(wg + (s * KT2 + kp) * PAIR, w[s][2 * kp], w[s][2 * kp + 1]);
        }
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) S[kt] = mm2(vnb[0], vnb[1], bgt[0][kt], bgt[1][kt], x[kt]);
        if (later) {
            // R[k'][v] += sum_tok G[tok][k'] do[tok][v]
#pragma unroll
            for (int j = 0; j < VT; ++j) R[j] = mm(gt, dot[j], R[j]);
        }
        signal_add(&flags[4 + pp]);
    }
    if (later) {
        float* rseg = a.rseg + rec * (K * V);
        const Frag<float> identf = ident_frag<float>();
#pragma unroll
        for (int j = 0; j < VT; ++j) {
            Frag<float> f;
            f.v = R[j];
            f = transpose(f, identf);
            *reinterpret_cast<f32x4*>(rseg + (j * KT + wv) * TILE + 4 * l) = f.v;
        }
    }
}

// ---- consumers, reverse direction ------------------------------------------------------------------------------------
template <typename T, int K, int V>
__device__ __forceinline__ void fused_consumer_rev(const FusedArgs<T>& a, char* smem, int n, int h, int seg, int s0, int s1, int wv) {
    typedef FusedLds<T, K, V, FUSED_REV> L;
    constexpr int KT = K / 16, VT = V / 16, KT2 = KT / 2;
    constexpr SlotB B = L::SB;
    const ChunkArgs<T>& p = a.c;
    int* const flags = reinterpret_cast<int*>(smem + L::FLAGS);
    const int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H, vt = wv;
    const int nst = s1 - s0;
    const int64_t soff = ((int64_t)n * H + h) * K * V + 16 * vt + c;

    f32x4 dS[KT];   // lane (g,c) reg i of tile kt = dS[16kt + 4g + i][16vt + c]
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) dS[kt] = zero4();
    if (p.dht) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) dS[kt][i] = p.dht[soff + (int64_t)(16 * kt + 4 * g + i) * V];
    }
    // The gradient entering this segment from the right: through the later segments, last one first,
    //   dS <- M_s^T dS + R_s   (as fragments: X^T <- X^T Q^T + A^T, tile (in, out) of the record at index in * KT + out).
    // Nothing waits for the producers here, so only the chain's own latency counts: the records of up to CHAIN_STAGE
    // segments are requested at once, a quarter of each transition record by each of the four consumer waves, which
    // share them through LDS as split operands; the consumers meet at two counters of their own (the producers are
    // at work meanwhile, so no workgroup barrier).
    {
        static_assert(VT == 4 && KT == 4, "a quarter of a record per consumer wave");
        constexpr int NQ = KT * KT / 4, STG = L::CHAIN_STAGE;
        // (one lane address for the whole area, opaque to the compiler: the area lies beyond the reach of an LDS
        // instruction's immediate offset from zero, and a register per tile address would not fit)
        int sMo = L::CHAIN + 4 * l * (int)sizeof(T);
        asm volatile("" : "+v"(sMo));
        T* const sM = reinterpret_cast<T*>(smem + sMo);
        const int64_t rec0 = ((int64_t)n * H + h) * a.nseg;
        int batch = 0, s = a.nseg - 1;
        while (s > seg) {
            int step[STG], ns = 0, q0, q1;
#pragma unroll
            for (int b = 0; b < STG; ++b) {
                step[b] = 0;
                while (s > seg) {
                    seg_range(p.st, n, a.nseg, s, q0, q1);
                    if (q1 > q0) break;
                    --s;
                }
                if (s > seg) { step[b] = s--; ns = b + 1; }
            }
            f32x4 mq[STG][NQ], add[STG][KT];
#pragma unroll
            for (int b = 0; b < STG; ++b) {
                if (b < ns) {
                    const float* mrec = a.mt + (rec0 + step[b]) * (K * K) + wv * NQ * TILE + 4 * l;
#pragma unroll
                    for (int i = 0; i < NQ; ++i) mq[b][i] = *reinterpret_cast<const f32x4*>(mrec + i * TILE);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < STG; ++b) {
                if (b < ns) {
                    const float* rrec = a.rseg + (rec0 + step[b]) * (K * V) + vt * KT * TILE + 4 * l;
#pragma unroll
                    for (int kt = 0; kt < KT; ++kt) add[b][kt] = *reinterpret_cast<const f32x4*>(rrec + kt * TILE);
                }
            }
            // every consumer has read the previous round's records out of LDS
            if (batch > 0 && !wait_ge(&flags[25], VT * batch, &flags[8])) { if (l == 0) *a.err = FUSED_ABORTED + 3; return; }
#pragma unroll
            for (int b = 0; b < STG; ++b) {
                if (b < ns) {
#pragma unroll
                    for (int i = 0; i < NQ; ++i) {
                        Split<T> q;
                        split(mq[b][i], q);
                        st_frag(sM + ((b * 2 + 0) * KT * KT + wv * NQ + i) * TILE, q.hi);
                        st_frag(sM + ((b * 2 + 1) * KT * KT + wv * NQ + i) * TILE, q.lo);
                    }
                }
            }
            signal_add(&flags[24]);
            if (!wait_ge(&flags[24], VT * (batch + 1), &flags[8])) { if (l == 0) *a.err = FUSED_ABORTED + 3; return; }
#pragma unroll
            for (int b = 0; b < STG; ++b) {
                if (b < ns) {
                    Split<T> xs[KT];
#pragma unroll
                    for (int kt = 0; kt < KT; ++kt) split(dS[kt], xs[kt]);
#pragma unroll
                    for (int ko = 0; ko < KT; ++ko) {
                        f32x4 acc = add[b][ko];
#pragma unroll
                        for (int ki = 0; ki < KT; ++ki) {
                            Split<T> q;
                            q.hi = ld_frag(sM + ((b * 2 + 0) * KT * KT + ki * KT + ko) * TILE);
                            q.lo = ld_frag(sM + ((b * 2 + 1) * KT * KT + ki * KT + ko) * TILE);
                            acc = mm_split(xs[ki], q, acc);
                        }
                        dS[ko] = acc;
                    }
                }
            }
            signal_add(&flags[25]);
            ++batch;
        }
    }

    for (int t = 0; t < nst; ++t) {
        const int pp = t & (FNP - 1), it = t / FNP;
        if (!wait_ge(&flags[pp], 2 * (it + 1), &flags[8])) { if (l == 0) *a.err = FUSED_ABORTED + 3; return; }
        const char* slot = smem + pp * L::SLOT;
        const int cid = s1 - 1 - t;
        const int64_t chw = (int64_t)h * p.st.nch + cid;
        const T* sWT = reinterpret_cast<const T*>(slot + B.W);
        const T* sBG = reinterpret_cast<const T*>(slot + B.BGT);
        const T* sQGT = reinterpret_cast<const T*>(slot + B.QGT);
        const float* sEGL = reinterpret_cast<const float*>(slot + B.EGL);
        Frag<T> aq[2], bg[2][KT], qgt[KT], wt[2][KT];
        f32x4 egl[KT];
        ld_pair(reinterpret_cast<const T*>(slot + B.AQBT), aq[0], aq[1]);
        const Frag<T> doT = ld_tile(reinterpret_cast<const T*>(slot + L::DOT) + wv * TILE);
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) {
            ld_pair(sBG + (0 * KT2 + kp) * PAIR, bg[0][2 * kp], bg[0][2 * kp + 1]);
            ld_pair(sBG + (1 * KT2 + kp) * PAIR, bg[1][2 * kp], bg[1][2 * kp + 1]);
            ld_pair(sQGT + kp * PAIR, qgt[2 * kp], qgt[2 * kp + 1]);
            ld_pair(sWT + (2 * kp) * PAIR, wt[0][2 * kp], wt[1][2 * kp]);
            ld_pair(sWT + (2 * kp + 1) * PAIR, wt[0][2 * kp + 1], wt[1][2 * kp + 1]);
            egl[2 * kp] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (2 * kp) + 4 * g);
            egl[2 * kp + 1] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (2 * kp + 1) + 4 * g);
        }
        // the stand-alone reverse scan's step (scan_impl.cuh), operation for operation
        Frag<T> dsb[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) dsb[kt] = to_frag<T>(dS[kt]);
        // (products one by one before those in twos, as in the forward direction; x: dv_new of both ranks, then the state)
        f32x4 x[2 + KT];
        x[0] = mm(doT, aq[0], zero4());
        x[1] = mm(doT, aq[1], zero4());
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) x[2 + kt] = mm(doT, qgt[kt], dS[kt] * egl[kt]);
        settle<T>(x);
        f32x4 dvn[2] = {x[0], x[1]};
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) {
            dvn[0] = mm2(dsb[2 * kp], dsb[2 * kp + 1], bg[0][2 * kp], bg[0][2 * kp + 1], dvn[0]);
            dvn[1] = mm2(dsb[2 * kp], dsb[2 * kp + 1], bg[1][2 * kp], bg[1][2 * kp + 1], dvn[1]);
        }
        const Frag<T> dvb[2] = {to_frag<T>(dvn[0]), to_frag<T>(dvn[1])};
        T* dhc = p.ws.DHC + chw * (K * V) + vt * PAIR;
        T* dvp = p.ws.DVN + chw * (2 * CH * V) + vt * PAIR;
#pragma unroll
        for (int kp = 0; kp < KT2; ++kp) st_pair2_past(dhc + kp * (VT * PAIR), dsb[2 * kp], dsb[2 * kp + 1]);
        st_pair2_past(dvp, dvb[0], dvb[1]);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) dS[kt] = mm2(dvb[0], dvb[1], wt[0][kt], wt[1][kt], x[2 + kt]);
        signal_add(&flags[4 + pp]);
    }
    if (seg == 0 && p.dh0) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) p.dh0[soff + (int64_t)(16 * kt + 4 * g + i) * V] = dS[kt][i];
    }
}

// ---- the kernel ------------------------------------------------------------------------------------------------------
// grid = (H, nseg, N); block = 64 (V/16 + 2 FNP): waves 0 .. V/16-1 consume, the rest produce in pairs
template <typename T, bool GKF32, int K, int V, int MODE, bool HD>
__global__ __launch_bounds__(64 * (V / 16 + 2 * FNP)) void fused_kernel(FusedArgs<T> a) {
    typedef FusedLds<T, K, V, MODE> L;
    __shared__ __attribute__((aligned(16))) char smem[L::BYTES];
    const int h = blockIdx.x, seg = blockIdx.y;
    const int n = scan_sequence(a.c.st, blockIdx.z);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int s0, s1;
    seg_range(a.c.st, n, a.nseg, seg, s0, s1);
    // an empty segment leaves nothing behind (whoever chains the segments skips it), except that the first one of an
    // empty sequence still passes the state through
    if (s1 <= s0 && seg > 0) return;
    if (threadIdx.x < 32) reinterpret_cast<int*>(smem + L::FLAGS)[threadIdx.x] = 0;
    __syncthreads();
    if (wv < V / 16) {
        if constexpr (MODE == FUSED_REV) fused_consumer_rev<T, K, V>(a, smem, n, h, seg, s0, s1, wv);
        else if constexpr (MODE == FUSED_CKPT) fused_consumer_ckpt<T, K, V, GKF32>(a, smem, n, h, seg, s0, s1, wv);
        else fused_consumer_fwd<T, K, V, MODE>(a, smem, n, h, seg, s0, s1, wv);
    } else {
        const int pp = (wv - V / 16) >> 1, half = (wv - V / 16) & 1;
        if constexpr (L::SOLVES) fused_producer<T, GKF32, K, V, MODE, HD>(a, smem, n, h, seg, s0, s1, pp, half);
        else fused_replay<T, GKF32, K, V, MODE, HD>(a, smem, n, h, seg, s0, s1, pp, half);
    }
}

// ---- forward pass, second kernel: the true entering states, and their part of the output ----------------------------
// grid = (H, nseg * FIXUP_PARTS, N), 256 threads.  blockIdx.y / FIXUP_PARTS = s in 1 .. nseg-1: segment s (chain the
// records of segments 0 .. s-1 into S_in(s), keep it as the boundary record, add G S_in(s) to the segment's local
// outputs); 0: the final state (all segments chained).  The kernel is a chain of dependent steps between two launches,
// so everything is arranged for its latency: all loads that do not depend on the chain are issued at the start (the
// first chunks' operands, the records of up to FIXUP_STAGE chain steps); the transition records, which every wave needs
// whole, are loaded a quarter by each wave and shared through LDS as split operands; wave j chains column block j of
// the state (the blocks are independent); FIXUP_PARTS workgroups share the chunks of a segment, each repeating the
// chain, so that a workgroup's share of the chunks is in flight from the start as well.
// The local outputs and G lie in memory as the waves take them (copy_out): 16.1 -> 12.8 us for 4 x 2048 tokens of 16 heads in four segments,
// where requests for 16 rows had met 16 cache lines each; those two read and o written are 9 at copy rate.
constexpr int FIXUP_PARTS = 2;                            // workgroups that share one segment's chunks (measured: 1, 2, 4 -> 12.8, 12.8, 16.0 us)
constexpr int FIXUP_STAGE = 3;                            // chain steps whose records are in LDS at a time
template <typename T, int K, int V>
__global__ __launch_bounds__(256) void fixup_kernel(FusedArgs<T> a) {
    constexpr int KT = K / 16, VT = V / 16, NB = 2, NQ = KT * KT / 4;
    static_assert(VT == 4 && KT == 4 && sizeof(T) == 2, "one column block per wave, a quarter of a transition record per wave");
    constexpr int OROW = V * (int)sizeof(T) + 16;
    __shared__ __attribute__((aligned(16))) char stage[4][CH * OROW];
    __shared__ __attribute__((aligned(16))) T sS[VT * KT * TILE];          // S_in as operand tiles [vt][kt]
    __shared__ __attribute__((aligned(16))) T sM[FIXUP_STAGE][2][KT * KT * TILE];   // transition records, hi and lo halves
    const ChunkArgs<T>& p = a.c;
    const int h = blockIdx.x;
    const int n = scan_sequence(p.st, blockIdx.z);
    const int ty = (int)blockIdx.y / FIXUP_PARTS, part = (int)blockIdx.y % FIXUP_PARTS;
    const int target = ty == 0 ? a.nseg : ty;                            // chain segments 0 .. target-1
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H, vt = wv;
    int s0 = 0, s1 = 0;
    if (target < a.nseg) {
        seg_range(p.st, n, a.nseg, target, s0, s1);
        // this workgroup's share of the segment's chunks
        const int per = (s1 - s0 + FIXUP_PARTS - 1) / FIXUP_PARTS;
        s0 = min(s0 + part * per, s1);
        s1 = min(s0 + per, s1);
        if (s1 <= s0 || (part > 0 && !a.ol)) return;
    } else if (!p.ht || part > 0) return;
    const int64_t rec0 = ((int64_t)n * H + h) * a.nseg;
    const int64_t soff = ((int64_t)n * H + h) * K * V + 16 * vt + c;

    int c0, c1;
    seq_chunks(p.st, n, c0, c1);
    int64_t bos, eos;
    seq_bounds(p.st, n, bos, eos);
    Frag<T> G[NB][KT];
    f32x4 OLr[NB][VT];
    auto request = [&](int first) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int cid = min(first + 4 * b, s1 - 1);   // past the end: the last chunk again, never used
            const int64_t chw = (int64_t)h * p.st.nch + cid;
            const T* gw = a.gw + chw * (CH * K);
            const float* ol = a.ol + chw * (CH * V) + 4 * l;
#pragma unroll
            for (int kp = 0; kp < KT / 2; ++kp) ld_pair(gw + kp * PAIR, G[b][2 * kp], G[b][2 * kp + 1]);
#pragma unroll
            for (int j = 0; j < VT; ++j) OLr[b][j] = *reinterpret_cast<const f32x4*>(ol + j * TILE);
        }
    };
    const bool outputs = target < a.nseg && a.ol != nullptr;
    if (outputs) request(s0 + wv);

    // S[kt]: lane (g,c) reg i = S[16kt + 4g + i][16vt + c].  Segment 0 ran from the initial state itself; only where it
    // is empty does the chain start from the initial state here.
    f32x4 S[KT];
    int q0, q1;
    seg_range(p.st, n, a.nseg, 0, q0, q1);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
        if (q1 > q0) {
            S[kt] = *reinterpret_cast<const f32x4*>(a.sloc + rec0 * (K * V) + (vt * KT + kt) * TILE + 4 * l);
        } else {
            S[kt] = zero4();
            if (p.h0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) S[kt][i] = p.h0[soff + (int64_t)(16 * kt + 4 * g + i) * V];
            }
        }
    }
    // the chain, FIXUP_STAGE non-empty segments at a time
    int s = 1;
    while (s < target) {
        int step[FIXUP_STAGE], ns = 0;
#pragma unroll
        for (int b = 0; b < FIXUP_STAGE; ++b) {
            step[b] = 0;
            while (s < target) {
                seg_range(p.st, n, a.nseg, s, q0, q1);
                if (q1 > q0) break;
                ++s;
            }
            if (s < target) { step[b] = s++; ns = b + 1; }
        }
        f32x4 mq[FIXUP_STAGE][NQ], add[FIXUP_STAGE][KT];
#pragma unroll
        for (int b = 0; b < FIXUP_STAGE; ++b) {
            if (b < ns) {
                const float* mrec = a.mseg + (rec0 + step[b]) * (K * K) + wv * NQ * TILE + 4 * l;
                const float* srec = a.sloc + (rec0 + step[b]) * (K * V) + vt * KT * TILE + 4 * l;
#pragma unroll
                for (int i = 0; i < NQ; ++i) mq[b][i] = *reinterpret_cast<const f32x4*>(mrec + i * TILE);
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) add[b][kt] = *reinterpret_cast<const f32x4*>(srec + kt * TILE);
            }
        }
        __syncthreads();                                  // the previous round's records have been used
#pragma unroll
        for (int b = 0; b < FIXUP_STAGE; ++b) {
            if (b < ns) {
#pragma unroll
                for (int i = 0; i < NQ; ++i) {
                    Split<T> q;
                    split(mq[b][i], q);
                    st_tile(sM[b][0] + (wv * NQ + i) * TILE, q.hi);
                    st_tile(sM[b][1] + (wv * NQ + i) * TILE, q.lo);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < FIXUP_STAGE; ++b) {
            if (b < ns) {
                // X^T <- X^T Q^T + A^T in split 2-byte products (the error of fp32 products); tile
                // (out, in) of the record is at index out * KT + in
                Split<T> xs[KT];
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) split(S[kt], xs[kt]);
#pragma unroll
                for (int ko = 0; ko < KT; ++ko) {
                    f32x4 acc = add[b][ko];
#pragma unroll
                    for (int ki = 0; ki < KT; ++ki) {
                        Split<T> q;
                        q.hi = ld_tile(sM[b][0] + (ko * KT + ki) * TILE);
                        q.lo = ld_tile(sM[b][1] + (ko * KT + ki) * TILE);
                        acc = mm_split(xs[ki], q, acc);
                    }
                    S[ko] = acc;
                }
            }
        }
    }
    if (target == a.nseg) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) p.ht[soff + (int64_t)(16 * kt + 4 * g + i) * V] = S[kt][i];
        return;
    }
    if (a.sin_out && part == 0) {
        float* so = a.sin_out + (rec0 + target) * (K * V) + vt * KT * TILE;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) *reinterpret_cast<f32x4*>(so + kt * TILE + 4 * l) = S[kt];
    }
    if (!a.ol) return;                                    // chaining only (the backward pass re-deriving the states)
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) st_tile(sS + (vt * KT + kt) * TILE, to_frag<T>(S[kt]));
    __syncthreads();
    Frag<T> Sb[VT][KT];
#pragma unroll
    for (int j = 0; j < VT; ++j)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            // the channels that G's fragment kt has on this lane: 32 (kt / 2) + 8 g + 4 (kt % 2) .. + 3
            const int ch = 8 * g + 4 * (kt & 1);
            Sb[j][kt].v = *reinterpret_cast<const s16x4*>(sS + (j * KT + (kt & ~1) + ch / 16) * TILE + 4 * (ch % 16 / 4 * 16 + c));
        }
    char* const st = stage[wv];
    for (int first = s0 + wv; first < s1; first += 4 * NB) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int cid = first + 4 * b;
            if (cid < s1) {
                const int64_t tok0 = bos + (int64_t)(cid - c0) * CH;
                const int len = (int)min((int64_t)CH, eos - tok0);
#pragma unroll
                for (int j = 0; j < VT; ++j) {
                    f32x4 o = OLr[b][j];
#pragma unroll
                    for (int kt = 0; kt < KT; kt += 2) o = mm2(G[b][kt], G[b][kt + 1], Sb[j][kt], Sb[j][kt + 1], o);
                    st_frag(reinterpret_cast<T*>(st + c * OROW) + 16 * j + 4 * g, to_frag<T>(o));
                }
                // whole rows, 16 bytes a lane (the wave's own staging area: LDS accesses of one wave complete in order)
                constexpr int LPR = V * (int)sizeof(T) / 16, RPI = 64 / LPR;
#pragma unroll
                for (int r0 = 0; r0 < CH; r0 += RPI) {
                    const int r = r0 + l / LPR, e = (l % LPR) * 16;
                    const i32x4 x = *reinterpret_cast<const i32x4*>(st + r * OROW + e);
                    if (r < len) st_past(reinterpret_cast<i32x4*>(reinterpret_cast<char*>(p.o + ((tok0 + r) * H + h) * V) + e), x);
                }
            }
        }
        if (first + 4 * NB < s1) request(first + 4 * NB);
    }
}

}  // namespace hdla
