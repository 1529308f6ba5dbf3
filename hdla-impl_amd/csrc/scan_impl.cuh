// The two inter-chunk state scans: the only sequential part of the chunked operator.
//
// scan_fwd replaces HRDPLR/fwd_triton.py:808-968 (state recurrence, h checkpoints, v_new, final state) and, in
// the forward pass, also HRDPLR/fwd_triton.py:984-1095 (the output o), so the forward pass never writes h.
// scan_bwd replaces HRDPLR/bwd_triton.py:127-222 (reverse recurrence of the state gradient, dh checkpoints,
// dh0) fused with the dv_new part of HRDPLR/bwd_triton.py:30-105.
//
// A wave owns one 16-column block of the fp32 state of a (sequence, head) for the whole sequence, in
// registers as the row fragment of S^T (rows = value column, inner = channel), which is at once the operand
// layout of the next product: w S, qg S and the rank updates chain through registers with no cross-lane
// movement.  A workgroup holds NWC such waves; a head's V/16 column blocks are split over (V/16)/NWC workgroups.  (KS = 2: two waves
// a block, half of the channels each, which hand each other their parts of v_new through LDS, one barrier more a step.  A step of 4-byte elements is
// bound by its products, 27 of 128 cycles at K = 64 with the output, and so a little more than half as long.)
//
// This file: 4-byte elements, and the chaining of the segments' records for both element sizes (2-byte elements: scan_out.cuh,
// scan_grad.cuh).  All column blocks of a head need the same w / kg / bg / qg tiles: a workgroup fetches the chunk's shared operand block
// (one contiguous block per chunk, written by the prep kernel) once for its NWC waves, which hold a register ring of their shares of the
// blocks to come and hand them to LDS.  Three LDS slots rotate with ONE LDS-only barrier per chunk (global loads stay in flight across it):
//    step t:  barrier                      block t+1 (written during step t-1) becomes visible
//             share of block t+2 -> slot (t+2) % 3          (its last readers finished before the barrier)
//             phase 1: v_new (operands already in registers, read during step t-1); the operands of the state update from slot t % 3
//             phase 2: state update; the phase-1 operands of chunk t+1 from slot (t+1) % 3
// so every LDS read has a phase of matrix products between its issue and its first use.
#pragma once
#include "hdla_common.cuh"
#include "scan_shapes.h"

namespace hdla {

constexpr int NSLOT = 3;

template <typename T, int K, int V, int NWC, int KS = 1> struct ScanCfg {
    static constexpr int VT = V / 16, SPLIT = VT / NWC;   // workgroups per head
    static constexpr int KB = K * (int)sizeof(T);         // bytes of one operand row
    static constexpr int THREADS = 64 * NWC * KS;
    // KS = 2, K = 64: two waves a column block, half of the channels each.  v_new and its gradient are then two sums over the channels, of either half; one wave forms
    // them so too, so that the bits do not depend on how many do.
    static constexpr bool HALVES = K == 64;
    static_assert(KS == 1 || (KS == 2 && HALVES), "");
    // 16-byte pieces that waves of a column block hand each other: the parts of both v_new, and of o
    static constexpr int HANDED = KS > 1 ? NWC * KS * 3 * 64 : 1;
    // Depth of the register ring of block shares (chunks in flight from global memory) and of the waves' own tiles; a multiple of the
    // number of slots so that slot numbers are static in the unrolled loops; 0: no ring, one chunk at a time.
    static constexpr int DR = KB <= 256 ? 3 : 0;
    // Whether LDS reads are issued a phase ahead of their use as described above, or left where the compiler
    // puts them (the shapes whose operands would not fit the register file twice over) ...
    static constexpr bool pipelined(bool with_o) { return KB <= 256 && !(NWC == 8 && with_o); }
    // ... and whether that includes the operands of the state update.  They are issued a few at a time between the products, not all of them
    // before the phase: K = V = 64, 2 x 1003 tokens of 8 heads, before the phase -> spread: records 45 -> 39 us, forward scan 22.5 -> 21.0,
    // scan pair 27.7 -> 26.3.
    static constexpr bool early_update_reads() { return KB <= 256 && NWC <= 4; }
};

// A shared operand block as the waves that load it see it: NI pieces of 1 KiB, lane l taking 16 bytes of each.  The first NT pieces hold
// tiles that are handed to LDS transposed, so a lane must hold whole fragments of them: such a piece is one tile of a pair, 16 of every 32 bytes.
__device__ __forceinline__ int piece_off(int i, int l, bool tiles) { return tiles ? (i >> 1) * 2048 + l * 32 + (i & 1) * 16 : i * 1024 + l * 16; }
// the whole block is contiguous in global memory (forward scans)
struct BlockOne {
    const char* p;
    __device__ __forceinline__ const char* piece(int i, int l, bool) const { return p + i * 1024 + l * 16; }
};
// reverse scan: W and BGT (NIF pieces) and the piece holding EGL come from the forward-scan block of the (chunk,
// head), the rest is the reverse-scan block
template <typename T, int K> struct BlockTwo {
    const char *f, *r;
    __device__ __forceinline__ const char* piece(int i, int l, bool tiles) const {
        constexpr SlotB S = slot_bwd(K, sizeof(T));
        static_assert(S.EGL_SRC % 1024 == 0, "EGL starts a piece");
        if (i < S.NIF) return f + piece_off(i, l, tiles);
        if (i == S.NIF) return f + S.EGL_SRC + l * 16;
        return r + (i - S.NIF - 1) * 1024 + l * 16;
    }
};

// 16 bytes of fragments, the tile transposed (a product with the identity: exact)
template <typename T> __device__ __forceinline__ i32x4 transpose_piece(i32x4 x) {
    Frag<T> f;
    f.v = __builtin_bit_cast(f32x4, x);
    return __builtin_bit_cast(i32x4, transpose(f, ident_frag<T>()).v);
}

// one wave's share of a shared operand block: the pieces w, w+NLD, ... of its NI pieces
template <typename T, int NI, int NLD, int NT = 0> struct Share {
    static constexpr int CNT = (NI + NLD - 1) / NLD;
    static_assert(NT % NLD == 0 && NT < NI, "whether a piece is transposed must not depend on the wave");
    i32x4 a[CNT];
    template <typename Blk> __device__ __forceinline__ void load(const Blk& blk, int w) {
        const int l = lane_id();
#pragma unroll
        for (int j = 0; j < CNT; ++j) {
            const int i = min(w + j * NLD, NI - 1);       // the last pieces may be fetched twice; never out of range
            a[j] = *reinterpret_cast<const i32x4*>(blk.piece(i, l, j * NLD < NT));
        }
    }
    __device__ __forceinline__ void to_lds(char* slot, int w) const {
        const int l = lane_id();
#pragma unroll
        for (int j = 0; j < CNT; ++j) {
            const int i = min(w + j * NLD, NI - 1);
            const bool tiles = j * NLD < NT;
            *reinterpret_cast<i32x4*>(slot + piece_off(i, l, tiles)) = tiles ? transpose_piece<T>(a[j]) : a[j];
        }
    }
};

// What a scan leaves:
//   OUT_O      forward pass: the output rows;
//   OUT_STATE  forward scan of the backward pass: the chunk's state checkpoint, [K/32][V/16] tile pairs.  v_new is not
//              checkpointed: the chunk_grad kernel rebuilds it from this checkpoint, w and u;
//   OUT_GRAD   reverse scan: the same for dS, and tile pairs of dv_new;
//   OUT_SUM    summary of a time segment: the record, written at the end
enum ScanOut { OUT_O, OUT_STATE, OUT_GRAD, OUT_SUM };
constexpr int SCAN_TARGET_WORKGROUPS = 256;               // compute units of the device

// ---- time segments -------------------------------------------------------------------------------------------
// Few (sequence, head) pairs leave most of the device idle while each of them walks its chunks one after the other, at
// 0.5 to 4 us a chunk.  There a sequence is cut into nseg time segments: the state leaving a segment is affine in the
// state entering it, S_out = M S_in + S_loc, and so is the state gradient on the way back.  A first launch walks all
// segments at once from a zero state (OUT_SUM: no output but the record) and, on K more columns that start as the
// identity and take no input of the chunks, for M; scan_chain_kernel chains the records into the states that enter the
// segments; then the scans run as they do for whole sequences, every segment from its own state.  Twice the steps,
// nseg times as many of them at once (scan_segments in api.hip says when).
//
// At the end of a segment: column block j of the state, or (trans) of the transition matrix X, whose tile (kt, j) is kept
// with rows k, inner k', which is how the chain takes it.  turned: where the backward pass will find its own, or null: what the state's gradient
// meets on its way back through a segment is the transpose of what the state met on its way there.
template <typename T, int K, int KS>
__device__ __forceinline__ void store_record(const f32x4 (&S)[K / 16 / KS], int kt0, float* loc, float* tr, float* turned, int64_t rec, int V, int j, bool trans) {
    constexpr int KT = K / 16, KTW = KT / KS;
    if (trans) {
        const Frag<float> ident = ident_frag<float>();
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt) {
            Frag<float> f;
            f.v = S[kt];
            f = transpose(f, ident);                      // exact: fp32 products with ones and zeros
            *reinterpret_cast<f32x4*>(tr + rec * (K * K) + ((kt0 + kt) * KT + j) * TILE + 4 * lane_id()) = f.v;
        }
        if (turned) {
#pragma unroll
            for (int kt = 0; kt < KTW; ++kt) *reinterpret_cast<f32x4*>(turned + rec * (K * K) + (j * KT + kt0 + kt) * TILE + 4 * lane_id()) = S[kt];
        }
    } else {
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt) *reinterpret_cast<f32x4*>(loc + rec * (K * V) + (j * KT + kt0 + kt) * TILE + 4 * lane_id()) = S[kt];
    }
}
// the columns a segment starts from when it does not start from h0 / dht: the chained state, zeros, or the identity
template <typename T, int K, bool SUM, int KS>
__device__ __forceinline__ void load_entry(f32x4 (&S)[K / 16 / KS], int kt0, const float* in, int64_t rec, int V, int j, bool trans) {
    const int l = lane_id(), g = l >> 4, c = l & 15;
#pragma unroll
    for (int kt = 0; kt < K / 16 / KS; ++kt) {
        if (!SUM) S[kt] = *reinterpret_cast<const f32x4*>(in + rec * (K * V) + (j * (K / 16) + kt0 + kt) * TILE + 4 * l);
        else if (trans) {
#pragma unroll
            for (int i = 0; i < 4; ++i) S[kt][i] = (16 * (kt0 + kt) + 4 * g + i == 16 * j + c) ? 1.f : 0.f;
        } else S[kt] = zero4();
    }
}

// ---- forward -------------------------------------------------------------------------------------------------
// split: which of the SPLIT groups of NWC column blocks; from SPLIT on (OUT_SUM only), of the transition matrix's
template <typename T, int K, int V, int NWC, ScanOut OUT, int KS>
__device__ __forceinline__ void scan_fwd_body(const ChunkArgs<T>& p, char* smem, f32x4* handed, int n, int seg, int split) {
    constexpr bool WRITE_O = OUT == OUT_O, SUM = OUT == OUT_SUM;
    typedef ScanCfg<T, K, V, NWC, KS> C;
    constexpr int KT = K / 16, KT2 = KT / 2, VT = V / 16, KTW = KT / KS, KTW2 = KTW / 2;
    constexpr BlkF B = blk_fwd(K, sizeof(T), WRITE_O);
    constexpr bool PIPE = C::pipelined(WRITE_O), PIPE_UPD = PIPE && C::early_update_reads();
    constexpr int SLOT = B.SIZE, NI = SLOT / 1024;

    const int h = blockIdx.x;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cb = wv % NWC, ks = KS == 1 ? 0 : wv / NWC, kt0 = ks * KTW, kp0 = kt0 / 2;   // own column block and channel tiles
    const bool trans = SUM && split >= C::SPLIT;
    const int vt0 = (trans ? split - C::SPLIT : split) * NWC;     // first column block of this workgroup
    const int own0 = trans ? 0 : vt0;                     // of its tiles of u^T, v^T (transition columns take none: never used)
    const int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H;
    int cs, ce, c0, c1;
    seq_chunks(p.st, n, cs, ce);
    seg_range(cs, ce, p.seg.nseg, seg, c0, c1);
    int64_t bos, eos;
    seq_bounds(p.st, n, bos, eos);
    bos += (int64_t)(c0 - cs) * CH;                       // the segment's first token
    const int64_t rec = ((int64_t)n * p.H + h) * p.seg.nseg + seg;
    const int64_t chw0 = (int64_t)h * p.st.nch;
    const int nchunks = c1 - c0, last = c1 - 1;
    // block of step t; steps past the end of the sequence are clamped, so every load is unconditional (a load
    // that may or may not have been issued would make the compiler wait for all outstanding loads)
    auto blk = [&](int t) __attribute__((always_inline)) {
        const int64_t chw = chw0 + min(c0 + t, last);
        // (the forward pass's blocks are B.SIZE apart; those the backward pass reads may be a forward pass's, further apart)
        const char* b = reinterpret_cast<const char*>(p.ws.W) + chw * (WRITE_O ? B.SIZE : p.ws.sa_stride);
        return BlockOne{b};
    };

    const int vt = vt0 + cb;
    // state block: lane (g,c) reg i of tile kt = S[16kt + 4g + i][16vt + c]
    f32x4 S[KTW];
    const int64_t soff = ((int64_t)n * H + h) * K * V + 16 * vt + c;
#pragma unroll
    for (int kt = 0; kt < KTW; ++kt) S[kt] = zero4();
    if (seg > 0) {
        load_entry<T, K, SUM, KS>(S, kt0, p.seg.in, rec, V, vt, trans);
    } else if (p.h0) {
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) S[kt][i] = p.h0[soff + (int64_t)(16 * (kt0 + kt) + 4 * g + i) * V];
    }
    struct Own { Frag<T> ut[2], vtt; };                   // the tiles only this wave reads
    auto load_own = [&](Own& o, int t) __attribute__((always_inline)) {
        const int64_t chw = chw0 + min(c0 + t, last);
        ld_pair(p.ws.UT + (chw * VT + own0 + cb % VT) * PAIR, o.ut[0], o.ut[1]);
        o.vtt = ld_tile(p.ws.VTT + (chw * VT + own0 + cb % VT) * TILE);
    };

    Frag<T> w[2][KTW];                                     // phase-1 operands; when pipelined, read a step ahead
    auto read_w = [&](const char* slot, int kp) __attribute__((always_inline)) {
        const T* sW = reinterpret_cast<const T*>(slot + B.W);
        ld_pair(sW + (0 * KT2 + kp0 + kp) * PAIR, w[0][2 * kp], w[0][2 * kp + 1]);
        ld_pair(sW + (1 * KT2 + kp0 + kp) * PAIR, w[1][2 * kp], w[1][2 * kp + 1]);
    };
    auto read_w_all = [&](const char* slot) __attribute__((always_inline)) {
#pragma unroll
        for (int kp = 0; kp < KTW2; ++kp) read_w(slot, kp);
    };

    // one chunk: shared operands from `slot`, the phase-1 operands of the next chunk from `slot_next`
    auto step = [&](const char* slot, const char* slot_next, Own own, int t) __attribute__((always_inline)) {
        const int cid = c0 + t;
        const int64_t chw = chw0 + cid;
        const int64_t tok0 = bos + (int64_t)t * CH;
        const int len = (int)min((int64_t)CH, eos - tok0);
        if (SUM && trans) { own.ut[0] = zero_frag<T>(); own.ut[1] = zero_frag<T>(); own.vtt = zero_frag<T>(); }
        const T* sBGT = reinterpret_cast<const T*>(slot + B.BGT);
        const T* sKGT = reinterpret_cast<const T*>(slot + B.KGT);
        const float* sEGL = reinterpret_cast<const float*>(slot + B.EGL);
        Frag<T> qg[WRITE_O ? KTW : 1], aqk, aqb[2], kgt[KTW], bgt[2][KTW];
        f32x4 egl[KTW];
        auto read_qg = [&](int kp) __attribute__((always_inline)) {
            ld_pair(reinterpret_cast<const T*>(slot + B.QG) + (kp0 + kp) * PAIR, qg[2 * kp], qg[2 * kp + 1]);
        };
        auto read_upd = [&](int kp) __attribute__((always_inline)) {
            ld_pair(sKGT + (kp0 + kp) * PAIR, kgt[2 * kp], kgt[2 * kp + 1]);
            ld_pair(sBGT + (0 * KT2 + kp0 + kp) * PAIR, bgt[0][2 * kp], bgt[0][2 * kp + 1]);
            ld_pair(sBGT + (1 * KT2 + kp0 + kp) * PAIR, bgt[1][2 * kp], bgt[1][2 * kp + 1]);
            egl[2 * kp] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (kt0 + 2 * kp) + 4 * g);
            egl[2 * kp + 1] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (kt0 + 2 * kp + 1) + 4 * g);
        };
        if (WRITE_O) {
            ld_pair(reinterpret_cast<const T*>(slot + B.AQB), aqb[0], aqb[1]);
            aqk = ld_tile(reinterpret_cast<const T*>(slot + B.AQK));
        }
        Frag<T> sb[KTW];
        // v_new^T (rows value, inner token) = u^T + S^T w^T; what is read on the way is used a group of products later or after
        f32x4 vn[2] = {to_f32(own.ut[0]), to_f32(own.ut[1])}, rest = zero4();
        if (ks) { vn[0] = zero4(); vn[1] = zero4(); }
        if constexpr (KS == 1 && PIPE && C::HALVES) {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) sb[kt] = to_frag<T>(S[kt]);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                if (WRITE_O) read_qg(r);
                if (PIPE_UPD && !WRITE_O) read_upd(r);
                __builtin_amdgcn_sched_barrier(0);
                if (r) vn[0] += rest;                     // (in the shadow of the products)
                rest = zero4();
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) {
                    f32x4& x = kt < KT2 ? vn[r] : rest;
                    x = mm(sb[kt], w[r][kt], x);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            f32x4 x2[2] = {zero4(), zero4()};
#pragma unroll
            for (int kp = 0; kp < KTW2; ++kp) {
                if (PIPE && WRITE_O) read_qg(kp);
                if (PIPE_UPD && !WRITE_O) read_upd(kp);
                if (!PIPE) read_w(slot, kp);
                if (PIPE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kt = 2 * kp; kt < 2 * kp + 2; ++kt) {
                    sb[kt] = to_frag<T>(S[kt]);
                    f32x4 (&x)[2] = C::HALVES && kt >= KT2 ? x2 : vn;
                    x[0] = mm(sb[kt], w[0][kt], x[0]);
                    x[1] = mm(sb[kt], w[1][kt], x[1]);
                }
                if (PIPE) __builtin_amdgcn_sched_barrier(0);
            }
            if (KS == 1 && C::HALVES) { vn[0] += x2[0]; rest = x2[1]; }
        }
        f32x4* const mine = handed + (cb * KS + ks) * 192 + l;
        const f32x4* const other = handed + (cb * KS + (ks ^ 1)) * 192 + l;
        if (KS > 1) { mine[0] = vn[0]; mine[64] = vn[1]; }
        f32x4 o = zero4();
        auto out_of_state = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int kp = 0; kp < KTW2; ++kp) {
                if (PIPE_UPD) read_upd(kp);
                if (!PIPE) read_qg(kp);
                if (PIPE) __builtin_amdgcn_sched_barrier(0);
                o = mm(qg[2 * kp], sb[2 * kp], o);
                o = mm(qg[2 * kp + 1], sb[2 * kp + 1], o);
                if (PIPE) __builtin_amdgcn_sched_barrier(0);
            }
        };
        // o (rows token, inner value) = qg S + A_qk v + sum_s A_qb^s v_new_s, one sum in this order: the wave of the channels' first half begins it
        // and the one of the second half goes on, when the first two of these are there
        if (WRITE_O && !ks) {
            out_of_state();
            if (KS > 1) mine[128] = o;
        }
        if (KS > 1) lds_barrier();
        if (WRITE_O && KS > 1 && ks) {
            o = other[128];
            out_of_state();
        }
        if (WRITE_O && ks == KS - 1) o = mm(aqk, own.vtt, o);
        Frag<T> vnb[2];
        auto sum_up = [&]() __attribute__((always_inline)) {
            if (KS > 1) { vn[0] += other[0]; vn[1] += other[64]; }
            else if (C::HALVES) vn[1] += rest;
            vnb[0] = to_frag<T>(vn[0]);
            vnb[1] = to_frag<T>(vn[1]);
        };
        if (WRITE_O || KS > 1) sum_up();
        if (PIPE) __builtin_amdgcn_sched_barrier(0);
        if (OUT == OUT_STATE) {
            // checkpoint of the entering state, as the fragments held here (tile pairs, 16 bytes per lane, whole
            // cache lines): the chunk_grad kernel turns them the way it needs them
            T* hc = p.ws.HC + chw * (K * V) + vt * PAIR;
            constexpr int HSTR = VT * PAIR;               // elements between the pairs of consecutive channel tiles
#pragma unroll
            for (int kp = 0; kp < KTW2; ++kp) st_pair2(hc + (kp0 + kp) * HSTR, sb[2 * kp], sb[2 * kp + 1]);
        }
        if (WRITE_O && ks == KS - 1) {
            o = mm(aqb[0], vnb[0], o);
            o = mm(aqb[1], vnb[1], o);
            if (c < len) st_frag(p.o + ((tok0 + c) * H + h) * V + 16 * vt + 4 * g, to_frag<T>(o));
        }
        // S <- exp(g_last) S + kg^T v + sum_s bg_s^T v_new_s
#pragma unroll
        for (int kp = 0; kp < KTW2; ++kp) {
            if (!PIPE_UPD) read_upd(kp);
            if (PIPE) {                             // (those of phase 1, whose products have taken them already)
                read_w(slot_next, kp);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int kt = 2 * kp; kt < 2 * kp + 2; ++kt) S[kt] = mm(own.vtt, kgt[kt], S[kt] * egl[kt]);
            if (kp == 0 && !WRITE_O && KS == 1) sum_up();   // (in the shadow of these)
#pragma unroll
            for (int kt = 2 * kp; kt < 2 * kp + 2; ++kt) {
                S[kt] = mm(vnb[0], bgt[0][kt], S[kt]);
                S[kt] = mm(vnb[1], bgt[1][kt], S[kt]);
            }
            if (PIPE) __builtin_amdgcn_sched_barrier(0);
        }
    };

    if (nchunks > 0) {
        constexpr int DR = C::DR;
        int done = 0;
        if constexpr (DR > 0) {
            Share<T, NI, NWC * KS> sh[DR];
            Own own[DR];
#pragma unroll
            for (int d = 0; d < DR; ++d) {
                sh[d].load(blk(d), wv);
                load_own(own[d], d);
            }
            sh[0].to_lds(smem, wv);
            sh[1].to_lds(smem + SLOT, wv);
            sh[0].load(blk(DR), wv);
            sh[1].load(blk(DR + 1), wv);
            lds_barrier();
            if (PIPE) read_w_all(smem);
            const int nfull = nchunks / DR;
#pragma unroll 1
            for (int gi = 0; gi < nfull; ++gi) {
#pragma unroll
                for (int j = 0; j < DR; ++j) {            // DR is a multiple of NSLOT: step gi*DR+j uses slot j % 3
                    const int t = gi * DR + j;
                    lds_barrier();
                    sh[(j + 2) % DR].to_lds(smem + ((j + 2) % NSLOT) * SLOT, wv);
                    sh[(j + 2) % DR].load(blk(t + 2 + DR), wv);
                    step(smem + (j % NSLOT) * SLOT, smem + ((j + 1) % NSLOT) * SLOT, own[j], t);
                    // refilled only after the last use: a register that is loaded while its old value is still
                    // live needs a copy, and the copy would wait for the load just issued
                    load_own(own[j], t + DR);
                }
            }
            done = nfull * DR;
        } else {
            Share<T, NI, NWC * KS> tmp;
            tmp.load(blk(0), wv);
            tmp.to_lds(smem, wv);
            tmp.load(blk(1), wv);
            tmp.to_lds(smem + SLOT, wv);
            lds_barrier();
            if (PIPE) read_w_all(smem);
        }
        // what is left (fewer than a ring of chunks, or all of them without a ring): one at a time, same protocol
        if (done < nchunks) {
            Own cur;
            load_own(cur, done);
#pragma unroll 1
            for (int t = done; t < nchunks; ++t) {
                lds_barrier();
                Share<T, NI, NWC * KS> tmp;
                tmp.load(blk(t + 2), wv);
                Own nxt;
                load_own(nxt, t + 1);
                step(smem + (t % NSLOT) * SLOT, smem + ((t + 1) % NSLOT) * SLOT, cur, t);
                tmp.to_lds(smem + ((t + 2) % NSLOT) * SLOT, wv);
                cur = nxt;
            }
        }
    }
    if (SUM) {
        store_record<T, K, KS>(S, kt0, p.seg.loc, p.seg.tr, p.seg.turned, rec, V, vt, trans);
    } else if (p.ht && seg == p.seg.nseg - 1) {
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) p.ht[soff + (int64_t)(16 * (kt0 + kt) + 4 * g + i) * V] = S[kt][i];
    }
}

// ---- backward ------------------------------------------------------------------------------------------------
// Step t handles chunk c1-1-t.
template <typename T, int K, int V, int NWC, ScanOut OUT, int KS>
__device__ __forceinline__ void scan_bwd_body(const ChunkArgs<T>& p, char* smem, f32x4* handed, int n, int seg, int split) {
    constexpr bool SUM = OUT == OUT_SUM;
    typedef ScanCfg<T, K, V, NWC, KS> C;
    constexpr int KT = K / 16, KT2 = KT / 2, VT = V / 16, KTW = KT / KS, KTW2 = KTW / 2;
    // LDS slot: [BG | WT] (BGT and W of the forward-scan block, transposed on their way in) | EGL | QGT | AQBT
    constexpr SlotB B = slot_bwd(K, sizeof(T));
    constexpr int SBWD = blk_bwd(K, sizeof(T)).SIZE, NT = B.NIF;
    const int SFWD = p.ws.sa_stride;
    constexpr bool PIPE = C::pipelined(false), PIPE_UPD = PIPE && C::early_update_reads();
    constexpr int NI = B.SIZE / 1024, SLOT = B.SIZE;

    const int h = blockIdx.x;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cb = wv % NWC, ks = KS == 1 ? 0 : wv / NWC, kt0 = ks * KTW, kp0 = kt0 / 2;   // own column block and channel tiles
    const bool trans = SUM && split >= C::SPLIT;
    const int vt0 = (trans ? split - C::SPLIT : split) * NWC;
    const int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H;
    int cs, ce, c0, c1;
    seq_chunks(p.st, n, cs, ce);
    seg_range(cs, ce, p.seg.nseg, seg, c0, c1);
    int64_t bos, eos;
    seq_bounds(p.st, n, bos, eos);
    bos += (int64_t)(c0 - cs) * CH;
    const int64_t rec = ((int64_t)n * p.H + h) * p.seg.nseg + seg;
    const int64_t chw0 = (int64_t)h * p.st.nch;
    const int nchunks = c1 - c0, first = c1 - 1;
    auto blk = [&](int t) __attribute__((always_inline)) {
        const int64_t slot = chw0 + max(first - t, c0);
        return BlockTwo<T, K>{reinterpret_cast<const char*>(p.ws.W) + slot * SFWD, reinterpret_cast<const char*>(p.ws.QGT) + slot * SBWD};
    };

    const int vt = vt0 + cb;
    f32x4 dS[KTW];   // lane (g,c) reg i of tile kt = dS[16kt + 4g + i][16vt + c]
    const int64_t soff = ((int64_t)n * H + h) * K * V + 16 * vt + c;
#pragma unroll
    for (int kt = 0; kt < KTW; ++kt) dS[kt] = zero4();
    if (seg < p.seg.nseg - 1) {
        load_entry<T, K, SUM, KS>(dS, kt0, p.seg.rin, rec, V, vt, trans);
    } else if (p.dht) {
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) dS[kt][i] = p.dht[soff + (int64_t)(16 * (kt0 + kt) + 4 * g + i) * V];
    }
    const Frag<T> ident = ident_frag<T>();
    // rows of do; rows past the end of a ragged chunk alias its last row and are zeroed where used
    auto load_own = [&](Frag<T>& don, int t) __attribute__((always_inline)) {
        const int cid = max(first - t, c0);
        const int64_t tok0 = bos + (int64_t)(cid - c0) * CH;
        const int len = (int)min((int64_t)CH, eos - tok0);
        don = ld_frag(p.dout + ((tok0 + min(c, len - 1)) * H + h) * V + 16 * (trans ? 0 : vt) + 4 * g);
    };

    Frag<T> aq[2], bg[2][KTW];                             // phase-1 operands; when pipelined, read a step ahead
    auto read_bg = [&](const char* slot, int kp) __attribute__((always_inline)) {
        const T* sBG = reinterpret_cast<const T*>(slot + B.BGT);
        ld_pair(sBG + (0 * KT2 + kp0 + kp) * PAIR, bg[0][2 * kp], bg[0][2 * kp + 1]);
        ld_pair(sBG + (1 * KT2 + kp0 + kp) * PAIR, bg[1][2 * kp], bg[1][2 * kp + 1]);
    };
    auto read_p1_all = [&](const char* slot) __attribute__((always_inline)) {
        ld_pair(reinterpret_cast<const T*>(slot + B.AQBT), aq[0], aq[1]);
#pragma unroll
        for (int kp = 0; kp < KTW2; ++kp) read_bg(slot, kp);
    };

    auto step = [&](const char* slot, const char* slot_next, Frag<T> don, int t) __attribute__((always_inline)) {
        const int cid = first - t;
        const int64_t chw = chw0 + cid;
        const T* sWT = reinterpret_cast<const T*>(slot + B.W);
        const T* sQGT = reinterpret_cast<const T*>(slot + B.QGT);
        const float* sEGL = reinterpret_cast<const float*>(slot + B.EGL);
        Frag<T> qgt[KTW], wt[2][KTW];
        f32x4 egl[KTW];
        auto read_upd = [&](int kp) __attribute__((always_inline)) {
            ld_pair(sQGT + (kp0 + kp) * PAIR, qgt[2 * kp], qgt[2 * kp + 1]);
            ld_pair(sWT + (0 * KT2 + kp0 + kp) * PAIR, wt[0][2 * kp], wt[0][2 * kp + 1]);
            ld_pair(sWT + (1 * KT2 + kp0 + kp) * PAIR, wt[1][2 * kp], wt[1][2 * kp + 1]);
            egl[2 * kp] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (kt0 + 2 * kp) + 4 * g);
            egl[2 * kp + 1] = *reinterpret_cast<const f32x4*>(sEGL + 16 * (kt0 + 2 * kp + 1) + 4 * g);
        };
        if (!PIPE) ld_pair(reinterpret_cast<const T*>(slot + B.AQBT), aq[0], aq[1]);
        Frag<T> dsb[KTW];
        const int len = (int)min((int64_t)CH, eos - (bos + (int64_t)(cid - c0) * CH));
        if (c >= len || trans) don = zero_frag<T>();
        const Frag<T> doT = transpose(don, ident);          // rows value, inner token
        // dv_new_s^T (rows value, inner token) = do^T A_qb^s + dS^T bg_s^T; what is read here is used a phase later
        f32x4 dvn[2] = {zero4(), zero4()}, rest = zero4();
        if (!ks) {
            dvn[0] = mm(doT, aq[0], zero4());
            dvn[1] = mm(doT, aq[1], zero4());
        }
        if constexpr (KS == 1 && PIPE_UPD && C::HALVES) {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) dsb[kt] = to_frag<T>(dS[kt]);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                read_upd(r);
                __builtin_amdgcn_sched_barrier(0);
                if (r) dvn[0] += rest;                    // (in the shadow of the products)
                rest = zero4();
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) {
                    f32x4& x = kt < KT2 ? dvn[r] : rest;
                    x = mm(dsb[kt], bg[r][kt], x);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            f32x4 x2[2] = {zero4(), zero4()};
#pragma unroll
            for (int kp = 0; kp < KTW2; ++kp) {
                if (PIPE_UPD) read_upd(kp);
                if (!PIPE) read_bg(slot, kp);
                if (PIPE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kt = 2 * kp; kt < 2 * kp + 2; ++kt) {
                    dsb[kt] = to_frag<T>(dS[kt]);
                    f32x4 (&x)[2] = C::HALVES && kt >= KT2 ? x2 : dvn;
                    x[0] = mm(dsb[kt], bg[0][kt], x[0]);
                    x[1] = mm(dsb[kt], bg[1][kt], x[1]);
                }
                if (PIPE) __builtin_amdgcn_sched_barrier(0);
            }
            if (KS == 1 && C::HALVES) { dvn[0] += x2[0]; rest = x2[1]; }
        }
        f32x4* const mine = handed + (cb * KS + ks) * 192 + l;
        const f32x4* const other = handed + (cb * KS + (ks ^ 1)) * 192 + l;
        if (KS > 1) {
            mine[0] = dvn[0];
            mine[64] = dvn[1];
            lds_barrier();
        }
        Frag<T> dvb[2];
        auto sum_up = [&]() __attribute__((always_inline)) {
            if (KS > 1) { dvn[0] += other[0]; dvn[1] += other[64]; }
            else if (C::HALVES) dvn[1] += rest;
            dvb[0] = to_frag<T>(dvn[0]);
            dvb[1] = to_frag<T>(dvn[1]);
        };
        // gradient of the state leaving the chunk and of v_new, as the fragments held here (tile pairs)
        if constexpr (!SUM) {
            T* dhc = p.ws.DHC + chw * (K * V) + vt * PAIR;
            constexpr int HSTR = VT * PAIR;
#pragma unroll
            for (int kp = 0; kp < KTW2; ++kp) st_pair2(dhc + (kp0 + kp) * HSTR, dsb[2 * kp], dsb[2 * kp + 1]);
        }
        // dS <- exp(g_last) dS + qg^T do + sum_s w_s^T dv_new_s
#pragma unroll
        for (int kp = 0; kp < KTW2; ++kp) {
            if (!PIPE_UPD) read_upd(kp);
            if (PIPE) {                             // (those of phase 1, whose products have taken them already)
                if (kp == 0) ld_pair(reinterpret_cast<const T*>(slot_next + B.AQBT), aq[0], aq[1]);
                read_bg(slot_next, kp);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int kt = 2 * kp; kt < 2 * kp + 2; ++kt) dS[kt] = mm(doT, qgt[kt], dS[kt] * egl[kt]);
            if (kp == 0) sum_up();                          // (in the shadow of these)
#pragma unroll
            for (int kt = 2 * kp; kt < 2 * kp + 2; ++kt) {
                dS[kt] = mm(dvb[0], wt[0][kt], dS[kt]);
                dS[kt] = mm(dvb[1], wt[1][kt], dS[kt]);
            }
            if (PIPE) __builtin_amdgcn_sched_barrier(0);
        }
        if (!SUM && !ks) st_pair2(p.ws.DVN + chw * (2 * CH * V) + vt * PAIR, dvb[0], dvb[1]);
    };

    if (nchunks > 0) {
        constexpr int DR = C::DR;
        int done = 0;
        if constexpr (DR > 0) {
            Share<T, NI, NWC * KS, NT> sh[DR];
            Frag<T> own[DR];
#pragma unroll
            for (int d = 0; d < DR; ++d) {
                sh[d].load(blk(d), wv);
                load_own(own[d], d);
            }
            sh[0].to_lds(smem, wv);
            sh[1].to_lds(smem + SLOT, wv);
            sh[0].load(blk(DR), wv);
            sh[1].load(blk(DR + 1), wv);
            lds_barrier();
            if (PIPE) read_p1_all(smem);
            const int nfull = nchunks / DR;
#pragma unroll 1
            for (int gi = 0; gi < nfull; ++gi) {
#pragma unroll
                for (int j = 0; j < DR; ++j) {
                    const int t = gi * DR + j;
                    lds_barrier();
                    sh[(j + 2) % DR].to_lds(smem + ((j + 2) % NSLOT) * SLOT, wv);
                    sh[(j + 2) % DR].load(blk(t + 2 + DR), wv);
                    step(smem + (j % NSLOT) * SLOT, smem + ((j + 1) % NSLOT) * SLOT, own[j], t);
                    load_own(own[j], t + DR);             // after the last use of the old value: no copy, no wait
                }
            }
            done = nfull * DR;
        } else {
            Share<T, NI, NWC * KS, NT> tmp;
            tmp.load(blk(0), wv);
            tmp.to_lds(smem, wv);
            tmp.load(blk(1), wv);
            tmp.to_lds(smem + SLOT, wv);
            lds_barrier();
            if (PIPE) read_p1_all(smem);
        }
        if (done < nchunks) {
            Frag<T> cur;
            load_own(cur, done);
#pragma unroll 1
            for (int t = done; t < nchunks; ++t) {
                lds_barrier();
                Share<T, NI, NWC * KS, NT> tmp;
                tmp.load(blk(t + 2), wv);
                Frag<T> nxt;
                load_own(nxt, t + 1);
                step(smem + (t % NSLOT) * SLOT, smem + ((t + 1) % NSLOT) * SLOT, cur, t);
                tmp.to_lds(smem + ((t + 2) % NSLOT) * SLOT, wv);
                cur = nxt;
            }
        }
    }
    if (SUM) {
        store_record<T, K, KS>(dS, kt0, p.seg.rloc, p.seg.rtr, nullptr, rec, V, vt, trans);
    } else if (p.dh0 && seg == 0) {
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) p.dh0[soff + (int64_t)(16 * (kt0 + kt) + 4 * g + i) * V] = dS[kt][i];
    }
}

// ---- kernels ---------------------------------------------------------------------------------------------------
// grid = (H, directions * SPLIT, N * segments): blockIdx.y = direction * SPLIT + split; blockIdx.z counts the sequences
// (segment fastest), packed ones from the longest down.  Workgroups start in the order of their linear index (x fastest):
// the workgroups of one (sequence, head) are H apart, which puts them on the same XCD (and its L2, where they share the
// chunk blocks) when H is a multiple of 8, and when the launch has more workgroups than the device holds at once, the long
// sequences, which decide when the launch ends, start first and the short ones fill in behind them.
// Where the sequences share the device by their lengths: sequence, width and column blocks of the unit-th workgroup of a head.  False: there are
// fewer.  The longest sequence's come first.
template <int V> __device__ __forceinline__ bool scan_share(const SeqTab& st, int unit, int shift, int& n, int& code, int& split) {
    static_assert(SHARE_MAX_N <= 64, "a lane a sequence");
    const int l = lane_id();
    const uint32_t e = l < st.N ? (uint32_t)st.order[l] : 0u;
    const int own = l < st.N ? (V / 64) << (e >> shift & 3) : 0;
    int end = own;
#pragma unroll
    for (int d = 1; d < SHARE_MAX_N; d <<= 1) {
        const int x = __shfl_up(end, d);
        end += l >= d ? x : 0;
    }
    const int r = __builtin_popcountll(__ballot(l < st.N && end <= unit));
    if (r >= st.N) return false;
    const uint32_t er = __builtin_amdgcn_readlane(e, r);
    n = (int)(er & ORDER_SEQ);
    code = (int)(er >> shift & 3);
    split = unit - __builtin_amdgcn_readlane(end - own, r);
    return true;
}
template <typename T, int K, int V, int NWC, int KS, bool WRITE_O>
__global__ __launch_bounds__((ScanCfg<T, K, V, NWC, KS>::THREADS)) void scan_fwd_kernel(ChunkArgs<T> p) {
    constexpr ScanOut OUT = WRITE_O ? OUT_O : OUT_STATE;
    __shared__ __attribute__((aligned(16))) char smem[NSLOT * blk_fwd(K, sizeof(T), WRITE_O).SIZE];
    __shared__ f32x4 handed[ScanCfg<T, K, V, NWC, KS>::HANDED];
    const int z = blockIdx.z / p.seg.nseg, seg = blockIdx.z % p.seg.nseg;
    scan_fwd_body<T, K, V, NWC, OUT, KS>(p, smem, handed, scan_sequence(p.st, z), seg, blockIdx.y);
}
template <typename T, int K, int V, int NWC, int KS>
__global__ __launch_bounds__((ScanCfg<T, K, V, NWC, KS>::THREADS)) void scan_bwd_kernel(ChunkArgs<T> p) {
    __shared__ __attribute__((aligned(16))) char smem[NSLOT * slot_bwd(K, sizeof(T)).SIZE];
    __shared__ f32x4 handed[ScanCfg<T, K, V, NWC, KS>::HANDED];
    const int z = blockIdx.z / p.seg.nseg, seg = blockIdx.z % p.seg.nseg;
    scan_bwd_body<T, K, V, NWC, OUT_GRAD, KS>(p, smem, handed, scan_sequence(p.st, z), seg, blockIdx.y);
}
// Both scans of the backward pass in one launch: they depend on the prep kernel only, not on each other.
template <typename T, int K, int V, int NWC, int KS>
__global__ __launch_bounds__((ScanCfg<T, K, V, NWC, KS>::THREADS)) void scan_pair_kernel(ChunkArgs<T> p) {
    constexpr int NF = NSLOT * blk_fwd(K, sizeof(T), false).SIZE;
    constexpr int NB = NSLOT * slot_bwd(K, sizeof(T)).SIZE;
    constexpr int SPLIT = ScanCfg<T, K, V, NWC, KS>::SPLIT;
    __shared__ __attribute__((aligned(16))) char smem[NF > NB ? NF : NB];
    __shared__ f32x4 handed[ScanCfg<T, K, V, NWC, KS>::HANDED];
    const int z = blockIdx.z / p.seg.nseg, seg = blockIdx.z % p.seg.nseg;
    const int n = scan_sequence(p.st, z);
    if (blockIdx.y < SPLIT) scan_fwd_body<T, K, V, NWC, OUT_STATE, KS>(p, smem, handed, n, seg, blockIdx.y);
    else scan_bwd_body<T, K, V, NWC, OUT_GRAD, KS>(p, smem, handed, n, seg, blockIdx.y - SPLIT);
}
// The segments' records: grid = (H, directions * (V + K) / 16 / NWC, N * (segments - 1)); forward the segments before the
// last, in reverse those behind the first.  first_y: blockIdx.y counts from there on (SEG_BWD_KEPT: the reverse direction's V / 16 / NWC, which
// leave out the transitions' columns; see sum_splits).
template <typename T, int K, int V, int NWC, int KS, bool BOTH>
__global__ __launch_bounds__((ScanCfg<T, K, V, NWC, KS>::THREADS)) void scan_sum_kernel(ChunkArgs<T> p, int first_y) {
    constexpr int NF = NSLOT * blk_fwd(K, sizeof(T), false).SIZE;
    constexpr int NB = NSLOT * slot_bwd(K, sizeof(T)).SIZE;
    constexpr int SPLIT = ScanCfg<T, K, V, NWC, KS>::SPLIT, COLS = (V + K) / 16 / NWC;
    __shared__ __attribute__((aligned(16))) char smem[BOTH && NB > NF ? NB : NF];
    __shared__ f32x4 handed[ScanCfg<T, K, V, NWC, KS>::HANDED];
    const int z = blockIdx.z / (p.seg.nseg - 1), seg = blockIdx.z % (p.seg.nseg - 1);
    const int n = scan_sequence(p.st, z), y = blockIdx.y + first_y, split = y % COLS;
    if (!BOTH || y < COLS) {
        if (seg == 0 && split >= SPLIT) return;           // starts from h0: nobody asks for its transition
        scan_fwd_body<T, K, V, NWC, OUT_SUM, KS>(p, smem, handed, n, seg, split);
    } else {
        if (seg + 1 == p.seg.nseg - 1 && split >= SPLIT) return;
        scan_bwd_body<T, K, V, NWC, OUT_SUM, KS>(p, smem, handed, n, seg + 1, split);
    }
}
// The records chained into what enters the segments, X <- M_s X + X_loc(s) from the segment that starts the sequence (or, in
// reverse, ends it): grid = (H, directions * V/16, N), one wave per 16 rows of the state's column block; blockIdx.y counts from first_y on.  A chain of
// dependent steps, so a step is kept short: the wave's rows of the next transition matrix are requested a step ahead, the
// waves exchange their rows through LDS (split operands: the error of fp32 products), one barrier a step.
// With 4-byte elements the sums are 64-bit (v_mfma_f64_16x16x4_f64): in fp32 a chain step rounds a state K / 4 times more than the
// scan of a whole sequence does.  Measured against a float64 evaluation, training steps on 2 x 1003 tokens of 8 heads, K = V = 64,
// slow decay: with fp32 sums the errors of outputs and gradients were 1.0 to 1.6 % larger than those of whole sequences (2.9e-7),
// with 64-bit sums they are the same (1.0002 +- 0.0002 for the outputs); 222.8 / 223.7 us, runs of one side differing by 1 %.
typedef double f64x4 __attribute__((ext_vector_type(4)));
template <typename T> struct ChainState { typedef Split<T> shared; };
template <> struct ChainState<float> { typedef f64x4 shared; };
template <typename T, int K, int V>
__global__ __launch_bounds__(64 * (K / 16)) void scan_chain_kernel(ChunkArgs<T> p, int first_y) {
    constexpr int KT = K / 16, VT = V / 16;
    constexpr bool WIDE = sizeof(T) == 4;
    typedef typename ChainState<T>::shared Shared;
    __shared__ __attribute__((aligned(16))) Shared sx[2][KT][64];
    const int y = blockIdx.y + first_y, h = blockIdx.x, vt = y % VT, n = blockIdx.z, nseg = p.seg.nseg;
    const bool rev = y >= VT;
    const int kt = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id();
    const float* const loc = rev ? p.seg.rloc : p.seg.loc;
    const float* const tr = rev ? p.seg.rtr : p.seg.tr;
    float* const in = rev ? p.seg.rin : p.seg.in;
    const int64_t rec0 = ((int64_t)n * p.H + h) * nseg;
    // step i handles the i-th segment from the start of the chain
    auto rec = [&](int i) { return rec0 + (rev ? nseg - 1 - i : i); };
    const int own = (vt * KT + kt) * TILE + 4 * l;
    // Register i of lane (g, c) of a 64-bit result is row g + 4 i of the product: the rows of the transition matrix are handed over
    // in the order in which that is row 4 g + i, as everywhere else.
    const int row = WIDE ? (l & 48) + 4 * (l & 3) + ((l >> 2) & 3) : l;
    auto request = [&](int i, f32x4 (&m)[KT], f32x4& a) __attribute__((always_inline)) {
        i = min(i, nseg - 2);                             // past the end: never used
        a = *reinterpret_cast<const f32x4*>(loc + rec(i) * (K * V) + own);
#pragma unroll
        for (int ki = 0; ki < KT; ++ki) m[ki] = *reinterpret_cast<const f32x4*>(tr + rec(i) * (K * K) + (kt * KT + ki) * TILE + 4 * row);
    };
    const f32x4 first = *reinterpret_cast<const f32x4*>(loc + rec(0) * (K * V) + own);
    f32x4 m[KT], add;
    request(1, m, add);
    if constexpr (WIDE) {
        f64x4 x = __builtin_convertvector(first, f64x4);
        for (int i = 1; i < nseg; ++i) {
            *reinterpret_cast<f32x4*>(in + rec(i) * (K * V) + own) = __builtin_convertvector(x, f32x4);
            if (i == nseg - 1) break;
            sx[i & 1][kt][l] = x;
            __syncthreads();
            x = __builtin_convertvector(add, f64x4);
            f64x4 q[KT];
#pragma unroll
            for (int ki = 0; ki < KT; ++ki) q[ki] = __builtin_convertvector(m[ki], f64x4);
            request(i + 1, m, add);
#pragma unroll
            for (int ki = 0; ki < KT; ++ki) {
                const f64x4 xs = sx[i & 1][ki][l];
#pragma unroll
                for (int s = 0; s < 4; ++s) x = __builtin_amdgcn_mfma_f64_16x16x4f64(q[ki][s], xs[s], x, 0, 0, 0);
            }
        }
    } else {
        f32x4 x = first;
        for (int i = 1; i < nseg; ++i) {
            *reinterpret_cast<f32x4*>(in + rec(i) * (K * V) + own) = x;
            if (i == nseg - 1) break;
            Split<T> xs;
            split(x, xs);
            sx[i & 1][kt][l] = xs;
            __syncthreads();
            x = add;
            Split<T> q[KT];
#pragma unroll
            for (int ki = 0; ki < KT; ++ki) split(m[ki], q[ki]);
            request(i + 1, m, add);
#pragma unroll
            for (int ki = 0; ki < KT; ++ki) x = mm_split(sx[i & 1][ki][l], q[ki], x);
        }
    }
}

// ---- launchers -------------------------------------------------------------------------------------------------
template <typename T, int K, int V, int NWC, int KS>
static hipError_t launch_scan_nwc(const ChunkArgs<T>& a, ScanKind kind, hipStream_t stream) {
    typedef ScanCfg<T, K, V, NWC, KS> C;
    dim3 grid(a.H, C::SPLIT * (kind == SCAN_PAIR ? 2 : 1), a.st.N * a.seg.nseg), block(C::THREADS);
    switch (kind) {
        case SCAN_FWD_O: hipLaunchKernelGGL((scan_fwd_kernel<T, K, V, NWC, KS, true>), grid, block, 0, stream, a); break;
        case SCAN_FWD: hipLaunchKernelGGL((scan_fwd_kernel<T, K, V, NWC, KS, false>), grid, block, 0, stream, a); break;
        case SCAN_BWD: hipLaunchKernelGGL((scan_bwd_kernel<T, K, V, NWC, KS>), grid, block, 0, stream, a); break;
        case SCAN_PAIR: hipLaunchKernelGGL((scan_pair_kernel<T, K, V, NWC, KS>), grid, block, 0, stream, a); break;
    }
    return hipGetLastError();
}

template <typename T, int K, int V>
hipError_t launch_scan_shape(const ChunkArgs<T>& a, ScanKind kind, hipStream_t stream) {
    // V = 128: all eight column blocks of a head in a workgroup are two waves a SIMD, which wait for each other's products, while compute units without
    // a workgroup have nothing to do.  Four of them a workgroup take 0.6 of the step (and fetch a chunk's operands twice), so: where twice the workgroups
    // come in rounds that are the sooner done.  us, fp32 forward passes, eight -> four, K = V = 128 / K = 64: 64 lanes of 19 chunks 165 -> 118 / 102 -> 75, 80 of
    // 22 201 -> 146 / 114 -> 82, 128 of 19 201 -> 160 / 120 -> 92, but 160 of 19 219 -> 250 / 131 -> 141, 256 of 13 195 -> 219 / 123 -> 132, and again 320 of 13
    // 301 -> 296 / 186 -> 175; 10 packed sequences of 8 heads, 3546 tokens 418 -> 278 / 231 -> 148.  The same bits.
    const long long lanes = (long long)a.H * a.st.N * a.seg.nseg * (kind == SCAN_PAIR ? 2 : 1);
    // K = 64, few sequences: two waves a column block, two blocks a workgroup, where these fit the device.  us, one wave a block -> two, fp32, V = 64 / V = 128:
    // forward passes of 64 lanes of 19 chunks 68.7 -> 61.3 / 73.5 -> 66.3, 128 of 19 83 -> 76 / (not chosen), 2 of 19 44 -> 40 / 46 -> 42, 10 packed sequences of 8
    // heads, 3546 tokens 142 -> 120; training steps of 64 lanes of 13 134 -> 122 / 173 -> 169, 2 x 1003 tokens of 8 heads 173 -> 169; where it is not chosen 0.99 to
    // 1.01.  Errors against float64, two sums over the channels instead of one, now to before: 0.92 (da) to 0.98 (dk), o 0.96 (3 shapes, 4 inputs each).
    if constexpr (K == 64) {
        if (lanes * (V / 32) <= SCAN_TARGET_WORKGROUPS) return launch_scan_nwc<T, K, V, 2, 2>(a, kind, stream);
    }
    if constexpr (V == 128) {
        auto rounds = [](long long workgroups) { return (workgroups + SCAN_TARGET_WORKGROUPS - 1) / SCAN_TARGET_WORKGROUPS; };
        if (6 * rounds(2 * lanes) < 10 * rounds(lanes)) return launch_scan_nwc<T, K, V, 4, 1>(a, kind, stream);
    }
    return launch_scan_nwc<T, K, V, V / 16, 1>(a, kind, stream);
}

template <typename T, int K, int V>
static hipError_t launch_scan_chain(const ChunkArgs<T>& a, SegStart what, hipStream_t stream) {
    hipLaunchKernelGGL((scan_chain_kernel<T, K, V>), dim3(a.H, V / 16 * (what == SEG_BWD ? 2 : 1), a.st.N), dim3(64 * (K / 16)), 0, stream, a,
                       what == SEG_BWD_KEPT ? V / 16 : 0);
    return hipGetLastError();
}
// workgroups of a (sequence, head, segment) in the launch of the segments' records, and the first of them.  With `turned` the forward direction's
// leave the reverse one's transitions, whose columns, the last ones of the launch, are then not asked for.
template <int K, int V, int NWC> static int sum_splits(SegStart what, bool turned) {
    constexpr int state = V / 16 / NWC, all = (V + K) / 16 / NWC;
    return what == SEG_BWD_KEPT ? state : what != SEG_BWD ? all : turned ? all + state : 2 * all;
}
template <int K, int V, int NWC> static int sum_first(SegStart what) { return what == SEG_BWD_KEPT ? (V + K) / 16 / NWC : 0; }
template <typename T, int K, int V, int NWC, int KS>
static hipError_t launch_scan_sum(const ChunkArgs<T>& a, SegStart what, dim3 grid, hipStream_t stream) {
    const dim3 block(ScanCfg<T, K, V, NWC, KS>::THREADS);
    const int first = sum_first<K, V, NWC>(what);
    if (what == SEG_BWD || what == SEG_BWD_KEPT) hipLaunchKernelGGL((scan_sum_kernel<T, K, V, NWC, KS, true>), grid, block, 0, stream, a, first);
    else hipLaunchKernelGGL((scan_sum_kernel<T, K, V, NWC, KS, false>), grid, block, 0, stream, a, first);
    return hipGetLastError();
}
template <typename T, int K, int V>
hipError_t launch_scan_segments_shape(const ChunkArgs<T>& a, SegStart what, hipStream_t stream) {
    // four column blocks per workgroup, each fetches the chunks' operands once for them; or two, where these fit the device (launch_scan_shape)
    auto grid = [&](int splits) { return dim3(a.H, splits, a.st.N * (a.seg.nseg - 1)); };
    hipError_t e = hipErrorInvalidValue;
    bool done = false;
    if constexpr (K == 64) {
        const dim3 g = grid(sum_splits<K, V, 2>(what, a.seg.turned));
        done = (long long)g.x * g.y * g.z <= SCAN_TARGET_WORKGROUPS;
        if (done) e = launch_scan_sum<T, K, V, 2, 2>(a, what, g, stream);
    }
    if (!done) e = launch_scan_sum<T, K, V, 4, 1>(a, what, grid(sum_splits<K, V, 4>(what, a.seg.turned)), stream);
    return e == hipSuccess ? launch_scan_chain<T, K, V>(a, what, stream) : e;
}

}  // namespace hdla
