// The forward pass's scan for 2-byte elements: the state recurrence and the output o (HRDPLR/fwd_triton.py:808-1095), and the
// records of time segments in the forward direction; without the output, the backward pass's forward scan.  (The reverse one:
// scan_grad.cuh; 4-byte elements: scan_impl.cuh.)  Computing
// waves hold a 16-column block of the fp32 state for the whole sequence; those of NWC blocks and NM waves that move data make a workgroup.
//
// A sequence is a chain of steps, and up to some 32 heads in flight the time is the number of steps of the longest sequence times
// the time of one, whatever the traffic (0.69 us at K = V = 128 in the form it had, that of scan_impl.cuh with four more waves that moved data, with 4 heads as with 32).  What a step costs
// is the instructions of a wave that has its SIMD to itself, some five cycles each, the latencies of the chain through the state (product ->
// conversion -> product -> exchange -> product), and what waits at its barrier.  So:
//  * products in twos (mm2), those with one product a sum first, one settle; b^T is stored with the two ranks of a channel tile side by
//    side, as the state update takes it; the walk is compiled without branches;
//  * at K = 128 two waves share a column block, a half of its channels each: half of the conversions, decays and products per wave, against
//    one exchange of v_new's parts through LDS, at the barrier that a step has anyway;
//  * the chunks' blocks go from global memory straight to LDS (global_load_lds), SLOTS chunks ahead, by waves that do nothing else;
//  * u = Tm (A_ak v) is formed here by a wave of its own, a chunk ahead, from the chunk's (I - A_ab)^-1 and A_ak and the workgroup's columns
//    of v (in the computing waves it cost 0.14 us a step: a chain of five dependent products).  The kernel that prepares the
//    chunks does not read v and writes 3 KB instead of u and v^T, 12 KB of its 70 a chunk and head at K = V = 128: 236 -> 192 us for 16384
//    tokens of 16 heads.  The products and roundings are the ones it had.  On the backward pass's workspace likewise, where that wave turns (I - A_ab)^-1 first
//    (chunk_grad wants it the other way round): a training step of 16384 tokens of 16 heads 1700 -> 1649 us, of 2 x 1537 of 8 191 -> 182.
// Measured, us, before -> after (when it was built), 2048 tokens a sequence: K = V = 128, 16 heads 88 -> 73, 32 heads 92 -> 79, 64 heads 105 -> 101, 128 heads
// 167 -> 146; K = 64, V = 128, 128 heads 116 -> 98; K = 128, V = 64, 32 heads 87 -> 72.  From 48 heads on a step waits for its loads: 82 us
// of the 101 where they never leave the L2, 70 without them; touching the blocks' lines 12 chunks ahead made it 105.
#pragma once
#include "hdla_common.cuh"
#include "hdla_launch.h"
#include "scan_impl.cuh"

namespace hdla {

// HD: with the HDLA parameterisation b_2 is k, so the gated copies of the two are the same tiles: kg^T is neither stored nor moved nor read (4 of a chunk and head's 42
// KB that prep moves at K = V = 128, of 37 that a forward pass's scan does).  us as a graph's replay, before -> after, the same bits, K = V = 128: forward pass of 4 x 2048 tokens of 16 heads 183 -> 164, 5003 packed
// 111 -> 108, 1 x 2048 79.8 -> 77.9; training step of 2 x 1537 of 8 162.3 -> 159.0; K = 128, V = 64, 1 x 3000 of 16 254 -> 248; K = 64, V = 128, 2 x 2000 of 4, forward 49.4 -> 48.7.
template <int K, int V, int NWC, ScanOut OUT, bool HD> struct OutCfg {
    static constexpr bool WITH_O = OUT == OUT_O;
    static constexpr int VT = V / 16, SPLIT = VT / NWC, KT = K / 16;
    static constexpr BlkF STORED = blk_fwd(K, 2, true);
    // 1-KiB pieces of a chunk's block that the scan needs (without o: without q's and the scores'), and where they are in LDS: HD without the CUT pieces from AT on
    static constexpr int CUT = HD ? KT / 2 : 0, AT = STORED.KGT / 1024;
    static constexpr int NI = (WITH_O ? STORED.SIZE : STORED.EGL + 1024) / 1024 - CUT, SLOT = NI * 1024;
    static constexpr BlkF slot_of(BlkF b) { b.EGL -= CUT * 1024; b.QG -= CUT * 1024; b.AQB -= CUT * 1024; b.AQK -= CUT * 1024; return b; }
    static constexpr BlkF B = slot_of(STORED);
    static __device__ __forceinline__ int stored(int i) { return HD && i >= AT ? i + CUT : i; }
    // computing waves of a column block, each holding KH channel tiles of the state
    static constexpr int PARTS = K / 64, KH = KT / PARTS, NC = NWC * PARTS;
    static constexpr int NL = 2, NM = NL + 1 + WITH_O;    // waves that load, with the one that forms u and the one that copies the output out
    static constexpr int CNT = (NI + NL - 1) / NL;        // loads of a wave per chunk (the last pieces may be fetched twice)
    static constexpr int THREADS = 64 * (NC + NM);
    static constexpr int OROW = 16 * NWC * 2 + 16, OB = WITH_O ? CH * OROW : 0;   // output rows of a step, padded; two of them
    static constexpr int UB = NWC * 1536;                 // u^T (a pair) and v^T (a tile) of the column blocks; two chunks' of them
    // what the waves of a column block hand each other: two tiles each, and from the second one its part of the output; two steps' of it
    static constexpr int XP = (WITH_O ? 5 : 4) * 1024, XB = PARTS > 1 ? NWC * XP : 0;
    static constexpr int REST = 2 * (OB + UB + XB);
    // as many slots as LDS holds, or as half of it does where that is enough (two workgroups on a compute unit)
    static constexpr int ROOM = (4 * SLOT + REST <= 80 * 1024 ? 80 : 160) * 1024 - REST;
    static constexpr int MOST = 62 / CNT + 1 < 8 ? 62 / CNT + 1 : 8, SLOTS = ROOM / SLOT < MOST ? ROOM / SLOT : MOST;
    static_assert(SLOTS >= 3 && (SLOTS - 1) * CNT < 63, "a chunk to read, the next one, and one on its way; the memory counter's range");
    static constexpr int OUTBOX = SLOTS * SLOT, UBUF = OUTBOX + 2 * OB, XBUF = UBUF + 2 * UB, BYTES = XBUF + 2 * XB;
};

// Roles of the NM waves behind the computing ones: NL that load, the one that forms, the one that copies the output out.  The forming wave comes first, then
// (with the output) the copying one, so that none of them is on a SIMD with a computing wave where there are one or two of those: waves go round
// the four SIMDs, and the forming one has half as many instructions a step as a computing one, a loading one a tenth.  It also finds its
// rows of v and do by 32-bit offsets from one base, 76 -> 55 instructions a chunk.  us a training step, before -> order -> both: K = 64, V = 128, 2 x 900 tokens
// of 16 heads 112.3 -> 109.5 -> 107.5 (while the passes read u 109.1), 2 x 1400 152.5 -> 148.4 -> 144.7, K = V = 64, 1 x 256 of 2 35.7 -> 35.8 -> 35.5 (35.2),
// K = V = 128, 2 x 1537 of 8 175.7 -> 169.4 -> 168.4, K = 128, V = 64, 2 x 900 of 16 133.9 -> 129.6 -> 129.8.  A forward pass that keeps nothing goes without: its forming
// wave does not turn (I - A_ab)^-1 and was done in time, and one that is done sooner meets the computing waves in LDS: K = V = 128, 2 x 1537 of 8
// heads 68.5 -> 68.6 -> 69.5, 2 x 1000 49.3 -> 49.6 -> 50.1 (segments' records by themselves: 22.1 -> 20.4).
template <typename C> __device__ __forceinline__ int forming_first(int wave) { return (wave + C::NL) % C::NM; }

// OUT_O: with the output; OUT_STATE: the forward scan of the backward pass, which leaves the state that enters each chunk; OUT_SUM:
// records of segments.
// KEPT: on a workspace of the backward pass (or that it will read, PREP_KEEP): (I - A_ab)^-1 is there turned, as chunk_grad takes it, A_ak in a place of its
// own, and b^T's pairs are of two channel tiles, as the reverse scan takes them.  The same products in the same order: the same bits.
// KEPT 2 (PREP_STATES): the states that enter the chunks are left for the backward pass, and q's part of the block is not the kept buffer's.
template <int K, int V, int NWC, ScanOut OUT, int KEPT, bool HD>
__device__ __forceinline__ void scan_out_body(const ChunkArgs<bf16>& p, char* smem, int n, int seg, int split) {
    typedef OutCfg<K, V, NWC, OUT, HD> C;
    typedef bf16 T;
    constexpr bool WITH_O = OUT == OUT_O, SUM = OUT == OUT_SUM;
    constexpr bool FWD = WITH_O && !KEPT, STATES = KEPT == 2;   // a forward pass that keeps nothing (see forming_first)
    constexpr int KT = C::KT, KT2 = KT / 2, SLOTS = C::SLOTS, SLOT = C::SLOT, PARTS = C::PARTS, KH = C::KH, KH2 = KH / 2;
    constexpr BlkF B = C::B;
    const int h = blockIdx.x;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool trans = SUM && split >= C::SPLIT;          // columns of the segment's transition matrix
    const int vt0 = (trans ? split - C::SPLIT : split) * NWC;
    const int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H;
    int cs, ce, c0, c1;
    seq_chunks(p.st, n, cs, ce);
    seg_range(cs, ce, p.seg.nseg, seg, c0, c1);
    int64_t bos, eos;
    seq_bounds(p.st, n, bos, eos);
    bos += (int64_t)(c0 - cs) * CH;                       // the segment's first token
    const int64_t rec = ((int64_t)n * H + h) * p.seg.nseg + seg;
    const int64_t chw0 = (int64_t)h * p.st.nch + c0;
    const int nchunks = c1 - c0, last = nchunks - 1;

    if (wv >= C::NC) {
        // ---- waves that move data.  Barriers: one closing the prologue, one per step, one handing over the last output; the computing
        // waves execute the same sequence.  From the barrier of step t on chunk t + 1 is in LDS and the slot of chunk t is free.
        if (nchunks <= 0) return;
        const int hw = FWD ? wv - C::NC : forming_first<C>(wv - C::NC);
        if (hw < C::NL) {
            const int stride = KEPT ? p.ws.sa_stride : C::STORED.SIZE;
            const char* const blk = reinterpret_cast<const char*>(p.ws.W) + chw0 * stride + l * 16;
            constexpr int PRE = STATES ? blk_fwd(K, 2, false).SIZE / 1024 - C::CUT : C::NI, STRIDE_Q = blk_q(K, 2);
            const char* const blk_of_q = reinterpret_cast<const char*>(p.ws.QG) + chw0 * STRIDE_Q + l * 16;
            int slot = 0;
            auto load = [&](int t) __attribute__((always_inline)) {
                // past the end: the last chunk again, never looked at
                const char* const bt = blk + (int64_t)min(t, last) * stride;
                const char* const qt = blk_of_q + (int64_t)min(t, last) * STRIDE_Q;
#pragma unroll
                for (int j = 0; j < C::CNT; ++j) {
                    const int i = min(hw + j * C::NL, C::NI - 1);
                    const char* const src = !STATES || i < PRE ? bt + C::stored(i) * 1024 : qt + (i - PRE) * 1024;
                    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                                     (__attribute__((address_space(3))) void*)(smem + slot * SLOT + i * 1024), 16, 0, 0);
                }
                slot = slot + 1 == SLOTS ? 0 : slot + 1;
            };
#pragma unroll
            for (int d = 0; d < SLOTS; ++d) load(d);
            wait_loads<(SLOTS - 1) * C::CNT>();           // chunk 0 is there
            __builtin_amdgcn_s_barrier();
            for (int t = 0; t < nchunks; ++t) {
                wait_loads<(SLOTS - 2) * C::CNT>();       // chunk t + 1
                __builtin_amdgcn_s_barrier();
                load(t + SLOTS);                          // where chunk t was
            }
            if (WITH_O) __builtin_amdgcn_s_barrier();
            wait_loads<0>();                              // nothing may arrive in LDS that is no longer this workgroup's
        } else if (hw == C::NL) {
            // v^T and u = Tm (A_ak v) of the workgroup's column blocks, a chunk ahead, with the roundings of the kernel that prepared the
            // chunk in u's place.  The operands come through registers, UD chunks ahead.
            constexpr int UD = 3;
            struct Own { i32x4 tm[3]; Frag<T> v[NWC]; };
            const Frag<T> ident = ident_frag<T>();
            // rows of v; behind the end of the last chunk its last row again
            auto len_of = [&](int t) __attribute__((always_inline)) { return (int)min((int64_t)CH, eos - (bos + (int64_t)min(t, last) * CH)); };
            const int len_last = len_of(last);
            const uint32_t row = (uint32_t)(H * V) * sizeof(T), whole = c * row + 8 * g, ragged = min(c, len_last - 1) * row + 8 * g;
            const T* const v0 = p.v + (bos * H + h) * V + 16 * (trans ? 0 : vt0);
            auto rows = [&](int t) __attribute__((always_inline)) {
                if constexpr (FWD) return p.v + ((bos + (int64_t)t * CH + min(c, len_of(t) - 1)) * H + h) * V + 16 * vt0 + 4 * g;
                else return at(v0 + (int64_t)t * (CH * H * V), t == last ? ragged : whole);
            };
            auto request = [&](int t) __attribute__((always_inline)) {
                t = min(t, last);
                Own o;
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const T* const from = !KEPT ? p.ws.TM + (chw0 + t) * (3 * PAIR) + i * PAIR : i < 2 ? p.ws.TM + (chw0 + t) * (2 * PAIR) + i * PAIR
                                                                                                       : p.ws.AAK + (chw0 + t) * PAIR;
                    o.tm[i] = *reinterpret_cast<const i32x4*>(from + 8 * l);
                }
#pragma unroll
                for (int j = 0; j < NWC; ++j) o.v[j] = ld_frag(rows(t) + (trans ? 0 : 16 * j));
                return o;
            };
            auto pair = [](i32x4 x, Frag<T>& f0, Frag<T>& f1) __attribute__((always_inline)) {
                const s16x8 y = __builtin_bit_cast(s16x8, x);
                f0.v = __builtin_shufflevector(y, y, 0, 1, 2, 3);
                f1.v = __builtin_shufflevector(y, y, 4, 5, 6, 7);
            };
            auto form = [&](int t, const Own& o) __attribute__((always_inline)) {
                const int len = FWD ? len_of(t) : t < last ? CH : len_last;
                T* const ub = reinterpret_cast<T*>(smem + C::UBUF + (t & 1) * C::UB);
                Frag<T> tm[2][2], aak[2], vT[NWC], mT[NWC][2];
                pair(o.tm[0], tm[0][0], tm[0][1]);
                pair(o.tm[1], tm[1][0], tm[1][1]);
                pair(o.tm[2], aak[0], aak[1]);
                if constexpr (KEPT) {
#pragma unroll
                    for (int s = 0; s < 2; ++s)
#pragma unroll
                        for (int r = 0; r < 2; ++r) tm[s][r] = transpose(tm[s][r], ident);
                }
#pragma unroll
                for (int j = 0; j < NWC; ++j) vT[j] = transpose((c >= len || trans) ? zero_frag<T>() : o.v[j], ident);
#pragma unroll
                for (int j = 0; j < NWC; ++j)
#pragma unroll
                    for (int r = 0; r < 2; ++r) mT[j][r] = to_frag<T>(mm(vT[j], aak[r], zero4()));
#pragma unroll
                for (int j = 0; j < NWC; ++j) {
                    st_tile(ub + j * (3 * TILE) + PAIR, vT[j]);
                    st_pair2(ub + j * (3 * TILE), to_frag<T>(mm2(mT[j][0], mT[j][1], tm[0][0], tm[0][1], zero4())),
                             to_frag<T>(mm2(mT[j][0], mT[j][1], tm[1][0], tm[1][1], zero4())));
                }
            };
            Own own[UD];                                  // chunk t in own[t % UD]
#pragma unroll
            for (int d = 0; d < UD; ++d) own[d] = request(d);
            form(0, own[0]);
            own[0] = request(UD);
            lds_barrier();
            auto step = [&](int t, Own& o) __attribute__((always_inline)) {
                form(t + 1, o);
                o = request(t + 1 + UD);
                lds_barrier();
            };
            // (unrolled: a register moved on while its load is on the way would wait for it)
            int t0 = 0;
#pragma unroll 1
            for (; t0 + UD <= nchunks; t0 += UD) {
#pragma unroll
                for (int j = 0; j < UD; ++j) step(t0 + j, own[(j + 1) % UD]);
            }
#pragma unroll
            for (int j = 0; j < UD - 1; ++j)
                if (t0 + j < nchunks) step(t0 + j, own[(j + 1) % UD]);
            if (WITH_O) lds_barrier();
        } else if constexpr (WITH_O) {
            // Outputs past the caches from 4 MiB a call on, an XCD's L2: below, the blocks' parts of a line meet there, and the kernel's end does not wait
            // for memory.  Calls in us, past -> near: 2 x 28 and 2 x 100 tokens of 12 heads, K = V = 128, 13.6 -> 13.1 and 18.6 -> 18.2; 2 x 1537 of 8
            // 63.7 -> 63.7; 2 x 2000 of 16 95 -> 104.
            const bool past = (int64_t)p.st.nch * H * (CH * V * 2) >= (4 << 20);
            __builtin_amdgcn_s_barrier();
            for (int t = 0; t <= nchunks; ++t) {
                lds_barrier();
                if (t == 0) continue;
                // rows of o: 16-byte pieces, LPR lanes a row
                constexpr int LPR = 2 * NWC, RPI = 64 / LPR;
                const int64_t tok0 = bos + (int64_t)(t - 1) * CH;
                const int len = (int)min((int64_t)CH, eos - tok0);
                const char* ob = smem + C::OUTBOX + ((t - 1) & 1) * C::OB;
#pragma unroll
                for (int r0 = 0; r0 < CH; r0 += RPI) {
                    const int r = r0 + l / LPR, e = (l % LPR) * 16;
                    if (r < len) {
                        const i32x4 x = *reinterpret_cast<const i32x4*>(ob + r * C::OROW + e);
                        i32x4* const to = reinterpret_cast<i32x4*>(reinterpret_cast<char*>(p.o + ((tok0 + r) * H + h) * V + 16 * vt0) + e);
                        if (past) st_past(to, x);
                        else st_near(to, x);
                    }
                }
            }
        }
        return;
    }

    // ---- computing wave: channel tiles kt0 .. kt0 + KH of column block vt.  Lane (g,c) reg i of S[k] = S[16 (kt0 + k) + 4g + i][16vt + c]
    const int col = wv / PARTS, part = wv % PARTS, kt0 = part * KH;
    const int vt = vt0 + col;
    f32x4 S[KH];
    const int64_t soff = ((int64_t)n * H + h) * K * V + 16 * vt + c;
#pragma unroll
    for (int k = 0; k < KH; ++k) {
        const int kt = kt0 + k;
        S[k] = zero4();
        if (seg > 0) {
            if (!SUM) S[k] = *reinterpret_cast<const f32x4*>(p.seg.in + rec * (K * V) + (vt * KT + kt) * TILE + 4 * l);
            else if (trans) {
#pragma unroll
                for (int i = 0; i < 4; ++i) S[k][i] = (16 * kt + 4 * g + i == 16 * vt + c) ? 1.f : 0.f;
            }
        } else if (p.h0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) S[k][i] = p.h0[soff + (int64_t)(16 * kt + 4 * g + i) * V];
        }
    }
    // The walk, compiled for each part by itself: a wave alone on its SIMD pays some five cycles for every instruction, branches more
    auto walk = [&](auto part_) __attribute__((always_inline)) {
        constexpr int part = decltype(part_)::value, kt0 = part * KH;
        // Two waves of one column block: each has its SIMD to itself, and a step is its chain of latencies: 960 cycles, of them 200 until the parts are on
        // their way into LDS, 140 to the barrier, 270 until v_new is there, 350 for the products.  Left to itself the compiler put the products of x and of
        // o before those that the next step waits for.  Measured, us for the scan, before -> after, the same bits: K = V = 128, 97 chunks, 16 heads 44.3 -> 41.6,
        // 44, 8 heads 22.3 -> 21.2; K = 128, V = 64, 63 chunks, 16 heads 30.0 -> 28.3; both backward scans 45 -> 43, 22.9 -> 20.4, 30.5 -> 29.3.  With two blocks,
        // or at K = 64, it was the same time.  Four waves a block (a channel tile pair each) took 47: the parts of four have to be read and added.
        constexpr bool ALONE = NWC == 1 && PARTS > 1;
        constexpr bool first = part == 0, from_u = part == PARTS - 1;   // the wave with the output, and the one that starts v_new from u
        // A chunk's operands, read as soon as the chunk before has been through with their registers: half a step and more before they are used
        Frag<T> w[2][KH], qg[WITH_O ? KH : 1], kgt[HD ? 1 : KH], bgt[2][KH], aqk, aqb[2], ut[2], vtt;
        f32x4 egl[KH];
        // (the lane's offset is all of an address that the wave holds in vector registers: the rest is the slot's and immediate)
        const uint32_t lo = 16 * l, ge = 16 * g;
        auto pair_at = [&](uint32_t so, int off, Frag<T>& f0, Frag<T>& f1) __attribute__((always_inline)) {
            const s16x8 y = *reinterpret_cast<const s16x8*>(smem + so + lo + off);
            f0.v = __builtin_shufflevector(y, y, 0, 1, 2, 3);
            f1.v = __builtin_shufflevector(y, y, 4, 5, 6, 7);
        };
        auto read_u = [&](int t) __attribute__((always_inline)) {
            const T* ub = reinterpret_cast<const T*>(smem + C::UBUF + (t & 1) * C::UB) + col * (3 * TILE);
            if constexpr (from_u) ld_pair(ub, ut[0], ut[1]);
            vtt = ld_tile(ub + PAIR);
        };
        auto read_first = [&](uint32_t so) __attribute__((always_inline)) {
#pragma unroll
            for (int kp = 0; kp < KH2; ++kp) {
                pair_at(so, B.W + (part * KH2 + kp) * 1024, w[0][2 * kp], w[0][2 * kp + 1]);
                pair_at(so, B.W + (KT2 + part * KH2 + kp) * 1024, w[1][2 * kp], w[1][2 * kp + 1]);
            }
#pragma unroll
            for (int kp = 0; kp < KH2; ++kp) {
                if constexpr (WITH_O) pair_at(so, B.QG + (part * KH2 + kp) * 1024, qg[2 * kp], qg[2 * kp + 1]);
                if constexpr (!HD) pair_at(so, B.KGT + (part * KH2 + kp) * 1024, kgt[2 * kp], kgt[2 * kp + 1]);
            }
#pragma unroll
            for (int k = 0; k < KH; ++k) egl[k] = *reinterpret_cast<const f32x4*>(smem + so + ge + B.EGL + 64 * (kt0 + k));
            if constexpr (WITH_O && first) aqk.v = *reinterpret_cast<const s16x4*>(smem + so + lo / 2 + B.AQK);
        };
        auto read_rest = [&](uint32_t so) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < KH; ++k) {
                if constexpr (!KEPT) pair_at(so, B.BGT + (kt0 + k) * 1024, bgt[0][k], bgt[1][k]);
                else {                                    // half a pair each, into the place that the product wants it in
                    const int at = B.BGT + (kt0 + k) / 2 * 1024 + (k & 1) * 8;
                    bgt[0][k].v = *reinterpret_cast<const s16x4*>(smem + so + lo + at);
                    bgt[1][k].v = *reinterpret_cast<const s16x4*>(smem + so + lo + at + KT2 * 1024);
                }
            }
            if constexpr (WITH_O && first) pair_at(so, B.AQB, aqb[0], aqb[1]);
        };
        // the column block's area: the parts of the first wave, then those of the second
        char* const xcol = smem + C::XBUF + col * C::XP + l * 16;
        lds_barrier();
        read_u(0);
        read_first(0);
        read_rest(0);
        uint32_t so = 0;
#pragma unroll 1
        for (int t = 0; t < nchunks; ++t) {
            so = so == (SLOTS - 1) * SLOT ? 0 : so + SLOT;
            char* const xt = xcol + (t & 1) * C::XB;
            // ---- own channels' part of v_new^T (rows value, inner token) = u^T + S^T w^T, and of qg S
            Frag<T> sb[KH];
            f32x4 vn[2] = {zero4(), zero4()}, o = zero4();
            if constexpr (from_u) { vn[0] = to_f32(ut[0]); vn[1] = to_f32(ut[1]); }
#pragma unroll
            for (int kp = 0; kp < KH2; ++kp) {
                sb[2 * kp] = to_frag<T>(S[2 * kp]);
                sb[2 * kp + 1] = to_frag<T>(S[2 * kp + 1]);
                vn[0] = mm2(sb[2 * kp], sb[2 * kp + 1], w[0][2 * kp], w[0][2 * kp + 1], vn[0]);
                vn[1] = mm2(sb[2 * kp], sb[2 * kp + 1], w[1][2 * kp], w[1][2 * kp + 1], vn[1]);
            }
            if constexpr (WITH_O) {
#pragma unroll
                for (int kp = 0; kp < KH2; ++kp) o = mm2(qg[2 * kp], qg[2 * kp + 1], sb[2 * kp], sb[2 * kp + 1], o);
            }
            if constexpr (OUT == OUT_STATE || STATES) {
                // checkpoint of the entering state, as the fragments held here (tile pairs, 16 bytes per lane, whole cache lines): the
                // chunk_grad kernel turns them the way it needs them
                T* const hc = p.ws.HC + (chw0 + t) * (K * V) + (part * KH2 * (V / 16) + vt) * PAIR;
#pragma unroll
                for (int kp = 0; kp < KH2; ++kp) st_pair2_past(hc + kp * (V / 16) * PAIR, sb[2 * kp], sb[2 * kp + 1]);
            }
            // ---- what is one product a sum: the chunk's own part of the state, A_qk v
            f32x4 x[KH + 1];
#pragma unroll
            for (int k = 0; k < KH; ++k) x[k] = mm(vtt, HD ? bgt[1][k] : kgt[HD ? 0 : k], S[k] * egl[k]);
            x[KH] = zero4();
            if constexpr (WITH_O && first) x[KH] = mm(aqk, vtt, x[KH]);
            if constexpr (PARTS > 1) {
                *reinterpret_cast<f32x4*>(xt + part * 2048) = vn[0];
                *reinterpret_cast<f32x4*>(xt + part * 2048 + 1024) = vn[1];
                if constexpr (WITH_O && !first) *reinterpret_cast<f32x4*>(xt + 4096) = o;
            }
            // (alone on its SIMD, a wave has the products of x issued in front of the barrier, while the parts are on their way into LDS, and those of S in
            // front of o's: see ALONE)
            if constexpr (ALONE) __builtin_amdgcn_sched_barrier(0);
            // the parts are there; so are chunk t + 1 and its u, and chunk t has been read by all
            lds_barrier();
            f32x4 ov[2], oo;
            if constexpr (PARTS > 1) {
                ov[0] = *reinterpret_cast<const f32x4*>(xt + (1 - part) * 2048);
                ov[1] = *reinterpret_cast<const f32x4*>(xt + (1 - part) * 2048 + 1024);
                if constexpr (WITH_O && first) oo = *reinterpret_cast<const f32x4*>(xt + 4096);
            }
            __builtin_amdgcn_sched_barrier(0);            // (before the reads of the next chunk: they are what is waited for)
            read_u(t + 1);
            read_first(so);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!ALONE) settle<T>(x);
            if constexpr (PARTS > 1) {
                vn[0] += ov[0];
                vn[1] += ov[1];
            }
            const Frag<T> vnb[2] = {to_frag<T>(vn[0]), to_frag<T>(vn[1])};
            // ---- S <- exp(g_last) S + kg^T v + sum_s bg_s^T v_new_s
#pragma unroll
            for (int k = 0; k < KH; ++k) S[k] = mm2(vnb[0], vnb[1], bgt[0][k], bgt[1][k], x[k]);
            if constexpr (ALONE) __builtin_amdgcn_sched_barrier(0);
            if constexpr (WITH_O && first) {
                // o (rows token, inner value) = A_qk v + qg S + sum_s A_qb^s v_new_s
                if constexpr (PARTS > 1) o += oo;
                o = mm2(aqb[0], aqb[1], vnb[0], vnb[1], o + x[KH]);
            }
            __builtin_amdgcn_sched_barrier(0);
            read_rest(so);
            if constexpr (WITH_O && first) st_frag(reinterpret_cast<T*>(smem + C::OUTBOX + (t & 1) * C::OB + c * C::OROW) + 16 * col + 4 * g, to_frag<T>(o));
        }
        if (WITH_O) lds_barrier();                          // hands over the last output
    };
    if (nchunks > 0) {
        if (PARTS == 1 || part == 0) walk(std::integral_constant<int, 0>());
        else walk(std::integral_constant<int, PARTS - 1>());
    }
    if (SUM) {
        // the record: column block vt of the state, or (trans) of the transition matrix, whose tile (kt, vt) is kept with rows k, inner k'
        const Frag<float> identf = ident_frag<float>();
#pragma unroll
        for (int k = 0; k < KH; ++k) {
            const int kt = kt0 + k;
            if (trans) {
                Frag<float> f;
                f.v = S[k];
                f = transpose(f, identf);                 // exact: fp32 products with ones and zeros
                *reinterpret_cast<f32x4*>(p.seg.tr + rec * (K * K) + (kt * KT + vt) * TILE + 4 * l) = f.v;
                if (p.seg.turned) *reinterpret_cast<f32x4*>(p.seg.turned + rec * (K * K) + (vt * KT + kt) * TILE + 4 * l) = S[k];
            } else {
                *reinterpret_cast<f32x4*>(p.seg.loc + rec * (K * V) + (vt * KT + kt) * TILE + 4 * l) = S[k];
            }
        }
    } else if (p.ht && seg == p.seg.nseg - 1) {
#pragma unroll
        for (int k = 0; k < KH; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) p.ht[soff + (int64_t)(16 * (kt0 + k) + 4 * g + i) * V] = S[k][i];
    }
}

// grid = (H, SPLIT, N * segments), as the other scans' (scan_impl.cuh)
template <int K, int V, int NWC, int KEPT, bool HD>
__global__ __launch_bounds__((OutCfg<K, V, NWC, OUT_O, HD>::THREADS)) void scan_out_kernel(ChunkArgs<bf16> p) {
    __shared__ __attribute__((aligned(16))) char smem[OutCfg<K, V, NWC, OUT_O, HD>::BYTES];
    const int z = blockIdx.z / p.seg.nseg, seg = blockIdx.z % p.seg.nseg;
    scan_out_body<K, V, NWC, OUT_O, KEPT, HD>(p, smem, scan_sequence(p.st, z), seg, blockIdx.y);
}
// Packed sequences that share the device by their lengths (see share_device, prep.hip): grid = (H, workgroups of a head).  Waves that a narrow
// workgroup has no use for end at once; barriers are among those that are left.  Measured, us, one width for all -> this, K = V = 128, 16 heads: forward
// pass of 1731 + 37 + 2204 + 1031 tokens 136 -> 131 (the scan 81 -> 72), of 9000 in 6 sequences, the longest 3700, 298 -> 262, of 6000 in 12 of
// similar lengths 137.7 -> 138.0; 12000 in 12, 8 heads 209 -> 186; training steps of 6000 in 6 748 -> 683, of 1500 in 7, 12 heads 174 -> 153, of
// 16384 in 4 1726 -> 1705 (its two scans are at their traffic, 2.2 GB in 520 us, in every width).  Where one block a workgroup for all fits the device,
// that is faster still and stays.  Beyond 32 sequences the device is full with the widest workgroups for all but the last few steps.
template <int K, int V, int KEPT, bool HD>
__global__ __launch_bounds__((OutCfg<K, V, 4, OUT_O, HD>::THREADS)) void scan_out_share_kernel(ChunkArgs<bf16> p) {
    typedef OutCfg<K, V, 4, OUT_O, HD> C4;
    typedef OutCfg<K, V, 2, OUT_O, HD> C2;
    typedef OutCfg<K, V, 1, OUT_O, HD> C1;
    __shared__ __attribute__((aligned(16))) char smem[C4::BYTES > C2::BYTES ? (C4::BYTES > C1::BYTES ? C4::BYTES : C1::BYTES) : C2::BYTES > C1::BYTES ? C2::BYTES : C1::BYTES];
    int n, code, split;
    if (!scan_share<V>(p.st, blockIdx.y, ORDER_OUT, n, code, split)) return;
    if (code == 0) scan_out_body<K, V, 4, OUT_O, KEPT, HD>(p, smem, n, 0, split);
    else if (code == 1) { if ((int)threadIdx.x < C2::THREADS) scan_out_body<K, V, 2, OUT_O, KEPT, HD>(p, smem, n, 0, split); }
    else if ((int)threadIdx.x < C1::THREADS) scan_out_body<K, V, 1, OUT_O, KEPT, HD>(p, smem, n, 0, split);
}
// the segments' records in the forward direction: grid = (H, (V + K) / 16 / NWC, N * (segments - 1))
template <int K, int V, int NWC, bool HD>
__global__ __launch_bounds__((OutCfg<K, V, NWC, OUT_SUM, HD>::THREADS)) void scan_out_sum_kernel(ChunkArgs<bf16> p) {
    __shared__ __attribute__((aligned(16))) char smem[OutCfg<K, V, NWC, OUT_SUM, HD>::BYTES];
    const int z = blockIdx.z / (p.seg.nseg - 1), seg = blockIdx.z % (p.seg.nseg - 1);
    if (seg == 0 && (int)blockIdx.y >= OutCfg<K, V, NWC, OUT_SUM, HD>::SPLIT) return;   // starts from h0: nobody asks for its transition
    scan_out_body<K, V, NWC, OUT_SUM, 0, HD>(p, smem, scan_sequence(p.st, z), seg, blockIdx.y);
}

template <int K, int V, int NWC, bool HD> static hipError_t launch_scan_out_nwc(const ChunkArgs<bf16>& a, int kept, hipStream_t stream) {
    typedef OutCfg<K, V, NWC, OUT_O, HD> C;
    const dim3 grid(a.H, C::SPLIT, a.st.N * a.seg.nseg), block(C::THREADS);
    if (kept == 2) hipLaunchKernelGGL((scan_out_kernel<K, V, NWC, 2, HD>), grid, block, 0, stream, a);
    else if (kept) hipLaunchKernelGGL((scan_out_kernel<K, V, NWC, 1, HD>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((scan_out_kernel<K, V, NWC, 0, HD>), grid, block, 0, stream, a);
    return hipGetLastError();
}
// Column blocks a workgroup: as few as give each workgroup a compute unit of its own (every workgroup fetches the chunks' blocks for
// itself).  A forward pass, us, two blocks and one, 128 chunks in one segment: K = V = 128, 1 lane 82 and 73, 16 lanes 102 and 96, 32 lanes 135 and
// 127; K = 64, V = 128, 8 lanes 71 and 59, 32 lanes 88 and 79; of 16 chunks K = V = 128 22.3 and 20.8.  The scan alone, two and four: K = V = 128,
// 128 heads 193 and 146, 64 heads 101 and 114.
template <int K, int V, bool HD> static hipError_t launch_scan_out_hd(const ChunkArgs<bf16>& a, int kept, hipStream_t stream) {
    constexpr int VT = V / 16;
    const int lanes = a.H * a.st.N * a.seg.nseg;
    if (lanes * VT <= SCAN_TARGET_WORKGROUPS) return launch_scan_out_nwc<K, V, 1, HD>(a, kept, stream);
    if (scan_shares(a.st.cu, a.st.N, a.H, V, a.seg.nseg, 1)) {
        const dim3 grid(a.H, share_most(a.H, 1, a.st.N, V)), block(OutCfg<K, V, 4, OUT_O, HD>::THREADS);
        if (kept == 2) hipLaunchKernelGGL((scan_out_share_kernel<K, V, 2, HD>), grid, block, 0, stream, a);
        else if (kept) hipLaunchKernelGGL((scan_out_share_kernel<K, V, 1, HD>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((scan_out_share_kernel<K, V, 0, HD>), grid, block, 0, stream, a);
        return hipGetLastError();
    }
    if (lanes * (VT / 2) <= SCAN_TARGET_WORKGROUPS) return launch_scan_out_nwc<K, V, 2, HD>(a, kept, stream);
    return launch_scan_out_nwc<K, V, 4, HD>(a, kept, stream);
}
template <int K, int V> hipError_t launch_scan_out_shape(const ChunkArgs<bf16>& a, int kept, hipStream_t stream) {
    return a.beta ? launch_scan_out_hd<K, V, true>(a, kept, stream) : launch_scan_out_hd<K, V, false>(a, kept, stream);
}
// the segments' records, chained into what enters the segments
template <int K, int V> hipError_t launch_scan_out_segments_shape(const ChunkArgs<bf16>& a, hipStream_t stream) {
    constexpr int NWC = 4;
    const dim3 grid(a.H, (V + K) / 16 / NWC, a.st.N * (a.seg.nseg - 1)), block(OutCfg<K, V, NWC, OUT_SUM, false>::THREADS);
    if (a.beta) hipLaunchKernelGGL((scan_out_sum_kernel<K, V, NWC, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((scan_out_sum_kernel<K, V, NWC, false>), grid, block, 0, stream, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? launch_scan_chain<bf16, K, V>(a, SEG_FWD, stream) : e;
}

}  // namespace hdla
