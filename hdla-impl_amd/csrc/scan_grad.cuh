// The scans of the backward pass for 2-byte elements.  scan_rev: the reverse recurrence of the state gradient, its checkpoints and dh0
// (HRDPLR/bwd_triton.py:127-222) with dv_new (HRDPLR/bwd_triton.py:30-105); the forward one, which leaves the states that enter the
// chunks, is scan_out.cuh's without the output.  They need the prep kernel only, not each other, and run as one launch.
//
// What bounds a step and how it is laid out: see scan_out.cuh, whose division of work the reverse scan has (two waves a column block at
// K = 128, blocks straight to LDS, a wave of its own for what does not depend on the state: here do^T and do^T A_qb).  Two things differ:
//  * it takes b and w turned, rows channel and rows token, which the block holds the other way round: ds_read_tr16_b64, the
//    transposing LDS read, gives them, half a pair each, so that the two ranks of a tile come to lie side by side as mm2 wants them.
//    Sixteen lanes of such a read take every fourth 16-byte piece of a tile pair's, all from the same banks; so the pieces of row group
//    g lie turned by 4 g, which the lanes that ask for them from global memory see to, and those sixteen meet each bank once;
//  * the results, the gradients of states and of v_new, leave straight from the computing waves (16 bytes a lane, whole lines; nothing
//    waits for them; through LDS and a wave that copies them it was the same time).
// Measured, us for the launch with both scans, before (scan_impl.cuh's form, four waves that moved data and turned tiles by products with the
// identity) -> after: K = V = 128, 2048 tokens, 32 heads 151 -> 144, 64 heads 227 -> 215, 128 heads 452 -> 433; 1537 tokens, 16 heads 81 -> 64;
// four sequences of 16384 tokens together, the longest 6144, 16 heads 568 -> 523; K = 64, V = 128, 16 heads 62 -> 54.  With many heads it is the
// traffic (K = V = 128: 72 KiB written and some 60 read a chunk and head: at copy rate 220 us for the 64 heads); with few the chain of steps,
// 0.48 us each, and beside it the writes: 16 heads 64 us, 47 with every chunk's results written to one place, 45 with its loads from one too.
#pragma once
#include "scan_out.cuh"

namespace hdla {

template <int K, int V, int NWC, bool SUM> struct RevCfg {
    static constexpr int VT = V / 16, SPLIT = VT / NWC, KT = K / 16;
    // LDS slot: W and BGT (turned by 4 g), EGL, QGT; a_qb goes to the wave that forms do^T A_qb
    static constexpr SlotB B = slot_bwd(K, 2);
    static constexpr int NI = B.AQBT / 1024, SLOT = NI * 1024;
    static_assert(B.AQBT % 1024 == 0, "whole pieces");
    static constexpr int PARTS = K / 64, KH = KT / PARTS, NC = NWC * PARTS;
    static constexpr int NL = 2, NM = NL + 1;
    static constexpr int CNT = (NI + NL - 1) / NL;
    static constexpr int THREADS = 64 * (NC + NM);
    static constexpr int DB = NWC * 2560;                 // do^T (a tile) and do^T A_qb^s (two of fp32) of the column blocks; two chunks' of them
    static constexpr int XP = 4 * 1024, XB = PARTS > 1 ? NWC * XP : 0;   // the parts of dv_new that the waves of a column block hand each other
    static constexpr int REST = 2 * (DB + XB);
    static constexpr int ROOM = (4 * SLOT + REST <= 80 * 1024 ? 80 : 160) * 1024 - REST;
    static constexpr int MOST = 62 / CNT + 1 < 8 ? 62 / CNT + 1 : 8, SLOTS = ROOM / SLOT < MOST ? ROOM / SLOT : MOST;
    static_assert(SLOTS >= 3 && (SLOTS - 1) * CNT < 63, "a chunk to read, the next one, and one on its way; the memory counter's range");
    static constexpr int DBUF = SLOTS * SLOT, XBUF = DBUF + 2 * DB, BYTES = XBUF + 2 * XB;
};

// Step t handles chunk c1 - 1 - t.
template <int K, int V, int NWC, bool SUM>
__device__ __forceinline__ void scan_rev_body(const ChunkArgs<bf16>& p, char* smem, int n, int seg, int split) {
    typedef RevCfg<K, V, NWC, SUM> C;
    typedef bf16 T;
    constexpr int KT = C::KT, KT2 = KT / 2, VT = C::VT, SLOTS = C::SLOTS, SLOT = C::SLOT, PARTS = C::PARTS, KH = C::KH, KH2 = KH / 2;
    constexpr SlotB B = C::B;
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
    const int nchunks = c1 - c0, last = nchunks - 1;
    const int64_t chw0 = (int64_t)h * p.st.nch + c0;      // chunk of step t: chw0 + last - t

    if (wv >= C::NC) {
        // ---- waves that move data; barriers as in scan_out.cuh, without one for a last output
        if (nchunks <= 0) return;
        const int hw = forming_first<C>(wv - C::NC);
        if (hw < C::NL) {
            const int sf = p.ws.sa_stride;
            constexpr int SB = blk_bwd(K, 2).SIZE;
            const char* const fwd = reinterpret_cast<const char*>(p.ws.W) + chw0 * sf;
            const char* const rev = reinterpret_cast<const char*>(p.ws.QGT) + chw0 * SB;
            const int turned = ((l & 48) + ((l - 4 * g) & 15)) * 16, plain = l * 16;
            int slot = 0;
            auto load = [&](int t) __attribute__((always_inline)) {
                const int at = max(last - t, 0);          // past the end: the segment's first chunk again, never looked at
                const char* const ft = fwd + (int64_t)at * sf;
                const char* const rt = rev + (int64_t)at * SB;
#pragma unroll
                for (int j = 0; j < C::CNT; ++j) {
                    const int i = min(hw + j * C::NL, C::NI - 1);
                    const char* const src = i < B.NIF ? ft + i * 1024 + turned : i == B.NIF ? ft + B.EGL_SRC + plain : rt + (i - B.NIF - 1) * 1024 + plain;
                    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                                     (__attribute__((address_space(3))) void*)(smem + slot * SLOT + i * 1024), 16, 0, 0);
                }
                slot = slot + 1 == SLOTS ? 0 : slot + 1;
            };
#pragma unroll
            for (int d = 0; d < SLOTS; ++d) load(d);
            wait_loads<(SLOTS - 1) * C::CNT>();           // step 0's is there
            __builtin_amdgcn_s_barrier();
            for (int t = 0; t < nchunks; ++t) {
                wait_loads<(SLOTS - 2) * C::CNT>();       // step t + 1's
                __builtin_amdgcn_s_barrier();
                load(t + SLOTS);                          // where step t's was
            }
            wait_loads<0>();                              // nothing may arrive in LDS that is no longer this workgroup's
        } else {
            // do^T and do^T A_qb^s of the workgroup's column blocks, a chunk ahead; the operands come through registers, UD chunks ahead
            constexpr int UD = 3;
            struct Own { i32x4 aq; Frag<T> d[NWC]; };
            const Frag<T> ident = ident_frag<T>();
            // rows of do, as those of v in scan_out.cuh
            const int len_last = (int)min((int64_t)CH, eos - (bos + (int64_t)last * CH));
            const uint32_t row = (uint32_t)(H * V) * sizeof(T), whole = c * row + 8 * g, ragged = min(c, len_last - 1) * row + 8 * g;
            const T* const do0 = p.dout + (bos * H + h) * V + 16 * (trans ? 0 : vt0);
            auto request = [&](int t) __attribute__((always_inline)) {
                const int i = max(last - t, 0);
                Own o;
                o.aq = *reinterpret_cast<const i32x4*>(reinterpret_cast<const char*>(p.ws.QGT) + (chw0 + i) * blk_bwd(K, 2).SIZE +
                                                       blk_bwd(K, 2).AQBT + 16 * l);
#pragma unroll
                for (int j = 0; j < NWC; ++j) o.d[j] = ld_frag(at(do0 + (int64_t)i * (CH * H * V) + (trans ? 0 : 16 * j), i == last ? ragged : whole));
                return o;
            };
            auto form = [&](int t, const Own& o) __attribute__((always_inline)) {
                const int len = t > 0 ? CH : len_last;
                char* const db = smem + C::DBUF + (t & 1) * C::DB;
                const s16x8 y = __builtin_bit_cast(s16x8, o.aq);
                Frag<T> aq[2], doT[NWC];
                aq[0].v = __builtin_shufflevector(y, y, 0, 1, 2, 3);
                aq[1].v = __builtin_shufflevector(y, y, 4, 5, 6, 7);
#pragma unroll
                for (int j = 0; j < NWC; ++j) doT[j] = transpose((c >= len || trans) ? zero_frag<T>() : o.d[j], ident);
#pragma unroll
                for (int j = 0; j < NWC; ++j) {
                    st_tile(reinterpret_cast<T*>(db + j * 2560), doT[j]);
#pragma unroll
                    for (int s = 0; s < 2; ++s) *reinterpret_cast<f32x4*>(db + j * 2560 + 512 + s * 1024 + 16 * l) = mm(doT[j], aq[s], zero4());
                }
            };
            Own own[UD];                                  // step t's in own[t % UD]
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
            int t0 = 0;
#pragma unroll 1
            for (; t0 + UD <= nchunks; t0 += UD) {
#pragma unroll
                for (int j = 0; j < UD; ++j) step(t0 + j, own[(j + 1) % UD]);
            }
#pragma unroll
            for (int j = 0; j < UD - 1; ++j)
                if (t0 + j < nchunks) step(t0 + j, own[(j + 1) % UD]);
        }
        return;
    }

    // ---- computing wave: channel tiles kt0 .. kt0 + KH of column block vt.  Lane (g,c) reg i of dS[k] = dS[16 (kt0 + k) + 4g + i][16vt + c]
    const int col = wv / PARTS, part = wv % PARTS, kt0 = part * KH;
    const int vt = vt0 + col;
    f32x4 dS[KH];
    const int64_t soff = ((int64_t)n * H + h) * K * V + 16 * vt + c;
#pragma unroll
    for (int k = 0; k < KH; ++k) {
        const int kt = kt0 + k;
        dS[k] = zero4();
        if (seg < p.seg.nseg - 1) {
            if (!SUM) dS[k] = *reinterpret_cast<const f32x4*>(p.seg.rin + rec * (K * V) + (vt * KT + kt) * TILE + 4 * l);
            else if (trans) {
#pragma unroll
                for (int i = 0; i < 4; ++i) dS[k][i] = (16 * kt + 4 * g + i == 16 * vt + c) ? 1.f : 0.f;
            }
        } else if (p.dht) {
#pragma unroll
            for (int i = 0; i < 4; ++i) dS[k][i] = p.dht[soff + (int64_t)(16 * kt + 4 * g + i) * V];
        }
    }
    auto walk = [&](auto part_) __attribute__((always_inline)) {
        constexpr int part = decltype(part_)::value, kt0 = part * KH;
        constexpr bool ALONE = NWC == 1 && PARTS > 1;
        constexpr bool first = part == 0, from_do = part == PARTS - 1;   // the wave that stores dv_new, and the one that starts it from do
        Frag<T> bg[2][KH], wt[2][KH], qgt[KH], doT;
        f32x4 egl[KH], e[2];
        const uint32_t lo = 16 * l, ge = 16 * g;
        // see ld_turned: row group s % 4 of row 4 g + s / 4, its pieces turned by 4 (s % 4)
        const int rg = c & 3;
        const uint32_t lt = (16 * rg + ((4 * g + (c >> 2) + 4 * rg) & 15)) * 16;
        auto turned_at = [&](uint32_t so, int off, int kt) __attribute__((always_inline)) {
            return ld_turned(smem + so + lt + (off + kt / 2 * 1024 + (kt & 1) * 8));
        };
        auto read_do = [&](int t) __attribute__((always_inline)) {
            const char* const db = smem + C::DBUF + (t & 1) * C::DB + col * 2560;
            doT = ld_tile(reinterpret_cast<const T*>(db));
            if constexpr (from_do) {
                e[0] = *reinterpret_cast<const f32x4*>(db + 512 + lo);
                e[1] = *reinterpret_cast<const f32x4*>(db + 1536 + lo);
            }
        };
        auto read_first = [&](uint32_t so) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < KH; ++k) {
                bg[0][k] = turned_at(so, B.BGT, kt0 + k);
                bg[1][k] = turned_at(so, B.BGT + KT2 * 1024, kt0 + k);
            }
#pragma unroll
            for (int kp = 0; kp < KH2; ++kp) {
                const s16x8 y = *reinterpret_cast<const s16x8*>(smem + so + lo + (B.QGT + (part * KH2 + kp) * 1024));
                qgt[2 * kp].v = __builtin_shufflevector(y, y, 0, 1, 2, 3);
                qgt[2 * kp + 1].v = __builtin_shufflevector(y, y, 4, 5, 6, 7);
            }
#pragma unroll
            for (int k = 0; k < KH; ++k) egl[k] = *reinterpret_cast<const f32x4*>(smem + so + ge + (B.EGL + 64 * (kt0 + k)));
        };
        auto read_rest = [&](uint32_t so) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < KH; ++k) {
                wt[0][k] = turned_at(so, B.W, kt0 + k);
                wt[1][k] = turned_at(so, B.W + KT2 * 1024, kt0 + k);
            }
        };
        char* const xcol = smem + C::XBUF + col * C::XP + l * 16;
        lds_barrier();
        read_do(0);
        read_first(0);
        read_rest(0);
        uint32_t so = 0;
#pragma unroll 1
        for (int t = 0; t < nchunks; ++t) {
            so = so == (SLOTS - 1) * SLOT ? 0 : so + SLOT;
            char* const xt = xcol + (t & 1) * C::XB;
            const int64_t chw = chw0 + (last - t);
            // ---- own channels' part of dv_new_s^T (rows value, inner token) = do^T A_qb^s + dS^T bg_s^T
            Frag<T> dsb[KH];
            f32x4 dvn[2] = {zero4(), zero4()};
            if constexpr (from_do) { dvn[0] = e[0]; dvn[1] = e[1]; }
#pragma unroll
            for (int kp = 0; kp < KH2; ++kp) {
                dsb[2 * kp] = to_frag<T>(dS[2 * kp]);
                dsb[2 * kp + 1] = to_frag<T>(dS[2 * kp + 1]);
                dvn[0] = mm2(dsb[2 * kp], dsb[2 * kp + 1], bg[0][2 * kp], bg[0][2 * kp + 1], dvn[0]);
                dvn[1] = mm2(dsb[2 * kp], dsb[2 * kp + 1], bg[1][2 * kp], bg[1][2 * kp + 1], dvn[1]);
            }
            // ---- gradient of the state leaving the chunk, as the fragments held here (tile pairs)
            if constexpr (!SUM) {
                T* const dhc = p.ws.DHC + chw * (K * V) + (part * KH2 * VT + vt) * PAIR;
#pragma unroll
                for (int kp = 0; kp < KH2; ++kp) st_pair2_past(dhc + kp * VT * PAIR, dsb[2 * kp], dsb[2 * kp + 1]);
            }
            // ---- what is one product a sum: the chunk's own part of the state's gradient
            f32x4 x[KH];
#pragma unroll
            for (int k = 0; k < KH; ++k) x[k] = mm(doT, qgt[k], dS[k] * egl[k]);
            if constexpr (PARTS > 1) {
                *reinterpret_cast<f32x4*>(xt + part * 2048) = dvn[0];
                *reinterpret_cast<f32x4*>(xt + part * 2048 + 1024) = dvn[1];
            }
            if constexpr (ALONE) __builtin_amdgcn_sched_barrier(0);       // (x in front of the barrier, as in scan_out.cuh)
            // the parts are there; so are step t + 1's block and do, and step t's has been read by all
            lds_barrier();
            f32x4 ov[2];
            if constexpr (PARTS > 1) {
                ov[0] = *reinterpret_cast<const f32x4*>(xt + (1 - part) * 2048);
                ov[1] = *reinterpret_cast<const f32x4*>(xt + (1 - part) * 2048 + 1024);
            }
            __builtin_amdgcn_sched_barrier(0);            // (before the reads of the next chunk: they are what is waited for)
            read_do(t + 1);
            read_first(so);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!ALONE) settle<T>(x);
            if constexpr (PARTS > 1) {
                dvn[0] += ov[0];
                dvn[1] += ov[1];
            }
            const Frag<T> dvb[2] = {to_frag<T>(dvn[0]), to_frag<T>(dvn[1])};
            // ---- dS <- exp(g_last) dS + qg^T do + sum_s w_s^T dv_new_s
#pragma unroll
            for (int k = 0; k < KH; ++k) dS[k] = mm2(dvb[0], dvb[1], wt[0][k], wt[1][k], x[k]);
            if constexpr (!SUM && first) st_pair2_past(p.ws.DVN + chw * (2 * CH * V) + vt * PAIR, dvb[0], dvb[1]);
            __builtin_amdgcn_sched_barrier(0);
            read_rest(so);
        }
    };
    if (nchunks > 0) {
        if (PARTS == 1 || part == 0) walk(std::integral_constant<int, 0>());
        else walk(std::integral_constant<int, PARTS - 1>());
    }
    if (SUM) {
        const Frag<float> identf = ident_frag<float>();
#pragma unroll
        for (int k = 0; k < KH; ++k) {
            const int kt = kt0 + k;
            if (trans) {
                Frag<float> f;
                f.v = dS[k];
                f = transpose(f, identf);                 // exact: fp32 products with ones and zeros
                *reinterpret_cast<f32x4*>(p.seg.rtr + rec * (K * K) + (kt * KT + vt) * TILE + 4 * l) = f.v;
            } else {
                *reinterpret_cast<f32x4*>(p.seg.rloc + rec * (K * V) + (vt * KT + kt) * TILE + 4 * l) = dS[k];
            }
        }
    } else if (p.dh0 && seg == 0) {
#pragma unroll
        for (int k = 0; k < KH; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) p.dh0[soff + (int64_t)(16 * (kt0 + k) + 4 * g + i) * V] = dS[k][i];
    }
}

template <int K, int V, int NWC, bool HD> constexpr int grad_lds() {
    return OutCfg<K, V, NWC, OUT_STATE, HD>::BYTES > RevCfg<K, V, NWC, false>::BYTES ? OutCfg<K, V, NWC, OUT_STATE, HD>::BYTES : RevCfg<K, V, NWC, false>::BYTES;
}
// grid = (H, directions * SPLIT, N * segments), as scan_impl.cuh's; blockIdx.y counts from the forward scan's splits on, or (first_dir 1) from
// the reverse one's
template <int K, int V, int NWC, bool HD>
__global__ __launch_bounds__((RevCfg<K, V, NWC, false>::THREADS)) void scan_grad_kernel(ChunkArgs<bf16> p, int first_dir) {
    typedef OutCfg<K, V, NWC, OUT_STATE, HD> F;
    typedef RevCfg<K, V, NWC, false> R;
    static_assert(F::THREADS == R::THREADS, "one launch");
    __shared__ __attribute__((aligned(16))) char smem[grad_lds<K, V, NWC, HD>()];
    const int z = blockIdx.z / p.seg.nseg, seg = blockIdx.z % p.seg.nseg;
    const int n = scan_sequence(p.st, z), y = blockIdx.y + first_dir * R::SPLIT;
    if (y < R::SPLIT) scan_out_body<K, V, NWC, OUT_STATE, 1, HD>(p, smem, n, seg, y);
    else scan_rev_body<K, V, NWC, false>(p, smem, n, seg, y - R::SPLIT);
}
// packed sequences that share the device by their lengths, as scan_out_share_kernel; the two directions in turn
template <int K, int V, bool HD>
__global__ __launch_bounds__((RevCfg<K, V, 4, false>::THREADS)) void scan_grad_share_kernel(ChunkArgs<bf16> p) {
    constexpr int B1 = grad_lds<K, V, 1, HD>(), B2 = grad_lds<K, V, 2, HD>(), B4 = grad_lds<K, V, 4, HD>();
    __shared__ __attribute__((aligned(16))) char smem[B4 > B2 ? (B4 > B1 ? B4 : B1) : B2 > B1 ? B2 : B1];
    int n, code, split;
    if (!scan_share<V>(p.st, blockIdx.y >> 1, ORDER_GRAD, n, code, split)) return;
    const bool rev = blockIdx.y & 1;
    auto walk = [&](auto nwc) __attribute__((always_inline)) {
        constexpr int NWC = decltype(nwc)::value;
        if ((int)threadIdx.x >= RevCfg<K, V, NWC, false>::THREADS) return;
        if (rev) scan_rev_body<K, V, NWC, false>(p, smem, n, 0, split);
        else scan_out_body<K, V, NWC, OUT_STATE, 1, HD>(p, smem, n, 0, split);
    };
    if (code == 0) walk(std::integral_constant<int, 4>());
    else if (code == 1) walk(std::integral_constant<int, 2>());
    else walk(std::integral_constant<int, 1>());
}
// the reverse scan alone, behind a forward pass that has left the entering states: in the widths of that one's scan (a direction has as many slots).
// us a training step, two blocks a workgroup for all -> this, 16 heads, K = V = 128: 16384 tokens in 4 sequences 1443 -> 1425, 9000 in 6, the longest 3700, 905 -> 855
template <int K, int V>
__global__ __launch_bounds__((RevCfg<K, V, 4, false>::THREADS)) void scan_rev_share_kernel(ChunkArgs<bf16> p) {
    constexpr int B1 = RevCfg<K, V, 1, false>::BYTES, B2 = RevCfg<K, V, 2, false>::BYTES, B4 = RevCfg<K, V, 4, false>::BYTES;
    __shared__ __attribute__((aligned(16))) char smem[B4 > B2 ? (B4 > B1 ? B4 : B1) : B2 > B1 ? B2 : B1];
    int n, code, split;
    if (!scan_share<V>(p.st, blockIdx.y, ORDER_OUT, n, code, split)) return;
    if (code == 0) scan_rev_body<K, V, 4, false>(p, smem, n, 0, split);
    else if (code == 1) { if ((int)threadIdx.x < RevCfg<K, V, 2, false>::THREADS) scan_rev_body<K, V, 2, false>(p, smem, n, 0, split); }
    else if ((int)threadIdx.x < RevCfg<K, V, 1, false>::THREADS) scan_rev_body<K, V, 1, false>(p, smem, n, 0, split);
}
// the segments' records on a workspace of the backward pass (or that it will read): grid and first_y as scan_sum_kernel's
template <int K, int V, int NWC, bool HD>
__global__ __launch_bounds__((RevCfg<K, V, NWC, true>::THREADS)) void scan_grad_sum_kernel(ChunkArgs<bf16> p, int first_y) {
    typedef OutCfg<K, V, NWC, OUT_SUM, HD> F;
    typedef RevCfg<K, V, NWC, true> R;
    static_assert(F::THREADS == R::THREADS, "one launch");
    constexpr int COLS = (V + K) / 16 / NWC;
    __shared__ __attribute__((aligned(16))) char smem[F::BYTES > R::BYTES ? F::BYTES : R::BYTES];
    const int z = blockIdx.z / (p.seg.nseg - 1), seg = blockIdx.z % (p.seg.nseg - 1);
    const int n = scan_sequence(p.st, z), y = blockIdx.y + first_y, split = y % COLS;
    if (y < COLS) {
        if (seg == 0 && split >= R::SPLIT) return;        // starts from h0: nobody asks for its transition
        scan_out_body<K, V, NWC, OUT_SUM, 1, HD>(p, smem, n, seg, split);
    } else {
        if (seg + 1 == p.seg.nseg - 1 && split >= R::SPLIT) return;
        scan_rev_body<K, V, NWC, true>(p, smem, n, seg + 1, split);
    }
}

template <int K, int V, int NWC> static hipError_t launch_scan_grad_nwc(const ChunkArgs<bf16>& a, ScanKind kind, hipStream_t stream) {
    typedef RevCfg<K, V, NWC, false> C;
    const dim3 grid(a.H, C::SPLIT * (kind == SCAN_PAIR ? 2 : 1), a.st.N * a.seg.nseg);
    if (a.beta) hipLaunchKernelGGL((scan_grad_kernel<K, V, NWC, true>), grid, dim3(C::THREADS), 0, stream, a, (int)(kind == SCAN_BWD));
    else hipLaunchKernelGGL((scan_grad_kernel<K, V, NWC, false>), grid, dim3(C::THREADS), 0, stream, a, (int)(kind == SCAN_BWD));
    return hipGetLastError();
}
// Column blocks a workgroup: as few as give each workgroup a compute unit of its own.  K = V = 128, 2 x 1537 tokens of 8 heads, one and two
// blocks: 64 and 69 us; 64 heads of 2048 tokens, two and four: 274 and 215 (four sequences of very unequal length: 511 and 523).
template <int K, int V> hipError_t launch_scan_grad_shape(const ChunkArgs<bf16>& a, ScanKind kind, hipStream_t stream) {
    constexpr int VT = V / 16;
    const int lanes = a.H * a.st.N * a.seg.nseg * (kind == SCAN_PAIR ? 2 : 1);
    if (lanes * VT <= SCAN_TARGET_WORKGROUPS) return launch_scan_grad_nwc<K, V, 1>(a, kind, stream);
    if (kind == SCAN_PAIR && scan_shares(a.st.cu, a.st.N, a.H, V, a.seg.nseg, 2)) {
        const dim3 grid(a.H, 2 * share_most(a.H, 2, a.st.N, V)), block(RevCfg<K, V, 4, false>::THREADS);
        if (a.beta) hipLaunchKernelGGL((scan_grad_share_kernel<K, V, true>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((scan_grad_share_kernel<K, V, false>), grid, block, 0, stream, a);
        return hipGetLastError();
    }
    if (kind == SCAN_BWD && scan_shares(a.st.cu, a.st.N, a.H, V, a.seg.nseg, 1)) {
        hipLaunchKernelGGL((scan_rev_share_kernel<K, V>), dim3(a.H, share_most(a.H, 1, a.st.N, V)), dim3(RevCfg<K, V, 4, false>::THREADS), 0, stream, a);
        return hipGetLastError();
    }
    if (lanes * (VT / 2) <= SCAN_TARGET_WORKGROUPS) return launch_scan_grad_nwc<K, V, 2>(a, kind, stream);
    return launch_scan_grad_nwc<K, V, 4>(a, kind, stream);
}
template <int K, int V> hipError_t launch_scan_grad_segments_shape(const ChunkArgs<bf16>& a, SegStart what, hipStream_t stream) {
    constexpr int NWC = 4;
    typedef RevCfg<K, V, NWC, true> C;
    const dim3 grid(a.H, sum_splits<K, V, NWC>(what, a.seg.turned), a.st.N * (a.seg.nseg - 1)), block(C::THREADS);
    if (a.beta) hipLaunchKernelGGL((scan_grad_sum_kernel<K, V, NWC, true>), grid, block, 0, stream, a, (sum_first<K, V, NWC>(what)));
    else hipLaunchKernelGGL((scan_grad_sum_kernel<K, V, NWC, false>), grid, block, 0, stream, a, (sum_first<K, V, NWC>(what)));
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? launch_scan_chain<bf16, K, V>(a, what, stream) : e;
}

}  // namespace hdla
