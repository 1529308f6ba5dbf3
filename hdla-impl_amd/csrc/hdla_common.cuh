// Shared device-side building blocks of the HDLA rank-2 DPLR delta-rule kernels for gfx950 (CDNA4, wave64).
//
// Everything in the chunked path is phrased as products of 16x16 tiles held in MFMA register fragments.
// A "row fragment" F(X) of a 16 x 16 tile X is 4 values per lane: lane (g, c) = (lane / 16, lane % 16)
// holds X[c][4g .. 4g+3], i.e. row c, four consecutive entries of the inner (contracted) dimension.
//
//     mm(F(P), F(Q), acc)   accumulates   Z = P * Q^T   as a row fragment:  lane (g,c) reg i  +=  Z[c][4g+i]
//
// so the rows of the first argument become the rows of the result and the rows of the second argument become
// the inner index of the result.  The result of one product is therefore directly the operand of the next one
// (after conversion to the operand type), which is what lets the inter-chunk state scan run entirely in
// registers.  The two instantiations are bf16 operands (v_mfma_f32_16x16x16_bf16) and fp32 operands
// (four v_mfma_f32_16x16x4_f32 steps with the inner index permuted to match); both accumulate in fp32.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "hdla_ws.h"

namespace hdla {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int CH = 16;       // tokens per chunk
constexpr int MID = 7;       // token whose cumulative log-decay centres the factorised scores
constexpr int RANK = 2;      // rank of the a/b update
constexpr int TILE = 256;    // elements of one 16x16 tile (64 lanes x 4)

template <typename T> struct Frag;
template <> struct Frag<bf16> { s16x4 v; };
template <> struct Frag<float> { f32x4 v; };

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// ---- conversions -------------------------------------------------------------------------------------------
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) {
    // round to nearest even; inputs here are finite by construction
    __bf16 h = (__bf16)f;
    return __builtin_bit_cast(uint16_t, h);
}

template <typename T> __device__ __forceinline__ Frag<T> to_frag(f32x4 a);
template <> __device__ __forceinline__ Frag<bf16> to_frag<bf16>(f32x4 a) {
    // two v_cvt_pk_bf16_f32 (round to nearest even), results already packed in operand order
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const f32x2 lo = {a[0], a[1]}, hi = {a[2], a[3]};
    u32x2 w;
    w[0] = __builtin_bit_cast(unsigned, __builtin_convertvector(lo, bf16x2));
    w[1] = __builtin_bit_cast(unsigned, __builtin_convertvector(hi, bf16x2));
    Frag<bf16> r;
    r.v = __builtin_bit_cast(s16x4, w);
    return r;
}
template <> __device__ __forceinline__ Frag<float> to_frag<float>(f32x4 a) { Frag<float> r; r.v = a; return r; }

__device__ __forceinline__ f32x4 to_f32(Frag<bf16> a) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 w = __builtin_bit_cast(u32x2, a.v);
    f32x4 r;
    r[0] = __uint_as_float(w[0] << 16); r[1] = __uint_as_float(w[0] & 0xffff0000u);
    r[2] = __uint_as_float(w[1] << 16); r[3] = __uint_as_float(w[1] & 0xffff0000u);
    return r;
}
__device__ __forceinline__ f32x4 to_f32(Frag<float> a) { return a.v; }

// Tells the optimiser that x may have changed (it has not, and no instruction is emitted): what is computed from x
// after this point stays after it, in particular inside a loop in which x does not change, instead of being hoisted
// out of the loop and kept in registers across it.
__device__ __forceinline__ void pin(Frag<bf16>& x) { asm volatile("" : "+v"(x.v)); }
__device__ __forceinline__ void pin(f32x4& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void hold(Frag<bf16>& x) { pin(x); }
__device__ __forceinline__ void hold(Frag<float>& x) { pin(x.v); }
__device__ __forceinline__ void pin(Frag<float>&) {}     // fp32 operands are used as they are: nothing to hoist

// The value of x is not needed any more; x is left with whatever its registers hold (no instruction).  For what is refilled under a
// condition: without this the old value stays in its registers until then, for the case that it is not.
template <typename X> __device__ __forceinline__ void forget(X& x) { asm volatile("" : "=v"(x)); }

__device__ __forceinline__ f32x4 zero4() { f32x4 z = {0.f, 0.f, 0.f, 0.f}; return z; }

// ---- the tile product --------------------------------------------------------------------------------------
// acc[lane(g,c)][i] += sum_k P[c][k] * Q[4g+i][k]     (frows = F(P), finner = F(Q))
__device__ __forceinline__ f32x4 mm(Frag<bf16> frows, Frag<bf16> finner, f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(finner.v, frows.v, acc, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mm(Frag<float> frows, Frag<float> finner, f32x4 acc) {
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(finner.v[s], frows.v[s], acc, 0, 0, 0);
    return acc;
}

// Two products of 2-byte operands in one instruction, acc += P0 Q0^T + P1 Q1^T: the 16x16x32 MFMA, whose operands are two
// tiles' fragments side by side (which inner index a lane's element stands for is free as long as both operands agree).
// Measured, cycles of a SIMD an instruction: 16 either way, also in a chain through the accumulator, so it is two products
// in the time of one.
// An accumulator must not go from mm to mm2 or back without settle(): a result is handed to the next product's accumulator
// inside the matrix unit, which works between two instructions of one shape, and the compiler, which takes the two shapes for one
// in this respect, inserts no wait.  Measured: with less than 5 wait states in between the second product adds to another
// number (back to back, a relative difference of 0.5 to 0.6; from 5 on none); results used as operands, or by vector
// instructions, are waited for correctly.  test_mfma_chains.py looks through the built kernels for such pairs.
// Where it counts: the fused kernels' waves wait mostly for the instructions of the others on their SIMD.  Forward kernel, 4 x 2048
// tokens of 16 heads, K = V = 64: 354 -> 222 products a chunk and head, 72.2 -> 69.5 us (the chain of a consumer's step half as long).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ bf16x8 side_by_side(Frag<bf16> x, Frag<bf16> y) {
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(x.v, y.v, 0, 1, 2, 3, 4, 5, 6, 7));
}
__device__ __forceinline__ f32x4 mm2(Frag<bf16> p0, Frag<bf16> p1, Frag<bf16> q0, Frag<bf16> q1, f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(side_by_side(q0, q1), side_by_side(p0, p1), acc, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mm2(Frag<float> p0, Frag<float> p1, Frag<float> q0, Frag<float> q1, f32x4 acc) {
    return mm(p1, q1, mm(p0, q0, acc));
}
// the accumulators x have left the matrix unit: 8 wait states between what produced them and what uses them
template <typename T, int N> __device__ __forceinline__ void settle(f32x4 (&x)[N]) {
    if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
        asm volatile("s_nop 7");
#pragma unroll
        for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
    }
}

// Split operands for the score products of the bf16 path: x = hi + lo with both halves bf16, and
// P Q^T ~ (Ph + Pl) (Qh + Ql)^T, which removes the rounding of the decayed operands (the largest single
// contribution to the forward error) at the price of one more MFMA per product: [Ph Ph] [Qh Ql]^T and [Pl Pl] [Qh Ql]^T.
// fp32 operands need no split.
template <typename T> struct Split;
template <> struct Split<bf16> { Frag<bf16> hi, lo; };
template <> struct Split<float> { Frag<float> hi; };
__device__ __forceinline__ void split(f32x4 x, Split<bf16>& s) {
    s.hi = to_frag<bf16>(x);
    s.lo = to_frag<bf16>(x - to_f32(s.hi));
}
__device__ __forceinline__ void split(f32x4 x, Split<float>& s) { s.hi.v = x; }
__device__ __forceinline__ f32x4 mm_split(const Split<bf16>& p, const Split<bf16>& q, f32x4 acc) {
    acc = mm2(p.lo, p.lo, q.hi, q.lo, acc);
    return mm2(p.hi, p.hi, q.hi, q.lo, acc);
}
__device__ __forceinline__ f32x4 mm_split(const Split<float>& p, const Split<float>& q, f32x4 acc) { return mm(p.hi, q.hi, acc); }
// one p against several q: the halves of p one after the other, so that only one is held twice at a time
template <int N> __device__ __forceinline__ void mm_split(const Split<bf16>& p, const Split<bf16>* const (&q)[N], f32x4* const (&acc)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) *acc[i] = mm2(p.lo, p.lo, q[i]->hi, q[i]->lo, *acc[i]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < N; ++i) *acc[i] = mm2(p.hi, p.hi, q[i]->hi, q[i]->lo, *acc[i]);
}

// F(I16): used to transpose a tile with one product, F(X^T) = mm(F(I), F(X)).
template <typename T> __device__ __forceinline__ Frag<T> ident_frag() {
    const int l = lane_id(), g = l >> 4, c = l & 15;
    f32x4 e;
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = (c == 4 * g + i) ? 1.f : 0.f;
    return to_frag<T>(e);
}
template <typename T> __device__ __forceinline__ Frag<T> transpose(Frag<T> x, Frag<T> ident) {
    return to_frag<T>(mm(ident, x, zero4()));
}

// The same of 4-byte elements through LDS, bit for bit: as a product it is four of 32 cycles, and prep and chunk_grad wait for products (a quarter and
// more of theirs were these).  scratch: TURN_SCRATCH bytes of the wave's own, 16-byte aligned (accesses of one wave complete in order: no barrier, and
// the area can be used again at once); rows padded so that neither the writes nor the reads meet a bank twice.  Measured, us, products -> this,
// K = V = 64: chunk_grad of 1008 (chunk, head) 52.8 -> 49.1, of 1408, beta form, 62 -> 57, prep 29.9 -> 26.2, of 8192 104 -> 99; K = 64, V = 128, 1008
// 87 -> 79 and 33 -> 30; K = 128, V = 64 56 -> 52.5.  Not in the reverse scan, which turns tiles between the layouts of its LDS slots: 27.2 -> 29.0.
constexpr int TURN_ROW = 20, TURN_SCRATCH = 16 * TURN_ROW * 4;
__device__ __forceinline__ Frag<float> turn(Frag<float> x, Frag<float>, char* scratch) {
    const int l = lane_id(), g = l >> 4, c = l & 15;
    float* const t = reinterpret_cast<float*>(scratch);
    *reinterpret_cast<f32x4*>(t + c * TURN_ROW + 4 * g) = x.v;
    Frag<float> r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r.v[i] = t[(4 * g + i) * TURN_ROW + c];
    return r;
}
__device__ __forceinline__ Frag<bf16> turn(Frag<bf16> x, Frag<bf16> ident, char*) { return transpose(x, ident); }

// Address = uniform base (it stays in scalar registers) + a 32-bit byte offset per lane.  This is the form the
// global memory instructions take directly: one address register per lane instead of two, no 64-bit vector adds.
template <typename T> __device__ __forceinline__ T* at(T* ubase, uint32_t byte_off) {
    return reinterpret_cast<T*>(reinterpret_cast<char*>(ubase) + byte_off);
}
template <typename T> __device__ __forceinline__ const T* at(const T* ubase, uint32_t byte_off) {
    return reinterpret_cast<const T*>(reinterpret_cast<const char*>(ubase) + byte_off);
}

// ---- fragment loads / stores -------------------------------------------------------------------------------
// four consecutive elements at p (8-byte aligned for bf16, 16-byte aligned for fp32)
__device__ __forceinline__ Frag<bf16> ld_frag(const bf16* p) { Frag<bf16> r; r.v = *reinterpret_cast<const s16x4*>(p); return r; }
__device__ __forceinline__ Frag<float> ld_frag(const float* p) { Frag<float> r; r.v = *reinterpret_cast<const f32x4*>(p); return r; }
__device__ __forceinline__ void st_frag(bf16* p, Frag<bf16> f) { *reinterpret_cast<s16x4*>(p) = f.v; }
__device__ __forceinline__ void st_frag(float* p, Frag<float> f) { *reinterpret_cast<f32x4*>(p) = f.v; }
template <typename T> __device__ __forceinline__ Frag<T> zero_frag() { return to_frag<T>(zero4()); }

// Masked load without a branch: p must be a readable address on every lane (callers clamp the row index);
// lanes with ok == false get zeros by a select after the load.  A branch around the load would stop the
// compiler from batching the loads of an unrolled loop, so every load would pay its own memory latency.
template <typename T> __device__ __forceinline__ Frag<T> ld_frag_sel(const T* p, bool ok) {
    Frag<T> f = ld_frag(p);
    Frag<T> z = zero_frag<T>();
    Frag<T> r;
    r.v = ok ? f.v : z.v;
    return r;
}

// one element stores (used for the strided, 4-rows-per-lane writes of row-major checkpoints)
__device__ __forceinline__ void st_elem(bf16* p, float x) { p->x = f2bf(x); }
__device__ __forceinline__ void st_elem(float* p, float x) { *p = x; }
__device__ __forceinline__ float ld_elem(const bf16* p) { return bf2f(p->x); }
__device__ __forceinline__ float ld_elem(const float* p) { return *p; }

// whole tile in fragment order: lane l owns elements [4l, 4l+4) of a 256-element block
template <typename T> __device__ __forceinline__ Frag<T> ld_tile(const T* tile) { return ld_frag(tile + 4 * lane_id()); }
template <typename T> __device__ __forceinline__ void st_tile(T* tile, Frag<T> f) { st_frag(tile + 4 * lane_id(), f); }

// Two tiles that one consumer lane always needs together are stored interleaved as a pair (1024 bytes for bf16):
// element 8*lane + 4*which + i, so that both fragments arrive with one 16-byte load per lane.  The scans are
// limited by the number of memory instructions a wave may have in flight, not by bytes.
typedef short s16x8 __attribute__((ext_vector_type(8)));
constexpr int PAIR = 2 * TILE;
__device__ __forceinline__ void ld_pair(const bf16* pair, Frag<bf16>& f0, Frag<bf16>& f1) {
    const s16x8 x = *reinterpret_cast<const s16x8*>(pair + 8 * lane_id());
    f0.v = __builtin_shufflevector(x, x, 0, 1, 2, 3);
    f1.v = __builtin_shufflevector(x, x, 4, 5, 6, 7);
}
__device__ __forceinline__ void ld_pair(const float* pair, Frag<float>& f0, Frag<float>& f1) {
    f0.v = *reinterpret_cast<const f32x4*>(pair + 8 * lane_id());
    f1.v = *reinterpret_cast<const f32x4*>(pair + 8 * lane_id() + 4);
}
template <typename T> __device__ __forceinline__ Frag<T> ld_pair_one(const T* pair, int which) {
    return ld_frag(pair + 8 * lane_id() + 4 * which);
}
template <typename T> __device__ __forceinline__ void st_pair(T* pair, int which, Frag<T> f) {
    st_frag(pair + 8 * lane_id() + 4 * which, f);
}
// both tiles of a pair at once: whole 16-byte pieces, so no cache line is ever written in two halves
__device__ __forceinline__ void st_pair2(bf16* pair, Frag<bf16> f0, Frag<bf16> f1) {
    const s16x8 x = __builtin_shufflevector(f0.v, f1.v, 0, 1, 2, 3, 4, 5, 6, 7);
    *reinterpret_cast<s16x8*>(pair + 8 * lane_id()) = x;
}
__device__ __forceinline__ void st_pair2(float* pair, Frag<float> f0, Frag<float> f1) {
    *reinterpret_cast<f32x4*>(pair + 8 * lane_id()) = f0.v;
    *reinterpret_cast<f32x4*>(pair + 8 * lane_id() + 4) = f1.v;
}

// Past the caches (non-temporal): results that a launch writes once and in whole lines and that are not read before much else is -- the checkpoints of
// states and state gradients, v_new's gradient, o, the inputs' gradients -- and loads of what nobody reads again.  Kept by the caches they put out
// what the next launch reads, the operator's inputs first.  A copy of 256 MiB goes at 5.9 TB/s without and 6.3 with it.  Measured, us a training step,
// without -> with, the same bits: K = V = 64, 16 heads, 4 x 2048 tokens 285 -> 266 (checkpoint and reverse kernels 56 -> 49 and 54 -> 47,
// chunk_grad 100 -> 94), 2 x 2048 154 -> 151, 1 x 2048 122 -> 120; K = V = 128, 1 x 2048 253 -> 225, 4 x 2048 801 -> 788, 16384 packed 1701 -> 1696, 2 x 1537 of 8 heads
// 191 -> 183.  Not so: what prep leaves (packed prefill of 5003 tokens 121 -> 132), local outputs and G of the fused forward kernel (fixup 12 -> 15), the
// checkpoints' loads, which two waves make each (chunk_grad at K = V = 128 520 -> 655), the inputs' last loads (nothing at K = 64, 1696 -> 1714).
template <typename X> __device__ __forceinline__ void st_past(X* p, X x) { __builtin_nontemporal_store(x, p); }
// The other side of a branch beside st_past: the compiler makes one store of the two otherwise, and that an ordinary one.
template <typename X> __device__ __forceinline__ void st_near(X* p, X x) {
    __builtin_amdgcn_sched_barrier(0);
    *p = x;
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void st_pair2_past(bf16* pair, Frag<bf16> f0, Frag<bf16> f1) {
    st_past(reinterpret_cast<s16x8*>(pair + 8 * lane_id()), __builtin_shufflevector(f0.v, f1.v, 0, 1, 2, 3, 4, 5, 6, 7));
}
__device__ __forceinline__ void ld_pair_past(const bf16* pair, Frag<bf16>& f0, Frag<bf16>& f1) {
    const s16x8 x = __builtin_nontemporal_load(reinterpret_cast<const s16x8*>(pair + 8 * lane_id()));
    f0.v = __builtin_shufflevector(x, x, 0, 1, 2, 3);
    f1.v = __builtin_shufflevector(x, x, 4, 5, 6, 7);
}
__device__ __forceinline__ void ld_pair_past(const float* pair, Frag<float>& f0, Frag<float>& f1) { ld_pair(pair, f0, f1); }

// lane (g, c)'s four elements of column c of a tile: of 16 lanes, lane s names the piece with row group s % 4 of row 4 g + s / 4, and lane c
// gets element c % 4 of the pieces c / 4 + 4 i
__device__ __forceinline__ Frag<bf16> ld_turned(const char* p) {
    Frag<bf16> f;
    f.v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
    return f;
}

// where lane l's piece of a tile in fragment order is, in bytes, for the tile turned
__device__ __forceinline__ int turned_tile(int l) { return (16 * (l & 3) + (l >> 4) * 4 + ((l >> 2) & 3)) * 8; }

// workgroup barrier that orders LDS accesses only: global loads issued before it may still be outstanding
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// all but the last n of this wave's memory accesses are complete
template <int N> __device__ __forceinline__ void wait_loads() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
    asm volatile("" ::: "memory");
}

// ---- rows of a tensor into fragments, through LDS -----------------------------------------------------------
// The lanes of a fragment run over the rows first.  Loaded straight from a row-major tensor an instruction touches 64
// separate pieces of 8 bytes, and the vector cache's address unit takes them one by one: the fused kernels' waves spent
// thousands of cycles a chunk waiting for their loads to be ISSUED (the unit held up by the cache for 27 % of the time).
// With four lanes to a row, 16 bytes each, there are half the instructions and whole 64-byte pieces; they change lanes in a
// scratch area of the wave's own in LDS (accesses of one wave complete in order: no barrier, and the area can be used again
// at once).  Measured, 4 x 2048 tokens, 16 heads, K = V = 64: fused forward kernel 82 -> 72 us, checkpoint kernel 68 -> 57,
// reverse kernel 69 -> 54.
typedef int i32x4 __attribute__((ext_vector_type(4)));
constexpr int ROWS_TILE = 576;                            // distance of the two tiles: 512 bytes and 16 banks
constexpr int ROWS_SCRATCH = ROWS_TILE + 512;
// l: the lane.  It holds bytes [16 (l & 3), 16 (l & 3) + 16) of row l >> 2 of 16 rows x 32 channels of 2-byte elements: both channel tiles
__device__ __forceinline__ void rows_to_tiles(char* scratch, int l, i32x4 x, Frag<bf16>& f0, Frag<bf16>& f1) {
    const int r = l >> 2, q = l & 3;
    *reinterpret_cast<i32x4*>(scratch + (q >> 1) * ROWS_TILE + r * 32 + (q & 1) * 16) = x;
    const char* mine = scratch + (l & 15) * 32 + (l >> 4) * 8;
    f0 = ld_frag(reinterpret_cast<const bf16*>(mine));
    f1 = ld_frag(reinterpret_cast<const bf16*>(mine + ROWS_TILE));
}
// the same of 16 rows x 16 channels of fp32: one tile
__device__ __forceinline__ f32x4 rows_to_tile(char* scratch, int l, f32x4 x) {
    *reinterpret_cast<f32x4*>(scratch + l * 16) = x;
    return *reinterpret_cast<const f32x4*>(scratch + (l & 15) * 64 + (l >> 4) * 16);
}

// N neighbouring channel tiles of the rows of a chunk on the way from global memory: load() requests them, tiles() gives the
// fragments.  base: the chunk's first row at the first of the channels (uniform); stride: elements from row to row; len: valid
// rows (those past the end alias the last valid one and come out as zeros).  In general every lane loads what its fragments
// hold; two tiles of 2-byte elements come four lanes to a row, 16 bytes each, and change lanes in `scratch` (rows_to_tiles).
// Measured at K = V = 128 bf16, 16384 tokens of 16 heads, lane loads -> rows: prep 248 -> 236 us, chunk_grad 561 -> 541; with
// 4-byte elements, where a lane's piece is 16 bytes as it is, the detour cost 1 us of prep's 23 (2 x 1003 tokens of 8 heads),
// and at K = 64 a chunk_grad wave has one tile a tensor and the training step of 4 x 2048 tokens took the same 306 us.
template <typename T, int N> struct TileLoad {
    Frag<T> x[N];
    __device__ __forceinline__ void load(const T* base, uint32_t stride, int len, int l) {
        const uint32_t off = min(l & 15, len - 1) * stride + 4 * (l >> 4);
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] = ld_frag(at(base, (off + 16 * j) * (uint32_t)sizeof(T)));
    }
    __device__ __forceinline__ void tiles(char*, int len, int l, Frag<T> (&f)[N]) const {
        const Frag<T> z = zero_frag<T>();
#pragma unroll
        for (int j = 0; j < N; ++j) f[j].v = (l & 15) < len ? x[j].v : z.v;
    }
};
template <> struct TileLoad<bf16, 2> {
    i32x4 x;
    __device__ __forceinline__ void load(const bf16* base, uint32_t stride, int len, int l) {
        x = *reinterpret_cast<const i32x4*>(at(base, (min(l >> 2, len - 1) * stride + 8 * (l & 3)) * 2));
    }
    __device__ __forceinline__ void tiles(char* scratch, int len, int l, Frag<bf16> (&f)[2]) const {
        const i32x4 z = {0, 0, 0, 0};
        rows_to_tiles(scratch, l, (l >> 2) < len ? x : z, f[0], f[1]);
    }
};

// gk may be stored as bf16 or fp32 independently of the other inputs (compile-time switch GKF32);
// same contract as ld_frag_sel: the address is readable on every lane, masked lanes read zero.
template <bool GKF32> __device__ __forceinline__ f32x4 ld_gk4(const void* base, int64_t elem_off, bool ok) {
    f32x4 x;
    if (GKF32) x = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(base) + elem_off);
    else x = to_f32(ld_frag(reinterpret_cast<const bf16*>(base) + elem_off));
    return ok ? x : zero4();
}
template <bool GKF32> __device__ __forceinline__ void st_gk4(void* base, int64_t elem_off, f32x4 x) {
    if (GKF32) *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(base) + elem_off) = x;
    else st_frag(reinterpret_cast<bf16*>(base) + elem_off, to_frag<bf16>(x));
}

// ---- x = 1 / (1 + e): sigmoids of N values, whose exponentials e^-x are in e -------------------------------
// The quotient is one step of Newton's method on the hardware reciprocal: for every fp32 number from 1 to 2^126 that is, bit for
// bit, the IEEE quotient (all 1,056,964,609 of them compared; the reciprocal alone is another number for 113,107,050), in three
// instructions instead of ten.  Beyond (x < -87.3, where it is subnormal or zero), if the wave finds any such value, the division.
// Measured, 8192 x 1024 bf16, division / this / the reciprocal alone: layer_pre forward 27.6 / 22.5 / 21.8 us, backward 30.6 / 28.1 /
// 27.8; a layer training step is 1.8 % slower with the division than with the reciprocal, with this 0.6 %.
template <int N> __device__ __forceinline__ void sigmoid_of_exp(const float (&e)[N], float (&x)[N]) {
    float big = 0.f;
#pragma unroll
    for (int j = 0; j < N; ++j) { x[j] = 1.f + e[j]; big = fmaxf(big, x[j]); }
    if (__any(big > 0x1p126f)) {
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] = 1.f / x[j];
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const float r = __builtin_amdgcn_rcpf(x[j]);
            x[j] = __builtin_fmaf(__builtin_fmaf(-x[j], r, 1.f), r, r);
        }
    }
}

// ---- exp: fast hardware exp2 for the bf16 path, full-accuracy expf for the fp32 path -----------------------
template <typename T> __device__ __forceinline__ float exp_t(float x);
template <> __device__ __forceinline__ float exp_t<bf16>(float x) { return __expf(x); }
template <> __device__ __forceinline__ float exp_t<float>(float x) { return expf(x); }
template <typename T> __device__ __forceinline__ f32x4 exp4(f32x4 x) {
    f32x4 r; r[0] = exp_t<T>(x[0]); r[1] = exp_t<T>(x[1]); r[2] = exp_t<T>(x[2]); r[3] = exp_t<T>(x[3]); return r;
}

// ---- sequence / chunk addressing ---------------------------------------------------------------------------
struct ChunkPos {
    int64_t tok0;  // first token row of the chunk on the flattened axis
    int len;       // valid tokens in the chunk (1..16)
    int n;         // sequence
};

// A value that is the same on every lane of the wave, moved to scalar registers.  What is read from a table arrives in
// vector registers even when the index is uniform; addresses formed from it would then be 64-bit vector arithmetic
// for every access, where a scalar base and a 32-bit lane offset do.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ int64_t uniform(int64_t x) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)x >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Token rows [bos, eos) of packed sequence n, forced into 0 <= bos <= eos <= total: the table comes from the caller
// and is not validated on the device, and no value in it may take an access outside the tensors.
__device__ __forceinline__ void packed_bounds(const int64_t* cu, int n, int64_t total, int64_t& bos, int64_t& eos) {
    bos = min(max(cu[n], (int64_t)0), total);
    eos = min(max(cu[n + 1], bos), total);
}

// (cid: the same on every lane)
__device__ __forceinline__ bool locate_chunk(const SeqTab& st, int cid, ChunkPos& cp) {
    if (st.cu == nullptr) {
        if (cid >= st.N * st.NT) return false;
        cp.n = cid / st.NT;
        const int ic = cid - cp.n * st.NT;
        cp.tok0 = (int64_t)cp.n * st.T + (int64_t)ic * CH;
        cp.len = min(CH, st.T - ic * CH);
        return true;
    }
    if (cid >= uniform(st.chunk_off[st.N])) return false;
    cp.n = uniform(st.chunk_seq[cid]);
    const int ic = cid - uniform(st.chunk_off[cp.n]);
    int64_t bos, eos;
    packed_bounds(st.cu, cp.n, st.T, bos, eos);
    cp.tok0 = uniform(bos) + (int64_t)ic * CH;
    cp.len = (int)min((int64_t)CH, uniform(eos) - cp.tok0);
    return cp.len > 0;
}

// The same without a table, for at most FEW_SEQS packed sequences: a wave reads the bounds of all of them, a sequence a lane, and adds up their chunks.
// One round of loads, where the table is three of them one after the other.
constexpr int FEW_SEQS = 64;
struct FewSeqs {
    int64_t bos, eos;  // of lane n's sequence
    int chunks, end;   // its chunks, and where they end: their sum so far, no more than `nch` (sums of larger ones may not fit)
};
template <int CTRL, int ROWS> __device__ __forceinline__ int add_lanes(int x, int most) {
    return min(x + __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false), most);
}
__device__ __forceinline__ FewSeqs few_seqs(const int64_t* cu, int N, int T, int nch) {
    FewSeqs f;
    const int n = lane_id();
    packed_bounds(cu, min(n, N - 1), T, f.bos, f.eos);
    f.chunks = n < N ? (int)((f.eos - f.bos + CH - 1) / CH) : 0;
    f.end = min(f.chunks, nch);
    f.end = add_lanes<0x111, 0xf>(f.end, nch);    // row_shr:1
    f.end = add_lanes<0x112, 0xf>(f.end, nch);
    f.end = add_lanes<0x114, 0xf>(f.end, nch);
    f.end = add_lanes<0x118, 0xf>(f.end, nch);
    f.end = add_lanes<0x142, 0xa>(f.end, nch);    // row_bcast:15, into the second and the fourth row of lanes
    f.end = add_lanes<0x143, 0xc>(f.end, nch);    // row_bcast:31, into the third and the fourth
    return f;
}
__device__ __forceinline__ int of_lane(int x, int n) { return __builtin_amdgcn_readlane(x, n); }
__device__ __forceinline__ int64_t of_lane(int64_t x, int n) {
    return (int64_t)(((uint64_t)(uint32_t)of_lane((int)((uint64_t)x >> 32), n) << 32) | (uint32_t)of_lane((int)(uint32_t)x, n));
}
// (cid: the same on every lane; all lanes)
__device__ __forceinline__ bool locate_few(const SeqTab& st, int cid, ChunkPos& cp) {
    const FewSeqs f = few_seqs(st.cu, st.N, st.T, st.nch);
    if (cid >= of_lane(f.end, 63)) return false;
    cp.n = __builtin_popcountll(__ballot(f.end <= cid));
    const int c0 = cp.n ? of_lane(f.end, cp.n - 1) : 0;
    cp.tok0 = of_lane(f.bos, cp.n) + (int64_t)(cid - c0) * CH;
    cp.len = (int)min((int64_t)CH, of_lane(f.eos, cp.n) - cp.tok0);
    return cp.len > 0;
}

// the z-th sequence in the order in which workgroups start: packed ones from the longest down (all that `order` is read with, but for scan_share)
__device__ __forceinline__ int scan_sequence(const SeqTab& st, int z) { return st.cu ? st.order[z] & ORDER_SEQ : z; }
// chunk range [c0, c1) of sequence n (n: the same on every lane)
__device__ __forceinline__ void seq_chunks(const SeqTab& st, int n, int& c0, int& c1) {
    if (st.cu == nullptr) { c0 = n * st.NT; c1 = c0 + st.NT; }
    else { c0 = uniform(st.chunk_off[n]); c1 = uniform(st.chunk_off[n + 1]); }
}

// token rows [bos, eos) of sequence n on the flattened axis (n: the same on every lane)
__device__ __forceinline__ void seq_bounds(const SeqTab& st, int n, int64_t& bos, int64_t& eos) {
    if (st.cu == nullptr) { bos = (int64_t)n * st.T; eos = bos + st.T; }
    else {
        packed_bounds(st.cu, n, st.T, bos, eos);
        bos = uniform(bos);
        eos = uniform(eos);
    }
}

// chunk range [s0, s1) of time segment `seg` of the chunks [c0, c1) of a sequence
__device__ __forceinline__ void seg_range(int c0, int c1, int nseg, int seg, int& s0, int& s1) {
    const int len = (c1 - c0 + nseg - 1) / nseg;
    s0 = min(c0 + seg * len, c1);
    s1 = min(s0 + len, c1);
}

// ---- per-chunk decay quantities in fragment layout ---------------------------------------------------------
// lane (g,c) holds token c of the chunk and channels 16*kt + 4g + i.  The 16 lanes of a group are one DPP "row",
// so prefix sums, suffix sums and sums over the tokens of a chunk are row_shr / row_shl / mirror additions on
// the vector ALU (out-of-row lanes read 0), with no LDS round trips.
template <int CTRL> __device__ __forceinline__ float dpp0(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ f32x4 dpp0(f32x4 x) {
    f32x4 r; r[0] = dpp0<CTRL>(x[0]); r[1] = dpp0<CTRL>(x[1]); r[2] = dpp0<CTRL>(x[2]); r[3] = dpp0<CTRL>(x[3]); return r;
}
__device__ __forceinline__ f32x4 scan16_incl(f32x4 x) {     // inclusive prefix sum over the 16 lanes of a group
    x += dpp0<0x111>(x);    // row_shr:1
    x += dpp0<0x112>(x);    // row_shr:2
    x += dpp0<0x114>(x);    // row_shr:4
    x += dpp0<0x118>(x);    // row_shr:8
    return x;
}
__device__ __forceinline__ f32x4 rscan16_incl(f32x4 x) {    // inclusive suffix sum over the 16 lanes of a group
    x += dpp0<0x101>(x);    // row_shl:1
    x += dpp0<0x102>(x);
    x += dpp0<0x104>(x);
    x += dpp0<0x108>(x);
    return x;
}
__device__ __forceinline__ f32x4 sum16(f32x4 x) {           // sum over the 16 lanes of a group, on all of them
    x += dpp0<0xB1>(x);     // quad_perm:[1,0,3,2]
    x += dpp0<0x4E>(x);     // quad_perm:[2,3,0,1]
    x += dpp0<0x141>(x);    // row_half_mirror
    x += dpp0<0x140>(x);    // row_mirror
    return x;
}
__device__ __forceinline__ f32x4 bcast16(f32x4 x, int src) {  // value of lane `src` of the own 16-lane group
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __shfl(x[i], src, 16);
    return r;
}
// the same with a compile-time source lane: one DPP move per register (row_newbcast), no LDS round trip
template <int SRC> __device__ __forceinline__ f32x4 bcast16(f32x4 x) {
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        r[i] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x[i]), 0x150 + SRC, 0xf, 0xf, true));
    return r;
}
// value held by the lane 32 positions away (v_permlane32_swap exchanges the two halves of the wave)
__device__ __forceinline__ float xor32(float x) {
    const int xi = __float_as_int(x);
    auto r = __builtin_amdgcn_permlane32_swap(xi, xi, false, false);
    return __int_as_float(lane_id() < 32 ? r[1] : r[0]);
}

// value held by the lane 16 positions away within each half of the wave (v_permlane16_swap exchanges odd and even
// rows of 16 lanes between two registers)
__device__ __forceinline__ float xor16(float x) {
    const int xi = __float_as_int(x);
    auto r = __builtin_amdgcn_permlane16_swap(xi, xi, false, false);     // r[0] rows: x0 x0 x2 x2, r[1]: x1 x1 x3 x3
    return __int_as_float((lane_id() & 16) ? r[0] : r[1]);
}
// Sums over the `width` lanes (1 to 64, a power of two, the same on all) of a lane's neighbourhood, on all of them: a butterfly on the vector ALU, within 16
// lanes by DPP (the mirrors meet sums that are the same on four, or eight, neighbours), beyond by swaps of rows of lanes.  Additions and
// order are those of a butterfly of __shfl_xor, and so are the bits; that one goes through LDS, at some 60 cycles a stage.
template <int N> __device__ __forceinline__ void sum_lanes(float (&x)[N], int width) {
    auto stage = [&](auto other) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] += other(x[i]);
    };
    if (width > 1) stage([](float v) __attribute__((always_inline)) { return dpp0<0xB1>(v); });     // quad_perm:[1,0,3,2]
    if (width > 2) stage([](float v) __attribute__((always_inline)) { return dpp0<0x4E>(v); });     // quad_perm:[2,3,0,1]
    if (width > 4) stage([](float v) __attribute__((always_inline)) { return dpp0<0x141>(v); });    // row_half_mirror
    if (width > 8) stage([](float v) __attribute__((always_inline)) { return dpp0<0x140>(v); });    // row_mirror
    if (width > 16) stage([](float v) __attribute__((always_inline)) { return xor16(v); });
    if (width > 32) stage([](float v) __attribute__((always_inline)) { return xor32(v); });
}
__device__ __forceinline__ float sum_lanes(float x, int width) {
    float v[1] = {x};
    sum_lanes<1>(v, width);
    return v[0];
}

// Sums over the lanes that lie CG (16 or 32) apart, on all of them
template <int CG> __device__ __forceinline__ void sum_rows(f32x4& x) {
    static_assert(CG == 16 || CG == 32, "rows or halves of a wavefront");
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (CG == 16) x[i] += xor16(x[i]);
        x[i] += xor32(x[i]);
    }
}

// sum over the four lanes c, c+16, c+32, c+48, on all of them
__device__ __forceinline__ float sum_groups(float x) {
    x += xor16(x);
    x += xor32(x);
    return x;
}


// ---- decay factors of the factorised score products --------------------------------------------------------------
// A score sums q_i[ch] k_j[ch] exp(gi_i[ch] - gi_j[ch]) over channels (j <= i; likewise with a, ge on the row side and b
// on the inner side).  To be a matrix product the decay must factorise: exp(gi_i - m) exp(m - gi_j) with a centre m per
// channel.  One centre (gi of token MID) serves the whole 16 x 16 tile as long as no exponent gi_i - m, ge_i - m exceeds
// SAFE_RANGE in magnitude: the factors then stay within e^+-70, inside the range of the element types with room for
// the operands themselves.  Beyond that (a channel that loses more than e^-70 over eight tokens) exp(gi_i - m) would
// overflow for pairs on one side of the centre, so the tile is assembled from three products whose exponents are all
// <= 0 or bounded:
//   pass 0: rows 8..15 x inner 0..7, centre token 7: gi_i - m <= 0 and m - gi_j <= 0, exact;
//   pass 1: rows 0..7 x inner 0..7, centre token 3;      pass 2: rows 8..15 x inner 8..15, centre token 11:
//           inside a half the per-token log-decay is clamped at -PASS_CLAMP first, so no exponent exceeds 4 tokens x
//           PASS_CLAMP = 80.  A pair (i, j) whose span holds a clamped token has weight < e^-20 = 2e-9 either way, and
//           every other pair is exact, so each weight is within 2e-9 (absolute) of its true value.
// Tokens outside a pass's rows / inner range get the factor 0, and what the passes leave above the diagonal is removed
// by the causal masks as before.
constexpr float SAFE_RANGE = 70.f;
constexpr float PASS_CLAMP = 20.f;

// ---- the same factors in base 2 (2-byte element types) --------------------------------------------------------------
// A channel tile needs e^{gi-m}, e^{m-gi}, e^{ge-m} for its scores and e^{gi}, e^{ge}, e^{gl-gi}, e^{gl} for the gated copies.
// An exponential is 16 cycles of a SIMD (a quarter-rate instruction) and a multiplication before it; but ge of a token is
// gi of the token before it, and the second group is the first times e^{m} and e^{gl-m}: three exponentials and lane moves
// in place of seven.  Products of two factors of the safe range stay inside that of fp32; a tile beyond it (its scores
// take the strong-decay route) forms the second group directly.  A product carries one rounding of 2^-24 more than an exponential,
// which beside operands of 8 bits is not seen.  All kernels take their factors so: fused producers, prep, chunk_grad.  Errors against a float64
// evaluation, relative to a build with every factor an exponential of its own, mean of 10 training steps of 2 x 256 tokens, outputs, final state and all
// gradients: K = V = 64, 8 heads (fused) 0.9997 to 1.0001, K = V = 128, 4 heads (classic) 0.9995 to 1.0000, with sixteen times the decay 0.9999 to 1.0001;
// standard errors up to 0.0004.  The products save 1.3 us of a training step of 4 x 2048 tokens and 0.3 us of a forward pass.
// Measured on 8192 tokens x 16 heads, K = V = 64 (with the producers' reordering in the fused kernels that came with it):
// forward 75.2 -> 73.8 us, checkpoints 78.6 -> 76.1, reverse 70.7 -> 69.0.
constexpr float LOG2E = 1.44269504088896340736f;
constexpr float SAFE_FACTOR = 2.5154386709191670e30f;    // e^SAFE_RANGE
__device__ __forceinline__ f32x4 exp2_4(f32x4 x) {
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_exp2f(x[i]);
    return r;
}
// value of the token before (lane c - 1 of the 16-lane group); `first` on the group's first lane
__device__ __forceinline__ f32x4 prev_token(f32x4 x, f32x4 first) {
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        r[i] = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(first[i]), __float_as_int(x[i]), 0x111, 0xf, 0xf, false));   // row_shr:1
    return r;
}
template <typename T> struct TileDecay;
template <> struct TileDecay<bf16> {
    f32x4 eq, ek, ea;                                     // e^{gi-m}, e^{m-gi}, e^{ge-m}
    f32x4 egi, ege, edn, egl;                             // e^{gi}, e^{ge}, e^{gl-gi}, e^{gl}
    bool strong;                                          // a factor beyond the safe range (the same on every lane)
    // g4: log-decay of the lane's token and channels; c: the token; check: whether the tile may be a strong one
    __device__ __forceinline__ TileDecay(f32x4 g4, int c, bool check = true) {
        const f32x4 gi = scan16_incl(g4 * LOG2E), m = bcast16<MID>(gi);
        eq = exp2_4(gi - m);
        ek = exp2_4(m - gi);
        const uint32_t flip = c == 0 ? 0x80000000u : 0u;
        f32x4 mm_;
#pragma unroll
        for (int i = 0; i < 4; ++i) mm_[i] = __uint_as_float(__float_as_uint(m[i]) ^ flip);
        const f32x4 em = exp2_4(mm_);                     // e^{-m} on the first token, e^{m} on the others
        float big = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) big = fmaxf(fmaxf(big, em[i]), fmaxf(eq[i], ek[i]));
        strong = check && __any(!(big <= SAFE_FACTOR)) != 0;
        ea = prev_token(eq, em);
        egi = eq * bcast16<1>(em);
        edn = ek * bcast16<CH - 1>(eq);
        if (check) {                                      // formed here, where the lane moves are part of the products, and not behind the branch
            pin(egi);
            pin(edn);
        }
        if (strong) {
            egi = exp2_4(gi);
            edn = exp2_4(bcast16<CH - 1>(gi) - gi);
        }
        const f32x4 one = {1.f, 1.f, 1.f, 1.f};
        ege = prev_token(egi, one);
        egl = bcast16<CH - 1>(egi);
    }
};
// 4-byte element types: every factor an exponential of its own.  With a token's exclusive ones taken from the token before it, the outputs of
// 2000 tokens of 8 heads were 0.1 % further from a float64 evaluation (standard error 0.01 %); with products more so.
template <> struct TileDecay<float> {
    f32x4 eq, ek, ea, egi, ege, edn, egl;
    bool strong;
    __device__ __forceinline__ TileDecay(f32x4 g4, int, bool check = true) {
        const f32x4 gi = scan16_incl(g4), ge = gi - g4, m = bcast16<MID>(gi), gl = bcast16<CH - 1>(gi);
        eq = exp4<float>(gi - m);
        ek = exp4<float>(m - gi);
        ea = exp4<float>(ge - m);
        egi = exp4<float>(gi);
        ege = exp4<float>(ge);
        edn = exp4<float>(gl - gi);
        egl = bcast16<CH - 1>(egi);
        float big = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) big = fmaxf(big, fmaxf(fabsf(gi[i] - m[i]), fabsf(ge[i] - m[i])));
        strong = check && __any(!(big <= SAFE_RANGE)) != 0;
    }
};

struct DecayPass {
    static constexpr int COUNT = 3;
    int centre;          // token whose cumulative decay centres the pass
    bool rows, cols;     // does this lane's token take part on the row side (q, a) / on the inner side (k, b)
    bool clamp;
    __device__ __forceinline__ DecayPass(int ps, int c) {
        centre = ps == 0 ? MID : ps == 1 ? MID / 2 : MID + (CH - MID) / 2;
        rows = ps == 1 ? c <= MID : c > MID;
        cols = ps == 2 ? c > MID : c <= MID;
        clamp = ps != 0;
    }
    // gi, ge: inclusive / exclusive cumulative log-decay of the lane's token (four channels)
    template <typename T> __device__ __forceinline__ void factors(f32x4 gi, f32x4 ge, f32x4& eq, f32x4& ek, f32x4& ea) const {
        if (clamp) {                                      // uniform over the wave
            f32x4 g = gi - ge;
#pragma unroll
            for (int i = 0; i < 4; ++i) g[i] = fmaxf(g[i], -PASS_CLAMP);
            gi = scan16_incl(g);
            ge = gi - g;
        }
        const f32x4 m = bcast16(gi, centre);
        const f32x4 z = zero4();
        f32x4 dq = gi - m, dk = m - gi, da = ge - m;
#pragma unroll
        for (int i = 0; i < 4; ++i) { dq[i] = fminf(dq[i], 80.f); dk[i] = fminf(dk[i], 80.f); da[i] = fminf(da[i], 80.f); }
        eq = rows ? exp4<T>(dq) : z;
        ek = cols ? exp4<T>(dk) : z;
        ea = rows ? exp4<T>(da) : z;
    }
};

}  // namespace hdla
