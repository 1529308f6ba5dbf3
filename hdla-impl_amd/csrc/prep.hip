// prep kernel: everything of a 16-token chunk that does not depend on the recurrent state.
//
// Replaces, for one (chunk, head) per workgroup, the reference's chunk-local cumsum (fla chunk_rwkv6_fwd_cumsum,
// called at HRDPLR/hrdplr.py:44), the two score kernels (HRDPLR/fwd_triton.py:22-290 and :305-514), the
// triangular inverse (HRDPLR/fwd_triton.py:601-667) and the WY kernel (HRDPLR/fwd_triton.py:685-790).
// The four score matrices never reach HBM: they are MFMA accumulators, (I - A_ab)^-1 is solved in LDS, and
// w, u and the gated copies are written once, in the fragment order the state scans read them in.
//
// A wave handles 64 channels: K = 64 is one wave per (chunk, head); K = 128 is a workgroup of two, each with its
// half of the channel tiles and of the value tiles.  The score tiles are sums over channels: the two exchange
// their parts through LDS and each then solves the (small) triangular system for itself.  One wave with all 128
// channels needs the whole register file, and at one wave per SIMD nothing hides its memory round trips.
#include "hdla_common.cuh"
#include "hdla_launch.h"

namespace hdla {

// ---- chunk table for packed variable-length batches ----------------------------------------------------------
constexpr int ORDER_MAX_N = 2048;      // beyond this many sequences they are taken as they come (ranking is quadratic)
constexpr int TABLE_THREADS = 256;
// More than FEW_SEQS sequences (fewer: few_table): workgroup 0 builds the table; with at most ORDER_MAX_N sequences, workgroups 1 .. ceil(N / 256) rank the sequences by
// their chunk counts, one sequence a thread (they form the counts from cu themselves, so they wait for nobody).
// The workgroups behind them clear the rows of the outputs that belong to no sequence.  Each looks the table over for itself
// and, where it is a partition of the T tokens, is done: all of them together are in the shadow of workgroup 0 (clearing the
// outputs for every call took 88 of 2050 us of a training step on 16384 tokens, H = 16, K = V = 128).  A table that does not
// decrease leaves out only what lies before its first and behind its last entry (a batch padded at its end); one that does may
// leave out anything, and the outputs are cleared whole.
// Measured, 16384 tokens of 16 heads, K = V = 128, the last 200 in no sequence, forward and backward pass: 1.62 ms (a full batch 1.64);
// with all outputs cleared by workgroup 0, two bytes a lane, 21.6.
struct ClearRange { long long lo, hi; };                  // tokens [0, lo) and [hi, T)
__device__ __forceinline__ ClearRange uncovered(const int64_t* cu, int N, int T, int t, int threads) {
    int decreases = 0;
    for (int n = t; n < N; n += threads) decreases |= cu[n + 1] < cu[n];
    ClearRange r;
    r.lo = min(max(cu[0], (int64_t)0), (int64_t)T);
    r.hi = min(max(cu[N], (int64_t)r.lo), (int64_t)T);
    if (__syncthreads_or(decreases)) r.lo = r.hi = T;
    return r;
}
// n bytes at p (both multiples of 2) become zero, 16 bytes a store between the first and the last multiple of 16; i of `count` threads
__device__ __forceinline__ void clear_bytes(char* p, long long n, long long i, long long count) {
    const long long head = min((long long)(-reinterpret_cast<uintptr_t>(p) & 15), n), body = (n - head) & ~15LL;
    for (long long e = 16 * i; e < body; e += 16 * count) *reinterpret_cast<i32x4*>(p + head + e) = i32x4{0, 0, 0, 0};
    if (i < 8) {
        if (2 * i < head) *reinterpret_cast<uint16_t*>(p + 2 * i) = 0;
        if (head + body + 2 * i < n) *reinterpret_cast<uint16_t*>(p + head + body + 2 * i) = 0;
    }
}
// (all threads of `groups` workgroups, of which this is the one numbered `group`)
__device__ __forceinline__ void clear_uncovered(const int64_t* cu, int N, int T, const PackedOut& out, int group, int groups, int t, int threads) {
    const ClearRange r = uncovered(cu, N, T, t, threads);
    const long long count = (long long)groups * threads, i = (long long)group * threads + t;
    for (int b = 0; b < out.n; ++b) {
        char* const p = static_cast<char*>(out.p[b]);
        clear_bytes(p, r.lo * out.row[b], i, count);
        clear_bytes(p + r.hi * out.row[b], (T - r.hi) * out.row[b], i, count);
    }
}
__global__ __launch_bounds__(TABLE_THREADS) void clear_uncovered_kernel(const int64_t* cu, int N, int T, PackedOut out) {
    clear_uncovered(cu, N, T, out, blockIdx.x, gridDim.x, threadIdx.x, TABLE_THREADS);
}
// How wide the workgroups of each sequence are in the scans of the backward and the forward pass.  A workgroup of fewer column blocks takes a shorter
// step, but more workgroups read a chunk's block.  Unequal lengths want unequal widths: a launch ends with its longest sequence, which walks its last
// steps on a device that the others have left.  Candidates: every length in every width as the time that no sequence may exceed where a
// narrower workgroup helps it; of these the one whose longest walk, or whose work spread over the slots, is least.  (Column blocks never meet: the
// results have the same bits in every width.)  Times of a step of 4, 2 and
// 1 blocks, 10 ns, one sequence of 16 heads alone on the device, K = V = 128: forward 81, 60, 58, both scans 105, 87, 78 (K = 64: 42, 35, 34; 59,
// 51, 45); the choice needs their ratios only, and with K = 128's it is at K = 64 as good as with its own (1203 random batches: 0.4 and 0.3 % over the best
// of its candidates on average, 14 and 13 % at the most).
constexpr float SHARE_STEP[2][3] = {{81.f, 60.f, 58.f}, {105.f, 87.f, 78.f}}, SHARE_PROLOGUE = 6.f;
// More workgroups than slots leave gaps behind them.  Over 1500 random batches of 2 to 14 sequences, the choice against the best of its candidates with the
// workgroups dealt out one by one: 0.3 % on average, 12 % at the most (without the factor 0.8 and 41 %; one width for all 17 and 40 %).
constexpr float SHARE_PACKING = 1.15f;
struct ShareLds {
    float steps[SHARE_MAX_N];                             // of the sequences from the longest down, and which they are
    int seq[SHARE_MAX_N];
    unsigned long long best[2];
};
__device__ __forceinline__ int share_code(int pass, float steps, float limit) {
    return steps * SHARE_STEP[pass][0] <= limit ? 0 : steps * SHARE_STEP[pass][1] <= limit ? 1 : 2;
}
// (all threads; returns the bits that go beside order[t])
__device__ __forceinline__ int share_device(ShareLds& sh, int N, int H, int V, int t, int threads) {
    if (t < 2) sh.best[t] = ~0ull;
    __syncthreads();
    auto limit = [&](int pass, int i) { return sh.steps[i / 3] * SHARE_STEP[pass][i % 3]; };
    for (int i = t; i < 6 * N; i += threads) {
        const int pass = i >= 3 * N, cand = pass ? i - 3 * N : i;
        const float x = limit(pass, cand);
        float chain = 0.f, work = 0.f;
        int groups = 0;
        for (int j = 0; j < N; ++j) {
            const int code = share_code(pass, sh.steps[j], x), g = (V / 64) << code;
            const float time = sh.steps[j] * SHARE_STEP[pass][code];
            chain = max(chain, time);
            work += time * (float)g;
            groups += g;
        }
        if (groups <= share_most(H, 1 + pass, N, V)) {
            const int slots = share_slots(H, 1 + pass);
            const float cost = groups <= slots ? chain : max(chain, SHARE_PACKING * work / (float)slots);
            atomicMin(&sh.best[pass], (unsigned long long)__float_as_uint(cost) << 32 | (unsigned)cand);
        }
    }
    __syncthreads();
    int codes = 0;
    if (t < N) {
        codes = share_code(0, sh.steps[t], limit(0, (int)(unsigned)sh.best[0])) << ORDER_OUT;
        codes |= (int)((unsigned)share_code(1, sh.steps[t], limit(1, (int)(unsigned)sh.best[1])) << ORDER_GRAD);
    }
    return codes;
}
// A table of at most FEW_SEQS sequences, in registers: work 0 writes chunk_off and chunk_seq, work 1 ranks the sequences (V: as in
// launch_chunk_table).  All threads of a workgroup, at least a wave, each wave for itself but for the widths.
__device__ __forceinline__ void few_table(int work, const int64_t* cu, int N, int T, int nch, int H, int V, int32_t* chunk_off, int32_t* chunk_seq,
                                          ShareLds& sh, int t, int threads) {
    const FewSeqs f = few_seqs(cu, N, T, nch);
    if (work == 0) {
        if (t < N) chunk_off[t + 1] = f.end;
        if (t == 0) chunk_off[0] = 0;
        for (int n = 0, c0 = 0; n < N; ++n) {
            const int c1 = of_lane(f.end, n);
            for (int cid = c0 + t; cid < c1; cid += threads) chunk_seq[cid] = n;
            c0 = c1;
        }
        return;
    }
    int32_t* const order = chunk_off + N + 1;
    const int n = lane_id();
    int r = 0;
    for (int m = 0; m < N; ++m) {
        const int other = of_lane(f.chunks, m);
        r += other > f.chunks || (other == f.chunks && m < n) ? 1 : 0;
    }
    if (V == 0 || N == 1 || N > SHARE_MAX_N) {
        if (t < N) order[r] = n;
        return;
    }
    if (t < N) {
        sh.steps[r] = (float)f.chunks + SHARE_PROLOGUE;
        sh.seq[r] = n;
    }
    const int codes = share_device(sh, N, H, V, t, threads);
    if (t < N) order[t] = sh.seq[t] | codes;
}
__global__ __launch_bounds__(TABLE_THREADS) void build_chunk_table_kernel(const int64_t* cu, int N, int T, int nch, int H, int V,
                                                                          int32_t* chunk_off, int32_t* chunk_seq, int rankers, PackedOut out) {
    constexpr int LONG_SEQ = 64, LONG_LIST = 512;
    __shared__ long long strip[2][TABLE_THREADS];
    __shared__ __attribute__((aligned(16))) int32_t len[ORDER_MAX_N];
    __shared__ int n_long, long_seq[LONG_LIST], long_c0[LONG_LIST], long_c1[LONG_LIST];
    const int t = threadIdx.x;
    auto chunks_of = [&](int n) {
        int64_t bos, eos;
        packed_bounds(cu, n, T, bos, eos);
        return (long long)((eos - bos + CH - 1) / CH);
    };
    int32_t* order = chunk_off + N + 1;
    if ((int)blockIdx.x > rankers) {
        clear_uncovered(cu, N, T, out, (int)blockIdx.x - 1 - rankers, (int)gridDim.x - 1 - rankers, t, TABLE_THREADS);
        return;
    }
    __shared__ ShareLds sh;
    if (N <= FEW_SEQS) {
        few_table(blockIdx.x, cu, N, T, nch, H, V, chunk_off, chunk_seq, sh, t, TABLE_THREADS);
        return;
    }
    if (blockIdx.x > 0) {
        // order[r] = the sequence with the r-th most chunks (ties by index): the scans start their workgroups in this
        // order, so that when there are more workgroups than compute units the long sequences are not the ones that
        // wait.  All counts go to LDS (entries past N hold -1 and rank behind everything); a thread reads them four at
        // a time against its own.
        for (int n = t; n < ORDER_MAX_N; n += TABLE_THREADS) len[n] = n < N ? (int)min(chunks_of(n), (long long)0x7fffffff) : -1;
        __syncthreads();
        const int n = ((int)blockIdx.x - 1) * TABLE_THREADS + t;
        if (n >= N) return;
        const int mine = len[n];
        int r = 0;
        for (int m = 0; m < N; m += 4) {
            const i32x4 lm = *reinterpret_cast<const i32x4*>(&len[m]);
#pragma unroll
            for (int j = 0; j < 4; ++j) r += (lm[j] > mine || (lm[j] == mine && m + j < n)) ? 1 : 0;
        }
        order[r] = n;
        return;
    }
    // chunk_off = exclusive prefix sum of the sequences' chunk counts: every thread sums a strip of consecutive
    // sequences, the strip sums are scanned in LDS, and the strips are walked a second time.
    const int per = (N + TABLE_THREADS - 1) / TABLE_THREADS;
    const int n0 = min(t * per, N), n1 = min(n0 + per, N);
    long long own = 0;
#pragma unroll 8
    for (int n = n0; n < n1; ++n) own += chunks_of(n);
    strip[0][t] = own;
    if (t == 0) n_long = 0;
    __syncthreads();
    int cur = 0;
    for (int d = 1; d < TABLE_THREADS; d <<= 1) {         // inclusive scan, one doubling step per round
        strip[cur ^ 1][t] = strip[cur][t] + (t >= d ? strip[cur][t - d] : 0);
        cur ^= 1;
        __syncthreads();
    }
    // chunk_off, and chunk_seq: a thread writes the entries of its own strip's sequences; sequences of more than
    // LONG_SEQ chunks are put on a list and written by the whole workgroup afterwards (a thread that finds the list
    // full writes its own).  Offsets never go beyond the slots the workspace has (cannot happen for a non-decreasing
    // table that ends at T).
    long long acc = strip[cur][t] - own;
    for (int n = n0; n < n1; ++n) {
        const long long nx = acc + chunks_of(n);
        const int c0 = (int)min(acc, (long long)nch), c1 = (int)min(nx, (long long)nch);
        acc = nx;
        chunk_off[n] = c0;
        int slot = LONG_LIST;
        if (c1 - c0 > LONG_SEQ) slot = atomicAdd(&n_long, 1);
        if (slot < LONG_LIST) { long_seq[slot] = n; long_c0[slot] = c0; long_c1[slot] = c1; }
        else for (int cid = c0; cid < c1; ++cid) chunk_seq[cid] = n;
    }
    if (t == 0) chunk_off[N] = (int)min(strip[cur][TABLE_THREADS - 1], (long long)nch);
    __syncthreads();
    const int nl = min(n_long, LONG_LIST);
    for (int i = 0; i < nl; ++i)
        for (int cid = long_c0[i] + t; cid < long_c1[i]; cid += TABLE_THREADS) chunk_seq[cid] = long_seq[i];
    if (N > ORDER_MAX_N)                                  // too many to rank: as they come
        for (int n = t; n < N; n += TABLE_THREADS) order[n] = n;
}

// The table as the work of prep_kernel's last workgroups, where a wave has a lane for each sequence: a launch of 4 to 8 us less that everything waited
// for, and prep_kernel's other workgroups find their chunks by themselves (locate_few).  us, forward passes, table first -> this: 90 tokens in 4 sequences,
// 4 heads 15.8 -> 13.0; 520 in 8, 8 heads, K = V = 128 27.5 -> 23.2; 3000 in 12, 16 heads, K = 64, V = 128 54.3 -> 47.4, in 30, K = V = 128 98.6 -> 91.8;
// 5003 in 4 130.7 -> 127.0; fp32, 700 in 4 61.6 -> 57.1; training step of 16384 in 4 1649 -> 1634.  The fused route, whose first kernel walks
// sequences, has the table first, in registers too: 2500 tokens in 5, 16 heads 52.0 -> 50.1.  FEW_CLEARERS: as many threads at K = 128 as the other launch's workgroups,
// four times as large, have.  A training step with 14384 of 16384 rows to clear, 16 heads, K = V = 128, by 256 / 512 / 1024 of them 394 / 386 / 384 us (by a launch of its own in
// front 387), K = 64, V = 128 233 / 240 / 234 (247); batches without such rows the same.
struct FewTable {
    int32_t *chunk_off, *chunk_seq;       // null: the table is there
    int V;
    PackedOut out;
};
static_assert(FEW_SEQS == 64 && SHARE_MAX_N <= FEW_SEQS, "a lane each (prep_makes_table)");
constexpr int FEW_CLEARERS = 1024;

constexpr int LDP = 36;   // padded row length of the 32x32 LDS matrices (keeps 16-byte row alignment)

// MODE: what the kernel leaves in the workspace -- PREP_FWD: what the forward pass's scan reads (which also forms the
// output); PREP_BWD: what the two scans of the backward pass and the chunk_grad kernels read; PREP_KEEP: both, for a
// forward pass whose workspace the backward pass will use instead of running this kernel again; PREP_STATES: the same beside the states that
// enter the chunks, where what only the forward pass reads is in a place of its own.
enum PrepMode { PREP_FWD = 0, PREP_BWD = 1, PREP_KEEP = 2, PREP_STATES = 3 };
// Waves a SIMD: what the registers of a wave allow.  Three of 2-byte elements (with fp32 decays beside plain a, b: two): a tile's factors, operands
// and gated copies are done with before the next one's begin, the copies that need nothing else leave at once, and (I - A_ab)^-1 lies where the
// parts of the score tiles were (20 KB of LDS a workgroup of two waves instead of 37).  Three exponentials a tile instead of seven (TileDecay).
// Measured, us, before (all copies formed behind (I - A_ab)^-1 from inputs and decays kept for that, 216 registers) -> after: K = V = 128, 16384
// tokens of 16 heads, forward / backward mode 190 / 237 -> 176 / 222, which is 5.7 TB/s of their traffic; with the HDLA parameterisation 5003 tokens
// of 16 heads 62 -> 52, 3074 tokens of 8 heads, both modes in one, 26 -> 23.  4-byte elements, 1008 chunks and heads (a wave a SIMD): the same.
template <typename T, bool GKF32, bool HD> constexpr int prep_waves() { return sizeof(T) == 2 && (HD || !GKF32) ? 3 : 2; }
template <typename T, bool GKF32, int K, int V, int MODE, bool HD>
__global__ __launch_bounds__(K) __attribute__((amdgpu_waves_per_eu(prep_waves<T, GKF32, HD>(), prep_waves<T, GKF32, HD>()))) void prep_kernel(ChunkArgs<T> p, FewTable few) {
    constexpr bool BWD = MODE == PREP_BWD;                // neither the output's score tiles nor qg are needed
    constexpr bool WB = MODE != PREP_FWD;                 // the backward pass's extras are
    // the forward pass's scan of 2-byte elements forms u itself and takes the ranks of b^T side by side (scan_out.cuh): v is not read
    constexpr bool SCAN_U = MODE == PREP_FWD && sizeof(T) == 2;
    // The other scans of 2-byte elements form u too, from (I - A_ab)^-1, A_ak and v; u is written where chunk_grad reads it (its REBUILD_U), or where the
    // caller has named the classic route, whose buffers can be looked at (UT is given).  This mode at K = V = 128, 16384 tokens of 16 heads, us: 221 -> 178,
    // for 12 KB not written and v not read of 85 a chunk and head.
    constexpr bool WRITE_U = sizeof(T) == 4 || GKF32;
    constexpr bool KG_IS_B = HD && sizeof(T) == 2;    // kg^T is bg_2^T, which the scans of 2-byte elements know (OutCfg)
    constexpr int NWP = K / 64;                       // waves per (chunk, head)
    constexpr int KTW = 4, VT = V / 16, VTW = VT / NWP, KT2 = K / 32;
    constexpr bool APART = MODE == PREP_STATES;
    constexpr int SAS = blk_fwd(K, sizeof(T), !BWD && !APART).SIZE / (int)sizeof(T);   // elements between (chunk, head) slots
    constexpr int SQS = APART ? blk_q(K, sizeof(T)) / (int)sizeof(T) : SAS;            // and between those of q's tiles and A_qb
    constexpr int SBS = blk_bwd(K, sizeof(T)).SIZE / (int)sizeof(T);
    constexpr int NPART = BWD ? 8 : 9;                                    // score tiles that are summed over the waves
    // Per wave: A_ab, rank-major, and (I - A_ab)^-1.  A wave's matrices lie where the other wave's parts of the score tiles were, which it
    // has then read and nobody else does.
    constexpr int MAT = 32 * LDP;
    static_assert(NPART * 256 <= 2 * MAT, "");
    __shared__ __attribute__((aligned(16))) float sMat[NWP][2 * MAT];
    // rows on their way to fragments; 4-byte elements: tiles that are turned
    __shared__ __attribute__((aligned(16))) char sRows[NWP][sizeof(T) == 4 ? TURN_SCRATCH : ROWS_SCRATCH];
    __shared__ float sSum[NWP * CH];
    __shared__ int sStrong[NWP];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* const sN = sMat[w];
    float* const sT = sN + MAT;
    char* const scratch = sRows[w];
    const int kt0 = w * KTW, vt0 = w * VTW;                              // first own channel tile / value tile

    // Which of the two indices runs fastest over the workgroups decides which rows of the [token][head][channel]
    // tensors the workgroups resident at one time touch.  Measured: with rows of 4 KiB and more, neighbouring
    // workgroups should be the heads of one chunk (together they read whole rows; chunk-fastest, all of them would
    // touch the same few hundred bytes of every row, a fraction of the HBM channels); with shorter rows the chunks
    // of one head, whose workspace records are contiguous.
    const bool head_fastest = (uint32_t)(p.H * K) * sizeof(T) >= 4096;
    if (few.chunk_off && (int)blockIdx.x >= p.H * p.st.nch) {
        const int work = (int)blockIdx.x - p.H * p.st.nch, rest = (int)gridDim.x - p.H * p.st.nch - 2;
        if (work < 2)
            few_table(work, p.st.cu, p.st.N, p.st.T, p.st.nch, p.H, few.V, few.chunk_off, few.chunk_seq, *reinterpret_cast<ShareLds*>(sMat), threadIdx.x, K);
        else clear_uncovered(p.st.cu, p.st.N, p.st.T, few.out, work - 2, rest, threadIdx.x, K);
        return;
    }
    const int cid = head_fastest ? blockIdx.x / p.H : blockIdx.x % p.st.nch;
    const int h = head_fastest ? blockIdx.x % p.H : blockIdx.x / p.st.nch;
    ChunkPos cp;
    if (!(few.chunk_off ? locate_few(p.st, cid, cp) : locate_chunk(p.st, cid, cp))) return;
    const int l = lane_id(), g = l >> 4, c = l & 15;
    const int H = p.H;
    const bool rowok = c < cp.len;
    const int64_t tok = cp.tok0 + min(c, cp.len - 1);   // rows past the end alias the last valid row, masked by rowok
    const int64_t chw = (int64_t)h * p.st.nch + cid;                // chunk-head slot in the workspace
    const float scale = p.scale;

    // ---- phase A: decays, the score tiles (rows i, inner j) and the gated copies --------------------------------
    f32x4 aqk = zero4(), aqb[2] = {zero4(), zero4()}, aak[2] = {zero4(), zero4()};
    f32x4 aab[2][2] = {{zero4(), zero4()}, {zero4(), zero4()}};
    const Frag<T> ident = ident_frag<T>();
    Frag<T> ag[2][KTW];                                    // of the own channel tiles; index kt below is local, kt0 + kt global
    typedef std::conditional_t<GKF32, float, bf16> G;
    typedef TileLoad<T, 2> Load;
    typedef TileLoad<G, 2> LoadG;
    const T* const qrow = p.q + (cp.tok0 * H + h) * K + 16 * kt0;
    const T* const krow = p.k + (cp.tok0 * H + h) * K + 16 * kt0;
    const G* const grow = reinterpret_cast<const G*>(p.gk) + (cp.tok0 * H + h) * K + 16 * kt0;
    const T* const arow = HD ? nullptr : p.a + (cp.tok0 * RANK * H + h) * K + 16 * kt0;
    const T* const brow = HD ? nullptr : p.b + (cp.tok0 * RANK * H + h) * K + 16 * kt0;
    const T* const vrow = p.v + (cp.tok0 * H + h) * V + 16 * vt0;
    // two channel tiles of a token: log-decay, q, k, a, b, requested and as fragments
    struct Request { Load q, k, a[2], b[2]; LoadG g; };
    struct Inputs { f32x4 g; Frag<T> q, k, a[2], b[2]; };
    auto request = [&](int kp, Request& x) __attribute__((always_inline)) {
        x.g.load(grow + 32 * kp, H * K, cp.len, l);
        x.k.load(krow + 32 * kp, H * K, cp.len, l);
        x.q.load(qrow + 32 * kp, H * K, cp.len, l);
        if (!HD) {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                x.a[r].load(arow + r * H * K + 32 * kp, RANK * H * K, cp.len, l);
                x.b[r].load(brow + r * H * K + 32 * kp, RANK * H * K, cp.len, l);
            }
        }
    };
    // (both pairs at once: each takes half of the rows' cache lines, and with the second one requested when the first had been used, and three
    // waves a SIMD, the lines had left the L2: 190 -> 208 us for 16384 tokens of 16 heads, K = V = 128; this way 176)
    Request req[KTW / 2];
#pragma unroll
    for (int kp = 0; kp < KTW / 2; ++kp) request(kp, req[kp]);
    __builtin_amdgcn_sched_barrier(0);
    // HDLA parameterisation: a_1 = -beta k, a_2 = beta k (beta s - f), b_1 = f k, b_2 = k with f = exp(gk) and
    // s = sum over ALL channels of k^2 f (two waves exchange their channels' parts)
    float beta_t = 0.f, s_t = 0.f;
    if (HD) beta_t = rowok ? ld_elem(p.beta + tok * H + h) : 0.f;
    f32x4 gks[HD ? KTW : 1];
    Frag<T> ks[HD ? KTW : 1];
    if (HD) {
#pragma unroll
        for (int kp = 0; kp < KTW / 2; ++kp) {
            Frag<G> fg[2];
            Frag<T> f[2];
            req[kp].g.tiles(scratch, cp.len, l, fg);
            req[kp].k.tiles(scratch, cp.len, l, f);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int kt = 2 * kp + e;
                gks[kt] = to_f32(fg[e]);
                ks[kt] = f[e];
                const f32x4 k4 = to_f32(f[e]), kf = k4 * k4 * exp4<T>(gks[kt]);
                s_t += kf[0] + kf[1] + kf[2] + kf[3];
            }
        }
        s_t = sum_groups(s_t);
        if (NWP > 1) {
            if (g == 0) sSum[w * CH + c] = s_t;
            __syncthreads();
            s_t = 0.f;
#pragma unroll
            for (int ww = 0; ww < NWP; ++ww) s_t += sSum[ww * CH + c];
        }
        if (WB && sizeof(T) == 2 && w == 0 && g == 0) p.ws.SUM[chw * CH + c] = s_t;
    }
    // held: with the HDLA parameterisation k and the decays are there already, from the sum
    auto inputs = [&](int kp, const Request& x, Inputs (&in)[2], bool held) __attribute__((always_inline)) {
        Frag<T> f[2];
        Frag<G> fg[2];
        if (!HD || !held) {
            x.g.tiles(scratch, cp.len, l, fg);
            x.k.tiles(scratch, cp.len, l, f);
#pragma unroll
            for (int e = 0; e < 2; ++e) { in[e].g = to_f32(fg[e]); in[e].k = f[e]; }
        } else {
#pragma unroll
            for (int e = 0; e < 2; ++e) { in[e].g = gks[HD ? 2 * kp + e : 0]; in[e].k = ks[HD ? 2 * kp + e : 0]; }
        }
        x.q.tiles(scratch, cp.len, l, f);
#pragma unroll
        for (int e = 0; e < 2; ++e) in[e].q = f[e];
        if (!HD) {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                x.a[r].tiles(scratch, cp.len, l, f);
#pragma unroll
                for (int e = 0; e < 2; ++e) in[e].a[r] = f[e];
                x.b[r].tiles(scratch, cp.len, l, f);
#pragma unroll
                for (int e = 0; e < 2; ++e) in[e].b[r] = f[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const f32x4 kk = to_f32(in[e].k), f4 = exp4<T>(in[e].g);
                in[e].a[0] = to_frag<T>(kk * (-beta_t));
                in[e].a[1] = to_frag<T>(kk * ((beta_t * s_t - f4) * beta_t));
                in[e].b[0] = to_frag<T>(f4 * kk);
                in[e].b[1] = in[e].k;
            }
        }
    };
    // 2-byte elements: one tile's factors and operands at a time, for the registers
    constexpr bool TIGHT = sizeof(T) == 2;
    bool strong = false;
#pragma unroll
    for (int kp = 0; kp < KTW / 2; ++kp) {
        Inputs in[2];
        inputs(kp, req[kp], in, true);
        Frag<T> kgT[2], bgT[2][2], qg[2];                  // [..][tile of the stored pair]
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int kt = 2 * kp + e;
            // Every score is a dense product of operands decayed relative to the middle of the chunk: exp(gi_i - gi_j) =
            // exp(gi_i - m) exp(m - gi_j) with m = gi of token MID.  That is done here for every chunk, tile by tile as the
            // inputs arrive; it is only valid while the exponents stay within +-SAFE_RANGE, which is checked afterwards.
            const TileDecay<T> d(in[e].g, c);
            strong |= d.strong;
            qg[e] = to_frag<T>(to_f32(in[e].q) * d.egi * scale);
            if (!KG_IS_B) kgT[e] = turn(to_frag<T>(to_f32(in[e].k) * d.edn), ident, scratch);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                ag[r][kt] = to_frag<T>(to_f32(in[e].a[r]) * d.ege);
                if (TIGHT) hold(ag[r][kt]);                          // formed here, not where it is used: that would keep a and its factors instead
                bgT[r][e] = turn(to_frag<T>(to_f32(in[e].b[r]) * d.edn), ident, scratch);
            }
            // (the same from all tokens' lanes: without a branch in the way of the scheduler)
            *reinterpret_cast<f32x4*>(p.ws.EGL + chw * (SAS * (int)sizeof(T) / 4) + 16 * (kt0 + kt) + 4 * g) = d.egl;
            if (TIGHT) __builtin_amdgcn_sched_barrier(0);
            // (pin(): converted to fp32 again rather than held so from above)
            if (!HD) {
                pin(in[e].q); pin(in[e].k);
#pragma unroll
                for (int r = 0; r < 2; ++r) { pin(in[e].a[r]); pin(in[e].b[r]); }
            }
            Split<T> kh, bh[2];
            split(to_f32(in[e].k) * d.ek, kh);
            split(to_f32(in[e].b[0]) * d.ek, bh[0]);
            split(to_f32(in[e].b[1]) * d.ek, bh[1]);
            {
                Split<T> qh;
                split(to_f32(in[e].q) * d.eq * scale, qh);
                aqk = mm_split(qh, kh, aqk);
#pragma unroll
                for (int s = 0; s < 2; ++s) aqb[s] = mm_split(qh, bh[s], aqb[s]);
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                if (TIGHT) __builtin_amdgcn_sched_barrier(0);
                Split<T> ah;
                split(to_f32(in[e].a[r]) * d.ea, ah);
                aak[r] = mm_split(ah, kh, aak[r]);
#pragma unroll
                for (int s = 0; s < 2; ++s) aab[r][s] = mm_split(ah, bh[s], aab[r][s]);
            }
            if (TIGHT) __builtin_amdgcn_sched_barrier(0);
        }
        const int pair = kt0 / 2 + kp;
        if (!KG_IS_B) st_pair2(p.ws.KGT + chw * SAS + pair * PAIR, kgT[0], kgT[1]);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (SCAN_U) st_pair2(p.ws.BGT + chw * SAS + (2 * pair + s) * PAIR, bgT[0][s], bgT[1][s]);   // (s: the tile of the pair)
            else st_pair2(p.ws.BGT + chw * SAS + (s * KT2 + pair) * PAIR, bgT[s][0], bgT[s][1]);
        }
        if (!BWD) st_pair2(p.ws.QG + chw * SQS + pair * PAIR, qg[0], qg[1]);
        if (WB) st_pair2(p.ws.QGT + chw * SBS + pair * PAIR, turn(qg[0], ident, scratch), turn(qg[1], ident, scratch));
    }
    // Each wave decides for its own channels (the parts of the score tiles add up whichever way they were formed); the
    // backward pass records the decision per (chunk, head) for the chunk_grad kernels.  Where a channel decays too
    // strongly for the single centre, what was accumulated above may hold infinities: it is thrown away and the tiles
    // are formed again, from inputs read again, by passes whose exponents cannot overflow (see DecayPass).
    if (WB && l == 0) {
        if (NWP == 1) p.ws.STRONG[chw] = strong;
        else sStrong[w] = strong;
    }
    if (strong) {
        aqk = zero4();
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            aqb[s] = zero4(); aak[s] = zero4(); aab[0][s] = zero4(); aab[1][s] = zero4();
        }
        // this path is rare and must not cost the common one registers: one tile and one operand at a time
#pragma unroll 1
        for (int ps = 0; ps < DecayPass::COUNT; ++ps) {
            const DecayPass dp(ps, c);
#pragma unroll 1
            for (int kp = 0; kp < KTW / 2; ++kp) {
                Request x;
                Inputs in[2];
                request(kp, x);
                inputs(kp, x, in, false);
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const f32x4 gi = scan16_incl(in[e].g);
                    f32x4 eq, ek, ea;
                    dp.factors<T>(gi, gi - in[e].g, eq, ek, ea);
                    Split<T> qh, kh, bh[2];
                    split(to_f32(in[e].k) * ek, kh);
                    split(to_f32(in[e].q) * eq * scale, qh);
                    aqk = mm_split(qh, kh, aqk);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        split(to_f32(in[e].b[s]) * ek, bh[s]);
                        aqb[s] = mm_split(qh, bh[s], aqb[s]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        Split<T> ah;
                        split(to_f32(in[e].a[r]) * ea, ah);
                        aak[r] = mm_split(ah, kh, aak[r]);
                        aab[r][0] = mm_split(ah, bh[0], aab[r][0]);
                        aab[r][1] = mm_split(ah, bh[1], aab[r][1]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
    }
    // v is used last (phase D) but requested here: the barriers in between would otherwise keep its loads, and a
    // full round trip to HBM, behind everything else
    Load lv[VTW / 2];
    if (!SCAN_U && WRITE_U)
#pragma unroll
    for (int vp = 0; vp < VTW / 2; ++vp) lv[vp].load(vrow + 32 * vp, H * V, cp.len, l);
    if (NWP > 1) {
        // sums over all channels: every wave leaves its parts in LDS and adds the others'
        f32x4* const tiles[9] = {&aak[0], &aak[1], &aab[0][0], &aab[0][1], &aab[1][0], &aab[1][1],
                                 &aqb[0], &aqb[1], &aqk};
#pragma unroll
        for (int i = 0; i < NPART; ++i) *reinterpret_cast<f32x4*>(&sMat[NWP - 1 - w][(i * 64 + l) * 4]) = *tiles[i];
        __syncthreads();
        static_assert(NWP <= 2, "the other wave");
#pragma unroll
        for (int i = 0; i < NPART; ++i) *tiles[i] += *reinterpret_cast<const f32x4*>(&sMat[w][(i * 64 + l) * 4]);
        if (WB && w == 0 && l == 0) {
            int any = 0;
#pragma unroll
            for (int ww = 0; ww < NWP; ++ww) any |= sStrong[ww];
            p.ws.STRONG[chw] = any;
        }
    }
    // causal masks: lane (g,c) reg i is entry (row c, inner 4g+i)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int j = 4 * g + i;
        const bool le = j <= c, lt = j < c;
        if (!le) { aqk[i] = 0.f; aqb[0][i] = 0.f; aqb[1][i] = 0.f; }
        if (!lt) { aak[0][i] = 0.f; aak[1][i] = 0.f; aab[0][0][i] = 0.f; aab[0][1][i] = 0.f; aab[1][0][i] = 0.f; aab[1][1][i] = 0.f; }
    }
    if (w == 0) {
        if (!BWD) {
            st_tile(p.ws.AQK + chw * SAS, to_frag<T>(aqk));
            st_pair2(p.ws.AQB + chw * SQS, to_frag<T>(aqb[0]), to_frag<T>(aqb[1]));
        }
        if (BWD || WB) {
            // the other orientation is the rounded tile turned (a product with the identity: exact), in every mode, so
            // that a backward pass finds the same bytes whether it recomputes them or reads what a forward pass kept
            st_pair2(p.ws.AQBT + chw * SBS, turn(to_frag<T>(aqb[0]), ident, scratch), turn(to_frag<T>(aqb[1]), ident, scratch));
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int s = 0; s < 2; ++s)
            *reinterpret_cast<f32x4*>(&sN[(16 * r + c) * LDP + 16 * s + 4 * g]) = aab[r][s];
    __syncthreads();

    // ---- phase B: (I - A_ab)^-1 -----------------------------------------------------------------------------------
    // In token halves, L = tokens 0..7 and H = 8..15 (both ranks: 16 rows each):
    //   (I - A)^-1 = [[T_LL, 0], [T_HL, T_HH]],  T_LL = (I - A_LL)^-1,  T_HH = (I - A_HH)^-1,  T_HL = T_HH A_HL T_LL.
    // The diagonal blocks by forward substitution over tokens, in registers, both at once: lane (r, half, column) builds
    // one column of the rows (r, i) of its half, one token per step, the entries of the other rank's rows coming from the
    // lane 32 positions away (eight steps and a quarter of the dependent multiply-adds of one substitution over all
    // sixteen tokens).  The block below the diagonal is two 16 x 16 x 16 products, in split operands like the score
    // products for 2-byte elements (the error of fp32 products), in fp32 products otherwise.
    {
        const int r = l >> 5, hf = (l >> 4) & 1, sc = (l >> 3) & 1, jc = l & 7;
        const int col = 16 * sc + 8 * hf + jc;
        float x[8], y[8];                        // own rows (r, j) and the partner's rows (1-r, j) of column col
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float* nrow = &sN[(16 * r + 8 * hf + i) * LDP + 8 * hf];
            float acc0 = (sc == r && jc == i) ? 1.f : 0.f, acc1 = 0.f;
#pragma unroll
            for (int j4 = 0; j4 < (i + 3) / 4; ++j4) {
                const f32x4 co = *reinterpret_cast<const f32x4*>(nrow + 16 * r + 4 * j4);         // own rank block
                const f32x4 cx = *reinterpret_cast<const f32x4*>(nrow + 16 * (1 - r) + 4 * j4);   // other rank block
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
            sT[(16 * r + 8 * hf + i) * LDP + col] = x[i];
            if (hf == 0) sT[(16 * r + i) * LDP + col + 8] = 0.f;      // rows of L, columns of H: zero
        }
        // (the wave reads below what its other lanes wrote above: LDS accesses of one wave complete in order)
        // 16 x 16 matrices in (rank, token of the half) order: row c = 8 rank + token, inner 4g .. 4g+3 likewise
        const int rr = c >> 3, ii = c & 7, ss = g >> 1, j0 = 4 * (g & 1);
        const f32x4 ahl = *reinterpret_cast<const f32x4*>(&sN[(16 * rr + 8 + ii) * LDP + 16 * ss + j0]);
        const f32x4 thh = *reinterpret_cast<const f32x4*>(&sT[(16 * rr + 8 + ii) * LDP + 16 * ss + 8 + j0]);
        f32x4 tllT;                              // T_LL^T: row c is column c of T_LL
#pragma unroll
        for (int e = 0; e < 4; ++e) tllT[e] = sT[(16 * ss + j0 + e) * LDP + 16 * rr + ii];
        Split<T> pa, pb;
        split(tllT, pa);
        split(ahl, pb);
        const f32x4 xT = mm_split(pa, pb, zero4());   // (A_HL T_LL)^T = T_LL^T A_HL^T
        split(thh, pa);
        split(xT, pb);
        const f32x4 thl = mm_split(pa, pb, zero4());  // T_HH (A_HL T_LL)
        *reinterpret_cast<f32x4*>(&sT[(16 * rr + 8 + ii) * LDP + 16 * ss + j0]) = thl;
        __syncthreads();
    }
    Frag<T> tm[2][2];   // F(Tm^{s s'}): rows i, inner j
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
            tm[s][s2] = to_frag<T>(*reinterpret_cast<const f32x4*>(&sT[(16 * s + c) * LDP + 16 * s2 + 4 * g]));
    if (WB && w == NWP - 1) {
        // for the chunk_grad kernel: the four blocks transposed, as fragments (two tile pairs), ready to load
        T* tmw = p.ws.TM + chw * 1024;
#pragma unroll
        for (int s = 0; s < 2; ++s) st_pair2(tmw + s * PAIR, turn(tm[s][0], ident, scratch), turn(tm[s][1], ident, scratch));
    }

    // ---- phase C: w = Tm ag, two channel tiles (one stored pair) at a time ---------------------------------------
#pragma unroll
    for (int kp = 0; kp < KTW / 2; ++kp) {
        Frag<T> fw[2][2];                                     // [..][tile of the pair]
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const Frag<T> agT[2] = {turn(ag[0][2 * kp + e], ident, scratch), turn(ag[1][2 * kp + e], ident, scratch)};
#pragma unroll
            for (int s = 0; s < 2; ++s) fw[s][e] = to_frag<T>(mm2(tm[s][0], tm[s][1], agT[0], agT[1], zero4()));
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) st_pair2(p.ws.W + chw * SAS + (s * KT2 + kt0 / 2 + kp) * PAIR, fw[s][0], fw[s][1]);
    }

    // ---- phase D: u = Tm (A_ak v), kept transposed (rows value, inner token) ---------------------------------
    const Frag<T> aakf[2] = {to_frag<T>(aak[0]), to_frag<T>(aak[1])};
    if (SCAN_U) {
        if (w == NWP - 1) {
            T* tma = p.ws.TM + chw * (3 * PAIR);
#pragma unroll
            for (int s = 0; s < 2; ++s) st_pair2(tma + s * PAIR, tm[s][0], tm[s][1]);
            st_pair2(tma + 2 * PAIR, aakf[0], aakf[1]);
        }
        return;
    }
    if (sizeof(T) == 2 && w == NWP - 1) st_pair2(p.ws.AAK + chw * PAIR, aakf[0], aakf[1]);
    const bool vtt = sizeof(T) == 4 || p.ws.VTT;
    if (!WRITE_U) {
        if (!p.ws.UT) return;
#pragma unroll
        for (int vp = 0; vp < VTW / 2; ++vp) lv[vp].load(vrow + 32 * vp, H * V, cp.len, l);
    }
    Frag<T> rv[2];
#pragma unroll
    for (int vl = 0; vl < VTW; ++vl) {
        const int vt = vt0 + vl;
        if (vl % 2 == 0) lv[vl / 2].tiles(scratch, cp.len, l, rv);
        const Frag<T> vT = turn(rv[vl % 2], ident, scratch);
        if (vtt) st_tile(p.ws.VTT + (chw * VT + vt) * TILE, vT);
        const Frag<T> mT[2] = {to_frag<T>(mm(vT, aakf[0], zero4())), to_frag<T>(mm(vT, aakf[1], zero4()))};
        Frag<T> fu[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            fu[s] = to_frag<T>(mm2(mT[0], mT[1], tm[s][0], tm[s][1], zero4()));
        }
        st_pair2(p.ws.UT + (chw * VT + vt) * PAIR, fu[0], fu[1]);
    }
}

// workgroups that look for rows to clear: one for every 16 KiB they might have to write, as many as fill the device (of 256 threads 512), and fewer
// where each has a long table to read first
static int clearing_workgroups(int N, int T, const PackedOut& out, int fill = 512) {
    long long bytes = 0;
    for (int b = 0; b < out.n; ++b) bytes += out.row[b] * T;
    const long long most = max(32, min(fill, (1 << 20) / N));
    return (int)min((bytes + 16383) / 16384, most);
}
// kg^T out of bg_2^T for those who look at the classic route's buffers (KG_IS_B above; a store of its own in prep_kernel cost all calls 0.5 us of 48).  RANKS: the pairs are the ranks of a tile.
// A workgroup a slot, of 64 threads
template <int K, bool RANKS>
__global__ __launch_bounds__(64) void kg_of_b_kernel(const bf16* bgt, bf16* kgt, int stride) {
    typedef uint2 Four;                               // four elements
    const int64_t at = (int64_t)blockIdx.x * stride;
    const Four* const from = reinterpret_cast<const Four*>(bgt + at);
    Four* const to = reinterpret_cast<Four*>(kgt + at);
    const int l = lane_id();
#pragma unroll
    for (int pair = 0; pair < K / 32; ++pair)
#pragma unroll
        for (int s = 0; s < 2; ++s)
            to[pair * (PAIR / 4) + 2 * l + s] = RANKS ? from[(2 * pair + s) * (PAIR / 4) + 2 * l + 1] : from[(K / 32 + pair) * (PAIR / 4) + 2 * l + s];
}
template <typename T, int K, int V, bool HD>
static hipError_t launch_prep_kv(const ChunkArgs<T>& a, int mode, const FewTable& few, hipStream_t stream) {
    const int makers = few.chunk_off ? 2 + clearing_workgroups(a.st.N, a.st.T, few.out, FEW_CLEARERS) : 0;
    dim3 grid(a.st.nch * a.H + makers), block(K);
    constexpr bool kAlwaysF32 = sizeof(T) == 4;
    const bool gkf32 = kAlwaysF32 || a.gk_f32;
    constexpr int STATES = sizeof(T) == 2 ? PREP_STATES : PREP_KEEP;
    if (sizeof(T) == 4 && mode == PREP_STATES) return hipErrorInvalidValue;
#define HDLA_PREP_LAUNCH(GK, MODE) hipLaunchKernelGGL((prep_kernel<T, GK, K, V, MODE, HD>), grid, block, 0, stream, a, few)
    if (gkf32) {
        if (mode == PREP_FWD) HDLA_PREP_LAUNCH(true, PREP_FWD);
        else if (mode == PREP_BWD) HDLA_PREP_LAUNCH(true, PREP_BWD);
        else if (mode == PREP_KEEP) HDLA_PREP_LAUNCH(true, PREP_KEEP);
        else HDLA_PREP_LAUNCH(true, STATES);
    } else {
        if (mode == PREP_FWD) HDLA_PREP_LAUNCH(kAlwaysF32, PREP_FWD);
        else if (mode == PREP_BWD) HDLA_PREP_LAUNCH(kAlwaysF32, PREP_BWD);
        else if (mode == PREP_KEEP) HDLA_PREP_LAUNCH(kAlwaysF32, PREP_KEEP);
        else HDLA_PREP_LAUNCH(kAlwaysF32, STATES);
    }
#undef HDLA_PREP_LAUNCH
    if constexpr (HD && sizeof(T) == 2) {
        if (a.ws.KGT) {
            const int stride = a.ws.sa_stride / (int)sizeof(T);
            if (mode == PREP_FWD) hipLaunchKernelGGL((kg_of_b_kernel<K, true>), dim3(a.st.nch * a.H), dim3(64), 0, stream, a.ws.BGT, a.ws.KGT, stride);
            else hipLaunchKernelGGL((kg_of_b_kernel<K, false>), dim3(a.st.nch * a.H), dim3(64), 0, stream, a.ws.BGT, a.ws.KGT, stride);
        }
    }
    return hipGetLastError();
}

template <typename T, bool HD>
static hipError_t launch_prep_hd(const ChunkArgs<T>& a, int K, int V, int mode, const FewTable& few, hipStream_t stream) {
    if (K == 64 && V == 64) return launch_prep_kv<T, 64, 64, HD>(a, mode, few, stream);
    if (K == 128 && V == 128) return launch_prep_kv<T, 128, 128, HD>(a, mode, few, stream);
    if (K == 64 && V == 128) return launch_prep_kv<T, 64, 128, HD>(a, mode, few, stream);
    if (K == 128 && V == 64) return launch_prep_kv<T, 128, 64, HD>(a, mode, few, stream);
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_prep(const ChunkArgs<T>& a, int K, int V, int mode, const PackedOut* out, int share_V, hipStream_t stream) {
    FewTable few{};
    if (out) few = FewTable{const_cast<int32_t*>(a.st.chunk_off), const_cast<int32_t*>(a.st.chunk_seq), share_V, *out};
    return a.beta ? launch_prep_hd<T, true>(a, K, V, mode, few, stream) : launch_prep_hd<T, false>(a, K, V, mode, few, stream);
}
template hipError_t launch_prep<bf16>(const ChunkArgs<bf16>&, int, int, int, const PackedOut*, int, hipStream_t);
template hipError_t launch_prep<float>(const ChunkArgs<float>&, int, int, int, const PackedOut*, int, hipStream_t);

hipError_t launch_clear_uncovered(const int64_t* cu, int N, int T, const PackedOut& out, hipStream_t stream) {
    const int clearers = clearing_workgroups(N, T, out);
    if (clearers == 0) return hipSuccess;
    hipLaunchKernelGGL(clear_uncovered_kernel, dim3(clearers), dim3(TABLE_THREADS), 0, stream, cu, N, T, out);
    return hipGetLastError();
}
hipError_t launch_chunk_table(const int64_t* cu, int N, int T, int nch, int H, int V, int32_t* chunk_off, int32_t* chunk_seq,
                              const PackedOut& out, hipStream_t stream) {
    const int rankers = N <= ORDER_MAX_N ? (N + TABLE_THREADS - 1) / TABLE_THREADS : 0, clearers = clearing_workgroups(N, T, out);
    hipLaunchKernelGGL(build_chunk_table_kernel, dim3(1 + rankers + clearers), dim3(TABLE_THREADS), 0, stream, cu, N, T, nch, H, V, chunk_off,
                       chunk_seq, rankers, out);
    return hipGetLastError();
}

}  // namespace hdla
