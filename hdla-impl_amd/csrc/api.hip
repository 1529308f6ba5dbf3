// C ABI of libhdla_hip.so: argument checks, workspace layout and the launch sequences of the three entry points.
#include "../../include/hdla_hip.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "fused_shapes.h"
#include "hdla_launch.h"
#include "host_path.h"
#include "hdla_ws.h"

using namespace hdla;

namespace {

constexpr int CHUNK = 16;
constexpr int AAK_STRIDE = 512, AAK_STRIDE_RECORD = 1024;    // elements between the tile pairs of A_ak: by themselves, in the record beside those of A_qb

inline size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// max_dim: 128 for the chunked entry points, 256 for the token-serial ones
int check_dims(const hdla_dims* d, int max_dim = 128) {
    if (!d) return HDLA_ERR_NULL;
    if (d->R != 2) return HDLA_ERR_RANK;
    if (d->B < 1 || d->T < 0 || d->H < 1 || d->N < 1) return HDLA_ERR_SHAPE;
    auto ok = [&](int x) { return x == 64 || x == 128 || (x == 256 && max_dim >= 256); };
    if (!ok(d->K) || !ok(d->V)) return HDLA_ERR_SHAPE;
    if (d->H > 65535) return HDLA_ERR_SHAPE;
    if (d->in_dtype != HDLA_BF16 && d->in_dtype != HDLA_FP32) return HDLA_ERR_DTYPE;
    if (d->gk_dtype != HDLA_BF16 && d->gk_dtype != HDLA_FP32) return HDLA_ERR_DTYPE;
    if (d->in_dtype == HDLA_FP32 && d->gk_dtype != HDLA_FP32) return HDLA_ERR_DTYPE;
    if (d->cu_seqlens) { if (d->B != 1) return HDLA_ERR_SEQ; }
    else if (d->N != d->B) return HDLA_ERR_SEQ;
    if (d->route != HDLA_ROUTE_AUTO && d->route != HDLA_ROUTE_CLASSIC && d->route != HDLA_ROUTE_FUSED && d->route != HDLA_ROUTE_PLAIN) return HDLA_ERR_ROUTE;
    if (d->segments < 0) return HDLA_ERR_ROUTE;
    return HDLA_OK;
}

// ---- the fused route (fused_impl.cuh) ----------------------------------------------------------------------------
constexpr int FUSED_MAX_SEGMENTS = 64;       // the segments are chained serially by every workgroup that needs them: about a
                                             // microsecond a segment, against 2.5 for every chunk a segment is shorter
constexpr int FUSED_MIN_SEGMENT_CHUNKS = 8;  // fewer would cost precision, see fused_segments
constexpr int FUSED_TARGET_WORKGROUPS = 256; // one workgroup per compute unit

// the shapes the fused kernels are built for
bool fused_shape(const hdla_dims* d) { return d->in_dtype == HDLA_BF16 && d->K == 64 && d->V == 64; }
// Few short sequences, where the choice is the library's (neither route nor segments asked for): the classic kernels.  A fused workgroup
// takes some 8 us for each round of four chunks of its segment, which is never shorter than eight chunks; the classic kernels prepare all
// chunks at once and then walk them at 0.35 us each.  Below six chunks there is little to walk either way, from 32 on there are four fused
// segments, and beyond 64 lanes the classic kernels' traffic counts.  Measured, us on the device, forward pass / training step, fused ->
// classic: 2 lanes of 16 chunks 27/55 -> 20/46, 8 of 12 28/60 -> 19/44, 16 of 24 34/75 -> 25/65, 64 of 8 22/60 -> 22/56, 64 of 24 37/97 -> 34/95; but
// 8 of 4 22/35 and 22/37, 32 of 32 31/82 and 33/85, 64 of 48 47/140 and 49/160, 128 of 8 23/69 and 30/76.
constexpr int SHORT_MIN_CHUNKS = 6, SHORT_MAX_CHUNKS = 4 * FUSED_MIN_SEGMENT_CHUNKS - 1, SHORT_MAX_LANES = 64;
bool few_short_sequences(const hdla_dims* d, int least = SHORT_MIN_CHUNKS) {
    if (!fused_shape(d) || d->route != HDLA_ROUTE_AUTO || d->segments > 0) return false;
    const long long chunks = ((d->T + CHUNK - 1) / CHUNK) / (d->cu_seqlens ? std::max(d->N, 1) : 1);
    return (long long)d->N * d->H <= SHORT_MAX_LANES && chunks >= least && chunks <= SHORT_MAX_CHUNKS;
}
// The forward pass alone only where the fused route would cut a sequence into segments: below, its workgroup walks the whole
// sequence and a prompt cut into pieces at chunk boundaries comes out in the bits of the whole one, which a line among these lengths would
// end; and up to four chunks, one round in one launch, it is the sooner one.  Measured, us on the device, fused / classic:
// 12 lanes of 2 chunks 8.6/10.4, 4 10.1/11.4, 8 16.8/13.4, 15 28.9/16.7, 30 34/24; 64 lanes of 2 8.8/11.3, 8 17.2/16.6, 15 29/23, 30 38/31.
constexpr int SHORT_MIN_CHUNKS_FWD = 2 * FUSED_MIN_SEGMENT_CHUNKS;
int short_least(int pass) { return pass == HDLA_PASS_FWD ? SHORT_MIN_CHUNKS_FWD : SHORT_MIN_CHUNKS; }
// whether the plain entry points take the fused route for these dimensions; HDLA_ROUTE_FUSED on another shape is an error.
// with_boundary: a boundary (or record) buffer is given: then it is the fused route's.
int pick_route(const hdla_dims* d, int pass, bool with_boundary, bool& fused) {
    fused = d->route != HDLA_ROUTE_CLASSIC && d->route != HDLA_ROUTE_PLAIN && fused_shape(d) && (with_boundary || !few_short_sequences(d, short_least(pass)));
    if (d->route == HDLA_ROUTE_FUSED && !fused) return HDLA_ERR_ROUTE;
    return HDLA_OK;
}
// Time segments per sequence: as many as give every compute unit a workgroup, of eight chunks at the least.  Segments of four
// chunks are faster where few (sequence, head) lanes leave the device idle (us, forward pass / training step, eight -> four:
// 2 lanes of 16 chunks 26/75 -> 20/70, 8 of 63 44/126 -> 32/96, 16 of 125 50/158 -> 49/141), but the states entering the later
// segments reach the outputs through G, which is rounded to 2 bytes once more than what a whole scan multiplies: with twice the
// segments the gradients are further from a float64 evaluation (mean of 12 inputs: by 0.3 to 0.4 % of the error for 2 lanes of 16
// chunks, by 0.1 to 0.2 % for 16 of 125, by 0.04 to 0.09 % for 8 of 63; standard errors 0.15, 0.02, 0.02 %).  Splitting the
// entering states and the transitions into two 2-byte halves each takes half of that away, for 3 us of a forward pass of 81.
int fused_segments(const hdla_dims* d) {
    if (d->segments > 0) return d->segments < FUSED_MAX_SEGMENTS ? d->segments : FUSED_MAX_SEGMENTS;
    const long long lanes = (long long)d->N * d->H;
    const long long chunks_per_seq = ((d->T + CHUNK - 1) / CHUNK) / (d->cu_seqlens ? d->N : 1);
    int nseg = 1;
    while (nseg * 2 <= FUSED_MAX_SEGMENTS && lanes * nseg * 2 <= FUSED_TARGET_WORKGROUPS &&
           chunks_per_seq / (nseg * 2) >= FUSED_MIN_SEGMENT_CHUNKS) nseg *= 2;
    return nseg;
}

// ---- time segments of the stand-alone scans (scan_impl.cuh, scan_out.cuh, scan_grad.cuh): where a whole sequence per workgroup would leave most of the
// device idle.  A launch for the segments' records, one that chains them, then the scans on shorter sequences: twice the steps,
// of which nseg run at once.
constexpr int SCAN_MAX_SEGMENTS = 32;
// Records (lanes x segments) of a segment count asked for: a record is a state and a matrix of K x K, a few of them per pass, and
// a sequence's segments share a grid dimension with the sequences (65535).  The device is full long before this many.
constexpr long long SCAN_MAX_RECORDS = 4096;
// 2-byte elements: the time of a pass's scans (us), from the launches a number of segments makes.  A step takes what its chain of
// products does, which grows with K, until the lanes in flight read more than comes in meanwhile; so does one of the records' launch, which
// has the transitions' columns beside the state's; then there are these two launches, and the records chained one behind the other.
// Fitted to passes of 32 to 400 chunks and 1 to 32 lanes, K, V in {64, 128}, each in 1, 4, 8, 16 and 32 segments (216 shapes): the choice costs
// 0.2 % (forward) and 0.6 % (backward pass) more than the best of these, 6 and 9 % at the most.  A least length for every number of lanes, 13 chunks forward and 7
// backward, cost 3.8 and 5.4 %, 40 and 27 % at the most.  us, forward / backward pass in one segment -> in 4 -> in 8 (* the choice), K = V = 128:
// 2 lanes of 97 chunks 61/68 -> 57/65 -> 49*/58*, 8 lanes of 64 50*/70* -> 52/78 -> 50/84, 16 lanes of 97 77*/162* -> 77/190 -> 87/206,
// 24 lanes of 97 84*/241* -> 113/270 -> 118/293, 8 lanes of 313 175/336 -> 144/297 -> 110*/292*.
struct ScanTime { double step, step_k, load, rec, rec_k, rec_load, launches, chain, chain_k; int most; };   // most: lanes x segments
constexpr ScanTime SCAN_TIME_FWD{0.18, 0.13, 0.0024, 0.37, 0.12, 0.0015, 6.5, 0.04, 0.73, 128},
    SCAN_TIME_BWD{0.26, 0.20, 0.0042, 0.29, 0.16, 0.0054, 21., 0.37, 0.49, 64};
// The backward pass that is given the forward one's transitions: the records' launch has the reverse direction's state columns only.
constexpr ScanTime SCAN_TIME_BWD_KEPT{0.26, 0.20, 0.0042, 0.61, 0.37, 0.0030, 0.5, -0.19, 2.07, 128};
// chunks: of a sequence on average; longest: of the longest one, whose chain of steps the launch waits for.
double scan_time(const ScanTime& t, const hdla_dims* d, double lanes, long long chunks, long long longest, int nseg) {
    const double k = d->K / 64., v = d->V / 64., columns = &t == &SCAN_TIME_BWD_KEPT ? v : k + v;
    const double steps = (double)((chunks + nseg - 1) / nseg), chain = (double)((longest + nseg - 1) / nseg);
    const double walk = std::max(chain * (t.step + t.step_k * k), steps * t.load * lanes * nseg * k * v);
    if (nseg == 1) return walk;
    return walk + std::max(chain * (t.rec + t.rec_k * k), steps * t.rec_load * lanes * (nseg - 1) * k * columns) + t.launches +
           nseg * (t.chain + t.chain_k * k);
}
// The lengths of packed sequences are on the device: the longest one is taken for 1.6 times the average.  128 batches of 2 to 12 sequences
// of random lengths, forward / backward pass over the best of the five: 5.7 / 3.3 % on average (1.0: 6.4 / 3.5, 2.5: 6.4 / 3.5; a least length as
// above: 6.3 / 4.2).
constexpr double PACKED_LONGEST = 1.6;
long long average_chunks(const hdla_dims* d) { return ((d->T + CHUNK - 1) / CHUNK) / (d->cu_seqlens ? d->N : 1); }
long long longest_chunks(const hdla_dims* d) { return d->cu_seqlens && d->N > 1 ? (long long)(average_chunks(d) * PACKED_LONGEST) : average_chunks(d); }
int scan_segments(const hdla_dims* d, bool bwd) {
    if (d->route != HDLA_ROUTE_AUTO) return 1;
    const long long lanes = (long long)d->N * d->H;
    if (d->segments > 0) return (int)std::max(1LL, std::min<long long>({d->segments, SCAN_MAX_SEGMENTS, SCAN_MAX_RECORDS / lanes}));
    const long long chunks = average_chunks(d);
    int nseg = 1;
    if (d->in_dtype != HDLA_FP32) {
        const ScanTime& t = bwd ? SCAN_TIME_BWD : SCAN_TIME_FWD;
        const long long longest = longest_chunks(d);
        double best = scan_time(t, d, (double)lanes, chunks, longest, 1);
        for (int n = 4; n <= SCAN_MAX_SEGMENTS && lanes * n <= t.most; n *= 2) {      // (two only make up for the second walk)
            const double x = scan_time(t, d, (double)lanes, chunks, longest, n);
            if (x < best) { best = x; nseg = n; }
        }
        return nseg;
    }
    // 4-byte elements: a step takes 2-4 us; beyond 128 lanes x segments the records' launch needs more than one round on the
    // device.  us, forward / backward pass, one segment -> as many as chosen here: K = V = 64, 16 lanes of 63 chunks 148/216 ->
    // 72/152 (8); K = V = 128, 4 lanes of 125 chunks 816/894 -> 155/282 (16).
    while (nseg * 2 <= SCAN_MAX_SEGMENTS && lanes * nseg * 2 <= 128 && chunks / (nseg * 2) >= 4) nseg *= 2;
    return nseg >= 4 ? nseg : 1;
}

// Segments of the passes that keep and are given a forward pass's workspace: as many as asked for (hdla_keep_plan's choice), one where
// nothing is said.
int kept_segments(const hdla_dims* d) { return d->segments > 0 ? scan_segments(d, false) : 1; }

// What a training call keeps of its forward pass where nothing else is said: all that the prep kernel forms, which the backward pass would form
// again (in 16 bits 1.06 to 1.25 times the inputs' bytes, in 32 1.3 to 1.7), and the records of the segments; of one call this much, 0.1 % of the device's memory (what all of them hold,
// the caller bounds: native.cpp, kept_room).  With its scratch a call's backward pass
// then has 5 % more than one that recomputes has, median of 949 shapes, 45 % at the most, where the forward pass alone is in segments.  us on the device, a training step
// that keeps the inputs -> this: 1 x 256 tokens, 2 heads, K = V = 64 43 -> 37; 2 x 1537 tokens, 8 heads, K = V = 128 214 -> 185;
// 4 x 1000 tokens, 16 heads 430 -> 393; 4 x 500, 8 heads 127 -> 107; fp32, 2 x 1003 tokens, 8 heads, K = V = 64 227 -> 190.
constexpr size_t KEEP_MOST = (size_t)256 << 20;
// Segments of the two passes of such a call (return, bwd).  The forward pass has those it has without gradients, and so the same bits (what recomputes a
// part of a model runs one pass without and one with them); the backward pass takes these, whose entering states and transitions are there,
// or, with 2-byte elements, none where that is the sooner by more than the times above are off by.  us, a training step in one segment -> in four forward and
// one backward -> four -> eight in both passes (* the choice), K = V = 128: 16 lanes of 200 chunks 402 -> 392 -> 384* -> 386, 16 of 313 654 -> 608 ->
// 571* -> 560, 12 of 128 207 -> 204 -> 217* -> 219; 16 of 97 in one, four, eight 182* -> 211 -> 214.  (Eight in both for the second, and for 4-byte elements at K = 128 four from
// 8 chunks on, 166 -> 137 for 16 lanes of 8, would need a forward pass in other segments than without gradients.)
int kept_plan_segments(const hdla_dims* d, int32_t& bwd) {
    const int fwd = bwd = scan_segments(d, false);
    if (fwd == 1 || d->segments > 0 || d->in_dtype == HDLA_FP32) return fwd;
    const double lanes = (double)d->N * d->H;
    const long long chunks = average_chunks(d), longest = longest_chunks(d);
    const auto time = [&](int n) { return scan_time(SCAN_TIME_BWD_KEPT, d, lanes, chunks, longest, n); };
    if (time(1) < 0.95 * time(fwd)) bwd = 1;
    return fwd;
}

// Whether a training call can leave the states that enter the chunks as well (hdla_states_plan), 2.0 times the inputs' bytes in all at K = V = 128 where the chunks'
// operands alone are 1.1: the forward pass's scan has them, and the backward pass's reverse scan has the device to itself.  Not where both scans of that
// pass fit the device in their narrowest workgroups: side by side they take no longer than one.  us a training step, without the states -> with them, 2-byte elements, K = V = 128:
// 16384 tokens of 16 heads in 4 sequences, where nothing is kept otherwise, 1630 -> 1424 (the pair of scans 510 -> 328, the forward pass's 253 -> 378, prep 348 -> 190), 4 x 2048, beta
// form 717 -> 627; K = 64, V = 128, 32 x 300 of 32 1071 -> 880; K = 128, V = 64, 16 x 1000 of 16, beta form 983 -> 757.  On the other side of the line, as a graph's replay, 16 lanes of 63 chunks
// 116 -> 115, 16 of 97 162 -> 159, 8 of 63 98.4 -> 98.0.  Which calls take them: native.cpp, chunk_forward.  STATES_MOST: what calls may hold on a device in all (kept_room there).
constexpr size_t STATES_MOST = (size_t)1 << 30;
constexpr long long SCAN_PAIR_WORKGROUPS = 256;               // one a compute unit (launch_scan_grad_shape)
bool leaves_states(const hdla_dims* d) {
    if (2LL * d->N * d->H * (d->V / 16) <= SCAN_PAIR_WORKGROUPS || d->in_dtype != HDLA_BF16 || d->route != HDLA_ROUTE_AUTO || d->segments > 1) return false;
    return scan_segments(d, false) == 1 && scan_segments(d, true) == 1;
}

struct FusedLayout {
    size_t OL, GW, SLOC, MSEG, RSEG, SIN, ERR;                 // fused kernels' own
    size_t HC, DHC, DVN, TM, UT, W, SUM, STRONG;               // what chunk_grad reads (backward pass; UT and W beside fp32 decays)
    size_t MT, AQ;                                             // and the rest of the record
    size_t CHUNK_OFF, CHUNK_SEQ;
    size_t total;
    int nch, nseg;
};
constexpr int PASS_BWD_RECORD = -2;          // a backward pass that is given the record (hdla_record_workspace_bytes)
int make_fused_layout(const hdla_dims* d, int pass, FusedLayout& L) {
    const int rc = check_dims(d);
    if (rc) return rc;
    if (d->N > 65535) return HDLA_ERR_SHAPE;
    const int NT = (d->T + CHUNK - 1) / CHUNK;
    const long long nch64 = d->cu_seqlens ? (long long)NT + d->N : (long long)d->B * NT;
    if (nch64 * d->H > 0x7fff0000LL) return HDLA_ERR_SHAPE;
    L = FusedLayout{};
    L.nch = (int)nch64;
    L.nseg = fused_segments(d);
    const size_t es = 2, K = d->K, V = d->V;
    const size_t chw = (size_t)d->H * (size_t)L.nch, recs = (size_t)d->N * d->H * L.nseg;
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += up256(bytes); return o; };
    L.ERR = take(256);
    if (pass != PASS_BWD_RECORD) {                            // of the passes that form the segments' records
        L.SLOC = take(recs * K * V * 4);
        L.MSEG = take(recs * K * K * 4);
    }
    if (pass == HDLA_PASS_FWD) {
        L.OL = take(chw * 16 * V * 4);
        L.GW = take(chw * 16 * K * es);
    } else {
        L.RSEG = take(recs * K * V * 4);
        if (pass == HDLA_PASS_BWD) {                               // what a record holds
            L.SIN = take(recs * K * V * 4);
            L.MT = take(recs * K * K * 4);
            L.GW = L.nseg > 1 ? take(chw * 16 * K * es) : 0;
            L.AQ = take(chw * 1024 * es);
            L.TM = take(chw * 1024 * es);
            L.STRONG = take(chw * 4);
        }
        L.HC = take(chw * K * V * es);
        L.DHC = take(chw * K * V * es);
        L.DVN = take(chw * 2 * 16 * V * es);
        if (d->gk_dtype == HDLA_FP32) { L.UT = take(chw * 2 * V * 16 * es); L.W = take(chw * 2 * K * 16 * es); }
        L.SUM = take(chw * 64);
    }
    if (d->cu_seqlens) {
        L.CHUNK_OFF = take((size_t)(2 * d->N + 1) * 4);
        L.CHUNK_SEQ = take((size_t)(L.nch > 0 ? L.nch : 1) * 4);
    }
    L.total = off;
    return HDLA_OK;
}
size_t fused_boundary_bytes(const hdla_dims* d) {
    const int nseg = fused_segments(d);
    return nseg > 1 ? (size_t)d->N * d->H * nseg * d->K * d->V * 4 : 0;
}
// The record a forward pass hands to the backward pass: the boundary states (first, so that a record is a boundary), the
// segments' transitions, and per (chunk, head) what the score tiles come to (fused_impl.cuh).
struct FusedRecord { size_t SIN, MT, GW, TM, AQ, STRONG, total; };
FusedRecord fused_record(const hdla_dims* d, const FusedLayout& L) {
    FusedRecord r{};
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += up256(bytes); return o; };
    const size_t chw = (size_t)d->H * (size_t)L.nch, recs = (size_t)d->N * d->H * L.nseg;
    r.SIN = take(fused_boundary_bytes(d));
    if (L.nseg > 1) { r.MT = take(recs * d->K * d->K * 4); r.GW = take(chw * 16 * d->K * 2); }
    r.TM = take(chw * 1024 * 2);
    r.AQ = take(chw * 1024 * 2);
    r.STRONG = take(chw * 4);
    r.total = off;
    return r;
}

// pass: HDLA_PASS_FWD, _BWD, _FWD_KEEP (a forward pass that leaves what the backward pass needs of it), _BWD_KEPT (the
// scratch of a backward pass that runs on such a workspace: only what its own scans write), PASS_FWD_STATES and PASS_BWD_STATES (the same two where the
// states that enter the chunks are left as well)
constexpr int PASS_FWD_STATES = 4, PASS_BWD_STATES = 5;
int make_layout(const hdla_dims* d, int pass, WsLayout& L, int& nch) {
    const int rc = check_dims(d);
    if (rc) return rc;
    if (d->N > 65535) return HDLA_ERR_SHAPE;
    const int NT = (d->T + CHUNK - 1) / CHUNK;
    const long long nch64 = d->cu_seqlens ? (long long)NT + d->N : (long long)d->B * NT;
    if (nch64 * d->H > 0x7fff0000LL) return HDLA_ERR_SHAPE;        // one workgroup per (chunk, head), one grid dimension (and room for the strided loops over them)
    nch = (int)nch64;
    const size_t es = d->in_dtype == HDLA_BF16 ? 2 : 4;
    const size_t chw = (size_t)d->H * (size_t)nch;
    const size_t K = d->K, V = d->V;
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += up256(bytes); return o; };
    L = WsLayout{};
    const bool states = pass == PASS_FWD_STATES;
    const bool prep_out = pass != HDLA_PASS_BWD_KEPT && pass != PASS_BWD_STATES;   // what the prep kernel writes
    const bool with_o = pass == HDLA_PASS_FWD || pass == HDLA_PASS_FWD_KEEP;
    const bool bwd_parts = pass == HDLA_PASS_BWD || pass == HDLA_PASS_FWD_KEEP || states;
    const bool scan_out = pass == HDLA_PASS_BWD || pass == HDLA_PASS_BWD_KEPT || pass == PASS_BWD_STATES;
    if (prep_out) {
        const BlkF bf = blk_fwd(d->K, (int)es, with_o);
        const size_t sa = take(chw * (size_t)bf.SIZE);
        L.SA_STRIDE = bf.SIZE;
        L.W = sa + bf.W; L.BGT = sa + bf.BGT; L.KGT = sa + bf.KGT; L.EGL = sa + bf.EGL;
        if (states) L.AQK = sa + blk_fwd(d->K, (int)es, true).AQK;   // (q's tiles and A_qb are in the forward pass's own workspace)
        if (with_o) { L.QG = sa + bf.QG; L.AQB = sa + bf.AQB; L.AQK = sa + bf.AQK; }
        if (pass == HDLA_PASS_FWD && es == 2) {
            L.TM = take(chw * 1536 * es);                         // the scan forms u itself (scan_out.cuh)
        } else {
            // (2-byte elements: the scans form u and v^T themselves.  chunk_grad reads u beside fp32 decays; v^T is there, and u, for whoever names the classic
            // route and looks at a backward pass's buffers.  The library's own plans name the plain one: us a training step that finds no room to keep its
            // forward pass, classic -> plain, 4 x 1000 tokens of 16 heads, K = V = 128 413 -> 392, 4 x 2048, K = 64, V = 128 490 -> 465.)
            const bool shown = pass == HDLA_PASS_BWD && d->route == HDLA_ROUTE_CLASSIC;
            if (d->gk_dtype == HDLA_FP32 || shown) L.UT = take(chw * 2 * V * 16 * es);
            if (es == 4 || shown) L.VTT = take(chw * V * 16 * es);
            if (es == 2) { L.AAK = take(chw * 512 * es); L.SUM = take(chw * 64); }
        }
    }
    if (bwd_parts) {
        const BlkB bb = blk_bwd(d->K, (int)es);
        const size_t sb = take(chw * (size_t)bb.SIZE);
        L.SB_STRIDE = bb.SIZE;
        L.QGT = sb + bb.QGT; L.AQBT = sb + bb.AQBT;
        L.TM = take(chw * 1024 * es);
        L.STRONG = take(chw * 4);
    }
    if (scan_out) {
        if (pass != PASS_BWD_STATES) L.HC = take(chw * K * V * es);
        L.DHC = take(chw * K * V * es);
        L.DVN = take(chw * 2 * 16 * V * es);
    }
    if (states) L.HC = take(chw * K * V * es);
    if (d->cu_seqlens && prep_out) {
        L.CHUNK_OFF = take((size_t)(2 * d->N + 1) * 4);          // chunk_off [N+1], then order [N]
        L.CHUNK_SEQ = take((size_t)(nch > 0 ? nch : 1) * 4);
    }
    const int nseg = states || pass == PASS_BWD_STATES ? 1 : pass == HDLA_PASS_FWD || pass == HDLA_PASS_BWD ? scan_segments(d, pass == HDLA_PASS_BWD) : kept_segments(d);
    if (nseg > 1) {
        const size_t recs = (size_t)d->N * d->H * nseg, state = recs * K * V * 4, matrix = recs * K * K * 4;
        if (prep_out) { L.SEG_LOC = take(state); L.SEG_TR = take(matrix); L.SEG_IN = take(state); }
        if (pass == HDLA_PASS_FWD_KEEP) L.SEG_RTR = take(matrix);
        if (pass == HDLA_PASS_BWD) { L.SEG_RLOC = take(state); L.SEG_RTR = take(matrix); L.SEG_RIN = take(state); }
        if (pass == HDLA_PASS_BWD_KEPT) { L.SEG_RLOC = take(state); L.SEG_RIN = take(state); }
    }
    // (behind the rest: where a backward pass finds what it reads does not depend on the routes that the two passes are called with)
    if (pass == HDLA_PASS_FWD_KEEP && d->route == HDLA_ROUTE_CLASSIC && !L.UT) L.UT = take(chw * 2 * V * 16 * es);
    L.total = off > 0 ? off : 256;
    return HDLA_OK;
}

// what the prep kernel writes (and the sequence tables) lives in `prep_ws`, laid out by LP; what the scans of the
// backward pass write lives in `scan_ws`, laid out by LS (the same buffer and layout unless the backward pass runs on a
// kept forward workspace)
template <typename T>
void bind_ws(ChunkArgs<T>& a, const hdla_dims* d, const WsLayout& LP, void* prep_ws, const WsLayout& LS, void* scan_ws, int nch) {
    char* base = static_cast<char*>(prep_ws);
    auto at = [&](size_t o) { return reinterpret_cast<T*>(base + o); };
    a.ws.W = at(LP.W); a.ws.UT = LP.UT ? at(LP.UT) : nullptr; a.ws.BGT = at(LP.BGT);
    a.ws.KGT = sizeof(T) == 2 && a.beta && d->route != HDLA_ROUTE_CLASSIC ? nullptr : at(LP.KGT);   // (nobody's, then: prep.hip, KG_IS_B)
    a.ws.VTT = LP.VTT ? at(LP.VTT) : nullptr; a.ws.AAK = at(LP.AAK); a.ws.aak_stride = AAK_STRIDE;
    a.ws.SUM = reinterpret_cast<float*>(base + LP.SUM);
    a.ws.QG = at(LP.QG); a.ws.AQK = at(LP.AQK); a.ws.AQB = at(LP.AQB);
    a.ws.AQBT = at(LP.AQBT); a.ws.QGT = at(LP.QGT);
    a.ws.EGL = reinterpret_cast<float*>(base + LP.EGL);
    a.ws.TM = at(LP.TM);
    a.ws.STRONG = reinterpret_cast<int32_t*>(base + LP.STRONG);
    a.ws.sa_stride = (int)LP.SA_STRIDE;
    char* sbase = static_cast<char*>(scan_ws);
    a.ws.HC = reinterpret_cast<T*>(sbase + LS.HC); a.ws.DHC = reinterpret_cast<T*>(sbase + LS.DHC);
    a.ws.DVN = reinterpret_cast<T*>(sbase + LS.DVN);
    a.st.cu = d->cu_seqlens;
    a.st.chunk_off = d->cu_seqlens ? reinterpret_cast<const int32_t*>(base + LP.CHUNK_OFF) : nullptr;
    a.st.chunk_seq = d->cu_seqlens ? reinterpret_cast<const int32_t*>(base + LP.CHUNK_SEQ) : nullptr;
    a.st.order = d->cu_seqlens ? a.st.chunk_off + d->N + 1 : nullptr;
    a.st.T = d->T;
    a.st.NT = (d->T + CHUNK - 1) / CHUNK;
    a.st.N = d->N;
    a.st.nch = nch;
}

template <typename T> PackedOut packed_outputs(const hdla_dims* d, const ChunkArgs<T>& a) {
    PackedOut out{};
    const long long H = d->H, k = H * d->K * (long long)sizeof(T), v = H * d->V * (long long)sizeof(T);
    out.add(a.o, v);
    out.add(a.dq, k); out.add(a.dk, k); out.add(a.dv, v); out.add(a.da, 2 * k); out.add(a.db, 2 * k);
    out.add(a.dgk, H * d->K * (a.gk_f32 ? 4 : 2)); out.add(a.dbeta, H * (long long)sizeof(T));
    return out;
}

inline bool bad_ws(const void* p, size_t have, size_t need) {
    return !p || (reinterpret_cast<uintptr_t>(p) & 255) || have < need;
}

// what a forward pass that leaves the states has for itself
size_t states_fwd_workspace(const hdla_dims* d, int nch) { return std::max<size_t>(256, up256((size_t)d->H * nch * blk_q(d->K, 2))); }

// pass: HDLA_PASS_FWD / _BWD on `workspace`; HDLA_PASS_FWD_KEEP on `kept`; HDLA_PASS_BWD_KEPT on `kept` (read) and
// `workspace` (what the scans write); PASS_FWD_STATES and PASS_BWD_STATES on both
template <typename T>
int run_chunk(const hdla_dims* d, int pass, const void* q, const void* k, const void* v, const void* a_,
              const void* b, const void* gk, const float* h0, void* o, float* ht, const void* d_o,
              const float* dht, void* dq, void* dk, void* dv, void* da, void* db, void* dgk, float* dh0,
              void* workspace, size_t workspace_bytes, hipStream_t stream, int stages = HDLA_STAGE_ALL,
              const void* beta = nullptr, void* dbeta = nullptr, void* kept = nullptr, size_t kept_bytes = 0) {
    WsLayout LP, LS;
    int nch = 0;
    const bool states = pass == PASS_FWD_STATES || pass == PASS_BWD_STATES;
    const bool fwd = pass == HDLA_PASS_FWD || pass == HDLA_PASS_FWD_KEEP || pass == PASS_FWD_STATES;
    const bool on_kept = pass == HDLA_PASS_FWD_KEEP || pass == HDLA_PASS_BWD_KEPT || states;
    hdla_dims kept_dims = *d;
    if (pass == HDLA_PASS_BWD_KEPT && d->route == HDLA_ROUTE_CLASSIC) kept_dims.route = HDLA_ROUTE_PLAIN;   // (what this pass reads)
    int rc = make_layout(&kept_dims, states ? PASS_FWD_STATES : on_kept ? HDLA_PASS_FWD_KEEP : pass, LP, nch);
    if (rc) return rc;
    void* prep_ws = on_kept ? kept : workspace;
    if (bad_ws(prep_ws, on_kept ? kept_bytes : workspace_bytes, LP.total)) return HDLA_ERR_WORKSPACE;
    LS = LP;
    if (pass == PASS_FWD_STATES && bad_ws(workspace, workspace_bytes, states_fwd_workspace(d, nch))) return HDLA_ERR_WORKSPACE;
    if (pass == HDLA_PASS_BWD_KEPT || pass == PASS_BWD_STATES) {
        rc = make_layout(d, pass, LS, nch);
        if (rc) return rc;
        if (bad_ws(workspace, workspace_bytes, LS.total)) return HDLA_ERR_WORKSPACE;
        // (the records lie where their number puts them: another number's buffer, which another size shows, would be read wrongly)
        if (!states && kept_segments(d) > 1 && kept_bytes != LP.total) return HDLA_ERR_WORKSPACE;
    }
    ChunkArgs<T> a{};
    a.q = static_cast<const T*>(q); a.k = static_cast<const T*>(k); a.v = static_cast<const T*>(v);
    a.a = static_cast<const T*>(a_); a.b = static_cast<const T*>(b);
    a.gk = gk; a.gk_f32 = d->gk_dtype == HDLA_FP32;
    a.H = d->H; a.scale = d->scale;
    a.h0 = h0; a.ht = fwd ? ht : nullptr; a.o = static_cast<T*>(o);
    a.dout = static_cast<const T*>(d_o); a.dht = dht; a.dh0 = dh0;
    a.dq = static_cast<T*>(dq); a.dk = static_cast<T*>(dk); a.dv = static_cast<T*>(dv);
    a.da = static_cast<T*>(da); a.db = static_cast<T*>(db); a.dgk = dgk;
    a.beta = static_cast<const T*>(beta); a.dbeta = static_cast<T*>(dbeta);
    bind_ws(a, d, LP, prep_ws, LS, pass == HDLA_PASS_BWD_KEPT || pass == PASS_BWD_STATES ? workspace : prep_ws, nch);
    if (states) a.ws.HC = reinterpret_cast<T*>(static_cast<char*>(kept) + LP.HC);
    if (pass == PASS_FWD_STATES) {
        constexpr int es = 2;
        const BlkF b = blk_fwd(d->K, es, true);
        a.ws.QG = static_cast<T*>(workspace);
        a.ws.AQB = reinterpret_cast<T*>(static_cast<char*>(workspace) + (b.AQB - b.QG));
    }
    a.seg = SegRec{1, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    const int nseg = states ? 1 : on_kept ? kept_segments(d) : scan_segments(d, !fwd);
    if (nseg > 1) {
        const auto at = [](void* base, size_t o) { return reinterpret_cast<float*>(static_cast<char*>(base) + o); };
        a.seg = SegRec{nseg, at(prep_ws, LP.SEG_LOC), at(prep_ws, LP.SEG_TR), at(prep_ws, LP.SEG_IN), nullptr, nullptr, nullptr, nullptr};
        if (!fwd) { a.seg.rloc = at(workspace, LS.SEG_RLOC); a.seg.rtr = at(prep_ws, LP.SEG_RTR); a.seg.rin = at(workspace, LS.SEG_RIN); }
        // (a backward pass that is told its number of segments: the transitions as one on a kept workspace meets them, so that its bits do not depend on
        // whether there was room to keep one)
        if (pass == HDLA_PASS_FWD_KEEP || (pass == HDLA_PASS_BWD && d->segments > 0)) a.seg.turned = at(prep_ws, LP.SEG_RTR);
    }
    hipError_t e;
    if (pass == PASS_BWD_STATES) stages &= ~HDLA_STAGE_SCAN_FWD;   // the forward pass has left what it leaves
    if (pass == HDLA_PASS_BWD_KEPT || pass == PASS_BWD_STATES) {
        stages &= ~HDLA_STAGE_PREP;                                // the forward pass has run it
        if (d->cu_seqlens) {
            e = launch_clear_uncovered(d->cu_seqlens, d->N, d->T, packed_outputs(d, a), stream);
            if (e != hipSuccess) return (int)e;
        }
    }
    if (stages & HDLA_STAGE_PREP) {
        // whether one of the scans on this table is shared out by the sequences' lengths (a kept one: of either pass, the backward one's in as many segments
        // or one)
        const bool shares = sizeof(T) == 2 && scan_shares(d->cu_seqlens, d->N, d->H, d->V, pass == HDLA_PASS_FWD_KEEP ? 1 : nseg, pass == HDLA_PASS_FWD ? 1 : 2);
        const int share_V = shares ? d->V : 0;
        const PackedOut out = packed_outputs(d, a);
        const bool made = prep_makes_table(d->cu_seqlens, d->N, d->H, nch);
        if (d->cu_seqlens && !made) {
            e = launch_chunk_table(d->cu_seqlens, d->N, d->T, nch, d->H, share_V, const_cast<int32_t*>(a.st.chunk_off), const_cast<int32_t*>(a.st.chunk_seq),
                                   out, stream);
            if (e != hipSuccess) return (int)e;
        }
        if (nch > 0) {
            e = launch_prep<T>(a, d->K, d->V, pass == HDLA_PASS_FWD ? 0 : pass == HDLA_PASS_BWD ? 1 : pass == PASS_FWD_STATES ? 3 : 2, made ? &out : nullptr, share_V, stream);
            if (e != hipSuccess) return (int)e;
        }
    }
    if (a.seg.nseg > 1 && (stages & HDLA_STAGE_CHAIN)) {
        const SegStart what = pass == HDLA_PASS_FWD ? SEG_FWD : pass == HDLA_PASS_FWD_KEEP ? SEG_FWD_KEPT : pass == HDLA_PASS_BWD ? SEG_BWD : SEG_BWD_KEPT;
        e = launch_scan_segments<T>(a, d->K, d->V, what, stream);
        if (e != hipSuccess) return (int)e;
    }
    // the two scans of the backward pass are independent of each other: one launch when both are asked for
    const bool pair = !fwd && (stages & HDLA_STAGE_SCAN_FWD) && (stages & HDLA_STAGE_SCAN_BWD);
    if (pair) {
        e = launch_scan_pair<T>(a, d->K, d->V, stream);
        if (e != hipSuccess) return (int)e;
    } else if (stages & HDLA_STAGE_SCAN_FWD) {
        e = fwd ? launch_scan_out<T>(a, d->K, d->V, pass == PASS_FWD_STATES ? 2 : pass == HDLA_PASS_FWD_KEEP, stream) : launch_scan_fwd<T>(a, d->K, d->V, stream);
        if (e != hipSuccess) return (int)e;
    }
    if (!fwd) {
        if (!pair && (stages & HDLA_STAGE_SCAN_BWD)) {
            e = launch_scan_bwd<T>(a, d->K, d->V, stream);
            if (e != hipSuccess) return (int)e;
        }
        if (nch > 0 && (stages & HDLA_STAGE_CHUNK_GRAD)) {
            e = launch_chunk_grad<T>(a, d->K, d->V, stream);
            if (e != hipSuccess) return (int)e;
        }
    }
    return HDLA_OK;
}

// The fused route's launch sequences.  Forward: fused kernel (+ fixup kernel when there are several segments).  When
// `boundary` is given it leaves the states entering the segments there, or, if there is room for it, the whole record.
// Backward: (without a record: summary pass, which writes one to the workspace; without the states: chaining) checkpoint
// kernel, reverse kernel, chunk_grad.
int run_fused(const hdla_dims* d, bool fwd, const void* q, const void* k, const void* v, const void* a_, const void* b,
              const void* beta, const void* gk, const float* h0, void* o, float* ht, const void* d_o, const float* dht,
              void* dq, void* dk, void* dv, void* da, void* db, void* dbeta, void* dgk, float* dh0, void* boundary,
              size_t boundary_bytes, void* workspace, size_t workspace_bytes, hipStream_t stream,
              int stages = HDLA_STAGE_ALL) {
    typedef bf16 T;
    FusedLayout L;
    int rc = make_fused_layout(d, fwd ? HDLA_PASS_FWD : HDLA_PASS_BWD, L);
    if (rc) return rc;
    const FusedRecord R = fused_record(d, L);
    char* const rec = boundary && boundary_bytes >= R.total ? static_cast<char*>(boundary) : nullptr;
    if (!fwd && rec) rc = make_fused_layout(d, PASS_BWD_RECORD, L);
    if (rc) return rc;
    if (bad_ws(workspace, workspace_bytes, L.total)) return HDLA_ERR_WORKSPACE;
    if (boundary && (L.nseg > 1) && (boundary_bytes < fused_boundary_bytes(d) || (reinterpret_cast<uintptr_t>(boundary) & 15)))
        return HDLA_ERR_WORKSPACE;
    if (rec && (reinterpret_cast<uintptr_t>(rec) & 15)) return HDLA_ERR_WORKSPACE;
    char* base = static_cast<char*>(workspace);
    FusedArgs<T> f{};
    ChunkArgs<T>& a = f.c;
    a.q = static_cast<const T*>(q); a.k = static_cast<const T*>(k); a.v = static_cast<const T*>(v);
    a.a = static_cast<const T*>(a_); a.b = static_cast<const T*>(b);
    a.gk = gk; a.gk_f32 = d->gk_dtype == HDLA_FP32;
    a.H = d->H; a.scale = d->scale;
    a.h0 = h0; a.ht = fwd ? ht : nullptr; a.o = static_cast<T*>(o);
    a.dout = static_cast<const T*>(d_o); a.dht = dht; a.dh0 = dh0;
    a.dq = static_cast<T*>(dq); a.dk = static_cast<T*>(dk); a.dv = static_cast<T*>(dv);
    a.da = static_cast<T*>(da); a.db = static_cast<T*>(db); a.dgk = dgk;
    a.beta = static_cast<const T*>(beta); a.dbeta = static_cast<T*>(dbeta);
    a.ws.HC = reinterpret_cast<T*>(base + L.HC); a.ws.DHC = reinterpret_cast<T*>(base + L.DHC);
    a.ws.DVN = reinterpret_cast<T*>(base + L.DVN);
    a.ws.UT = reinterpret_cast<T*>(base + L.UT); a.ws.W = reinterpret_cast<T*>(base + L.W);
    f.gw = reinterpret_cast<T*>(base + L.GW);
    if (rec) {
        a.ws.TM = reinterpret_cast<T*>(rec + R.TM); a.ws.STRONG = reinterpret_cast<int32_t*>(rec + R.STRONG);
        f.aq = reinterpret_cast<T*>(rec + R.AQ);
        if (L.nseg > 1) { f.mt = reinterpret_cast<float*>(rec + R.MT); f.gw = reinterpret_cast<T*>(rec + R.GW); }
    } else if (!fwd) {
        a.ws.TM = reinterpret_cast<T*>(base + L.TM); a.ws.STRONG = reinterpret_cast<int32_t*>(base + L.STRONG);
        f.aq = reinterpret_cast<T*>(base + L.AQ);
        f.mt = reinterpret_cast<float*>(base + L.MT);
    }
    a.ws.AAK = f.aq; a.ws.aak_stride = AAK_STRIDE_RECORD;          // (of the record's pairs, the first)
    a.ws.SUM = reinterpret_cast<float*>(base + L.SUM);
    a.ws.sa_stride = 2 * d->K * 16 * 2;                            // chunk_grad's view of w: [2][K/16] tiles per slot
    a.st.cu = d->cu_seqlens;
    a.st.chunk_off = d->cu_seqlens ? reinterpret_cast<const int32_t*>(base + L.CHUNK_OFF) : nullptr;
    a.st.chunk_seq = d->cu_seqlens ? reinterpret_cast<const int32_t*>(base + L.CHUNK_SEQ) : nullptr;
    a.st.order = d->cu_seqlens ? a.st.chunk_off + d->N + 1 : nullptr;
    a.st.T = d->T; a.st.NT = (d->T + CHUNK - 1) / CHUNK; a.st.N = d->N; a.st.nch = L.nch;
    f.nseg = L.nseg;
    f.sloc = reinterpret_cast<float*>(base + L.SLOC); f.mseg = reinterpret_cast<float*>(base + L.MSEG);
    f.rseg = reinterpret_cast<float*>(base + L.RSEG);
    f.err = reinterpret_cast<int*>(base + L.ERR);
    hipError_t e;
    if (d->cu_seqlens && (stages & HDLA_STAGE_PREP)) {
        e = launch_chunk_table(d->cu_seqlens, d->N, d->T, L.nch, d->H, 0, reinterpret_cast<int32_t*>(base + L.CHUNK_OFF),
                               reinterpret_cast<int32_t*>(base + L.CHUNK_SEQ), packed_outputs(d, a), stream);
        if (e != hipSuccess) return (int)e;
    }
    if (fwd) {
        f.ol = reinterpret_cast<float*>(base + L.OL);
        f.sin_out = static_cast<float*>(boundary);
        if (stages & HDLA_STAGE_SCAN_FWD) {
            e = launch_fused<T>(f, d->K, d->V, FUSED_FWD, stream);
            if (e != hipSuccess) return (int)e;
        }
        if (L.nseg > 1 && (stages & HDLA_STAGE_CHAIN)) {
            e = launch_fixup<T>(f, d->K, d->V, stream);
            if (e != hipSuccess) return (int)e;
        }
        return HDLA_OK;
    }
    f.sin = static_cast<const float*>(boundary);
    // no record: one pass over the inputs for it, and its segments chained into the states that enter them (a caller that
    // runs the stages one by one may leave this one out once the workspace holds them; one segment has no stage of its own
    // for it)
    if (!rec && (stages & (L.nseg > 1 ? HDLA_STAGE_CHAIN : HDLA_STAGE_SCAN_FWD))) {
        e = launch_fused<T>(f, d->K, d->V, FUSED_SUM, stream);
        if (e != hipSuccess) return (int)e;
    }
    if (L.nseg > 1 && !boundary) {
        f.sin_out = reinterpret_cast<float*>(base + L.SIN);
        if (stages & HDLA_STAGE_CHAIN) {
            e = launch_fixup<T>(f, d->K, d->V, stream);
            if (e != hipSuccess) return (int)e;
        }
        f.sin = f.sin_out;
    }
    if (stages & HDLA_STAGE_SCAN_FWD) {
        e = launch_fused<T>(f, d->K, d->V, FUSED_CKPT, stream);
        if (e != hipSuccess) return (int)e;
    }
    if (stages & HDLA_STAGE_SCAN_BWD) {
        e = launch_fused<T>(f, d->K, d->V, FUSED_REV, stream);
        if (e != hipSuccess) return (int)e;
    }
    if (L.nch > 0 && (stages & HDLA_STAGE_CHUNK_GRAD)) {
        e = launch_chunk_grad<T>(a, d->K, d->V, stream);
        if (e != hipSuccess) return (int)e;
    }
    return HDLA_OK;
}

}  // namespace

// ---- scratch memory of the entry point that allocates nothing ------------------------------------------------
// One array per GPU, part of the loaded code object, held until the process ends.  In host code the array's name is
// only a handle for hipGetSymbolAddress; the address kernels can use is looked up once per device and kept here.
// (No `used` attribute on the array: with it the compiler keeps the symbol local to the code object, where the runtime's
// lookup by name fails; the host-side reference below is what keeps the array and makes its symbol visible.)
static __device__ __align__(256) unsigned char scratch[HDLA_STATIC_WORKSPACE_BYTES];
static constexpr int MAX_DEVICES = 64;
static std::atomic<void*> g_scratch_ptr[MAX_DEVICES];

// Device address of `scratch` on the current device (looked up on the first call per device); nullptr and *err set
// on failure.  Two threads racing on the first call both obtain the same address.
static void* static_scratch(int* err) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) { *err = (int)e; return nullptr; }
    if (dev < 0 || dev >= MAX_DEVICES) { *err = HDLA_ERR_SHAPE; return nullptr; }
    void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (p) return p;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) { *err = e != hipSuccess ? (int)e : HDLA_ERR_WORKSPACE; return nullptr; }
    g_scratch_ptr[dev].store(p, std::memory_order_release);
    return p;
}

extern "C" {

int hdla_version(void) { return HDLA_VERSION; }

const char* hdla_strerror(int code) {
    switch (code) {
        case HDLA_OK: return "success";
        case HDLA_ERR_NULL: return "a required pointer is NULL";
        case HDLA_ERR_SHAPE: return "unsupported shape (need K,V in {64,128}, or 256 as well for the token-serial entry points; B,H,N >= 1, T >= 0, H,N <= 65535, chunks x heads < 2^31)";
        case HDLA_ERR_RANK: return "only rank R = 2 is supported";
        case HDLA_ERR_DTYPE: return "unsupported dtype (in_dtype bf16|fp32; gk fp32, or bf16 with bf16 inputs)";
        case HDLA_ERR_WORKSPACE: return "workspace is NULL, not 256-byte aligned, smaller than hdla_workspace_bytes(), or kept with another number of segments";
        case HDLA_ERR_ALIGN: return "tensor pointers must be 16-byte aligned";
        case HDLA_ERR_SEQ: return "cu_seqlens needs B == 1; without it N must equal B";
        case HDLA_ERR_ROUTE: return "route must be HDLA_ROUTE_AUTO, _CLASSIC, _PLAIN or _FUSED (the fused route: bf16 inputs, K = V = 64) and segments >= 0";
        case HDLA_ERR_STATIC_LIMIT: return "the call needs more scratch memory than the built-in HDLA_STATIC_WORKSPACE_BYTES; use hdla_chunk_fwd with a caller-owned workspace";
        default: return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown error code";
    }
}

size_t hdla_workspace_bytes(const hdla_dims* dims, int pass) {
    WsLayout L;
    int nch;
    if (pass < HDLA_PASS_FWD || pass > HDLA_PASS_BWD_KEPT) return 0;
    if (check_dims(dims)) return 0;
    bool fused;
    if (pick_route(dims, pass, true, fused)) return 0;
    size_t need = 0;
    if (fused && (pass == HDLA_PASS_FWD || pass == HDLA_PASS_BWD)) {
        FusedLayout F;
        if (make_fused_layout(dims, pass, F)) return 0;
        need = F.total;
        if (!few_short_sequences(dims, short_least(pass))) return need;   // (of these the call decides: enough for either)
    }
    if (make_layout(dims, pass, L, nch)) return 0;
    return std::max(need, L.total);
}

size_t hdla_boundary_bytes(const hdla_dims* dims) {
    bool fused;
    if (check_dims(dims) || pick_route(dims, HDLA_PASS_FWD, true, fused) || !fused) return 0;
    return fused_boundary_bytes(dims);
}

size_t hdla_record_bytes(const hdla_dims* dims) {
    bool fused;
    FusedLayout L;
    if (check_dims(dims) || pick_route(dims, HDLA_PASS_BWD, false, fused) || !fused || make_fused_layout(dims, HDLA_PASS_BWD, L)) return 0;
    return fused_record(dims, L).total;
}

size_t hdla_record_workspace_bytes(const hdla_dims* dims) {
    FusedLayout L;
    if (!hdla_record_bytes(dims)) return hdla_workspace_bytes(dims, HDLA_PASS_BWD);
    return make_fused_layout(dims, PASS_BWD_RECORD, L) ? 0 : L.total;
}

size_t hdla_keep_plan(const hdla_dims* dims, int32_t* fwd_segments, int32_t* bwd_segments) {
    bool fused_fwd, fused_bwd;
    if (!fwd_segments || !bwd_segments || check_dims(dims) || dims->T < 1) return 0;
    if (pick_route(dims, HDLA_PASS_FWD, false, fused_fwd) || pick_route(dims, HDLA_PASS_BWD, false, fused_bwd) || fused_fwd || fused_bwd) return 0;
    hdla_dims d = *dims;
    WsLayout L;
    int nch;
    d.segments = kept_plan_segments(dims, *bwd_segments);
    *fwd_segments = d.segments;
    if (make_layout(&d, HDLA_PASS_FWD_KEEP, L, nch) || L.total > KEEP_MOST) return 0;
    return L.total;
}

size_t hdla_states_plan(const hdla_dims* dims, size_t* fwd_workspace, size_t* bwd_workspace) {
    bool fused_fwd, fused_bwd;
    if (!fwd_workspace || !bwd_workspace || check_dims(dims) || dims->T < 1 || !leaves_states(dims)) return 0;
    if (pick_route(dims, HDLA_PASS_FWD, false, fused_fwd) || pick_route(dims, HDLA_PASS_BWD, false, fused_bwd) || fused_fwd || fused_bwd) return 0;
    WsLayout L, S;
    int nch;
    if (make_layout(dims, PASS_FWD_STATES, L, nch) || L.total > STATES_MOST || make_layout(dims, PASS_BWD_STATES, S, nch)) return 0;
    *fwd_workspace = states_fwd_workspace(dims, nch);
    *bwd_workspace = S.total;
    return L.total;
}

int hdla_workspace_layout(const hdla_dims* dims, int pass, hdla_ws_layout* out) {
    if (!out) return HDLA_ERR_NULL;
    if (pass < HDLA_PASS_FWD || pass > HDLA_PASS_BWD_KEPT) return HDLA_ERR_SHAPE;
    WsLayout L;
    int nch;
    int rc = check_dims(dims);
    if (rc) return rc;
    bool fused;
    rc = pick_route(dims, pass, false, fused);
    if (rc) return rc;
    if (fused && (pass == HDLA_PASS_FWD || pass == HDLA_PASS_BWD)) {
        FusedLayout F;
        rc = make_fused_layout(dims, pass, F);
        if (rc) return rc;
        *out = hdla_ws_layout{};
        out->nch = F.nch;
        out->UT = F.UT; out->TM = F.TM; out->HC = F.HC; out->DHC = F.DHC; out->DVN = F.DVN; out->STRONG = F.STRONG;
        out->W = F.W; out->SA_STRIDE = pass == HDLA_PASS_BWD ? 2 * dims->K * 16 * 2 : 0;
        out->CHUNK_OFF = F.CHUNK_OFF; out->CHUNK_SEQ = F.CHUNK_SEQ;
        out->total = F.total;
        out->ERR = F.ERR;
        if (pass == HDLA_PASS_BWD) { out->AAK = F.AQ; out->AAK_STRIDE = AAK_STRIDE_RECORD * 2; out->SUM = F.SUM; }
        return HDLA_OK;
    }
    rc = make_layout(dims, pass, L, nch);
    if (rc) return rc;
    out->nch = nch;
    out->W = L.W; out->UT = L.UT; out->KGT = L.KGT; out->BGT = L.BGT; out->VTT = L.VTT; out->EGL = L.EGL;
    out->QG = L.QG; out->AQK = L.AQK; out->AQB = L.AQB;
    out->AQBT = L.AQBT; out->QGT = L.QGT; out->TM = L.TM;
    out->SA_STRIDE = L.SA_STRIDE; out->SB_STRIDE = L.SB_STRIDE;
    out->HC = L.HC; out->DHC = L.DHC; out->DVN = L.DVN; out->STRONG = L.STRONG;
    out->CHUNK_OFF = L.CHUNK_OFF; out->CHUNK_SEQ = L.CHUNK_SEQ;
    out->total = L.total;
    out->ERR = -1;
    out->AAK = L.AAK; out->AAK_STRIDE = L.AAK ? AAK_STRIDE * 2 : 0; out->SUM = L.SUM;
    return HDLA_OK;
}

// forward pass of either form (a, b given, or beta) on the route the dimensions select
static int chunk_fwd_any(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a, const void* b,
                         const void* beta, const void* gk, const float* h0, void* o, float* ht, void* boundary,
                         size_t boundary_bytes, void* workspace, size_t workspace_bytes, void* stream) {
    int rc = check_dims(dims);
    if (rc) return rc;
    if (dims->T > 0 && (!q || !k || !v || !gk || !o || (!beta && (!a || !b)))) return HDLA_ERR_NULL;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(a) || !aligned16(b) || !aligned16(gk) ||
        !aligned16(o) || !aligned16(h0) || !aligned16(ht)) return HDLA_ERR_ALIGN;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (beta) { a = nullptr; b = nullptr; }
    bool fused;
    rc = pick_route(dims, HDLA_PASS_FWD, boundary != nullptr, fused);
    if (rc) return rc;
    if (fused)
        return run_fused(dims, true, q, k, v, a, b, beta, gk, h0, o, ht, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                         nullptr, nullptr, nullptr, nullptr, boundary, boundary_bytes, workspace, workspace_bytes, s);
    if (dims->in_dtype == HDLA_BF16)
        return run_chunk<bf16>(dims, 0, q, k, v, a, b, gk, h0, o, ht, nullptr, nullptr, nullptr, nullptr, nullptr,
                               nullptr, nullptr, nullptr, nullptr, workspace, workspace_bytes, s, HDLA_STAGE_ALL, beta, nullptr);
    return run_chunk<float>(dims, 0, q, k, v, a, b, gk, h0, o, ht, nullptr, nullptr, nullptr, nullptr, nullptr,
                            nullptr, nullptr, nullptr, nullptr, workspace, workspace_bytes, s, HDLA_STAGE_ALL, beta, nullptr);
}

static int chunk_bwd_any(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a, const void* b,
                         const void* beta, const void* gk, const float* h0, const void* d_o, const float* dht, void* dq,
                         void* dk, void* dv, void* da, void* db, void* dbeta, void* dgk, float* dh0, const void* boundary,
                         size_t boundary_bytes, void* workspace, size_t workspace_bytes, void* stream) {
    int rc = check_dims(dims);
    if (rc) return rc;
    if (dims->T > 0 && (!q || !k || !v || !gk || !d_o || !dq || !dk || !dv || !dgk)) return HDLA_ERR_NULL;
    if (dims->T > 0 && (beta ? !dbeta : (!a || !b || !da || !db))) return HDLA_ERR_NULL;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(a) || !aligned16(b) || !aligned16(gk) ||
        !aligned16(d_o) || !aligned16(dq) || !aligned16(dk) || !aligned16(dv) || !aligned16(da) || !aligned16(db) ||
        !aligned16(dgk) || !aligned16(h0) || !aligned16(dht) || !aligned16(dh0)) return HDLA_ERR_ALIGN;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (beta) { a = nullptr; b = nullptr; da = nullptr; db = nullptr; }
    bool fused;
    rc = pick_route(dims, HDLA_PASS_BWD, boundary != nullptr, fused);
    if (rc) return rc;
    if (fused)
        return run_fused(dims, false, q, k, v, a, b, beta, gk, h0, nullptr, nullptr, d_o, dht, dq, dk, dv, da, db, dbeta, dgk,
                         dh0, const_cast<void*>(boundary), boundary_bytes, workspace, workspace_bytes, s);
    if (dims->in_dtype == HDLA_BF16)
        return run_chunk<bf16>(dims, 1, q, k, v, a, b, gk, h0, nullptr, nullptr, d_o, dht, dq, dk, dv, da, db, dgk,
                               dh0, workspace, workspace_bytes, s, HDLA_STAGE_ALL, beta, dbeta);
    return run_chunk<float>(dims, 1, q, k, v, a, b, gk, h0, nullptr, nullptr, d_o, dht, dq, dk, dv, da, db, dgk,
                            dh0, workspace, workspace_bytes, s, HDLA_STAGE_ALL, beta, dbeta);
}

int hdla_chunk_fwd(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a,
                   const void* b, const void* gk, const float* h0, void* o, float* ht,
                   void* workspace, size_t workspace_bytes, void* stream) {
    if (dims && dims->T > 0 && (!a || !b)) return HDLA_ERR_NULL;
    return chunk_fwd_any(dims, q, k, v, a, b, nullptr, gk, h0, o, ht, nullptr, 0, workspace, workspace_bytes, stream);
}

int hdla_chunk_fwd_static(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a,
                          const void* b, const void* gk, const float* h0, void* o, float* ht, void* stream) {
    size_t need = hdla_workspace_bytes(dims, 0);
    if (need == 0) { const int rc = check_dims(dims); return rc ? rc : HDLA_ERR_SHAPE; }
    // the records of the scans' segments are what a call can do without
    hdla_dims whole = *dims;
    if (need > (size_t)HDLA_STATIC_WORKSPACE_BYTES && dims->segments == 0 && !fused_shape(dims)) {
        whole.segments = 1;
        dims = &whole;
        need = hdla_workspace_bytes(dims, 0);
    }
    if (need > (size_t)HDLA_STATIC_WORKSPACE_BYTES) return HDLA_ERR_STATIC_LIMIT;
    int err = 0;
    void* ws = static_scratch(&err);
    if (!ws) return err;
    // every byte of the workspace that a kernel of the forward pass reads has been written by an earlier kernel of
    // the same call, so nothing has to be cleared between calls
    return hdla_chunk_fwd(dims, q, k, v, a, b, gk, h0, o, ht, ws, (size_t)HDLA_STATIC_WORKSPACE_BYTES, stream);
}

int hdla_chunk_bwd(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a,
                   const void* b, const void* gk, const float* h0, const void* d_o, const float* dht,
                   void* dq, void* dk, void* dv, void* da, void* db, void* dgk, float* dh0,
                   void* workspace, size_t workspace_bytes, void* stream) {
    return chunk_bwd_any(dims, q, k, v, a, b, nullptr, gk, h0, d_o, dht, dq, dk, dv, da, db, nullptr, dgk, dh0, nullptr, 0,
                         workspace, workspace_bytes, stream);
}

int hdla_param_chunk_fwd(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* beta,
                         const void* gk, const float* h0, void* o, float* ht,
                         void* workspace, size_t workspace_bytes, void* stream) {
    if (!beta) return HDLA_ERR_NULL;
    return chunk_fwd_any(dims, q, k, v, nullptr, nullptr, beta, gk, h0, o, ht, nullptr, 0, workspace, workspace_bytes, stream);
}

int hdla_param_chunk_bwd(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* beta,
                         const void* gk, const float* h0, const void* d_o, const float* dht,
                         void* dq, void* dk, void* dv, void* dbeta, void* dgk, float* dh0,
                         void* workspace, size_t workspace_bytes, void* stream) {
    if (!beta) return HDLA_ERR_NULL;
    return chunk_bwd_any(dims, q, k, v, nullptr, nullptr, beta, gk, h0, d_o, dht, dq, dk, dv, nullptr, nullptr, dbeta, dgk,
                         dh0, nullptr, 0, workspace, workspace_bytes, stream);
}

int hdla_chunk_fwd_b(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a, const void* b,
                     const void* beta, const void* gk, const float* h0, void* o, float* ht, void* boundary,
                     size_t boundary_bytes, void* workspace, size_t workspace_bytes, void* stream) {
    return chunk_fwd_any(dims, q, k, v, a, b, beta, gk, h0, o, ht, boundary, boundary_bytes, workspace, workspace_bytes, stream);
}

int hdla_chunk_bwd_b(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a, const void* b,
                     const void* beta, const void* gk, const float* h0, const void* d_o, const float* dht, void* dq,
                     void* dk, void* dv, void* da, void* db, void* dbeta, void* dgk, float* dh0, const void* boundary,
                     size_t boundary_bytes, void* workspace, size_t workspace_bytes, void* stream) {
    return chunk_bwd_any(dims, q, k, v, a, b, beta, gk, h0, d_o, dht, dq, dk, dv, da, db, dbeta, dgk, dh0, boundary,
                         boundary_bytes, workspace, workspace_bytes, stream);
}

// pass: HDLA_PASS_FWD_KEEP or PASS_FWD_STATES
static int chunk_fwd_kept(const hdla_dims* dims, int pass, const void* q, const void* k, const void* v, const void* a,
                          const void* b, const void* beta, const void* gk, const float* h0, void* o, float* ht,
                          void* kept, size_t kept_bytes, void* workspace, size_t workspace_bytes, void* stream) {
    if (dims->T > 0 && (!q || !k || !v || !gk || !o || (!beta && (!a || !b)))) return HDLA_ERR_NULL;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(a) || !aligned16(b) || !aligned16(gk) ||
        !aligned16(o) || !aligned16(h0) || !aligned16(ht)) return HDLA_ERR_ALIGN;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (beta) { a = nullptr; b = nullptr; }
    if (dims->in_dtype == HDLA_BF16)
        return run_chunk<bf16>(dims, pass, q, k, v, a, b, gk, h0, o, ht, nullptr, nullptr, nullptr, nullptr,
                               nullptr, nullptr, nullptr, nullptr, nullptr, workspace, workspace_bytes, s, HDLA_STAGE_ALL, beta, nullptr,
                               kept, kept_bytes);
    return run_chunk<float>(dims, pass, q, k, v, a, b, gk, h0, o, ht, nullptr, nullptr, nullptr, nullptr,
                            nullptr, nullptr, nullptr, nullptr, nullptr, workspace, workspace_bytes, s, HDLA_STAGE_ALL, beta, nullptr,
                            kept, kept_bytes);
}
int hdla_chunk_fwd_keep(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a,
                        const void* b, const void* beta, const void* gk, const float* h0, void* o, float* ht,
                        void* kept, size_t kept_bytes, void* stream) {
    const int rc = check_dims(dims);
    if (rc) return rc;
    return chunk_fwd_kept(dims, HDLA_PASS_FWD_KEEP, q, k, v, a, b, beta, gk, h0, o, ht, kept, kept_bytes, nullptr, 0, stream);
}
int hdla_chunk_fwd_states(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a, const void* b, const void* beta, const void* gk,
                          const float* h0, void* o, float* ht, void* kept, size_t kept_bytes, void* workspace, size_t workspace_bytes, void* stream) {
    const int rc = check_dims(dims);
    if (rc) return rc;
    if (!leaves_states(dims)) return HDLA_ERR_SHAPE;
    return chunk_fwd_kept(dims, PASS_FWD_STATES, q, k, v, a, b, beta, gk, h0, o, ht, kept, kept_bytes, workspace, workspace_bytes, stream);
}

static int chunk_bwd_kept(const hdla_dims* dims, int pass, const void* q, const void* k, const void* v, const void* a,
                          const void* b, const void* beta, const void* gk, const float* h0, const void* d_o,
                          const float* dht, void* dq, void* dk, void* dv, void* da, void* db, void* dbeta, void* dgk,
                          float* dh0, void* kept, size_t kept_bytes, void* workspace, size_t workspace_bytes,
                          void* stream) {
    if (dims->T > 0 && (!q || !k || !v || !gk || !d_o || !dq || !dk || !dv || !dgk)) return HDLA_ERR_NULL;
    if (dims->T > 0 && (beta ? !dbeta : (!a || !b || !da || !db))) return HDLA_ERR_NULL;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(a) || !aligned16(b) || !aligned16(gk) ||
        !aligned16(d_o) || !aligned16(dq) || !aligned16(dk) || !aligned16(dv) || !aligned16(da) || !aligned16(db) ||
        !aligned16(dgk) || !aligned16(h0) || !aligned16(dht) || !aligned16(dh0)) return HDLA_ERR_ALIGN;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (beta) { a = nullptr; b = nullptr; da = nullptr; db = nullptr; }
    if (dims->in_dtype == HDLA_BF16)
        return run_chunk<bf16>(dims, pass, q, k, v, a, b, gk, h0, nullptr, nullptr, d_o, dht, dq, dk, dv, da,
                               db, dgk, dh0, workspace, workspace_bytes, s, HDLA_STAGE_ALL, beta, dbeta, kept, kept_bytes);
    return run_chunk<float>(dims, pass, q, k, v, a, b, gk, h0, nullptr, nullptr, d_o, dht, dq, dk, dv, da,
                            db, dgk, dh0, workspace, workspace_bytes, s, HDLA_STAGE_ALL, beta, dbeta, kept, kept_bytes);
}
int hdla_chunk_bwd_kept(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a,
                        const void* b, const void* beta, const void* gk, const float* h0, const void* d_o,
                        const float* dht, void* dq, void* dk, void* dv, void* da, void* db, void* dbeta, void* dgk,
                        float* dh0, void* kept, size_t kept_bytes, void* workspace, size_t workspace_bytes,
                        void* stream) {
    const int rc = check_dims(dims);
    if (rc) return rc;
    return chunk_bwd_kept(dims, HDLA_PASS_BWD_KEPT, q, k, v, a, b, beta, gk, h0, d_o, dht, dq, dk, dv, da, db, dbeta, dgk, dh0, kept, kept_bytes, workspace,
                          workspace_bytes, stream);
}
int hdla_chunk_bwd_states(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a, const void* b, const void* beta, const void* gk,
                          const float* h0, const void* d_o, const float* dht, void* dq, void* dk, void* dv, void* da, void* db, void* dbeta, void* dgk, float* dh0,
                          void* kept, size_t kept_bytes, void* workspace, size_t workspace_bytes, void* stream) {
    const int rc = check_dims(dims);
    if (rc) return rc;
    if (!leaves_states(dims)) return HDLA_ERR_SHAPE;
    return chunk_bwd_kept(dims, PASS_BWD_STATES, q, k, v, a, b, beta, gk, h0, d_o, dht, dq, dk, dv, da, db, dbeta, dgk, dh0, kept, kept_bytes, workspace,
                          workspace_bytes, stream);
}

int hdla_chunk_stages(const hdla_dims* dims, int pass, int stages, const void* q, const void* k, const void* v,
                      const void* a, const void* b, const void* gk, const float* h0, void* o, float* ht,
                      const void* d_o, const float* dht, void* dq, void* dk, void* dv, void* da, void* db, void* dgk,
                      float* dh0, void* workspace, size_t workspace_bytes, void* stream) {
    const int rc = check_dims(dims);
    if (rc) return rc;
    if (pass != 0 && pass != 1) return HDLA_ERR_SHAPE;
    if (!q || !k || !v || !a || !b || !gk) return HDLA_ERR_NULL;
    if (pass == 0 ? !o : (!d_o || !dq || !dk || !dv || !da || !db || !dgk)) return HDLA_ERR_NULL;
    hipStream_t s = static_cast<hipStream_t>(stream);
    bool fused;
    const int rr = pick_route(dims, pass, false, fused);
    if (rr) return rr;
    if (fused)
        return run_fused(dims, pass == 0, q, k, v, a, b, nullptr, gk, h0, o, ht, d_o, dht, dq, dk, dv, da, db, nullptr, dgk, dh0,
                         nullptr, 0, workspace, workspace_bytes, s, stages);
    if (dims->in_dtype == HDLA_BF16)
        return run_chunk<bf16>(dims, pass, q, k, v, a, b, gk, h0, o, ht, d_o, dht, dq, dk, dv, da, db, dgk, dh0,
                               workspace, workspace_bytes, s, stages);
    return run_chunk<float>(dims, pass, q, k, v, a, b, gk, h0, o, ht, d_o, dht, dq, dk, dv, da, db, dgk, dh0,
                            workspace, workspace_bytes, s, stages);
}

static int run_recurrent(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a,
                         const void* b, const void* beta, const void* gk, int reverse, const float* h0, void* o,
                         float* ht, void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e;
    if (dims->in_dtype == HDLA_BF16) {
        RecurrentArgs<bf16> r{};
        r.q = static_cast<const bf16*>(q); r.k = static_cast<const bf16*>(k); r.v = static_cast<const bf16*>(v);
        r.a = static_cast<const bf16*>(a); r.b = static_cast<const bf16*>(b);
        r.beta = static_cast<const bf16*>(beta);
        r.gk = gk; r.gk_f32 = dims->gk_dtype == HDLA_FP32;
        r.H = dims->H; r.T_ = dims->T; r.N = dims->N; r.scale = dims->scale; r.reverse = reverse;
        r.cu = dims->cu_seqlens; r.h0 = h0; r.ht = ht; r.o = static_cast<bf16*>(o);
        e = launch_recurrent<bf16>(r, dims->K, dims->V, s);
    } else {
        RecurrentArgs<float> r{};
        r.q = static_cast<const float*>(q); r.k = static_cast<const float*>(k); r.v = static_cast<const float*>(v);
        r.a = static_cast<const float*>(a); r.b = static_cast<const float*>(b);
        r.beta = static_cast<const float*>(beta);
        r.gk = gk; r.gk_f32 = 1;
        r.H = dims->H; r.T_ = dims->T; r.N = dims->N; r.scale = dims->scale; r.reverse = reverse;
        r.cu = dims->cu_seqlens; r.h0 = h0; r.ht = ht; r.o = static_cast<float*>(o);
        e = launch_recurrent<float>(r, dims->K, dims->V, s);
    }
    return e == hipSuccess ? HDLA_OK : (int)e;
}

int hdla_recurrent_fwd(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a,
                       const void* b, const void* gk, int reverse, const float* h0, void* o, float* ht,
                       void* stream) {
    const int rc = check_dims(dims, 256);
    if (rc) return rc;
    if (dims->T > 0 && (!q || !k || !v || !a || !b || !gk || !o)) return HDLA_ERR_NULL;
    if (!aligned16(h0) || !aligned16(ht)) return HDLA_ERR_ALIGN;
    return run_recurrent(dims, q, k, v, a, b, nullptr, gk, reverse, h0, o, ht, stream);
}

int hdla_param_recurrent_fwd(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* beta,
                             const void* gk, int reverse, const float* h0, void* o, float* ht, void* stream) {
    const int rc = check_dims(dims, 256);
    if (rc) return rc;
    if (!beta) return HDLA_ERR_NULL;
    if (dims->T > 0 && (!q || !k || !v || !gk || !o)) return HDLA_ERR_NULL;
    if (!aligned16(h0) || !aligned16(ht)) return HDLA_ERR_ALIGN;
    return run_recurrent(dims, q, k, v, nullptr, nullptr, beta, gk, reverse, h0, o, ht, stream);
}

}  // extern "C"
