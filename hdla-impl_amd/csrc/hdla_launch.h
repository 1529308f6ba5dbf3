// Host-callable launchers of the HIP kernels (one per device stage); defined in the .hip files, used by api.hip.
#pragma once
#include <hip/hip_runtime.h>

#include "hdla_ws.h"

namespace hdla {

// Outputs of a call on a packed batch.  The kernels write the rows of the sequences; a table that is not a partition of the
// tokens (it may come unchecked from the device) leaves rows that belong to none, and these are to read as zeros.
struct PackedOut {
    void* p[7];
    long long row[7];         // bytes a token, multiples of 2
    int n;
    void add(void* q, long long b) { if (q) { p[n] = q; row[n++] = b; } }
};
// (V: where a scan on the table is shared out by the sequences' lengths (scan_shares); else 0, and `order` holds no widths)
hipError_t launch_chunk_table(const int64_t* cu, int N, int T, int nch, int H, int V, int32_t* chunk_off, int32_t* chunk_seq,
                              const PackedOut& out, hipStream_t stream);
// only what clears the rows that belong to no sequence
hipError_t launch_clear_uncovered(const int64_t* cu, int N, int T, const PackedOut& out, hipStream_t stream);

// K, V in {64, 128}; returns hipErrorInvalidValue for any other pair.
// mode: 0 = for the forward pass, 1 = for the backward pass, 2 = forward pass whose workspace the backward pass will use, 3 = the same with the
// states that enter the chunks in it (2-byte elements)
// out: with it the launch leaves the chunk table too and does launch_chunk_table's other work (prep_makes_table says whether it can); share_V as V there
inline bool prep_makes_table(const int64_t* cu, int N, int H, int nch) { return cu && N <= 64 /* FEW_SEQS */ && nch > 0 && (long long)H * nch < 0x7ffff000LL; }
template <typename T> hipError_t launch_prep(const ChunkArgs<T>& a, int K, int V, int mode, const PackedOut* out, int share_V, hipStream_t stream);
// the two scans of the backward pass
template <typename T> hipError_t launch_scan_fwd(const ChunkArgs<T>& a, int K, int V, hipStream_t stream);
// the scan of the forward pass, with the output (kept: 0 after launch_prep of mode 0, 1 of mode 2, 2 of mode 3)
template <typename T> hipError_t launch_scan_out(const ChunkArgs<T>& a, int K, int V, int kept, hipStream_t stream);
template <typename T> hipError_t launch_scan_bwd(const ChunkArgs<T>& a, int K, int V, hipStream_t stream);
// both in one launch
template <typename T> hipError_t launch_scan_pair(const ChunkArgs<T>& a, int K, int V, hipStream_t stream);
// several time segments per sequence: what the scans above start their segments from
enum SegStart {
    SEG_FWD,          // of launch_scan_out, after launch_prep of mode 0
    SEG_FWD_KEPT,     // the same after mode 2
    SEG_BWD,          // of the two scans of the backward pass, after mode 1 (with seg.turned: rtr as SEG_FWD_KEPT leaves it)
    SEG_BWD_KEPT      // the reverse scan's alone, on the states and transitions that SEG_FWD_KEPT left
};
template <typename T> hipError_t launch_scan_segments(const ChunkArgs<T>& a, int K, int V, SegStart what, hipStream_t stream);
template <typename T> hipError_t launch_chunk_grad(const ChunkArgs<T>& a, int K, int V, hipStream_t stream);
template <typename T> hipError_t launch_recurrent(const RecurrentArgs<T>& a, int K, int V, hipStream_t stream);

}  // namespace hdla
