// Argument block and host entry points of the fused chunk kernels (fused_impl.cuh); each mode is compiled in its own
// translation unit (fused_*.hip) so that the build can run them in parallel.
#pragma once
#include "hdla_launch.h"

namespace hdla {

// FUSED_FWD: forward pass (o, or o_local and G for segments > 0; segment records; with ws.TM set: the record for the backward
// pass).  FUSED_SUM: the same without the outputs (what a backward pass runs first when the forward pass left no record).
// FUSED_CKPT: the backward pass's forward half: state checkpoints, u and w where chunk_grad reads them, R of the segments.
// FUSED_REV: the reverse scan of the state gradient: dS checkpoints, dv_new, dh0.
enum FusedMode { FUSED_FWD = 0, FUSED_SUM = 1, FUSED_CKPT = 2, FUSED_REV = 3 };

template <typename T>
struct FusedArgs {
    ChunkArgs<T> c;
    int nseg;              // time segments per sequence
    // records per (sequence, head, segment), fp32 tiles in fragment order (see fused_impl.cuh)
    float* sloc;           // [N][H][nseg][K*V]
    float* mseg;           // [N][H][nseg][K*K]
    float* rseg;           // [N][H][nseg][K*V]
    const float* sin;      // [N][H][nseg][K*V]  states entering the segments (read by FUSED_CKPT)
    float* sin_out;        // the same record, written by fixup_kernel (nullable)
    float* ol;             // [H][nch][V/16] fp32 tiles  local outputs of segments > 0 (forward pass); null: fixup_kernel only chains
    // the record (with c.ws.TM and c.ws.STRONG): written by FUSED_FWD and FUSED_SUM, read by FUSED_CKPT and FUSED_REV
    float* mt;             // [N][H][nseg][K*K]     transposed transitions of segments > 0 (nullable)
    T* gw;                 // [H][nch][K/8][16][8]  G of segments > 0 (the forward pass's fixup_kernel needs it as well)
    T* aq;                 // [H][nch][2][2 tiles]  A_ak, A_qb
    int* err;              // set nonzero by a wave whose bounded wait ran out
};

// K = V = 64, 2-byte elements only; hipErrorInvalidValue otherwise
template <typename T> hipError_t launch_fused(const FusedArgs<T>& a, int K, int V, int mode, hipStream_t stream);
template <typename T> hipError_t launch_fixup(const FusedArgs<T>& a, int K, int V, hipStream_t stream);

// per-mode instantiations
template <typename T, int MODE> hipError_t launch_fused_mode(const FusedArgs<T>& a, hipStream_t stream);

}  // namespace hdla
