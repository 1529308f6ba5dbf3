// Entry points of libhdla_hip.so that native.cpp calls beside those of include/hdla_hip.h.  Both are built together: they are no part of the C ABI and of
// its version number.
#pragma once
#include "../../include/hdla_hip.h"

extern "C" {
// A training call that leaves its backward pass, beside what hdla_chunk_fwd_keep leaves, the states that enter the chunks: that pass runs the reverse
// scan alone.  hdla_states_plan: bytes of the buffer to hold between the passes, 0 where it does not pay or is too large (a gibibyte; whether a call takes it, native.cpp says); fwd_workspace, bwd_workspace: bytes of scratch of the
// two calls.  One segment in both passes; the results, and those of a backward pass without the buffer (HDLA_ROUTE_PLAIN), are the same bits.
size_t hdla_states_plan(const hdla_dims* dims, size_t* fwd_workspace, size_t* bwd_workspace);
int hdla_chunk_fwd_states(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a, const void* b, const void* beta, const void* gk,
                          const float* h0, void* o, float* ht, void* kept, size_t kept_bytes, void* workspace, size_t workspace_bytes, void* stream);
int hdla_chunk_bwd_states(const hdla_dims* dims, const void* q, const void* k, const void* v, const void* a, const void* b, const void* beta, const void* gk,
                          const float* h0, const void* d_o, const float* dht, void* dq, void* dk, void* dv, void* da, void* db, void* dbeta, void* dgk, float* dh0,
                          void* kept, size_t kept_bytes, void* workspace, size_t workspace_bytes, void* stream);
// hdla_layer_pre_bwd into a dy whose rows are lddy elements (ldy at the least, whole 16 bytes): its padding reaches there.
int hdla_layer_pre_bwd_to(const hdla_pre_dims* dims, const void* y, const void* dq, const void* dk, const void* dv, const void* dbeta, void* dy, int32_t lddy, void* stream);
// y [M, N] = x [M, K] W, W [N, K] taken turned or (turned) [K, N] as it is; bf16, sums in 32 bits.  N and K in eights (turned: N in 64s), rows 16 bytes aligned.
int hdla_tile_gemm(int32_t M, int32_t N, int32_t K, const void* x, int64_t ldx, const void* w, int64_t ldw, int32_t turned, void* y, int64_t ldy, void* stream);
}
