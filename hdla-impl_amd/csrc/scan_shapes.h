// Entry points of the scan kernels per element type and head shape; each shape is compiled in its own
// translation unit (scan_*.hip) so that the build can run them in parallel.
#pragma once
#include "hdla_launch.h"

namespace hdla {

enum ScanKind { SCAN_FWD_O, SCAN_FWD, SCAN_BWD, SCAN_PAIR };   // forward scan with / without the output, reverse, both

template <typename T, int K, int V> hipError_t launch_scan_shape(const ChunkArgs<T>& a, ScanKind kind, hipStream_t stream);
// the forward pass's scan for 2-byte elements, and its segments' records and entering states (scan_out.cuh)
template <int K, int V> hipError_t launch_scan_out_shape(const ChunkArgs<bf16>& a, int kept, hipStream_t stream);
template <int K, int V> hipError_t launch_scan_out_segments_shape(const ChunkArgs<bf16>& a, hipStream_t stream);   // SEG_FWD
// the scans of the backward pass for 2-byte elements, and their segments' (scan_grad.cuh)
template <int K, int V> hipError_t launch_scan_grad_shape(const ChunkArgs<bf16>& a, ScanKind kind, hipStream_t stream);
template <int K, int V> hipError_t launch_scan_grad_segments_shape(const ChunkArgs<bf16>& a, SegStart what, hipStream_t stream);   // the others
// several time segments: the segments' records, then the states and state gradients that enter them
template <typename T, int K, int V> hipError_t launch_scan_segments_shape(const ChunkArgs<T>& a, SegStart what, hipStream_t stream);

}  // namespace hdla
