// Scan kernels, bf16 inputs, head sizes K=64 V=64, K=64 V=128 (see scan_out.cuh, scan_grad.cuh).
#include "scan_grad.cuh"

namespace hdla {
template hipError_t launch_scan_out_shape<64, 64>(const ChunkArgs<bf16>&, int, hipStream_t);
template hipError_t launch_scan_out_segments_shape<64, 64>(const ChunkArgs<bf16>&, hipStream_t);
template hipError_t launch_scan_grad_shape<64, 64>(const ChunkArgs<bf16>&, ScanKind, hipStream_t);
template hipError_t launch_scan_grad_segments_shape<64, 64>(const ChunkArgs<bf16>&, SegStart, hipStream_t);
template hipError_t launch_scan_out_shape<64, 128>(const ChunkArgs<bf16>&, int, hipStream_t);
template hipError_t launch_scan_out_segments_shape<64, 128>(const ChunkArgs<bf16>&, hipStream_t);
template hipError_t launch_scan_grad_shape<64, 128>(const ChunkArgs<bf16>&, ScanKind, hipStream_t);
template hipError_t launch_scan_grad_segments_shape<64, 128>(const ChunkArgs<bf16>&, SegStart, hipStream_t);
}  // namespace hdla
