// Host-side dispatch of the scan kernels by head shape (kernels: scan_out.cuh and scan_grad.cuh, fp32 scan_impl.cuh; compiled in scan_*.hip).
#include "scan_shapes.h"

namespace hdla {

template <typename T>
static hipError_t launch_scan(const ChunkArgs<T>& a, int K, int V, ScanKind kind, hipStream_t stream) {
    if constexpr (sizeof(T) == 2) {
        if (K == 64 && V == 64) return launch_scan_grad_shape<64, 64>(a, kind, stream);
        if (K == 128 && V == 128) return launch_scan_grad_shape<128, 128>(a, kind, stream);
        if (K == 64 && V == 128) return launch_scan_grad_shape<64, 128>(a, kind, stream);
        if (K == 128 && V == 64) return launch_scan_grad_shape<128, 64>(a, kind, stream);
        return hipErrorInvalidValue;
    } else {
        if (K == 64 && V == 64) return launch_scan_shape<T, 64, 64>(a, kind, stream);
        if (K == 128 && V == 128) return launch_scan_shape<T, 128, 128>(a, kind, stream);
        if (K == 64 && V == 128) return launch_scan_shape<T, 64, 128>(a, kind, stream);
        if (K == 128 && V == 64) return launch_scan_shape<T, 128, 64>(a, kind, stream);
        return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t launch_scan_fwd(const ChunkArgs<T>& a, int K, int V, hipStream_t stream) {
    return launch_scan<T>(a, K, V, SCAN_FWD, stream);
}
template <typename T>
hipError_t launch_scan_out(const ChunkArgs<T>& a, int K, int V, int kept, hipStream_t stream) {
    if constexpr (sizeof(T) == 2) {
        if (K == 64 && V == 64) return launch_scan_out_shape<64, 64>(a, kept, stream);
        if (K == 128 && V == 128) return launch_scan_out_shape<128, 128>(a, kept, stream);
        if (K == 64 && V == 128) return launch_scan_out_shape<64, 128>(a, kept, stream);
        if (K == 128 && V == 64) return launch_scan_out_shape<128, 64>(a, kept, stream);
        return hipErrorInvalidValue;
    }
    return launch_scan<T>(a, K, V, SCAN_FWD_O, stream);
}
template <typename T>
hipError_t launch_scan_bwd(const ChunkArgs<T>& a, int K, int V, hipStream_t stream) {
    return launch_scan<T>(a, K, V, SCAN_BWD, stream);
}
template <typename T>
hipError_t launch_scan_pair(const ChunkArgs<T>& a, int K, int V, hipStream_t stream) {
    return launch_scan<T>(a, K, V, SCAN_PAIR, stream);
}
template <typename T>
hipError_t launch_scan_segments(const ChunkArgs<T>& a, int K, int V, SegStart what, hipStream_t stream) {
    if constexpr (sizeof(T) == 2) {
        if (K == 64 && V == 64) return what == SEG_FWD ? launch_scan_out_segments_shape<64, 64>(a, stream) : launch_scan_grad_segments_shape<64, 64>(a, what, stream);
        if (K == 128 && V == 128) return what == SEG_FWD ? launch_scan_out_segments_shape<128, 128>(a, stream) : launch_scan_grad_segments_shape<128, 128>(a, what, stream);
        if (K == 64 && V == 128) return what == SEG_FWD ? launch_scan_out_segments_shape<64, 128>(a, stream) : launch_scan_grad_segments_shape<64, 128>(a, what, stream);
        if (K == 128 && V == 64) return what == SEG_FWD ? launch_scan_out_segments_shape<128, 64>(a, stream) : launch_scan_grad_segments_shape<128, 64>(a, what, stream);
        return hipErrorInvalidValue;
    } else {
        if (K == 64 && V == 64) return launch_scan_segments_shape<T, 64, 64>(a, what, stream);
        if (K == 128 && V == 128) return launch_scan_segments_shape<T, 128, 128>(a, what, stream);
        if (K == 64 && V == 128) return launch_scan_segments_shape<T, 64, 128>(a, what, stream);
        if (K == 128 && V == 64) return launch_scan_segments_shape<T, 128, 64>(a, what, stream);
        return hipErrorInvalidValue;
    }
}
template hipError_t launch_scan_segments<bf16>(const ChunkArgs<bf16>&, int, int, SegStart, hipStream_t);
template hipError_t launch_scan_segments<float>(const ChunkArgs<float>&, int, int, SegStart, hipStream_t);
template hipError_t launch_scan_fwd<bf16>(const ChunkArgs<bf16>&, int, int, hipStream_t);
template hipError_t launch_scan_fwd<float>(const ChunkArgs<float>&, int, int, hipStream_t);
template hipError_t launch_scan_out<bf16>(const ChunkArgs<bf16>&, int, int, int, hipStream_t);
template hipError_t launch_scan_out<float>(const ChunkArgs<float>&, int, int, int, hipStream_t);
template hipError_t launch_scan_bwd<bf16>(const ChunkArgs<bf16>&, int, int, hipStream_t);
template hipError_t launch_scan_bwd<float>(const ChunkArgs<float>&, int, int, hipStream_t);
template hipError_t launch_scan_pair<bf16>(const ChunkArgs<bf16>&, int, int, hipStream_t);
template hipError_t launch_scan_pair<float>(const ChunkArgs<float>&, int, int, hipStream_t);

}  // namespace hdla
