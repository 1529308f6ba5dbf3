// Several sums over partial results in one launch.  Each of them is a few workgroups' round trip to memory, 5 to 6 us as a launch of its own.
// What bounds it: reading the partial results (25 MB for the first of these) behind one latency; the loads of eight at a time are on their way together.  The
// three sums of a training step of the layer (16 tiles in 16 shares, two low-rank weight gradients, the norm's weight) 5.4 + 5.0 + 6.2 -> 9.8 us; the step,
// 4 x 2048 tokens, d = 1024 670 -> 667, 4 x 1024 405 -> 399, 4 x 2048, d = 512 382 -> 376.
#include "sums.cuh"

#include <cstring>

namespace hdla {

constexpr int SUMS_MOST = 8;
struct SumJobs { SumJob job[SUMS_MOST]; int end[SUMS_MOST]; };     // end: of each job's workgroups
__global__ __launch_bounds__(256) void sums_kernel(SumJobs p) {
    int at = 0, block = (int)blockIdx.x;
#pragma unroll
    for (int i = 0; i < SUMS_MOST - 1; ++i)
        if ((int)blockIdx.x >= p.end[i]) { at = i + 1; block = (int)blockIdx.x - p.end[i]; }
    const SumJob& j = p.job[at];
    if (j.kind == SUM_PARTS) sum_parts(j, block);
    else if (j.kind == SUM_ROWS) sum_rows_of_groups(j.part, j.out[0], j.f32, j.n, j.G, j.E, block);
    else if (j.kind == SUM_TILES) sum_tiles(j, block);
}

static int run_sums(const SumJob* jobs, int count, hipStream_t stream) {
    SumJobs p{};
    int used = 0, blocks = 0;
    for (int i = 0; i < count; ++i) {
        if (jobs[i].kind == SUM_NONE || jobs[i].blocks == 0) continue;
        p.job[used] = jobs[i];
        p.end[used++] = blocks += jobs[i].blocks;
    }
    for (int i = used; i < SUMS_MOST; ++i) p.end[i] = blocks;
    if (!blocks) return HDLA_OK;
    hipLaunchKernelGGL(sums_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, p);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? HDLA_OK : (int)e;
}

int sum_now_or_later(const SumJob& job, hdla_sum* later, hipStream_t stream) {
    if (!later) return run_sums(&job, 1, stream);
    std::memset(later, 0, sizeof(*later));
    std::memcpy(later, &job, sizeof(job));
    return HDLA_OK;
}

}  // namespace hdla

using namespace hdla;

extern "C" int hdla_run_sums(const hdla_sum* sums, int32_t count, void* stream) {
    if (count < 0 || count > SUMS_MOST) return HDLA_ERR_SHAPE;
    if (count && !sums) return HDLA_ERR_NULL;
    SumJob jobs[SUMS_MOST];
    long long blocks = 0;
    for (int i = 0; i < count; ++i) {
        std::memcpy(&jobs[i], &sums[i], sizeof(SumJob));
        if (jobs[i].kind < SUM_NONE || jobs[i].kind > SUM_TILES || jobs[i].blocks < 0) return HDLA_ERR_SHAPE;
        blocks += jobs[i].blocks;
    }
    if (blocks > 0x7fffffffLL) return HDLA_ERR_SHAPE;
    return run_sums(jobs, count, static_cast<hipStream_t>(stream));
}
