// Small tables of the host (row offsets of the experts, lists of problems) to device memory, through a kernel's arguments.
//
// A copy from pageable host memory waits for everything in front of it on the stream, and the host with it: a grouped linear
// layer whose offsets went that way left the GPU idle for 25 - 40 us in front of its GEMM.  A kernel's arguments are taken
// when the launch is queued, so the caller's array may go as soon as the call returns, and nothing waits.
#include "lowp_device.h"

namespace {

// at most 4 KB of arguments per launch
constexpr int kWords = 960;
struct Words { int32_t v[kWords]; };

__global__ __launch_bounds__(256) void words_to_device(Words w, int n, int32_t *__restrict__ out)
{
    for (int i = threadIdx.x; i < n; i += 256) out[i] = w.v[i];
}

}  // namespace

extern "C" int lp_host_table(const int32_t *src, int64_t n, int32_t *dst, lp_stream_t stream)
{
    LP_REQUIRE(n >= 0, "lp_host_table: negative length");
    if (n == 0) return LP_OK;
    LP_REQUIRE(src && dst, "lp_host_table: null pointer");
    for (int64_t i = 0; i < n; i += kWords) {
        Words w;
        const int part = (int)(n - i < kWords ? n - i : kWords);
        for (int k = 0; k < part; ++k) w.v[k] = src[i + k];
        for (int k = part; k < kWords; ++k) w.v[k] = 0;
        hipLaunchKernelGGL(words_to_device, dim3(1), dim3(256), 0, (hipStream_t)stream, w, part, dst + i);
    }
    return lowp::check_launch("lp_host_table");
}

namespace {

__global__ void raise_flag(int32_t *flag) { __hip_atomic_store(flag, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM); }

}  // namespace

extern "C" int lp_host_flag(int32_t *flag, lp_stream_t stream)
{
    LP_REQUIRE(flag, "lp_host_flag: null pointer");
    hipLaunchKernelGGL(raise_flag, dim3(1), dim3(1), 0, (hipStream_t)stream, flag);
    return lowp::check_launch("lp_host_flag");
}
