// Small tables of the host (row offsets of the experts, lists of problems) to device memory, through a kernel's arguments, and
// the results of listed problems that have nothing to compute.
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

// Bound by the write of the slots; a workgroup clears 16 KB.  One launch for all of them: a fill per slot took the host 5 us
// each (a weight gradient with 32 of 64 experts empty, 2048 x 2048 each: 326 us a call with a fill per slot, 175 so; 224 of
// 256, 1408 x 2048: 1271 / 357).
constexpr int kClear = 256 * 16 * 4;

__global__ __launch_bounds__(256) void zero_slots(char *__restrict__ C, int64_t slot_bytes, int64_t total, const int32_t *__restrict__ slots, int per)
{
    const int64_t slot = slots[blockIdx.x / per];
    if (slot < 0 || slot >= total) return;
    const int64_t first = (int64_t)(blockIdx.x % per) * kClear + threadIdx.x * 16;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (first + i * 4096 < slot_bytes) __builtin_nontemporal_store(lowp::u32x4{0, 0, 0, 0}, (lowp::u32x4 *)(C + slot * slot_bytes + first + i * 4096));
}

}  // namespace

extern "C" int lp_zero_slots(void *C, int64_t slot_bytes, int64_t total, const int32_t *slots, int n, lp_stream_t stream)
{
    LP_REQUIRE(slot_bytes >= 0 && slot_bytes % 16 == 0 && total >= 0 && n >= 0, "lp_zero_slots: bad size");
    if (n == 0 || slot_bytes == 0) return LP_OK;
    LP_REQUIRE(C && slots, "lp_zero_slots: null pointer");
    const int64_t per = (slot_bytes + kClear - 1) / kClear;
    LP_REQUIRE(per <= 0x7FFFFFFF, "lp_zero_slots: slot too large");
    const int most = (int)(0x7FFFFFFF / per);              // slots a launch's grid holds
    for (int i = 0; i < n; i += most) {
        const int part = n - i < most ? n - i : most;
        hipLaunchKernelGGL(zero_slots, dim3((unsigned)(part * per)), dim3(256), 0, (hipStream_t)stream, (char *)C, slot_bytes, total, slots + i, (int)per);
        if (n - i <= most) break;
    }
    return lowp::check_launch("lp_zero_slots");
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
