// math_check.hip -- the render kernels' reciprocal, root and pack against their plain forms, over ranges of bit
// patterns (ptgpu_check_math).  Every image's bits rest on their being equal.
#include "render_device.hpp"

namespace ptgpu {

// A wave takes 64 patterns in a row, so its fast forms run where all of them are in range, as in a render.
template <int WHICH>
__global__ __launch_bounds__(256) void k_check_math(unsigned first, unsigned long long count, const float *tab,
                                                    unsigned long long *wrong) {
    __shared__ float s_tab[kPackEntries];
    for (int i = threadIdx.x; i < kPackEntries; i += blockDim.x) s_tab[i] = tab[i];
    __syncthreads();
    unsigned bad = 0;
    for (unsigned long long i = (unsigned long long)blockIdx.x * 256 + threadIdx.x; i < count;
         i += (unsigned long long)gridDim.x * 256) {
        const float x = __uint_as_float(first + (unsigned)i);
        if (WHICH == PTGPU_CHECK_PACK) {
            bad += to_int_tab(x, s_tab) != to_int(x);
        } else {
            const float a = WHICH == PTGPU_CHECK_RCP ? rcp_exact(x) : sqrt_exact(x);
            const float b = WHICH == PTGPU_CHECK_RCP ? 1.0f / x : sqrtf(x);
            bad += __float_as_uint(a) != __float_as_uint(b) && !(a != a && b != b);
        }
    }
    if (bad) atomicAdd(wrong, (unsigned long long)bad);
}

}  // namespace ptgpu

extern "C" int ptgpu_check_math(ptgpu_ctx *ctx, int which, unsigned first, unsigned long long count,
                                unsigned long long *wrong) {
    using namespace ptgpu;
    PT_CHECK(ctx && wrong, PTGPU_ERR_INVALID, "null argument");
    PT_CHECK(which >= PTGPU_CHECK_RCP && which <= PTGPU_CHECK_PACK, PTGPU_ERR_INVALID, "check %d", which);
    PT_CHECK(count <= (1ull << 32), PTGPU_ERR_INVALID, "%llu patterns: binary32 has 2^32", count);
    PT_NO_CAPTURE(ctx, "a check of the math");
    PT_HIP(hipSetDevice(ctx->device));
    DevBuf sum;
    PT_TRY(sum.ensure(8));
    int st = fill_u32(ctx->stream, sum.p, 0u, 2);
    if (st == PTGPU_OK) {
        const dim3 grid((unsigned)(8 * ctx->cu_count)), block(256);
        auto *d = sum.as<unsigned long long>();
        const float *tab = ctx->pack_tab.as<float>();
        if (which == PTGPU_CHECK_RCP) hipLaunchKernelGGL(k_check_math<PTGPU_CHECK_RCP>, grid, block, 0, ctx->stream, first, count, tab, d);
        else if (which == PTGPU_CHECK_SQRT) hipLaunchKernelGGL(k_check_math<PTGPU_CHECK_SQRT>, grid, block, 0, ctx->stream, first, count, tab, d);
        else hipLaunchKernelGGL(k_check_math<PTGPU_CHECK_PACK>, grid, block, 0, ctx->stream, first, count, tab, d);
        st = hipGetLastError() == hipSuccess && hipMemcpyAsync(wrong, d, 8, hipMemcpyDeviceToHost, ctx->stream) == hipSuccess &&
                     hipStreamSynchronize(ctx->stream) == hipSuccess ? PTGPU_OK : PTGPU_ERR_HIP;
    }
    sum.release();
    return st;
}
