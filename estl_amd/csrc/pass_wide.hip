// pass_wide.hip -- k_pass_wide: one global Stockham pass with 32 values per thread
// (pass_wide.h), FP32 or FP16 storage, compiled once per direction (-DESTL_PASS_DIR).
#include "pass_wide.h"

#ifndef ESTL_PASS_DIR
#error "compile pass_wide.hip with -DESTL_PASS_DIR=-1 or +1"
#endif

namespace estl {

template <int LOG2B, int DIR, int LOG2T, int MODE, typename ST>
__global__ void __launch_bounds__(1 << (LOG2B - 5 + LOG2T)) __attribute__((amdgpu_waves_per_eu(4)))
k_pass_wide(const ST *__restrict__ in, ST *__restrict__ out, PassArgs a) {
    __shared__ float lds[WideTile<LOG2B, LOG2T, MODE>::lds_floats];
    if constexpr (!__is_same(ST, float2)) row_scale<LOG2B, LOG2T>(a, blockIdx.x);
    wide_tile<LOG2B, DIR, LOG2T, MODE>(in, out, a, blockIdx.x, lds);
}

template <int LOG2B, int LOG2T, typename ST>
static hipError_t launch_t(const void *in, void *out, const PassArgs &a, hipStream_t st) {
    const int lcpr = a.log2n - LOG2B;
    if (lcpr < LOG2T) return hipErrorInvalidValue;
    const long tiles = a.batch << (lcpr - LOG2T);
    if (tiles > 0x7fffffffL) return hipErrorInvalidValue;
    auto kernel = a.A == 1 ? k_pass_wide<LOG2B, ESTL_PASS_DIR, LOG2T, kWideFirst, ST>
                           : k_pass_wide<LOG2B, ESTL_PASS_DIR, LOG2T, kWideMiddle, ST>;
    if (a.A > 1 && a.log2S < LOG2T) {
        if constexpr (LOG2B > 7) kernel = k_pass_wide<LOG2B, ESTL_PASS_DIR, LOG2T, kWideLast, ST>;
        else return hipErrorInvalidValue;  // pass_is_wide: k_fft_pass's
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(WideTile<LOG2B, LOG2T, 0>::threads), 0, st,
                       static_cast<const ST *>(in), static_cast<ST *>(out), a);
    return hipGetLastError();
}

template <typename ST>
static hipError_t launch_w(int log2b, int log2t, const void *in, void *out, const PassArgs &a, hipStream_t st) {
    switch (log2b * 16 + log2t) {
#define WIDE(B, T) \
    case B * 16 + T: return launch_t<B, T, ST>(in, out, a, st);
        WIDE(7, 6) WIDE(8, 5) WIDE(8, 6) WIDE(9, 4) WIDE(9, 5) WIDE(10, 4)
#undef WIDE
        default: return hipErrorInvalidValue;
    }
}

#if ESTL_PASS_DIR < 0
#define ESTL_WIDE_LAUNCHER launch_pass_wide_fwd
#else
#define ESTL_WIDE_LAUNCHER launch_pass_wide_bwd
#endif

hipError_t ESTL_WIDE_LAUNCHER(int log2b, int log2t, bool fp16, const void *in, void *out, const PassArgs &a,
                              hipStream_t st) {
    return fp16 ? launch_w<f16x2>(log2b, log2t, in, out, a, st) : launch_w<float2>(log2b, log2t, in, out, a, st);
}

}  // namespace estl
