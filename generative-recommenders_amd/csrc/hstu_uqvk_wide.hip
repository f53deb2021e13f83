// The producer's kernel with 64 rows per wave (libhstu_linear.so).  A translation unit of its own because it is compiled with the
// matrix instructions' VGPR form: the normalised rows fill the accumulation registers, the sums stay where vector
// instructions can read them (with the other form the kernel copies 64 registers per column block and spills).
#include "hstu_uqvk_wide_kernel.h"

#include <atomic>
#include <cstdio>

// defined in hstu_linear.hip; internal to the library
extern "C" __attribute__((visibility("hidden"))) void hstu_linear_set_last_error(const char* text);

namespace {

int fail(const char* what, hipError_t e) {
    char text[256];
    snprintf(text, sizeof(text), "%s: %s", what, hipGetErrorString(e));
    hstu_linear_set_last_error(text);
    return -7;
}

template <class TT, int KT, bool OUT8>
int launch(hstu::UqvkFusedParams p, hipStream_t stream) {
    auto kern = hstu::hstu_uqvk_wide_kernel<TT, KT, OUT8>;
    static std::atomic<bool> attr_done[64];  // (a function attribute belongs to the device it was set on)
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev >= 64) dev = -1;
    if (dev < 0 || !attr_done[dev]) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, hstu::kWideLds<KT>);
        if (e != hipSuccess) return fail("fused uqvk kernel attribute", e);
        if (dev >= 0) attr_done[dev] = true;
    }
    p.units = (int)((p.rows + hstu::kWideRows - 1) / hstu::kWideRows) * (p.n_out / hstu::kWideCols);
    const int grid = p.units < 256 ? p.units : 256;  // one workgroup per CU
    p.chunks_per_wg = p.units / grid;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), hstu::kWideLds<KT>, stream, p);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail("fused uqvk kernel launch", e);
}

template <class TT>
int launch_width(const hstu::UqvkFusedParams& p, int d_model, hipStream_t stream) {
    switch (d_model) {
        case 256: return p.out8 ? launch<TT, 4, true>(p, stream) : launch<TT, 4, false>(p, stream);
        case 384: return p.out8 ? launch<TT, 6, true>(p, stream) : launch<TT, 6, false>(p, stream);
        default: return p.out8 ? launch<TT, 8, true>(p, stream) : launch<TT, 8, false>(p, stream);
    }
}

}  // namespace

// d_model: 256, 384 or 512
int hstu_uqvk_wide_launch(const hstu::UqvkFusedParams& p, int d_model, bool bf16, hipStream_t stream) {
    return bf16 ? launch_width<hstu::Bf16>(p, d_model, stream) : launch_width<hstu::Fp16>(p, d_model, stream);
}
