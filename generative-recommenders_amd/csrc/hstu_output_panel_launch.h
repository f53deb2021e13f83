// Launching the one-kernel output step for more than a few rows (hstu_output_panel_kernel.h); part of hstu_uqvk.hip, which is compiled with the matrix
// instructions' VGPR form: the sums are few, and the vector instructions of the epilogue read them.
#pragma once
#include "hstu_output_panel_kernel.h"
#include "hstu_output_wide_kernel.h"

#include <atomic>
#include <cstdio>

// defined in hstu_linear.hip; internal to the library
extern "C" __attribute__((visibility("hidden"))) void hstu_linear_set_last_error(const char* text);
namespace {

template <class TT, bool GROUP, int D, int RB, int NW>
int launch_shape(const hstu::OutputPanelParams& p, hipStream_t stream) {
    typedef hstu::OutputPanel<D, RB, NW> Geo;
    auto kern = hstu::hstu_output_panel_kernel<TT, GROUP, D, RB, NW>;
    static std::atomic<bool> attr_done[64];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev >= 64) dev = -1;
    hipError_t e = hipSuccess;
    if (dev < 0 || !attr_done[dev]) {  // (a function attribute belongs to the device it was set on)
        e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Geo::kLds);
        if (e == hipSuccess && dev >= 0) attr_done[dev] = true;
    }
    if (e == hipSuccess) {
        const long long octets = ((p.nm.rows + Geo::kRows - 1) / Geo::kRows + 7) / 8;
        hipLaunchKernelGGL(kern, dim3((unsigned)(octets * 8 * (p.n / Geo::kCols))), dim3(NW * 64), Geo::kLds, stream, p);
        e = hipGetLastError();
    }
    if (e == hipSuccess) return 0;
    char text[256];
    snprintf(text, sizeof(text), "output panel kernel: %s", hipGetErrorString(e));
    hstu_linear_set_last_error(text);
    return -7;
}

template <class TT, bool GROUP, int D>
int launch_form(const hstu::OutputPanelParams& p, int form, hipStream_t stream) {
    if constexpr (D <= 256)
        if (form == hstu::kPanel64x128) return launch_shape<TT, GROUP, D, 2, 4>(p, stream);
    if (form == hstu::kPanel32x128) return launch_shape<TT, GROUP, D, 1, 4>(p, stream);
    if (form == hstu::kPanel64x256 && p.n % 256 == 0) return launch_shape<TT, GROUP, D, 2, 8>(p, stream);
    hstu_linear_set_last_error("output panel kernel: no such form for this shape");
    return -6;
}

template <class TT, bool GROUP>
int launch_width(const hstu::OutputPanelParams& p, int form, hipStream_t stream) {
    switch (p.nm.d) {
        case 128: return launch_form<TT, GROUP, 128>(p, form, stream);
        case 256: return launch_form<TT, GROUP, 256>(p, form, stream);
        case 384: return launch_form<TT, GROUP, 384>(p, form, stream);
        default: return launch_form<TT, GROUP, 512>(p, form, stream);
    }
}

}  // namespace

namespace {

template <class TT, bool GROUP, int D>
int launch_wide(const hstu::OutputPanelParams& p, hipStream_t stream) {
    auto kern = hstu::hstu_output_wide_kernel<TT, GROUP, D>;
    static std::atomic<bool> attr_done[64];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev >= 64) dev = -1;
    hipError_t e = hipSuccess;
    if (dev < 0 || !attr_done[dev]) {
        e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, hstu::kOutWideLds);
        if (e == hipSuccess && dev >= 0) attr_done[dev] = true;
    }
    if (e == hipSuccess) {
        const long long items = (p.nm.rows + hstu::kOutWideRows - 1) / hstu::kOutWideRows * (p.n / hstu::kOutWideCols);
        hipLaunchKernelGGL(kern, dim3((unsigned)(items < 256 ? items : 256)), dim3(hstu::kOutWideWaves * 64), hstu::kOutWideLds, stream, p);
        e = hipGetLastError();
    }
    if (e == hipSuccess) return 0;
    char text[256];
    snprintf(text, sizeof(text), "wide output kernel: %s", hipGetErrorString(e));
    hstu_linear_set_last_error(text);
    return -7;
}

template <class TT, bool GROUP>
int launch_wide_width(const hstu::OutputPanelParams& p, hipStream_t stream) {
    switch (p.nm.d) {
        case 256: return launch_wide<TT, GROUP, 256>(p, stream);
        case 384: return launch_wide<TT, GROUP, 384>(p, stream);
        case 512: return launch_wide<TT, GROUP, 512>(p, stream);
        default: return launch_wide<TT, GROUP, 1024>(p, stream);
    }
}

}  // namespace

// p.nm.d: 256, 384, 512 or 1024; all three blocks; p.n a multiple of 512
int hstu_output_wide_launch(const hstu::OutputPanelParams& p, bool bf16, bool group, hipStream_t stream) {
    if (bf16) return group ? launch_wide_width<hstu::Bf16, true>(p, stream) : launch_wide_width<hstu::Bf16, false>(p, stream);
    return group ? launch_wide_width<hstu::Fp16, true>(p, stream) : launch_wide_width<hstu::Fp16, false>(p, stream);
}

// p.nm.d: 128, 256, 384 or 512; form: one that output_panel_form or output_panel_tail_form gives for it
int hstu_output_panel_launch(const hstu::OutputPanelParams& p, int form, bool bf16, bool group, hipStream_t stream) {
    if (bf16) return group ? launch_width<hstu::Bf16, true>(p, form, stream) : launch_width<hstu::Bf16, false>(p, form, stream);
    return group ? launch_width<hstu::Fp16, true>(p, form, stream) : launch_width<hstu::Fp16, false>(p, form, stream);
}
