// The pipelined forward kernels for the delta form with runs fitted to the lengths (decode_fitted in hstu_common.h): the FIT
// variants, in a translation unit of their own so that they compile beside the others.
#include "hstu_hip.h"

#include <hip/hip_runtime.h>

#include "hstu_fwd_pp_kernel.h"
#include "hstu_fwd_stream_kernel.h"

namespace {

template <class TT, int D>
void launch(const hstu::FwdParams& p, int cfg, int grid_per_xcd, hipStream_t stream) {
    const dim3 grid((unsigned)grid_per_xcd * 8);
    if (cfg == 2) hipLaunchKernelGGL((hstu::hstu_fwd_stream_kernel<TT, D, D, 64, true>), grid, dim3(512), 0, stream, p);
    else hipLaunchKernelGGL((hstu::hstu_fwd_pp_kernel<TT, D, D, 64, 1, true>), grid, dim3(256), 0, stream, p);
}

template <class TT>
void launch_dim(const hstu::FwdParams& p, int dim, int cfg, int grid_per_xcd, hipStream_t stream) {
    if (dim == 32) launch<TT, 32>(p, cfg, grid_per_xcd, stream);
    else if (dim == 64) launch<TT, 64>(p, cfg, grid_per_xcd, stream);
    else launch<TT, 128>(p, cfg, grid_per_xcd, stream);
}

}  // namespace

// The caller has checked the arguments (dim 32, 64 or 128; cfg 2 or 3) and looks at hipGetLastError.
extern "C" __attribute__((visibility("hidden"))) void hstu_hip_launch_fitted(const hstu::FwdParams* p, int dtype, int dim, int cfg, int grid_per_xcd,
                                                                           hipStream_t stream) {
    if (dtype == HSTU_BF16) launch_dim<hstu::Bf16>(*p, dim, cfg, grid_per_xcd, stream);
    else if (dtype == HSTU_FP16) launch_dim<hstu::Fp16>(*p, dim, cfg, grid_per_xcd, stream);
    else launch_dim<hstu::Fp8>(*p, dim, cfg, grid_per_xcd, stream);
}
