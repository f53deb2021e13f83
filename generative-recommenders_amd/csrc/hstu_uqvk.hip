// The producer's kernels and the one-kernel output step (libhstu_linear.so).  A translation unit of its own because of how it is compiled: see hstu_uqvk_launch.h.
#include "hstu_uqvk_launch.h"
#include "hstu_output_panel_launch.h"

// d_model: 128, 256, 384 or 512
int hstu_uqvk_launch(const hstu::UqvkFusedParams& p, int d_model, bool bf16, hipStream_t stream) {
    return p.out8 ? launch_mode<hstu::kUqvkForward8>(p, d_model, bf16, stream) : launch_mode<hstu::kUqvkForward>(p, d_model, bf16, stream);
}
