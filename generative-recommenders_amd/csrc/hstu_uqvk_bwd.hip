// Products of the dense steps' backward on the producer's kernels (libhstu_linear.so); compiled as hstu_uqvk.hip is.
#include "hstu_uqvk_launch.h"

// depth: 128, 256, 384 or 512; n_out a multiple of 128
int hstu_uqvk_grad_u_launch(const hstu::UqvkFusedParams& p, int depth, bool bf16, hipStream_t stream) {
    return launch_mode<hstu::kUqvkGradU>(p, depth, bf16, stream);
}
// Whether the product with a transposed matrix is these kernels' or the library GEMM's (choose_product).
bool hstu_product_t_takes(int64_t rows, int depth, int n) {
    if ((depth != 128 && depth != 256 && depth != 384 && depth != 512) || n <= 0 || n % 128 != 0 || n > (1 << 20) || rows > 0x7fffffffLL) return false;
    return choose_product(rows, n, depth / 64).kernel != Kernel::kLibrary;
}
int hstu_product_t_launch(const hstu::UqvkFusedParams& p, int depth, bool bf16, hipStream_t stream) {
    return launch_mode<hstu::kProductT>(p, depth, bf16, stream);
}
