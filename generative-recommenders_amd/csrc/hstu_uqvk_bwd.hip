// Products of the dense steps' backward on the producer's kernels (libhstu_linear.so); compiled as hstu_uqvk.hip is.
#include "hstu_uqvk_launch.h"

// depth: 128, 256, 384 or 512; n_out a multiple of 128
int hstu_uqvk_grad_u_launch(const hstu::UqvkFusedParams& p, int depth, bool bf16, hipStream_t stream) {
    return launch_mode<hstu::kUqvkGradU>(p, depth, bf16, stream);
}
// Whether the product with a transposed matrix is these kernels' or the library GEMM's.  Theirs, us against the library's: up to depth 256
// (54000 rows into 768 columns 30 / 50, 100000 into 256 30 / 35); where all column units are waves of one round (33 rows of depth 512 into
// 1536 columns 4.6 / 5.1); into 1024 columns and more (8000 rows into 1536 25 / 28, 12000 35 / 44; 3000 14.2 / 11.8, but the library's call costs the
// host 5 us more); where the kernel with 64 rows per wave has its units (139264 rows into 1536 216 / 320, 54000 into 512 44 / 64).  The library's: few
// columns of depth 384 and 512 between these (30000 rows into 512 columns 30 / 23, 54000 into 128 33 / 19).
bool hstu_product_t_takes(int64_t rows, int depth, int n) {
    if ((depth != 128 && depth != 256 && depth != 384 && depth != 512) || n % 128 != 0 || n > (1 << 20) || rows > 0x7fffffffLL) return false;
    if (depth <= 256 || n >= 1024 || (rows + 31) / 32 * (n / 128) <= 512) return true;
    return n >= 512 && (rows + 255) / 256 * (n / 64) >= kProductWide;
}
int hstu_product_t_launch(const hstu::UqvkFusedParams& p, int depth, bool bf16, hipStream_t stream) {
    return launch_mode<hstu::kProductT>(p, depth, bf16, stream);
}
