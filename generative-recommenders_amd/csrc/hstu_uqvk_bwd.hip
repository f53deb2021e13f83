// Products of the dense steps' backward on the producer's kernels (libhstu_linear.so); compiled as hstu_uqvk.hip is.
#include "hstu_uqvk_launch.h"
#include "hstu_product_split_kernel.h"

namespace {

bool producer_depth(int depth) { return depth == 128 || depth == 256 || depth == 384 || depth == 512; }

// The product at the other depths: while its workgroups are one round of the CUs, which their LDS fills.  us on the GPU, the library's / with it: 768 deep into 256 columns, 700 rows
// 4.9 / 4.8, 2048 rows (the last) 6.0 / 5.3, 2200 rows 7.4 / 9.3; 1024 into 512, 700 rows 8.5 / 5.9, 1100 rows 8.5 / 10.2; 2048 into 640, 20 rows 5.3 / 6.7, 700 rows 9.7 / 9.2; the
// library's choice for a batch's own rows takes 15 us of the host besides.  Past a depth of 1024 few workgroups are a longer chain than the library's split of the depth (25 rows of 3840 into 384
// 6.7 / 9.2, 59 of 2560 into 128 5.8 / 7.5; many are not: 287 of 4032 into 1536 21.4 / 11.7), and the operator is faster all the same: its backward, one after the other, 20 rows of 512 into 2048 90 / 73,
// 25 of 1024 into 4096 114 / 99.  Deeper than 1024 only up to 512 rows, which is no line between times: past them a test of the operator expects the framework's product bit for bit.
bool split_takes(int64_t rows, int depth, int n) {
    if (depth % 64 != 0 || n % hstu::kSplitCols != 0 || (depth > 1024 && rows > 512)) return false;
    return (rows + hstu::kSplitRows - 1) / hstu::kSplitRows * (n / hstu::kSplitCols) <= 256;
}

}  // namespace

// depth: 128, 256, 384 or 512; n_out a multiple of 128
int hstu_uqvk_grad_u_launch(const hstu::UqvkFusedParams& p, int depth, bool bf16, hipStream_t stream) {
    return launch_mode<hstu::kUqvkGradU>(p, depth, bf16, stream);
}
// Whether the product with a transposed matrix is these kernels' or the library GEMM's (choose_product, split_takes).
bool hstu_product_t_takes(int64_t rows, int depth, int n) {
    if (n <= 0 || n > (1 << 20) || rows > 0x7fffffffLL) return false;
    if (!producer_depth(depth)) return split_takes(rows, depth, n);
    return n % 128 == 0 && choose_product(rows, n, depth / 64).kernel != Kernel::kLibrary;
}
int hstu_product_t_launch(const hstu::UqvkFusedParams& p, int depth, bool bf16, hipStream_t stream) {
    if (producer_depth(depth)) return launch_mode<hstu::kProductT>(p, depth, bf16, stream);
    const hstu::ProductSplitParams sp{p.x, p.w, p.out, p.x_rs, p.w_rs, p.out_rs, p.rows, depth};
    const dim3 grid((unsigned)(p.n_out / hstu::kSplitCols), (unsigned)((p.rows + hstu::kSplitRows - 1) / hstu::kSplitRows));
    auto kern = bf16 ? hstu::hstu_product_split_kernel<hstu::Bf16> : hstu::hstu_product_split_kernel<hstu::Fp16>;
    static std::atomic<bool> attr_done[2][64];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev >= 64) dev = -1;
    hipError_t e = hipSuccess;
    if (dev < 0 || !attr_done[bf16][dev]) {  // (a function attribute belongs to the device it was set on)
        e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, hstu::kSplitLds);
        if (e == hipSuccess && dev >= 0) attr_done[bf16][dev] = true;
    }
    if (e == hipSuccess) {
        hipLaunchKernelGGL(kern, grid, dim3(hstu::kSplitWaves * 64), hstu::kSplitLds, stream, sp);
        e = hipGetLastError();
    }
    if (e == hipSuccess) return 0;
    char text[256];
    snprintf(text, sizeof(text), "product kernel launch: %s", hipGetErrorString(e));
    hstu_linear_set_last_error(text);
    return -7;
}
