// Launching the kernels of hstu_uqvk_kernel.h and hstu_uqvk_wide_kernel.h: which one a call takes.  Shared by the translation units that
// instantiate them (hstu_uqvk.hip: the producer; hstu_uqvk_bwd.hip: products of its backward), which are compiled with the matrix
// instructions' VGPR form: the rows fill the accumulation registers, the sums stay where vector instructions can read them (with
// the other form the kernels copy their sums per column block and spill).
#pragma once
#include "hstu_uqvk_kernel.h"
#include "hstu_uqvk_wide_kernel.h"

#include <atomic>
#include <cstdio>
#include <type_traits>

// defined in hstu_linear.hip; internal to the library
extern "C" __attribute__((visibility("hidden"))) void hstu_linear_set_last_error(const char* text);
int hstu_uqvk_fused_launch(hstu::UqvkFusedParams p, int d_model, bool bf16, hipStream_t stream);

namespace {

int fail(const char* what, hipError_t e) {
    char text[256];
    snprintf(text, sizeof(text), "%s: %s", what, hipGetErrorString(e));
    hstu_linear_set_last_error(text);
    return -7;
}

// Launches `kern` with `lds` bytes of dynamic LDS, of which it never asks for more than `most`.
int launch(void (*kern)(hstu::UqvkFusedParams), std::atomic<bool> (&attr_done)[64], int most, int lds, dim3 grid, const hstu::UqvkFusedParams& p,
           hipStream_t stream) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev >= 64) dev = -1;
    if (dev < 0 || !attr_done[dev]) {  // (a function attribute belongs to the device it was set on)
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, most);
        if (e != hipSuccess) return fail("fused uqvk kernel attribute", e);
        if (dev >= 0) attr_done[dev] = true;
    }
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, stream, p);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail("fused uqvk kernel launch", e);
}

template <class TT, int KT, int MODE>
int launch_wide(hstu::UqvkFusedParams p, hipStream_t stream) {
    static std::atomic<bool> attr_done[64];
    p.units = (int)((p.rows + hstu::kWideRows - 1) / hstu::kWideRows) * (p.n_out / hstu::kWideCols);
    const int grid = p.units < 256 ? p.units : 256;  // one workgroup per CU
    p.units_per_wave = p.units / grid;
    return launch(hstu::hstu_uqvk_wide_kernel<TT, KT, MODE>, attr_done, hstu::kWideLds<KT>, hstu::kWideLds<KT>, dim3((unsigned)grid), p, stream);
}

template <class TT, int KT, int RB, int NB, int MODE>
int launch_rows(hstu::UqvkFusedParams p, int units_per_wave, hipStream_t stream) {
    static std::atomic<bool> attr_done[64];
    typedef hstu::UqvkRows<KT, RB, NB> Geo;
    const long long blocks = (p.rows + RB * 32 - 1) / (RB * 32);
    const int units = (p.n_out / NB + 3) / 4;  // of a wave that walks its quarter of all columns
    p.units_per_wave = units_per_wave < units ? units_per_wave : units;
    const unsigned splits = (unsigned)((units + p.units_per_wave - 1) / p.units_per_wave);
    return launch(hstu::hstu_uqvk_rows_kernel<TT, KT, RB, NB, MODE>, attr_done, Geo::lds(hstu::kUqvkMostUnits), Geo::lds(p.units_per_wave),
                  dim3((unsigned)blocks, splits), p, stream);
}

enum class Kernel { kRows32, kRows64, kFused, kWide, kLibrary };
struct Choice {
    Kernel kernel;
    int units_per_wave;
};

// The kernel of the product with a transposed matrix, or the library GEMM.  No norm to repeat, but only the products to gain from.  us, these kernels' / the
// library's, whose time jumps by half between neighbouring sizes (depth 512 into 1024 columns: 10000 rows 17.6, 12000 33.3), so that no line suits all.
//   * kRows32 while all column units can be waves of their own in one round, two workgroups per CU: depth 512, 1000 rows into 1536 columns 6.4 / 8.4,
//     8000 into 256 6.8 / 9.4.
//   * kWide at depth 256 from 6 units (row blocks of 256 x column blocks of 64) per CU on: 17000 rows into 2048 columns 27.6 / 50, kRows64 34.8; 8000 into
//     6144 29.1 / 40, 46.8.  At depth 384 and 512 from more than 4 (depth 512, 17000 rows into 1024 34.5 / 42.1, 54000 into 1536 94 / 134; at 4 units 32768
//     into 512 26.2 / 22.8), but for what kRows64 does in one round with up to 6 units per wave (12000 rows into 1536 32.0, kWide 34.6, the library 46).
//   * At depth 384 and 512, W above the 4 MB of an XCD's L2: kRows32 with one workgroup per CU, kWide from 2.75 units on, the library between them
//     (depth 512 into 6144 columns, 100 rows 4.8 / 7.2, 200 rows 10.0 / 8.2, 1000 rows 20.0 / 14.6, 2000 rows 21.0 / 28.4, 4000 rows 29.9 / 41).
//     From 3 MB at depth 512 the library too between kRows32 (of 4 MB: with one workgroup per CU) and kWide (into 3072 columns, 1300 rows 11.9 / 10.0, 2315 16.7 /
//     13.6, 4533 24.8 / 19.9, 5400 33.2 / 44.5; into 4096, 450 rows 8.4 / 7.0, 900 11.9 / 9.1, 2000 17.0 / 15.2, 3764 29.0 / 21.2, 4100 33.4 / 36.8).
//   * Otherwise there into fewer than 1024 columns the library (5000 rows into 768 10.1 / 9.7), from there kRows64: with one unit per wave (1100 rows into
//     2048 8.6 / 10.0), with several where they give seven tenths of the CUs a workgroup (2600 rows into 2560 14.9 / 19.0, 12000 into 1024 23.2 / 33.3;
//     fewer: 3000 rows into 1536 13.2 / 11.9, 5000 into 2048 23.6 / 17.3).
//   * Up to depth 256 kRows64, in one round with as many units per wave as that takes (54000 rows of depth 256 into 768 columns 30 / 50, 12000 of depth 128
//     into 1536 13.5 / 26), and in several but for 256 columns of depth 256 in the second (54000 rows 17.3 / 15.2, 100000 29.5 / 34.9).
Choice choose_product(int64_t rows, int n, int kt) {
    const long long wide_units = (rows + 255) / 256 * (n / 64), blocks32 = (rows + 31) / 32, blocks64 = (rows + 63) / 64;
    const int quarter32 = n / 128, quarter = kt <= 4 ? quarter32 : (quarter32 + 1) / 2;
    const bool large = kt > 4 && (long long)n * kt * 128 > (4 << 20);
    const bool wide = kt >= 4 && n >= 512 && wide_units >= (kt == 4 ? 1536 : large ? 704 : 1025) && wide_units <= 0x7fffffffLL;
    if (blocks32 * quarter32 <= (kt > 4 && (long long)n * kt * 128 >= (4 << 20) ? 256 : 512)) return {Kernel::kRows32, 1};
    if (kt > 4 && (large || n < 1024 || (kt == 8 && n >= 3072))) return {wide ? Kernel::kWide : Kernel::kLibrary, 0};
    if (kt == 4 && wide) return {Kernel::kWide, 0};
    const int round = kt <= 4 ? 512 : 256;
    for (int per = 1; per <= (kt <= 4 ? hstu::kUqvkMostUnits : 8); per *= 2) {
        const long long workgroups = blocks64 * ((quarter + per - 1) / per);
        if (workgroups > round) continue;
        if (wide && per == 8 && quarter > 6) break;
        if (kt > 4 && per > 1 && workgroups * 10 < round * 7) return {Kernel::kLibrary, 0};
        return {Kernel::kRows64, per};
    }
    if (wide) return {Kernel::kWide, 0};
    if (kt == 4 && n == 256 && blocks64 <= 1024) return {Kernel::kLibrary, 0};
    return {Kernel::kRows64, hstu::kUqvkMostUnits};
}

// The kernel of the gradient of u.  us, against what stood here before, layer norm + library GEMM + hstu_uqvk_silu_bwd.
//   * kRows32 and kRows64 in one round as for the producer (choose), and up to depth 256 in more rounds too (depth 256, 90000 rows into 512 columns 83 / 126).
//   * Several rounds at depth 384 and 512: kRows32, each workgroup all columns, two per CU, up to 384 columns (depth 384 into 128, 60000 rows 41.8 / 44.3, kRows64
//     58.9: half its waves have no unit; depth 512 into 384, 20000 rows 32.1 / 36.0, kRows64 42.7), and into more while it has few rounds: depth 512 into 512,
//     60000 rows 80.8 / 96.5, kRows64 87.3; 90000 rows 147.8, kRows64 140.5; depth 384 into 1024, 20000 rows 54.6 / 59.0, kRows64 65.9.
//   * Beyond, kRows64 with the columns divided so that rounds x (the rows' preparation, about two units' time, + units) is smallest: depth 384 into 2048,
//     24000 rows 4 units per wave 114, 8 125 / 129; 60000 rows 8 units 252, 4 280 / 312.  Just past one round it stays up to 8 % behind (depth 384 into 768,
//     16500 rows 46.5 / 43.1).
Choice choose_grad_u(int64_t rows, int n, int kt) {
    const int quarter32 = n / 128, quarter = kt <= 4 ? quarter32 : (quarter32 + 1) / 2, round = kt <= 4 ? 512 : 256;
    const long long blocks32 = (rows + 31) / 32, blocks64 = (rows + 63) / 64;
    if (blocks32 * quarter32 <= 512) return {Kernel::kRows32, 1};
    if (n <= 256 && kt > 4 && blocks32 <= 1024) return {Kernel::kRows32, quarter32};
    for (int per = 1; per <= (kt <= 4 ? hstu::kUqvkMostUnits : 8); per *= 2)
        if (blocks64 * ((quarter + per - 1) / per) <= round) return {Kernel::kRows64, per};
    if (kt <= 4) return {Kernel::kRows64, hstu::kUqvkMostUnits};
    if (n <= 384 || (n <= 1024 && blocks32 * quarter32 <= 9216)) return {Kernel::kRows32, quarter32};
    Choice best{Kernel::kRows64, 1};
    double least = 1e300;
    for (int per = 1; per <= hstu::kUqvkMostUnits; per *= 2) {
        const int splits = (quarter + per - 1) / per;
        const double cost = (double)((blocks64 * splits + 255) / 256) * (2 + (double)quarter / splits);
        if (cost < least) least = cost, best.units_per_wave = per;
    }
    return best;
}

// The kernel of a call of the producer.  All sizes in us, this rule's choice against the kernel on the other side of the line.
//   * kWide where its work, row blocks of 256 x column blocks of 64, gives each CU 16 units or more; below that the rows' preparation, 256
//     at a time on one CU, outweighs the faster matrix phase.  Against kFused, d_model 512 into 2048 columns: 26000 rows 91 / 87, 32768
//     85 / 100, 139264 329 / 408; into 4096: 12000 rows 87 / 83, 16384 88 / 98.  Against kRows64, d_model 256 into 2048: 24000 rows 52 / 48,
//     45000 77 / 88; into 512: 90000 rows 61 / 52.  Columns: into 256 it is slower at every size (300000 rows of d_model 512: 197 / 177).
//   * kRows32 while all column units can be waves of their own in one round of workgroups, two per CU: d_model 512 into 2048 columns, 1000
//     rows 10.3, kRows64 12.4; 2000 rows (two rounds) 18.5 / 13.8.  Few columns, up to 256: up to two rounds of workgroups that hold all of
//     them: d_model 512 into 128 columns, 24000 rows 14.5, kRows64 23.0, kFused 17.8; 90000 rows 45.5 / 72.1 / 41.1.  d_model 384: only where
//     they are no slower than kFused there (into 128 columns, 24000 rows 13.6 / 13.5, 30000 15.6 / 14.1; into 256, 30000 22.9 / 22.8, 30700 23.1 / 21.6).
//   * kRows64, dividing the columns over as many workgroups as one round holds (one per CU, two up to d_model 256): d_model 512 into 2048,
//     4000 rows with 2 units per wave 21.3, with 1 29.0, with 4 27.5.  More rounds, and more than 8 units per wave, are kFused's at d_model
//     384 and 512 (into 512 columns, 24000 rows 35.1 / 33.4, 90000 rows 109 / 88; into 4096, 12000 rows 92 / 81), more than 4 at d_model 384 (into
//     2048, 8200 rows 40.7 / 34.1), 8 for fewer than 176 workgroups (d_model 512 into 4096, 5100 rows 44.8 / 41.1, 6000 45.4 / 48.2), and, where W exceeds an
//     XCD's 4 MB of L2, more than 4 (d_model 512 into 6144, 5400 rows 67 / 60) or than 160 workgroups that each read it (into 8192, 2000 rows 49.0 / 35.7;
//     into 5120, 2000 rows 31.3 / 32.7), and kRows64's below (d_model 256 into 512 columns, 45000 rows 29.3 / 38.3).
Choice choose(const hstu::UqvkFusedParams& p, int kt, int mode) {
    if (mode == hstu::kProductT) return choose_product(p.rows, p.n_out, kt);
    if (mode == hstu::kUqvkGradU) return choose_grad_u(p.rows, p.n_out, kt);
    const long long wide_units = (p.rows + 255) / 256 * (p.n_out / 64);
    const bool whole64 = p.n_silu % 64 == 0;  // (SiLU per 64 columns)
    if (kt >= 4 && p.n_out >= 512 && whole64 && wide_units >= 4096 && wide_units <= 0x7fffffffLL) return {Kernel::kWide, 0};
    const int quarter32 = p.n_out / 128;  // column units of a wave that walks a quarter of the columns
    const long long blocks32 = (p.rows + 31) / 32, blocks64 = (p.rows + 63) / 64;
    if (blocks32 * quarter32 <= 512) return {Kernel::kRows32, 1};
    if (p.n_out <= 256 && kt > 4 && blocks32 <= (kt == 8 ? 1024 : p.n_out == 128 ? 512 : 940)) return {Kernel::kRows32, quarter32};
    const int quarter = kt <= 4 ? quarter32 : (quarter32 + 1) / 2, round = kt <= 4 ? 512 : 256;
    if (kt <= 4 || whole64) {
        const bool large = kt > 4 && (long long)p.n_out * kt * 128 > (4 << 20);
        for (int per = 1; per <= (kt <= 4 ? hstu::kUqvkMostUnits : kt == 8 && !large ? 8 : 4); per *= 2) {
            const long long workgroups = blocks64 * ((quarter + per - 1) / per);
            if (workgroups > round) continue;
            if (kt > 4 && (large ? workgroups > 160 : per == 8 && workgroups < 176)) break;
            return {Kernel::kRows64, per};
        }
        if (kt <= 4) return {Kernel::kRows64, hstu::kUqvkMostUnits};
    }
    return {Kernel::kFused, 0};
}

template <class TT, int KT, int MODE>
int launch_depth(const hstu::UqvkFusedParams& p, hipStream_t stream) {
    const Choice c = choose(p, KT, MODE);
    if constexpr (KT >= 4 && MODE != hstu::kUqvkGradU)
        if (c.kernel == Kernel::kWide) return launch_wide<TT, KT, MODE>(p, stream);
    if constexpr (KT > 4 && (MODE == hstu::kUqvkForward || MODE == hstu::kUqvkForward8))
        if (c.kernel == Kernel::kFused) return hstu_uqvk_fused_launch(p, KT * 64, std::is_same<TT, hstu::Bf16>::value, stream);
    if (c.kernel == Kernel::kRows32) return launch_rows<TT, KT, 1, 32, MODE>(p, c.units_per_wave, stream);
    return launch_rows<TT, KT, 2, (KT <= 4 ? 32 : 64), MODE>(p, c.units_per_wave, stream);
}

template <class TT, int MODE>
int launch_type(const hstu::UqvkFusedParams& p, int d_model, hipStream_t stream) {
    switch (d_model) {
        case 128: return launch_depth<TT, 2, MODE>(p, stream);
        case 256: return launch_depth<TT, 4, MODE>(p, stream);
        case 384: return launch_depth<TT, 6, MODE>(p, stream);
        default: return launch_depth<TT, 8, MODE>(p, stream);
    }
}

template <int MODE>
int launch_mode(const hstu::UqvkFusedParams& p, int d_model, bool bf16, hipStream_t stream) {
    return bf16 ? launch_type<hstu::Bf16, MODE>(p, d_model, stream) : launch_type<hstu::Fp16, MODE>(p, d_model, stream);
}

}  // namespace
