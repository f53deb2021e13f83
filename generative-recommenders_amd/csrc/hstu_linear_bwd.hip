// Backward of the dense steps (libhstu_linear.so): the norm-multiply step of the output projection, the layer norm of the producer,
// the SiLU on its u columns, and the gradients of the weights (hstu_wgrad_kernel.h).  The other products are plain GEMMs and the
// caller's.
//
// The row-wise kernels are bound by HBM, so every kernel reads each row once and writes each result once: one wave per row with 16-byte
// accesses as in the forward kernels, statistics recomputed from the row in registers (nothing is saved by the forward), the
// dropout mask regenerated from its Philox stream.  The gradients of the norm's weight and bias are sums over all rows: a wave
// keeps its share in fp32 registers, a workgroup adds its four waves in LDS and writes one partial row, and a second small
// kernel adds the partial rows in order -- no atomics, the same bits from run to run.
#include "hstu_rows.h"
#include "hstu_wgrad_kernel.h"

#include <atomic>
#include <cstdio>

// defined in hstu_linear.hip; internal to the library
extern "C" __attribute__((visibility("hidden"))) void hstu_linear_set_last_error(const char* text);

namespace {

using namespace hstu;

constexpr int kMaxPartials = 1024;  // workgroups, and partial rows, of a kernel that sums over rows

long long row_workgroups(long long rows) {
    const long long wgs = (rows + 3) / 4;
    return wgs < kMaxPartials ? wgs : kMaxPartials;
}

int launch_status(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) return 0;
    char text[256];
    snprintf(text, sizeof(text), "%s: %s", what, hipGetErrorString(e));
    hstu_linear_set_last_error(text);
    return -7;
}

// Column sums of `partial` [n, cols] in fp32, rounded once: columns [0, half) go to out0, the rest to out1.  A workgroup takes 64
// columns, its 16 waves every 16th row each.
template <class E>
__global__ __launch_bounds__(1024) void hstu_sum_partials_kernel(const float* partial, int n, int cols, int half, E* out0, E* out1) {
    __shared__ float part[16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    float sum = 0.f;
    if (c < cols) {
#pragma unroll 8
        for (int i = wave; i < n; i += 16) sum += partial[(int64_t)i * cols + c];
    }
    part[wave][lane] = sum;
    __syncthreads();
    if (wave == 0 && c < cols) {
#pragma unroll
        for (int w = 1; w < 16; ++w) sum += part[w][lane];
        if (c < half) out0[c] = (E)sum;
        else out1[c - half] = (E)sum;
    }
}

// Adds the four waves' per-lane sums (lane: NCH chunks of 8 columns) in LDS and writes the workgroup's partial row [2 * d].
template <int NCH>
__device__ __forceinline__ void write_partial_row(float (&dw)[NCH][8], float (&db)[NCH][8], int d, float* lds, float* row) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, chunks = d >> 3;
    for (int w = 0; w < 4; ++w) {
        if (wave == w) {
#pragma unroll
            for (int i = 0; i < NCH; ++i) {
                const int c = lane + 64 * i;
                if (c < chunks) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        lds[c * 8 + j] = (w ? lds[c * 8 + j] : 0.f) + dw[i][j];
                        lds[d + c * 8 + j] = (w ? lds[d + c * 8 + j] : 0.f) + db[i][j];
                    }
                }
            }
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < 2 * d; i += 256) row[i] = lds[i];
}

// ---- layer norm ---------------------------------------------------------------------------------------------------------
// dx = rstd (g - mean(g) - xhat mean(g xhat)), g = dy * weight; dweight = sum dy xhat, dbias = sum dy.
template <class V8, int NCH>
__global__ __launch_bounds__(256) void hstu_layer_norm_bwd_kernel(const char* x, int64_t x_rs, const char* weight, float eps, const char* dy,
                                                                  int64_t dy_rs, char* dx, int64_t dx_rs, int64_t rows, int d, float* partial) {
    typedef decltype(V8{}[0] + V8{}[0]) E;
    extern __shared__ float lds[];
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = (int64_t)gridDim.x * 4;
    const int chunks = d >> 3;
    const float inv_d = 1.0f / (float)d;
    float w[NCH][8], dw[NCH][8], db[NCH][8];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = lane + 64 * i;
        V8 wv{};
        if (c < chunks) wv = *(const V8*)(weight + (int64_t)c * 16);
#pragma unroll
        for (int j = 0; j < 8; ++j) w[i][j] = (float)wv[j], dw[i][j] = db[i][j] = 0.f;
    }
    for (int64_t r = wave; r < rows; r += nwaves) {
        V8 xv[NCH], gv[NCH];
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = lane + 64 * i;
            xv[i] = V8{}, gv[i] = V8{};
            if (c < chunks) {
                xv[i] = *(const V8*)(x + (r * x_rs + (int64_t)c * 8) * 2);
                gv[i] = *(const V8*)(dy + (r * dy_rs + (int64_t)c * 8) * 2);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) sum += (float)xv[i][j];
        }
        const float mean = wave_sum(sum) * inv_d;
        float sq = 0.f;
#pragma unroll
        for (int i = 0; i < NCH; ++i)
            if (lane + 64 * i < chunks)
#pragma unroll
                for (int j = 0; j < 8; ++j) sq += ((float)xv[i][j] - mean) * ((float)xv[i][j] - mean);
        const float rstd = __builtin_amdgcn_rsqf(wave_sum(sq) * inv_d + eps);
        float s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int i = 0; i < NCH; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float xh = ((float)xv[i][j] - mean) * rstd, dyj = (float)gv[i][j], g = dyj * w[i][j];
                dw[i][j] += dyj * xh, db[i][j] += dyj;  // (lanes past the row hold zeros in dy)
                s1 += g, s2 += g * xh;
            }
        s1 = wave_sum(s1) * inv_d, s2 = wave_sum(s2) * inv_d;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = lane + 64 * i;
            if (c < chunks) {
                V8 o;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    o[j] = (E)(rstd * ((float)gv[i][j] * w[i][j] - s1 - ((float)xv[i][j] - mean) * rstd * s2));
                *(V8*)(dx + (r * dx_rs + (int64_t)c * 8) * 2) = o;
            }
        }
    }
    write_partial_row<NCH>(dw, db, d, lds, partial + (int64_t)blockIdx.x * 2 * d);
}

// ---- norm * u, concatenated -----------------------------------------------------------------------------------------------
struct NormMulBwdParams {
    NormMulParams f;  // the forward's; joined: null, or where the recomputed `joined` goes
    const char* dj;   // gradient of `joined`
    char *d_attn, *d_u;
    int64_t dj_rs, da_rs, du_rs;
    float* partial;
};

// Which of eight elements at column `col` survive, as factors (0 or the scale); all ones without dropout.
__device__ __forceinline__ void keep8(const DropoutParams& d, int64_t r, int64_t width, int64_t col, float (&keep)[8]) {
    if (d.thresh == 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) keep[j] = 1.f;
        return;
    }
    const uint64_t group = (uint64_t)(r * width + col) >> 2;
    const PhiloxWords a = dropout_words(d, group), b = dropout_words(d, group + 1);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        keep[j] = a.w[j] >= d.thresh ? d.scale : 0.f;
        keep[4 + j] = b.w[j] >= d.thresh ? d.scale : 0.f;
    }
}

// One wave per row.  Reads attn, u and the gradient of `joined`; writes the gradients of attn and u and, on request, `joined`
// itself (the weight gradient's operand).  GROUP: statistics, weight and bias per head, as in the forward kernel.
template <class V8, int NCH, bool GROUP>
__global__ __launch_bounds__(256) void hstu_norm_mul_bwd_kernel(NormMulBwdParams q) {
    typedef decltype(V8{}[0] + V8{}[0]) E;
    extern __shared__ float lds[];
    const NormMulParams& p = q.f;
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = (int64_t)gridDim.x * 4;
    const int chunks = p.d >> 3;
    float w[NCH][GROUP ? 1 : 8], b[NCH][GROUP ? 1 : 8];
    float dw[NCH][8], db[NCH][8];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = lane + 64 * i;
        V8 wv{}, bv{};
        if (c < chunks) {
            if constexpr (GROUP) {
                const int head = c / p.group_lanes;
                wv[0] = ((const E*)p.weight)[head], bv[0] = ((const E*)p.bias)[head];
            } else {
                wv = *(const V8*)(p.weight + (int64_t)c * 16), bv = *(const V8*)(p.bias + (int64_t)c * 16);
            }
        }
#pragma unroll
        for (int j = 0; j < (GROUP ? 1 : 8); ++j) w[i][j] = (float)wv[j], b[i][j] = (float)bv[j];
#pragma unroll
        for (int j = 0; j < 8; ++j) dw[i][j] = db[i][j] = 0.f;
    }
    const float inv_n = GROUP ? 1.0f / (float)(p.group_lanes * 8) : 1.0f / (float)p.d;
    // sums over the elements a norm's statistics cover: the row, or the lanes of one head
    auto reduce = [&](float (&v)[NCH]) __attribute__((always_inline)) {
        if constexpr (GROUP) {
#pragma unroll
            for (int i = 0; i < NCH; ++i) {
                for (int k = 1; k < p.group_lanes; k <<= 1) v[i] += __shfl_xor(v[i], k, 64);
                v[i] *= inv_n;
            }
        } else {
            float t = 0.f;
#pragma unroll
            for (int i = 0; i < NCH; ++i) t += v[i];
            t = wave_sum(t) * inv_n;
#pragma unroll
            for (int i = 0; i < NCH; ++i) v[i] = t;
        }
    };
    for (int64_t r = wave; r < p.rows; r += nwaves) {
        V8 xraw[NCH], uraw[NCH], gu[NCH], gx[NCH], gy[NCH];
        const char* grow = q.dj + r * q.dj_rs * 2;
        float mean[NCH], rstd[NCH];
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = lane + 64 * i;
            xraw[i] = uraw[i] = gu[i] = gx[i] = gy[i] = V8{};
            if (c < chunks) {
                xraw[i] = *(const V8*)(p.attn + (r * p.attn_rs + (int64_t)c * 8) * 2);
                uraw[i] = *(const V8*)(p.u + (r * p.u_rs + (int64_t)c * 8) * 2);
                gy[i] = *(const V8*)(grow + ((int64_t)p.off_y + c * 8) * 2);
                if (p.off_u >= 0) gu[i] = *(const V8*)(grow + ((int64_t)p.off_u + c * 8) * 2);
                if (p.off_x >= 0) gx[i] = *(const V8*)(grow + ((int64_t)p.off_x + c * 8) * 2);
            }
            mean[i] = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) mean[i] += (float)xraw[i][j];
        }
        reduce(mean);
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            rstd[i] = 0.f;
            if (lane + 64 * i < chunks)
#pragma unroll
                for (int j = 0; j < 8; ++j) rstd[i] += ((float)xraw[i][j] - mean[i]) * ((float)xraw[i][j] - mean[i]);
        }
        reduce(rstd);
#pragma unroll
        for (int i = 0; i < NCH; ++i) rstd[i] = __builtin_amdgcn_rsqf(rstd[i] + p.eps);

        float s1[NCH], s2[NCH];  // means of g = d(norm) * weight and of g * xhat
        float g[NCH][8];
        char* jrow = p.joined + r * p.joined_rs * 2;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = lane + 64 * i;
            s1[i] = s2[i] = 0.f;
            if (c < chunks) {
                float keep[8];
                V8 jv, du;
                float d_u[8];
                // the copied u block
#pragma unroll
                for (int j = 0; j < 8; ++j) d_u[j] = 0.f;
                if (p.off_u >= 0) {
                    keep8(p.drop, r, p.width, (int64_t)p.off_u + c * 8, keep);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float uf = (float)uraw[i][j], sg = p.silu_u ? sigmoid_f(uf) : 1.f;
                        jv[j] = (E)(uf * sg * keep[j]);
                        // (group norm: the slope of SiLU(u), which feeds both blocks, is applied at the end)
                        d_u[j] = (float)gu[i][j] * keep[j] * (!GROUP && p.silu_u ? sg * (1.f + uf * (1.f - sg)) : 1.f);
                    }
                    if (p.joined) *(V8*)(jrow + ((int64_t)p.off_u + c * 8) * 2) = jv;
                }
                // y = gate(u) * (xhat * weight + bias)
                keep8(p.drop, r, p.width, (int64_t)p.off_y + c * 8, keep);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float uf = (float)uraw[i][j];
                    float gate = uf, slope = 1.f;
                    if (GROUP ? p.silu_u != 0 : p.mul_act != HSTU_MUL_U_NONE) {
                        const float sg = sigmoid_f(uf), silu_slope = sg * (1.f + uf * (1.f - sg));
                        const bool sigmoid = !GROUP && p.mul_act == HSTU_MUL_U_SIGMOID;
                        gate = sigmoid ? sg : uf * sg;
                        slope = sigmoid ? sg * (1.f - sg) : silu_slope;
                    }
                    const float wj = w[i][GROUP ? 0 : j], bj = b[i][GROUP ? 0 : j];
                    const float xh = ((float)xraw[i][j] - mean[i]) * rstd[i], normed = xh * wj + bj, dy = (float)gy[i][j] * keep[j];
                    jv[j] = (E)(gate * normed * keep[j]);
                    const float dn = dy * gate;
                    dw[i][j] += dn * xh, db[i][j] += dn;
                    g[i][j] = dn * wj;
                    s1[i] += g[i][j], s2[i] += g[i][j] * xh;
                    if constexpr (GROUP) d_u[j] = (d_u[j] + dy * normed) * slope;
                    else d_u[j] += dy * normed * slope;
                    du[j] = (E)d_u[j];
                }
                if (p.joined) *(V8*)(jrow + ((int64_t)p.off_y + c * 8) * 2) = jv;
                *(V8*)(q.d_u + (r * q.du_rs + (int64_t)c * 8) * 2) = du;
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) g[i][j] = 0.f;
            }
        }
        reduce(s1);
        reduce(s2);
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = lane + 64 * i;
            if (c < chunks) {
                float dx[8];
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    dx[j] = rstd[i] * (g[i][j] - s1[i] - ((float)xraw[i][j] - mean[i]) * rstd[i] * s2[i]);
                V8 o;
                if (p.off_x >= 0) {
                    float keep[8];
                    V8 jv;
                    keep8(p.drop, r, p.width, (int64_t)p.off_x + c * 8, keep);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        jv[j] = (E)((float)xraw[i][j] * keep[j]);
                        dx[j] += (float)gx[i][j] * keep[j];
                    }
                    if (p.joined) *(V8*)(jrow + ((int64_t)p.off_x + c * 8) * 2) = jv;
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = (E)dx[j];
                *(V8*)(q.d_attn + (r * q.da_rs + (int64_t)c * 8) * 2) = o;
            }
        }
    }
    if constexpr (GROUP) {
        // one weight and bias per head: the head's first lane of each wave holds the sum over its lanes; a partial row is [2 * heads]
        const int heads = chunks / p.group_lanes, wv = threadIdx.x >> 6;
        float* mine = lds + wv * 2 * heads;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = lane + 64 * i;
            float a = 0.f, e = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) a += dw[i][j], e += db[i][j];
            for (int k = 1; k < p.group_lanes; k <<= 1) a += __shfl_xor(a, k, 64), e += __shfl_xor(e, k, 64);
            if (c < chunks && c % p.group_lanes == 0) mine[c / p.group_lanes] = a, mine[heads + c / p.group_lanes] = e;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < 2 * heads; i += 256)
            q.partial[(int64_t)blockIdx.x * 2 * heads + i] = lds[i] + lds[2 * heads + i] + lds[4 * heads + i] + lds[6 * heads + i];
    } else {
        write_partial_row<NCH>(dw, db, p.d, lds, q.partial + (int64_t)blockIdx.x * 2 * p.d);
    }
}

// ---- SiLU -----------------------------------------------------------------------------------------------------------------
// v <- du * (derivative of SiLU at v + bias) in place; eight elements per thread.
template <class V8>
__global__ __launch_bounds__(256) void hstu_silu_bwd_kernel(char* v, int64_t v_rs, const char* bias, const char* du, int64_t du_rs, int64_t rows,
                                                            int chunks) {
    typedef decltype(V8{}[0] + V8{}[0]) E;
    const int64_t total = rows * chunks;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t r = i / chunks, c = i - r * chunks;
        V8* vp = (V8*)(v + (r * v_rs + c * 8) * 2);
        const V8 x = *vp, b = *(const V8*)(bias + c * 16), g = *(const V8*)(du + (r * du_rs + c * 8) * 2);
        V8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float f = (float)x[j] + (float)b[j], sg = sigmoid_f(f);
            o[j] = (E)((float)g[j] * sg * (1.f + f * (1.f - sg)));
        }
        *vp = o;
    }
}

// How the rows of a weight gradient are split: as many workgroups as the chip has CUs (one fits a CU) where the rows allow at
// least two tiles of 32 rows each; more only repeats fp32 sums (256 KB each, written and read once).  The byte offsets inside a
// split stay below 2^31.
struct WgradPlan {
    int tiles_m, tiles_n, splits, rows_per_split;
    size_t partial_bytes, colsum_bytes;
};
WgradPlan wgrad_plan(int m, int n, int64_t rows, int64_t stride) {
    WgradPlan pl;
    pl.tiles_m = (m + kWgTile - 1) / kWgTile, pl.tiles_n = (n + kWgTile - 1) / kWgTile;
    const int64_t tiles = (int64_t)pl.tiles_m * pl.tiles_n;
    int64_t want = 256 / tiles;
    if (want > rows / (2 * kWgDepth)) want = rows / (2 * kWgDepth);
    const int64_t most_rows = ((int64_t)1 << 30) / (stride * 2);  // of a split
    if (want < (rows + most_rows - 1) / most_rows) want = (rows + most_rows - 1) / most_rows;
    if (want < 1) want = 1;
    pl.rows_per_split = (int)(((rows + want - 1) / want + kWgDepth - 1) / kWgDepth * kWgDepth);
    pl.splits = (int)((rows + pl.rows_per_split - 1) / pl.rows_per_split);
    pl.partial_bytes = (size_t)pl.splits * tiles * kWgTileFloats * sizeof(float);
    pl.colsum_bytes = (size_t)pl.splits * n * sizeof(float);
    return pl;
}

template <class TT>
int launch_wgrad(const WgradParams& p, typename TT::elem* out, typename TT::elem* colsum, hipStream_t stream) {
    auto kern = hstu_wgrad_kernel<TT>;
    static std::atomic<bool> attr_done[64];  // (a function attribute belongs to the device it was set on)
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev >= 64) dev = -1;
    if (dev < 0 || !attr_done[dev]) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kWgLds) != hipSuccess)
            return launch_status("weight gradient kernel attribute");
        if (dev >= 0) attr_done[dev] = true;
    }
    const int tiles = p.tiles_m * p.tiles_n;
    hipLaunchKernelGGL(kern, dim3((unsigned)((tiles * p.splits + 7) / 8 * 8)), dim3(kWgWaves * 64), kWgLds, stream, p);
    int rc = launch_status("weight gradient kernel launch");
    if (rc != 0) return rc;
    const int tile_blocks = tiles * (kWgTileFloats / 4 / 256), sum_blocks = colsum ? (p.n + 255) / 256 : 0;
    hipLaunchKernelGGL((hstu_wgrad_reduce_kernel<typename TT::elem>), dim3((unsigned)(tile_blocks + sum_blocks)), dim3(256), 0, stream, p, out, colsum,
                       tile_blocks);
    return launch_status("weight gradient reduce kernel launch");
}

template <class E>
void sum_partials(const float* partial, long long n, int cols, int half, void* out0, void* out1, hipStream_t stream) {
    hipLaunchKernelGGL((hstu_sum_partials_kernel<E>), dim3((unsigned)((cols + 63) / 64)), dim3(1024), 0, stream, partial, (int)n, cols, half, (E*)out0,
                       (E*)out1);
}

bool misaligned(std::initializer_list<const void*> ptrs, std::initializer_list<int64_t> strides) {
    uintptr_t all = 0;
    for (const void* p : ptrs) all |= (uintptr_t)p;
    for (int64_t s : strides) all |= (uintptr_t)((s & 7) << 1);
    return (all & 15) != 0;
}

}  // namespace

extern "C" {

size_t hstu_uqvk_layer_norm_bwd_workspace_bytes(int64_t rows, int32_t d_model) {
    return rows <= 0 || d_model <= 0 ? 0 : (size_t)row_workgroups(rows) * 2 * d_model * sizeof(float);
}

int hstu_uqvk_layer_norm_bwd(const void* x, int64_t x_row_stride, const void* weight, float eps, const void* dy, int64_t dy_row_stride, void* dx,
                             int64_t dx_row_stride, void* d_weight, void* d_bias, int64_t rows, int32_t d, int32_t dtype, void* workspace,
                             int64_t workspace_bytes, void* stream_) {
    hstu_linear_set_last_error("");
    if (rows <= 0 || d <= 0 || (d & 7) != 0 || d > 4096 || x_row_stride < d || dy_row_stride < d || dx_row_stride < d) return -5;
    if (dtype != 0 && dtype != 1) return -2;
    if (!x || !weight || !dy || !dx || !d_weight || !d_bias || !workspace) return -1;
    if (misaligned({x, weight, dy, dx, workspace}, {x_row_stride, dy_row_stride, dx_row_stride})) return -4;
    if (workspace_bytes < (int64_t)hstu_uqvk_layer_norm_bwd_workspace_bytes(rows, d)) return -5;
    hipStream_t stream = (hipStream_t)stream_;
    const long long wgs = row_workgroups(rows);
    const int nch = (d / 8 + 63) / 64;
    float* partial = (float*)workspace;
#define HSTU_LNB(V8, N)                                                                                                                 \
    hipLaunchKernelGGL((hstu_layer_norm_bwd_kernel<V8, N>), dim3((unsigned)wgs), dim3(256), 2 * d * sizeof(float), stream, (const char*)x, \
                       x_row_stride, (const char*)weight, eps, (const char*)dy, dy_row_stride, (char*)dx, dx_row_stride, rows, d, partial)
#define HSTU_LNB_N(V8)                                                                                                     \
    do {                                                                                                                   \
        if (nch <= 1) HSTU_LNB(V8, 1); else if (nch <= 2) HSTU_LNB(V8, 2); else if (nch <= 4) HSTU_LNB(V8, 4); else HSTU_LNB(V8, 8); \
    } while (0)
    if (dtype == 0) HSTU_LNB_N(bf16x8_t); else HSTU_LNB_N(f16x8_t);
#undef HSTU_LNB_N
#undef HSTU_LNB
    int rc = launch_status("layer norm backward kernel launch");
    if (rc != 0) return rc;
    if (dtype == 0) sum_partials<__bf16>(partial, wgs, 2 * d, d, d_weight, d_bias, stream);
    else sum_partials<_Float16>(partial, wgs, 2 * d, d, d_weight, d_bias, stream);
    return launch_status("partial sum kernel launch");
}

size_t hstu_output_norm_mul_bwd_workspace_bytes(const HstuOutputArgs* a) {
    if (!a || a->rows <= 0 || a->heads <= 0 || a->linear_dim <= 0) return 0;
    const size_t cols = a->group_norm ? (size_t)a->heads : (size_t)a->heads * a->linear_dim;
    return (size_t)row_workgroups(a->rows) * 2 * cols * sizeof(float);
}

int hstu_output_norm_mul_bwd(const HstuOutputArgs* a, const HstuNormMulGrads* g, void* stream_) {
    hstu_linear_set_last_error("");
    if (!a || !g) return -1;
    NormMulBwdParams q;
    int rc = norm_mul_params(a, g->joined, g->joined ? g->joined_row_stride : (int64_t)output_blocks(a) * a->heads * a->linear_dim, false, q.f);
    if (rc != 0) return rc;
    if (a->rows == 0) return -5;  // nothing to sum: the caller's gradients are zero
    const int d = q.f.d, cols = a->group_norm ? a->heads : d;
    if (g->d_joined_row_stride < q.f.width || g->d_attn_row_stride < d || g->d_u_row_stride < d) return -5;
    if (!g->d_joined || !g->d_attn || !g->d_u || !g->d_norm_weight || !g->d_norm_bias || !g->workspace) return -1;
    if (misaligned({g->d_joined, g->d_attn, g->d_u, g->workspace}, {g->d_joined_row_stride, g->d_attn_row_stride, g->d_u_row_stride})) return -4;
    if (g->workspace_bytes < (int64_t)hstu_output_norm_mul_bwd_workspace_bytes(a)) return -5;
    hipStream_t stream = (hipStream_t)stream_;
    q.dj = (const char*)g->d_joined, q.dj_rs = g->d_joined_row_stride;
    q.d_attn = (char*)g->d_attn, q.da_rs = g->d_attn_row_stride, q.d_u = (char*)g->d_u, q.du_rs = g->d_u_row_stride;
    q.partial = (float*)g->workspace;
    const long long wgs = row_workgroups(a->rows);
    const int nch = (d / 8 + 63) / 64;
    const size_t lds = (a->group_norm ? 8 * a->heads : 2 * d) * sizeof(float);
#define HSTU_NMB(V8, N, G) hipLaunchKernelGGL((hstu_norm_mul_bwd_kernel<V8, N, G>), dim3((unsigned)wgs), dim3(256), lds, stream, q)
#define HSTU_NMB_N(V8, G)                                                                                                           \
    do {                                                                                                                            \
        if (nch <= 1) HSTU_NMB(V8, 1, G); else if (nch <= 2) HSTU_NMB(V8, 2, G); else if (nch <= 4) HSTU_NMB(V8, 4, G); else HSTU_NMB(V8, 8, G); \
    } while (0)
    if (a->dtype == 0) {
        if (a->group_norm) HSTU_NMB_N(bf16x8_t, true); else HSTU_NMB_N(bf16x8_t, false);
    } else {
        if (a->group_norm) HSTU_NMB_N(f16x8_t, true); else HSTU_NMB_N(f16x8_t, false);
    }
#undef HSTU_NMB_N
#undef HSTU_NMB
    rc = launch_status("norm-mul backward kernel launch");
    if (rc != 0) return rc;
    if (a->dtype == 0) sum_partials<__bf16>(q.partial, wgs, 2 * cols, cols, g->d_norm_weight, g->d_norm_bias, stream);
    else sum_partials<_Float16>(q.partial, wgs, 2 * cols, cols, g->d_norm_weight, g->d_norm_bias, stream);
    return launch_status("partial sum kernel launch");
}

int hstu_uqvk_silu_bwd(void* pre, int64_t pre_row_stride, const void* bias, const void* du, int64_t du_row_stride, int64_t rows, int64_t width, int32_t dtype,
                       void* stream_) {
    hstu_linear_set_last_error("");
    if (rows < 0 || width <= 0 || (width & 7) != 0 || width > (1 << 30) || pre_row_stride < width || du_row_stride < width) return -5;
    if (dtype != 0 && dtype != 1) return -2;
    if (rows == 0) return 0;
    if (!pre || !bias || !du) return -1;
    if (misaligned({pre, bias, du}, {pre_row_stride, du_row_stride})) return -4;
    long long wgs = (rows * (width / 8) + 255) / 256;
    if (wgs > 256 * 16) wgs = 256 * 16;
    hipStream_t stream = (hipStream_t)stream_;
    if (dtype == 0)
        hipLaunchKernelGGL((hstu_silu_bwd_kernel<bf16x8_t>), dim3((unsigned)wgs), dim3(256), 0, stream, (char*)pre, pre_row_stride, (const char*)bias,
                           (const char*)du, du_row_stride, rows, (int)(width / 8));
    else
        hipLaunchKernelGGL((hstu_silu_bwd_kernel<f16x8_t>), dim3((unsigned)wgs), dim3(256), 0, stream, (char*)pre, pre_row_stride, (const char*)bias,
                           (const char*)du, du_row_stride, rows, (int)(width / 8));
    return launch_status("SiLU backward kernel launch");
}

size_t hstu_linear_weight_grad_workspace_bytes(int32_t m, int32_t n, int64_t rows, int64_t a_row_stride, int64_t b_row_stride) {
    if (m <= 0 || n <= 0 || rows <= 0 || a_row_stride < m || b_row_stride < n) return 0;
    const WgradPlan pl = wgrad_plan(m, n, rows, a_row_stride > b_row_stride ? a_row_stride : b_row_stride);
    return pl.partial_bytes + pl.colsum_bytes;
}

int hstu_linear_weight_grad(const void* a, int64_t a_row_stride, int32_t m, const void* b, int64_t b_row_stride, int32_t n, int64_t rows,
                            int32_t dtype, void* out, void* b_sums, void* workspace, int64_t workspace_bytes, void* stream_) {
    hstu_linear_set_last_error("");
    if (m <= 0 || n <= 0 || (m & 7) != 0 || (n & 7) != 0 || m > 65536 || n > 65536 || rows <= 0 || rows > 0x7fffffffLL) return -5;
    if (a_row_stride < m || b_row_stride < n || a_row_stride > (1 << 22) || b_row_stride > (1 << 22)) return -5;
    if (dtype != 0 && dtype != 1) return -2;
    if (!a || !b || !out || !workspace) return -1;
    if (misaligned({a, b, out, workspace}, {a_row_stride, b_row_stride})) return -4;
    if (workspace_bytes < (int64_t)hstu_linear_weight_grad_workspace_bytes(m, n, rows, a_row_stride, b_row_stride)) return -5;
    const WgradPlan pl = wgrad_plan(m, n, rows, a_row_stride > b_row_stride ? a_row_stride : b_row_stride);
    WgradParams p;
    p.a = (const char*)a, p.b = (const char*)b;
    p.a_rsb = (unsigned)(a_row_stride * 2), p.b_rsb = (unsigned)(b_row_stride * 2);
    p.m = m, p.n = n, p.rows = rows, p.rows_per_split = pl.rows_per_split;
    p.tiles_m = pl.tiles_m, p.tiles_n = pl.tiles_n, p.splits = pl.splits;
    p.partial = (float*)workspace;
    p.colsum = b_sums ? (float*)((char*)workspace + pl.partial_bytes) : nullptr;
    hipStream_t stream = (hipStream_t)stream_;
    if (dtype == 0) return launch_wgrad<Bf16>(p, (__bf16*)out, (__bf16*)b_sums, stream);
    return launch_wgrad<Fp16>(p, (_Float16*)out, (_Float16*)b_sums, stream);
}

}  // extern "C"
