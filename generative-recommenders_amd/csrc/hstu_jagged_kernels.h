// Row copies between two jagged (or dense-per-batch) 2-D tensors and their per-batch concatenation: the data
// format either side of the attention path (cache (+) delta -> full K/V, full -> cache | delta).  Pure byte
// movement, bound by HBM bandwidth; results are bit-identical to an index copy by definition.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace hstu {

struct JaggedCopyParams {
    char* left;
    char* right;
    char* joined;
    int64_t left_rs, right_rs, joined_rs;  // row strides in bytes
    int64_t row_bytes;
    const void* offsets_left;   // NULL = dense: exactly max_len_left rows per batch
    const void* offsets_right;
    int offsets_left_i64, offsets_right_i64;
    int batch;
    int max_len_left, max_len_right;
};

__device__ __forceinline__ int64_t jagged_offset(const void* offsets, int is_i64, int dense_len, int b) {
    if (!offsets) return (int64_t)dense_len * b;
    return is_i64 ? ((const int64_t*)offsets)[b] : (int64_t)((const int*)offsets)[b];
}

// Accesses 0 .. total - 1 of a block by the 256 threads of a workgroup, four of a thread in flight, loads first: the compiler does not move a load over
// a store that might be the same place, and a cold copy needs many bytes in flight.  where(i, src, dst) says what access i is.  Whole rounds are
// unconditional, and a last round has only the accesses it needs, of which a thread's last one is conditional: with four conditional accesses in
// every round a large copy paid for the conditions (32 sequences of 2256 rows of 8 KB 261 us, so 247) and a small block for addresses that nobody used
// (tails of 256 rows of 128 bytes, 32 sequences, 2.3 us, so 2.1).
template <int VEC, class INDEX, class WHERE>
__device__ __forceinline__ void copy_accesses(INDEX total, WHERE&& where) {
    typedef __attribute__((ext_vector_type(4))) int v16;
    typedef std::conditional_t<VEC == 16, v16, std::conditional_t<VEC == 8, int64_t, std::conditional_t<VEC == 4, int, std::conditional_t<VEC == 2, short, char>>>> V;
    auto round = [&](auto count, auto whole, INDEX base) __attribute__((always_inline)) {
        constexpr int N = decltype(count)::value;
        const INDEX last = base + (N - 1) * 256 + threadIdx.x;
        const bool there = decltype(whole)::value || last < total;
        V x[N];
        char* dst[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const char* src;
            where(j < N - 1 ? base + j * 256 + threadIdx.x : there ? last : base, src, dst[j]);  // (past the end: read an access that there is)
            x[j] = *(const V*)src;
        }
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (j < N - 1 || there) *(V*)dst[j] = x[j];
    };
    INDEX base = 0;
    for (; total - base >= 1024; base += 1024) round(std::integral_constant<int, 4>{}, std::true_type{}, base);
    const INDEX left = total - base;
    if (left > 768) round(std::integral_constant<int, 4>{}, std::false_type{}, base);
    else if (left > 512) round(std::integral_constant<int, 3>{}, std::false_type{}, base);
    else if (left > 256) round(std::integral_constant<int, 2>{}, std::false_type{}, base);
    else if (left > 0) round(std::integral_constant<int, 1>{}, std::false_type{}, base);
}

// One workgroup per (batch, block of ROWS joined rows).  joined row r of batch b is left row r if r < len_left(b),
// else right row r - len_left(b); the joined tensor starts batch b at offset_left[b] + offset_right[b].
// SPLIT = false: left, right -> joined (concat_2D_jagged); SPLIT = true: joined -> left, right (split_2D_jagged).
// VEC = bytes moved per thread and access (16, 8, 4, 2 or 1: the largest that divides row_bytes, every stride
// and every base address).  INDEX counts a block's accesses: 32 bits wherever they suffice (a 64-bit division is some hundred instructions).
template <bool SPLIT, int VEC, int ROWS, class INDEX>
__global__ __launch_bounds__(256) void hstu_jagged_copy_kernel(const JaggedCopyParams p) {
    const int b = blockIdx.y;
    const int64_t ol = jagged_offset(p.offsets_left, p.offsets_left_i64, p.max_len_left, b);
    const int64_t orr = jagged_offset(p.offsets_right, p.offsets_right_i64, p.max_len_right, b);
    int64_t len_l = jagged_offset(p.offsets_left, p.offsets_left_i64, p.max_len_left, b + 1) - ol;
    int64_t len_r = jagged_offset(p.offsets_right, p.offsets_right_i64, p.max_len_right, b + 1) - orr;
    const int64_t r0 = (int64_t)blockIdx.x * ROWS;
    if (r0 >= len_l + len_r) return;
    const int64_t r1 = r0 + ROWS < len_l + len_r ? r0 + ROWS : len_l + len_r;
    const INDEX vec_per_row = (INDEX)(p.row_bytes / VEC);
    const INDEX total = (INDEX)(r1 - r0) * vec_per_row;
    copy_accesses<VEC>(total, [&](INDEX i, const char*& src, char*& dst) __attribute__((always_inline)) {
        const INDEX row = i / vec_per_row;
        const int64_t r = r0 + (int64_t)row;
        const int64_t c = (int64_t)(i - row * vec_per_row) * VEC;
        char* part = r < len_l ? p.left + (ol + r) * p.left_rs : p.right + (orr + r - len_l) * p.right_rs;
        char* whole = p.joined + (ol + orr + r) * p.joined_rs;
        src = (SPLIT ? whole : part) + c;
        dst = (SPLIT ? part : whole) + c;
    });
}

// joined[offsets_joined[b+1] - tail_len + i] = tail[b * tail_len + i]: writes a dense block of `tail_len` rows per
// batch over the last rows of every sequence of a jagged tensor, in place.  With a K/V cache kept in the layout
// "history rows, then tail_len spare rows" per sequence this replaces the concatenation of the whole history with
// the new rows by a copy of the new rows alone.  One workgroup per (batch, block of `rows` tail rows); 16 rows of 1 KB
// are one round of four accesses per thread (32 rows in eight rounds of one, a load behind every store, took 3.7 us for 100 rows of each of 5
// sequences where this takes 2.3, 4.6 for 256 rows of each of 32 where this takes 3.7).  The arguments fit 64 bytes: a second line of them,
// fetched from the host's memory, costs 0.3 us.
template <int VEC, class INDEX>
__global__ __launch_bounds__(256) void hstu_jagged_write_tail_kernel(char* joined, int64_t joined_rs, const void* offsets,
                                                                     int offsets_i64, int rows, const char* tail, int64_t tail_rs,
                                                                     int64_t row_bytes, int tail_len) {
    const int b = blockIdx.y;
    const int64_t end = jagged_offset(offsets, offsets_i64, 0, b + 1);
    const int64_t start = jagged_offset(offsets, offsets_i64, 0, b);
    if (end - start < tail_len) return;  // contract: every sequence holds at least tail_len rows
    const int r0 = blockIdx.x * rows;
    if (r0 >= tail_len) return;
    const int r1 = r0 + rows < tail_len ? r0 + rows : tail_len;
    const INDEX vec_per_row = (INDEX)(row_bytes / VEC);
    const INDEX total = (INDEX)(r1 - r0) * vec_per_row;
    const char* const from = tail + ((int64_t)b * tail_len + r0) * tail_rs;
    char* const to = joined + (end - tail_len + r0) * joined_rs;
    copy_accesses<VEC>(total, [&](INDEX i, const char*& src, char*& dst) __attribute__((always_inline)) {
        const INDEX row = i / vec_per_row;
        const int64_t c = (int64_t)(i - row * vec_per_row) * VEC;
        src = from + (int64_t)row * tail_rs + c;
        dst = to + (int64_t)row * joined_rs + c;
    });
}

}  // namespace hstu
