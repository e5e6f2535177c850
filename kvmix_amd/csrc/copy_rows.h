// Strided copies as blocks of a launch: the copy kernel's own (copy_rows.hip) and those that run beside the quantizers when a
// cache grows (quant_pack.hip).
#pragma once

#include "kvmix_common.h"


namespace kvmix {

constexpr int kCopyItems = 16;     // copies per launch
constexpr int kCopyPieces = 4;     // 16-byte pieces per thread
constexpr int kCopyThreads = 256;

// n / d for n < 2^31: (n * mul) >> shift, exact
struct CopyDiv {
    uint32_t d, mul, shift;
};

struct CopyItem {
    const uint8_t *src;
    uint8_t *dst;
    int64_t src_os, src_is, dst_os, dst_is;  // bytes
    int64_t row_bytes;
    uint32_t pieces;                         // in all
    CopyDiv per_row, inner;                  // pieces per row, rows per outer slice
};

struct CopyArgs {
    CopyItem item[kCopyItems];
    uint32_t first[kCopyItems + 1];          // first block of each item
    int count;
};

typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(2)));

__device__ __forceinline__ uint32_t copy_div(uint32_t n, const CopyDiv &c)
{
    return (uint32_t)(((uint64_t)n * c.mul) >> c.shift);
}

// Block `block` of the copies: a thread moves four 16-byte pieces, all read before the first is written; neighbouring
// threads have neighbouring pieces of a row.  Rows start where the concatenation puts them (scales: any multiple of two
// bytes), so the accesses are unaligned ones; the last piece of a row is moved back to end with it, and what it shares
// with its neighbour is written twice with the same bytes.  Rows shorter than a piece go two bytes at a time.
__device__ __forceinline__ void copy_block(const CopyArgs &a, uint32_t block)
{
    int i = 0;
    while (i + 1 < a.count && block >= a.first[i + 1]) i++;
    const CopyItem it = a.item[i];  // (by value: read before the first store)
    const uint32_t p0 = (block - a.first[i]) * (kCopyThreads * kCopyPieces) + threadIdx.x;
    const int64_t last = it.row_bytes - 16;
    const uint8_t *from[kCopyPieces];
    uint8_t *to[kCopyPieces];
#pragma unroll
    for (int u = 0; u < kCopyPieces; u++) {
        const uint32_t p = p0 + u * kCopyThreads < it.pieces ? p0 + u * kCopyThreads : it.pieces - 1;
        const uint32_t row = copy_div(p, it.per_row), o = copy_div(row, it.inner);
        const int64_t at = (int64_t)(p - row * it.per_row.d) * 16, r = row - o * it.inner.d;
        const int64_t in = last < 0 ? 0 : (at < last ? at : last);
        from[u] = it.src + o * it.src_os + r * it.src_is + in;
        to[u] = it.dst + o * it.dst_os + r * it.dst_is + in;
    }
    if (last < 0) {
        for (int u = 0; u < kCopyPieces; u++) {
            for (int64_t b = 0; b < it.row_bytes; b += 2) *(uint16_t *)(to[u] + b) = *(const uint16_t *)(from[u] + b);
        }
        return;
    }
    uint4u v[kCopyPieces];
#pragma unroll
    for (int u = 0; u < kCopyPieces; u++) v[u] = *(const uint4u *)from[u];
#pragma unroll
    for (int u = 0; u < kCopyPieces; u++) *(uint4u *)to[u] = v[u];
}

inline CopyDiv copy_divisor(uint32_t d)
{
    int s = 0;
    while ((1ull << s) < d) s++;
    CopyDiv c;
    c.d = d;
    c.shift = 31 + s;
    c.mul = (uint32_t)(((1ull << (31 + s)) + d - 1) / d);
    return c;
}

// everything is checked before anything is launched
inline int copy_check(const kvmix_copy_rows_t *items, int count)
{
    if (count < 0) return KVMIX_ERR_SHAPE;
    if (count > 0 && !items) return KVMIX_ERR_NULL;
    for (int i = 0; i < count; i++) {
        const kvmix_copy_rows_t &p = items[i];
        if (p.outer < 0 || p.inner < 0 || p.row_bytes < 0 || p.row_bytes % 2 != 0) return KVMIX_ERR_SHAPE;
        if (p.outer == 0 || p.inner == 0 || p.row_bytes == 0) continue;
        if (!p.src || !p.dst) return KVMIX_ERR_NULL;
        if (((uintptr_t)p.src | (uintptr_t)p.dst | (uintptr_t)p.src_outer_stride | (uintptr_t)p.src_inner_stride |
             (uintptr_t)p.dst_outer_stride | (uintptr_t)p.dst_inner_stride) % 2 != 0)
            return KVMIX_ERR_SHAPE;
        if (p.dst_inner_stride < p.row_bytes && p.inner > 1) return KVMIX_ERR_SHAPE;
        if (p.outer > (1ll << 31) || p.inner > (1ll << 31) || p.row_bytes > (1ll << 40)) return KVMIX_ERR_UNSUPPORTED;
        const __int128 pieces = (__int128)p.outer * p.inner * ((p.row_bytes + 15) / 16);
        if (pieces > 0x7fffffff - kCopyThreads * kCopyPieces) return KVMIX_ERR_UNSUPPORTED;
    }
    return KVMIX_OK;
}

inline bool copy_is_empty(const kvmix_copy_rows_t &p) { return p.outer == 0 || p.inner == 0 || p.row_bytes == 0; }

// one more copy of a launch (there is room for kCopyItems)
inline void copy_add(CopyArgs &a, const kvmix_copy_rows_t &p)
{
    int64_t inner = p.inner, outer = p.outer, row = p.row_bytes;
    if (p.src_inner_stride == row && p.dst_inner_stride == row) {  // rows that follow one another on both sides are one
        row *= inner;
        inner = 1;
        if (p.src_outer_stride == row && p.dst_outer_stride == row) {
            row *= outer;
            outer = 1;
        }
    }
    CopyItem &it = a.item[a.count];
    it.src = (const uint8_t *)p.src;
    it.dst = (uint8_t *)p.dst;
    it.src_os = p.src_outer_stride;
    it.src_is = p.src_inner_stride;
    it.dst_os = p.dst_outer_stride;
    it.dst_is = p.dst_inner_stride;
    it.row_bytes = row;
    it.per_row = copy_divisor((uint32_t)((row + 15) / 16));
    it.inner = copy_divisor((uint32_t)inner);
    it.pieces = (uint32_t)(outer * inner) * it.per_row.d;
    a.first[a.count + 1] = a.first[a.count] + (it.pieces + kCopyThreads * kCopyPieces - 1) / (kCopyThreads * kCopyPieces);
    a.count++;
}

}  // namespace kvmix
