// Several strided copies in one launch: what growing a cache by concatenation moves.  An append operator has three (codes,
// scales, minima), a decode step on the 9-tuple four for its tails and six more when it flushes
// (models/modeling_llama_KVmix.py:117-118,134-139,162-167); one by one each costs a launch for a few megabytes.
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

// Bound by HBM.  A thread moves four 16-byte pieces, all read before the first is written; neighbouring threads have
// neighbouring pieces of a row.  Rows start where the concatenation puts them (scales: any multiple of two bytes), so the
// accesses are unaligned ones; the last piece of a row is moved back to end with it, and what it shares with its
// neighbour is written twice with the same bytes.  Rows shorter than a piece go two bytes at a time.
// Measured (both append operators on 2304 cached tokens, batch 4, 2-bit keys and 4-bit values: 78 MB read and written):
// six copies and two quantizers 40 us of GPU time and 69 per call with their launches, two and two 28 per call.
__global__ void __launch_bounds__(kCopyThreads) copy_rows(CopyArgs a)
{
    int i = 0;
    while (i + 1 < a.count && blockIdx.x >= a.first[i + 1]) i++;
    const CopyItem &it = a.item[i];
    const uint32_t p0 = (blockIdx.x - a.first[i]) * (kCopyThreads * kCopyPieces) + threadIdx.x;
    const int64_t last = it.row_bytes - 16;
    uint4u v[kCopyPieces];
    uint8_t *to[kCopyPieces];
#pragma unroll
    for (int u = 0; u < kCopyPieces; u++) {
        const uint32_t p = p0 + u * kCopyThreads < it.pieces ? p0 + u * kCopyThreads : it.pieces - 1;
        const uint32_t row = copy_div(p, it.per_row), o = copy_div(row, it.inner);
        const int64_t at = (int64_t)(p - row * it.per_row.d) * 16, r = row - o * it.inner.d;
        const uint8_t *from = it.src + o * it.src_os + r * it.src_is;
        to[u] = it.dst + o * it.dst_os + r * it.dst_is;
        if (last >= 0) {
            from += at < last ? at : last;
            to[u] += at < last ? at : last;
            v[u] = *(const uint4u *)from;
        } else {
            for (int64_t b = 0; b < it.row_bytes; b += 2) *(uint16_t *)(to[u] + b) = *(const uint16_t *)(from + b);
        }
    }
    if (last < 0) return;
#pragma unroll
    for (int u = 0; u < kCopyPieces; u++) *(uint4u *)to[u] = v[u];
}

namespace {

CopyDiv copy_divisor(uint32_t d)
{
    int s = 0;
    while ((1ull << s) < d) s++;
    CopyDiv c;
    c.d = d;
    c.shift = 31 + s;
    c.mul = (uint32_t)(((1ull << (31 + s)) + d - 1) / d);
    return c;
}

}  // namespace
}  // namespace kvmix

using namespace kvmix;

extern "C" int kvmix_copy_rows(const kvmix_copy_rows_t *items, int count, kvmix_stream_t stream)
{
    if (count < 0) return KVMIX_ERR_SHAPE;
    if (count == 0) return KVMIX_OK;
    if (!items) return KVMIX_ERR_NULL;
    for (int i = 0; i < count; i++) {  // everything is checked before anything is launched
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
    CopyArgs a;
    a.count = 0;
    a.first[0] = 0;
    auto launch = [&]() {
        if (a.count == 0) return KVMIX_OK;
        copy_rows<<<dim3(a.first[a.count]), kCopyThreads, 0, (hipStream_t)stream>>>(a);
        a.count = 0;
        return launch_status();
    };
    for (int i = 0; i < count; i++) {
        const kvmix_copy_rows_t &p = items[i];
        if (p.outer == 0 || p.inner == 0 || p.row_bytes == 0) continue;
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
        if (++a.count == kCopyItems) {
            const int rc = launch();
            if (rc != KVMIX_OK) return rc;
        }
    }
    return launch();
}
