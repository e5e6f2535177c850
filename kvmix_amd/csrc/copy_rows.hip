// Several strided copies in one launch: what growing a cache by concatenation moves.  An append operator has three (codes,
// scales, minima), a decode step on the 9-tuple four for its tails and six more when it flushes
// (models/modeling_llama_KVmix.py:117-118,134-139,162-167); one by one each costs a launch for a few megabytes.
#include "copy_rows.h"

namespace kvmix {

// Bound by HBM; what a block does is copy_block (copy_rows.h).
// Measured (the copies of both append operators on 2304 cached tokens, batch 4, 2-bit keys and 4-bit values: 78 MB read and
// written): three copies each 40 us of GPU time with the quantizers, one launch each 24.5 (beside the quantizers: grow_kv_flush).
__global__ void __launch_bounds__(kCopyThreads) copy_rows(CopyArgs a)
{
    copy_block(a, blockIdx.x);
}

}  // namespace kvmix

using namespace kvmix;

extern "C" int kvmix_copy_rows(const kvmix_copy_rows_t *items, int count, kvmix_stream_t stream)
{
    const int chk = copy_check(items, count);
    if (chk != KVMIX_OK) return chk;
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
        if (copy_is_empty(items[i])) continue;
        copy_add(a, items[i]);
        if (a.count == kCopyItems) {
            const int rc = launch();
            if (rc != KVMIX_OK) return rc;
        }
    }
    return launch();
}
