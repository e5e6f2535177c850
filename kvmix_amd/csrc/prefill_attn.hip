// Dense attention of a prompt: out = softmax(q k^T / sqrt(D) + mask) v, fp16 operands, fp32 logits, softmax and sums, no
// [Q, T] matrix in memory.  It is the prompt branch of the attention layer where nobody reads the probabilities
// (models/modeling_llama_KVmix.py:252-266); query head h reads kv head h / heads_per_kv, nothing is repeated.
//
// The mask is any additive [1 or batch, 1 or heads, Q, T] tensor, fp32 or fp16.  It is taken as the prompt branch takes
// it: clamped below at the lowest finite half and rounded to fp16, added in fp32; a row in which everything is masked
// weighs all its positions alike.  prefill_mask_classes reads it once and sorts the tiles of 32 queries by 64 keys into
// skipped (everything masked), plain (all zero), binary (entries masked or zero: one bit each is kept) and mixed; the
// attention kernel never loads the first, needs no mask for the second, eight bytes per query for the third and adds the
// mask itself in the last only, so that a causal or padding mask costs half the products and next to no reads.
// A skipped position weighs exp(l - l' - 65504) against some position of its row: zero as long as the row's largest mask
// entry is above -30000 (rows where it is not have no skipped tiles) and the logits differ by less than 35000; q.k of
// more than 65504 = 5800 sqrt(128) is an infinity in the reference's own half-precision logits.
#include "kvmix_common.h"

namespace kvmix {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2 __attribute__((ext_vector_type(2)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 half4u __attribute__((ext_vector_type(4), aligned(2)));

constexpr int kPreWaves = 4;  // 32 queries each
constexpr int kPreK = 64;     // keys per tile
constexpr int kClassWaves = 16;
constexpr int kClassCols = 4 * kWave;  // columns a wave reads per row and load
constexpr float kHalfLowest = -65504.0f;
constexpr float kLog2e = 1.44269504088896340736f;
enum { kTileSkip = 0, kTilePlain = 1, kTileMixed = 2, kTileBinary = 3 };
enum { kHasLive = 1, kHasOther = 2, kHasMixed = 4 };  // some entry not masked, not zero, neither
constexpr int kClassChunk = 2 * kClassCols;           // columns of a block of prefill_mask_classes
constexpr int64_t kMaxClassBlocks = 65535;            // ... and such blocks along a row

struct PrefillArgs {
    const _Float16 *q, *k, *v;
    _Float16 *out;
    int64_t q_bs, q_hs, q_ts, k_bs, k_hs, k_ts, v_bs, v_hs, v_ts, o_bs, o_hs, o_ts;
    const void *mask;
    int mask_f32;
    int64_t m_bs, m_hs, m_rs;
    int flag_b, flag_h;        // mask slice of (batch b, head h): b * flag_b + h * flag_h
    const uint8_t *flags;      // [mask slices][key tiles][query parts]: what the tile of a part's 32 queries holds (kHas*)
    const uint2 *rows;         // [mask slices][query parts][chunks]: bit per query, with an entry not `absorbed` (x), of at least -30000 (y)
    const uint64_t *bits;      // [mask slices][query parts][key tiles][32 queries]: bit 16 j + i = key 4 i + j is masked
    int heads, heads_per_kv, q_len, kv_len, q_tiles, k_tiles, parts, chunks;  // parts: 32 queries each, whole blocks of them
    float scale;
    int far;                   // a tile's rows lie too far apart for 32-bit offsets
};

__device__ __forceinline__ float prefill_mask_value(float v)
{
    v = v < kHalfLowest ? kHalfLowest : v;  // (a NaN stays one)
    return (float)(_Float16)v;
}

// entries [col, col + 4) of a mask row; what lies at or past `cols` is not read and comes back as `beyond`
template <typename T>
__device__ __forceinline__ void mask_four(const T *row, int col, int cols, float beyond, float *v)
{
    if (col + 4 <= cols) {
        if constexpr (sizeof(T) == 4) {
            const float4u w = *(const float4u *)(row + col);
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = w[j];
        } else {
            const half4u w = *(const half4u *)(row + col);
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = (float)w[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = col + j < cols ? (float)row[col + j] : beyond;
    }
}

// What the tiles of 32 queries by 64 keys hold, eight tiles to a block, and per query whether these columns have an entry above
// `absorbed` (x) and one of at least -30000 (y); attention makes the classes out of both.  Bound by the ballots (twenty
// instructions per entry and lane) and by the latency of one round of loads: two rows per wave, two loads of each in flight.
// With whole rows to a block a mask of 2048 x 2048 kept 64 CUs busy and the rest idle (B = 4, 32 heads, T = 512, one round of
// blocks, with attention: 37.3 -> 35.0 us; B = 1, T = 4096 213 -> 202).
template <typename T>
__global__ void __launch_bounds__(kClassWaves * kWave) prefill_mask_classes(PrefillArgs a, uint64_t *bits, uint8_t *flags, uint2 *rows,
                                                                             int64_t mask_heads)
{
    constexpr int TILES = kClassChunk / kPreK;
    __shared__ uint32_t tile_bits[TILES];  // per key tile: kHas*
    __shared__ uint32_t row_bits[2];       // rows with an entry above `absorbed`, rows with an entry of at least -30000
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int64_t slice = blockIdx.y;
    const int r0 = blockIdx.x * 32, valid = a.q_len - r0 < 32 ? a.q_len - r0 : 32;
    const T *base = (const T *)a.mask + (slice / mask_heads) * a.m_bs + (slice % mask_heads) * a.m_hs;
    // what the prompt branch takes for a row masked everywhere: see KVmixAttention._prompt_attention
    const float absorbed = sizeof(T) == 2 ? kHalfLowest : -1e30f;
    if (threadIdx.x < TILES) tile_bits[threadIdx.x] = 0;
    if (threadIdx.x < 2) row_bits[threadIdx.x] = 0;
    const int c0 = blockIdx.z * kClassChunk, tile0 = c0 / kPreK;
    float v[2][2][4];
#pragma unroll
    for (int u = 0; u < 2; u++) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int row = 2 * wave + r;
            mask_four(base + (int64_t)(r0 + row < a.q_len ? r0 + row : a.q_len - 1) * a.m_rs, c0 + u * kClassCols + 4 * lane, a.kv_len,
                      0.0f, v[u][r]);
        }
    }
    __syncthreads();
    uint32_t live[2] = {0, 0}, tight[2] = {0, 0};
    uint64_t *tile_rows = bits + (slice * a.parts + blockIdx.x) * a.k_tiles * 32;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int col = c0 + u * kClassCols + 4 * lane;
        const int tile = tile0 + u * (kClassCols / kPreK) + lane / 16;
        uint32_t some = 0, other = 0, neither = 0;
#pragma unroll
        for (int r = 0; r < 2; r++) {
            uint64_t masked = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float m = v[u][r][j];
                masked |= (__ballot(m <= kHalfLowest) >> (lane & 48) & 0xffff) << (16 * j);
                const uint32_t in = col + j < a.kv_len && 2 * wave + r < valid ? 1 : 0;
                some |= m <= kHalfLowest ? 0 : in;
                other |= m == 0.0f ? 0 : in;
                neither |= m == 0.0f || m <= kHalfLowest ? 0 : in;
                live[r] |= m <= absorbed ? 0 : in;
                tight[r] |= m < -30000.0f ? 0 : in;
            }
            if (lane % 16 == 0 && tile < a.k_tiles) tile_rows[(int64_t)tile * 32 + 2 * wave + r] = masked;
        }
        const uint64_t s = __ballot(some != 0), o = __ballot(other != 0), n = __ballot(neither != 0);
        if (lane % 16 == 0 && tile < a.k_tiles) {
            const uint32_t kinds = ((s >> lane) & 0xffff ? kHasLive : 0u) | ((o >> lane) & 0xffff ? kHasOther : 0u) | ((n >> lane) & 0xffff ? kHasMixed : 0u);
            if (kinds) atomicOr(&tile_bits[tile - tile0], kinds);
        }
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const bool l = __ballot(live[r] != 0) != 0, t = __ballot(tight[r] != 0) != 0;
        if (lane == 0) {
            if (l) atomicOr(&row_bits[0], 1u << (2 * wave + r));
            if (t) atomicOr(&row_bits[1], 1u << (2 * wave + r));
        }
    }
    __syncthreads();
    if (threadIdx.x < TILES && tile0 + (int)threadIdx.x < a.k_tiles)
        flags[(slice * a.k_tiles + tile0 + threadIdx.x) * (int64_t)a.parts + blockIdx.x] = (uint8_t)tile_bits[threadIdx.x];
    if (threadIdx.x == 0) rows[(slice * a.parts + blockIdx.x) * a.chunks + blockIdx.z] = make_uint2(row_bits[0], row_bits[1]);
}

// The class of a tile of 32 queries of which `rows` exist: `loose`: some row has no entry of at least -30000 (no tile may be
// skipped then), `all_dead`: every row is masked everywhere (with queries of zero all positions count alike).
__device__ __forceinline__ uint32_t tile_class(uint32_t has, bool loose, bool all_dead, bool any_row)
{
    const uint32_t c = has & kHasMixed ? kTileMixed : (has & kHasOther ? kTileBinary : kTilePlain);
    return !any_row ? (uint32_t)kTileSkip : all_dead ? (uint32_t)kTilePlain : !(has & kHasLive) && !loose ? (uint32_t)kTileSkip : c;
}

// LDS layouts, both [64][D] as loaded, the 16-byte pieces of a row exchanged by the row's low bits so that the reading side
// is free of bank conflicts: keys are read a piece per lane, sixteen rows at a time, values transposed (ds_read_tr), sixteen
// lanes taking 4 rows of 16 dimensions.
template <int D>
__device__ __forceinline__ int key_piece(int key, int c)
{
    return D == 128 ? key * 256 + ((c ^ (key & 15)) << 4) : key * 128 + ((c ^ ((key >> 1) & 7)) << 4);
}

template <int D>
__device__ __forceinline__ int value_piece(int key, int c)
{
    return D == 128 ? key * 256 + ((c ^ ((key & 3) << 2)) << 4) : key * 128 + ((c ^ (((key >> 1) & 1) << 2)) << 4);
}

// Four values of a lane's column out of rows of 16 halves: each lane of sixteen names its quarter of one of four rows.
typedef short short4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ half4 read_transposed(const uint8_t *at)
{
    return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4 *)at));
}

// One block: 128 queries of one head, 32 to a wave, over the key tiles that some of them needs.  Bound by the matrix cores and
// the vector ALU beside them (exponentials, conversions, rescaling: 230 instructions per wave and tile; both together fill
// 95 % of the cycles), so everything else is kept off that path.  The logits are computed transposed (32x32x16, keys as
// rows): a lane then holds 32 logits of ONE query, the softmax needs a single exchange between the two halves of a wave, and
// the probabilities are already the right-hand operand of out^T = v^T p^T.  The mask's entries are added to the finished
// logits (sums that start from them round at their size at every step: 2.5 times the error under a mask of -10000).  Keys
// and values go from memory straight to LDS, a tile ahead of the products, from one offset per lane and addresses that are
// the same for a wave (a row's address per piece took 66 instructions per tile, a third of them at a quarter of the rate);
// values are transposed by the reads that take them (ds_read_tr), not on the way through registers (16 of them, 46
// instructions, 8 stores with bank conflicts: 26 % of the LDS's cycles).  Two blocks share a CU.  Reading operands a step
// or two ahead of their products, fewer scheduling barriers and wave priorities changed nothing (353 -> 345..356 us without
// a mask); eight waves on 256 queries lose more to the causal border than they save in reads.
// Measured (us per call with the mask's classes, causal fp32 mask; values through registers and head after head -> now): B =
// 4, 32 heads, T = 2048 316 -> 236 (without a mask 420 -> 353, 780 TFLOP/s); B = 1, T = 4096 291 -> 202; B = 4, T = 512 46 -> 35;
// 32 / 8 heads: B = 4, T = 2048 358 -> 256, B = 1, T = 1001 58 -> 46.  A mask that is mixed in every tile (a bias per
// distance below the diagonal), B = 2, 32 heads, T = 2048: 283 -> 176.  Error against float64 relative to the norm, keys with
// an outlier channel, causal, T = 300 / 1500 / 2048: 2.35 / 2.37 / 2.41e-4; with the maximum moved from 2^8 on only 2.40 /
// 2.52 / 2.59e-4 (238 us).
template <int D, bool SPLIT>
__global__ void __launch_bounds__(kPreWaves * kWave) __attribute__((amdgpu_waves_per_eu(2, 2))) prefill_attn(PrefillArgs a)
{
    constexpr int W = kPreWaves;
    constexpr int KS = D / 16, DT = D / 32, CPR = D / 8;   // k-steps of q.k^T, 32-row tiles of out^T, pieces per row
    constexpr int KL = kPreK * CPR / (W * kWave);  // key pieces a thread moves per tile
    constexpr int kTileBytes = kPreK * D * 2;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2][2][kTileBytes];
    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave), col = lane & 31, h2 = lane >> 5;

    // Under a mask the longest (causal) query tiles of all heads first, so that the blocks that end a launch are short ones;
    // blocks are dealt to the XCDs in turn, and neighbouring heads stay on one (its L2 then holds what they share).  Head
    // after head left a last head whose long tiles ran on alone: B = 4, 32 heads, T = 2048 260 -> 239 us, a bias per distance
    // 248 -> 173.  Without a mask all blocks are alike, and the query tiles of one head after the other share more (363 against
    // 377 us).
    const uint32_t n = gridDim.x, l = blockIdx.x, xcd = l % 8, per = n / 8, rem = n % 8, q_tiles = a.q_tiles, heads = n / q_tiles, nth = l % heads;
    const uint32_t job = xcd * per + (xcd < rem ? xcd : rem) + l / 8;
    const int qt = (int)(q_tiles - 1 - (a.flags ? l / heads : job % q_tiles));
    const uint32_t bh = !a.flags ? job / q_tiles : heads % 8 == 0 ? nth % 8 * (heads / 8) + nth / 8 : nth;
    const int b = (int)(bh / (uint32_t)a.heads), head = (int)(bh % (uint32_t)a.heads);
    const _Float16 *kp = a.k + b * a.k_bs + (head / a.heads_per_kv) * a.k_hs;
    const _Float16 *vp = a.v + b * a.v_bs + (head / a.heads_per_kv) * a.v_hs;
    const int64_t slice = (int64_t)b * a.flag_b + (int64_t)head * a.flag_h;
    const uint32_t *flags = a.flags ? (const uint32_t *)(a.flags + slice * a.k_tiles * a.parts) + qt : nullptr;  // a byte per wave
    const int flag_step = a.parts / W;

    const int query = (qt * W + wave) * 32 + col, row = query < a.q_len ? query : a.q_len - 1;
    half8 qv[KS];
    {
        const _Float16 *qp = a.q + b * a.q_bs + head * a.q_hs + (int64_t)row * a.q_ts + 8 * h2;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) qv[ks] = *(const half8 *)(qp + 16 * ks);
    }
    // per part of the block: whether it has rows, is loose or all dead (tile_class), the same in all lanes
    uint32_t part_kind = 0;
    if (a.flags) {
        uint32_t live = 0, tight = 0;
        const uint2 *rows = a.rows + (slice * a.parts + qt * W + (lane & (W - 1))) * a.chunks;
        for (int i = 0; i < a.chunks; i++) live |= rows[i].x, tight |= rows[i].y;
        const int valid = a.q_len - (qt * W + (lane & (W - 1))) * 32;
        const uint32_t mine = valid <= 0 ? 0 : valid >= 32 ? 0xffffffffu : (1u << valid) - 1;
        const uint64_t any_row = __ballot(mine != 0), loose = __ballot((tight & mine) != mine), all_dead = __ballot((live & mine) == 0);
        part_kind = (uint32_t)(any_row & 15) | (uint32_t)(loose & 15) << 4 | (uint32_t)(all_dead & 15) << 8;
        const uint32_t wave_live = __builtin_amdgcn_readlane(live, wave);  // (lanes 0..3: the block's parts)
        if (!(wave_live >> (row & 31) & 1)) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) qv[ks] = half8{};
        }
    }

    // the key tiles that some query of the block needs, in order
    int window = -kWave;
    uint64_t pending = 0;
    uint32_t classes = 0, cls = 0;
    auto next_tile = [&]() -> int {
        while (pending == 0) {
            window += kWave;
            if (window >= a.k_tiles) return -1;
            const int t = window + lane;
            classes = 0x01010101u;
            if (flags && t < a.k_tiles) {
                const uint32_t has = flags[(int64_t)t * flag_step];
                classes = 0;
#pragma unroll
                for (int w = 0; w < W; w++)
                    classes |= tile_class(has >> (8 * w), part_kind >> (4 + w) & 1, part_kind >> (8 + w) & 1, part_kind >> w & 1) << (8 * w);
            }
            classes = t < a.k_tiles ? classes : 0;
            pending = __ballot(classes != 0);
        }
        const int bit = __builtin_ctzll(pending);
        pending &= pending - 1;
        cls = __builtin_amdgcn_readlane(classes, bit);
        return window + bit;
    };

    // Pieces of a tile go from memory straight to LDS, where a wave's 64 lie one after the other: lane by lane the one that
    // belongs there.  Instructions of a tile are 64 * W / CPR rows apart, a multiple of what the pieces are exchanged by, so
    // a lane has one offset for all of them and the rest of an address is the same for the wave.
    constexpr int STEP = W * kWave / CPR;  // rows between a thread's pieces
    const int own_row = tid / CPR, own_k = key_piece<D>(own_row, tid % CPR) >> 4, own_v = value_piece<D>(own_row, tid % CPR) >> 4;
    const uint32_t k_off = (uint32_t)(own_row * (int)a.k_ts + (own_k % CPR) * 8), v_off = (uint32_t)(own_row * (int)a.v_ts + (own_v % CPR) * 8);
    auto to_lds = [&](const _Float16 *from, uint8_t *to) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from, (__attribute__((address_space(3))) void *)to, 16, 0, 0);
    };
    auto load_tile = [&](int t, int into) {
        const int k0 = t * kPreK;
        uint8_t *k_to = lds[into][0] + wave * kWave * 16, *v_to = lds[into][1] + wave * kWave * 16;
        if (__builtin_expect(k0 + kPreK <= a.kv_len && !a.far, 1)) {
            const _Float16 *kb = kp + (int64_t)k0 * a.k_ts, *vb = vp + (int64_t)k0 * a.v_ts;
#pragma unroll
            for (int i = 0; i < KL; i++) {
                to_lds(kb + k_off, k_to + i * W * kWave * 16);
                to_lds(vb + v_off, v_to + i * W * kWave * 16);
                kb += STEP * a.k_ts, vb += STEP * a.v_ts;
            }
        } else {  // rows past the end repeat the last one
            const int last = a.kv_len - 1;
#pragma unroll
            for (int i = 0; i < KL; i++) {
                const int64_t key = min(k0 + own_row + i * STEP, last);
                to_lds(kp + key * a.k_ts + (own_k % CPR) * 8, k_to + i * W * kWave * 16);
                to_lds(vp + key * a.v_ts + (own_v % CPR) * 8, v_to + i * W * kWave * 16);
            }
        }
    };
    // (... of the values zeros: weight zero times an infinite one is NaN.  Behind the wait for the tile and a barrier.)
    auto clear_past_end = [&](int t, int buf) {
        if (__builtin_expect((t + 1) * kPreK > a.kv_len, 0)) {
            for (int i = tid; i < kTileBytes / 16; i += W * kWave) {
                if (t * kPreK + i / CPR >= a.kv_len) *(half8 *)(lds[buf][1] + i * 16) = half8{};
            }
            __syncthreads();
        }
    };

    // a lane's pieces of the first 32 rows: step ks, kk is the piece at an exclusive or with 32 bytes times the step
    const int k_at = key_piece<D>(col, h2);
    // ... and a lane's place in the transposed reads of the values: row (lane % 16) / 4 of four, four dimensions of sixteen;
    // dimension tile t is at an exclusive or with 64 bytes times the tile
    const int v_at = value_piece<D>(4 * h2 + (lane & 15) / 4, 2 * ((lane >> 4) & 1) + (lane & 3) / 2) + (lane & 1) * 8;

    floatx16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++) o[t] = floatx16{};
    float m = -1e30f, sum = 0.0f;  // in units of log2 (a finite start: a tile of logits of -inf weighs zero)
    const float c = a.scale * kLog2e, unscale = 1.0f / a.scale;

    int tile = next_tile(), buf = 0;
    if (tile >= 0) load_tile(tile, 0);
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (tile >= 0) clear_past_end(tile, 0);
    while (tile >= 0) {
        const int k0 = tile * kPreK, mine = (int)(cls >> (8 * wave)) & 255;
        uint64_t masked = 0;
        if (mine == kTileBinary)
            masked = a.bits[((slice * a.parts + qt * W + wave) * a.k_tiles + tile) * 32 + col] >> h2;
        const int next = next_tile();
        if (next >= 0) load_tile(next, buf ^ 1);  // (that buffer was last read before the barrier that ended the iteration before)
        if (mine != kTileSkip) {
            // logits, transposed: a lane has keys 8 (i / 4) + 4 h2 + i % 4 of two times 32 for its one query
            floatx16 s[2] = {floatx16{}, floatx16{}};
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const half8 kk = *(const half8 *)(lds[buf][0] + (k_at ^ (ks << 5)) + t * 32 * 2 * D);
                    s[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kk, qv[ks], s[t], 0, 0, 0);
                }
                if (ks % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (all reads of a tile ahead of its products would spill)
            }
            // the mask's entries, divided by the scale that follows, are added to the finished sums: one rounding at their size
            if (mine == kTileBinary && k0 + kPreK <= a.kv_len) {
                const uint32_t word[2] = {(uint32_t)masked, (uint32_t)(masked >> 32)};
#pragma unroll
                for (int i = 0; i < 32; i++) {
                    const int bit = 16 * (i % 4) + 8 * (i / 16) + 2 * (i % 16 / 4);
                    s[i / 16][i % 16] += word[bit / 32] >> (bit % 32) & 1 ? kHalfLowest * unscale : 0.0f;
                }
            } else if (mine != kTilePlain) {
                int r = query;  // (what follows from it is not kept across the tiles)
                asm volatile("" : "+v"(r));
                const int64_t mask_row = b * a.m_bs + head * a.m_hs + (int64_t)(r < a.q_len ? r : a.q_len - 1) * a.m_rs;
                auto add_mask = [&](const auto *entries) {
#pragma unroll
                    for (int g = 0; g < 8; g++) {
                        float v[4];
                        mask_four(entries + mask_row, k0 + 32 * (g / 4) + 8 * (g % 4) + 4 * h2, a.kv_len, 0.0f, v);
#pragma unroll
                        for (int j = 0; j < 4; j++) s[g / 4][4 * (g % 4) + j] += prefill_mask_value(v[j]) * unscale;
                        __builtin_amdgcn_sched_barrier(0);  // (a load at a time: more would spill, and took longer)
                    }
                };
                if (a.mask_f32) add_mask((const float *)a.mask);
                else add_mask((const _Float16 *)a.mask);
            }
            if (k0 + kPreK > a.kv_len) {
#pragma unroll
                for (int i = 0; i < 32; i++) {
                    if (k0 + 32 * (i / 16) + 8 * (i % 16 / 4) + 4 * h2 + i % 4 >= a.kv_len) s[i / 16][i % 16] = -__builtin_inff();
                }
            }
            float top = s[0][0];
#pragma unroll
            for (int t = 0; t < 2; t++) {
#pragma unroll
                for (int i = 0; i < 16; i++) top = fmaxf(top, s[t][i]);
            }
            {
                const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(top), __float_as_uint(top), false, false);
                top = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * c;
            }
            // With probabilities in two parts the maximum is only moved when it has grown by more than 2^8: below that they
            // stay well inside fp16's range, and rescaling the 64 sums of a lane costs a quarter of a tile's products.  In
            // one part the largest has to be exactly one, or its rounding is the largest error of the row.
            if (__any(top > (SPLIT ? m + 8.0f : m))) {
                const float grown = fmaxf(m, top);
                const float shrink = __builtin_amdgcn_exp2f(m - grown);
                m = grown;
                sum *= shrink;
#pragma unroll
                for (int t = 0; t < DT; t++) o[t] *= shrink;
            }
            half8 ph[2], pl[2];
            auto probs = [&](int kk) {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float p = __builtin_amdgcn_exp2f(fmaf(s[kk / 2][8 * (kk % 2) + i], c, -m));
                    const _Float16 hi = (_Float16)p;
                    ph[kk % 2][i] = hi;
                    if constexpr (SPLIT) {
                        sum += p;
                        pl[kk % 2][i] = (_Float16)(p - (float)hi);
                    } else if (i % 2) {  // the sum of what the products weigh with: a common part of the roundings drops out
                        sum = __builtin_amdgcn_fdot2(half2{ph[kk % 2][i - 1], hi}, half2{(_Float16)1.0f, (_Float16)1.0f}, sum, false);
                    }
                }
            };
            probs(0);
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {  // (a step's probabilities between the products of the one before)
#pragma unroll
                for (int t = 0; t < DT; t++) {
                    const uint8_t *at = lds[buf][1] + (v_at ^ (t << 6)) + kk * 16 * 2 * D;
                    const half4 v0 = read_transposed(at), v1 = read_transposed(at + 8 * 2 * D);
                    const half8 vv = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
                    o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vv, ph[kk % 2], o[t], 0, 0, 0);
                    if constexpr (SPLIT) o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vv, pl[kk % 2], o[t], 0, 0, 0);
                }
                if (kk < 3) probs(kk + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        buf ^= 1;
        __builtin_amdgcn_s_waitcnt(0x0f70);  // the pieces on their way to LDS (vmcnt 0)
        __syncthreads();
        if (next >= 0) clear_past_end(next, buf);
        tile = next;
    }
    if (query >= a.q_len) return;
    {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
        sum = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    const float inv = 1.0f / sum;
    _Float16 *op = a.out + b * a.o_bs + head * a.o_hs + (int64_t)query * a.o_ts + 4 * h2;
#pragma unroll
    for (int t = 0; t < DT; t++) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            half4 w;
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = (_Float16)(o[t][4 * g + j] * inv);
            *(half4 *)(op + 32 * t + 8 * g) = w;
        }
    }
}

namespace {

constexpr int64_t kMaxKeyTiles = 8192;
static_assert(kMaxKeyTiles * kPreK / kClassChunk <= kMaxClassBlocks, "chunks of a row along a grid dimension");

int prefill_check(const kvmix_prefill_attn_t *p)
{
    if (!p) return KVMIX_ERR_NULL;
    if (p->batch < 0 || p->heads <= 0 || p->kv_heads <= 0 || p->q_len < 0 || p->kv_len < 0) return KVMIX_ERR_SHAPE;
    if (p->heads % p->kv_heads != 0) return KVMIX_ERR_HEADS;
    if (p->head_dim != 64 && p->head_dim != 128) return KVMIX_ERR_UNSUPPORTED;
    if (p->kv_len > kMaxKeyTiles * kPreK || p->q_len > (1 << 24) || p->heads > (1 << 24)) return KVMIX_ERR_UNSUPPORTED;
    // launches that fit a grid: a block per 128 queries and head, mask slices along y
    if ((__int128)p->batch * p->heads * ((p->q_len + 32 * kPreWaves - 1) / (32 * kPreWaves)) > 0x7fffffff) return KVMIX_ERR_UNSUPPORTED;
    // 16-byte loads and 8-byte stores
    const int64_t strides[] = {p->q_batch_stride, p->q_head_stride, p->q_token_stride, p->k_batch_stride, p->k_head_stride,
                               p->k_token_stride, p->v_batch_stride, p->v_head_stride, p->v_token_stride};
    for (int64_t s : strides)
        if (s < 0 || s % 8 != 0) return KVMIX_ERR_UNSUPPORTED;
    if (((uintptr_t)p->q | (uintptr_t)p->k | (uintptr_t)p->v) % 16 != 0 || (uintptr_t)p->out % 8 != 0) return KVMIX_ERR_UNSUPPORTED;
    if (p->out_batch_stride % 4 != 0 || p->out_head_stride % 4 != 0 || p->out_token_stride % 4 != 0) return KVMIX_ERR_UNSUPPORTED;
    if (p->mask) {
        if (p->mask_dtype != KVMIX_F16 && p->mask_dtype != KVMIX_F32) return KVMIX_ERR_DTYPE;
        if ((p->mask_batch != 1 && p->mask_batch != p->batch) || (p->mask_heads != 1 && p->mask_heads != p->heads)) return KVMIX_ERR_SHAPE;
        if ((__int128)p->mask_batch * p->mask_heads > 65535) return KVMIX_ERR_UNSUPPORTED;
        if (p->mask_batch_stride < 0 || p->mask_head_stride < 0 || p->mask_row_stride < 0) return KVMIX_ERR_SHAPE;
    }
    return KVMIX_OK;
}

int64_t prefill_flag_bytes(const kvmix_prefill_attn_t *p)
{
    const int64_t parts = (p->q_len + 32 * kPreWaves - 1) / (32 * kPreWaves) * kPreWaves, kt = (p->kv_len + kPreK - 1) / kPreK;
    return p->mask_batch * p->mask_heads * parts * kt;  // (a byte per tile of 32 queries; its bits take 256)
}

int64_t prefill_chunks(const kvmix_prefill_attn_t *p) { return (p->kv_len + kClassChunk - 1) / kClassChunk; }

}  // namespace
}  // namespace kvmix

using namespace kvmix;

extern "C" int64_t kvmix_prefill_attention_workspace_bytes(const kvmix_prefill_attn_t *p)
{
    if (prefill_check(p) != KVMIX_OK || !p->mask) return 0;
    const int64_t kt = (p->kv_len + kPreK - 1) / kPreK;  // (per part and key tile a flag and 256 bytes of bits; per part and chunk two words)
    return kt ? 257 * prefill_flag_bytes(p) + 8 + prefill_flag_bytes(p) / kt * prefill_chunks(p) * 8 : 0;
}

extern "C" int kvmix_prefill_attention_supported(const kvmix_prefill_attn_t *p)
{
    return prefill_check(p) == KVMIX_OK ? 1 : 0;
}

extern "C" int kvmix_prefill_attention(const kvmix_prefill_attn_t *p, void *workspace, int64_t workspace_bytes, kvmix_stream_t stream)
{
    const int rc = prefill_check(p);
    if (rc != KVMIX_OK) return rc;
    if (p->batch == 0 || p->q_len == 0) return KVMIX_OK;
    if (p->kv_len == 0) return KVMIX_ERR_UNSUPPORTED;  // (no position to average)
    if (!p->q || !p->k || !p->v || !p->out) return KVMIX_ERR_NULL;
    PrefillArgs a;
    a.q = (const _Float16 *)p->q;
    a.k = (const _Float16 *)p->k;
    a.v = (const _Float16 *)p->v;
    a.out = (_Float16 *)p->out;
    a.q_bs = p->q_batch_stride, a.q_hs = p->q_head_stride, a.q_ts = p->q_token_stride;
    a.k_bs = p->k_batch_stride, a.k_hs = p->k_head_stride, a.k_ts = p->k_token_stride;
    a.v_bs = p->v_batch_stride, a.v_hs = p->v_head_stride, a.v_ts = p->v_token_stride;
    a.o_bs = p->out_batch_stride, a.o_hs = p->out_head_stride, a.o_ts = p->out_token_stride;
    a.heads = (int)p->heads;
    a.heads_per_kv = (int)(p->heads / p->kv_heads);
    a.q_len = (int)p->q_len;
    a.kv_len = (int)p->kv_len;
    a.q_tiles = (int)((p->q_len + 32 * kPreWaves - 1) / (32 * kPreWaves));
    a.parts = a.q_tiles * kPreWaves;
    a.k_tiles = (int)((p->kv_len + kPreK - 1) / kPreK);
    a.scale = p->scale;
    a.mask = p->mask;
    a.mask_f32 = p->mask_dtype == KVMIX_F32;
    a.m_bs = p->mask_batch > 1 ? p->mask_batch_stride : 0;
    a.m_hs = p->mask_heads > 1 ? p->mask_head_stride : 0;
    a.m_rs = p->mask_row_stride;
    a.far = p->k_token_stride >= (1 << 24) || p->v_token_stride >= (1 << 24);
    a.flags = nullptr;
    a.rows = nullptr;
    a.chunks = 0;
    a.bits = nullptr;
    a.flag_b = a.flag_h = 0;
    const int64_t blocks = p->batch * p->heads * a.q_tiles;
    hipStream_t st = (hipStream_t)stream;
    if (p->mask) {
        const int64_t slices = p->mask_batch * p->mask_heads;
        if (!workspace || (uintptr_t)workspace % 8 != 0 || workspace_bytes < kvmix_prefill_attention_workspace_bytes(p)) return KVMIX_ERR_WORKSPACE;
        uint64_t *bits = (uint64_t *)workspace;
        uint8_t *flags = (uint8_t *)workspace + 256 * prefill_flag_bytes(p);
        uint2 *rows = (uint2 *)((uint8_t *)workspace + 256 * prefill_flag_bytes(p) + (prefill_flag_bytes(p) + 7) / 8 * 8);
        a.chunks = (int)prefill_chunks(p);
        const dim3 grid((unsigned)a.parts, (unsigned)slices, (unsigned)a.chunks);
        if (a.mask_f32) prefill_mask_classes<float><<<grid, kClassWaves * kWave, 0, st>>>(a, bits, flags, rows, p->mask_heads);
        else prefill_mask_classes<_Float16><<<grid, kClassWaves * kWave, 0, st>>>(a, bits, flags, rows, p->mask_heads);
        if (launch_status() != KVMIX_OK) return KVMIX_ERR_LAUNCH;
        a.flags = flags;
        a.rows = rows;
        a.bits = bits;
        a.flag_h = p->mask_heads > 1 ? 1 : 0;
        a.flag_b = p->mask_batch > 1 ? (int)p->mask_heads : 0;
    }
    const dim3 grid((unsigned)blocks), block(kPreWaves * kWave);
    // What the routines that served these calls before held the probabilities in: with one query head per kv head fp16,
    // with grouped heads fp32, here two fp16 parts (their sum is within 2^-22).  The second part costs half as many
    // products again (B = 4, 32 / 32 heads, T = 2048, causal, before values were read transposed: 293 us without, 328 with it).
    const bool split = a.heads_per_kv > 1;
    if (p->head_dim == 128) split ? prefill_attn<128, true><<<grid, block, 0, st>>>(a) : prefill_attn<128, false><<<grid, block, 0, st>>>(a);
    else split ? prefill_attn<64, true><<<grid, block, 0, st>>>(a) : prefill_attn<64, false><<<grid, block, 0, st>>>(a);
    return launch_status();
}
