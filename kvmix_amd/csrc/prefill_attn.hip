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

struct PrefillArgs {
    const _Float16 *q, *k, *v;
    _Float16 *out;
    int64_t q_bs, q_hs, q_ts, k_bs, k_hs, k_ts, v_bs, v_hs, v_ts, o_bs, o_hs, o_ts;
    const void *mask;
    int mask_f32;
    int64_t m_bs, m_hs, m_rs;
    int flag_b, flag_h;        // mask slice of (batch b, head h): b * flag_b + h * flag_h
    const uint8_t *flags;      // [mask slices][key tiles][query parts]: class of the tile of a part's 32 queries
    const uint8_t *dead;       // [mask slices][Q]
    const uint64_t *bits;      // [mask slices][query parts][key tiles][32 queries]: bit 16 j + i = key 4 i + j is masked
    int heads, heads_per_kv, q_len, kv_len, q_tiles, k_tiles, parts;  // parts: 32 queries each, whole blocks of them
    float scale;
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

// Classes of the tiles of 32 queries (one block) by 64 keys, and which rows are masked everywhere.  Bound by the latency of
// reading the mask once (13 us at T = 2048; the loads of the mixed tiles alone cost the attention kernel 90); two rows per wave and four loads of each in flight, since a block is all the work there is for 32 queries.
template <typename T>
__global__ void __launch_bounds__(kClassWaves * kWave) prefill_mask_classes(PrefillArgs a, uint64_t *bits, uint8_t *flags, uint8_t *dead,
                                                                             int64_t mask_heads)
{
    extern __shared__ uint32_t tile_bits[];  // per key tile: some entry not masked (1), not zero (2), neither (4)
    __shared__ uint32_t row_bits[2];         // rows with an entry above `absorbed`, rows with an entry of at least -30000
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int64_t slice = blockIdx.y;
    const int r0 = blockIdx.x * 32, valid = a.q_len - r0 < 32 ? a.q_len - r0 : 32;
    const T *base = (const T *)a.mask + (slice / mask_heads) * a.m_bs + (slice % mask_heads) * a.m_hs;
    // what the prompt branch takes for a row masked everywhere: see KVmixAttention._prompt_attention
    const float absorbed = sizeof(T) == 2 ? kHalfLowest : -1e30f;
    for (int t = threadIdx.x; t < a.k_tiles; t += kClassWaves * kWave) tile_bits[t] = 0;
    if (threadIdx.x < 2) row_bits[threadIdx.x] = 0;
    __syncthreads();
    uint32_t live[2] = {0, 0}, tight[2] = {0, 0};
    uint64_t *tile_rows = bits + (slice * a.parts + blockIdx.x) * a.k_tiles * 32;
    for (int c0 = 0; c0 < a.kv_len; c0 += 4 * kClassCols) {
        float v[4][2][4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int row = 2 * wave + r;
                mask_four(base + (int64_t)(r0 + row < a.q_len ? r0 + row : a.q_len - 1) * a.m_rs, c0 + u * kClassCols + 4 * lane,
                          a.kv_len, 0.0f, v[u][r]);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int col = c0 + u * kClassCols + 4 * lane;
            const int tile = (c0 + u * kClassCols) / kPreK + lane / 16;
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
                const uint32_t kinds = ((s >> lane) & 0xffff ? 1u : 0u) | ((o >> lane) & 0xffff ? 2u : 0u) | ((n >> lane) & 0xffff ? 4u : 0u);
                if (kinds) atomicOr(&tile_bits[tile], kinds);
            }
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
    const uint32_t rows = valid <= 0 ? 0 : (valid == 32 ? 0xffffffffu : (1u << valid) - 1);
    const bool all_dead = (row_bits[0] & rows) == 0, loose = (row_bits[1] & rows) != rows;
    uint8_t *f = flags + slice * a.k_tiles * a.parts + blockIdx.x;
    for (int t = threadIdx.x; t < a.k_tiles; t += kClassWaves * kWave) {
        const uint32_t kinds = tile_bits[t];
        int c = kinds & 4 ? kTileMixed : (kinds & 2 ? kTileBinary : kTilePlain);
        if (!(kinds & 1) && !loose) c = kTileSkip;
        if (all_dead) c = kTilePlain;  // (with queries of zero: all positions alike, whatever the one mask value is)
        f[t * (int64_t)a.parts] = valid <= 0 ? kTileSkip : c;
    }
    if ((int)threadIdx.x < valid) dead[slice * a.q_len + r0 + threadIdx.x] = !(row_bits[0] >> threadIdx.x & 1);
}

// LDS layouts, both free of bank conflicts on the reading side.  Keys: [64][D] as loaded, the 16-byte pieces of a row
// exchanged by the row's low bits.  Values: transposed, [D][64 keys], the keys of each sixteen in the order in which the
// lanes hold the probabilities (groups of four: 0 2 1 3), so that a lane's eight values of one dimension are one piece.
template <int D>
__device__ __forceinline__ int key_piece(int key, int c)
{
    return D == 128 ? key * 256 + ((c ^ (key & 15)) << 4) : key * 128 + ((c ^ ((key >> 1) & 7)) << 4);
}

__device__ __forceinline__ int value_piece(int d, int c)
{
    return d * 128 + ((c ^ ((d >> 1) & 7)) << 4);
}

// One block: 128 queries of one head, 32 to a wave, over the key tiles that some of them needs.  Bound by the matrix
// cores and the exponentials beside them, so everything else is kept off that path.  The logits are computed transposed
// (32x32x16, keys as rows): a lane then holds 32 logits of ONE query, the softmax needs a single exchange between the two
// halves of a wave, and the probabilities are already the right-hand operand of out^T = v^T p^T (the order of the keys
// inside a product is free: the values are stored in LDS in that order).  The mask's entries are added to the finished
// logits (sums that start from them round at their size at every step: 2.5 times the error under a mask of -10000).  Keys
// go from memory straight to LDS, values through registers (transposed on the way), both one tile ahead of the products;
// two blocks share a CU.  Eight waves on 256 queries read keys and values half as often but lose more to the causal
// border (T = 2048: 409 against 400 us with split probabilities).  Measured (us per call with the mask's classes, causal
// fp32 mask; torch's fused routine after preparing the mask -> this): B = 4, 32 heads, T = 2048 739 -> 293 (without a
// mask 720 TFLOP/s); B = 1, T = 4096 927 -> 285; B = 4, T = 512 57 -> 42; 32 / 8 heads: B = 4, T = 2048 6012 -> 326, B =
// 1, T = 1001 442 -> 54.  A mask that is mixed in every tile (a bias per distance below the diagonal), B = 2, 32 heads, T
// = 2048: 273 (504 from sums that start there).  Error against float64 relative to the norm, keys with an outlier
// channel, causal, T = 300 / 1500 / 2048: 2.35 / 2.37 / 2.41e-4, the routine before 2.36 / 2.39 / 2.42e-4; with the
// maximum moved from 2^8 on only 2.45 / 2.58 / 2.68e-4 (268 us).
template <int D, bool SPLIT>
__global__ void __launch_bounds__(kPreWaves * kWave) __attribute__((amdgpu_waves_per_eu(2, 2))) prefill_attn(PrefillArgs a)
{
    constexpr int W = kPreWaves;
    constexpr int KS = D / 16, DT = D / 32, CPR = D / 8;   // k-steps of q.k^T, 32-row tiles of out^T, pieces per row
    constexpr int KL = kPreK * CPR / (W * kWave);  // key pieces a thread moves per tile
    constexpr int kTileBytes = kPreK * D * 2;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2][2][kTileBytes];
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, col = lane & 31, h2 = lane >> 5;

    // consecutive blocks of one XCD: the query tiles of one head after the other, the longest (causal) ones first
    const int64_t n = gridDim.x, l = blockIdx.x, xcd = l % 8, per = n / 8, rem = n % 8;
    const int64_t job = xcd * per + (xcd < rem ? xcd : rem) + l / 8;
    const int qt = a.q_tiles - 1 - (int)(job % a.q_tiles);
    const int64_t bh = job / a.q_tiles;
    const int b = (int)(bh / a.heads), head = (int)(bh % a.heads);
    const _Float16 *kp = a.k + b * a.k_bs + (head / a.heads_per_kv) * a.k_hs;
    const _Float16 *vp = a.v + b * a.v_bs + (head / a.heads_per_kv) * a.v_hs;
    const int64_t slice = (int64_t)b * a.flag_b + (int64_t)head * a.flag_h;
    const uint32_t *flags = a.flags ? (const uint32_t *)(a.flags + slice * a.k_tiles * a.parts) + qt : nullptr;  // a byte per wave
    const int flag_step = a.parts / W;

    const int query = (qt * W + wave) * 32 + col, row = query < a.q_len ? query : a.q_len - 1;
    half8 qv[KS];
    {
        const _Float16 *qp = a.q + b * a.q_bs + head * a.q_hs + (int64_t)row * a.q_ts + 8 * h2;
        const bool off = a.flags && a.dead[slice * a.q_len + row];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            qv[ks] = *(const half8 *)(qp + 16 * ks);
            if (off) qv[ks] = half8{};
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
            classes = t < a.k_tiles ? (flags ? flags[(int64_t)t * flag_step] : 0x01010101u) : 0;
            pending = __ballot(classes != 0);
        }
        const int bit = __builtin_ctzll(pending);
        pending &= pending - 1;
        cls = __builtin_amdgcn_readlane(classes, bit);
        return window + bit;
    };

    half8 vr[4];
    const int vd = tid % CPR, vg = tid / CPR;  // value pieces: dimensions [8 vd, 8 vd + 8) of keys [4 vg, 4 vg + 4)
    auto load_tile = [&](int t, int into) {
        const int k0 = t * kPreK, last = a.kv_len - 1;
#pragma unroll
        for (int i = 0; i < KL; i++) {
            // straight to LDS, where a wave's 64 pieces lie one after the other: lane by lane the piece that belongs there
            const int first = (wave + i * W) * kWave, p = first + lane, key = k0 + p / CPR;
            const int at = key_piece<D>(p / CPR, p % CPR) >> 4;
            const _Float16 *from = kp + (int64_t)(key < last ? key : last) * a.k_ts + (at % CPR) * 8;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from,
                                             (__attribute__((address_space(3))) void *)(lds[into][0] + first * 16), 16, 0, 0);
        }
        if (vg < kPreK / 4) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int key = k0 + 4 * vg + i;
                vr[i] = *(const half8 *)(vp + (int64_t)(key < last ? key : last) * a.v_ts + vd * 8);
            }
        }
    };
    auto store_tile = [&](int t, int buf) {
        if (vg < kPreK / 4) {
            if (__builtin_expect((t + 1) * kPreK > a.kv_len, 0)) {  // (the last value again past the end: weight zero times an infinite one is NaN)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (t * kPreK + 4 * vg + i >= a.kv_len) vr[i] = half8{};
            }
            const int c = 2 * (vg >> 2) + (vg & 1), at = 8 * ((vg >> 1) & 1);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const half4 w = {vr[0][i], vr[1][i], vr[2][i], vr[3][i]};
                *(half4 *)(lds[buf][1] + value_piece(8 * vd + i, c) + at) = w;
            }
        }
    };

    // a lane's pieces of the first 32 rows: step ks, kk is the piece at an exclusive or with 32 bytes times the step
    const int k_at = key_piece<D>(col, h2), v_at = value_piece(col, h2);

    floatx16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++) o[t] = floatx16{};
    float m = -1e30f, sum = 0.0f;  // in units of log2 (a finite start: a tile of logits of -inf weighs zero)
    const float c = a.scale * kLog2e, unscale = 1.0f / a.scale;

    int tile = next_tile(), buf = 0;
    if (tile >= 0) {
        load_tile(tile, 0);
        store_tile(tile, 0);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
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
                    const half8 vv = *(const half8 *)(lds[buf][1] + (v_at ^ (kk << 5)) + t * 32 * 2 * kPreK);
                    o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vv, ph[kk % 2], o[t], 0, 0, 0);
                    if constexpr (SPLIT) o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vv, pl[kk % 2], o[t], 0, 0, 0);
                }
                if (kk < 3) probs(kk + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        buf ^= 1;
        if (next >= 0) store_tile(next, buf);
        __builtin_amdgcn_s_waitcnt(0x0f70);  // the key pieces on their way to LDS (vmcnt 0)
        __syncthreads();
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

constexpr int64_t kMaxKeyTiles = 8192;  // (a word of LDS each in prefill_mask_classes)

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

}  // namespace
}  // namespace kvmix

using namespace kvmix;

extern "C" int64_t kvmix_prefill_attention_workspace_bytes(const kvmix_prefill_attn_t *p)
{
    if (prefill_check(p) != KVMIX_OK || !p->mask) return 0;
    return 257 * prefill_flag_bytes(p) + p->mask_batch * p->mask_heads * p->q_len;
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
    a.flags = nullptr;
    a.dead = nullptr;
    a.bits = nullptr;
    a.flag_b = a.flag_h = 0;
    const int64_t blocks = p->batch * p->heads * a.q_tiles;
    hipStream_t st = (hipStream_t)stream;
    if (p->mask) {
        const int64_t slices = p->mask_batch * p->mask_heads;
        if (!workspace || (uintptr_t)workspace % 8 != 0 || workspace_bytes < kvmix_prefill_attention_workspace_bytes(p)) return KVMIX_ERR_WORKSPACE;
        uint64_t *bits = (uint64_t *)workspace;
        uint8_t *flags = (uint8_t *)workspace + 256 * prefill_flag_bytes(p), *dead = flags + prefill_flag_bytes(p);
        const dim3 grid((unsigned)a.parts, (unsigned)slices);
        const size_t lds = (size_t)a.k_tiles * 4;
        if (a.mask_f32) prefill_mask_classes<float><<<grid, kClassWaves * kWave, lds, st>>>(a, bits, flags, dead, p->mask_heads);
        else prefill_mask_classes<_Float16><<<grid, kClassWaves * kWave, lds, st>>>(a, bits, flags, dead, p->mask_heads);
        if (launch_status() != KVMIX_OK) return KVMIX_ERR_LAUNCH;
        a.flags = flags;
        a.dead = dead;
        a.bits = bits;
        a.flag_h = p->mask_heads > 1 ? 1 : 0;
        a.flag_b = p->mask_batch > 1 ? (int)p->mask_heads : 0;
    }
    const dim3 grid((unsigned)blocks), block(kPreWaves * kWave);
    // What the routines that served these calls before held the probabilities in: with one query head per kv head fp16,
    // with grouped heads fp32, here two fp16 parts (their sum is within 2^-22).  The second part costs half as many
    // products again: B = 4, 32 / 32 heads, T = 2048, causal 293 us without, 328 with it.
    const bool split = a.heads_per_kv > 1;
    if (p->head_dim == 128) split ? prefill_attn<128, true><<<grid, block, 0, st>>>(a) : prefill_attn<128, false><<<grid, block, 0, st>>>(a);
    else split ? prefill_attn<64, true><<<grid, block, 0, st>>>(a) : prefill_attn<64, false><<<grid, block, 0, st>>>(a);
    return launch_status();
}
