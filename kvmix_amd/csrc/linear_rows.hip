// The projections of a decode step: y[m][n] = sum_k x[m][k] w[n][k] for a handful of rows m (one per sequence),
// fp16 operands, fp32 sums.  Together they stream the weights of the model once per token, which is most of what a
// step moves, so what bounds them is HBM and the launches between them.  What stands around a projection in a
// decoder layer (models/modeling_llama_KVmix.py:84-112,268-283 and the stock layer around it) is folded in:
//
//   before  RMSNorm of x (every block normalises the rows it holds: the rows are a few kilobytes, the weights megabytes)
//   after   + residual | silu(gate) * up | RoPE and the append of the new token to the cache tails | fp16 -> fp32
//
// each with the roundings of the fp16 tensor expression it stands for.
#include "kvmix_common.h"

namespace kvmix {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

struct LinearArgs {
    const _Float16 *x, *norm;
    const _Float16 *w0, *w1, *w2;
    int64_t x_rs, w_rs;
    int64_t rows0, rows1, rows2;  // rows of w0, w1, w2
    int m, k;
    int pieces;                   // row tiles' worth of outputs per block (rows, or pairs of rows)
    float eps;
    // epilogues
    const uint16_t *residual;
    void *out;
    int64_t res_rs, out_rs;
    // rope
    const uint16_t *cos, *sin;
    int64_t cs_bs;                // elements between two sequences' angles (0: shared)
    uint16_t *k_tail, *v_tail;
    const int64_t *k_slot_dev, *v_slot_dev;
    int64_t kt_bs, kt_hs, kt_ts, vt_bs, vt_hs, vt_ts, k_slots, v_slots, k_slot, v_slot;
    int half;                     // head dimension / 2
};

enum { kEpiPlain = 0, kEpiFloat = 1, kEpiResidual = 2, kEpiSwiglu = 3, kEpiRope = 4 };

constexpr int kLinWaves = 8;

// Chunks per wave that a kernel of CH of them always has to itself: it is chosen only for more than the next smaller one holds.
__device__ constexpr int lin_full_chunks(int ch) { return ch <= 2 ? 0 : (ch <= 8 ? ch - 2 : ch - 3); }

__device__ __forceinline__ float lin_rounded(float v)
{
    uint32_t bits = f32_to_h16(v);
    asm volatile("" : "+v"(bits));  // keeps the rounding to fp16 from being contracted away
    return h16_to_f32((uint16_t)bits);
}

// Bound by HBM and, for the small ones, by what a launch costs before its bytes count.  A block takes `pieces` outputs
// (rows of w, or pairs of rows for the epilogues that combine two) and its eight waves slice K by 128-element chunks,
// round-robin, so that the block reads whole contiguous rows.  A wave keeps its slice of all x rows in registers for its
// whole life: lane = (row i of a tile or sequence i of a group of four, chunk part b), which is at once the A operand (four
// rows of w) and the B operand (four sequences) of v_mfma_f32_4x4x4, whose sixteen blocks take sixteen parts of K.  One
// load instruction is then 256 contiguous bytes of each of four rows (the 16x16x32 shape reads 64 bytes of each of sixteen
// rows and x again for every tile: 4.3-4.9 TB/s at best, 3.6 for sixteen sequences).  Two tiles are in flight while a
// third is multiplied; sums over lanes go by row swaps and DPP (through LDS shuffles: 31.4 instead of 25.8 us for sixteen
// sequences, k = 4096, n = 12288), a tile's sums leave through LDS and there is no barrier until the end.
// Measured (graph replay, weights from HBM; the library's product with the torch kernels around it -> this, us), four
// sequences, k = 4096: q/k/v n = 12288 with norm and RoPE 28.1 + 4.8 -> 20.7; n = 4096 with residual 14.9 -> 8.8; gate and
// up n = 22016 with norm and product 64.8 -> 33.1 (5.4 TB/s); n = 32000 with norm, fp32 67.6 -> 46.5 (5.6 TB/s); k = 11008,
// n = 4096 with residual 33.7 -> 20.6.  Sixteen sequences: 28.5 + 4.8 -> 25.8, 14.9 -> 12.0, 65.4 -> 39.6, 68.2 -> 55.0.
template <int CH, int MG, bool NORM, int EPI>
__global__ void __launch_bounds__(kLinWaves * kWave) linear_rows(LinearArgs a)
{
    constexpr bool PAIR = EPI == kEpiSwiglu || EPI == kEpiRope;
    constexpr int RT = PAIR ? 2 : 1;  // row tiles per step
    constexpr int MC = 4 * MG;
    extern __shared__ float part[];   // [waves][RT * pieces][MC]
    __shared__ float sq[kLinWaves][MC];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, i = lane & 3, b = lane >> 2;
    const int chunks = a.k / 128, wave_s = __builtin_amdgcn_readfirstlane(wave);
    const int64_t units = EPI == kEpiSwiglu ? a.rows0 : (EPI == kEpiRope ? (a.rows0 + a.rows1 + a.rows2) / 2 : a.rows0);
    const int64_t q0 = (int64_t)blockIdx.x * a.pieces;
    const int count = (int)(units - q0 < a.pieces ? units - q0 : a.pieces);
    const int tiles = (count + 3) / 4;

    // the weight row behind unit q of tile half r
    auto row_ptr = [&](int64_t q, int r) -> const _Float16 * {
        q = q < units ? q : units - 1;
        if constexpr (EPI == kEpiSwiglu) {
            return (r ? a.w1 : a.w0) + q * a.w_rs;
        } else if constexpr (EPI == kEpiRope) {
            const int64_t head = (uint32_t)q / (uint32_t)a.half;  // (rows of 256 bytes and more: fewer than 2^31)
            int64_t row = head * 2 * a.half + (q - head * a.half) + (r ? a.half : 0);
            if (row < a.rows0) return a.w0 + row * a.w_rs;
            row -= a.rows0;
            if (row < a.rows1) return a.w1 + row * a.w_rs;
            return a.w2 + (row - a.rows1) * a.w_rs;
        } else {
            return a.w0 + q * a.w_rs;
        }
    };

    half8 xv[MG][CH], wv[2][RT][CH];
    int off[CH];
#pragma unroll
    for (int j = 0; j < CH; j++) {
        const int c = wave + kLinWaves * j;
        off[j] = (c < chunks ? c : chunks - 1) * 128 + b * 8;
    }
    // (past the last tile every lane reads the same sixteen bytes: loads behind a branch would be waited for at once)
    auto load = [&](int t, half8 (&d)[RT][CH]) {
        const bool in = t < tiles;
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const _Float16 *p = in ? row_ptr(q0 + 4 * t + i, r) : a.w0;
#pragma unroll
            for (int j = 0; j < CH; j++)
                d[r][j] = __builtin_nontemporal_load(reinterpret_cast<const half8 *>(p + (in ? off[j] : 0)));
        }
    };
    // x first (it is in the L2), the first weights right behind it
#pragma unroll
    for (int g = 0; g < MG; g++) {
        const int m = g * 4 + i;
        const _Float16 *p = a.x + (int64_t)(m < a.m ? m : a.m - 1) * a.x_rs;
#pragma unroll
        for (int j = 0; j < CH; j++) xv[g][j] = *reinterpret_cast<const half8 *>(p + off[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    load(0, wv[0]);
    load(1, wv[1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < CH; j++) {  // (a chunk past the end repeats the last one's weights: both sides are made zero)
        if (wave + kLinWaves * j >= chunks) {
#pragma unroll
            for (int g = 0; g < MG; g++) xv[g][j] = half8{0, 0, 0, 0, 0, 0, 0, 0};
        }
    }
    if constexpr (NORM) {
        float nw[CH][8];
#pragma unroll
        for (int j = 0; j < CH; j++) {
            const half8 h = *reinterpret_cast<const half8 *>(a.norm + off[j]);
#pragma unroll
            for (int e = 0; e < 8; e++) nw[j][e] = wave_s + kLinWaves * j < chunks ? (float)h[e] : 0.f;
        }
#pragma unroll
        for (int g = 0; g < MG; g++) {
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < CH; j++) {
#pragma unroll
                for (int e = 0; e < 8; e++) s = fmaf((float)xv[g][j][e], (float)xv[g][j][e], s);
            }
#pragma unroll
            for (int o = 4; o <= 32; o *= 2) s += __shfl_xor(s, o);
            if (lane < 4) sq[wave][g * 4 + lane] = s;
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < MG; g++) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < kLinWaves; w++) s += sq[w][g * 4 + i];
            const float rstd = 1.0f / sqrtf(s / (float)a.k + a.eps);
#pragma unroll
            for (int j = 0; j < CH; j++) {
#pragma unroll
                for (int e = 0; e < 8; e++) xv[g][j][e] = (_Float16)fmaf((float)xv[g][j][e], rstd * nw[j][e], -0.0f);
            }
        }
    }
    auto work = [&](int t, const half8 (&d)[RT][CH]) {
#pragma unroll
        for (int r = 0; r < RT; r++) {
            floatx4 acc[MG];
#pragma unroll
            for (int g = 0; g < MG; g++) acc[g] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < CH; j++) {
                half8 ww = d[r][j];
                if (j >= lin_full_chunks(CH)) {  // (zero times an infinite weight would be NaN)
                    const uint32_t keep = wave_s + kLinWaves * j < chunks ? 0xffffffffu : 0;
                    ww = __builtin_bit_cast(half8, __builtin_bit_cast(uint4v, ww) & keep);
                }
                const half4 lo = {ww[0], ww[1], ww[2], ww[3]}, hi = {ww[4], ww[5], ww[6], ww[7]};
#pragma unroll
                for (int g = 0; g < MG; g++) {
                    const half8 xx = xv[g][j];
                    acc[g] = __builtin_amdgcn_mfma_f32_4x4x4f16(lo, half4{xx[0], xx[1], xx[2], xx[3]}, acc[g], 0, 0, 0);
                    acc[g] = __builtin_amdgcn_mfma_f32_4x4x4f16(hi, half4{xx[4], xx[5], xx[6], xx[7]}, acc[g], 0, 0, 0);
                }
            }
            // sum over the sixteen blocks (lane bits 2..5): two halving steps leave one row per lane, two plain ones finish
#pragma unroll
            for (int g = 0; g < MG; g++) {
                float v = halving_sum<16>(halving_sum<32>(acc[g][0], acc[g][2], lane), halving_sum<32>(acc[g][1], acc[g][3], lane), lane);
                v += row_ror<8>(v);
                v += row_ror<4>(v);
                if ((lane & 12) == 0)
                    part[((int64_t)(wave * RT + r) * a.pieces + 4 * t + (lane >> 5) * 2 + (lane >> 4 & 1)) * MC + g * 4 + i] = v;
            }
        }
    };
    for (int t = 0; t < tiles; t += 2) {
        work(t, wv[0]);
        load(t + 2, wv[0]);
        __builtin_amdgcn_sched_barrier(0);
        if (t + 1 < tiles) work(t + 1, wv[1]);
        load(t + 3, wv[1]);
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();

    for (int e = threadIdx.x; e < count * MC; e += kLinWaves * kWave) {
        const int piece = e % count, m = e / count;  // neighbouring threads: neighbouring outputs of one sequence
        if (m >= a.m) break;
        float s[RT];
#pragma unroll
        for (int r = 0; r < RT; r++) {
            s[r] = 0.f;
#pragma unroll
            for (int w = 0; w < kLinWaves; w++) s[r] += part[((int64_t)(w * RT + r) * a.pieces + piece) * MC + m];
        }
        const int64_t q = q0 + piece;
        if constexpr (EPI == kEpiPlain) {
            ((uint16_t *)a.out)[m * a.out_rs + q] = f32_to_h16(s[0]);
        } else if constexpr (EPI == kEpiFloat) {
            ((float *)a.out)[m * a.out_rs + q] = lin_rounded(s[0]);
        } else if constexpr (EPI == kEpiResidual) {
            ((uint16_t *)a.out)[m * a.out_rs + q] = f32_to_h16(h16_to_f32(a.residual[m * a.res_rs + q]) + lin_rounded(s[0]));
        } else if constexpr (EPI == kEpiSwiglu) {
            const float gate = lin_rounded(s[0]), up = lin_rounded(s[1]);
            const float act = lin_rounded(gate / (1.0f + expf(-gate)));
            ((uint16_t *)a.out)[m * a.out_rs + q] = f32_to_h16(act * up);
        } else {
            const int D = 2 * a.half;
            const int64_t head = (uint32_t)q / (uint32_t)a.half;  // (rows of 256 bytes and more: fewer than 2^31)
            const int d = (int)(q - head * a.half);
            float x1 = lin_rounded(s[0]), x2 = lin_rounded(s[1]);
            const int64_t heads = a.rows0 / D, kv = a.rows1 / D;
            uint16_t *dst;
            if (head < heads) {
                dst = (uint16_t *)a.out + m * a.out_rs + head * D;
            } else if (head < heads + kv) {
                const int64_t slot = a.k_slot_dev ? *a.k_slot_dev : a.k_slot;
                if (slot < 0 || slot >= a.k_slots) continue;  // a slot from device memory never leads out of the window
                dst = a.k_tail + m * a.kt_bs + (head - heads) * a.kt_hs + slot * a.kt_ts;
            } else {
                const int64_t slot = a.v_slot_dev ? *a.v_slot_dev : a.v_slot;
                if (slot < 0 || slot >= a.v_slots) continue;
                dst = a.v_tail + m * a.vt_bs + (head - heads - kv) * a.vt_hs + slot * a.vt_ts;
                dst[d] = f32_to_h16(x1);
                dst[d + a.half] = f32_to_h16(x2);
                continue;
            }
            const uint16_t *cs = a.cos + m * a.cs_bs, *sn = a.sin + m * a.cs_bs;
            const float c1 = h16_to_f32(cs[d]), c2 = h16_to_f32(cs[d + a.half]);
            const float s1 = h16_to_f32(sn[d]), s2 = h16_to_f32(sn[d + a.half]);
            dst[d] = f32_to_h16(lin_rounded(x1 * c1) + lin_rounded(-x2 * s1));
            dst[d + a.half] = f32_to_h16(lin_rounded(x2 * c2) + lin_rounded(x1 * s2));
        }
    }
}

}  // namespace kvmix

using namespace kvmix;

namespace {

struct LinearPlan {
    int ch, mg, pieces;
    unsigned blocks;
    size_t lds;
};

// Rows of x a wave keeps: ch chunks of each of 4 * mg sequences, four registers per chunk and group of four sequences.
// The weights in flight take as many again per row tile, and a wave of this block size has 256 registers: the
// combinations refused below would spill or measured no faster than the library's product (k = 8192, sixteen sequences:
// 19.7 against 19.1 us; k = 14336, eight: 29.4 against 29.8).  One block per CU: every block reads all of x from the L2
// before it starts, and 512 or 1024 smaller blocks do that two or four times per CU (k = 4096, four sequences, 256 / 512 /
// 1024 blocks: n = 4096 8.8 / 9.8 / 11.9, n = 22016 33.1 / 35.5 / 41.8 us).
bool linear_plan(const kvmix_linear_rows_t *p, LinearPlan *pl)
{
    const int64_t chunks = (p->k / 128 + kLinWaves - 1) / kLinWaves;
    const bool pair = p->epilogue == KVMIX_LINEAR_SWIGLU || p->epilogue == KVMIX_LINEAR_ROPE_APPEND;
    pl->ch = 0;
    for (int c : {2, 4, 6, 8, 11, 14}) {
        if (chunks <= c) {
            pl->ch = c;
            break;
        }
    }
    pl->mg = p->m <= 4 ? 1 : (p->m <= 8 ? 2 : 4);
    if (!pl->ch || p->m > 16) return false;
    const bool norm = p->norm_weight != nullptr;
    if (norm && p->epilogue == KVMIX_LINEAR_RESIDUAL) return false;  // (nothing in a decoder layer is both: no such instance)
    if (pl->ch > 8 && (pl->mg > 2 || pair || norm)) return false;
    if ((pl->ch > 6 && pl->mg > 2) || (pl->ch > 11 && pl->mg > 1)) return false;  // (no faster than the library's there)
    if (pl->ch > 6 && norm && pair && pl->mg > 1) return false;
    if (pl->ch > 4 && pl->mg > 2 && (pair || norm)) return false;
    const int64_t units = pair ? (p->epilogue == KVMIX_LINEAR_SWIGLU ? p->rows[0] : (p->rows[0] + p->rows[1] + p->rows[2]) / 2) : p->rows[0];
    const int rt = pair ? 2 : 1;
    int64_t target = 256;
#ifdef KVMIX_EXPERIMENT
    if (const char *e = getenv("KVMIX_LIN_BLOCKS")) target = atoi(e);
#endif
    int64_t pieces = ((units + target - 1) / target + 3) / 4 * 4;
    const int64_t most = (64 << 10) / (kLinWaves * rt * 4 * pl->mg * 4);  // (partial sums in LDS)
    if (pieces > most) pieces = most;
    if (pieces < 4) pieces = 4;  // (no rows at all: nothing is launched)
    pl->pieces = (int)pieces;
    pl->blocks = (unsigned)((units + pieces - 1) / pieces);
    pl->lds = (size_t)kLinWaves * rt * pieces * 4 * pl->mg * 4;
    return true;
}

template <int CH, int MG, bool NORM, int EPI>
int linear_launch(const LinearArgs &a, const LinearPlan &pl, hipStream_t st)
{
    hipLaunchKernelGGL((linear_rows<CH, MG, NORM, EPI>), dim3(pl.blocks), dim3(kLinWaves * kWave), pl.lds, st, a);
    return launch_status();
}

template <int CH, int MG>
int linear_epilogue(const LinearArgs &a, const LinearPlan &pl, int epi, bool norm, hipStream_t st)
{
    if constexpr (CH <= 8) {
        if (norm) {
            if constexpr (CH <= 4 || MG <= 2) {
                if (epi == KVMIX_LINEAR_PLAIN) return linear_launch<CH, MG, true, kEpiPlain>(a, pl, st);
                if (epi == KVMIX_LINEAR_FLOAT) return linear_launch<CH, MG, true, kEpiFloat>(a, pl, st);
            }
            if constexpr (CH <= 4 || MG <= 1 || (CH <= 6 && MG <= 2)) {
                if (epi == KVMIX_LINEAR_SWIGLU) return linear_launch<CH, MG, true, kEpiSwiglu>(a, pl, st);
                if (epi == KVMIX_LINEAR_ROPE_APPEND) return linear_launch<CH, MG, true, kEpiRope>(a, pl, st);
            }
            return KVMIX_ERR_UNSUPPORTED;
        }
        if constexpr (CH <= 4 || MG <= 2) {
            if (epi == KVMIX_LINEAR_SWIGLU) return linear_launch<CH, MG, false, kEpiSwiglu>(a, pl, st);
            if (epi == KVMIX_LINEAR_ROPE_APPEND) return linear_launch<CH, MG, false, kEpiRope>(a, pl, st);
        }
    }
    if (epi == KVMIX_LINEAR_PLAIN) return linear_launch<CH, MG, false, kEpiPlain>(a, pl, st);
    if (epi == KVMIX_LINEAR_FLOAT) return linear_launch<CH, MG, false, kEpiFloat>(a, pl, st);
    if (epi == KVMIX_LINEAR_RESIDUAL) return linear_launch<CH, MG, false, kEpiResidual>(a, pl, st);
    return KVMIX_ERR_UNSUPPORTED;
}

int linear_check(const kvmix_linear_rows_t *p)
{
    if (!p) return KVMIX_ERR_NULL;
    if (p->m < 0 || p->k <= 0 || p->rows[0] < 0 || p->rows[1] < 0 || p->rows[2] < 0 || p->x_stride < p->k || p->w_stride < p->k)
        return KVMIX_ERR_SHAPE;
    // 16-byte loads of whole 128-element chunks
    if (p->k % 128 != 0 || p->x_stride % 8 != 0 || p->w_stride % 8 != 0) return KVMIX_ERR_UNSUPPORTED;
    if (((uintptr_t)p->x | (uintptr_t)p->w[0] | (uintptr_t)p->w[1] | (uintptr_t)p->w[2] | (uintptr_t)p->norm_weight) % 16 != 0)
        return KVMIX_ERR_UNSUPPORTED;
    if (p->epilogue < KVMIX_LINEAR_PLAIN || p->epilogue > KVMIX_LINEAR_ROPE_APPEND) return KVMIX_ERR_UNSUPPORTED;
    if (p->epilogue == KVMIX_LINEAR_SWIGLU && p->rows[1] != p->rows[0]) return KVMIX_ERR_SHAPE;
    if (p->epilogue == KVMIX_LINEAR_ROPE_APPEND) {
        if (p->head_dim <= 0 || p->head_dim % 8 != 0) return KVMIX_ERR_UNSUPPORTED;
        if (p->rows[0] <= 0 || p->rows[1] <= 0 || p->rows[0] % p->head_dim || p->rows[1] % p->head_dim || p->rows[2] != p->rows[1])
            return KVMIX_ERR_SHAPE;
        if (p->rows[0] % p->rows[1] != 0) return KVMIX_ERR_HEADS;
        if (p->k_tail_slots < 0 || p->v_tail_slots < 0 || p->k_tail_token_stride < p->head_dim || p->v_tail_token_stride < p->head_dim)
            return KVMIX_ERR_SHAPE;
        if ((!p->k_slot_dev && (p->k_slot < 0 || p->k_slot >= p->k_tail_slots)) ||
            (!p->v_slot_dev && (p->v_slot < 0 || p->v_slot >= p->v_tail_slots)))
            return KVMIX_ERR_SHAPE;
    } else if (p->epilogue != KVMIX_LINEAR_SWIGLU && (p->rows[1] || p->rows[2])) {
        return KVMIX_ERR_SHAPE;
    }
    if (p->out_stride < p->rows[0] || (p->epilogue == KVMIX_LINEAR_RESIDUAL && p->residual_stride < p->rows[0])) return KVMIX_ERR_SHAPE;
    return KVMIX_OK;
}

}  // namespace

extern "C" int kvmix_linear_rows_supported(const kvmix_linear_rows_t *p)
{
    LinearPlan pl;
    return linear_check(p) == KVMIX_OK && linear_plan(p, &pl) ? 1 : 0;
}

extern "C" int kvmix_linear_rows(const kvmix_linear_rows_t *p, kvmix_stream_t stream)
{
    const int rc = linear_check(p);
    if (rc != KVMIX_OK) return rc;
    LinearPlan pl;
    if (!linear_plan(p, &pl)) return KVMIX_ERR_UNSUPPORTED;
    if (p->m == 0 || p->rows[0] == 0) return KVMIX_OK;
    if (!p->x || !p->w[0] || !p->out) return KVMIX_ERR_NULL;
    if (p->epilogue == KVMIX_LINEAR_RESIDUAL && !p->residual) return KVMIX_ERR_NULL;
    if (p->epilogue == KVMIX_LINEAR_SWIGLU && !p->w[1]) return KVMIX_ERR_NULL;
    if (p->epilogue == KVMIX_LINEAR_ROPE_APPEND && (!p->w[1] || !p->w[2] || !p->cos || !p->sin || !p->k_tail || !p->v_tail)) return KVMIX_ERR_NULL;
    LinearArgs a;
    a.x = (const _Float16 *)p->x;
    a.norm = (const _Float16 *)p->norm_weight;
    a.w0 = (const _Float16 *)p->w[0];
    a.w1 = (const _Float16 *)p->w[1];
    a.w2 = (const _Float16 *)p->w[2];
    a.x_rs = p->x_stride;
    a.w_rs = p->w_stride;
    a.rows0 = p->rows[0];
    a.rows1 = p->rows[1];
    a.rows2 = p->rows[2];
    a.m = (int)p->m;
    a.k = (int)p->k;
    a.pieces = pl.pieces;
    a.eps = p->norm_eps;
    a.residual = (const uint16_t *)p->residual;
    a.out = p->out;
    a.res_rs = p->residual_stride;
    a.out_rs = p->out_stride;
    a.cos = (const uint16_t *)p->cos;
    a.sin = (const uint16_t *)p->sin;
    a.cs_bs = p->cos_sin_batch_stride;
    a.k_tail = (uint16_t *)p->k_tail;
    a.v_tail = (uint16_t *)p->v_tail;
    a.k_slot_dev = p->k_slot_dev;
    a.v_slot_dev = p->v_slot_dev;
    a.kt_bs = p->k_tail_batch_stride;
    a.kt_hs = p->k_tail_head_stride;
    a.kt_ts = p->k_tail_token_stride;
    a.vt_bs = p->v_tail_batch_stride;
    a.vt_hs = p->v_tail_head_stride;
    a.vt_ts = p->v_tail_token_stride;
    a.k_slots = p->k_tail_slots;
    a.v_slots = p->v_tail_slots;
    a.k_slot = p->k_slot;
    a.v_slot = p->v_slot;
    a.half = (int)(p->head_dim / 2);
    const bool norm = p->norm_weight != nullptr;
    hipStream_t st = (hipStream_t)stream;
#define KVMIX_LINEAR_CASE(CH, MG) \
    if (pl.ch == CH && pl.mg == MG) return linear_epilogue<CH, MG>(a, pl, p->epilogue, norm, st);
    KVMIX_LINEAR_CASE(2, 1)
    KVMIX_LINEAR_CASE(2, 2)
    KVMIX_LINEAR_CASE(2, 4)
    KVMIX_LINEAR_CASE(4, 1)
    KVMIX_LINEAR_CASE(4, 2)
    KVMIX_LINEAR_CASE(4, 4)
    KVMIX_LINEAR_CASE(6, 1)
    KVMIX_LINEAR_CASE(6, 2)
    KVMIX_LINEAR_CASE(6, 4)
    KVMIX_LINEAR_CASE(8, 1)
    KVMIX_LINEAR_CASE(8, 2)
    KVMIX_LINEAR_CASE(11, 1)
    KVMIX_LINEAR_CASE(11, 2)
    KVMIX_LINEAR_CASE(14, 1)
#undef KVMIX_LINEAR_CASE
    return KVMIX_ERR_UNSUPPORTED;
}
