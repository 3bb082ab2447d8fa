// BH4 with 64 x 64 blocks (PL/bh4/kernel.py:23-36), forward and backward, on the fp16 matrix cores: the stages of
// bh4_block.hip, (H_NB (x) I_64) * blockdiag(H_64 W[r,s,n]) each, with the weights and the tokens' rows as two half-precision terms
// a number (split_mfma.h).
//
// The hash form runs the layer's whole front end for 8-bit codes: LayerNorm while the tile is loaded, the stages, z = decay * y +
// residual * LN(x) + bias on the accumulators (x is read again and normalised with the kept statistics), codes and scores.  A
// wavefront owns 16 output columns of every block, products on v_mfma_f32_16x16x32_f16 with the weights as A and the tokens as B, so
// that a lane ends up with four consecutive columns of one token in every block: the butterflies across blocks are register adds.
// Between two stages a token's row is scaled by a power of two, its largest to [2^14, 2^15), split, and written to the tile (hi and
// lo, 4 bytes a number, as much as it was in fp32); both terms are then normal half-precision numbers or smaller than 2^-38 of the
// row's largest, so neither needs a factor, the six instructions of a block add into one accumulator, and nothing overflows however a
// stage amplifies.  A row's scale depends on that row alone: its results do not depend on its neighbours.  A row with an infinity or
// NaN comes out as NaN.
//
// What bounds it: vector work (LayerNorm 18, a stage 9, hash 18 instructions a number) and the latencies between it and the products;
// with all weights from the L1 the hash form at 32768 tokens, D = 512, two repeats takes 113 us instead of 121, so the weights' way from
// the L2 (2.1 GB) is no more than a part.  The training form and the backward write 0.54 and 0.67 GB at that size, which go out at the
// memory's rate and hide little behind the products (137 and 128 us without them).  They go out as whole rows, turned round through LDS
// in fp32, where a wavefront stored 64 bytes of sixteen rows straight from its accumulators: 196 -> 166 and 200 -> 173 us, 209 -> 168 and
// 250 -> 195 in a training step; 16384, D = 1024 115 -> 99 and 106 -> 98; 32768, D = 256, four repeats 184 -> 175 and 185 -> 162.  Stores held
// back until the next product: 193 and 217, from spills.
// Products on the fp32 matrix cores (bh4_block.hip) take 16/3 of the time of these.  us, fp32 kernel -> this one, inputs in turn: hash
// 32768 tokens, D = 512, two repeats 202 -> 121; 16384, D = 1024 113 -> 73; 385, D = 512 18.6 -> 12.3.  Training form 278 -> 168; 385,
// D = 512 24.9 -> 15.5.  Backward in a training step 256 -> 195; few tokens 18.7 -> 12.2 and 2103, D = 1024 35.6 -> 23.0.
// Tried for the hash form: 32 tokens a workgroup in 4 wavefronts (124-149 us from build to build) and 8 (151), 64 in 8 (145), four
// blocks' weights ahead instead of two (134).  Error of the last stage against 64 bits 2.4e-7 (fp32 matrix cores 3.2e-7), input gradient
// 2.2e-7 (3.1e-7).
//
// A layer runs this forward with gradients and without, in train() and eval() (Hashing.forward_block, csrc/host.cpp): a projected
// value within rounding of zero takes either sign, with the sign the derivative of its score turns round, and a pass without
// gradients must not differ from one with them.  The training form is the hash form with stores: its codes and scores are the same
// bit for bit.  Against 64 bits, LayerNorm included, 200 rows of D = 512, fp32 kernel -> this one: z 3.1e-7 -> 2.4e-7, stage inputs
// 2.4e-7 -> 1.8e-7, scores 4.5e-7 -> 3.4e-7 (rows spread over e^1.5 in size: 3.2e-7, 2.4e-7, 4.6e-7 -> 2.4e-7, 1.9e-7, 3.9e-7).
#include <algorithm>

#include "split_mfma.h"

// the mix and the score keep the reference's operation order: no fused multiply-add
#pragma clang fp contract(off)

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int BS = 64;          // block size this file is built for
constexpr int PAD = 4;          // floats of padding per row of the fp32 tile
constexpr float TOP = 16384.f;  // what the largest of a row is scaled to at least (and less than twice that)

// Largest and smallest over the wavefront.
__device__ __forceinline__ void wave_range(float v, float &most, float &least) {
    most = least = v;
    auto step = [&](float m, float l) { most = fmaxf(most, m), least = fminf(least, l); };
    step(lane_xor<1>(most), lane_xor<1>(least));
    step(lane_xor<2>(most), lane_xor<2>(least));
    step(lane_xor<4>(most), lane_xor<4>(least));
    step(lane_xor<8>(most), lane_xor<8>(least));
    step(lane_xor<16>(most), lane_xor<16>(least));
    step(lane_xor<32>(most), lane_xor<32>(least));
}

// The 64-point transform of every block (bh4_block.hip: bh4_fold_kernel), split, ready for the product kernel.  One workgroup per
// stage, a wavefront per block.  The weights are scaled by a power of two, so that lo needs no factor.  The 64 numbers of an input
// column of a block are fp32 sums of the same 64, so what the split leaves of a small one of them is as good as it was; but a
// column's size is that of the weights, and a small column meets a large input (forward) or gives a small gradient (backward).  So:
//   columns that all lie within SPAN of the stage's largest number are scaled together, that number to [2^14, 2^15); a column still has
//     22 bits down to 2^-9 of its own largest, and is held to 2^-31 of that below;
//   else every column of every block by itself, its largest to [2^14, 2^15), and the product kernel multiplies by the way back: the
//     forward its rows, before it takes their largest, the backward what it has formed.
// At 32768 tokens, D = 512, two repeats the second costs 8, 13 and 5 us of hash, training form and backward, the choice between them 0, 4
// and 0.  With one scale for a stage's column (sixteen of the forward's) in all blocks, as it was, the relative error was 4e-5 where columns
// are spread over 1e8 and their inputs the other way round, and 4e-4 in the gradient of a small block; so it is 1.2e-7 and 1.9e-7, as it is
// for numbers of one size (fp32 kernel 1.7e-7 and 2.8e-7).
// Per block and product wavefront four fragments of 64 lanes x 8 numbers: hi of the first and the second eight columns of a lane's
// sixteen, then lo of them; behind all blocks the way back of every column over 2^14, [stage][64 * num_block], 0 for a column of zeros
// (its input must not set its row's scale), and [stage] the one of the stage's scale or 0.
constexpr float SPAN = 1.f / 256;
template <bool TRANSPOSED>
__device__ __forceinline__ void fold_split(const float *w, uint32_t *out, float *back, float *together) {
    __shared__ float range_s[2][16];
    const int num_block = blockDim.x / 64, wave = threadIdx.x >> 6;
    const int64_t blk = int64_t(blockIdx.x) * num_block + wave;
    const int i = threadIdx.x & 63;
    const float *src = w + blk * (BS * BS) + i;
    float v[BS];
#pragma unroll
    for (int o = 0; o < BS; ++o) v[o] = src[o * BS];
#pragma unroll
    for (int h = BS / 2; h >= 1; h >>= 1) {
#pragma unroll
        for (int o = 0; o < BS; ++o) {
            if ((o & h) == 0) {
                const float lo = v[o], hi = v[o + h];
                v[o] = lo + hi;
                v[o + h] = lo - hi;
            }
        }
    }
    float most = 0.f;
#pragma unroll
    for (int o = 0; o < BS; ++o) most = fmaxf(most, fabsf(v[o]));
    float largest, least;
    wave_range(most, largest, least);
    range_s[0][wave] = largest, range_s[1][wave] = least;
    __syncthreads();
    for (int n = 0; n < num_block; ++n) largest = fmaxf(largest, range_s[0][n]), least = fminf(least, range_s[1][n]);
    const bool one = least >= largest * SPAN;                 // uniform
    const PowerOfTwo p = scale_to_one(one ? largest : most);
    const float f = p.scale * TOP;
    back[blk * BS + i] = most > 0.f ? p.inverse * (1 / TOP) : 0.f;
    if (threadIdx.x == 0) together[blockIdx.x] = one ? p.inverse * (1 / TOP) : 0.f;
    // eight consecutive k of a row of the A operand as hi and lo: fragment (row / 16, (k % 16) / 8), lane 16 (k / 16) + row % 16
    uint4 *const dst = reinterpret_cast<uint4 *>(out + blk * (BS * BS));
    auto store8 = [&](int row, int k, const float (&x)[8]) {
        uint32_t h[4], l[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            h[e] = split_hi(x[2 * e], x[2 * e + 1], 1.f);
            l[e] = split_rest(x[2 * e], x[2 * e + 1], h[e]);
        }
        const int at = ((row / 16) * 4 + (k % 16) / 8) * 64 + 16 * (k / 16) + row % 16;
        dst[at] = make_uint4(h[0], h[1], h[2], h[3]);
        dst[at + 128] = make_uint4(l[0], l[1], l[2], l[3]);
    };
    if constexpr (TRANSPOSED) {
#pragma unroll
        for (int k = 0; k < BS; k += 8) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = v[k + e] * f;
            store8(i, k, x);
        }
    } else {
        // a lane has a column of the block: sixteen rows at a time turned round through the wavefront's own 16 x 65 floats of LDS
        extern __shared__ float turn[];
        float *const t = turn + wave * (16 * 65);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int o = 0; o < 16; ++o) t[o * 65 + i] = v[16 * g + o] * f;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int row = i % 16, k = 16 * (i / 16) + 8 * m;
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = t[row * 65 + k + e];
                store8(16 * g + row, k, x);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
}

// One of the two forms, or both (gridDim.y 2: a training step's, in one launch)
__global__ __launch_bounds__(1024) void bh4_fold_split_kernel(const float *w, float *out, float *out_t, int64_t numbers) {
    if (blockIdx.y == 0 && out) fold_split<false>(w, reinterpret_cast<uint32_t *>(out), out + numbers, out + numbers + numbers / BS);
    else fold_split<true>(w, reinterpret_cast<uint32_t *>(out_t), out_t + numbers, out_t + numbers + numbers / BS);
}

struct SplitArgs {
    const float *x;        // [B, H]
    const float *ln_w;     // [H] LayerNorm weight, or null: no LayerNorm
    const float *ln_b;     // [H]
    float ln_eps;
    const float *w;        // split weights
    const float *wback;    // [R*J][D] the way back of their columns, [R*J] of a stage's together
    const float *pbias;    // [T*8] or null
    int32_t *codes;        // [B, T]
    float *scores;         // [B, T]
    uint32_t *records;     // instead of codes and scores: the record stream of the four-lanes-per-token gather,
    int64_t rec_stride;    // [T/2][rec_stride][3] (lffn_quad_record_slot)
    int rec_tile;          // tokens per workgroup of the gather the records are written for
    float *z;              // training: [B, T*8] z, kept for the backward (backward from scores: read)
    const float *g_score;  // backward from scores: [B, T] gradient of the scores
    float4 *clear;         // backward from scores: an array to clear on the way (the sum of the weights' gradient), or null
    int64_t clear_n;
    float *bias_parts;     // backward from scores: [ceil(B/16), T*8] column sums of the gradient of z, or null
    float *row_stats;      // training, with LayerNorm: [B, 2] every row's mean and 1/sigma
    const float *gz;       // backward: [B, T*8] gradient of z
    float *g_x;            // backward: [R, B, H]
    float *stage_save;     // training: [R, J-1, B, D] inputs of stages 1 .. J-1;
                           // backward: [R, J, B, D] gradient before the product of each stage
    int64_t B;
    int H, R, J, T;
    float decay, residual;
};

__device__ __forceinline__ f32x4 mfma16(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// hi and lo of four numbers
__device__ __forceinline__ void split4(f32x4 v, uint2 &hi, uint2 &lo) {
    hi = make_uint2(split_hi(v.x, v.y, 1.f), split_hi(v.z, v.w, 1.f));
    lo = make_uint2(split_rest(v.x, v.y, hi.x), split_rest(v.z, v.w, hi.y));
}

// A workgroup has 16 tokens: 4 wavefronts (BG = 1) of 16 output columns of every block each, or 16 for small batches (BG = 4), in
// which wavefront group bg has blocks bg, bg + 4, ...: the butterflies across a wavefront's own blocks (strides 4 and up) stay
// between accumulators, the last two (strides 2 and 1) are a pass over the tile in LDS.
// Both do the same operations in the same order: the results are those of the other form bit for bit.
//
// BWD: the backward through the stages with the same machinery.  With G_{s+1} the gradient of a stage's output, the gradient of its
// input is  W'_s^T (H_NB (x) I_64) G_{s+1}  (H_64 is symmetric and already inside W' = H_64 W): the butterflies across blocks run
// BEFORE the product, which takes the folded weights in transposed fragment order, and nothing follows it.  The butterflied
// gradient P_s = (H_NB (x) I) G_{s+1} is also written to memory: the gradient w.r.t. the folded weights is the per-block product
// P_s^T U_s over all tokens (U_s = the stage's input, which the forward saved), formed by the caller.  First gradient: decay * grad z;
// result: grad x of this repeat = G_0[:, :H] + residual * grad z[:, :H].
//
// SCORES_BACKWARD: the same from z and the scores' gradient.  The gradient of z is formed where it is used, at the start and for the
// residual, and its columns' sums, the projection bias's gradient, go out with it.  32768 x 512, two repeats: 263 us where a kernel that
// formed it took 48, this one 200 and the sums 24.  Written to g_x at the start and read back at the end instead: 288; the scores'
// derivatives kept by the training form instead of z: 260 to 273, and the forward longer.
enum Form { HASH, TRAIN, BACKWARD, SCORES_BACKWARD };       // TRAIN: the hash form that also keeps what the backward needs

template <int NB, Form FORM, int BG>
__global__ __launch_bounds__(256 * BG, BG > 1 || NB <= 8 ? 4 : 2) void bh4_split_kernel(SplitArgs a) {
    constexpr bool BWD = FORM >= BACKWARD;
    constexpr bool SCORES = FORM == SCORES_BACKWARD;
    constexpr bool SAVE = FORM != HASH;           // the numbers between the stages go to memory
    static_assert(BG == 1 || (BG == 4 && NB >= 4), "the wide form: four groups of blocks");
    constexpr int TOK = 16;                       // tokens per workgroup
    constexpr int NWAVE = 4 * BG;
    constexpr int NBW = NB / BG;                  // blocks of a wavefront: bg + BG * n, n < NBW
    const float *__restrict__ x = a.x;
    const int64_t B = a.B;
    const int H = a.H, J = a.J;
    constexpr int D = BS * NB;
    constexpr int LDR = D + PAD;                  // floats of a row in fp32
    constexpr int LDP = 4 * LDR;                  // bytes of a tile row, hi and lo: 16 rows' reads of a fragment fall on different banks
    constexpr int AHEAD = NBW < 2 ? NBW : 2;     // blocks whose weights are on their way
    extern __shared__ __attribute__((aligned(16))) char lds[];
    char *const tile = lds;                       // [TOK] rows of LDP bytes: hi, then lo
    // [TOK][LDR] in fp32: the narrow form's in the tile's place, where a row's two terms lie within its own numbers
    float *const rows32 = reinterpret_cast<float *>(lds + (BG > 1 ? TOK * LDP : 0));
    float *const stats = rows32 + TOK * LDR;      // [TOK][2]: LayerNorm's mean and 1/sigma
    float *const unscale = stats + 2 * TOK;       // [TOK] 1 / scale of a token's row
    float *const most_s = unscale + TOK;          // [TOK][4] largest of a token's row in a wavefront's columns
    float *const lnw_s = most_s + 4 * TOK;        // hash form: [D] each LayerNorm's weight and bias, the projection's bias
    float *const lnb_s = lnw_s + D, *const pbias_s = lnb_s + D;
    float *const xs = reinterpret_cast<float *>(lds);      // hash form, after the last stage: codes and scores

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ow = wave & 3;                      // output columns [16*ow, 16*ow + 16) of each block
    const int bg = wave >> 2;                     // group of blocks of this wavefront
    const int c = lane & 15;                      // A operand: output column; B operand and result: token
    const int kq = lane >> 4;                     // operands: columns 16*kq .. + 15 of the block; result: output columns 4*kq .. + 3
    // A workgroup takes one repeat of its tokens: few tokens with several repeats are as many workgroups more.  The repeats of
    // GROUP tiles come one after the other in the grid (on the same XCDs, as that is a multiple of their number), so that what they share, the
    // tokens' rows forward, lines and pages of z and of the scores' gradient backward, is read close together.  32768 tokens, D = 512, two
    // repeats, all tiles of a repeat after all of the one before -> groups of 128: backward 244 -> 231 us, hash 2 to 4 us of a layer's 259 (groups of 64
    // the same, 256 241 of 238, 512 248); but the training form 168 -> 173, which keeps the old order.
    constexpr unsigned GROUP = 128;
    unsigned repeat = blockIdx.y, tile_no = blockIdx.x;
    if constexpr (FORM != TRAIN) {
        const unsigned in_order = blockIdx.y * gridDim.x + blockIdx.x, group = in_order / (GROUP * gridDim.y);
        const unsigned group_tiles = min(GROUP, gridDim.x - group * GROUP), in_group = in_order - group * (GROUP * gridDim.y);
        repeat = in_group / group_tiles;
        tile_no = group * GROUP + in_group % group_tiles;
    }
    const int r = __builtin_amdgcn_readfirstlane(repeat);
    tile_no = __builtin_amdgcn_readfirstlane(tile_no);
    const int64_t tok_base = int64_t(tile_no) * TOK;
    if (!BWD) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        for (int e = tid * 4; e < D; e += 256 * NWAVE) {
            const f32x4 one = {1.f, 1.f, 1.f, 1.f};
            *reinterpret_cast<f32x4 *>(lnw_s + e) = e >= H ? zero : a.ln_w ? *reinterpret_cast<const f32x4 *>(a.ln_w + e) : one;
            *reinterpret_cast<f32x4 *>(lnb_s + e) = e < H && a.ln_w ? *reinterpret_cast<const f32x4 *>(a.ln_b + e) : zero;
            const int col = r * D + e;
            *reinterpret_cast<f32x4 *>(pbias_s + e) = a.pbias && col < a.T * 8 ? *reinterpret_cast<const f32x4 *>(a.pbias + col) : zero;
        }
        __syncthreads();
    }

    f32x4 acc[NBW];

    // this wavefront's weights of a block: four fragments of 1 KB (hi, hi, lo, lo)
    uint4 wq[AHEAD][4];
    auto load_w = [&](int s, int n) {
        if (n >= NBW) {                           // the next stage's first blocks (after the last stage: a harmless re-read)
            n -= NBW;
            s = BWD ? max(s - 1, 0) : min(s + 1, J - 1);
        }
        const float *p = a.w + (size_t)((r * J + s) * NB + n * BG + bg) * (BS * BS) + ow * 1024 + lane * 4;
#pragma unroll
        for (int q = 0; q < 4; ++q) wq[n % AHEAD][q] = *reinterpret_cast<const uint4 *>(p + q * 256);
    };
    // this lane's token values of block n: 16 numbers as hi and lo fragments
    auto read_x = [&](int n, uint4 (&f)[4]) {
        const char *p = tile + c * LDP + (n * BG + bg) * 128 + kq * 32;
        f[0] = *reinterpret_cast<const uint4 *>(p);
        f[1] = *reinterpret_cast<const uint4 *>(p + 16);
        f[2] = *reinterpret_cast<const uint4 *>(p + 2 * D);
        f[3] = *reinterpret_cast<const uint4 *>(p + 2 * D + 16);
    };
    // four numbers of a token's row into the tile
    auto put = [&](int row, int col, f32x4 v) {
        uint2 hi, lo;
        split4(v, hi, lo);
        char *p = tile + row * LDP + col * 2;
        *reinterpret_cast<uint2 *>(p) = hi;
        *reinterpret_cast<uint2 *>(p + 2 * D) = lo;
    };

    // What the accumulators are to be multiplied with: the weights' part, and the way back of the lane's token.
    constexpr float INV_W = BWD ? 1.f : 1 / TOP;
    float inv_x = 1.f;
    // the way back of a stage's weights, over 2^14: of all together, or 0 and of columns col .. + 3
    // (no store of this kernel meets the weights: a scalar load)
    const auto *const each = (const __attribute__((address_space(4))) float *)(uintptr_t)(a.wback + size_t(a.R) * J * D + r * J);
    auto together_of = [&](int s) { return each[s]; };
    // of the stage whose product is next and the one after, requested a stage ahead (a product's LDS reads would wait for it)
    float together = together_of(BWD ? J - 1 : 0), together_next = together_of(BWD ? max(J - 2, 0) : min(1, J - 1));
    auto back_of = [&](int s, int col) { return *reinterpret_cast<const f32x4 *>(a.wback + size_t(r * J + s) * D + col); };
    // v[i] times the way back of four columns (a few at a time: registers), over 2^14 times f
    auto go_back = [&](int s, auto &v, auto col, float f) {
        constexpr int N = sizeof(v) / sizeof(v[0]);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            v[i] = v[i] * (back_of(s, col(i)) * f);
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto own_col = [&](int n) { return (n * BG + bg) * BS + 16 * ow + 4 * kq; };       // of the lane's accumulator n

    // acc = (blocks of the stage's weights) x (the tile's tokens)
    auto product = [&](int s) {
        const float own = together;
        inv_x = own != 0.f ? unscale[c] * (own * (BWD ? 1.f : TOP)) : unscale[c];
        together = together_next;
        uint4 xv[2][4];
        read_x(0, xv[0]);
        static_for<NBW>([&](auto n_c) {
            constexpr int n = decltype(n_c)::value;
            if constexpr (n > 0) load_w(s, n - 1 + AHEAD);
            if constexpr (n + 1 < NBW) read_x(n + 1, xv[(n + 1) % 2]);
            __builtin_amdgcn_sched_barrier(0);
            // the small terms first
            const uint4 (&w)[4] = wq[n % AHEAD], (&x4)[4] = xv[n % 2];
            acc[n] = mfma16(w[2], x4[0], (f32x4){0.f, 0.f, 0.f, 0.f});
            acc[n] = mfma16(w[0], x4[2], acc[n]);
            acc[n] = mfma16(w[3], x4[1], acc[n]);
            acc[n] = mfma16(w[1], x4[3], acc[n]);
            acc[n] = mfma16(w[0], x4[0], acc[n]);
            acc[n] = mfma16(w[1], x4[1], acc[n]);
            __builtin_amdgcn_sched_barrier(0);
        });
        load_w(s, NBW - 1 + AHEAD);
        together_next = together_of(BWD ? max(s - 2, 0) : min(s + 2, J - 1));
        if (BWD && own == 0.f) go_back(s, acc, own_col, 1.f);                   // uniform
    };

    // H_NB across the blocks of the accumulators, from stride NB / 2 down (wide form: down to BG)
    auto butterflies = [&]() {
#pragma unroll
        for (int h = NBW / 2; h >= 1; h >>= 1) {
#pragma unroll
            for (int n = 0; n < NBW; ++n) {
                if ((n & h) == 0) {
                    const f32x4 lo = acc[n], hi = acc[n + h];
                    acc[n] = lo + hi;
                    acc[n + h] = lo - hi;
                }
            }
        }
    };

    // The accumulators times f as rows of fp32 in LDS, and the four rows of a wavefront from there, NB vectors a lane: vector i of
    // lane l is row row_of(i), columns col_of(i) .. + 3.
    constexpr int ROW_LANES = D < 256 ? D / 4 : 64, ROW_VALUES = D < 256 ? 1 : D / 256;
    auto row_of = [&](int i) { return 4 * wave + (D < 256 ? i * (64 / ROW_LANES) + lane / ROW_LANES : i / ROW_VALUES); };
    auto col_of = [&](int i) { return 4 * (lane % ROW_LANES) + (D < 256 ? 0 : 256 * (i % ROW_VALUES)); };
    auto to_rows = [&](float f) {
#pragma unroll
        for (int n = 0; n < NBW; ++n)
            *reinterpret_cast<f32x4 *>(rows32 + c * LDR + own_col(n)) = acc[n] * f;
    };
    auto from_rows = [&](f32x4 (&v)[NB]) {
#pragma unroll
        for (int i = 0; i < NB; ++i) v[i] = *reinterpret_cast<const f32x4 *>(rows32 + row_of(i) * LDR + col_of(i));
    };

    // The accumulators (after butterflies()) become the tile of the product of stage s, and the rows of D floats at `save` where they are
    // kept: a token's row, forward times the way back of the columns that it meets where those are not scaled together, is scaled by the power of two that takes its largest
    // to [2^14, 2^15).
    auto hand_over = [&](int s, float *save) {
        if constexpr (BG > 1) {
            // strides 2 and 1, which take four wavefronts' accumulators: a pass over the tile in fp32, 16 bytes of blocks
            // 4 n .. 4 n + 3 per thread; the 16 NBW threads of a row are neighbours in a wavefront
            to_rows(INV_W);
            if (bg == 0 && ow == 0 && kq == 0) unscale[c] = inv_x;
            __syncthreads();
            if (tid < TOK * 16 * NBW) {
                const int row = tid / (16 * NBW), n = (tid / 16) % NBW, c4 = (tid % 16) * 4;
                const float *p = rows32 + row * LDR + n * BG * BS + c4;
                const float inv = unscale[row];
                f32x4 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const f32x4 *>(p + k * BS);
                const f32x4 s0 = v[0] + v[2], s1 = v[1] + v[3], d0 = v[0] - v[2], d1 = v[1] - v[3];
                v[0] = s0 + s1; v[1] = s0 - s1; v[2] = d0 + d1; v[3] = d0 - d1;
                const bool live = SAVE && tok_base + row < B;
                if (live) {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        __builtin_nontemporal_store(v[k] * inv, reinterpret_cast<f32x4 *>(save + size_t(row) * D + (n * BG + k) * BS + c4));
                }
                if (!BWD && together == 0.f) go_back(s, v, [&](int k) { return (n * BG + k) * BS + c4; }, TOP);
                float most = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e) most = fmaxf(most, fabsf(v[k][e]));
                most = fmaxf(most, lane_xor<1>(most));
                most = fmaxf(most, lane_xor<2>(most));
                most = fmaxf(most, lane_xor<4>(most));
                most = fmaxf(most, lane_xor<8>(most));
                if constexpr (NBW > 1) most = fmaxf(most, lane_xor<16>(most));
                if constexpr (NBW > 2) most = fmaxf(most, lane_xor<32>(most));
                const PowerOfTwo p2 = scale_to_one(most);
                if (tid % (16 * NBW) == 0) unscale[row] = inv * (p2.inverse * (1 / TOP));
#pragma unroll
                for (int k = 0; k < 4; ++k) put(row, (n * BG + k) * BS + c4, v[k] * (p2.scale * TOP));
            }
            __syncthreads();
        } else if constexpr (SAVE) {
            // the rows go out as whole lines: through LDS in fp32, and a wavefront has four rows from there
            __syncthreads();                      // every wavefront has read this stage's input
            to_rows(INV_W);
            if (ow == 0 && kq == 0) unscale[c] = inv_x;
            __syncthreads();
            f32x4 v[NB];
            from_rows(v);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int row = row_of(i);
                if (tok_base + row < B) __builtin_nontemporal_store(v[i] * unscale[row], reinterpret_cast<f32x4 *>(save + size_t(row) * D + col_of(i)));
            }
            if (!BWD && together == 0.f) go_back(s, v, col_of, TOP);
#pragma unroll
            for (int i = 0; i < NB; i += ROW_VALUES) {
                const int row = row_of(i);
                const float inv = unscale[row];
                float most = 0.f;
#pragma unroll
                for (int k = i; k < i + ROW_VALUES; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e) most = fmaxf(most, fabsf(v[k][e]));
                most = fmaxf(most, lane_xor<1>(most));
                most = fmaxf(most, lane_xor<2>(most));
                most = fmaxf(most, lane_xor<4>(most));
                most = fmaxf(most, lane_xor<8>(most));
                if constexpr (ROW_LANES == 32) most = fmaxf(most, lane_xor<16>(most));
                if constexpr (ROW_LANES == 64) most = rows_most(most);
                const PowerOfTwo p2 = scale_to_one(most);
#pragma unroll
                for (int k = i; k < i + ROW_VALUES; ++k) put(row, col_of(k), v[k] * (p2.scale * TOP));
                if (lane % ROW_LANES == 0) unscale[row] = inv * (p2.inverse * (1 / TOP));
            }
            __syncthreads();
        } else {
            if (together == 0.f) go_back(s, acc, own_col, TOP);
            f32x4 m4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int n = 0; n < NBW; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) m4[e] = fmaxf(m4[e], fabsf(acc[n][e]));
            m4 = m4 * INV_W;
            const float most = rows_most(fmaxf(fmaxf(m4.x, m4.y), fmaxf(m4.z, m4.w)));
            if (kq == 0) most_s[c * 4 + ow] = most;
            __syncthreads();                      // every wavefront has read this stage's input and left its largest
            const float4 m = *reinterpret_cast<const float4 *>(most_s + c * 4);
            const PowerOfTwo p2 = scale_to_one(fmaxf(fmaxf(m.x, m.y), fmaxf(m.z, m.w)));
            if (kq == 0 && ow == 0) unscale[c] = inv_x * (p2.inverse * (1 / TOP));
#pragma unroll
            for (int n = 0; n < NBW; ++n) put(c, own_col(n), acc[n] * (INV_W * TOP * p2.scale));
            __syncthreads();
        }
    };
    // wide form, after the last stage: the accumulators of strides 2 and 1 as well
    auto last_strides = [&]() {
        if constexpr (BG > 1) {
#pragma unroll
            for (int n = 0; n < NBW; ++n)
                *reinterpret_cast<f32x4 *>(rows32 + c * LDR + (n * BG + bg) * BS + 16 * ow + 4 * kq) = acc[n];
            __syncthreads();
            if (tid < TOK * 16 * NBW) {
                const int row = tid / (16 * NBW), n = (tid / 16) % NBW, c4 = (tid % 16) * 4;
                float *p = rows32 + row * LDR + n * BG * BS + c4;
                f32x4 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const f32x4 *>(p + k * BS);
                const f32x4 s0 = v[0] + v[2], s1 = v[1] + v[3], d0 = v[0] - v[2], d1 = v[1] - v[3];
                v[0] = s0 + s1; v[1] = s0 - s1; v[2] = d0 + d1; v[3] = d0 - d1;
#pragma unroll
                for (int k = 0; k < 4; ++k) *reinterpret_cast<f32x4 *>(p + k * BS) = v[k];
            }
            __syncthreads();
#pragma unroll
            for (int n = 0; n < NBW; ++n)
                acc[n] = *reinterpret_cast<const f32x4 *>(rows32 + c * LDR + (n * BG + bg) * BS + 16 * ow + 4 * kq);
        }
    };

#pragma unroll
    for (int n = 0; n < AHEAD; ++n) load_w(BWD ? J - 1 : 0, n);
    // Backward from scores: the workgroup's tokens' rows as NBW vectors of four columns a thread, a few
    // at a time; two neighbouring lanes have the eight columns of a score.
    auto z_gradient = [&](f32x4 z, float g) {
        const float zq[4] = {z.x, z.y, z.z, z.w};
        const ScorePart own = score_part(zq);
        const float twice = 2.0f * (own.sum + lane_xor<1>(own.sum)), g_over_p = g / (own.product * lane_xor<1>(own.product));
        f32x4 out;
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = score_derivative(zq[e], own.away[e], twice, g_over_p);
        return out;
    };
    auto z_gradients = [&](auto take) {
        constexpr int FEW = NBW < 4 ? NBW : 4;
        // (nontemporal, both times: kept, z would push out what the stages write, 32768 x 512 10 us of the step)
#pragma unroll 1
        for (int i0 = 0; i0 < NBW; i0 += FEW) {
            f32x4 z[FEW];
            float g[FEW];
            int at[FEW];
#pragma unroll
            for (int i = 0; i < FEW; ++i) {
                at[i] = tid + (i0 + i) * 256 * BG;
                const int64_t tok = min(tok_base + at[i] / (D / 4), B - 1);
                const int col = r * D + 4 * (at[i] % (D / 4));
                const bool in = col < a.T * 8;
                z[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(a.z + tok * (a.T * 8) + (in ? col : 0)));
                g[i] = a.g_score[tok * a.T + (in ? col / 8 : 0)];
                if (!in || tok_base + at[i] / (D / 4) >= B) g[i] = 0.f, z[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int i = 0; i < FEW; ++i) take(at[i] / (D / 4), 4 * (at[i] % (D / 4)), z_gradient(z[i], g[i]));
        }
    };
    if constexpr (BWD) {
        const int ncols = a.T * 8;
        // The matrix cores' sums are off to one side by a little, a twentieth of what a result is off in any direction; the gradient
        // of the weights, a sum over the tokens, would keep that, so every other token's row has its sign turned on the way.
        inv_x = c & 1 ? -1.f : 1.f;
        if constexpr (SCORES) {
            if (a.clear)
                for (int64_t i = (int64_t(blockIdx.y) * gridDim.x + blockIdx.x) * (256 * BG) + tid; i < a.clear_n;
                     i += int64_t(gridDim.x) * gridDim.y * (256 * BG))
                    a.clear[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            z_gradients([&](int row, int col, f32x4 g) { *reinterpret_cast<f32x4 *>(rows32 + row * LDR + col) = g; });
            __syncthreads();
            if (a.bias_parts) {
                for (int e = tid; e < D && r * D + e < ncols; e += 256 * BG) {
                    float sum = 0.f;
#pragma unroll
                    for (int t = 0; t < TOK; ++t) sum += rows32[t * LDR + e];
                    a.bias_parts[size_t(tile_no) * ncols + r * D + e] = sum;
                }
            }
#pragma unroll
            for (int n = 0; n < NBW; ++n)
                acc[n] = (a.decay * inv_x) * *reinterpret_cast<const f32x4 *>(rows32 + c * LDR + (n * BG + bg) * BS + 16 * ow + 4 * kq);
            if constexpr (BG > 1) __syncthreads();             // (the narrow form's hand_over begins with one)
        } else {
#pragma unroll
            for (int n = 0; n < NBW; ++n) {
                const int gcol = r * D + (n * BG + bg) * BS + 16 * ow + 4 * kq;
                f32x4 g = {0.f, 0.f, 0.f, 0.f};
                if (tok_base + c < B && gcol < ncols) g = *reinterpret_cast<const f32x4 *>(a.gz + (tok_base + c) * ncols + gcol);
                acc[n] = (a.decay * inv_x) * g;
            }
        }
#pragma unroll 1
        for (int s = J - 1; s >= 0; --s) {
            butterflies();
            hand_over(s, a.stage_save + ((size_t(r) * J + s) * B + tok_base) * D);
            product(s);
        }
    } else {
        // Sixteen lanes have a row (wide form: a wavefront, its sixteens every fourth 64 columns), 16 bytes a lane of every 64
        // columns, all loads in flight before the first use.  Columns at or beyond H are zero.  Sums are taken over every fourth 64
        // columns of a lane, then those, then the sixteen lanes, in either form.
        constexpr int QG = BG > 1 ? 4 : 1, NQ = NB / QG, SG = NB < 4 ? NB : 4, LANES = 16 * QG;
        const int l = tid & 15, g = QG > 1 ? (tid >> 4) & 3 : 0;
        auto row_sum = [&](const float (&part)[NQ]) {
            float sum[SG] = {};
#pragma unroll
            for (int i = 0; i < NQ; ++i) sum[QG > 1 ? 0 : i % SG] += part[i];
            float v = sum[0];
            if constexpr (QG > 1) {
                v += lane_xor<16>(v);
                v += lane_xor<32>(v);
            } else {
                if constexpr (SG > 1) v += sum[1];
                if constexpr (SG > 2) v += sum[2] + sum[3];
            }
            return lane_group_sum<16>(v);
        };
#pragma unroll
        for (int row = tid / LANES; row < TOK; row += 64 * NWAVE / LANES) {
            const int64_t tok = tok_base + row;
            const float *px = x + min(tok, B - 1) * H;
            f32x4 v[NQ];
            float part[NQ];
            auto column = [&](int i) { return (g + i * QG) * 64 + 4 * l; };
#pragma unroll
            for (int i = 0; i < NQ; ++i) v[i] = *reinterpret_cast<const f32x4 *>(px + min(column(i), H - 4));
            if (tok >= B || H < D) {
#pragma unroll
                for (int i = 0; i < NQ; ++i)
                    if (tok >= B || column(i) >= H) v[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
            if (a.ln_w) {
                // LayerNorm over the H valid columns (biased variance, two passes, eps inside the
                // square root: torch.nn.LayerNorm, PL/lookup.py:84,99)
#pragma unroll
                for (int i = 0; i < NQ; ++i) part[i] = (v[i].x + v[i].y) + (v[i].z + v[i].w);
                const float mean = row_sum(part) / float(H);
#pragma unroll
                for (int i = 0; i < NQ; ++i) {
                    v[i] = v[i] - mean;
                    const f32x4 sq = v[i] * v[i];
                    part[i] = (sq.x + sq.y) + (sq.z + sq.w);
                }
                if (H < D) {
#pragma unroll
                    for (int i = 0; i < NQ; ++i)
                        if (column(i) >= H) part[i] = 0.f;
                }
                const float rstd = 1.0f / sqrtf(row_sum(part) / float(H) + a.ln_eps);
#pragma unroll
                for (int i = 0; i < NQ; ++i)          // (weight and bias are zero beyond column H)
                    v[i] = v[i] * rstd * *reinterpret_cast<const f32x4 *>(lnw_s + column(i)) +
                           *reinterpret_cast<const f32x4 *>(lnb_s + column(i));
                if (tid % LANES == 0) {
                    stats[2 * row] = mean;
                    stats[2 * row + 1] = rstd;
                    if (SAVE && r == 0 && tok < B) *reinterpret_cast<float2 *>(a.row_stats + 2 * tok) = make_float2(mean, rstd);
                }
            }
            if (together == 0.f) go_back(0, v, column, TOP);
            float most = 0.f;
#pragma unroll
            for (int i = 0; i < NQ; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) most = fmaxf(most, fabsf(v[i][e]));
            most = fmaxf(most, lane_xor<1>(most));
            most = fmaxf(most, lane_xor<2>(most));
            most = fmaxf(most, lane_xor<4>(most));
            most = fmaxf(most, lane_xor<8>(most));
            if constexpr (QG > 1) {
                most = fmaxf(most, lane_xor<16>(most));
                most = fmaxf(most, lane_xor<32>(most));
            }
            const PowerOfTwo s = scale_to_one(most);
            if (tid % LANES == 0) unscale[row] = s.inverse * (1 / TOP);
#pragma unroll
            for (int i = 0; i < NQ; ++i) put(row, column(i), v[i] * (s.scale * TOP));
        }
        __syncthreads();
#pragma unroll 1
        for (int s = 0; s < J; ++s) {
            product(s);
            butterflies();
            if (s + 1 < J) hand_over(s + 1, SAVE ? a.stage_save + ((size_t(r) * (J - 1) + s) * B + tok_base) * D : nullptr);
        }
        last_strides();
    }
    const int64_t token = tok_base + c;
    if constexpr (BWD) {
        // grad x of this repeat: the first H columns, plus the residual path of the mix
        const int ncols = a.T * 8;
        if constexpr (SCORES) {                   // whole rows again
            __syncthreads();
            to_rows(inv_x);
            __syncthreads();
            z_gradients([&](int row, int col, f32x4 g) {
                f32x4 v = *reinterpret_cast<const f32x4 *>(rows32 + row * LDR + col);
                v = v + a.residual * g;           // (beyond T*8 columns: 0)
                if (tok_base + row < B && col < H) *reinterpret_cast<f32x4 *>(a.g_x + (size_t(r) * B + tok_base + row) * H + col) = v;
            });
        } else if constexpr (BG == 1) {
            __syncthreads();
            to_rows(inv_x);
            __syncthreads();
            f32x4 v[NB];
            from_rows(v);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int64_t tok = tok_base + row_of(i);
                const int xc = col_of(i);
                if (tok < B && xc < H) {
                    if (r * D + xc < ncols) v[i] = v[i] + a.residual * *reinterpret_cast<const f32x4 *>(a.gz + tok * ncols + r * D + xc);
                    *reinterpret_cast<f32x4 *>(a.g_x + (size_t(r) * B + tok) * H + xc) = v[i];
                }
            }
        } else if (token < B) {
#pragma unroll
            for (int n = 0; n < NBW; ++n) {
                const int xc = (n * BG + bg) * BS + 16 * ow + 4 * kq;
                if (xc < H) {
                    f32x4 o = acc[n] * inv_x;
                    if (r * D + xc < ncols) o = o + a.residual * *reinterpret_cast<const f32x4 *>(a.gz + token * ncols + r * D + xc);
                    *reinterpret_cast<f32x4 *>(a.g_x + (size_t(r) * B + token) * H + xc) = o;
                }
            }
        }
    } else {
        __syncthreads();                          // the tile has been read: it takes the codes and scores
        const int ncols = a.T * 8;
        constexpr int CROW = D / 8 + 1;                // padded: tokens down a column hit different banks
        int *cs = reinterpret_cast<int *>(xs);         // [TOK][CROW] codes of this repeat
        float *ss = xs + TOK * CROW;                   // [TOK][CROW] scores
        // the addresses below do not change from stage to stage; computed from an opaque
        // zero they are formed here instead of being kept in registers through the stages
        int opq = 0;
        asm volatile("" : "+v"(opq));
        const float mean = a.ln_w ? stats[2 * (c + opq)] : 0.f, rstd = a.ln_w ? stats[2 * (c + opq) + 1] : 1.f;
        // the token's input values for every block, all requested before the first use (tokens and columns beyond the end: the last
        // ones again, whose results go nowhere)
        f32x4 xin[NBW];
        const float *px = x + min(token + opq, B - 1) * H;
#pragma unroll
        for (int n = 0; n < NBW; ++n) xin[n] = *reinterpret_cast<const f32x4 *>(px + min((n * BG + bg) * BS + 16 * ow + 4 * kq, H - 4));
        __builtin_amdgcn_sched_barrier(0);
        // z of the lane's four columns of block n
        auto form_z = [&](int n) {
            const int xc = (n * BG + bg) * BS + 16 * ow + 4 * kq + opq;    // column of the padded input
            // (without LayerNorm or bias: 0, 1, 1, 0 and 0; the weight is zero beyond column H)
            const f32x4 xv = (xin[n] - mean) * rstd * *reinterpret_cast<const f32x4 *>(lnw_s + xc) +
                             *reinterpret_cast<const f32x4 *>(lnb_s + xc);
            const f32x4 z = a.decay * (INV_W * inv_x) * acc[n] + a.residual * xv +      // (decay times a power of two: as decay * y)
                            *reinterpret_cast<const f32x4 *>(pbias_s + xc);
            if (SAVE && BG > 1 && token < B && r * D + xc < ncols)
                __builtin_nontemporal_store(z, reinterpret_cast<f32x4 *>(a.z + token * ncols + r * D + xc));
            return z;
        };
        if constexpr (SAVE && BG == 1) {          // z as whole rows
#pragma unroll
            for (int n = 0; n < NBW; ++n) acc[n] = form_z(n);
            to_rows(1.f);
            __syncthreads();
            f32x4 v[NB];
            from_rows(v);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int64_t tok = tok_base + row_of(i);
                const int col = r * D + col_of(i);
                if (tok < B && col < ncols) __builtin_nontemporal_store(v[i], reinterpret_cast<f32x4 *>(a.z + tok * ncols + col));
            }
            __syncthreads();
        }
        auto z_of = [&](int n) {
            if constexpr (SAVE && BG == 1) return acc[n];
            else return form_z(n);
        };
        // Columns 8 g .. 8 g + 3 sit in the lane with even kq, 8 g + 4 .. 8 g + 7 in lane + 16.  Two groups of four are taken at a
        // time and exchanged between the lanes' rows, so that an even row has all eight columns of the first and an odd row of the
        // second: code, sum and product in column order (compute_code_score/torch_extension.cc:31-37), one division a lane.
        constexpr int ITEMS = NBW;
#pragma unroll
        for (int i = 0; i < ITEMS; i += 2) {
            const int i1 = i + 1 < ITEMS ? i + 1 : i;              // (a single one: with itself, the odd rows' copy is not used)
            const f32x4 za = z_of(i), zb = z_of(i1);
            float z[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const auto pair = __builtin_amdgcn_permlane16_swap(__float_as_uint(za[e]), __float_as_uint(zb[e]), false, false);
                z[e] = __uint_as_float(pair[0]);
                z[e + 4] = __uint_as_float(pair[1]);
            }
            int code = 0;
            float sum = fabsf(z[0]), prod = 1.0f + exp_minus_2a(fabsf(z[0]));
#pragma unroll
            for (int e = 0; e < 8; ++e)
                asm("v_cmp_lt_f32 vcc, 0, %1\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(code) : "v"(z[e]) : "vcc");
#pragma unroll
            for (int e = 1; e < 8; ++e) {
                sum = sum + fabsf(z[e]);
                prod = prod * (1.0f + exp_minus_2a(fabsf(z[e])));
            }
            // staged in LDS, written out row by row below: straight from here a store would scatter 4-byte pieces over 32 rows
            const bool odd = kq & 1;
            const int at = c * CROW + ((odd ? i1 : i) * BG + bg) * 8 + 2 * ow + (kq >> 1);
            if (ITEMS > 1 || !odd) {
                cs[at] = code;
                ss[at] = sum / prod;
            }
        }
        __syncthreads();
        if (a.records) {
            // records: per table pair three words per token, the workgroup's TOK tokens (whole
            // groups of 16: 192 contiguous bytes each) side by side; a token whose index has bit 1
            // set takes the pair's tables in the order (2k+1, 2k)
            static_assert((64 * NWAVE) % TOK == 0, "a thread stays on one token");
            const int row = tid % TOK;
            const int64_t tok = tok_base + row;
            const int64_t slot = tok < B ? lffn_quad_record_slot(tok, a.rec_tile) : 0;
            for (int kk = tid / TOK; kk < D / 16; kk += 64 * NWAVE / TOK) {
                const int pair = r * (D / 16) + kk;
                if (tok < B && 2 * pair + 1 < a.T) {
                    const int ca = cs[row * CROW + 2 * kk], cb = cs[row * CROW + 2 * kk + 1];
                    const float sa = ss[row * CROW + 2 * kk], sb = ss[row * CROW + 2 * kk + 1];
                    const bool second_first = (tok & 2) != 0;
                    uint32_t *dst = a.records + ((size_t)pair * a.rec_stride + slot) * LFFN_RECORD_WORDS;
                    dst[0] = __float_as_uint(second_first ? sb : sa);
                    dst[1] = __float_as_uint(second_first ? sa : sb);
                    dst[2] = second_first ? (unsigned)(cb | (ca << 8)) : (unsigned)(ca | (cb << 8));
                }
            }
        } else {
            // every wavefront writes the D/8 codes and scores of TOK/NWAVE tokens
#pragma unroll 1
            for (int i = 0; i < TOK / NWAVE; ++i) {
                const int row = wave * (TOK / NWAVE) + i;
                const int64_t tok = tok_base + row;
                if (tok >= B) break;
#pragma unroll
                for (int e0 = 0; e0 < D / 8; e0 += 64) {
                    const int e = e0 + lane;
                    const int tt = r * (D / 8) + e;
                    if (e < D / 8 && tt < a.T) {
                        a.codes[tok * a.T + tt] = cs[row * CROW + e];
                        a.scores[tok * a.T + tt] = ss[row * CROW + e];
                    }
                }
            }
        }
    }
}

template <int NB, Form FORM, int BG>
int launch_form(const SplitArgs &a, hipStream_t st) {
    constexpr int TOK = 16, D = BS * NB;
    constexpr size_t lds_bytes = (BG > 1 ? 2 : 1) * TOK * (D + PAD) * 4 + 7 * TOK * 4 + (FORM >= BACKWARD ? 0 : 3 * D * 4);
    static_assert(lds_bytes <= 160 * 1024);
    auto kern = bh4_split_kernel<NB, FORM, BG>;
    static LdsGrant granted;      // one record per kernel instantiation
    if (!lffn_grant_dynamic_lds(reinterpret_cast<const void *>(kern), lds_bytes, granted)) return LFFN_ERR_LAUNCH;
    const dim3 grid((unsigned)((a.B + TOK - 1) / TOK), (unsigned)a.R);
    hipLaunchKernelGGL(kern, grid, dim3(256 * BG), lds_bytes, st, a);
    return lffn_launch_status();
}

// The wide form where its workgroups leave no compute unit a second one: there 4 wavefronts wait for every latency of their own.
// Forward / backward, 4 -> 16 wavefronts: 2103 tokens, D = 1024 23.7 -> 20.9 / 31.2 -> 21.5 us; 385, D = 512 12.3 both / 15.3 ->
// 12.2; 600, D = 256, four repeats 9.6 -> 9.7 / 10.4 -> 9.4.  Two rounds of it: 4096, D = 512, two repeats 19.1 -> 26.8 / 30.7 -> 29.7.
constexpr int64_t WIDE_WORKGROUPS = 256;

template <int NB, Form FORM>
int launch_block(const SplitArgs &a, hipStream_t st) {
    if constexpr (NB >= 4)
        if ((a.B + 15) / 16 * a.R <= WIDE_WORKGROUPS) return launch_form<NB, FORM, 4>(a, st);
    return launch_form<NB, FORM, 1>(a, st);
}

template <Form FORM>
int dispatch_block(const SplitArgs &a, int64_t D, hipStream_t st) {
    switch (D / BS) {
        case 1: return launch_block<1, FORM>(a, st);
        case 2: return launch_block<2, FORM>(a, st);
        case 4: return launch_block<4, FORM>(a, st);
        case 8: return launch_block<8, FORM>(a, st);
        default: return launch_block<16, FORM>(a, st);
    }
}

}  // namespace

namespace {

int fold_split_entry(const float *w, float *out, float *out_t, int64_t stages, int64_t num_block, int64_t block_size, void *stream) {
    LFFN_REQUIRE(stages >= 0 && stages <= (1 << 20) && num_block >= 1, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(block_size == BS && lffn_is_pow2(num_block) && num_block <= 16, LFFN_ERR_UNSUPPORTED);
    if (stages == 0) return LFFN_OK;
    LFFN_REQUIRE(w && (out || out_t) && w != out && w != out_t && lffn_aligned16(out) && lffn_aligned16(out_t), LFFN_ERR_BAD_ARG);
    const size_t lds = out ? num_block * 16 * 65 * sizeof(float) : 0;
    static LdsGrant granted;
    if (lds > 50000 && !lffn_grant_dynamic_lds(reinterpret_cast<const void *>(bh4_fold_split_kernel), lds, granted)) return LFFN_ERR_LAUNCH;
    hipLaunchKernelGGL(bh4_fold_split_kernel, dim3((unsigned)stages, out && out_t ? 2 : 1), dim3((unsigned)(BS * num_block)), lds,
                       static_cast<hipStream_t>(stream), w, out, out_t, stages * num_block * (BS * BS));
    return lffn_launch_status();
}

}  // namespace

extern "C" int lffn_bh4_fold_split_f32(const float *w, float *w_split, int64_t stages, int64_t num_block, int64_t block_size,
                                       int32_t transposed, void *stream) {
    return fold_split_entry(w, transposed ? nullptr : w_split, transposed ? w_split : nullptr, stages, num_block, block_size, stream);
}

extern "C" int lffn_bh4_fold_split_both_f32(const float *w, float *w_split, float *w_split_t, int64_t stages, int64_t num_block,
                                            int64_t block_size, void *stream) {
    LFFN_REQUIRE(stages == 0 || (w_split && w_split_t && w_split != w_split_t), LFFN_ERR_BAD_ARG);
    return fold_split_entry(w, w_split, w_split_t, stages, num_block, block_size, stream);
}

namespace {

// the hash forms' arguments, checked
int front_args(const lffn_block_front *f, const float *x, int64_t B, SplitArgs &a) {
    LFFN_REQUIRE(f, LFFN_ERR_BAD_ARG);
    const int64_t H = f->H, D = f->D, R = f->R, J = f->J, T = f->T;
    LFFN_REQUIRE(B >= 0 && R >= 1 && J >= 1 && D >= 1 && H >= 1 && H <= D && T >= 0, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(H % 4 == 0 && J <= 64, LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(lffn_is_pow2(D) && D >= BS && D <= 1024, LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(R <= 4096 && B <= (int64_t(1) << 31) - 1 && T <= (1 << 24), LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(T * 8 <= R * D, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(!f->ln_weight || (f->ln_bias && f->ln_eps >= 0.f), LFFN_ERR_BAD_ARG);
    if (B == 0 || T == 0) return LFFN_OK;
    LFFN_REQUIRE(x && f->w_split && (f->records || (f->codes && f->scores)), LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(!f->records || (T % 2 == 0 && lffn_record_layout_ok(B, f->record_stride, f->tokens_per_workgroup) &&
                                 (uintptr_t)f->records % 4 == 0), LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(x) && lffn_aligned16(f->w_split) && lffn_aligned16(f->proj_bias) && lffn_aligned16(f->ln_weight) &&
                     lffn_aligned16(f->ln_bias), LFFN_ERR_BAD_ARG);
    a.x = x; a.ln_w = f->ln_weight; a.ln_b = f->ln_bias; a.ln_eps = f->ln_eps; a.w = f->w_split;
    a.wback = f->w_split + R * J * D * BS; a.pbias = f->proj_bias; a.codes = f->codes; a.scores = f->scores;
    a.records = f->records; a.rec_stride = f->record_stride; a.rec_tile = f->tokens_per_workgroup;
    a.B = B; a.H = (int)H; a.R = (int)R; a.J = (int)J; a.T = (int)T; a.decay = f->decay; a.residual = f->residual;
    return LFFN_OK;
}

}  // namespace

extern "C" int lffn_bh4_block_front_split_f32(const lffn_block_front *f, const float *x, int64_t B, void *stream) {
    SplitArgs a{};
    const int rc = front_args(f, x, B, a);
    return rc != LFFN_OK || B == 0 || f->T == 0 ? rc : dispatch_block<HASH>(a, f->D, static_cast<hipStream_t>(stream));
}

extern "C" int lffn_bh4_block_front_train_split_f32(const lffn_block_front *f, const float *x, float *z, float *stage_inputs,
                                                     float *row_stats, int64_t B, void *stream) {
    SplitArgs a{};
    const int rc = front_args(f, x, B, a);
    if (rc != LFFN_OK || B == 0 || f->T == 0) return rc;
    LFFN_REQUIRE(f->codes && f->scores && !f->records && z && (stage_inputs || f->J == 1) && (row_stats || !f->ln_weight), LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(z) && lffn_aligned16(stage_inputs) && (uintptr_t)row_stats % 8 == 0, LFFN_ERR_BAD_ARG);
    a.z = z; a.stage_save = stage_inputs; a.row_stats = row_stats;
    return dispatch_block<TRAIN>(a, f->D, static_cast<hipStream_t>(stream));
}

namespace {

__global__ __launch_bounds__(256) void clear_kernel(float4 *p, int64_t n) {
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// the backwards' arguments, checked
int back_args(const float *w_split_t, float *g_x, float *stage_grads, int64_t B, int64_t H, int64_t D, int64_t R, int64_t J, int64_t T,
              int64_t block_size, float decay, float residual, SplitArgs &a) {
    LFFN_REQUIRE(B >= 0 && R >= 1 && J >= 1 && D >= 1 && H >= 1 && H <= D && T >= 1, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(H % 4 == 0 && J <= 64, LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(block_size == BS && lffn_is_pow2(D) && D >= BS && D <= 1024, LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(R <= 4096 && B <= (int64_t(1) << 31) - 1 && T <= (1 << 24), LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(T * 8 <= R * D, LFFN_ERR_BAD_ARG);
    if (B == 0) return LFFN_OK;
    LFFN_REQUIRE(w_split_t && g_x && stage_grads, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(w_split_t) && lffn_aligned16(g_x) && lffn_aligned16(stage_grads), LFFN_ERR_BAD_ARG);
    a.w = w_split_t; a.wback = w_split_t + R * J * D * BS; a.g_x = g_x; a.stage_save = stage_grads;
    a.B = B; a.H = (int)H; a.R = (int)R; a.J = (int)J; a.T = (int)T; a.decay = decay; a.residual = residual;
    return LFFN_OK;
}

}  // namespace

extern "C" int lffn_bh4_block_bwd_split_f32(const float *g_z, const float *w_split_t, float *g_x, float *stage_grads, int64_t B,
                                            int64_t H, int64_t D, int64_t R, int64_t J, int64_t T, int64_t block_size, float decay,
                                            float residual, void *stream) {
    SplitArgs a{};
    const int rc = back_args(w_split_t, g_x, stage_grads, B, H, D, R, J, T, block_size, decay, residual, a);
    if (rc != LFFN_OK || B == 0) return rc;
    LFFN_REQUIRE(g_z && lffn_aligned16(g_z), LFFN_ERR_BAD_ARG);
    a.gz = g_z;
    return dispatch_block<BACKWARD>(a, D, static_cast<hipStream_t>(stream));
}

extern "C" int lffn_bh4_block_score_bwd_split_f32(const float *z, const float *g_score, const float *w_split_t, float *g_x,
                                                  float *stage_grads, float *bias_parts, float *clear, int64_t clear_n, int64_t B,
                                                  int64_t H, int64_t D, int64_t R, int64_t J, int64_t T, int64_t block_size, float decay,
                                                  float residual, void *stream) {
    SplitArgs a{};
    const int rc = back_args(w_split_t, g_x, stage_grads, B, H, D, R, J, T, block_size, decay, residual, a);
    if (rc != LFFN_OK) return rc;
    LFFN_REQUIRE(!clear || (clear_n >= 0 && clear_n % 4 == 0 && lffn_aligned16(clear)), LFFN_ERR_BAD_ARG);
    if (B == 0) {                                 // nothing but that
        if (!clear || clear_n == 0) return LFFN_OK;
        hipLaunchKernelGGL(clear_kernel, dim3((unsigned)std::min<int64_t>((clear_n / 4 + 255) / 256, 4096)), dim3(256), 0,
                           static_cast<hipStream_t>(stream), reinterpret_cast<float4 *>(clear), clear_n / 4);
        return lffn_launch_status();
    }
    LFFN_REQUIRE(z && g_score && lffn_aligned16(z), LFFN_ERR_BAD_ARG);
    a.clear = reinterpret_cast<float4 *>(clear); a.clear_n = clear ? clear_n / 4 : 0;
    a.z = const_cast<float *>(z); a.g_score = g_score; a.bias_parts = bias_parts;
    return dispatch_block<SCORES_BACKWARD>(a, D, static_cast<hipStream_t>(stream));
}
