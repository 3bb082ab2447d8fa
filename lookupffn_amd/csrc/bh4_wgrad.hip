// Weight gradient of the BH4 stages with 64x64 blocks: for every stage s = (r, j) and block n
//
//   g[s][n][o][i] += sum over tokens b of  p[s][b][64n + o] * u[s][b][64n + i]
//
// p[s]: [B, D] the gradient in front of the stage's block product (what lffn_bh4_block_bwd_f32
// writes), u[s]: the stage's input: x [B, H], zero beyond column H, for j = 0, else the saved
// input [B, D] of stage j (what lffn_bh4_block_hash_train_f32 keeps).  With ln_w the stage-0 input is
// LayerNorm(x), formed on load from x and the rows' kept mean and 1/sigma (the forward's LayerNorm ran
// inside its kernel and the normalised rows were never stored).  A batched product
// with a tiny output (64x64 per block) and a long sum (all tokens): one workgroup takes one
// block and a chunk of tokens, each of its four wavefronts sums a quarter of the chunk into a
// full 64x64 tile on the fp32 matrix cores (16 accumulator tiles), the four tiles are added in
// LDS and the workgroup adds its result to g with global atomics (g must hold the value to
// accumulate into, e.g. zero).
//
// Operands: a lane loads 16 bytes of a token's row of the block, lanes 0-15 cover the 256-byte
// row, the four lane groups take four consecutive tokens (the k index of
// v_mfma_f32_16x16x4_f32).  The four values of a lane feed four different output tiles, so
// tile j holds rows/columns 4*c + j (c = lane % 16): a fixed permutation undone when the tile
// is written.
#include "lffn_common.h"

#include <hip/amd_detail/amd_hip_unsafe_atomics.h>

// LayerNorm on load repeats the forward kernel's operations one by one: no fused multiply-add
#pragma clang fp contract(off)

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int BS = 64;
// Tokens per workgroup.  Every workgroup ends in 4096 atomic additions to the result, and too few workgroups leave the chip idle.  us
// at chunks of 4096 | 2048 | 1024 | 512 | 256 | 128 | 64 tokens (with LayerNorm in the first stage):
//   32768 tokens, D = 512, two repeats of four stages  237 | 209 | 208 | 216
//   16384, D = 1024, H = 768, one repeat               112 | 108 | 116 | 113
//    4096, D = 512                                                   25 | 16.1 | 19.4 | 27 | 40
//    2103, D = 1024, H = 768                                         24 | 24 | 23 | 25 | 38
//    1000, D = 512                                                        13.8 | 9.4 | 8.4 | 11.7
//     385, D = 512                                                        13.5 | 8.9 | 6.7 | 6.2
int chunk_tokens(int64_t B, int64_t D, int64_t blocks) {
    constexpr struct { int chunk, workgroups; } options[] = {{2048, 512}, {1024, 512}, {512, 256}, {256, 256}, {128, 256}};
    for (const auto &o : options)              // (32-bit offsets into a wavefront's quarter, two steps beyond its end included)
        if ((B + o.chunk - 1) / o.chunk * blocks >= o.workgroups && (o.chunk / 4 + 48) * D * 4 <= (int64_t(1) << 29)) return o.chunk;
    return 64;
}
constexpr int DEPTH = 4;          // token quads a step: their loads are in flight while the step before is multiplied

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// Tokens that a wavefront adds up from zero: a sum's rounding grows with its length.  Relative error against 64 bits and us, a chunk's sum
// in one | in runs of 64 tokens:
//   32768 tokens, D = 512, two repeats (chunks of 2048) 4.15e-7 | 1.77e-7, 214 | 224; 16384, D = 1024 (2048) 4.1e-7 | 1.7e-7, 103 | 104
//   16384, D = 512 (1024) 3.0e-7 | 1.7e-7, 54 | 54; 4096, D = 512 (512) 2.14e-7 | 1.62e-7, 17.8 | 18.2
// The first step of a run begun from zero in the instruction, four steps a turn: 42 spilled registers, 256 us.
constexpr int RUN = 64;
static_assert(RUN % (8 * DEPTH) == 0);

constexpr int ONCE = 2;           // a load's cache policy: nontemporal, read once

// What bounds it: memory (32768 tokens, D = 512, two repeats: 1.07 GB in 208 us, 5.1 TB/s; the products are 112 of it by themselves).  Loads
// that were branched around for a chunk's end waited for each other, four round trips a step: 277 us and 131 at 16384, D = 1024 instead
// of 199 and 91, 23 -> 16 at 4096, 10 -> 8.4 at 1000.  The nontemporal loads matter most behind the backward, whose stores they would push
// out of the memory-side cache line by line: both kernels in turn 473 -> 390 and 230 -> 186 us.
template <bool LN>
__global__ __launch_bounds__(256, 2) void bh4_wgrad_kernel(const float *stage_grads,
                                                           const float *x,
                                                           const float *stage_inputs,
                                                           float *g, int64_t B, int H, int D, int J,
                                                           const float *ln_w, const float *ln_b,
                                                           const float *row_stats, int chunk) {
    __shared__ float red[4][BS * BS / 4];          // a quarter of each wavefront's 64x64 tile
    const int n = blockIdx.y;
    const int s = blockIdx.z;                      // stage r * J + j
    const int r = s / J, j = s % J;
    const float *p = stage_grads + (size_t)s * B * D;
    const float *u = j == 0 ? x : stage_inputs + (size_t)(r * (J - 1) + j - 1) * B * D;
    const int Hu = j == 0 ? H : D;
    // a block of the first stage that lies wholly in the zero padding beyond column H has a zero input,
    // hence a zero gradient: g keeps what it holds (768 columns padded to 1024: 4 of 16 blocks)
    if (n * BS >= Hu) return;                      // uniform over the workgroup
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15;
    const int kq = lane >> 4;
    const int64_t tok_lo = int64_t(blockIdx.x) * chunk + wave * (chunk / 4);
    const int live = (int)max<int64_t>(0, min<int64_t>(chunk / 4, B - tok_lo));
    const bool u_live = n * BS + 4 * c < Hu;       // Hu % 4 == 0: the four columns are all in or all out
    const bool ln = LN && j == 0;                  // uniform over the workgroup

    // The wavefront's rows of the block as buffers that end with its last token: a load beyond it gives zeros, with no branch and no
    // wait in the way of the loads behind it.  (A lane whose columns of u are padding reads beyond the end throughout.)
    const int64_t first = min<int64_t>(tok_lo, B);
    const auto pr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p + first * D + n * BS), 0, max(0, (live * D - n * BS) * 4), 0x00020000);
    const auto ur = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(u + first * Hu + n * BS), 0, max(0, (live * Hu - n * BS) * 4), 0x00020000);
    const auto sr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(ln ? row_stats + 2 * first : p), 0, ln ? live * 8 : 0, 0x00020000);
    const int p_at = (kq * D + 4 * c) * 4, u_at = u_live ? (kq * Hu + 4 * c) * 4 : 0x40000000;

    f32x4 acc[4][4], total[4][4];                  // [o tile][i tile]
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = total[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto end_run = [&]() {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                total[a][b] += acc[a][b];
                acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
    };

    struct Step {
        u32x4 p[DEPTH], u[DEPTH];
        u32x2 stat[DEPTH];
    };
    auto fetch = [&](int t, Step &v, auto norm) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            v.p[d] = __builtin_amdgcn_raw_buffer_load_b128(pr, p_at + (t + 4 * d) * D * 4, 0, ONCE);
            v.u[d] = __builtin_amdgcn_raw_buffer_load_b128(ur, u_at + (t + 4 * d) * Hu * 4, 0, ONCE);
            if constexpr (decltype(norm)::value) v.stat[d] = __builtin_amdgcn_raw_buffer_load_b64(sr, (t + 4 * d + kq) * 8, 0, 0);
        }
        // (loads stay where they are issued: neither scheduler nor optimiser takes them past this point)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const Step &v) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            const f32x4 pa = __builtin_bit_cast(f32x4, v.p[d]), ub = __builtin_bit_cast(f32x4, v.u[d]);
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[a], ub[b], acc[a][b], 0, 0, 0);
        }
    };
    f32x4 lw = {0.f, 0.f, 0.f, 0.f}, lb = lw;      // this lane's four columns of LayerNorm's weight and bias
    if (ln && u_live) {
        lw = *reinterpret_cast<const f32x4 *>(ln_w + n * BS + 4 * c);
        lb = *reinterpret_cast<const f32x4 *>(ln_b + n * BS + 4 * c);
    }
    // LayerNorm of a step's rows, by the same operations as the forward's: (x - mean) * (1/sigma) * weight + bias
    auto normalise = [&](int t, Step &v) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            f32x4 h = (__builtin_bit_cast(f32x4, v.u[d]) - __uint_as_float(v.stat[d].x)) * __uint_as_float(v.stat[d].y) * lw + lb;
            asm("" : "+v"(h));                     // (selected from, not branched around)
            v.u[d] = t + 4 * d + kq < live && u_live ? __builtin_bit_cast(u32x4, h) : (u32x4){0u, 0u, 0u, 0u};
        }
    };
    // Two steps' registers in turn: a step's loads are issued in front of the products of the one before.
    auto run = [&](auto norm) {
        Step v0, v1;
        auto step = [&](int t, Step &now, Step &next) {
            fetch(t + 4 * DEPTH, next, norm);
            if constexpr (decltype(norm)::value) normalise(t, now);
            multiply(now);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        fetch(0, v0, norm);
        for (int t = 0; t < live; t += 8 * DEPTH) {
            step(t, v0, v1);
            if (t + 4 * DEPTH < live) step(t + 4 * DEPTH, v1, v0);
            if (t % RUN == RUN - 8 * DEPTH) end_run();
        }
        end_run();
    };
    if (ln) run(std::true_type{});
    else run(std::false_type{});

    // Tile (a, b), lane (c, kq), component r holds the sum for row o = 4*(4*kq + r) + a and
    // column i = 4*c + b.  Sum the four wavefronts through LDS, a quarter of the 64x64 block
    // (one value of a) at a time, then add to g.
    float *gb = g + ((size_t)s * (D / BS) + n) * BS * BS;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        __syncthreads();
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                red[wave][((4 * kq + r) * 16 + c) * 4 + b] = total[a][b][r];       // [o' = 4kq+r][c][b]
        __syncthreads();
        // 16 rows o' x 64 columns of this quarter: thread t adds element t, t+256, ...
        for (int e = threadIdx.x; e < BS * BS / 4; e += 256) {
            const float sum = (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
            const int op = e / 64, i = e % 64;                   // i = 4*c + b already in order
            unsafeAtomicAdd(gb + (4 * op + a) * BS + i, sum);
        }
    }
}

int wgrad_entry(const float *stage_grads, const float *x, const float *ln_weight, const float *ln_bias,
                const float *row_stats, const float *stage_inputs, float *g_folded, int64_t B, int64_t H, int64_t D,
                int64_t R, int64_t J, int64_t block_size, void *stream) {
    LFFN_REQUIRE(B >= 0 && D >= 1 && H >= 1 && H <= D && R >= 1 && J >= 1, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(block_size == BS && D % BS == 0 && D <= (1 << 20), LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(H % 4 == 0 && B <= (int64_t(1) << 31) - 1 && R * J <= 65535, LFFN_ERR_UNSUPPORTED);
    if (B == 0) return LFFN_OK;
    LFFN_REQUIRE(stage_grads && x && g_folded && (stage_inputs || J == 1), LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(stage_grads) && lffn_aligned16(x) && lffn_aligned16(stage_inputs) && lffn_aligned16(g_folded),
                 LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(!ln_weight || (ln_bias && row_stats && lffn_aligned16(ln_weight) && lffn_aligned16(ln_bias) &&
                                (uintptr_t)row_stats % 8 == 0), LFFN_ERR_BAD_ARG);
    const int chunk = chunk_tokens(B, D, D / BS * R * J);
    const int64_t chunks = (B + chunk - 1) / chunk;
    LFFN_REQUIRE(chunks <= 0x7fffffff && D / BS <= 65535, LFFN_ERR_UNSUPPORTED);
    hipLaunchKernelGGL(ln_weight ? bh4_wgrad_kernel<true> : bh4_wgrad_kernel<false>, dim3((unsigned)chunks, (unsigned)(D / BS), (unsigned)(R * J)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), stage_grads, x, stage_inputs, g_folded, B, (int)H, (int)D, (int)J,
                       ln_weight, ln_bias, row_stats, chunk);
    return lffn_launch_status();
}

}  // namespace

extern "C" int lffn_bh4_block_wgrad_f32(const float *stage_grads, const float *x, const float *stage_inputs,
                                        float *g_folded, int64_t B, int64_t H, int64_t D, int64_t R, int64_t J,
                                        int64_t block_size, void *stream) {
    return wgrad_entry(stage_grads, x, nullptr, nullptr, nullptr, stage_inputs, g_folded, B, H, D, R, J, block_size, stream);
}

extern "C" int lffn_ln_bh4_block_wgrad_f32(const float *stage_grads, const float *x, const float *ln_weight,
                                           const float *ln_bias, const float *row_stats, const float *stage_inputs,
                                           float *g_folded, int64_t B, int64_t H, int64_t D, int64_t R, int64_t J,
                                           int64_t block_size, void *stream) {
    LFFN_REQUIRE(ln_weight && ln_bias && row_stats, LFFN_ERR_BAD_ARG);
    return wgrad_entry(stage_grads, x, ln_weight, ln_bias, row_stats, stage_inputs, g_folded, B, H, D, R, J, block_size, stream);
}
