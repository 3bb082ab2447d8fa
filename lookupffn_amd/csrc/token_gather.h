// The gather-add of one token by one workgroup of eight or four wavefronts (PL/lookup.py:120-130, 108), for small batches:
//
//   out[row,:] = sum_t score_t * tables[t][code_t][:] (+ bias) (+ residual)
//
// A batch of a few tokens waits for memory round trips and nothing else, so as many row loads as possible are in flight: the
// wavefronts share the tables, eight tables at a time each with all column passes of those rows together, and their
// partial sums meet in LDS.  Up to 256 tokens, one to a compute unit, eight wavefronts (WAVES); beyond that four, two
// workgroups to a compute unit, where a second round of eight would wait for the first (384 tokens, 128 tables of 768
// fp32 columns: 33.9 us with eight, 27.1 with four; 256 tokens 21.1 with eight, 23.0 with four).
#pragma once

#include "lffn_common.h"

constexpr int64_t TOKEN_WIDE_MAX = 256;    // tokens up to which a token gets eight wavefronts
constexpr int TOKEN_MAX_T = 512;    // (code, score) pairs kept in LDS
constexpr int TOKEN_MAX_NC = 4;     // column passes of 256 in flight together; wider rows go in rounds of 1024

struct TokenGatherArgs {
    const void *tables;   // [T, S, Do], rows in the format of the kernel's FMT
    const float *obias;   // [Do] or null
    const float *gres;    // [B, Do] or null: added to the result
    float *gout;          // [B, Do]
    int T, S, Do;
    int part_cols = 0;    // columns of workgroup blockIdx.y of a token: a multiple of 256, or 0 for all of them
};

// Workgroups for a token, and the columns of each: as many as there are 256-column passes while the batch leaves compute units
// idle.  What comes before the gather is repeated by each; the sums of a column are the same.  One compute unit takes in a token's
// rows at some 60 bytes a clock, 393 KB of them at 128 tables of 768 fp32 columns: layer, us, 17 tokens 11.7 -> 9.3, 64 tokens 12.7 -> 11.5, 85
// tokens 13.2 -> 12.6; 512 tables of 1024 columns, 17 tokens 29.5 -> 14.9, 64 tokens 47 -> 28.
inline int token_parts(TokenGatherArgs &a, int64_t B) {
    const int passes = (a.Do + 255) / 256;
    const int64_t most = TOKEN_WIDE_MAX / (B > 0 ? B : 1);
    const int parts = (int)(most < passes ? most : passes);
    if (parts < 2) return 1;
    a.part_cols = (passes + parts - 1) / parts * 256;
    return (a.Do + a.part_cols - 1) / a.part_cols;
}

// four columns of a row as they are loaded, and their products with a score added up
template <int FMT>
using RowQuad = std::conditional_t<FMT == LFFN_ROWS_F32, float4, uint2>;

template <int FMT>
__device__ __forceinline__ void add_quad(float4 &acc, const RowQuad<FMT> &v, float s) {
    if constexpr (FMT == LFFN_ROWS_F32) {
        acc.x = fmaf(s, v.x, acc.x); acc.y = fmaf(s, v.y, acc.y); acc.z = fmaf(s, v.z, acc.z); acc.w = fmaf(s, v.w, acc.w);
    } else if constexpr (FMT == LFFN_ROWS_BF16) {
        acc.x = fmaf(s, bf16_lo(v.x), acc.x); acc.y = fmaf(s, bf16_hi(v.x), acc.y);
        acc.z = fmaf(s, bf16_lo(v.y), acc.z); acc.w = fmaf(s, bf16_hi(v.y), acc.w);
    } else {
        typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
        const half2_t a = __builtin_bit_cast(half2_t, v.x), b = __builtin_bit_cast(half2_t, v.y);
        acc.x = fmaf((float)a.x, s, acc.x); acc.y = fmaf((float)a.y, s, acc.y);
        acc.z = fmaf((float)b.x, s, acc.z); acc.w = fmaf((float)b.y, s, acc.w);
    }
}

// Columns [col0, col0 + 256 NC).  Loads are unconditional at clamped columns, so that none of them waits for another; what
// a clamped lane loaded is never stored.  Called by all wavefronts of the workgroup, with `pairs` visible to them.
template <int WAVES, int NC, int FMT, int ROWS>
__device__ __forceinline__ void token_gather_columns(const TokenGatherArgs &a, const uint2 *pairs,
                                                     float4 (*part)[TOKEN_MAX_NC][64], int64_t row, int col0, int wave,
                                                     int lane) {
    using Quad = RowQuad<FMT>;
    constexpr int ESZ = FMT == LFFN_ROWS_F32 ? 4 : 2;
    const char *tables = static_cast<const char *>(a.tables);
    int gc[NC];
    float4 acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int col = col0 + 256 * c + 4 * lane;
        gc[c] = col < a.Do ? col : 0;
        acc[c] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // bias and residual of the columns this wavefront will write, requested with the rows
    const int wcol = col0 + 256 * wave + 4 * lane;
    const bool writes = wave < NC && wcol < a.Do;
    float4 bb = make_float4(0.f, 0.f, 0.f, 0.f), rr = bb;
    if (writes && a.obias) bb = *reinterpret_cast<const float4 *>(a.obias + wcol);
    if (writes && a.gres) rr = *reinterpret_cast<const float4 *>(a.gres + row * a.Do + wcol);
    const int share = (a.T + WAVES - 1) / WAVES;
    const int t_lo = min(wave * share, a.T), t_hi = min(t_lo + share, a.T);
    for (int t0 = t_lo; t0 < t_hi; t0 += ROWS) {
        Quad rv[ROWS][NC];
        float sv[ROWS];
#pragma unroll
        for (int u = 0; u < ROWS; ++u) {
            const int tt = min(t0 + u, t_hi - 1);
            const uint2 pr = pairs[tt];
            sv[u] = t0 + u < t_hi ? __uint_as_float(pr.y) : 0.f;
            const char *rowp = tables + ((size_t)tt * a.S + pr.x) * a.Do * ESZ;
#pragma unroll
            for (int c = 0; c < NC; ++c) rv[u][c] = *reinterpret_cast<const Quad *>(rowp + gc[c] * ESZ);
        }
#pragma unroll
        for (int u = 0; u < ROWS; ++u)
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (t0 + u < t_hi) add_quad<FMT>(acc[c], rv[u][c], sv[u]);    // (uniform; a row past the end may hold anything)
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) part[wave][c][lane] = acc[c];
    __syncthreads();
    if (writes) {
        float4 o = part[0][wave][lane];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) {
            const float4 q = part[w][wave][lane];
            o.x += q.x; o.y += q.y; o.z += q.z; o.w += q.w;
        }
        if (a.obias) { o.x += bb.x; o.y += bb.y; o.z += bb.z; o.w += bb.w; }
        if (a.gres) { o.x += rr.x; o.y += rr.y; o.z += rr.z; o.w += rr.w; }
        *reinterpret_cast<float4 *>(a.gout + row * a.Do + wcol) = o;
    }
}

// PARTS: workgroup blockIdx.y has the token's columns from blockIdx.y * part_cols on, one or two passes at a time: their registers allow
// sixteen rows of a wavefront in flight.
template <int WAVES, int FMT, bool PARTS>
__device__ __forceinline__ void token_gather(const TokenGatherArgs &a, const uint2 *pairs, int64_t row, int wave, int lane) {
    __shared__ float4 part[WAVES][TOKEN_MAX_NC][64];
    if constexpr (PARTS) {
        const int first = blockIdx.y * a.part_cols, stop = min(a.Do, first + a.part_cols);
        for (int col0 = first; col0 < stop; col0 += 512) {
            if (col0 > first) __syncthreads();         // `part` has been read
            if (stop - col0 > 256) token_gather_columns<WAVES, 2, FMT, 16>(a, pairs, part, row, col0, wave, lane);
            else token_gather_columns<WAVES, 1, FMT, 16>(a, pairs, part, row, col0, wave, lane);
        }
        return;
    }
    for (int col0 = 0; col0 < a.Do; col0 += 256 * TOKEN_MAX_NC) {
        if (col0) __syncthreads();                     // `part` has been read
        switch (min(TOKEN_MAX_NC, (a.Do - col0 + 255) / 256)) {
            case 1: token_gather_columns<WAVES, 1, FMT, 8>(a, pairs, part, row, col0, wave, lane); break;
            case 2: token_gather_columns<WAVES, 2, FMT, 8>(a, pairs, part, row, col0, wave, lane); break;
            case 3: token_gather_columns<WAVES, 3, FMT, 8>(a, pairs, part, row, col0, wave, lane); break;
            default: token_gather_columns<WAVES, 4, FMT, 8>(a, pairs, part, row, col0, wave, lane); break;
        }
    }
}
