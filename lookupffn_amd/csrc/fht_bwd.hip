// Backward of the fused projection + hash for block size 1 and four stages, its transforms on the fp16 matrix cores, two terms a number
// (split_mfma.h).
//
//   z = decay * y + residual * pad(h) (+ bias),  y = FHT(d_3 * ... FHT(d_0 * pad(h))),  h = x or LayerNorm(x)   per repeat
//
// A transform of 1024 points is two products with the 32 x 32 matrix H of signs: the row as a matrix X[a][b] of 32 x 32, element
// 32 a + b, becomes H X H.  512 points are 16 x 32 and 256 points 8 x 32: a tile of 32 x 32 then holds two or four rows and the matrix
// on the left is block diagonal.  Signs (times 2^-5, so that nothing grows) are exact in half precision, so a number's hi and lo take
// one instruction each; what is rounded is lo, to 2^-23 of the number, twice a transform, and the sums: over rows of gradients and of inputs the
// result is closer to 64 bits than after ten rounded butterflies (tests/test_gpu_projection_bwd.py).
//
// Layouts.  In the first, lane l holds row a = l % 32 and columns b = mfma_row(i, l / 32), i = 0 .. 15: the operand on the left of a
// product over b, whose result has lane = b' and a in the registers, the operand on the right of a product over a.  That result is
// the second layout, lane = column b, registers = rows a = mfma_row(i, l / 32); the same two products, with the roles of the two
// sides changed, lead from it back to the first.  No value changes lanes otherwise, and a register's place within its instruction's sum is the
// order that the instruction hands its results out in, so the fragments of H are the same for both.  The inputs of the stages alternate between
// the layouts on the way up, and the gradients meet them in the same one on the way down.
//
// Bound by instruction issue: some 120 vector instructions a number at two wavefronts per SIMD, 60 of them in the 7 transforms (a
// transform's ten butterflies took 17 a number), the rest the diagonals, their gradients, the score's gradient and LayerNorm; a
// transform's 8 matrix instructions of 32 clocks lie under the other wavefront's.  16384 rows of 768, 1024 points: 131 -> 89 us.  One
// row's result is off by 2.0e-7 (butterflies 2.2e-7), a diagonal's gradient over 16384 rows by 2.6e-7 (2.8e-7).  A row with an infinity
// or NaN comes out as NaN, by itself.
#include "split_mfma.h"

#include "fht_bwd.h"

namespace {

constexpr int J = 4;
constexpr int LD = 36;                  // floats from one lane's part of a stage's diagonal to the next in LDS: b128 reads without conflicts

template <int LOGD>
struct Tile {
    static constexpr int D = 1 << LOGD, A = D / 32, ROWS = 32 / A;       // rows of a token's matrix, tokens in a tile
    static constexpr int PER = 16 / ROWS;                                 // registers of a token in the second layout
    static_assert(LOGD >= 8 && LOGD <= 10, "256, 512 and 1024 points");
};

__device__ __forceinline__ uint32_t max_u32(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t magnitude(float v) { return __float_as_uint(v) & 0x7FFFFFFFu; }

// The same operation over lanes l of a group of N = 8, 16 or 32 neighbours and over l and l + 32.
template <int N, typename F>
__device__ __forceinline__ float across(float v, F f) {
    v = f(v, lane_xor<1>(v));
    v = f(v, lane_xor<2>(v));
    v = f(v, lane_xor<4>(v));
    if constexpr (N >= 16) v = f(v, lane_xor<8>(v));
    if constexpr (N >= 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = f(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// A matrix of signs as the operand of a product over 32: row (or column) l % 32, times 2^-5; block diagonal with blocks of N.
template <int N>
__device__ __forceinline__ void signs(uint4 (&f)[2], int lane) {
    const int m = lane & 31, half = lane >> 5;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            uint32_t h[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int k = mfma_row(8 * s + j + u, half);
                h[u] = m / N == k / N ? (0x2800u | ((__popc(m & k) & 1) << 15)) : 0u;            // 2^-5
            }
            w[j / 2] = h[0] | (h[1] << 16);
        }
        f[s] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

struct Split {
    uint4 hi[2], lo[2];
};
__device__ __forceinline__ Split split16(const float (&v)[16]) {
    Split s;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        uint32_t h[4], l[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float a = v[8 * k + 2 * j], b = v[8 * k + 2 * j + 1];
            h[j] = split_hi(a, b, 1.f);
            l[j] = split_rest(a, b, h[j]);
        }
        s.hi[k] = make_uint4(h[0], h[1], h[2], h[3]);
        s.lo[k] = make_uint4(l[0], l[1], l[2], l[3]);
    }
    return s;
}

// The transform of a tile's rows, from the first layout to the second (FIRST) or back.  fa: signs over a, fb: over b.
// turned: 1 or -1, from tile to tile.  The matrix cores' sums are off to one side by a little, by an eighth of what a result is off
// in any direction; a sum over many rows would keep that, so every other row goes through with its sign turned.  (Gradient of the
// first diagonal, 16384 rows of 1024: off by 3.7e-7 without, 2.6e-7 with; butterflies 2.8e-7.)
template <int LOGD, bool FIRST>
__device__ __forceinline__ void transform(float (&v)[16], const uint4 (&fa)[2], const uint4 (&fb)[2], float turned, int lane) {
    using G = Tile<LOGD>;
    constexpr int N = G::ROWS, PER = G::PER;
    __builtin_amdgcn_sched_barrier(0);
    // The largest number of each row to 2^13 .. 2^14, and what takes the result back: 2^10 for the two products.  A row that is
    // not finite comes out as NaN, and for the others of its tile as zero.
    float in[FIRST ? 1 : N], out[FIRST ? N : 1];
    auto factors = [turned](uint32_t most, float &scale, float &back) {
        const PowerOfTwo p = scale_to_one(__uint_as_float(most));
        scale = p.scale * (turned * 8192.f);
        back = p.inverse * (turned * 0.125f);
        if (N > 1 && most >= 0x7F800000u) { scale = 0.f; back = __uint_as_float(0x7FC00000u); }
    };
    auto larger = [](float a, float b) { return __uint_as_float(max_u32(__float_as_uint(a), __float_as_uint(b))); };
    auto most_of = [&](int i0, int n) {
        if constexpr (N == 1) {
            float m = fabsf(v[i0]);
            for (int i = 1; i < n; ++i) m = fmaxf(m, fabsf(v[i0 + i]));
            return m;
        } else {                                              // (a NaN counts)
            uint32_t m = magnitude(v[i0]);
            for (int i = 1; i < n; ++i) m = max_u32(m, magnitude(v[i0 + i]));
            return __uint_as_float(m);
        }
    };
    bool all_finite = true;
    if constexpr (FIRST) {
        const float m = across<G::A>(most_of(0, 16), larger);
        float back;
        factors(__float_as_uint(m), in[0], back);
        if constexpr (N > 1) all_finite = __all(is_finite(m));
#pragma unroll
        for (int g = 0; g < N; ++g)
            out[g] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(back), g * G::A));
    } else {
        float back[N];
#pragma unroll
        for (int g = 0; g < N; ++g) {
            const float m = across<32>(most_of(g * PER, PER), larger);
            factors(__builtin_amdgcn_readfirstlane(__float_as_uint(m)), in[g], back[g]);
            if constexpr (N > 1) all_finite = all_finite && is_finite(m);
        }
        out[0] = back[0];
#pragma unroll
        for (int g = 1; g < N; ++g) out[0] = (lane & 31) / G::A == g ? back[g] : out[0];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] *= in[FIRST ? 0 : i / PER];
    if constexpr (N > 1) {
        if (!all_finite) {
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = in[FIRST ? 0 : i / PER] == 0.f ? 0.f : v[i];
        }
    }
    const uint4 (&f1)[2] = FIRST ? fb : fa, (&f2)[2] = FIRST ? fa : fb;
    Split s = split16(v);
    __builtin_amdgcn_sched_barrier(0);
    f32x16_t p{};
    p = mfma_f16(s.lo[0], f1[0], p);
    p = mfma_f16(s.lo[1], f1[1], p);
    p = mfma_f16(s.hi[0], f1[0], p);
    p = mfma_f16(s.hi[1], f1[1], p);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = p[i];
    s = split16(v);
    __builtin_amdgcn_sched_barrier(0);
    f32x16_t y{};
    y = mfma_f16(f2[0], s.lo[0], y);
    y = mfma_f16(f2[1], s.lo[1], y);
    y = mfma_f16(f2[0], s.hi[0], y);
    y = mfma_f16(f2[1], s.hi[1], y);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = y[i] * out[FIRST ? i / PER : 0];
}

template <int LOGD>
__global__ __launch_bounds__(256, 2) void project_hash_bwd_mfma_kernel(ProjectBwdArgs a) {
    using G = Tile<LOGD>;
    constexpr int D = G::D, A = G::A, N = G::ROWS;
    // A stage's diagonal as its layout reads it: [row a][column b] for stages 0 and 2, [b][a] for 1 and 3.
    __shared__ float diag[J][32 * LD];
    __shared__ float ln[2][32 * LD];             // LayerNorm's weight and bias, [row a][column b], 0 beyond H
    // Each lane's own, out of the way of its registers: the inputs of the first two stages and the sums of the gradient of z; at the end
    // the way from the wavefronts to the workgroup's sums.
    __shared__ float4 kept[2][4][4][64], sum_b[4][4][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5, m = lane & 31;
    const int r = blockIdx.y;
#pragma unroll
    for (int i = 0; i < J * D / 1024; ++i) {
        const int k = 4 * tid + 1024 * i, s = k / D, e = k % D, row = e / 32, col = e % 32;
        const float4 w = *reinterpret_cast<const float4 *>(a.diag + int64_t(r) * J * D + k);
        const int at = s & 1 ? col * LD + row : row * LD + col, step = s & 1 ? LD : 1;
        diag[s][at] = w.x; diag[s][at + step] = w.y; diag[s][at + 2 * step] = w.z; diag[s][at + 3 * step] = w.w;
    }
    for (int k = tid; k < D; k += 256) {
        const bool there = a.ln_w && k < a.H;
        ln[0][k / 32 * LD + k % 32] = there ? a.ln_w[k] : 0.f;
        ln[1][k / 32 * LD + k % 32] = there ? a.ln_b[k] : 0.f;
    }
    uint4 fa[2], fb[2];
    signs<A>(fa, lane);
    signs<32>(fb, lane);
    __syncthreads();

    const int own = m % A;                       // the first layout's row of the token's matrix
    // v *= (the stage's diagonal)
    auto scale_by_diag = [&](float (&v)[16], int s) {
        asm volatile("" ::: "memory");           // or the compiler keeps all four stages' in registers
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int at = 8 * q + 4 * half;
            const float4 w = *reinterpret_cast<const float4 *>(s & 1 ? &diag[s][m * LD + at % A] : &diag[s][own * LD + at]);
            v[4 * q] *= w.x; v[4 * q + 1] *= w.y; v[4 * q + 2] *= w.z; v[4 * q + 3] *= w.w;
        }
    };

    const int ncols = a.T * 8;
    const int64_t ntiles = (a.B + N - 1) / N;
    const int col0 = 32 * own + 4 * half;        // the first layout's columns: col0 + 8 q, and the three behind it
    auto load4 = [](float *v, const float *p, bool there) {            // p: where something can be read in any case
        const float4 w = *reinterpret_cast<const float4 *>(p);
        v[0] = there ? w.x : 0.f; v[1] = there ? w.y : 0.f; v[2] = there ? w.z : 0.f; v[3] = there ? w.w : 0.f;
    };
    float acc_d[J][16];
#pragma unroll
    for (int s = 0; s < J; ++s)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc_d[s][i] = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) sum_b[wave][q][lane] = make_float4(0.f, 0.f, 0.f, 0.f);

    for (int64_t tile = int64_t(blockIdx.x) * 4 + wave; tile < ntiles; tile += int64_t(gridDim.x) * 4) {
        // (rows from B on take the last row's input and a gradient of zero, and their result is not stored)
        const int64_t left = a.B - tile * N;
        const float turned = tile & 1 ? -1.f : 1.f;
        const bool live = m / A < left;
        const int ahead = live ? m / A : (int)left - 1;        // rows behind the tile's first
        float t[16], z[16], g[4];
        const float *xp = a.x + tile * N * a.H, *zp = a.z + tile * N * ncols, *gp = a.g_score + tile * N * a.T;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bool there = col0 + 8 * q < a.H;
            load4(t + 4 * q, xp + (ahead * a.H + (there ? col0 + 8 * q : 0)), there);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int col = r * D + col0 + 8 * q;
            const bool there = live && col < ncols;
            load4(z + 4 * q, zp + (ahead * ncols + (there ? col : 0)), there);
            g[q] = gp[ahead * a.T + (there ? col >> 3 : 0)];
            g[q] = there ? g[q] : 0.f;
        }
        float u[2][16];                          // the inputs of the last two stages
        if (a.ln_w) {                                         // uniform; as the forward: biased variance, two passes
            auto sum = [](float x, float y) { return x + y; };
            float s1 = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) s1 += t[i];
            const float mean = across<A>(s1, sum) / float(a.H);
            float s2 = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                t[i] = col0 + 8 * (i / 4) < a.H ? t[i] - mean : 0.f;        // H % 4 == 0: all four columns or none
                s2 += t[i] * t[i];
            }
            const float rstd = 1.0f / sqrtf(across<A>(s2, sum) / float(a.H) + a.ln_eps);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int at = own * LD + 8 * q + 4 * half;
                const float4 lw = *reinterpret_cast<const float4 *>(&ln[0][at]), lb = *reinterpret_cast<const float4 *>(&ln[1][at]);
                t[4 * q] = t[4 * q] * rstd * lw.x + lb.x;
                t[4 * q + 1] = t[4 * q + 1] * rstd * lw.y + lb.y;
                t[4 * q + 2] = t[4 * q + 2] * rstd * lw.z + lb.z;
                t[4 * q + 3] = t[4 * q + 3] * rstd * lw.w + lb.w;
            }
        }
        auto keep = [&](int s) {
            if (s < 2) {
#pragma unroll
                for (int q = 0; q < 4; ++q) kept[s][wave][q][lane] = make_float4(t[4 * q], t[4 * q + 1], t[4 * q + 2], t[4 * q + 3]);
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) u[s - 2][i] = t[i];
            }
        };
        keep(0);
        scale_by_diag(t, 0);
        transform<LOGD, true>(t, fa, fb, turned, lane);
        keep(1);
        scale_by_diag(t, 1);
        transform<LOGD, false>(t, fa, fb, turned, lane);
        keep(2);
        scale_by_diag(t, 2);
        transform<LOGD, true>(t, fa, fb, turned, lane);
        keep(3);

        // The gradient of z.  A group of eight columns sits in four registers of the two halves of the wavefront.
        float gz[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float zq[4] = {z[4 * q], z[4 * q + 1], z[4 * q + 2], z[4 * q + 3]};
            const ScorePart own = score_part(zq);
            const auto ss = __builtin_amdgcn_permlane32_swap(__float_as_uint(own.sum), __float_as_uint(own.sum), false, false);
            const auto pp = __builtin_amdgcn_permlane32_swap(__float_as_uint(own.product), __float_as_uint(own.product), false, false);
            const float twice = 2.0f * (__uint_as_float(ss[0]) + __uint_as_float(ss[1]));
            const float g_over_p = g[q] / (__uint_as_float(pp[0]) * __uint_as_float(pp[1]));
#pragma unroll
            for (int c = 0; c < 4; ++c) gz[4 * q + c] = score_derivative(zq[c], own.away[c], twice, g_over_p);
            float4 sb = sum_b[wave][q][lane];
            sb.x += gz[4 * q]; sb.y += gz[4 * q + 1]; sb.z += gz[4 * q + 2]; sb.w += gz[4 * q + 3];
            sum_b[wave][q][lane] = sb;
        }

        // back through the stages
#pragma unroll
        for (int i = 0; i < 16; ++i) t[i] = a.decay * gz[i];
        auto meet = [&](int s) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float4 v;
                if (s < 2) v = kept[s][wave][q][lane];
                else v = make_float4(u[s - 2][4 * q], u[s - 2][4 * q + 1], u[s - 2][4 * q + 2], u[s - 2][4 * q + 3]);
                acc_d[s][4 * q] += t[4 * q] * v.x; acc_d[s][4 * q + 1] += t[4 * q + 1] * v.y;
                acc_d[s][4 * q + 2] += t[4 * q + 2] * v.z; acc_d[s][4 * q + 3] += t[4 * q + 3] * v.w;
            }
            scale_by_diag(t, s);
        };
        transform<LOGD, true>(t, fa, fb, turned, lane);
        meet(3);
        transform<LOGD, false>(t, fa, fb, turned, lane);
        meet(2);
        transform<LOGD, true>(t, fa, fb, turned, lane);
        meet(1);
        transform<LOGD, false>(t, fa, fb, turned, lane);
        meet(0);
        // (formed here and not behind the stores' conditions, where the compiler would move every register out of the way)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            t[i] += a.residual * gz[i];
            asm volatile("" : "+v"(t[i]));
        }
        float *gx = a.g_x + (int64_t(r) * a.B + tile * N) * a.H;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (live && col0 + 8 * q < a.H)
                *reinterpret_cast<float4 *>(gx + (ahead * a.H + col0 + 8 * q)) =
                    make_float4(t[4 * q], t[4 * q + 1], t[4 * q + 2], t[4 * q + 3]);
    }

    // the workgroup's partial sums: over its four wavefronts and a tile's tokens, in that order
    float *red = reinterpret_cast<float *>(kept);
    auto flush = [&](const float (&acc)[16], bool second, float *dst) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int k = mfma_row(i, half);
            red[wave * 1024 + (second ? 32 * k + m : 32 * m + k)] = acc[i];
        }
        __syncthreads();
        for (int e = tid; e < D; e += 256) {
            float sum = 0.f;
#pragma unroll
            for (int k = 0; k < 4 * N; ++k) sum += red[k * D + e];
            dst[e] = sum;
        }
    };
#pragma unroll
    for (int s = 0; s < J; ++s) flush(acc_d[s], s & 1, a.part_d + ((int64_t(blockIdx.x) * a.R + r) * J + s) * D);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 v = sum_b[wave][q][lane];
        acc_d[0][4 * q] = v.x; acc_d[0][4 * q + 1] = v.y; acc_d[0][4 * q + 2] = v.z; acc_d[0][4 * q + 3] = v.w;
    }
    flush(acc_d[0], false, a.part_b + (int64_t(blockIdx.x) * a.R + r) * D);
}

}  // namespace

int lffn_internal_project_hash_bwd_mfma(const ProjectBwdArgs &a, int logd, int num_partials, hipStream_t st) {
    const dim3 grid((unsigned)num_partials, (unsigned)a.R);
    switch (logd) {
        case 8: hipLaunchKernelGGL((project_hash_bwd_mfma_kernel<8>), grid, dim3(256), 0, st, a); break;
        case 9: hipLaunchKernelGGL((project_hash_bwd_mfma_kernel<9>), grid, dim3(256), 0, st, a); break;
        case 10: hipLaunchKernelGGL((project_hash_bwd_mfma_kernel<10>), grid, dim3(256), 0, st, a); break;
        default: return LFFN_ERR_UNSUPPORTED;
    }
    return lffn_launch_status();
}
