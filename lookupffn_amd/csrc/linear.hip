// out[m, n] = sum_k x[m, k] w[n, k] + bias[n] (+ residual[m, n]) in fp32 on the fp16 matrix cores (split_mfma.h), up to three
// matrices w (query, key and value of an attention) in one launch.
//
// A workgroup owns a tile of BM x BN results and walks k in steps of 32.  A step's numbers are fetched as they lie (fp32, 16 bytes a
// lane, two steps ahead), split on the way into LDS (hi and lo planes of 64-byte rows, the four 16-byte pieces of a row turned by
// row / 4, so that sixteen rows' reads of one piece fall on different banks) and read back as operands; three buffers, so that a
// step's products need one barrier and its first operands are there when it starts.  The products, the splitting and the LDS
// traffic are spread through each other by scheduling groups: a matrix instruction covers five vector ones.
//
// Every row of x and w is scaled by a power of two of its own and the results are scaled back: any size of numbers goes.  The scale comes
// from 32 numbers spread over the row.  A tile with a row that is 128 times larger elsewhere comes out infinite and is done once more with
// the scales of the rows' largest numbers; what is not finite then, a third time in fp32, for which infinities and NaN are numbers like
// others.  16384 x 768 x 768 with a residual, us: 84, where every row outgrows its sample 208, with an infinity in every tile 470.  (The
// largest numbers looked for beforehand, one more pass over the rows for every tile: 97; 16 rows 13 -> 16, with the sample 13.)
//
// What bounds it: power.  16384 x 768 x 768, three matrices: 222 us, 261 TFLOP/s of fp32 product (783 of fp16) at 1.67 GHz; with
// zeros for numbers the same kernel runs at 2.37 GHz, 194 us.  Of its clocks 62 % are matrix instructions; LDS (writes 13 clocks per
// kilobyte, reads 4 to 7) and the splitting take as long as those beside them.  The library's fp32 product takes 426 us
// (136 TFLOP/s, 0.87 of the fp32 matrix cores' peak).  Error against 64 bits 2.0e-7 of the result (library 5.0e-7; 16 rows, where
// it splits k, 2.5e-7); as six products of three bfloat16 terms 1.6e-7, but 313 us.
//
// lffn_linear_norm_f32 takes the splitting out of the loop: a row of x is split for nine tiles, a row of w for 128, each time anew.
// LayerNorm's kernel writes its rows split instead (split_rows_kernel), with the rows of every w beside them, and a tile's numbers go
// into LDS as they come.  LayerNorm and the three matrices, us before -> now: 16384 x 768 254 -> 230, 32768 x 768 486 -> 434, 4096 x
// 1024 124 -> 107, 16384 x 512 131 -> 118, 2103 x 768 43 -> 42, 1024 x 768 31 -> 31, 512 x 768 24 -> 31 (its form is the one with
// tiles of 64 x 64 and no extra traffic for w): from 2048 rows on it is never slower.  Splitting w alone gives nothing, the launch
// costs what it saves (16384 x 768: 233 -> 228, one matrix 82 -> 84).
#include "split_mfma.h"


namespace {

constexpr int BK = 32;                                  // k of a step

struct LinearArgs {
    const float *x;              // [M, K]
    const float *residual;       // [M, N] or null
    const float *w[3], *b[3];    // [N, K], [N] or null, of every set
    const uint4 *split;          // rows of x and of every w by split_rows_kernel, [M + sets N][K / 8][hi, lo]
    const int *split_exponent;   // [M + sets N]
    float *out[3];               // [M, N]
    int64_t M;
    int N, K, sets;
};

struct SplitArgs {
    const float *x, *weight, *bias;      // [M, K], [K] or null: LayerNorm of the rows of x
    const float *w[3];                   // [N, K]
    uint4 *split;
    int *exponent;
    int64_t M, rows;                     // M + sets N
    int N, K;
    float eps;
};

constexpr int TOP = 13;             // the row's largest number: lo, times 2048, stays below 2^13
constexpr int TOP_OF_SAMPLE = 8;    // a sample's, which the row may outgrow 128 times

__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, lane_xor<1>(v));
    v = fmaxf(v, lane_xor<2>(v));
    v = fmaxf(v, lane_xor<4>(v));
    v = fmaxf(v, lane_xor<8>(v));
    v = fmaxf(v, lane_xor<16>(v));
    return fmaxf(v, lane_xor<32>(v));
}

// Rows of LayerNorm(x) and of every w as the products want them, eight hi and eight lo in the place of eight numbers, scaled by a
// power of two by their largest finite number.  A wavefront a row, NV x 16 bytes a lane; two lanes with the halves of eight numbers
// exchange them, so that one stores the hi and the other the lo and a row is written as it is read.  One launch in the place of
// LayerNorm's, 50 MB in and 50 out as that one (16384 x 768: 22 us with three matrices of 768 rows, PyTorch's LayerNorm 29).
template <int NV>
__global__ __launch_bounds__(256) void split_rows_kernel(SplitArgs a) {
    const int lane = threadIdx.x & 63, quads = a.K >> 2;
    const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (row >= a.rows) return;
    const bool norm = row < a.M;
    const int64_t wrow = row - a.M;
    const float4 *const from = reinterpret_cast<const float4 *>(norm ? a.x + row * a.K : a.w[wrow / a.N] + wrow % a.N * a.K);
    float v[NV][4];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int q = i * 64 + lane;
        const float4 u = q < quads ? from[q] : make_float4(0.f, 0.f, 0.f, 0.f);
        v[i][0] = u.x, v[i][1] = u.y, v[i][2] = u.z, v[i][3] = u.w;
    }
    if (norm) {
        float sum = 0.f, squares = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i) sum += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
        const float mean = lane_group_sum<64>(sum) / a.K;
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[i][e] -= mean;
                if (i * 64 + lane < quads) squares = fmaf(v[i][e], v[i][e], squares);
            }
        const float factor = 1.f / sqrtf(lane_group_sum<64>(squares) / a.K + a.eps);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int q = i * 64 + lane;
            const bool live = q < quads;
            const float4 m = live && a.weight ? reinterpret_cast<const float4 *>(a.weight)[q] : make_float4(1.f, 1.f, 1.f, 1.f);
            const float4 b = live && a.bias ? reinterpret_cast<const float4 *>(a.bias)[q] : make_float4(0.f, 0.f, 0.f, 0.f);
            v[i][0] = fmaf(v[i][0] * factor, m.x, b.x);
            v[i][1] = fmaf(v[i][1] * factor, m.y, b.y);
            v[i][2] = fmaf(v[i][2] * factor, m.z, b.z);
            v[i][3] = fmaf(v[i][3] * factor, m.w, b.w);
        }
    }
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (i * 64 + lane < quads && is_finite(v[i][e])) most = fmaxf(most, fabsf(v[i][e]));
    int exponent;
    const float scale = scale_to(wave_max(most), TOP, exponent);
    uint4 *const to = a.split + row * quads;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int q = i * 64 + lane;                    // (quads is even: both lanes of a pair are in or neither)
        const uint32_t h0 = split_hi(v[i][0], v[i][1], scale), h1 = split_hi(v[i][2], v[i][3], scale);
        const uint32_t l0 = split_lo(v[i][0], v[i][1], scale, h0), l1 = split_lo(v[i][2], v[i][3], scale, h1);
        const bool odd = lane & 1;
        const uint32_t o0 = __float_as_uint(lane_xor<1>(__uint_as_float(odd ? h0 : l0)));
        const uint32_t o1 = __float_as_uint(lane_xor<1>(__uint_as_float(odd ? h1 : l1)));
        if (q < quads) to[q] = odd ? make_uint4(o0, o1, l0, l1) : make_uint4(h0, h1, o0, o1);
    }
    if (lane == 0) a.exponent[row] = exponent;
}

// Four numbers of eight that are split, hi at p and lo 16 bytes on, as they were but for the last bits.
__device__ __forceinline__ float4 joined(const float *p, int exponent) {
    const uint2 h = *reinterpret_cast<const uint2 *>(p), l = *reinterpret_cast<const uint2 *>(p + 4);
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float hi = __builtin_bit_cast(f16x2_t, e < 2 ? h.x : h.y)[e & 1], lo = __builtin_bit_cast(f16x2_t, e < 2 ? l.x : l.y)[e & 1];
        y[e] = __builtin_amdgcn_ldexpf(is_finite(hi) ? fmaf(lo, 1 / SPLIT_LO, hi) : hi, exponent);
    }
    return make_float4(y[0], y[1], y[2], y[3]);
}

// WAVES_M x WAVES_N wavefronts of WM x WN tiles of 32 x 32 each.  SPLIT: x and w come split.
template <int WAVES_M, int WAVES_N, int WM, int WN, bool SPLIT>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, 2) void linear_kernel(LinearArgs a) {
    constexpr int BM = 32 * WM * WAVES_M, BN = 32 * WN * WAVES_N, THREADS = 64 * WAVES_M * WAVES_N;
    constexpr int BUF = 2 * (BM + BN) * 4;               // 16-byte pieces of a step's buffer
    constexpr int RSTEP = THREADS / 4;
    constexpr int NP = (BM + BN) / RSTEP;                // pieces of eight numbers a thread brings a step,
    constexpr bool REST = (BM + BN) % RSTEP != 0;        // and half a piece, of the last RSTEP / 2 rows
    constexpr int NC = NP + REST;
    constexpr int NR = 2 * (WM + WN);                    // fragments of half a step
    static_assert(BM % RSTEP == 0 && (BN % RSTEP == 0 || BN % RSTEP == RSTEP / 2) && NC <= 3);
    extern __shared__ __attribute__((aligned(16))) uint4 lds[];
    int *const exponent = reinterpret_cast<int *>(lds + 3 * BUF);         // [BM + BN] of the rows' scales
    int &outgrown = exponent[BM + BN];
    const int N = a.N, K = a.K;
    const int64_t M = a.M;
    // XCD b % 8 takes a contiguous range of the tiles, a tile of x against all matrices before the next
    const int per_set = (N + BN - 1) / BN, ntn = per_set * a.sets;
    const int nblk = gridDim.x, xcd = blockIdx.x & 7, q = nblk >> 3, rem = nblk & 7;
    const int tile = xcd * q + min(xcd, rem) + (blockIdx.x >> 3);
    const int64_t m0 = int64_t(tile / ntn) * BM;
    const int nt = tile % ntn, set = nt / per_set, n0 = (nt % per_set) * BN;
    const float *const w = a.w[set];
    const float *const xa = a.x + m0 * K, *const wb = w + int64_t(n0) * K;
    // (split or not, eight numbers are 32 bytes)
    const float *const xf = SPLIT ? reinterpret_cast<const float *>(a.split) + m0 * K : xa;
    const float *const wf = SPLIT ? reinterpret_cast<const float *>(a.split) + (M + int64_t(set) * N + n0) * K : wb;
    const float *const bias = a.b[set];
    float *const out = a.out[set] + m0 * N + n0;
    const float *const residual = a.residual ? a.residual + m0 * N + n0 : nullptr;
    const int rows = (int)min(int64_t(BM), M - m0), cols = min(BN, N - n0);
    bool bad;
    // The rows' scales from a sample of them, 32 numbers from all parts of a row; where one has outgrown its sample (the results are
    // infinite), the tile once more with the scales of the rows' largest numbers.
#pragma unroll 1
    for (int whole = 0;; ++whole) {
        // (an opaque zero: what follows from the lane is formed anew in each pass, and none of it kept through the results)
        int zero = 0;
        asm volatile("" : "+v"(zero));
        const int tid = threadIdx.x + zero, lane = tid & 63, wave = tid >> 6;
        const int wm = wave % WAVES_M, wn = wave / WAVES_M;
        // a thread's pieces of a step: eight numbers each of rows tid / 4 + RSTEP i, those of x before those of w
        const int chunk = tid & 3, row0 = tid >> 2;
        uint32_t src[NC];
        int dst[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int row = i < NP ? row0 + RSTEP * i : RSTEP * NP + (tid >> 3);
            if (i == NP) {
                src[i] = uint32_t(min(row - BM, N - 1 - n0)) * K + (tid & 7) * 4;
                dst[i] = 2 * BM * 4 + (row - BM) * 4 + (((tid & 7) >> 1) ^ ((row >> 2) & 3));
            } else if (RSTEP * i < BM) {
                src[i] = uint32_t(min(int64_t(row), M - 1 - m0)) * K + chunk * 8;
                dst[i] = row * 4 + (chunk ^ ((row >> 2) & 3));
            } else {
                src[i] = uint32_t(min(row - BM, N - 1 - n0)) * K + chunk * 8;
                dst[i] = 2 * BM * 4 + (row - BM) * 4 + (chunk ^ ((row >> 2) & 3));
            }
        }
        const int r = lane & 31, half = lane >> 5;
        const int arow = wm * 32 * WM + r, brow = wn * 32 * WN + r;
        int aoff[2], boff[2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            aoff[kk] = arow * 4 + ((kk * 2 + half) ^ ((arow >> 2) & 3));
            boff[kk] = 2 * BM * 4 + brow * 4 + ((kk * 2 + half) ^ ((brow >> 2) & 3));
        }
        float v[NC][8], scale[NC];
        auto fetch = [&](int i, int k0) {
            const int k = min(k0, K - BK);                  // (beyond the end: the last step again, never used)
            const float *const p = (RSTEP * i < BM ? xf : wf) + k;
            *reinterpret_cast<float4 *>(&v[i][0]) = *reinterpret_cast<const float4 *>(p + src[i]);
            if (i < NP) *reinterpret_cast<float4 *>(&v[i][4]) = *reinterpret_cast<const float4 *>(p + src[i] + 4);
        };
        uint32_t h[4];
        auto place = [&](uint4 *buf, int i, int p) {
            const int plane = (RSTEP * i < BM ? BM : BN) * 4;
            uint32_t o[4];
            if (SPLIT) {                                    // it comes as it goes; of the half piece a thread has one term
                const uint4 u = *reinterpret_cast<const uint4 *>(&v[i][i < NP ? 4 * p : 0]);
                if (i < NP) buf[dst[i] + p * plane] = u;
                else if (p == 0) buf[dst[i] + (tid & 1) * plane] = u;
                return;
            }
#pragma unroll
            for (int e = 0; e < (i < NP ? 4 : 2); ++e) {
                if (p == 0) o[e] = h[e] = split_hi(v[i][2 * e], v[i][2 * e + 1], scale[i]);
                else o[e] = split_lo(v[i][2 * e], v[i][2 * e + 1], scale[i], h[e]);
            }
            if (i < NP) buf[dst[i] + p * plane] = make_uint4(o[0], o[1], o[2], o[3]);
            else reinterpret_cast<uint2 *>(buf + dst[i] + p * plane)[tid & 1] = make_uint2(o[0], o[1]);
        };
        uint4 fa[2][WM][2], fb[2][WN][2];                   // [half of the step][tile][hi, lo]
        auto read = [&](const uint4 *buf, int kk, int n) {
            if (n < 2 * WM) {
                fa[kk][n % WM][n / WM] = buf[aoff[kk] + n / WM * BM * 4 + n % WM * 32 * 4];
            } else {
                n -= 2 * WM;
                fb[kk][n % WN][n / WN] = buf[boff[kk] + n / WN * BN * 4 + n % WN * 32 * 4];
            }
        };
        // steps 0 and 1 into their buffers, 2 on its way
        float most[NC] = {};
        auto take = [&](int i, const float *p) {            // (beyond the end: the row's last numbers again)
            const float4 f = *reinterpret_cast<const float4 *>(p);
            most[i] = fmaxf(fmaxf(most[i], fmaxf(fabsf(f.x), fabsf(f.y))), fmaxf(fabsf(f.z), fabsf(f.w)));
        };
        if (!SPLIT) {
            const int parts = whole ? K / BK : 1;
#pragma unroll 4
            for (int part = 0; part < parts; ++part)
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    // (a thread's share of the row's numbers: K / 4, of the half piece K / 8)
                    const float *const row = (RSTEP * i < BM ? xf : wf) + src[i];
                    if (i < NP) {
                        const float *const p = row + chunk * (K / 4 - 8) + part * 8;
                        take(i, p);
                        take(i, p + 4);
                    } else {
                        take(i, row + (tid & 7) * (K / 8 - 4) + part * 4);
                    }
                }
        }
#pragma unroll
        for (int i = 0; i < NC; ++i) fetch(i, 0);
        if (!SPLIT && tid == 0) outgrown = 0;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            if constexpr (SPLIT) {
                const int row = i < NP ? row0 + RSTEP * i : RSTEP * NP + (tid >> 3);
                if ((i < NP ? chunk : tid & 7) == 0)
                    exponent[row] = a.split_exponent[RSTEP * i < BM ? min(m0 + row, M - 1) : M + int64_t(set) * N + min(n0 + row - BM, N - 1)];
                place(lds, i, 0);
                place(lds, i, 1);
                fetch(i, BK);
                continue;
            }
            float m = fmaxf(most[i], lane_xor<1>(most[i]));
            m = fmaxf(m, lane_xor<2>(m));
            if (i == NP) m = fmaxf(m, lane_xor<4>(m));
            int back;
            scale[i] = scale_to(m, whole ? TOP : TOP_OF_SAMPLE, back);
            if (i < NP) {
                if (chunk == 0) exponent[row0 + RSTEP * i] = back;
            } else if ((tid & 7) == 0) {
                exponent[RSTEP * NP + (tid >> 3)] = back;
            }
            place(lds, i, 0);
            place(lds, i, 1);
            fetch(i, BK);
        }
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            place(lds + BUF, i, 0);
            place(lds + BUF, i, 1);
            fetch(i, 2 * BK);
        }
        lds_barrier();
        f32x16_t acc[WM][WN] = {}, low[WM][WN] = {};
        uint4 *cur = lds, *nxt = lds + BUF, *put = lds + 2 * BUF;
#pragma unroll
        for (int n = 0; n < NR; ++n) read(cur, 0, n);
#pragma unroll 1
        for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int t = 0; t < 3; ++t) {
                    const int g = kk * 3 + t;
#pragma unroll
                    for (int i = 0; i < WM; ++i)
#pragma unroll
                        for (int j = 0; j < WN; ++j) {
                            if (t == 0) low[i][j] = mfma_f16(fa[kk][i][1], fb[kk][j][0], low[i][j]);
                            if (t == 1) low[i][j] = mfma_f16(fa[kk][i][0], fb[kk][j][1], low[i][j]);
                            if (t == 2) acc[i][j] = mfma_f16(fa[kk][i][0], fb[kk][j][0], acc[i][j]);
                        }
#pragma unroll
                    for (int n = t * NR / 3; n < (t + 1) * NR / 3; ++n) read(kk ? nxt : cur, kk ^ 1, n);
                    if (g < 2 * NC) {
                        place(put, g / 2, g % 2);
                        if (g % 2) fetch(g / 2, k0 + 3 * BK);
                    }
#pragma unroll
                    for (int n = 0; n < WM * WN; ++n) {
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
                        if (n == 0) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                        else __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x20, 2, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            lds_barrier();
            uint4 *const o = cur;
            cur = nxt;
            nxt = put;
            put = o;
        }

        // Results: the lane has 16 rows of one column of every 32 x 32 tile.
        bad = false;
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            const int n = wn * 32 * WN + j * 32 + r;
            const float bv = bias ? bias[n0 + min(n, cols - 1)] : 0.f;
            const int back = exponent[BM + n];
#pragma unroll
            for (int i = 0; i < WM; ++i) {
                const int ml = wm * 32 * WM + i * 32;
                float res[16];
                if (residual) {
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        res[e] = residual[uint32_t(min(ml + mfma_row(e, half), rows - 1)) * N + min(n, cols - 1)];
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int m = ml + mfma_row(e, half);
                    float y = __builtin_amdgcn_ldexpf(fmaf(low[i][j][e], 1 / SPLIT_LO, acc[i][j][e]), exponent[m] + back);
                    bad |= !is_finite(y);
                    y += bv;
                    if (residual) y += res[e];
                    if (m < rows && n < cols) out[uint32_t(m) * N + n] = y;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (SPLIT || whole) break;
        if (__any(bad) && lane == 0) outgrown = 1;
        __syncthreads();
        const bool again = outgrown != 0;
        __syncthreads();                                    // (read by all before it is cleared)
        if (!again) return;
    }
    if (__any(bad)) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, half = lane >> 5;
        const int wm = wave % WAVES_M, wn = wave / WAVES_M;
        // the split does not carry infinities: the wavefront's results once more, on the fp32 matrix cores
#pragma unroll 1
        for (int t = 0; t < WM * WN; ++t) {
            const int n = wn * 32 * WN + t % WN * 32 + r, ml = wm * 32 * WM + t / WN * 32;
            const float *pa = xf + uint32_t(min(ml + r, rows - 1)) * K + (SPLIT ? 2 : 4) * half, *pb = wb + uint32_t(min(n, cols - 1)) * K + 4 * half;
            f32x16_t y = {};
#pragma unroll 2
            for (int k = 0; k < K; k += 8) {
                const float4 u = SPLIT ? joined(pa + k, exponent[ml + r]) : *reinterpret_cast<const float4 *>(pa + k), z = *reinterpret_cast<const float4 *>(pb + k);
                y = __builtin_amdgcn_mfma_f32_32x32x2f32(u.x, z.x, y, 0, 0, 0);
                y = __builtin_amdgcn_mfma_f32_32x32x2f32(u.y, z.y, y, 0, 0, 0);
                y = __builtin_amdgcn_mfma_f32_32x32x2f32(u.z, z.z, y, 0, 0, 0);
                y = __builtin_amdgcn_mfma_f32_32x32x2f32(u.w, z.w, y, 0, 0, 0);
            }
            const float bv = bias ? bias[n0 + min(n, cols - 1)] : 0.f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint32_t m = ml + mfma_row(e, half);
                if (m < rows && n < cols) out[m * N + n] = y[e] + bv + (residual ? residual[m * N + n] : 0.f);
            }
        }
    }
}

template <int WAVES_M, int WAVES_N, int WM, int WN, bool SPLIT>
int launch(const LinearArgs &a, void *stream) {
    constexpr int BM = 32 * WM * WAVES_M, BN = 32 * WN * WAVES_N;
    constexpr size_t lds = 3 * 2 * (BM + BN) * 64 + (BM + BN) * 4 + 4;
    static LdsGrant granted;
    if (lds > 65536 && !lffn_grant_dynamic_lds(reinterpret_cast<const void *>(&linear_kernel<WAVES_M, WAVES_N, WM, WN, SPLIT>), lds, granted))
        return LFFN_ERR_LAUNCH;
    const int64_t tiles = (a.M + BM - 1) / BM * ((a.N + BN - 1) / BN) * a.sets;
    LFFN_REQUIRE(tiles <= INT32_MAX, LFFN_ERR_UNSUPPORTED);
    linear_kernel<WAVES_M, WAVES_N, WM, WN, SPLIT><<<dim3(tiles), dim3(64 * WAVES_M * WAVES_N), lds, static_cast<hipStream_t>(stream)>>>(a);
    return lffn_launch_status();
}

}  // namespace

extern "C" int lffn_linear_f32(const float *x, const float *const *w, const float *const *bias, const float *residual, float *const *out,
                               int64_t sets, int64_t M, int64_t N, int64_t K, void *stream) {
    LFFN_REQUIRE(x && w && bias && out, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(sets >= 1 && M >= 0 && N >= 0 && K >= 0, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(x), LFFN_ERR_BAD_ARG);
    // (offsets within a tile, 256 rows of K or N numbers, are 32 bits)
    LFFN_REQUIRE(sets <= 3 && K % BK == 0 && K >= BK && N >= 1 && K <= (1 << 20) && N <= (1 << 20) && M <= INT64_C(1) << 40, LFFN_ERR_UNSUPPORTED);
    LinearArgs a{};
    for (int64_t s = 0; s < sets; ++s) {
        LFFN_REQUIRE(w[s] && out[s] && lffn_aligned16(w[s]), LFFN_ERR_BAD_ARG);
        a.w[s] = w[s];
        a.b[s] = bias[s];
        a.out[s] = out[s];
    }
    if (M == 0) return LFFN_OK;
    a.x = x;
    a.residual = residual;
    a.M = M;
    a.N = (int)N;
    a.K = (int)K;
    a.sets = (int)sets;
    // Time of each form in ns for K = 768, the same share of it for any other: a round of 256 tiles (one a compute unit) of 128 x 256
    // takes 43 us, of 128 x 192 36, of 128 x 128 27.5; tiles of 64 x 64 share compute units, 13 us at least and 8.6 per 256 tiles.
    // The middle one is the least a column when it fills its rounds and the widest does not: one matrix of 768 x 768 and 16384 rows is
    // two whole rounds of it against one and a half of 128 x 256 (84 against 94 us), three and 4096 rows one and a half against 1.1
    // (73 against 82 to 88).  Measured at 16 to 16384 rows of 512 to 1024: the form this picks is the fastest or within 3 % of it.
    auto tiles = [&](int64_t bm, int64_t bn) { return (M + bm - 1) / bm * ((N + bn - 1) / bn) * sets; };
    auto rounds = [&](int64_t bn) { return (tiles(128, bn) + 255) / 256; };
    const int64_t wide = rounds(256) * 43000, middle = rounds(192) * 36000, square = rounds(128) * 27500;
    int64_t small = tiles(64, 64) * 8600 / 256 + 4000;
    if (small < 13000) small = 13000;
    if (small <= wide && small <= middle && small <= square) return launch<2, 2, 1, 1, false>(a, stream);
    if (square < wide && square <= middle) return launch<4, 2, 1, 2, false>(a, stream);
    return middle < wide ? launch<4, 2, 1, 3, false>(a, stream) : launch<2, 4, 2, 2, false>(a, stream);
}

extern "C" int lffn_linear_norm_workspace_bytes(int64_t sets, int64_t M, int64_t N, int64_t K, int64_t *bytes) {
    LFFN_REQUIRE(bytes, LFFN_ERR_BAD_ARG);
    const bool taken = sets >= 1 && sets <= 3 && M >= 0 && M <= INT64_C(1) << 32 && N >= 1 && N <= (1 << 20) && K >= BK && K <= 2048 && K % BK == 0;
    *bytes = taken ? (M + sets * N) * (K + 1) * (int64_t)sizeof(float) : 0;
    return LFFN_OK;
}

extern "C" int lffn_linear_norm_f32(const float *x, const float *norm_weight, const float *norm_bias, float eps, const float *const *w,
                                    const float *const *bias, float *const *out, void *workspace, int64_t workspace_bytes, int64_t sets,
                                    int64_t M, int64_t N, int64_t K, void *stream) {
    LFFN_REQUIRE(x && w && bias && out, LFFN_ERR_BAD_ARG);
    int64_t need = 0;
    lffn_linear_norm_workspace_bytes(sets, M, N, K, &need);
    LFFN_REQUIRE(need > 0, LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(workspace && workspace_bytes >= need && lffn_aligned16(workspace), LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(x) && lffn_aligned16(norm_weight) && lffn_aligned16(norm_bias), LFFN_ERR_BAD_ARG);
    LinearArgs a{};
    SplitArgs p{};
    for (int64_t s = 0; s < sets; ++s) {
        LFFN_REQUIRE(w[s] && out[s] && lffn_aligned16(w[s]), LFFN_ERR_BAD_ARG);
        p.w[s] = a.w[s] = w[s];
        a.b[s] = bias[s];
        a.out[s] = out[s];
    }
    if (M == 0) return LFFN_OK;
    p.x = x;
    p.weight = norm_weight;
    p.bias = norm_bias;
    p.eps = eps;
    a.split = p.split = static_cast<uint4 *>(workspace);
    a.M = p.M = M;
    p.rows = M + sets * N;
    a.split_exponent = p.exponent = static_cast<int *>(workspace) + p.rows * K;
    a.N = p.N = (int)N;
    a.K = p.K = (int)K;
    a.sets = (int)sets;
    const dim3 grid((unsigned)((p.rows + 3) / 4)), block(256);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (K <= 256) split_rows_kernel<1><<<grid, block, 0, st>>>(p);
    else if (K <= 512) split_rows_kernel<2><<<grid, block, 0, st>>>(p);
    else if (K <= 768) split_rows_kernel<3><<<grid, block, 0, st>>>(p);
    else if (K <= 1024) split_rows_kernel<4><<<grid, block, 0, st>>>(p);
    else split_rows_kernel<8><<<grid, block, 0, st>>>(p);
    if (const int rc = lffn_launch_status(); rc != LFFN_OK) return rc;
    // as above, with the splitting out of the loop: a round of 128 x 256 40 us, of 128 x 192 32, of 128 x 128 23.5 (K = 768)
    auto rounds = [&](int64_t bn) { return ((M + 127) / 128 * ((N + bn - 1) / bn) * sets + 255) / 256; };
    const int64_t wide = rounds(256) * 40000, middle = rounds(192) * 32000, square = rounds(128) * 23500;
    if (square < wide && square <= middle) return launch<4, 2, 1, 2, true>(a, stream);
    return middle < wide ? launch<4, 2, 1, 3, true>(a, stream) : launch<2, 4, 2, 2, true>(a, stream);
}
