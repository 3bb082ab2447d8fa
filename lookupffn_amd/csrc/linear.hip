// out[m, n] = sum_k x[m, k] w[n, k] + bias[n] (+ residual[m, n]) in fp32 on the fp16 matrix cores (split_mfma.h), up to three
// matrices w (query, key and value of an attention) in one launch.
//
// A workgroup owns a tile of BM x BN results and walks k in steps of 32.  A step's numbers are fetched as they lie (fp32, 16 bytes a
// lane, two steps ahead), split on the way into LDS (hi and lo planes of 64-byte rows, the four 16-byte pieces of a row turned by
// row / 4, so that sixteen rows' reads of one piece fall on different banks) and read back as operands; three buffers, so that a
// step's products need one barrier and its first operands are there when it starts.  The products, the splitting and the LDS
// traffic are spread through each other by scheduling groups: a matrix instruction covers five vector ones.
//
// Every row of x and w is scaled by a power of two of its own, taken from its first 32 numbers, and the results are scaled back:
// any size of numbers goes, and a row that grows past its beginning 30000 times comes out infinite and is done again in fp32.
//
// What bounds it: power.  16384 x 768 x 768, three matrices: 222 us, 261 TFLOP/s of fp32 product (783 of fp16) at 1.67 GHz; with
// zeros for numbers the same kernel runs at 2.37 GHz, 194 us.  Of its clocks 62 % are matrix instructions; LDS (writes 13 clocks per
// kilobyte, reads 4 to 7) and the splitting take as long as those beside them.  The library's fp32 product takes 426 us
// (136 TFLOP/s, 0.87 of the fp32 matrix cores' peak).  Error against 64 bits 2.0e-7 of the result (library 5.0e-7; 16 rows, where
// it splits k, 2.5e-7); as six products of three bfloat16 terms 1.6e-7, but 313 us.
#include "split_mfma.h"


namespace {

constexpr int BK = 32;                                  // k of a step

struct LinearArgs {
    const float *x;              // [M, K]
    const float *residual;       // [M, N] or null
    const float *w[3], *b[3];    // [N, K], [N] or null, of every set
    float *out[3];               // [M, N]
    int64_t M;
    int N, K, sets;
};

// WAVES_M x WAVES_N wavefronts of WM x WN tiles of 32 x 32 each.
template <int WAVES_M, int WAVES_N, int WM, int WN>
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
    float *const inverse = reinterpret_cast<float *>(lds + 3 * BUF);      // [BM + BN] the rows' scales
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave % WAVES_M, wn = wave / WAVES_M;
    const int N = a.N, K = a.K;
    const int64_t M = a.M;
    // XCD b % 8 takes a contiguous range of the tiles, a tile of x against all matrices before the next
    const int per_set = (N + BN - 1) / BN, ntn = per_set * a.sets;
    const int nblk = gridDim.x, xcd = blockIdx.x & 7, q = nblk >> 3, rem = nblk & 7;
    const int tile = xcd * q + min(xcd, rem) + (blockIdx.x >> 3);
    const int64_t m0 = int64_t(tile / ntn) * BM;
    const int nt = tile % ntn, set = nt / per_set, n0 = (nt % per_set) * BN;
    const float *const w = a.w[set];

    // a thread's pieces of a step: eight numbers each of rows tid / 4 + RSTEP i, those of x before those of w
    const int chunk = tid & 3, row0 = tid >> 2;
    const float *const xa = a.x + m0 * K, *const wb = w + int64_t(n0) * K;
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
        const float *const p = (RSTEP * i < BM ? xa : wb) + k;
        *reinterpret_cast<float4 *>(&v[i][0]) = *reinterpret_cast<const float4 *>(p + src[i]);
        if (i < NP) *reinterpret_cast<float4 *>(&v[i][4]) = *reinterpret_cast<const float4 *>(p + src[i] + 4);
    };
    uint32_t h[4];
    auto place = [&](uint4 *buf, int i, int p) {
        const int plane = (RSTEP * i < BM ? BM : BN) * 4;
        uint32_t o[4];
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
    f32x16_t acc[WM][WN] = {}, low[WM][WN] = {};
#pragma unroll
    for (int i = 0; i < NC; ++i) fetch(i, 0);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        float most = 0.f;
#pragma unroll
        for (int e = 0; e < (i < NP ? 8 : 4); ++e) most = fmaxf(most, fabsf(v[i][e]));
        most = fmaxf(most, lane_xor<1>(most));
        most = fmaxf(most, lane_xor<2>(most));
        if (i == NP) most = fmaxf(most, lane_xor<4>(most));
        const PowerOfTwo s = scale_to_one(most);
        scale[i] = s.scale;
        if (i < NP) {
            if (chunk == 0) inverse[row0 + RSTEP * i] = s.inverse;
        } else if ((tid & 7) == 0) {
            inverse[RSTEP * NP + (tid >> 3)] = s.inverse;
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
    const float *const bias = a.b[set];
    float *const out = a.out[set] + m0 * N + n0;
    const float *const residual = a.residual ? a.residual + m0 * N + n0 : nullptr;
    const int rows = (int)min(int64_t(BM), M - m0), cols = min(BN, N - n0);
    bool bad = false;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
        const int n = wn * 32 * WN + j * 32 + r;
        const float bv = bias ? bias[n0 + min(n, cols - 1)] : 0.f, sb = inverse[BM + n];
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
                float y = fmaf(low[i][j][e], 1 / SPLIT_LO, acc[i][j][e]) * inverse[m] * sb;
                bad |= !is_finite(y);
                y += bv;
                if (residual) y += res[e];
                if (m < rows && n < cols) out[uint32_t(m) * N + n] = y;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (__any(bad)) {
        // the split does not carry infinities: the wavefront's results once more, on the fp32 matrix cores
#pragma unroll 1
        for (int t = 0; t < WM * WN; ++t) {
            const int n = wn * 32 * WN + t % WN * 32 + r, ml = wm * 32 * WM + t / WN * 32;
            const float *pa = xa + uint32_t(min(ml + r, rows - 1)) * K + 4 * half, *pb = wb + uint32_t(min(n, cols - 1)) * K + 4 * half;
            f32x16_t y = {};
#pragma unroll 2
            for (int k = 0; k < K; k += 8) {
                const float4 u = *reinterpret_cast<const float4 *>(pa + k), z = *reinterpret_cast<const float4 *>(pb + k);
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

template <int WAVES_M, int WAVES_N, int WM, int WN>
int launch(const LinearArgs &a, void *stream) {
    constexpr int BM = 32 * WM * WAVES_M, BN = 32 * WN * WAVES_N;
    constexpr size_t lds = 3 * 2 * (BM + BN) * 64 + (BM + BN) * 4;
    static LdsGrant granted;
    if (lds > 65536 && !lffn_grant_dynamic_lds(reinterpret_cast<const void *>(&linear_kernel<WAVES_M, WAVES_N, WM, WN>), lds, granted))
        return LFFN_ERR_LAUNCH;
    const int64_t tiles = (a.M + BM - 1) / BM * ((a.N + BN - 1) / BN) * a.sets;
    LFFN_REQUIRE(tiles <= INT32_MAX, LFFN_ERR_UNSUPPORTED);
    linear_kernel<WAVES_M, WAVES_N, WM, WN><<<dim3(tiles), dim3(64 * WAVES_M * WAVES_N), lds, static_cast<hipStream_t>(stream)>>>(a);
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
    if (small <= wide && small <= middle && small <= square) return launch<2, 2, 1, 1>(a, stream);
    if (square < wide && square <= middle) return launch<4, 2, 1, 2>(a, stream);
    return middle < wide ? launch<4, 2, 1, 3>(a, stream) : launch<2, 4, 2, 2>(a, stream);
}
