// Gradient of the layer's gather w.r.t. the tables, table-major with the
// gradient slice accumulated in LDS:
//
//   grad_tables[t, s, :] (+)= sum over tokens b with (code[b,t] & (S-1)) == s of score[b,t] * g[b,:]
//
// The reference computes this with one global fp32 atomicAdd per (token, table,
// column) (gather_kernel_fp32.cu:83-91).  Here a 1024-lane workgroup owns one
// table and a 64-column slice: their gradient (S rows x 64 columns) lives in LDS
// as DOUBLES (128 KiB for S = 256), zeroed at the start.  The workgroup streams
// over ALL tokens; a wavefront takes one token at a time, lane l holding column l
// of the slice, and adds score * g into the row the token's code selects with one
// ds_add_f64: 64 lanes hit 64 consecutive doubles, so an instruction never has a
// bank conflict or two lanes on one address, however skewed the code distribution
// is.  At the end the slice is rounded to fp32 and written to HBM with plain
// coalesced stores: no global atomics, and the output needs no zero-fill.
//
// Why doubles: on gfx950 the LDS fp32 atomic add is processed lane by lane (192
// clocks per 64-lane instruction measured), while the fp64 atomic add runs at the
// rate of an LDS integer atomic (under 10 clocks).  Accumulating in fp64 also makes
// the sum independent of the order in which wavefronts reach a row up to one fp32
// rounding at the end, so results repeat from run to run except where that final
// rounding sits on a tie.
//
// (row offset, score) pairs of 64 tokens are fetched by the 64 lanes at once (one
// token per lane), parked in a wavefront-private LDS strip and read back as a
// broadcast ds_read_b64 when their token comes up.
#include "lffn_common.h"

#include <hip/amd_detail/amd_hip_unsafe_atomics.h>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int WG = 1024;
constexpr int WAVES = WG / 64;
constexpr int COLS = 64;           // columns per slice = lanes per token
constexpr int MAX_S = 256;
constexpr int XCDS = 8;
constexpr int GDEPTH = 16;         // gradient rows in flight per wavefront

struct ScatterArgs {
    const int32_t *code;   // [B, T]
    const float *score;    // [B, T]
    const float *g;        // [B, Do]
    float *out;            // [T, S, Do]
    int64_t B;
    int T, S, Do;
    int nslices, per_xcd;
    int accumulate;
    int past_caches;       // lffn_rows_written_past_caches
};

__global__ __launch_bounds__(WG) void lookup_scatter_lds_kernel(ScatterArgs a) {
    extern __shared__ double lds[];                // [S][COLS] doubles, then [WAVES][64] uint2
    const int tab_elems = a.S * COLS;
    uint2 *strip = reinterpret_cast<uint2 *>(lds + tab_elems) + (threadIdx.x >> 6) * 64;

    const int xcd = blockIdx.x % XCDS;
    const int unit = xcd * a.per_xcd + blockIdx.x / XCDS;
    if (unit >= a.T * a.nslices) return;           // uniform over the workgroup
    // units that share a slice of g are neighbours, so they land on one XCD
    const int slice = unit / a.T;
    const int t = unit % a.T;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;

    for (int q = tid; q < tab_elems / 2; q += WG)
        reinterpret_cast<double2 *>(lds)[q] = make_double2(0.0, 0.0);
    __syncthreads();

    const int mask = a.S - 1;
    const float *gcol = a.g + (size_t)slice * COLS + lane;
    double *my_col = lds + lane;

    // The wavefront's token stream: batch k covers tokens wave*64 + k*1024 + [0, 64).
    // The wavefront number is made scalar so that all per-token address arithmetic
    // runs on the scalar unit; only the lane's column offset is a vector value.
    const int swave = __builtin_amdgcn_readfirstlane(wave);
    const int64_t first = int64_t(swave) * 64;
    const int64_t nbatch = first < a.B ? (a.B - first + WG - 1) / WG : 0;
    const int64_t last = a.B - 1;

    auto load_pair = [&](int64_t batch) {
        const int64_t tok = min<int64_t>(first + batch * WG + lane, last);
        uint2 pr;
        pr.x = (unsigned)((a.code[tok * a.T + t] & mask) * COLS);
        pr.y = __float_as_uint(a.score[tok * a.T + t]);
        return pr;
    };

    uint2 pr_next = make_uint2(0u, 0u);
    if (nbatch > 0) pr_next = load_pair(0);
    for (int64_t batch = 0; batch < nbatch; ++batch) {
        const int64_t base = first + batch * WG;
        strip[lane] = pr_next;     // wavefront-private: ordered by the LDS queue, no barrier needed
        pr_next = load_pair(batch + 1 < nbatch ? batch + 1 : batch);   // pairs run one batch ahead
        const int n = (int)min<int64_t>(64, a.B - base);
        const float *gp = gcol + base * a.Do;
        if (n == 64) {
#pragma unroll
            for (int i0 = 0; i0 < 64; i0 += GDEPTH) {
                float gv[GDEPTH];
                uint2 pr[GDEPTH];
#pragma unroll
                for (int u = 0; u < GDEPTH; ++u) gv[u] = gp[(size_t)(i0 + u) * a.Do];
#pragma unroll
                for (int u = 0; u < GDEPTH; ++u) pr[u] = strip[i0 + u];   // broadcast reads
#pragma unroll
                for (int u = 0; u < GDEPTH; ++u)
                    unsafeAtomicAdd(my_col + pr[u].x, (double)(__uint_as_float(pr[u].y) * gv[u]));
            }
        } else {
            for (int i = 0; i < n; ++i) {
                const uint2 pr = strip[i];
                unsafeAtomicAdd(my_col + pr.x, (double)(__uint_as_float(pr.y) * gp[(size_t)i * a.Do]));
            }
        }
    }
    __syncthreads();

    // flush: rows of table t x this slice, 16 lanes per 256-byte row segment
    for (int q = tid; q < a.S * (COLS / 4); q += WG) {
        const int row = q / (COLS / 4);
        const int v = q % (COLS / 4);
        const double2 lo = reinterpret_cast<double2 *>(lds)[2 * q];
        const double2 hi = reinterpret_cast<double2 *>(lds)[2 * q + 1];
        float4 val = make_float4((float)lo.x, (float)lo.y, (float)hi.x, (float)hi.y);
        float *dst = a.out + ((size_t)t * a.S + row) * a.Do + (size_t)slice * COLS + v * 4;
        if (a.accumulate) {
            const float4 old = *reinterpret_cast<const float4 *>(dst);
            val.x += old.x; val.y += old.y; val.z += old.z; val.w += old.w;
        }
        *reinterpret_cast<float4 *>(dst) = val;
    }
}

// The same for few tokens.  Most rows of the gradient are then zero and the rest sums of a few products, and the kernel above
// spends its time clearing and emptying 128 KB of LDS with one workgroup on a compute unit.  Here a workgroup owns 32 rows of a
// table, every groups-th: it lists the (token, score) pairs of each row, and a wavefront adds up a row's products in registers (in
// fp64, as above) and writes the whole row: plain streaming stores from many wavefronts.  A row's pairs are listed in any order, which
// fp64 sums do not show but for ties of the final rounding.  128 tables of 768 columns: 64 tokens 35.8 -> 18.2 us (100 MB
// written: 5.5 TB/s), 1024 tokens 76.5 -> 35.5, 2048 112 -> 77 (the sorted form 79); 512
// tables of 1024 columns: 64 tokens 179 -> 100, 1500 268 (sorted 261), 2048 409 (288).
//
// Rows of many pairs would leave that to one wavefront, a chain of loads (2048 tokens of which half fall on one row of 128 tables of
// 768 columns: 264 us).  A row of more than LONG_ROW pairs, and of four times the average, is summed by all workgroups of its
// table, a slice of the columns each: every one of them lists it beside its own short rows.  Half on one row 83 us, all on one 426 ->
// 69, codes with Zipf's distribution 219 -> 95-100 (112 above, whatever the distribution); evenly spread codes as before (77).
constexpr int ROWS_PER_WG = 32;
constexpr int LIST_MAX_B = LFFN_SCATTER_LIST_TOKENS;
constexpr int LIST_BATCHES = LIST_MAX_B / 256;
constexpr int LONG_ROW = 32;
constexpr int SLICE_QUADS = 16;                    // fewest columns of a slice, in fours

template <int NC>
__global__ __launch_bounds__(256) void lookup_scatter_list_kernel(ScatterArgs a, int groups, int long_from) {
    __shared__ int count[MAX_S], start[MAX_S], cursor[MAX_S], wave_sum[4], long_row[LIST_MAX_B / LONG_ROW], nlong;
    __shared__ double part[4][256];                // (columns by threads: no bank conflicts)
    extern __shared__ double lds[];
    uint2 *list = reinterpret_cast<uint2 *>(lds);  // [B]: the listed rows have no token in common
    const int unit = (int)(blockIdx.x % XCDS) * a.per_xcd + (int)(blockIdx.x / XCDS);     // neighbouring tables on one XCD
    if (unit >= a.T * groups) return;              // uniform over the workgroup
    const int t = unit / groups, group = unit % groups;
    const int nrows = min(ROWS_PER_WG, a.S);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto mine = [&](int r) { return (r & (groups - 1)) == group; };     // its rows: group + groups * i
    int row[LIST_BATCHES];
#pragma unroll
    for (int k = 0; k < LIST_BATCHES; ++k) {
        const int64_t b = tid + 256 * k;
        row[k] = b < a.B ? a.code[b * a.T + t] & (a.S - 1) : -1;
    }
    count[tid] = 0;
    if (tid == 0) nlong = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < LIST_BATCHES; ++k)
        if (row[k] >= 0) atomicAdd(&count[row[k]], 1);
    __syncthreads();
    {   // a row per thread: where its list starts, if it is listed here
        const int n = count[tid], listed = mine(tid) || n > long_from ? n : 0;
        int inc = listed;
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(inc, d);
            if (lane >= d) inc += v;
        }
        if (lane == 63) wave_sum[wave] = inc;
        if (n > long_from) long_row[atomicAdd(&nlong, 1)] = tid;
        __syncthreads();
        int before = inc - listed;
        for (int w = 0; w < wave; ++w) before += wave_sum[w];
        start[tid] = before;
        cursor[tid] = listed ? before : -1;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < LIST_BATCHES; ++k)
        if (row[k] >= 0 && (mine(row[k]) || count[row[k]] > long_from)) {
            const int b = tid + 256 * k;
            list[atomicAdd(&cursor[row[k]], 1)] = make_uint2((unsigned)b, __float_as_uint(a.score[(int64_t)b * a.T + t]));
        }
    __syncthreads();
    for (int i = wave; i < nrows; i += 4) {
        const int r = group + groups * i;
        const int n0 = __builtin_amdgcn_readfirstlane(start[r]), n1 = n0 + __builtin_amdgcn_readfirstlane(count[r]);
        if (n1 - n0 > long_from) continue;
        float *dst = a.out + ((size_t)t * a.S + r) * a.Do;
        for (int col0 = 0; col0 < a.Do; col0 += 256 * NC) {
            double acc[NC][4];
            int col[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                col[c] = col0 + 256 * c + 4 * lane;
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[c][e] = 0.0;
            }
            for (int i = n0; i < n1; i += 4) {
                float4 gv[4][NC];
                float sv[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint2 pr = list[min(i + u, n1 - 1)];
                    const float *gp = a.g + (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)pr.x) * a.Do;
                    sv[u] = __uint_as_float(pr.y);
#pragma unroll
                    for (int c = 0; c < NC; ++c) gv[u][c] = *reinterpret_cast<const float4 *>(gp + (col[c] < a.Do ? col[c] : 0));
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (i + u < n1) {                          // uniform
#pragma unroll
                        for (int c = 0; c < NC; ++c) {
                            acc[c][0] += (double)(sv[u] * gv[u][c].x); acc[c][1] += (double)(sv[u] * gv[u][c].y);
                            acc[c][2] += (double)(sv[u] * gv[u][c].z); acc[c][3] += (double)(sv[u] * gv[u][c].w);
                        }
                    }
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (col[c] >= a.Do) continue;
                float4 v = make_float4((float)acc[c][0], (float)acc[c][1], (float)acc[c][2], (float)acc[c][3]);
                if (a.accumulate) {
                    const float4 old = *reinterpret_cast<const float4 *>(dst + col[c]);
                    v.x += old.x; v.y += old.y; v.z += old.z; v.w += old.w;
                }
                if (a.past_caches) __builtin_nontemporal_store((f32x4){v.x, v.y, v.z, v.w}, reinterpret_cast<f32x4 *>(dst + col[c]));
                else *reinterpret_cast<float4 *>(dst + col[c]) = v;
            }
        }
    }
    // long rows: this workgroup's columns, in fours, a thread each; what threads that leaves share out the pairs
    const int quads = a.Do / 4, slices = min(groups, max(1, quads / SLICE_QUADS));
    if (group >= slices) return;                   // uniform
    const int q_end = (int)((int64_t)quads * (group + 1) / slices);
    for (int i = 0; i < nlong; ++i) {
        const int r = long_row[i], n0 = start[r], n = count[r];
        for (int q0 = (int)((int64_t)quads * group / slices); q0 < q_end; q0 += 64) {
            const int width = min(64, q_end - q0), shares = 256 / width, share = tid / width, q = q0 + tid % width;
            double acc[4] = {0.0, 0.0, 0.0, 0.0};
            if (share < shares)
                for (int k = share; k < n; k += 8 * shares) {
                    float4 gv[8];
                    float sv[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const uint2 pr = list[n0 + min(k + u * shares, n - 1)];
                        sv[u] = __uint_as_float(pr.y);
                        gv[u] = *reinterpret_cast<const float4 *>(a.g + (size_t)pr.x * a.Do + 4 * q);
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (k + u * shares < n) {
                            acc[0] += (double)(sv[u] * gv[u].x); acc[1] += (double)(sv[u] * gv[u].y);
                            acc[2] += (double)(sv[u] * gv[u].z); acc[3] += (double)(sv[u] * gv[u].w);
                        }
                }
#pragma unroll
            for (int e = 0; e < 4; ++e) part[e][tid] = acc[e];
            __syncthreads();
            if (tid < width) {
                for (int w = 1; w < shares; ++w)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e] += part[e][tid + w * width];
                float4 v = make_float4((float)acc[0], (float)acc[1], (float)acc[2], (float)acc[3]);
                float4 *dst = reinterpret_cast<float4 *>(a.out + ((size_t)t * a.S + r) * a.Do + 4 * q);
                if (a.accumulate) {
                    const float4 old = *dst;
                    v.x += old.x; v.y += old.y; v.z += old.z; v.w += old.w;
                }
                *dst = v;
            }
            __syncthreads();
        }
    }
}

int launch_list(const ScatterArgs &args, hipStream_t st) {
    ScatterArgs a = args;
    const int groups = a.S > ROWS_PER_WG ? a.S / ROWS_PER_WG : 1;
    a.past_caches = lffn_rows_written_past_caches(int64_t(a.T) * a.S, a.Do);
    a.per_xcd = (a.T * groups + XCDS - 1) / XCDS;
    const dim3 grid((unsigned)(a.per_xcd * XCDS));
    const size_t lds_bytes = (size_t)a.B * sizeof(uint2);
    const int average = (int)((a.B + a.S - 1) / a.S), long_from = 4 * average > LONG_ROW ? 4 * average : LONG_ROW;
    switch ((a.Do + 255) / 256) {
        case 1: hipLaunchKernelGGL(lookup_scatter_list_kernel<1>, grid, dim3(256), lds_bytes, st, a, groups, long_from); break;
        case 2: hipLaunchKernelGGL(lookup_scatter_list_kernel<2>, grid, dim3(256), lds_bytes, st, a, groups, long_from); break;
        case 3: hipLaunchKernelGGL(lookup_scatter_list_kernel<3>, grid, dim3(256), lds_bytes, st, a, groups, long_from); break;
        default: hipLaunchKernelGGL(lookup_scatter_list_kernel<4>, grid, dim3(256), lds_bytes, st, a, groups, long_from); break;
    }
    return lffn_launch_status();
}

__global__ __launch_bounds__(256) void fill_zero_kernel(float4 *p, int64_t n4) {
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n4; i += int64_t(gridDim.x) * 256)
        p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

}  // namespace

extern "C" int lffn_lookup_scatter_f32(const int32_t *code, const float *score, const float *g,
                                       float *grad_tables, int64_t B, int64_t T, int64_t S, int64_t Do,
                                       int32_t accumulate, void *stream) {
    LFFN_REQUIRE(B >= 0 && T >= 0 && Do >= 1, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_is_pow2(S) && S <= (1 << 24) && T * S <= 0x7fffffff, LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(Do % 64 == 0 && Do <= (1 << 20) && T <= (1 << 24), LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(B <= (int64_t(1) << 31) - 1, LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(grad_tables || T == 0, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE((code && score && g) || B * T == 0, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(grad_tables) && lffn_aligned16(g), LFFN_ERR_BAD_ARG);
    if (T == 0) return LFFN_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t units = T * (Do / COLS);
    if (S > MAX_S || units > (int64_t(1) << 24)) {
        // tables too large for the LDS slice: zero-fill, then global atomics
        if (!accumulate) {
            const int64_t n4 = T * S * Do / 4;
            hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((n4 + 255) / 256 < 65536 ? (n4 + 255) / 256 : 65536)), dim3(256), 0,
                               st, reinterpret_cast<float4 *>(grad_tables), n4);
            int rc = lffn_launch_status();
            if (rc != LFFN_OK) return rc;
        }
        if (B == 0) return LFFN_OK;
        return lffn_internal_lookup_scatter_atomic(code, score, g, grad_tables, B, T, S, Do, stream);
    }
    ScatterArgs a{};
    a.code = code; a.score = score; a.g = g; a.out = grad_tables;
    a.B = B; a.T = (int)T; a.S = (int)S; a.Do = (int)Do;
    a.nslices = (int)(Do / COLS);
    a.per_xcd = (int)((units + XCDS - 1) / XCDS);
    a.accumulate = accumulate;
    // The LDS form takes its time per round of one workgroup on each of 256 compute units: with a single round it is the faster one
    // (32 tables of 256 columns: 64 tokens 7.0 us against 7.7, 512 9.4 against 10.8).  So it is where a table is one workgroup of the
    // list form and has many tokens (128 tables of 32 x 768: 512 tokens 36.5 against 35, 1024 60.5 against 60.3, 2048 96 against 134).
    if (units > 256 && B <= (S > ROWS_PER_WG ? LIST_MAX_B : 512) && T * S <= (int64_t(1) << 30)) return launch_list(a, st);
    const size_t lds_bytes = size_t(S) * COLS * 8 + size_t(WAVES) * 64 * 8;
    static LdsGrant granted;      // one record per kernel instantiation
    if (!lffn_grant_dynamic_lds(reinterpret_cast<const void *>(lookup_scatter_lds_kernel), lds_bytes, granted)) return LFFN_ERR_LAUNCH;
    hipLaunchKernelGGL(lookup_scatter_lds_kernel, dim3(a.per_xcd * XCDS), dim3(WG), lds_bytes, st, a);
    return lffn_launch_status();
}
