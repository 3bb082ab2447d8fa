// Table gradient of the lookup layer without atomics on the accumulators:
//
//   grad_tables[t][code[b][t]][:] += score[b][t] * g[b][:]        (PL/gather/cuda/kernel.py:190-202,
//                                                                   PL/gather/cuda/extension/gather_kernel_fp32.cu:49)
//
// Three launches and a workspace.
//
// lookup_prep_kernel: code and score are [B, T]; a table's column is one value per 4*T bytes,
// and 64 lanes reading it are 64 separate requests, which made the sort four times slower
// than it is.  The kernel writes them transposed, [T, B] (codes masked, as 16-bit values).
//
// lookup_sort_pack_kernel: two jobs in one launch, by workgroup number.  The sort occupies one
// workgroup per table (128 of the 256 compute units at 128 tables) and is bound by latency; the
// copy of g to a slice-major layout [Do/32][B + 1][32] (in which the 128-byte row pieces of a slice
// are contiguous: with rows 4*Do bytes apart the pieces of one slice fall on a quarter of the L2
// channels) is pure memory traffic and depends on nothing: its workgroups fill the rest of the
// chip while the sort runs (23 + 25 us as two launches at 16384 tokens x 128 tables x 768).
//
// The sort: one workgroup per table sorts the tokens by their code for that
// table (a stable counting sort: per-wavefront histograms over contiguous token ranges,
// ranks inside a 64-token batch from ballots over the code bits) and writes (token, score)
// pairs bucket by bucket: into LDS first (a 16-bit token and a score per entry: at most 18432
// entries, 108 KB), from where the list goes to memory in whole lines; written straight
// from the ranks, every wavefront store was 64 separate 8-byte requests.  Every bucket is padded to a multiple of eight entries,
// so that eight consecutive entries always belong to one code, and the bucket boundaries are stored in units of eight entries.
// The padding names token B, whose row of the copy of g is zero (a token of the bucket with weight 0 would make a row of an
// infinite gradient NaN).
//
// lookup_scatter_sorted_kernel: one workgroup per (table, 32-column slice).  The sorted
// list is cut into equal pieces, one per wavefront, whatever the bucket sizes (a skewed code
// distribution costs nothing).  A wavefront walks its piece eight tokens at a time: lane
// group q = lane / 8 takes token q of the step, its eight lanes load the token's 128-byte
// piece of g and multiply-add it into registers; at a bucket boundary (wave-uniform,
// because of the padding) the eight partial sums are added across the lane groups and the
// row is stored.  Buckets cut by a piece boundary go to LDS and one wavefront adds the
// pieces in order after a barrier.  Every row of the slice is written exactly once with
// plain stores: no zero-fill, no atomics, and the sum order is fixed (run-to-run
// reproducible).  The slices are dealt to the XCDs so that the workgroups running on one
// XCD read the same 32 columns of g (2 MB at 16384 tokens), which then stay in its L2.
#include "lffn_common.h"

namespace {

constexpr int SORT_WG = 1024;
constexpr int SORT_WAVES = SORT_WG / 64;
constexpr int MAX_S = 512;
constexpr int XCDS = 8;
constexpr int SORT_DEPTH = 16;      // batches of 64 tokens whose loads are in flight per wavefront

constexpr int MWG = 512;             // main kernel: threads per workgroup
constexpr int MWAVES = MWG / 64;
constexpr int SC = 32;               // columns per slice: 8 lanes x float4
constexpr int U = 8;                 // steps (of eight tokens) per batch = one 64-entry load of pairs

struct PrepArgs {
    const int32_t *code;   // [B, T]
    const float *score;    // [B, T]
    const float *g;        // [B, Do]
    uint16_t *code_t;      // [T, Bp]
    float *score_t;        // [T, Bp]
    float *g_packed;       // [Do / SC][B + 1][SC], the last row zero
    float *sums;           // [ceil((B + 1) / PACK_TOKENS), Do] or null: column sums of the rows of g that a workgroup copies
    int64_t B, Bp;
    int T, S, Do, tiles_t;
};

// one 64 x 64 tile of code and score per workgroup
__global__ __launch_bounds__(256) void lookup_prep_kernel(PrepArgs a) {
    __shared__ int sc[64][65];
    __shared__ float ss[64][65];
    const int tid = threadIdx.x, lane = tid & 63, row0 = tid >> 6;
    const int64_t b0 = int64_t(blockIdx.x / a.tiles_t) * 64;
    const int t0 = (blockIdx.x % a.tiles_t) * 64;
    const int mask = a.S - 1;
    // all sixteen rows of a thread are requested before the first is used
    int cv[16];
    float sv[16];
    const int t_in = t0 + lane;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int64_t b = b0 + row0 + 4 * i;
        const bool live = b < a.B && t_in < a.T;
        cv[i] = live ? a.code[b * a.T + t_in] : 0;
        sv[i] = live ? a.score[b * a.T + t_in] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        sc[row0 + 4 * i][lane] = cv[i] & mask;
        ss[row0 + 4 * i][lane] = sv[i];
    }
    __syncthreads();
    const int64_t b_out = b0 + lane;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = row0 + 4 * i, t = t0 + r;
        if (b_out < a.B && t < a.T) {
            a.code_t[(size_t)t * a.Bp + b_out] = (uint16_t)sc[lane][r];
            a.score_t[(size_t)t * a.Bp + b_out] = ss[lane][r];
        }
    }
}

constexpr int PACK_TOKENS = 32;      // rows of g per workgroup of the slice-major copy
typedef float f32x4 __attribute__((ext_vector_type(4)));

// PACK_TOKENS rows of g, copied to the slice-major layout (workgroup `blk` of the copy); row B is the padding's.  A thread has four
// columns of every G-th row, so that their sum (the output bias's gradient) is a few additions and a pass over LDS (a
// launch of its own for them took 14 us at 16384 x 768, this one is no longer for it).  g is read nontemporally, since the copy is
// what is read from here on: training step at 16384 x 768 745 -> 738 us.
__device__ __forceinline__ void pack_rows(const PrepArgs &a, int64_t blk) {
    extern __shared__ int sm[];
    float4 *const part = reinterpret_cast<float4 *>(sm);     // [SORT_WG]
    const int64_t b0 = blk * PACK_TOKENS;
    for (int q0 = 0; q0 < a.Do / 4; q0 += SORT_WG) {
        const int q = min(a.Do / 4 - q0, SORT_WG), G = SORT_WG / q;
        const int grp = threadIdx.x / q, col = (q0 + (int)threadIdx.x % q) * 4;
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        // eight loads per thread in flight before the first store (a store must not overtake a load the compiler
        // cannot prove independent of it, so load-store pairs one after the other would each wait out a round trip)
        constexpr int DEPTH = 8;
        for (int r0 = grp < G ? grp : PACK_TOKENS; r0 < PACK_TOKENS; r0 += G * DEPTH) {
            float4 v[DEPTH];
#pragma unroll
            for (int i = 0; i < DEPTH; ++i) {
                const int64_t b = b0 + r0 + i * G;
                v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (r0 + i * G < PACK_TOKENS && b < a.B) {
                    const f32x4 w = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(a.g + (size_t)b * a.Do + col));
                    v[i] = make_float4(w.x, w.y, w.z, w.w);
                }
            }
#pragma unroll
            for (int i = 0; i < DEPTH; ++i) {
                const int64_t b = b0 + r0 + i * G;
                sum.x += v[i].x; sum.y += v[i].y; sum.z += v[i].z; sum.w += v[i].w;
                if (r0 + i * G < PACK_TOKENS && b <= a.B)
                    *reinterpret_cast<float4 *>(a.g_packed + ((size_t)(col / SC) * (a.B + 1) + b) * SC + col % SC) = v[i];
            }
        }
        if (!a.sums) continue;                                // uniform
        __syncthreads();                                      // (the columns before have been read)
        part[threadIdx.x] = sum;
        __syncthreads();
        if (grp == 0) {
            for (int k = 1; k < G; ++k) {
                const float4 t = part[threadIdx.x + k * q];
                sum.x += t.x; sum.y += t.y; sum.z += t.z; sum.w += t.w;
            }
            *reinterpret_cast<float4 *>(a.sums + blk * a.Do + col) = sum;
        }
    }
}

struct SortArgs {
    const uint16_t *code;  // [T, Bp], masked
    const float *score;    // [T, Bp]
    uint2 *pairs;          // [T, stride] (token, score bits)
    int32_t *off8;         // [T, S + 1] bucket starts, in units of eight entries
    int64_t B, Bp, stride;
    int T, S, nbits;
    int stage;             // the sorted list is collected in LDS and written out in whole lines (it fits: S <= 256)
};

__device__ __forceinline__ void sort_table(const SortArgs &a, const int t) {
    extern __shared__ int sm[];
    const int S = a.S;
    int *hist = sm;                    // [SORT_WAVES][S]: counts, then running write positions
    int *count = hist + SORT_WAVES * S;
    int *start = count + S;            // padded bucket starts (entries)
    int *total = start + S;
    float *sc_s = reinterpret_cast<float *>(total + 4);                       // [stride] scores of the sorted list
    unsigned short *tok_s = reinterpret_cast<unsigned short *>(sc_s + a.stride);   // [stride] tokens

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint16_t *code = a.code + (size_t)t * a.Bp;
    const float *score = a.score + (size_t)t * a.Bp;
    for (int q = tid; q < SORT_WAVES * S; q += SORT_WG) hist[q] = 0;
    __syncthreads();

    // A wavefront takes up to SORT_DEPTH batches of 64 consecutive tokens (the launch keeps B within 1024 * SORT_DEPTH).
    // Their codes and scores are loaded once, all loads in flight together, and stay in registers through both
    // passes, as does every token's rank among the tokens of its batch with the same code (from ballots over
    // the code bits): the first pass counts a batch's codes once per code (the lowest lane of each adds the
    // whole count: no two lanes of an instruction touch one counter, however skewed the codes are), the
    // second turns ranks into positions.
    const int64_t per = ((a.B + SORT_WG - 1) / SORT_WG) * 64;       // tokens per wavefront, whole batches
    const int64_t lo = min<int64_t>(a.B, wave * per), hi = min<int64_t>(a.B, lo + per);
    int *myh = hist + wave * S;
    int cv[SORT_DEPTH], rk[SORT_DEPTH];
    float sv[SORT_DEPTH];
#pragma unroll
    for (int k = 0; k < SORT_DEPTH; ++k) {
        const int64_t b = lo + 64 * k + lane;                    // loads are unconditional (clamped), so none waits for another
        const int64_t bc = min<int64_t>(b, a.B - 1);
        const int c = code[bc];
        sv[k] = score[bc];
        cv[k] = b < hi ? c : -1;
    }
#pragma unroll
    for (int k = 0; k < SORT_DEPTH; ++k) {
        rk[k] = 0;
        if (lo + 64 * k >= hi) continue;                         // uniform
        const bool live = cv[k] >= 0;
        const int c = live ? cv[k] : 0;
        unsigned long long m = __ballot(live);
        for (int bit = 0; bit < a.nbits; ++bit) {
            const bool mine = (c >> bit) & 1;
            const unsigned long long bb = __ballot(mine);
            m &= mine ? bb : ~bb;
        }
        const int rank = __popcll(m & ((1ull << lane) - 1ull));
        const int cnt = __popcll(m);
        rk[k] = rank | (cnt << 8);
        if (live && rank == 0) myh[c] += cnt;
    }
    __syncthreads();
    for (int c = tid; c < S; c += SORT_WG) {
        int sum = 0;
        for (int w = 0; w < SORT_WAVES; ++w) {
            const int v = hist[w * S + c];
            hist[w * S + c] = sum;
            sum += v;
        }
        count[c] = sum;
        start[c] = (sum + 7) & ~7;
    }
    __syncthreads();
    if (wave == 0) {                   // exclusive scan of the padded counts
        const int per_lane = (S + 63) / 64;
        int loc = 0;
        for (int k = 0; k < per_lane; ++k) {
            const int i = lane * per_lane + k;
            if (i < S) loc += start[i];
        }
        int inc = loc;
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(inc, d);
            if (lane >= d) inc += v;
        }
        int run = inc - loc;
        for (int k = 0; k < per_lane; ++k) {
            const int i = lane * per_lane + k;
            if (i < S) {
                const int v = start[i];
                start[i] = run;
                run += v;
            }
        }
        if (lane == 63) *total = inc;
    }
    __syncthreads();
    for (int c = tid; c < S; c += SORT_WG) {
        const int o = start[c];
        a.off8[(size_t)t * (S + 1) + c] = o >> 3;
        for (int w = 0; w < SORT_WAVES; ++w) hist[w * S + c] += o;
    }
    if (tid == 0) a.off8[(size_t)t * (S + 1) + S] = *total >> 3;
    __syncthreads();

    uint2 *out = a.pairs + (size_t)t * a.stride;
#pragma unroll
    for (int k = 0; k < SORT_DEPTH; ++k) {
        if (lo + 64 * k >= hi) continue;                         // uniform
        if (cv[k] >= 0) {
            const int c = cv[k], rank = rk[k] & 0xff, cnt = rk[k] >> 8;
            const int base = myh[c];                              // all lanes of a code read before its last lane writes
            if (a.stage) {                                        // uniform
                tok_s[base + rank] = (unsigned short)(lo + 64 * k + lane);
                sc_s[base + rank] = sv[k];
            } else {
                out[base + rank] = make_uint2((unsigned)(lo + 64 * k + lane), __float_as_uint(sv[k]));
            }
            if (rank == cnt - 1) myh[c] = base + cnt;
        }
    }
    __syncthreads();
    for (int c = tid; c < S; c += SORT_WG) {
        const int n = count[c], o = start[c];
        for (int p = n; p < ((n + 7) & ~7); ++p) {
            if (a.stage) {
                tok_s[o + p] = (unsigned short)a.B;
                sc_s[o + p] = 0.f;
            } else {
                out[o + p] = make_uint2((unsigned)a.B, 0u);
            }
        }
    }
    if (!a.stage) return;                                     // uniform
    __syncthreads();
    const int n_out = *total;
    for (int i = tid; i < n_out; i += SORT_WG) out[i] = make_uint2((unsigned)tok_s[i], __float_as_uint(sc_s[i]));
}

// workgroups [0, nsort): the sort of one table each; the others: PACK_TOKENS rows of the copy of g each
__global__ __launch_bounds__(SORT_WG) void lookup_sort_pack_kernel(SortArgs sa, PrepArgs pa, int nsort) {
    if ((int)blockIdx.x < nsort) sort_table(sa, (int)blockIdx.x);      // uniform over the workgroup
    else pack_rows(pa, int64_t(blockIdx.x) - nsort);
}

struct SortedArgs {
    const uint2 *pairs;    // table t's list starts at t * stride
    const int32_t *off8;   // [T, S + 1] bucket starts inside that list, in units of eight entries
    const float *g;        // [Do / SC][B + 1][SC]
    float *out;            // [rows, Do]; table t's rows from t * S on
    int64_t stride, rows;
    unsigned last_token;   // B: the padding's
    int T, S, Do, nslices, accumulate;
    int more;              // a later launch adds to these rows
};

__device__ __forceinline__ float4 add4(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

// v + (v of the lane 16 / 32 positions away): gfx950's row and half-wave swaps, no LDS traffic
__device__ __forceinline__ float add_xor16(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float add_xor32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// v + (v of lane ^ 8): a DPP rotation by eight inside the 16-lane row
__device__ __forceinline__ float add_xor8(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true));
}

// sum over the eight lane groups; afterwards every lane holds the total of its column group
__device__ __forceinline__ float4 sum_groups(float4 v) {
    v.x = add_xor32(add_xor16(add_xor8(v.x)));
    v.y = add_xor32(add_xor16(add_xor8(v.y)));
    v.z = add_xor32(add_xor16(add_xor8(v.z)));
    v.w = add_xor32(add_xor16(add_xor8(v.w)));
    return v;
}

// ADD: the sums are added to what a.out holds.  They are kept in LDS, and the rows read, added to and written at the end, eight of a
// thread's pieces in flight: read where a bucket ends, every row was waited for with all that was in flight behind it (the second
// 16384 tokens of 128 tables of 512 columns 264 -> 214 us; requested when the bucket begins 255, as atomic additions 249).
template <bool ADD>
__global__ __launch_bounds__(MWG) void lookup_scatter_sorted_kernel(SortedArgs a) {
    extern __shared__ int sm[];
    int *off = sm;                                            // [S + 1]
    int *flag = off + ((a.S + 1 + 3) & ~3);                     // [MWAVES][4]: head code, head closes, tail code
    float *slot = reinterpret_cast<float *>(flag + MWAVES * 4);   // [MWAVES][2][SC]
    float *row_s = slot + MWAVES * 2 * SC;                      // ADD: [S][SC]

    const int xcd = blockIdx.x % XCDS, idx = blockIdx.x / XCDS;
    const int slice = xcd + XCDS * (idx / a.T);
    const int t = idx % a.T;
    if (slice >= a.nslices) return;                           // uniform over the workgroup
    const int S = (int)min<int64_t>(a.S, a.rows - (int64_t)t * a.S);      // the last table of a row count that a.S does not divide

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = lane >> 3, j = lane & 7;
    for (int q = tid; q <= S; q += MWG) off[q] = a.off8[(size_t)t * (a.S + 1) + q];
    if (tid < MWAVES * 4) flag[tid] = -1;
    __syncthreads();

    float *orow = a.out + (size_t)t * a.S * a.Do + (size_t)slice * SC + j * 4;     // + code * Do
    // Rows that nothing adds to any more go out nontemporally: in the caches they would take the place of g.  Read again next, 32768 x 512,
    // that costs 7 us of 1490.  With a reader behind the pass, unlike the lists and the sums of few pairs (lffn_rows_written_past_caches), it
    // costs no more than it gives: a training step of 2500 tokens and more of 128 to 512 tables takes the same alone and with SGD, clipping
    // or Adam behind it; the operator's pass, plainly -> nontemporally, alone, with SGD, with Adam:
    //   4096 x 128 x 512  231 -> 226 (219 for 229 where the passes' results stay), 270 -> 264, 317 -> 318    3000 x 128 x 512  206 -> 204, 245 -> 239, 295 -> 298
    //   8192 x 64 x 512  217 -> 202, 232 -> 240, 283 -> 284    2500 x 128 x 768  266 -> 265, 332 -> 337, 462 -> 462    8192 x 256 x 512  601 -> 586, 671 -> 662
    auto store_row = [&](float *p, float4 v) {
        if (a.more) *reinterpret_cast<float4 *>(p) = v;                            // uniform
        else __builtin_nontemporal_store((f32x4){v.x, v.y, v.z, v.w}, reinterpret_cast<f32x4 *>(p));
    };
    if (!ADD)                                                 // rows no token points at
        for (int q = tid; q < S * 8; q += MWG) {
            const int c = q >> 3;
            if (off[c + 1] == off[c])
                *reinterpret_cast<float4 *>(a.out + ((size_t)t * a.S + c) * a.Do + (size_t)slice * SC + (q & 7) * 4) =
                    make_float4(0.f, 0.f, 0.f, 0.f);
        }

    const int n0 = off[0], n8 = off[S] - n0;
    const int s_lo = n0 + (int)((int64_t)wave * n8 / MWAVES), s_hi = n0 + (int)((int64_t)(wave + 1) * n8 / MWAVES);
    if (s_lo < s_hi) {
        // the bucket holding step s_lo: the last c with off[c] <= s_lo
        int lo = 0, hi = S;                                   // invariant: off[lo] <= s_lo < off[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (off[mid] <= s_lo) lo = mid; else hi = mid;
        }
        int cur = __builtin_amdgcn_readfirstlane(lo);
        int next_b = __builtin_amdgcn_readfirstlane(off[cur + 1]);
        bool head = off[cur] < s_lo;                          // the bucket began in an earlier piece
        const uint2 *pp = a.pairs + (size_t)t * a.stride;
        const float *gcol = a.g + (size_t)slice * SC * (size_t(a.last_token) + 1) + j * 4;
        const int64_t last_entry = (int64_t)s_hi * 8 - 1;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);

        auto flush = [&](bool continues) {
            const float4 v = sum_groups(acc);
            if (head) {
                if (lane < 8) *reinterpret_cast<float4 *>(slot + (wave * 2 + 0) * SC + j * 4) = v;
                if (lane == 0) { flag[wave * 4 + 0] = cur; flag[wave * 4 + 1] = continues ? 0 : 1; }
            } else if (continues) {
                if (lane < 8) *reinterpret_cast<float4 *>(slot + (wave * 2 + 1) * SC + j * 4) = v;
                if (lane == 0) flag[wave * 4 + 2] = cur;
            } else if (lane < 8) {
                if (ADD) *reinterpret_cast<float4 *>(row_s + cur * SC + j * 4) = v;
                else store_row(orow + (size_t)cur * a.Do, v);
            }
            head = false;
            acc = make_float4(0.f, 0.f, 0.f, 0.f);
        };

        uint2 pr = pp[min((int64_t)s_lo * 8 + lane, last_entry)];
        for (int step0 = s_lo; step0 < s_hi; step0 += U) {
            float4 gv[U];
            float sc[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const unsigned tok = min(__shfl(pr.x, u * 8 + grp), a.last_token);
                sc[u] = __uint_as_float(__shfl(pr.y, u * 8 + grp));
                gv[u] = *reinterpret_cast<const float4 *>(gcol + (size_t)tok * SC);
            }
            if (step0 + U < s_hi) pr = pp[min((int64_t)(step0 + U) * 8 + lane, last_entry)];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int step = step0 + u;
                if (step < s_hi) {                            // uniform
                    if (step == next_b) {                     // uniform: the bucket ended with the step before
                        flush(false);
                        do {
                            ++cur;
                            next_b = __builtin_amdgcn_readfirstlane(off[cur + 1]);
                        } while (next_b == step && cur < S - 1);   // skip codes without tokens
                    }
                    acc.x = fmaf(sc[u], gv[u].x, acc.x);
                    acc.y = fmaf(sc[u], gv[u].y, acc.y);
                    acc.z = fmaf(sc[u], gv[u].z, acc.z);
                    acc.w = fmaf(sc[u], gv[u].w, acc.w);
                }
            }
        }
        flush(next_b > s_hi);
    }
    __syncthreads();

    // buckets cut by piece boundaries: add their parts in order
    if (tid < 8) {
        float4 pend = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int w = 0; w < MWAVES; ++w) {
            const int hc = flag[w * 4 + 0];
            if (hc >= 0) {
                pend = add4(pend, *reinterpret_cast<const float4 *>(slot + (w * 2 + 0) * SC + j * 4));
                if (flag[w * 4 + 1] == 1) {
                    *reinterpret_cast<float4 *>(ADD ? row_s + hc * SC + j * 4 : orow + (size_t)hc * a.Do) = pend;
                    pend = make_float4(0.f, 0.f, 0.f, 0.f);
                }
            }
            if (flag[w * 4 + 2] >= 0) pend = *reinterpret_cast<const float4 *>(slot + (w * 2 + 1) * SC + j * 4);
        }
    }
    if constexpr (ADD) {
        __syncthreads();
        constexpr int DEPTH = 8;
        float *const first = a.out + (size_t)t * a.S * a.Do + (size_t)slice * SC;
        for (int q0 = tid; q0 < S * 8; q0 += MWG * DEPTH) {
            float4 v[DEPTH];
            bool live[DEPTH];
#pragma unroll
            for (int i = 0; i < DEPTH; ++i) {
                const int q = q0 + i * MWG, row = min(q >> 3, S - 1);
                live[i] = q < S * 8 && off[row + 1] > off[row];          // rows no token points at stay as they are
                if (live[i]) v[i] = *reinterpret_cast<const float4 *>(first + (size_t)row * a.Do + (q & 7) * 4);
            }
#pragma unroll
            for (int i = 0; i < DEPTH; ++i) {
                const int q = q0 + i * MWG;
                if (live[i])
                    store_row(first + (size_t)(q >> 3) * a.Do + (q & 7) * 4, add4(v[i], *reinterpret_cast<const float4 *>(row_s + q * 4)));
            }
        }
    }
}

// one workgroup per (table of a.S rows, slice)
int launch_sorted(SortedArgs a, hipStream_t st) {
    const int64_t per_xcd = (int64_t)((a.nslices + XCDS - 1) / XCDS) * a.T;
    const size_t lds = (((a.S + 1 + 3) & ~3) + MWAVES * 4) * sizeof(int) + size_t(MWAVES) * 2 * SC * sizeof(float);
    const dim3 grid((unsigned)(per_xcd * XCDS));
    if (a.accumulate) {
        const size_t add_lds = lds + size_t(a.S) * SC * sizeof(float);
        static LdsGrant granted;
        if (add_lds > 65000 && !lffn_grant_dynamic_lds(reinterpret_cast<const void *>(lookup_scatter_sorted_kernel<true>), add_lds, granted))
            return LFFN_ERR_LAUNCH;
        hipLaunchKernelGGL(lookup_scatter_sorted_kernel<true>, grid, dim3(MWG), add_lds, st, a);
    } else {
        hipLaunchKernelGGL(lookup_scatter_sorted_kernel<false>, grid, dim3(MWG), lds, st, a);
    }
    return lffn_launch_status();
}

inline int64_t pair_stride(int64_t B, int64_t S) { return ((B + 7) & ~int64_t(7)) + 8 * S; }

inline bool sorted_supported(int64_t B, int64_t T, int64_t S, int64_t Do) {
    return B >= 1 && T >= 1 && lffn_is_pow2(S) && S <= MAX_S && Do % SC == 0 && Do <= (1 << 20) &&
           B <= (int64_t(1) << 31) - 1 && T <= (1 << 20) && T * ((Do / SC + XCDS - 1) / XCDS) * XCDS <= 0x7fffffff;
}

inline int64_t pack_workgroups(int64_t Bc) { return (Bc + 1 + PACK_TOKENS - 1) / PACK_TOKENS; }
inline int64_t round16(int64_t v) { return (v + 15) & ~int64_t(15); }
inline int64_t padded_tokens(int64_t B) { return (B + 63) & ~int64_t(63); }

// Tokens are taken CHUNK at a time (later chunks add to the result of the earlier ones): a
// 32-column slice of 16384 rows of g is 2 MB and stays in an XCD's 4 MB L2 while the
// workgroups of that XCD walk it in 128 different orders; twice that no longer does.
constexpr int64_t CHUNK = 16384;

struct Workspace {
    int64_t pairs, off8, code_t, score_t, g_packed, total;    // byte offsets
};

inline Workspace workspace_layout(int64_t B, int64_t T, int64_t S, int64_t Do) {
    Workspace w{};
    const int64_t Bc = B < CHUNK ? B : CHUNK, Bp = padded_tokens(Bc);
    w.pairs = 0;
    w.off8 = w.pairs + T * pair_stride(Bc, S) * 8;
    w.code_t = w.off8 + round16(T * (S + 1) * 4);
    w.score_t = w.code_t + round16(T * Bp * 2);
    w.g_packed = w.score_t + round16(T * Bp * 4);
    w.total = w.g_packed + round16((Bc + 1) * Do * 4);
    return w;
}

}  // namespace

extern "C" int lffn_lookup_scatter_workspace_bytes(int64_t B, int64_t T, int64_t S, int64_t Do, int64_t *bytes) {
    LFFN_REQUIRE(bytes, LFFN_ERR_BAD_ARG);
    *bytes = sorted_supported(B, T, S, Do) ? workspace_layout(B, T, S, Do).total : 0;
    return LFFN_OK;
}

namespace {

// The sorted scatter over chunks of CHUNK tokens and, when grad_score is given, the score gradient of each
// chunk from the same slice-major copy of g the scatter reads (lookup_prep_kernel writes it once per chunk).
// grad_tables may be null (score gradient only).
int sorted_backward(const int32_t *code, const float *score, const float *g, const float *tables, float *grad_score,
                    float *grad_tables, float *sums, void *workspace, int64_t workspace_bytes, int64_t B, int64_t T, int64_t S,
                    int64_t Do, int32_t accumulate, void *stream) {
    const Workspace w = workspace_layout(B, T, S, Do);
    LFFN_REQUIRE(workspace_bytes >= w.total, LFFN_ERR_BAD_ARG);
    hipStream_t st = static_cast<hipStream_t>(stream);
    char *base = static_cast<char *>(workspace);
    uint2 *pairs = reinterpret_cast<uint2 *>(base + w.pairs);
    int32_t *off8 = reinterpret_cast<int32_t *>(base + w.off8);

    for (int64_t c0 = 0; c0 < B; c0 += CHUNK) {
        const int64_t Bc = B - c0 < CHUNK ? B - c0 : CHUNK;
        const int64_t stride = pair_stride(Bc, S), Bp = padded_tokens(Bc);

        PrepArgs pa{};
        pa.code = code + c0 * T; pa.score = score + c0 * T; pa.g = g + c0 * Do;
        pa.code_t = reinterpret_cast<uint16_t *>(base + w.code_t);
        pa.score_t = reinterpret_cast<float *>(base + w.score_t);
        pa.g_packed = reinterpret_cast<float *>(base + w.g_packed);
        pa.B = Bc; pa.Bp = Bp; pa.T = (int)T; pa.S = (int)S; pa.Do = (int)Do;
        pa.sums = sums;
        pa.tiles_t = (int)((T + 63) / 64);
        // (score gradient only: the codes and scores need no transposing or sorting, only g its slice-major copy)
        const int64_t transpose_blocks = grad_tables ? (Bp / 64) * pa.tiles_t : 0;
        const int64_t pack_blocks = pack_workgroups(Bc);
        if (sums) sums += pack_blocks * Do;
        const int64_t nsort = grad_tables ? T : 0;
        LFFN_REQUIRE(transpose_blocks <= 0x7fffffff && nsort + pack_blocks <= 0x7fffffff, LFFN_ERR_UNSUPPORTED);
        int rc = LFFN_OK;
        if (transpose_blocks > 0) {
            hipLaunchKernelGGL(lookup_prep_kernel, dim3((unsigned)transpose_blocks), dim3(256), 0, st, pa);
            rc = lffn_launch_status();
            if (rc != LFFN_OK) return rc;
        }
        SortArgs sa{};
        sa.code = pa.code_t; sa.score = pa.score_t; sa.pairs = pairs; sa.off8 = off8;
        sa.B = Bc; sa.Bp = Bp; sa.stride = stride; sa.T = (int)T; sa.S = (int)S; sa.nbits = lffn_log2(S);
        // histograms and bucket tables, then the sorted list itself (4 + 2 bytes per entry; tokens of a chunk fit 16 bits)
        static_assert(CHUNK < 65536, "tokens of a chunk and the padding's are staged as 16-bit values");
        static_assert(CHUNK <= int64_t(SORT_WG) * SORT_DEPTH, "a wavefront of the sort holds its tokens in registers");
        const size_t tables_lds = (size_t(SORT_WAVES) * S + 2 * S + 4 + 4) * sizeof(int);
        const size_t staged_lds = tables_lds + size_t(stride) * 6 + 16;
        sa.stage = staged_lds <= 160 * 1024 ? 1 : 0;            // 512-row tables: the list goes straight to memory
        size_t sort_lds = nsort ? (sa.stage ? staged_lds : tables_lds) : 0;
        if (pa.sums && sort_lds < SORT_WG * sizeof(float4)) sort_lds = SORT_WG * sizeof(float4);
        static LdsGrant granted;
        if (!lffn_grant_dynamic_lds(reinterpret_cast<const void *>(lookup_sort_pack_kernel), sort_lds, granted))
            return LFFN_ERR_LAUNCH;
        hipLaunchKernelGGL(lookup_sort_pack_kernel, dim3((unsigned)(nsort + pack_blocks)), dim3(SORT_WG), sort_lds, st, sa, pa,
                           (int)nsort);
        rc = lffn_launch_status();
        if (rc != LFFN_OK) return rc;

        if (grad_score) {
            // token b's 32 columns of slice s sit at g_packed + (s * (Bc + 1) + b) * 32
            if (!lffn_internal_lookup_inner_quad_try(pa.code, pa.g_packed, SC, (Bc + 1) * SC, tables, grad_score + c0 * T, Bc, T, S,
                                                     Do, stream, &rc))
                rc = lffn_lookup_inner_f32(pa.code, pa.g, tables, grad_score + c0 * T, Bc, T, S, Do, stream);
            if (rc != LFFN_OK) return rc;
        }
        if (!grad_tables) continue;

        SortedArgs ma{};
        ma.pairs = pairs; ma.off8 = off8; ma.g = pa.g_packed; ma.out = grad_tables; ma.stride = stride; ma.rows = T * S;
        ma.last_token = (unsigned)Bc;
        ma.T = (int)T; ma.S = (int)S; ma.Do = (int)Do; ma.nslices = (int)(Do / SC);
        ma.accumulate = (accumulate || c0 > 0) ? 1 : 0;
        ma.more = c0 + CHUNK < B ? 1 : 0;
        rc = launch_sorted(ma, st);
        if (rc != LFFN_OK) return rc;
    }
    return LFFN_OK;
}

}  // namespace

extern "C" int lffn_lookup_scatter_sorted_f32(const int32_t *code, const float *score, const float *g,
                                              float *grad_tables, void *workspace, int64_t workspace_bytes,
                                              int64_t B, int64_t T, int64_t S, int64_t Do, int32_t accumulate,
                                              void *stream) {
    LFFN_REQUIRE(B >= 0 && T >= 0 && S >= 1 && Do >= 1, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(sorted_supported(B, T, S, Do), LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(code && score && g && grad_tables && workspace, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(grad_tables) && lffn_aligned16(g) && lffn_aligned16(workspace), LFFN_ERR_BAD_ARG);
    return sorted_backward(code, score, g, nullptr, nullptr, grad_tables, nullptr, workspace, workspace_bytes, B, T, S, Do, accumulate,
                           stream);
}

// Both gradients of the layer's gather in one call with one workspace (lffn_lookup_scatter_workspace_bytes):
//   grad_score[b,t]  = < g[b,:], tables[t, code[b,t], :] >           (overwritten)
//   grad_tables[t,s] = sum over b with code[b,t] = s of score[b,t] * g[b,:]   (overwritten, or added to)
// Per chunk of 16384 tokens: one kernel transposes code and score and copies g slice-major, the score-gradient
// kernel and the sorted scatter both read that copy.
extern "C" int lffn_lookup_backward_sums_f32(const int32_t *code, const float *score, const float *g, const float *tables,
                                             float *grad_score, float *grad_tables, float *sums, void *workspace,
                                             int64_t workspace_bytes, int64_t B, int64_t T, int64_t S, int64_t Do,
                                             int32_t accumulate, void *stream) {
    LFFN_REQUIRE(B >= 0 && T >= 0 && S >= 1 && Do >= 1, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(sorted_supported(B, T, S, Do) && Do % 64 == 0, LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(code && g && workspace && (grad_score || grad_tables), LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE((!grad_score || tables) && (!grad_tables || score), LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(g) && lffn_aligned16(workspace) && (!grad_tables || lffn_aligned16(grad_tables)) &&
                     (!tables || lffn_aligned16(tables)) && lffn_aligned16(sums), LFFN_ERR_BAD_ARG);
    return sorted_backward(code, score, g, tables, grad_score, grad_tables, sums, workspace, workspace_bytes, B, T, S, Do,
                           accumulate, stream);
}

extern "C" int lffn_lookup_backward_f32(const int32_t *code, const float *score, const float *g, const float *tables,
                                        float *grad_score, float *grad_tables, void *workspace, int64_t workspace_bytes,
                                        int64_t B, int64_t T, int64_t S, int64_t Do, int32_t accumulate, void *stream) {
    return lffn_lookup_backward_sums_f32(code, score, g, tables, grad_score, grad_tables, nullptr, workspace, workspace_bytes, B, T, S,
                                         Do, accumulate, stream);
}

extern "C" int lffn_lookup_backward_sums_rows(int64_t B, int64_t *rows) {
    LFFN_REQUIRE(rows && B >= 0, LFFN_ERR_BAD_ARG);
    *rows = B / CHUNK * pack_workgroups(CHUNK) + (B % CHUNK ? pack_workgroups(B % CHUNK) : 0);
    return LFFN_OK;
}

// ---------------------------------------------------------------------------
// The same accumulation for flat row numbers (weighted_vector_scatter_add on any index array):
//
//   out[idx[b][i]][:] += w[b][i] * g[b][:]
//
// Fp32 atomics on the output rows run at 79 G/s on this part, one per product: 3.4 ms at 4096 x 128 x 512.  The
// accumulation above needs the (token, weight) pairs listed row by row instead, which takes one integer atomic per pair:
//   rows_rank_kernel    a pair's place among the pairs of its row: the value its atomic add on the row's counter returns, or a
//                       workgroup's one such add for all its pairs of the row
//   rows_claim_kernel   one workgroup per 256 rows (a "table" of the accumulation) scans their padded counts and takes that
//                       much of the list; which table's part comes first does not matter
//   rows_place_kernel   pairs into the list (and a row's padding, which names the zero row, by its first pair); other workgroups copy
//                       g slice-major
// The order inside a row is the order of arrival: sums differ from run to run in their last bit, as they did with
// atomics.
namespace {

constexpr int VT = 256;                 // rows per "table"

struct RowsArgs {
    const int32_t *idx;    // [B, I]
    const float *w;        // [B, I]
    const void *g;         // [B, Dv] fp32 or half
    int32_t *count;        // [tables * VT] pairs per row, then (one word) the list's end in units of eight entries
    int32_t *rank;         // [B * I]
    int32_t *off8;         // [tables, VT + 1]
    int32_t *flags;        // [TABLE_FLAGS] not zero where a row number lies outside its column's table, or null: not looked for
    uint2 *pairs;
    float *g_packed;       // [Dv / SC][B + 1][SC], the last row zero
    int64_t B, n, rows;
    int I, Dv, tables, place_blocks;
};

__device__ __forceinline__ int row_of(const RowsArgs &a, int64_t e) {
    const int64_t raw = a.idx[e], hi = a.rows - 1;
    return (int)(raw < 0 ? 0 : (raw > hi ? hi : raw));
}

// The counters to zero; with flags, what table_form_kernel (gather.hip) leaves there for these row numbers.
__global__ __launch_bounds__(1024) void rows_zero_kernel(RowsArgs a, int64_t n4) {
    __shared__ int s_bad[16];
    const int64_t first = int64_t(blockIdx.x) * 1024 + threadIdx.x, stride = int64_t(gridDim.x) * 1024;
    for (int64_t i = first; i < n4; i += stride) reinterpret_cast<int4 *>(a.count)[i] = make_int4(0, 0, 0, 0);
    if (!a.flags) return;                         // uniform
    int bad = 0, i = (int)(first % a.I);
    const int step = (int)(stride % a.I);
    for (int64_t e = first; e < a.n; e += stride) {
        bad |= (a.idx[e] >> 8) ^ i;
        i += step;
        if (i >= a.I) i -= a.I;
    }
    const unsigned long long m = __ballot(bad != 0);
    if ((threadIdx.x & 63) == 0) s_bad[threadIdx.x >> 6] = m != 0;
    __syncthreads();
    if (threadIdx.x == 0) {
        int any = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) any |= s_bad[w];
        a.flags[blockIdx.x] = any;
    }
}

__global__ __launch_bounds__(256) void rows_rank_kernel(RowsArgs a) {
    const int64_t stride = int64_t(gridDim.x) * 256;
    for (int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x; e < a.n; e += stride) a.rank[e] = atomicAdd(a.count + row_of(a, e), 1);
}

// The same for many tokens.  Row numbers as the layer forms them lie in table i in column i: then a workgroup has RANK_TOKENS tokens of
// RANK_COLS columns, counts them in LDS and takes their places from one add per row.  What bounds it is the adds that return something,
// 24 G/s: 4096 x 128 pairs, 32768 rows, 22 -> 7 us, 16000 x 64 41 -> 9.5, 2500 x 256 27 -> 8.  For other row numbers an add for every pair, in
// their order (in the order of the tables' form, sixteen bytes of a token's at a time, 22 -> 25 us, 45 -> 54).  From RANK_TABLES_TOKENS
// on: at 1024 tokens a row has four pairs in a table, and there is nothing to win.
constexpr int64_t RANK_TABLES_TOKENS = 2048;
constexpr int RANK_TOKENS = 1024, RANK_COLS = 4, RANK_WG = 1024;
__global__ __launch_bounds__(RANK_WG) void rows_rank_tables_kernel(RowsArgs a, int col_groups) {
    __shared__ int place[RANK_COLS * VT];
    constexpr int EACH = RANK_TOKENS * RANK_COLS / RANK_WG;
    if (table_guard_ends(TableGuard{a.flags, 1})) {           // uniform: not in table form
        const int64_t stride = int64_t(gridDim.x) * RANK_WG;
        for (int64_t e0 = int64_t(blockIdx.x) * RANK_WG + threadIdx.x; e0 < a.n; e0 += stride * EACH) {
            int rank[EACH];
#pragma unroll
            for (int k = 0; k < EACH; ++k) rank[k] = e0 + k * stride < a.n ? atomicAdd(a.count + row_of(a, e0 + k * stride), 1) : 0;
#pragma unroll
            for (int k = 0; k < EACH; ++k)
                if (e0 + k * stride < a.n) a.rank[e0 + k * stride] = rank[k];
        }
        return;
    }
    const int c = threadIdx.x % RANK_COLS, col0 = int(blockIdx.x % col_groups) * RANK_COLS, col = col0 + c;
    const int64_t b0 = int64_t(blockIdx.x / col_groups) * RANK_TOKENS + threadIdx.x / RANK_COLS;
    int row[EACH], rank[EACH];
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
        const int64_t b = b0 + k * (RANK_WG / RANK_COLS);
        row[k] = b < a.B && col < a.I ? row_of(a, b * a.I + col) : -1;
    }
    static_assert(RANK_COLS * VT == RANK_WG, "a counter per thread");
    place[threadIdx.x] = 0;
    __syncthreads();
    auto in_table = [&](int k) { return row[k] / VT == col; };            // (-1 / VT == 0, but such a thread writes nothing)
#pragma unroll
    for (int k = 0; k < EACH; ++k)
        if (row[k] >= 0) rank[k] = in_table(k) ? atomicAdd(&place[c * VT + row[k] % VT], 1) : atomicAdd(a.count + row[k], 1);
    __syncthreads();
    const int n = place[threadIdx.x];             // row threadIdx.x % VT of table col0 + threadIdx.x / VT
    if (n > 0) place[threadIdx.x] = atomicAdd(a.count + (size_t)col0 * VT + threadIdx.x, n);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EACH; ++k)
        if (row[k] >= 0)
            a.rank[(b0 + k * (RANK_WG / RANK_COLS)) * a.I + col] = rank[k] + (in_table(k) ? place[c * VT + row[k] % VT] : 0);
}

__global__ __launch_bounds__(VT) void rows_claim_kernel(RowsArgs a) {
    __shared__ int wave_sum_s[VT / 64], base_s;
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int mine = (a.count[t * VT + tid] + 7) >> 3;
    int inc = mine;
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(inc, d);
        if (lane >= d) inc += v;
    }
    if (lane == 63) wave_sum_s[wave] = inc;
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < VT / 64; ++w) {
        before += w < wave ? wave_sum_s[w] : 0;
        total += wave_sum_s[w];
    }
    if (tid == 0) base_s = atomicAdd(a.count + (size_t)a.tables * VT, total);
    __syncthreads();
    int32_t *off = a.off8 + (size_t)t * (VT + 1);
    off[tid] = base_s + before + inc - mine;
    if (tid == 0) off[VT] = base_s + total;
}

__device__ __forceinline__ float4 load4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ float4 load4(const _Float16 *p) {
    typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
    const half4_t h = *reinterpret_cast<const half4_t *>(p);
    return make_float4((float)h.x, (float)h.y, (float)h.z, (float)h.w);
}

template <typename G>
__global__ __launch_bounds__(256) void rows_place_kernel(RowsArgs a) {
    if ((int)blockIdx.x < a.place_blocks) {
        const int64_t stride = int64_t(a.place_blocks) * 256;
        for (int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x; e < a.n; e += stride) {
            const int row = row_of(a, e), rank = a.rank[e];
            const unsigned token = (unsigned)((uint32_t)e / (uint32_t)a.I);
            uint2 *list = a.pairs + (int64_t)a.off8[(row / VT) * (VT + 1) + row % VT] * 8;
            list[rank] = make_uint2(token, __float_as_uint(a.w[e]));
            if (rank == 0) {
                const int c = a.count[row];
                for (int p = c; p < ((c + 7) & ~7); ++p) list[p] = make_uint2((unsigned)a.B, 0u);
            }
        }
        return;
    }
    // four 16-byte pieces of g per thread, zeros past its end
    const int q = a.Dv / 4;
    const int64_t n = a.B * q, first = (int64_t(blockIdx.x) - a.place_blocks) * 1024 + threadIdx.x;
    float4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t e = first + 256 * i;
        v[i] = load4(static_cast<const G *>(a.g) + min(e, n - 1) * 4);
        if (e >= n) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t e = first + 256 * i;
        if (e < n + q) {
            const int64_t b = e / q;
            const int col = (int)(e - b * q) * 4;
            *reinterpret_cast<float4 *>(a.g_packed + ((size_t)(col / SC) * (a.B + 1) + b) * SC + col % SC) = v[i];
        }
    }
}

// The rows' sums where rows have few pairs or none (SPARSE_PAIRS on average or fewer): a wavefront adds up a row at a time over
// all its columns from g as it lies and writes it whole.  The slice-by-slice accumulation above reads every row's list once per 32
// columns, which for rows of a few pairs is most of its time.  All five launches, 64 tokens: 128 tables of 768 columns 55 -> 29 us,
// 512 of 1024 217 -> 125 us (537 MB written: 4.3 TB/s); 8 pairs a row, 2048 tokens of 128 x 512: 92 -> 60 us; 16 pairs a row 128 us
// either way, hence the limit.  A row of more than LONG_ROW pairs goes to the whole workgroup; with half of all pairs on one row a single
// compute unit's reads of g bound it (512 tokens of 128 x 768: 516 us by slices, 1275 so, 3437 by fp32 atomics; with a tenth 288 and 1174).
constexpr int64_t SPARSE_PAIRS = 8;
constexpr int LONG_ROW = 32;
constexpr int ROW_GROUP = 32;                         // rows of a workgroup

// acc += the pairs [i0, n) of a row, 64 at a time with `step` from one 64 to the next: a pair per lane, read from there
template <typename G, int NC, int U>
__device__ __forceinline__ void add_pairs(float4 (&acc)[NC], const G *g, const uint2 *list, int i0, int n, int step, int Dv, int col0,
                                          int lane) {
    for (int base = i0; base < n; base += step) {
        const int m = min(64, n - base);
        const uint2 mine = list[base + min(lane, m - 1)];
        for (int k = 0; k < m; k += U) {
            float4 v[U][NC];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const G *p = g + (size_t)(unsigned)__builtin_amdgcn_readlane((int)mine.x, min(k + u, m - 1)) * Dv;
#pragma unroll
                for (int c = 0; c < NC; ++c) v[u][c] = load4(p + (col0 + 256 * c < Dv ? col0 + 256 * c : 0));
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k + u < m) {                              // uniform
                    const float s = __int_as_float(__builtin_amdgcn_readlane((int)mine.y, k + u));
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        acc[c].x = fmaf(s, v[u][c].x, acc[c].x); acc[c].y = fmaf(s, v[u][c].y, acc[c].y);
                        acc[c].z = fmaf(s, v[u][c].z, acc[c].z); acc[c].w = fmaf(s, v[u][c].w, acc[c].w);
                    }
                }
        }
    }
}

template <typename G, int NC>
__global__ __launch_bounds__(256) void rows_sum_kernel(RowsArgs a, float *out, int accumulate, int past_caches) {
    __shared__ float4 part[4][NC][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t first = int64_t(blockIdx.x) * ROW_GROUP;
    const int nrows = (int)min<int64_t>(ROW_GROUP, a.rows - first);
    const G *g = static_cast<const G *>(a.g);
    // counts and list positions of the workgroup's rows, a row per lane
    const int64_t my_row = first + min(lane, nrows - 1);
    const int my_count = a.count[my_row], my_off = a.off8[(my_row / VT) * (VT + 1) + my_row % VT];
    auto list_of = [&](int r) { return a.pairs + (int64_t)__builtin_amdgcn_readlane(my_off, r) * 8; };
    auto store = [&](int r, int col, float4 v) {
        float4 *dst = reinterpret_cast<float4 *>(out + (first + r) * a.Dv + col);
        if (accumulate) {
            const float4 old = *dst;
            v.x += old.x; v.y += old.y; v.z += old.z; v.w += old.w;
        }
        if (past_caches) __builtin_nontemporal_store((f32x4){v.x, v.y, v.z, v.w}, reinterpret_cast<f32x4 *>(dst));      // uniform
        else *dst = v;
    };
    for (int col0 = 4 * lane; col0 - 4 * lane < a.Dv; col0 += 256 * NC) {
        for (int r = wave; r < nrows; r += 4) {
            const int n = __builtin_amdgcn_readlane(my_count, r);
            if (n > LONG_ROW) continue;
            float4 acc[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[c] = make_float4(0.f, 0.f, 0.f, 0.f);
            add_pairs<G, NC, 4>(acc, g, list_of(r), 0, n, 64, a.Dv, col0, lane);
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (col0 + 256 * c < a.Dv) store(r, col0 + 256 * c, acc[c]);
        }
        for (int r = 0; r < nrows; ++r) {                     // (the counts are the same for every wavefront)
            const int n = __builtin_amdgcn_readlane(my_count, r);
            if (n <= LONG_ROW) continue;
            float4 acc[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[c] = make_float4(0.f, 0.f, 0.f, 0.f);
            add_pairs<G, NC, 8>(acc, g, list_of(r), 64 * wave, n, 256, a.Dv, col0, lane);
#pragma unroll
            for (int c = 0; c < NC; ++c) part[wave][c][lane] = acc[c];
            __syncthreads();
            if (wave == 0) {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    float4 v = part[0][c][lane];
#pragma unroll
                    for (int w = 1; w < 4; ++w) {
                        const float4 q = part[w][c][lane];
                        v.x += q.x; v.y += q.y; v.z += q.z; v.w += q.w;
                    }
                    if (col0 + 256 * c < a.Dv) store(r, col0 + 256 * c, v);
                }
            }
            __syncthreads();
        }
    }
}

template <typename G>
int launch_rows_sum(const RowsArgs &a, float *out, int accumulate, hipStream_t st) {
    const dim3 grid((unsigned)((a.rows + ROW_GROUP - 1) / ROW_GROUP));
    const int past_caches = lffn_rows_written_past_caches(a.rows, a.Dv, sizeof(G) == 2);
    switch ((a.Dv + 255) / 256) {
        case 1: hipLaunchKernelGGL((rows_sum_kernel<G, 1>), grid, dim3(256), 0, st, a, out, accumulate, past_caches); break;
        case 2: hipLaunchKernelGGL((rows_sum_kernel<G, 2>), grid, dim3(256), 0, st, a, out, accumulate, past_caches); break;
        case 3: hipLaunchKernelGGL((rows_sum_kernel<G, 3>), grid, dim3(256), 0, st, a, out, accumulate, past_caches); break;
        default: hipLaunchKernelGGL((rows_sum_kernel<G, 4>), grid, dim3(256), 0, st, a, out, accumulate, past_caches); break;
    }
    return lffn_launch_status();
}

struct RowsWorkspace {
    int64_t count, rank, off8, pairs, g_packed, flags, total;
};

// Worth it from 3e6 products on (five launches, about 30 us of them whatever the size, against 79 G atomics/s; forward and backward at 512
// tokens of 32 x 256, 4e6 products: fp32 75 -> 71 us, half 155 -> 99; at 128 x 512, 64 tokens 104 -> 73 and 219 -> 99) and while
// the list that every slice reads is in proportion: at least one pair for every four rows of the output.
bool rows_supported(int64_t B, int64_t I, int64_t rows, int64_t Dv) {
    if (B < 1 || I < 1 || rows < 1 || Dv < SC || Dv % SC != 0 || Dv > (1 << 20)) return false;
    const int64_t Bc = B < CHUNK ? B : CHUNK, tables = (rows + VT - 1) / VT;
    return Bc * I < (int64_t(1) << 31) - 8 * 256 && rows <= (int64_t(1) << 30) && B * I * 4 >= rows &&
           double(B) * double(I) * double(Dv) >= 3e6 && tables * ((Dv / SC + XCDS - 1) / XCDS) * XCDS <= 0x7fffffff &&
           (Bc + 1) * Dv / 1024 < (int64_t(1) << 30);
}

RowsWorkspace rows_layout(int64_t B, int64_t I, int64_t rows, int64_t Dv) {
    RowsWorkspace w{};
    const int64_t Bc = B < CHUNK ? B : CHUNK, tables = (rows + VT - 1) / VT, n = Bc * I;
    w.count = 0;
    w.rank = round16((tables * VT + 1) * 4);
    w.off8 = w.rank + round16(n * 4);
    w.pairs = w.off8 + round16(tables * (VT + 1) * 4);
    w.g_packed = w.pairs + (n + 7 * (n < rows ? n : rows)) * 8 + 8;
    w.g_packed = round16(w.g_packed);
    w.flags = w.g_packed + (Bc + 1) * Dv * 4;               // (a multiple of 128)
    w.total = w.flags + TABLE_FLAGS * 4;
    return w;
}

}  // namespace

extern "C" int lffn_scatter_rows_workspace_bytes(int64_t B, int64_t I, int64_t out_size, int64_t Dv, int64_t *bytes) {
    LFFN_REQUIRE(bytes, LFFN_ERR_BAD_ARG);
    *bytes = rows_supported(B, I, out_size, Dv) ? rows_layout(B, I, out_size, Dv).total : 0;
    return LFFN_OK;
}

extern "C" int lffn_scatter_rows(const int32_t *idx, const void *g, const float *w, float *out, void *workspace,
                                 int64_t workspace_bytes, int64_t B, int64_t I, int64_t out_size, int64_t Dv, int32_t g_format,
                                 int32_t accumulate, void *stream) {
    LFFN_REQUIRE(g_format == LFFN_ROWS_F32 || g_format == LFFN_ROWS_F16, LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(rows_supported(B, I, out_size, Dv), LFFN_ERR_UNSUPPORTED);
    LFFN_REQUIRE(idx && g && w && out && workspace, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(g) && lffn_aligned16(out) && lffn_aligned16(workspace), LFFN_ERR_BAD_ARG);
    const RowsWorkspace l = rows_layout(B, I, out_size, Dv);
    LFFN_REQUIRE(workspace_bytes >= l.total, LFFN_ERR_BAD_ARG);
    hipStream_t st = static_cast<hipStream_t>(stream);
    char *base = static_cast<char *>(workspace);
    for (int64_t c0 = 0; c0 < B; c0 += CHUNK) {              // as above: a slice of g has to stay in an XCD's L2
        RowsArgs a{};
        a.B = B - c0 < CHUNK ? B - c0 : CHUNK;
        a.idx = idx + c0 * I; a.w = w + c0 * I;
        a.g = static_cast<const char *>(g) + c0 * Dv * (g_format == LFFN_ROWS_F16 ? 2 : 4);
        a.count = reinterpret_cast<int32_t *>(base + l.count);
        a.rank = reinterpret_cast<int32_t *>(base + l.rank);
        a.off8 = reinterpret_cast<int32_t *>(base + l.off8);
        a.pairs = reinterpret_cast<uint2 *>(base + l.pairs);
        a.g_packed = reinterpret_cast<float *>(base + l.g_packed);
        a.n = a.B * I; a.rows = out_size; a.I = (int)I; a.Dv = (int)Dv;
        a.tables = (int)((out_size + VT - 1) / VT);
        const int64_t blocks = (a.n + 255) / 256;
        a.place_blocks = (int)(blocks < 4096 ? blocks : 4096);
        const bool sparse = a.n <= SPARSE_PAIRS * out_size;      // (no slice-major copy of g)
        const int64_t pack_blocks = sparse ? 0 : ((a.B + 1) * (Dv / 4) + 1023) / 1024;
        const int64_t zero4 = l.rank / 16;                      // the counters and the list's end
        a.flags = a.B >= RANK_TABLES_TOKENS ? reinterpret_cast<int32_t *>(base + l.flags) : nullptr;
        const int64_t zero_blocks = (zero4 + 1023) / 1024;
        hipLaunchKernelGGL(rows_zero_kernel, dim3((unsigned)(a.flags || zero_blocks > TABLE_FLAGS ? TABLE_FLAGS : zero_blocks)), dim3(1024), 0, st, a,
                           zero4);
        if (a.flags) {
            const int col_groups = (int)((I + RANK_COLS - 1) / RANK_COLS);      // (workgroups: fewer than pairs)
            hipLaunchKernelGGL(rows_rank_tables_kernel, dim3((unsigned)((a.B + RANK_TOKENS - 1) / RANK_TOKENS * col_groups)), dim3(RANK_WG), 0,
                               st, a, col_groups);
        } else {
            hipLaunchKernelGGL(rows_rank_kernel, dim3((unsigned)a.place_blocks), dim3(256), 0, st, a);
        }
        hipLaunchKernelGGL(rows_claim_kernel, dim3((unsigned)a.tables), dim3(VT), 0, st, a);
        const dim3 grid((unsigned)(a.place_blocks + pack_blocks));
        if (g_format == LFFN_ROWS_F16) hipLaunchKernelGGL(rows_place_kernel<_Float16>, grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL(rows_place_kernel<float>, grid, dim3(256), 0, st, a);
        int rc = lffn_launch_status();
        if (rc != LFFN_OK) return rc;
        if (sparse) {
            const int add = (accumulate || c0 > 0) ? 1 : 0;
            rc = g_format == LFFN_ROWS_F16 ? launch_rows_sum<_Float16>(a, out, add, st) : launch_rows_sum<float>(a, out, add, st);
            if (rc != LFFN_OK) return rc;
            continue;
        }
        SortedArgs ma{};
        ma.pairs = a.pairs; ma.off8 = a.off8; ma.g = a.g_packed; ma.out = out; ma.stride = 0; ma.rows = out_size;
        ma.last_token = (unsigned)a.B;
        ma.T = a.tables; ma.S = VT; ma.Do = (int)Dv; ma.nslices = (int)(Dv / SC);
        ma.accumulate = (accumulate || c0 > 0) ? 1 : 0;
        ma.more = c0 + CHUNK < B ? 1 : 0;
        rc = launch_sorted(ma, st);
        if (rc != LFFN_OK) return rc;
    }
    return LFFN_OK;
}
