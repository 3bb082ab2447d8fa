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
// copy of g to a slice-major layout [ceil(Do / 64)][B + 1][64] (in which the 256-byte row pieces of a slice
// are contiguous: with rows 4*Do bytes apart the pieces of one slice fall on a part of the L2
// channels) is pure memory traffic and depends on nothing: its workgroups fill the rest of the
// chip while the sort runs (23 + 25 us as two launches at 16384 tokens x 128 tables x 768).
//
// The sort: one workgroup per table sorts the tokens by their code for that
// table (a stable counting sort: per-wavefront histograms over contiguous token ranges,
// ranks inside a 64-token batch from ballots over the code bits) and writes (token, score)
// pairs bucket by bucket: into LDS first (a 16-bit token and a score per entry, 98 KB at most), from where the list goes to memory in
// whole lines; written straight from the ranks, every wavefront store was 64 separate 8-byte requests.  More than SUB tokens are two
// lists, each sorted by half of the wavefronts (a workgroup per list: 28 -> 34 us at 16384 tokens).  Nothing is padded.
//
// lookup_scatter_sorted_kernel: one workgroup per (table, 64-column slice), or more of them, each for some of the table's rows, whose entries are a part of the
// table's lists: more than 256 rows leave no room in LDS for a second workgroup on a compute unit, and few tables of few columns would leave compute
// units idle (launch_sorted_form).  What bounds it is the compute unit's vector memory path: every
// pair's 256 bytes of g come out of the L2, random rows of any length at 33 TB/s where nothing else is asked for (57 bytes a clock of a
// compute unit), and it does so with the least beside them:
//   * 64 columns, so that a list is read once per 256 bytes of a row.  A slice of 16384 rows is then 4 MB, as much as an XCD's L2, and
//     its tokens are two lists whose rows are walked one after the other (as one list 275 -> 296 us at 16384 x 128 x 768); four lists
//     cost more bucket ends than they give (300).
//   * A list is cut into pieces of the same cost, one per wavefront, a bucket's end taken as END_COST entries: with the same number of entries, the
//     wavefront with the shortest buckets was waited for by all.  us, same entries -> same cost, codes by Zipf's law from row 0 on: 16384 x 128 x 768 349 -> 301,
//     16384 x 512 x 1024 1879 -> 1577, 4096 x 128 x 768 150 -> 101, 32768 x 32 x 512 249 -> 189; the same law, rows shuffled: 302 -> 298, 1555 -> 1530, 106 -> 97, 193 -> 177;
//     spread evenly: 292 -> 293, 1521 -> 1530, 95 -> 95, 170 -> 170.  (END_COST 4: 308, 1598, 109, 204 and 300, 1533, 98, 182; 8: 301, 1555, 98, 178 but evenly 294, 1535.)  A
//     wavefront takes four entries a step: lane group q = lane / 16 has entry q and its sixteen lanes the 256 bytes.  Entries
//     reach their lanes by DPP (through LDS, two permutes a step, it had 12.7 vector instructions a kilobyte for 9.3), and eight steps' loads are in flight all the
//     time: the register of a step that is done is loaded for the step eight on.
//   * A bucket ends between any two entries: then a step's lane groups are split by selects.  (Lists padded to whole steps cost 5 % of the
//     reads at 64 pairs a row and 18 % at 16.)
//   * A bucket's sum goes to LDS, where its row holds what earlier lists gave, and the rows are written at the end, whole: no store sits
//     among the loads (the counter that loads are waited for with counts stores too), no zero-fill and no atomics.  Buckets cut by
//     a piece boundary go to slots, and the wavefront in whose piece one ends adds its parts in order.  The sum order is fixed
//     (run-to-run reproducible), and eight partial sums of a bucket (four lane groups, even and odd steps) keep its error where it was.
// Eight wavefronts a workgroup, two of them a compute unit for their LDS; 12 or 16 wavefronts are slower (285, 310 us).  All launches,
// before (padded lists of 16384 tokens, 32 columns, rows stored as they end) -> now, sums in fp32, codes spread evenly, by Zipf's law in any order of the rows:
// 16384 x 128 x 768 317 -> 294 us, 322 -> 299; x 512 223 -> 204, 229 -> 206; 32768 x 128 x 512 445 -> 413, 457 -> 420; 8192 x 256 x 768 336 -> 279, 348 -> 283;
// 16384 x 512 x 1024 1532 -> 1524, 1545 -> 1529; of 512 rows 16384 x 128 x 768 348 -> 335, 369 -> 369; sums in doubles (in fp32 before) 4096 x 128 x 768 123 -> 95, 137 -> 97.  What is left at 16384 x 128 x 768, taken
// apart: without bucket ends -12 us, with lists from the L2 -28, rows from the L1 -47, all three 228 of 285, of which 25 to 35 are starts and ends of workgroups in step
// with each other.  Fetching the lists' lines or the next list's rows ahead through the scalar cache gives nothing, nor does a
// workgroup that stays for several slices.
#include "lffn_common.h"

#include <climits>

namespace {

constexpr int SORT_WG = 1024;
constexpr int SORT_WAVES = SORT_WG / 64;
constexpr int MAX_S = 512;
constexpr int XCDS = 8, COMPUTE_UNITS = 256;
constexpr int64_t CHUNK = LFFN_SCATTER_CHUNK_TOKENS;    // tokens of a launch: 16384
constexpr int64_t SUB = 8192;       // tokens whose pairs are sorted together, at most (all of a launch for sums in doubles)
constexpr int SORT_DEPTH = CHUNK / SORT_WG;    // batches of 64 tokens whose loads are in flight per wavefront

constexpr int SC = 64;               // columns per slice: 16 lanes x float4
constexpr int WAVES = 8;            // of the sums' workgroup
constexpr int MWG = WAVES * 64;
constexpr int RING = 8;              // loads in flight per wavefront
constexpr int MAX_BLOCK_ROWS = 256;  // rows of a table that lie together in LDS
constexpr int END_COST = 6;          // what a bucket's end costs, in entries
constexpr int CUTS = 2 * WAVES + 2;  // words about a list's pieces

struct PrepArgs {
    const int32_t *code;   // [B, T]
    const float *score;    // [B, T]
    const float *g;        // [B, Do]
    uint16_t *code_t;      // [T, Bp]
    float *score_t;        // [T, Bp]
    float *g_packed;       // [ceil(Do / SC)][B + 1][SC], the last row zero
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

// PACK_TOKENS rows of g, copied to the slice-major layout (workgroup `blk` of the copy); row B is zeros.  A thread has four
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
    uint2 *pairs;          // [subs, T, stride] (token, counted from the list's first on, and score bits)
    int32_t *off;          // [subs, T, S + 2] bucket starts in a list and its length; where the list starts, in units of eight entries
    int64_t B, Bp, sub_len, stride;      // list `sub` has the tokens [sub * sub_len, (sub + 1) * sub_len)
    int T, S, nbits, subs;
};

// The lists of table t: one, or two, to each half of the wavefronts one.
__device__ __forceinline__ void sort_table(const SortArgs &a, const int t) {
    extern __shared__ int sm[];
    const int S = a.S, waves = SORT_WAVES / a.subs;      // of a list
    int *hist = sm;                    // [SORT_WAVES][S]: counts, then running write positions
    int *start = hist + SORT_WAVES * S;                                        // [subs][S] bucket starts (entries)
    float *sc_s = reinterpret_cast<float *>(start + a.subs * S);                // [subs * stride] scores of the sorted lists
    unsigned short *tok_s = reinterpret_cast<unsigned short *>(sc_s + a.subs * a.stride);   // [subs * stride] tokens

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sub = wave / waves;
    const uint16_t *code = a.code + (size_t)t * a.Bp;
    const float *score = a.score + (size_t)t * a.Bp;
    for (int q = tid; q < SORT_WAVES * S; q += SORT_WG) hist[q] = 0;
    __syncthreads();

    // A wavefront takes up to SORT_DEPTH batches of 64 consecutive tokens (a list's length is a multiple of its wavefronts').
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
    for (int i = tid; i < a.subs * S; i += SORT_WG) {
        const int w0 = i / S * waves, c = i % S;
        int sum = 0;
        for (int w = w0; w < w0 + waves; ++w) {
            const int v = hist[w * S + c];
            hist[w * S + c] = sum;
            sum += v;
        }
        start[i] = sum;
    }
    __syncthreads();
    if (wave % waves == 0) {           // exclusive scan of the counts
        int *mine = start + sub * S;
        const int per_lane = (S + 63) / 64;
        int loc = 0;
        for (int k = 0; k < per_lane; ++k) {
            const int i = lane * per_lane + k;
            if (i < S) loc += mine[i];
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
                const int v = mine[i];
                mine[i] = run;
                run += v;
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < a.subs * S; i += SORT_WG) {
        const int q = i / S, c = i % S, o = start[i];
        a.off[((size_t)q * a.T + t) * (S + 2) + c] = o;
        for (int w = q * waves; w < (q + 1) * waves; ++w) hist[w * S + c] += q * (int)a.stride + o;
    }
    if (tid < a.subs) {
        const int64_t list = (int64_t)tid * a.T + t;
        a.off[list * (S + 2) + S] = (int)min(a.B - tid * a.sub_len, a.sub_len);
        a.off[list * (S + 2) + S + 1] = (int)(list * a.stride / 8);
    }
    __syncthreads();

#pragma unroll
    for (int k = 0; k < SORT_DEPTH; ++k) {
        if (lo + 64 * k >= hi) continue;                         // uniform
        if (cv[k] >= 0) {
            const int c = cv[k], rank = rk[k] & 0xff, cnt = rk[k] >> 8;
            const int base = myh[c];                              // all lanes of a code read before its last lane writes
            tok_s[base + rank] = (unsigned short)(lo - sub * a.sub_len + 64 * k + lane);
            sc_s[base + rank] = sv[k];
            if (rank == cnt - 1) myh[c] = base + cnt;
        }
    }
    __syncthreads();
    for (int q = 0; q < a.subs; ++q) {
        const int n = (int)min(a.B - q * a.sub_len, a.sub_len), first = q * (int)a.stride;
        uint2 *out = a.pairs + ((int64_t)q * a.T + t) * a.stride;
        for (int i = tid; i < n; i += SORT_WG) out[i] = make_uint2((unsigned)tok_s[first + i], __float_as_uint(sc_s[first + i]));
    }
}

// workgroups [0, nsort): the sort of one table each; the others: PACK_TOKENS rows of the copy of g each
__global__ __launch_bounds__(SORT_WG) void lookup_sort_pack_kernel(SortArgs sa, PrepArgs pa, int nsort) {
    if ((int)blockIdx.x < nsort) sort_table(sa, (int)blockIdx.x);      // uniform over the workgroup
    else pack_rows(pa, int64_t(blockIdx.x) - nsort);
}

struct SortedArgs {
    const uint2 *pairs;
    const int32_t *off;    // [subs, T, S + 2] as in SortArgs
    const float *g;        // [nslices][B + 1][SC], the last row zero
    float *out;            // [rows, Do]; table t's rows from t * S on
    int64_t rows;
    int B, sub_len;        // tokens, CHUNK at most, and those of a list
    int T, S, Do, nslices, subs, per_xcd, accumulate;
    int block_rows, block_bits;       // rows of a table that lie together in LDS: S >> block_bits
    int part_bits;         // and into how many parts their lists are cut, a workgroup each
    int more;              // a later launch adds to these rows
};

__device__ __forceinline__ float4 add4(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

// Sum over the four lane groups of a float4 that every lane holds for its four columns: two values change places with each swap, so that
// both sums take one addition, and a lane ends with one of its four (6 instructions; one value after the other takes 16).  Lane
// 16 r + i has column 4 i + {0, 2, 1, 3}[r].
__device__ __forceinline__ float sum_swapped32(float x, float y) {     // lanes 0-31: x of both halves, 32-63: y
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_swapped16(float x, float y) {     // rows of 16: x of rows 0 and 1, y of both, x of rows 2 and 3, y of both
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_groups(const float (&v)[4]) { return sum_swapped16(sum_swapped32(v[0], v[1]), sum_swapped32(v[2], v[3])); }
// the same of doubles, the two words of each on the same ways
template <bool HALVES>
__device__ __forceinline__ double sum_swapped(double x, double y) {
    const uint64_t a = __double_as_longlong(x), b = __double_as_longlong(y);
    auto swap = [](unsigned p, unsigned q) {
        return HALVES ? __builtin_amdgcn_permlane32_swap(p, q, false, false) : __builtin_amdgcn_permlane16_swap(p, q, false, false);
    };
    const auto lo = swap((unsigned)a, (unsigned)b), hi = swap((unsigned)(a >> 32), (unsigned)(b >> 32));
    return __longlong_as_double((uint64_t)hi[0] << 32 | lo[0]) + __longlong_as_double((uint64_t)hi[1] << 32 | lo[1]);
}
__device__ __forceinline__ double sum_groups(const double (&v)[4]) {
    return sum_swapped<false>(sum_swapped<true>(v[0], v[1]), sum_swapped<true>(v[2], v[3]));
}

// What lane u of a row of sixteen lanes holds, in all of them (a DPP operand of the instruction that uses it).
__device__ __forceinline__ int row_pick(int v, int u) {
#define LFFN_PICK(n) case n: return __builtin_amdgcn_mov_dpp(v, 0x150 + n, 0xF, 0xF, true)
    switch (u) {
        LFFN_PICK(0); LFFN_PICK(1); LFFN_PICK(2); LFFN_PICK(3); LFFN_PICK(4); LFFN_PICK(5); LFFN_PICK(6); LFFN_PICK(7);
        LFFN_PICK(8); LFFN_PICK(9); LFFN_PICK(10); LFFN_PICK(11); LFFN_PICK(12); LFFN_PICK(13); LFFN_PICK(14);
        default: return __builtin_amdgcn_mov_dpp(v, 0x15F, 0xF, 0xF, true);
    }
#undef LFFN_PICK
}

// ADD: the sums are added to what a.out holds.  Sum: float, or double (sums_in_doubles).
template <bool ADD, typename Sum>
__global__ __launch_bounds__(MWG, WAVES / 2) void lookup_scatter_sorted_kernel(SortedArgs a) {
    extern __shared__ float4 lds4[];
    const int R = a.block_rows;
    float *row_s = reinterpret_cast<float *>(lds4);             // [R][SC]: the rows' sums
    Sum *slot = reinterpret_cast<Sum *>(row_s + R * SC);        // [WAVES][2][SC], and where sums go that belong in no slot
    int *flag_s = reinterpret_cast<int *>(slot + (WAVES * 2 + 1) * SC);      // [2][WAVES][4]: head bucket, it closes here, tail bucket
    int *cut_s = flag_s + 2 * WAVES * 4;                        // [2][CUTS]: where pieces begin, the last one's end, the list's first line, rows that cuts fall to
    int *off_s = cut_s + 2 * CUTS;                              // [2][R + 1]

    // neighbouring tables of a slice on one XCD
    const int unit = (int)(blockIdx.x % XCDS) * a.per_xcd + (int)(blockIdx.x / XCDS), slice_units = a.T << (a.block_bits + a.part_bits);
    if (unit >= slice_units * a.nslices) return;              // uniform over the workgroup
    const int slice = unit / slice_units, block = unit - slice * slice_units >> a.part_bits, part = unit & ((1 << a.part_bits) - 1);
    const int t = block >> a.block_bits, row0 = (block - (t << a.block_bits)) * R;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = lane >> 4, i16 = lane & 15;
    const int my_col = i16 * 4 + (lane >> 5) + ((lane >> 3) & 2);
    // fp32: a column's place in the LDS as a whole, so that one index serves rows and slots; doubles: in the slots
    const int slot0 = ((sizeof(Sum) == 4 ? R : 0) + wave * 2) * SC + my_col, no_slot = WAVES * 2 * SC + my_col;

    static_assert(MAX_BLOCK_ROWS <= MWG, "a row a thread");
    auto offsets = [&](int sub) { return a.off + ((size_t)sub * a.T + t) * (a.S + 2) + row0; };
    // The rows [r0, r1) of the block are this workgroup's.  Parts are of the same cost, as near as whole rows allow: a row's entries and END_COST for
    // its end.
    int r0 = 0, r1 = R;
    if (a.part_bits > 0) {                                    // uniform
        const int q = min(tid, R - 1);
        int first = END_COST * a.subs * q, next = first + END_COST * a.subs, whole = END_COST * a.subs * R;
        for (int sub = 0; sub < a.subs; ++sub) {
            const int32_t *off = offsets(sub);
            first += off[q] - off[0];
            next += off[q + 1] - off[0];
            whole += off[R] - off[0];
        }
        const int from = part * whole >> a.part_bits, to = (part + 1) * whole >> a.part_bits;
        if (tid < R && first < to && to <= next) flag_s[1] = tid + 1;
        if (part == 0 ? tid == 0 : tid < R && first < from && from <= next) flag_s[0] = part == 0 ? 0 : tid + 1;
        __syncthreads();
        r0 = __builtin_amdgcn_readfirstlane(flag_s[0]);
        r1 = __builtin_amdgcn_readfirstlane(flag_s[1]);
    }
    // A list's offsets: thread q has those of row q, where its bucket starts and ends.  Pieces, too, are of the same cost: else the wavefront with the
    // shortest buckets would be waited for by all.  A piece begins in the row that its share of the cost falls to, on a whole line of pairs.
    int next_off = 0, next_end = 0, list_begin = 0, list_end = 0, list_line = 0;
    auto load_offsets = [&](int sub) {
        const int32_t *off = offsets(sub), *mine = off + min(tid, R - 1);
        next_off = mine[0];
        next_end = mine[1];
        list_begin = off[r0];
        list_end = off[r1];
        list_line = off[a.S + 1 - row0];
    };
    auto keep_offsets = [&](int sub) {
        int *off = off_s + (sub & 1) * (R + 1), *cuts = cut_s + (sub & 1) * CUTS;
        if (tid < R) off[tid] = next_off;
        if (tid == R - 1) off[R] = next_end;
        if (tid >= r0 && tid < r1) {
            const int first = next_off - list_begin + END_COST * (tid - r0), cost = next_end - next_off + END_COST;      // of the row
            const int whole = __builtin_amdgcn_readfirstlane(list_end - list_begin) + END_COST * (r1 - r0);
#pragma unroll
            for (int w = 1; w < WAVES; ++w) {
                const int at = (int)((unsigned)(w * whole) / WAVES) - first;
                if ((unsigned)at < (unsigned)cost) {
                    cuts[w] = max(min(next_off + at, next_end) & ~7, list_begin);
                    cuts[WAVES + 2 + w] = tid;
                }
            }
        }
        if (tid == 0) {
            cuts[0] = list_begin;
            cuts[WAVES] = list_end;
            cuts[WAVES + 1] = list_line;
            cuts[WAVES + 2] = r0;
        }
        if (r0 == r1 && tid > 0 && tid < WAVES) cuts[tid] = list_begin;      // no rows, no entries
    };
    load_offsets(0);
    for (int q = tid; q < R * (SC / 4); q += MWG) lds4[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    keep_offsets(0);
    __syncthreads();

    // What a wavefront knows of its piece of the list at hand, and its first pairs.
    int sub = 0;
    int e_lo, e_hi, cur, first_end, ends, head_bucket, tokens;
    const uint2 *pp;
    uint2 pr0, pr1;
    // The ends of 64 buckets, one a lane, so that nothing waits for LDS at a bucket's end; those that the piece does not reach lie
    // beyond every entry.
    auto load_ends = [&]() {
        int v = off_s[(sub & 1) * (R + 1) + min(first_end + lane, R)];
        v = v < e_hi ? v : INT_MAX;
        asm volatile("" : "+v"(v));                           // (waited for here, not where one is read)
        return v;
    };
    // 64 pairs as they lie, past the piece's end weight 0 and the row of zeros
    auto load_pairs = [&](int e) { return pp[min(e + lane, e_hi - 1)]; };
    auto begin_list = [&]() {
        const int *off = off_s + (sub & 1) * (R + 1);
        const int *cuts = cut_s + (sub & 1) * CUTS + wave;
        e_lo = __builtin_amdgcn_readfirstlane(cuts[0]);
        e_hi = __builtin_amdgcn_readfirstlane(cuts[1]);
        tokens = a.B - sub * a.sub_len;                       // the row of zeros, from the list's first token on
        pp = a.pairs + (int64_t)__builtin_amdgcn_readfirstlane(cuts[WAVES + 1 - wave]) * 8;
        head_bucket = -1;
        if (e_lo >= e_hi) return;                             // uniform
        pr0 = load_pairs(e_lo);
        pr1 = load_pairs(min(e_lo + 64, e_hi - 1));
        // the bucket holding entry e_lo, the last c with off[c] <= e_lo: the row that the cut fell to, a neighbour, or searched for
        cur = __builtin_amdgcn_readfirstlane(cuts[WAVES + 2]);
        int tries = 3;
        for (; tries > 0; --tries) {
            const int from = __builtin_amdgcn_readfirstlane(off[cur]), to = __builtin_amdgcn_readfirstlane(off[cur + 1]);
            if (from <= e_lo && e_lo < to) break;
            cur += from > e_lo ? -1 : 1;
        }
        if (tries == 0) {                                     // uniform
            int lo = r0, hi = r1;                             // invariant: off[lo] <= e_lo < off[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (off[mid] <= e_lo) lo = mid; else hi = mid;
            }
            cur = __builtin_amdgcn_readfirstlane(lo);
        }
        first_end = cur + 1;
        ends = load_ends();
        head_bucket = __builtin_amdgcn_readfirstlane(off[cur] < e_lo ? cur : -1);
    };
    begin_list();

    for (;;) {
        const bool last_list = sub + 1 == a.subs;
        if (!last_list) load_offsets(sub + 1);                // the next list's, on their way while this one is walked
        int *flag = flag_s + (sub & 1) * WAVES * 4;
        int closes = 0, goes_on = 0;
        if (e_lo < e_hi) {
            const int *off = off_s + (sub & 1) * (R + 1);
            int next_b = __builtin_amdgcn_readlane(ends, 0);
            closes = head_bucket >= 0 && __builtin_amdgcn_readfirstlane(off[cur + 1]) <= e_hi ? 1 : 0;
            constexpr int SUMS = sizeof(Sum) == 4 ? 2 : 1;    // the even and the odd steps', so that an fp32 sum is one of eight
            // where the sum of the bucket at hand goes: its row, or, if it began in an earlier piece, this wavefront's first slot.  Doubles,
            // whose rows hold nothing before, are written to both, the row of a cut bucket once more by whoever closes it, others' slot nobody's: a
            // branch here costs 3 to 8 % where codes have Zipf's distribution.
            int dst = head_bucket >= 0 ? slot0 : SUMS == 2 ? cur * SC + my_col : no_slot;
            float before = head_bucket >= 0 ? 0.f : row_s[cur * SC + my_col];      // what the row holds: the sum over earlier lists
            const char *gs = reinterpret_cast<const char *>(a.g + ((size_t)slice * (a.B + 1) + (size_t)sub * a.sub_len) * SC);
            Sum acc[SUMS][4];
            auto clear = [&]() {
#pragma unroll
                for (int e = 0; e < 4 * SUMS; ++e) acc[e >> 2][e & 3] = 0;
            };
            clear();
            auto flush = [&]() {
                if constexpr (SUMS == 2)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[0][e] += acc[1][e];
                const Sum v = sum_groups(acc[0]);
                if constexpr (SUMS == 2) {
                    row_s[dst] = before + v;
                } else {
                    slot[dst] = v;
                    row_s[cur * SC + my_col] = (float)v;
                }
            };
            // Lane i of group q gets the pair that the group takes in step i (loaded so, sixteen lanes would be sixteen lines).
            auto turned = [&](unsigned v) { return __builtin_amdgcn_ds_bpermute((i16 * 4 + grp) * 4, (int)v); };
            // (a launch's tokens: 32 bits hold the offset of a row in the slice)
            auto rows_of = [&](uint2 v, int e) {
                return turned((e + lane < e_hi ? min(v.x, (unsigned)tokens) : (unsigned)tokens) * unsigned(SC * 4));
            };
            auto weights_of = [&](uint2 v, int e) { return turned(e + lane < e_hi ? v.y : 0u); };
            auto load_row = [&](int rows, int u) {
                return *reinterpret_cast<const float4 *>(gs + (unsigned)(row_pick(rows, u) + i16 * 16));
            };
            auto add = [&](int odd, float w, float4 v, bool live) {
                Sum (&to)[4] = acc[odd % SUMS];
                const Sum x = fma((Sum)w, (Sum)v.x, to[0]), y = fma((Sum)w, (Sum)v.y, to[1]), z = fma((Sum)w, (Sum)v.z, to[2]),
                          u = fma((Sum)w, (Sum)v.w, to[3]);
                to[0] = live ? x : to[0];
                to[1] = live ? y : to[1];
                to[2] = live ? z : to[2];
                to[3] = live ? u : to[3];
            };
            // four entries from e on, one per lane group; a bucket may end before any of them
            auto take = [&](int e, int odd, float w, float4 v) {
                if (next_b >= e + 4) {                        // uniform
                    add(odd, w, v, true);
                    return;
                }
                int from = 0;
                do {
                    const int to = next_b - e;
                    add(odd, w, v, grp >= from && grp < to);      // (selected, not branched on: all control flow is the wavefront's)
                    flush();
                    const int end = next_b;
                    do {
                        ++cur;
                        if (cur + 1 - first_end == 64) {
                            first_end = cur + 1;
                            ends = load_ends();
                        }
                        next_b = __builtin_amdgcn_readlane(ends, cur + 1 - first_end);
                    } while (next_b == end);                  // skip codes without tokens
                    dst = SUMS == 2 ? cur * SC + my_col : no_slot;
                    if (SUMS == 2) before = row_s[dst];
                    clear();
                    from = to;
                } while (next_b < e + 4);
                add(odd, w, v, grp >= from);
            };

            int rows = rows_of(pr0, e_lo), w = weights_of(pr0, e_lo);
            float4 gv[RING];
#pragma unroll
            for (int u = 0; u < RING; ++u) gv[u] = load_row(rows, u);
            int e = e_lo;
            for (; e + 64 < e_hi; e += 64) {
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    take(e + 4 * u, u & 1, __int_as_float(row_pick(w, u)), gv[u]);
                    gv[u] = load_row(rows, u + 8);
                }
                rows = rows_of(pr1, e + 64);
                const int w_next = weights_of(pr1, e + 64);
                pr1 = load_pairs(min(e + 128, e_hi - 1));
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    take(e + 32 + 4 * u, u & 1, __int_as_float(row_pick(w, u + 8)), gv[u]);
                    gv[u] = load_row(rows, u);
                }
                w = w_next;
            }
            if (e + 32 < e_hi) {                              // uniform
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    take(e + 4 * u, u & 1, __int_as_float(row_pick(w, u)), gv[u]);
                    gv[u] = load_row(rows, u + 8);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (e + 32 + 4 * u < e_hi) take(e + 32 + 4 * u, u & 1, __int_as_float(row_pick(w, u + 8)), gv[u]);
            } else {
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (e + 4 * u < e_hi) take(e + 4 * u, u & 1, __int_as_float(row_pick(w, u)), gv[u]);
            }
            goes_on = cur != head_bucket && __builtin_amdgcn_readfirstlane(off[cur + 1]) > e_hi ? 1 : 0;      // in the next piece
            dst = goes_on ? slot0 + SC : dst;
            before = goes_on ? 0.f : before;
            flush();
        }
        flag[wave * 4 + 0] = head_bucket;                     // (every lane the same)
        flag[wave * 4 + 1] = closes;
        flag[wave * 4 + 2] = goes_on ? cur : -1;
        if (!last_list) keep_offsets(sub + 1);
        __syncthreads();
        // a bucket cut by piece boundaries: the wavefront in whose piece it ends adds its parts
        if (closes) {                                         // uniform
            Sum sum = slot[wave * 2 * SC + lane];
            for (int k = wave - 1; k >= 0; --k) {
                if (__builtin_amdgcn_readfirstlane(flag[k * 4 + 2]) >= 0) {
                    sum = slot[(k * 2 + 1) * SC + lane] + sum;
                    break;
                }
                if (__builtin_amdgcn_readfirstlane(flag[k * 4 + 0]) >= 0) sum = slot[k * 2 * SC + lane] + sum;
            }
            float &row = row_s[head_bucket * SC + lane];
            if constexpr (sizeof(Sum) == 4) row += sum;
            else row = (float)sum;
        }
        ++sub;
        if (!last_list) begin_list();
        __syncthreads();
        if (last_list) break;
    }

    // Rows that nothing adds to any more go out nontemporally: in the caches they would take the place of g.  Read again next, 32768 x 512,
    // that costs 7 us of 1490.  With a reader behind the pass, unlike the lists and the sums of few pairs (lffn_rows_written_past_caches), it
    // costs no more than it gives: a training step of 2500 tokens and more of 128 to 512 tables takes the same alone and with SGD, clipping
    // or Adam behind it; the operator's pass, plainly -> nontemporally, alone, with SGD, with Adam:
    //   4096 x 128 x 512  231 -> 226 (219 for 229 where the passes' results stay), 270 -> 264, 317 -> 318    3000 x 128 x 512  206 -> 204, 245 -> 239, 295 -> 298
    //   8192 x 64 x 512  217 -> 202, 232 -> 240, 283 -> 284    2500 x 128 x 768  266 -> 265, 332 -> 337, 462 -> 462    8192 x 256 x 512  601 -> 586, 671 -> 662
    const int64_t first_row = (int64_t)t * a.S + row0;
    const int rows = (int)min<int64_t>(r1, a.rows - first_row);      // the last table of a row count that a.S does not divide: fewer, or none
    if (i16 * 4 >= a.Do - slice * SC) return;                 // (the last slice may be half a one)
    // ADD: rows that no token points at stay as they are, to the bit, and are not touched (somebody else may be adding to them).  The offsets of both
    // lists are still there.
    auto live = [&](int row) {
        if (row >= rows) return false;
        if (!ADD) return true;
        const int *const o = off_s + row, *const o2 = o + (a.subs - 1) * (R + 1);
        return o[1] > o[0] || o2[1] > o2[0];
    };
    constexpr int DEPTH = 4;
    float *const first = a.out + (size_t)first_row * a.Do + (size_t)slice * SC + i16 * 4;
    for (int row_k = r0 + (tid >> 4); row_k < rows; row_k += MWG / 16 * DEPTH) {
        float4 v[DEPTH];
        bool mine[DEPTH];
#pragma unroll
        for (int k = 0; k < DEPTH; ++k) {
            const int row = row_k + k * (MWG / 16);
            mine[k] = live(row);
            if (ADD && mine[k]) v[k] = *reinterpret_cast<const float4 *>(first + (size_t)row * a.Do);
        }
#pragma unroll
        for (int k = 0; k < DEPTH; ++k) {
            const int row = row_k + k * (MWG / 16);
            if (!mine[k]) continue;
            const float4 sum = lds4[row * (SC / 4) + i16];
            v[k] = ADD ? add4(v[k], sum) : sum;
            float *p = first + (size_t)row * a.Do;
            if (a.more) *reinterpret_cast<float4 *>(p) = v[k];                     // uniform
            else __builtin_nontemporal_store((f32x4){v[k].x, v[k].y, v[k].z, v[k].w}, reinterpret_cast<f32x4 *>(p));
        }
    }
}

template <bool ADD, typename Sum>
int launch_sorted_form(SortedArgs a, hipStream_t st) {
    // 512 rows, whole -> two blocks, us, codes spread evenly, by Zipf's law in any order of the rows, in order from row 0 on: 16384 x 128 x 256 168 -> 132, 173 -> 151,
    // 188 -> 199; x 768 437 -> 335, 447 -> 369, 494 -> 521; 8192 x 64 x 1024 170 -> 126, 172 -> 136, 187 -> 184.
    a.block_rows = a.S < MAX_BLOCK_ROWS ? a.S : MAX_BLOCK_ROWS;
    a.block_bits = lffn_log2(a.S / a.block_rows);
    const int64_t blocks = (int64_t(a.T) << a.block_bits) * a.nslices;
    // As many parts as give every compute unit a workgroup, and twice as many where most of them would otherwise wait for the others' second.  us, whole
    // tables -> parts, codes as above: 65536 x 32 x 256 (128 workgroups) 335 -> 250, 346 -> 271, 371 -> 273; 16384 x 32 x 256 79 -> 60, 80 -> 67, 83 -> 62;
    // 32768 x 32 x 576 (288) 255 -> 218, 260 -> 235, 266 -> 232; 16384 x 32 x 768 (384) 125 -> 103, 127 -> 114, 128 -> 112; but 16384 x 100 x 256 (400) 117 -> 122,
    // 118 -> 127, 122 -> 136.
    auto more_parts = [&](int64_t least, int64_t most) {
        const int64_t units = blocks << a.part_bits;
        return units >= least && units <= most && a.block_rows >> a.part_bits > 16;
    };
    while (more_parts(0, COMPUTE_UNITS - 1)) ++a.part_bits;
    if (more_parts(COMPUTE_UNITS + 1, COMPUTE_UNITS * 3 / 2)) ++a.part_bits;
    const size_t lds = size_t(a.block_rows) * SC * sizeof(float) + (WAVES * 2 + 1) * SC * sizeof(Sum) +
                       (2 * WAVES * 4 + 2 * CUTS + size_t(2) * (a.block_rows + 1)) * sizeof(int);
    static LdsGrant granted;
    if (!lffn_grant_dynamic_lds(reinterpret_cast<const void *>(lookup_scatter_sorted_kernel<ADD, Sum>), lds, granted)) return LFFN_ERR_LAUNCH;
    a.per_xcd = (int)(((blocks << a.part_bits) + XCDS - 1) / XCDS);
    hipLaunchKernelGGL((lookup_scatter_sorted_kernel<ADD, Sum>), dim3((unsigned)(a.per_xcd * XCDS)), dim3(MWG), lds, st, a);
    return lffn_launch_status();
}

// Calls of fewer products than this and of at most CHUNK tokens have their sums in doubles: the LDS form (lookup_scatter.hip) has, which
// served the layer there and takes longer from LFFN_SCATTER_SORTED_WORK products on.  They cost little beside the loads (3000 tokens of
// 128 tables of 768 columns 81 -> 90 us, 4096 x 64 x 512 50 -> 53; the LDS form 192 and 64), and the error against 64 bits is 2.6e-8
// (fp32 5.5e-8 to 5.7e-8, the LDS form's products rounded to fp32 3.6e-8), whatever pieces cut: a row's parts stay doubles and are rounded once.
inline bool sums_in_doubles(int64_t B, int64_t T, int64_t Do) {
    return B <= CHUNK && double(B) * double(T) * double(Do) < LFFN_SCATTER_DOUBLE_WORK;
}

int launch_sorted(const SortedArgs &a, bool doubles, hipStream_t st) {
    if (doubles) return a.accumulate ? launch_sorted_form<true, double>(a, st) : launch_sorted_form<false, double>(a, st);
    return a.accumulate ? launch_sorted_form<true, float>(a, st) : launch_sorted_form<false, float>(a, st);
}

inline int64_t slices(int64_t Do) { return (Do + SC - 1) / SC; }
// One list of a chunk's tokens, or two: then half of the sort's wavefronts have the first, and all of them as many batches of 64.
// Sums in doubles are not taken apart (kept in fp32 between two lists, the error is 3.8e-8 instead of 2.6e-8 at 12000 tokens).
inline int64_t sub_lists(int64_t Bc, bool doubles = false) { return Bc > SUB && !doubles ? 2 : 1; }
inline int64_t list_tokens(int64_t Bc, bool doubles = false) {
    return sub_lists(Bc, doubles) > 1 ? (Bc + SORT_WG - 1) / SORT_WG * (SORT_WG / 2) : Bc;
}
inline int64_t pair_stride(int64_t Bc, bool doubles = false) { return (list_tokens(Bc, doubles) + 7) & ~int64_t(7); }      // (times their number: doubles' is no more)

inline bool sorted_supported(int64_t B, int64_t T, int64_t S, int64_t Do) {
    return B >= 1 && T >= 1 && lffn_is_pow2(S) && S <= MAX_S && Do % 32 == 0 && Do <= (1 << 20) &&
           B <= (int64_t(1) << 31) - 1 && T <= (1 << 20) && T * ((Do / 32 + XCDS - 1) / XCDS) * XCDS <= 0x7fffffff;
}

inline int64_t pack_workgroups(int64_t Bc) { return (Bc + 1 + PACK_TOKENS - 1) / PACK_TOKENS; }
inline int64_t round16(int64_t v) { return (v + 15) & ~int64_t(15); }
inline int64_t whole_rows(int64_t v) { return (v + SC * 4 - 1) / (SC * 4) * (SC * 4); }      // rows of the copy of g on whole lines
inline int64_t padded_tokens(int64_t B) { return (B + 63) & ~int64_t(63); }

// Tokens are taken CHUNK at a time (later chunks add to the result of the earlier ones): a
// list's 64 columns of 8192 rows of g are 2 MB and stay in an XCD's 4 MB L2 while the
// workgroups of that XCD walk them in as many orders; twice that no longer does.
static_assert(CHUNK <= 2 * SUB, "a chunk's tokens are one list or two");

struct Workspace {
    int64_t pairs, off, code_t, score_t, g_packed, total;    // byte offsets
};

inline Workspace workspace_layout(int64_t B, int64_t T, int64_t S, int64_t Do) {
    Workspace w{};
    const int64_t Bc = B < CHUNK ? B : CHUNK, Bp = padded_tokens(Bc);
    w.pairs = 0;
    w.off = w.pairs + sub_lists(Bc) * T * pair_stride(Bc) * 8;
    w.code_t = w.off + round16(sub_lists(Bc) * T * (S + 2) * 4);
    w.score_t = w.code_t + round16(T * Bp * 2);
    w.g_packed = whole_rows(w.score_t + T * Bp * 4);
    w.total = w.g_packed + (Bc + 1) * slices(Do) * SC * 4;
    return w;
}

}  // namespace

extern "C" int lffn_lookup_scatter_workspace_bytes(int64_t B, int64_t T, int64_t S, int64_t Do, int64_t *bytes) {
    LFFN_REQUIRE(bytes, LFFN_ERR_BAD_ARG);
    *bytes = sorted_supported(B, T, S, Do) ? workspace_layout(B, T, S, Do).total : 0;
    return LFFN_OK;
}

// Where the sorted form is the one to use.  From LFFN_SCATTER_DOUBLE_WORK products on it is; below, lffn_lookup_scatter_f32 sums in LDS, which
// takes 6.1 us per thousand tokens for every round of one workgroup (64 columns of a table) on each compute unit, whatever the round has.  The sorted form
// reads and writes g once more, which few tables of many columns don't repay.  Training step of the layer, us, LDS form -> sorted (whose copy of g gives the output
// bias's gradient, too):
//   more than one round     3000 x 48 x 384 157 -> 130, 16384 x 32 x 640 452 -> 349, 8192 x 128 x 256 303 -> 266; both gradients alone 4600 x 16 x 4096
//                           200 -> 180, 8192 x 16 x 2048 163 -> 167, but 4600 x 8 x 4096 113 -> 137, 8192 x 8 x 4096 181 -> 245
//   more than half a round  16384 x 48 x 256 282 -> 245, 4600 x 48 x 256 136 -> 132, 8192 x 32 x 448 186 -> 179, 16384 x 32 x 512 275 -> 249, 4600 x 64 x 256 149 -> 150,
//                           4600 x 32 x 512 160 -> 163, 16384 x 12 x 768 312 -> 294, 4600 x 16 x 768 142 -> 141; but 3000 x 16 x 1024 124 -> 130, 16384 x 16 x 1024 369 -> 382
//   half a round or less    8192 x 32 x 256 146 -> 132, 16384 x 8 x 1024 350 -> 330, 16384 x 4 x 1024 336 -> 293; but both gradients alone 8192 x 4 x 2048 78 -> 89,
//                           16384 x 1 x 4096 161 -> 224
// With 512 rows lffn_lookup_scatter_f32 has only atomics (both gradients of 16384 x 32 x 256 1785 -> 124), and columns that are no multiple of 64 it does not take.
extern "C" int lffn_lookup_scatter_plan(int64_t B, int64_t T, int64_t S, int64_t Do, int32_t *sorted) {
    LFFN_REQUIRE(sorted, LFFN_ERR_BAD_ARG);
    const double work = double(B) * double(T) * double(Do);
    *sorted = 0;
    if (!sorted_supported(B, T, S, Do) || B <= LFFN_SCATTER_LIST_TOKENS || work < LFFN_SCATTER_SORTED_WORK) return LFFN_OK;
    if (work >= LFFN_SCATTER_DOUBLE_WORK) {
        *sorted = 1;
    } else if (B <= CHUNK) {
        const int64_t workgroups = T * (Do / 64);
        const int64_t most_columns = workgroups > COMPUTE_UNITS ? 256 * T : workgroups > COMPUTE_UNITS / 2 ? 768 : 1024;
        *sorted = S > 256 || Do % 64 != 0 || Do <= most_columns ? 1 : 0;
    }
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
    int32_t *off = reinterpret_cast<int32_t *>(base + w.off);
    const bool doubles = sums_in_doubles(B, T, Do);

    for (int64_t c0 = 0; c0 < B; c0 += CHUNK) {
        const int64_t Bc = B - c0 < CHUNK ? B - c0 : CHUNK;
        const int64_t stride = pair_stride(Bc, doubles), Bp = padded_tokens(Bc);

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
        sa.code = pa.code_t; sa.score = pa.score_t; sa.pairs = pairs; sa.off = off;
        sa.B = Bc; sa.Bp = Bp; sa.sub_len = list_tokens(Bc, doubles); sa.stride = stride;
        sa.T = (int)T; sa.S = (int)S; sa.nbits = lffn_log2(S); sa.subs = (int)sub_lists(Bc, doubles);
        // histograms and bucket starts, then the sorted lists themselves (4 + 2 bytes per entry)
        static_assert(CHUNK <= 65536 && CHUNK % SORT_WG == 0, "a list's tokens are staged as 16-bit values, and held in registers");
        size_t sort_lds = nsort ? size_t(SORT_WAVES + sa.subs) * S * sizeof(int) + size_t(sa.subs) * stride * 6 : 0;
        if (pa.sums && sort_lds < SORT_WG * sizeof(float4)) sort_lds = SORT_WG * sizeof(float4);
        static LdsGrant granted;
        if (!lffn_grant_dynamic_lds(reinterpret_cast<const void *>(lookup_sort_pack_kernel), sort_lds, granted))
            return LFFN_ERR_LAUNCH;
        hipLaunchKernelGGL(lookup_sort_pack_kernel, dim3((unsigned)(nsort + pack_blocks)), dim3(SORT_WG), sort_lds, st, sa, pa,
                           (int)nsort);
        rc = lffn_launch_status();
        if (rc != LFFN_OK) return rc;

        if (grad_score) {
            // token b's 64 columns of slice s sit at g_packed + (s * (Bc + 1) + b) * 64
            if (!lffn_internal_lookup_inner_quad_try(pa.code, pa.g_packed, SC, (Bc + 1) * SC, tables, grad_score + c0 * T, Bc, T, S,
                                                     Do, B <= CHUNK, stream, &rc))
                rc = lffn_lookup_inner_f32(pa.code, pa.g, tables, grad_score + c0 * T, Bc, T, S, Do, stream);
            if (rc != LFFN_OK) return rc;
        }
        if (!grad_tables) continue;

        SortedArgs ma{};
        ma.pairs = pairs; ma.off = off; ma.g = pa.g_packed; ma.out = grad_tables; ma.rows = T * S; ma.B = (int)Bc;
        ma.T = (int)T; ma.S = (int)S; ma.Do = (int)Do; ma.nslices = (int)slices(Do); ma.subs = sa.subs;
        ma.sub_len = (int)sa.sub_len;
        ma.accumulate = (accumulate || c0 > 0) ? 1 : 0;
        ma.more = c0 + CHUNK < B ? 1 : 0;
        rc = launch_sorted(ma, doubles, st);
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
//   rows_claim_kernel   one workgroup per 256 rows (a "table" of the accumulation) scans their counts and takes that
//                       much of the list; which table's part comes first does not matter (more than SUB tokens: as if each of their
//                       two parts had rows of its own)
//   rows_place_kernel   pairs into the list; other workgroups copy
//                       g slice-major
// The order inside a row is the order of arrival: sums differ from run to run in their last bit, as they did with
// atomics.
namespace {

constexpr int VT = 256;                 // rows per "table"

struct RowsArgs {
    const int32_t *idx;    // [B, I]
    const float *w;        // [B, I]
    const void *g;         // [B, Dv] fp32 or half
    int32_t *count;        // [subs * tables * VT] pairs per row, then (one word) the lists' end in units of eight entries
    int32_t *rank;         // [B * I]
    int32_t *off;          // [subs * tables, VT + 2] as in SortArgs
    int32_t *flags;        // [TABLE_FLAGS] not zero where a row number lies outside its column's table, or null: not looked for
    uint2 *pairs;
    float *g_packed;       // [Dv / SC][B + 1][SC], the last row zero
    int64_t B, n, rows;
    int64_t sub_pairs;     // pairs of the tokens whose pairs are listed together (all of them or SUB tokens')
    int I, Dv, tables, subs, place_blocks;
};

__device__ __forceinline__ int row_of(const RowsArgs &a, int64_t e) {
    const int64_t raw = a.idx[e], hi = a.rows - 1;
    return (int)(raw < 0 ? 0 : (raw > hi ? hi : raw));
}
// the place of pair e's counter: its row's, among those of its part of the tokens
__device__ __forceinline__ int64_t counter_of(const RowsArgs &a, int64_t e) {
    return (e >= a.sub_pairs ? (int64_t)a.tables * VT : 0) + row_of(a, e);
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
    for (int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x; e < a.n; e += stride) a.rank[e] = atomicAdd(a.count + counter_of(a, e), 1);
}

// The same for many tokens.  Row numbers as the layer forms them lie in table i in column i: then a workgroup has RANK_TOKENS tokens of
// RANK_COLS columns, counts them in LDS and takes their places from one add per row.  What bounds it is the adds that return something,
// 24 G/s: 4096 x 128 pairs, 32768 rows, 22 -> 7 us, 16000 x 64 41 -> 9.5, 2500 x 256 27 -> 8 (neighbouring columns on one XCD: 7 -> 5.8).  For other row numbers an add for every pair, in
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
            for (int k = 0; k < EACH; ++k) rank[k] = e0 + k * stride < a.n ? atomicAdd(a.count + counter_of(a, e0 + k * stride), 1) : 0;
#pragma unroll
            for (int k = 0; k < EACH; ++k)
                if (e0 + k * stride < a.n) a.rank[e0 + k * stride] = rank[k];
        }
        return;
    }
    // neighbouring groups of columns on one XCD, as rows_place_kernel has them
    const int per_xcd = (col_groups + XCDS - 1) / XCDS, group = int(blockIdx.x % XCDS) * per_xcd + int(blockIdx.x / XCDS % per_xcd);
    if (group >= col_groups) return;                          // uniform
    const int64_t b_first = int64_t(blockIdx.x / XCDS / per_xcd) * RANK_TOKENS;
    const int c = threadIdx.x % RANK_COLS, col0 = group * RANK_COLS, col = col0 + c;
    const int64_t b0 = b_first + threadIdx.x / RANK_COLS;
    static_assert(SUB % RANK_TOKENS == 0, "a workgroup's tokens are of one part");
    int32_t *const count = a.count + (b_first * a.I >= a.sub_pairs ? (size_t)a.tables * VT : 0);
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
        if (row[k] >= 0) rank[k] = in_table(k) ? atomicAdd(&place[c * VT + row[k] % VT], 1) : atomicAdd(count + row[k], 1);
    __syncthreads();
    const int n = place[threadIdx.x];             // row threadIdx.x % VT of table col0 + threadIdx.x / VT
    if (n > 0) place[threadIdx.x] = atomicAdd(count + (size_t)col0 * VT + threadIdx.x, n);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EACH; ++k)
        if (row[k] >= 0)
            a.rank[(b0 + k * (RANK_WG / RANK_COLS)) * a.I + col] = rank[k] + (in_table(k) ? place[c * VT + row[k] % VT] : 0);
}

__global__ __launch_bounds__(VT) void rows_claim_kernel(RowsArgs a) {
    __shared__ int wave_sum_s[VT / 64];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int mine = a.count[(size_t)t * VT + tid];
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
    int32_t *off = a.off + (size_t)t * (VT + 2);
    off[tid] = before + inc - mine;
    if (tid == 0) {
        off[VT] = total;
        off[VT + 1] = atomicAdd(a.count + (size_t)a.subs * a.tables * VT, (total + 7) >> 3);
    }
}

__device__ __forceinline__ float4 load4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ float4 load4(const _Float16 *p) {
    typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
    const half4_t h = *reinterpret_cast<const half4_t *>(p);
    return make_float4((float)h.x, (float)h.y, (float)h.z, (float)h.w);
}

constexpr int PLACE_COLS = 32;
template <typename G>
__global__ __launch_bounds__(256) void rows_place_kernel(RowsArgs a) {
    if ((int)blockIdx.x < a.place_blocks) {
        // An XCD takes an eighth of the columns, from PLACE_COLS of them on: where column i's rows are of table i, what is written to a line
        // of a list then meets in one L2 (4096 x 128 pairs 13.3 -> 8.4 us).
        const unsigned xcds = a.I >= PLACE_COLS ? XCDS : 1, cols = (unsigned)(a.I + xcds - 1) / xcds, col0 = blockIdx.x % xcds * cols;
        if (col0 >= (unsigned)a.I) return;                    // uniform
        const unsigned mine = min(cols, a.I - col0), pairs = (unsigned)a.B * mine;
        for (unsigned q = blockIdx.x / xcds * 256 + threadIdx.x; q < pairs; q += a.place_blocks / xcds * 256) {
            const unsigned b = q / mine;
            const int64_t e = (int64_t)b * a.I + col0 + (q - b * mine);
            const int64_t row = counter_of(a, e);
            const unsigned token = e >= a.sub_pairs ? b - (unsigned)SUB : b;
            const int32_t *off = a.off + row / VT * (VT + 2);
            a.pairs[(int64_t)off[VT + 1] * 8 + off[row % VT] + a.rank[e]] = make_uint2(token, __float_as_uint(a.w[e]));
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
// all its columns from g as it lies and writes it whole.  The slice-by-slice accumulation above reads every row's list once per 64
// columns and copies g first, which for rows of a few pairs is most of its time.  All five launches, us, by slices -> so, rows by chance: 2 pairs a row 128 x 512
// 45 -> 30, 512 x 1024 218 -> 128 (537 MB written: 4.2 TB/s); 4 pairs 53 -> 38, 260 -> 185, 32 x 256 22 -> 22; 6 pairs 58 -> 46, 297 -> 298, 128 x 768 74 -> 66; 8 pairs 58 -> 51,
// 303 -> 399, 75 -> 84, 26 -> 29; 16 pairs 75 -> 111, 449 -> 1006; by Zipf's law in any order of the rows 2 pairs 41 -> 41, 4 pairs 51 -> 56, 8 pairs 58 -> 81.  So the limit, set by a
// slower form by slices (16 pairs of 128 x 512 128 us either way), is some two pairs too high but for tables of few columns.  A row of more than LONG_ROW pairs goes to the whole workgroup; with half of all pairs on one row a single
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
    const int32_t *const off = a.off + first / VT * (VT + 2);      // (a workgroup's rows are of one table)
    static_assert(VT % ROW_GROUP == 0, "a workgroup's rows are of one table");
    const int my_count = a.count[my_row], my_off = off[my_row % VT];
    const uint2 *const pairs = a.pairs + (int64_t)off[VT + 1] * 8;
    auto list_of = [&](int r) { return pairs + __builtin_amdgcn_readlane(my_off, r); };
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
    int64_t count, rank, off, pairs, g_packed, flags, total;
};

// The lists that a launch walks: of all its tokens where rows are summed from g as it lies (SPARSE_PAIRS), of SUB tokens each otherwise.
inline bool rows_sparse(int64_t Bc, int64_t I, int64_t rows) { return Bc * I <= SPARSE_PAIRS * rows; }

// Worth it from 3e6 products on (five launches, about 30 us of them whatever the size, against 79 G atomics/s; forward and backward at 512
// tokens of 32 x 256, 4e6 products: fp32 75 -> 71 us, half 155 -> 99; at 128 x 512, 64 tokens 104 -> 73 and 219 -> 99) and while
// the list that every slice reads is in proportion: at least one pair for every four rows of the output.
bool rows_supported(int64_t B, int64_t I, int64_t rows, int64_t Dv) {
    if (B < 1 || I < 1 || rows < 1 || Dv < 32 || Dv % 32 != 0 || Dv > (1 << 20)) return false;
    const int64_t Bc = B < CHUNK ? B : CHUNK, tables = (rows + VT - 1) / VT;
    return Bc * I < (int64_t(1) << 31) - 8 * 256 && rows <= (int64_t(1) << 30) && B * I * 4 >= rows &&
           double(B) * double(I) * double(Dv) >= 3e6 && tables * ((Dv / 32 + XCDS - 1) / XCDS) * XCDS <= 0x7fffffff &&
           (Bc + 1) * Dv / 1024 < (int64_t(1) << 30);
}

RowsWorkspace rows_layout(int64_t B, int64_t I, int64_t rows, int64_t Dv) {
    RowsWorkspace w{};
    const int64_t Bc = B < CHUNK ? B : CHUNK, tables = (rows + VT - 1) / VT, n = Bc * I;
    const int64_t lists = sub_lists(Bc) * tables;               // (a shorter last launch has no more of them)
    w.count = 0;
    w.rank = round16((lists * VT + 1) * 4);
    w.off = w.rank + round16(n * 4);
    w.pairs = w.off + round16(lists * (VT + 2) * 4);
    w.g_packed = whole_rows(w.pairs + (n + 7 * lists) * 8 + 8);
    w.flags = w.g_packed + (Bc + 1) * slices(Dv) * SC * 4;
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
        a.off = reinterpret_cast<int32_t *>(base + l.off);
        a.pairs = reinterpret_cast<uint2 *>(base + l.pairs);
        a.g_packed = reinterpret_cast<float *>(base + l.g_packed);
        a.n = a.B * I; a.rows = out_size; a.I = (int)I; a.Dv = (int)Dv;
        a.tables = (int)((out_size + VT - 1) / VT);
        const int64_t blocks = (a.n + 255) / 256;
        a.place_blocks = (int)((blocks < 4096 ? blocks + XCDS - 1 : 4096) / XCDS * XCDS);
        const bool sparse = rows_sparse(a.B, I, out_size);       // (no slice-major copy of g)
        a.subs = sparse ? 1 : (int)sub_lists(a.B);
        a.sub_pairs = a.subs > 1 ? SUB * I : a.n;
        const int64_t pack_blocks = sparse ? 0 : ((a.B + 1) * (Dv / 4) + 1023) / 1024;
        const int64_t zero4 = l.rank / 16;                      // the counters and the list's end
        a.flags = a.B >= RANK_TABLES_TOKENS ? reinterpret_cast<int32_t *>(base + l.flags) : nullptr;
        const int64_t zero_blocks = (zero4 + 1023) / 1024;
        hipLaunchKernelGGL(rows_zero_kernel, dim3((unsigned)(a.flags || zero_blocks > TABLE_FLAGS ? TABLE_FLAGS : zero_blocks)), dim3(1024), 0, st, a,
                           zero4);
        if (a.flags) {
            const int col_groups = (int)((I + RANK_COLS - 1) / RANK_COLS);      // (workgroups: fewer than pairs)
            hipLaunchKernelGGL(rows_rank_tables_kernel, dim3((unsigned)((a.B + RANK_TOKENS - 1) / RANK_TOKENS * ((col_groups + XCDS - 1) / XCDS * XCDS))), dim3(RANK_WG), 0,
                               st, a, col_groups);
        } else {
            hipLaunchKernelGGL(rows_rank_kernel, dim3((unsigned)a.place_blocks), dim3(256), 0, st, a);
        }
        hipLaunchKernelGGL(rows_claim_kernel, dim3((unsigned)(a.subs * a.tables)), dim3(VT), 0, st, a);
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
        ma.pairs = a.pairs; ma.off = a.off; ma.g = a.g_packed; ma.out = out; ma.rows = out_size; ma.B = (int)a.B;
        ma.T = a.tables; ma.S = VT; ma.Do = (int)Dv; ma.nslices = (int)slices(Dv); ma.subs = a.subs;
        ma.sub_len = (int)(a.sub_pairs / I);
        ma.accumulate = (accumulate || c0 > 0) ? 1 : 0;
        ma.more = c0 + CHUNK < B ? 1 : 0;
        rc = launch_sorted(ma, false, st);
        if (rc != LFFN_OK) return rc;
    }
    return LFFN_OK;
}
