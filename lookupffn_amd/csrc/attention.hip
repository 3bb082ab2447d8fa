// softmax(q k^T / 8 - 1000 (1 - mask)) v of heads of 64 columns in fp32 (PL/layer.py:33-47), on the fp16 matrix cores
// (split_mfma.h).
//
// A workgroup has 128 queries of a head, 32 a wavefront, and walks the keys 64 at a time with the running maximum and sum of a
// softmax taken in one pass.  Keys and values are fetched as fp32 a step ahead and split on the way into LDS (two buffers; the values
// turned round, a column's keys side by side).  Scores are formed as keys x queries, so that a lane holds 16 keys' scores of one
// query of every 32: the softmax stays in the lane but for one exchange with the lane that has the other 16, and the weights are
// the next product's operand where they are (its k runs over the keys in the order the lane holds them; the values lie in that order).
//
// Scaling by powers of two, a largest number to 2^14 and more: queries each by their own, keys eight at a time (the eight that a
// wavefront splits and a lane's results of one row of four share a factor), a column of the values by its largest so far, weights by 2^14
// behind the power (an exponent near 14 would be rounded to 2^-21).  A value that outgrows its column's scale in a later step has the
// column's sums so far scaled down to the new one.  All are large enough for the lo term to be kept without a factor, so that one
// accumulator does.  The mask's largest term is taken off before the scores are formed (a softmax does not see it): a sentence of nothing
// but padding comes out 100 times closer to 64 bits than with -1000 in fp32.  Infinities and NaN are not carried by the split: a
// wavefront with such results does its queries again in fp32, key by key (2.1 ms where every wavefront has to).
//
// 32 x 512 tokens, 12 heads: 110 us, 235 TFLOP/s of fp32 product, of the same tensors again and again, 126 of three sets in turn (library,
// fp32 matrix cores: 490 and 35 for a copy); 113 with a scale
// for every key, 103 with one for all keys and one for all values taken from the first 64 (which lost numbers far smaller and sent
// numbers 500 times larger through the fp32 loop).  The three products' matrix instructions are 67 us of that at the rate a large
// half-precision product reaches, the vector work on a score (two multiply-adds, exp2, maximum, sum, split) as much again, partly
// beside them.  Error against 64 bits 3.4e-7 (library 4.6e-7), 17 tokens 1.5e-7 (1.9e-7).
#include "split_mfma.h"


namespace {

constexpr int HEAD = 64;                  // columns of a head
constexpr int QT = 128;                   // queries of a workgroup, 32 a wavefront
constexpr int KT = 64;                    // keys of a step
constexpr int PLANE = KT * 8;             // 16-byte pieces of a term of a step's keys or values
constexpr int BUF = 4 * PLANE;            // keys hi, lo, values hi, lo
constexpr float LOG2E = 1.4426950408889634f;
constexpr int TOP = 14;                   // a query's and a key's largest number goes to 2^14 and more, and a column's of the values among
constexpr float MOST_V = 65504.f;         // the keys seen so far, until a value outgrows this

struct AttentionArgs {
    const float *q, *k, *v;               // [B, L, heads, 64]
    const float *mask;                    // [B, L]
    float *out;                           // [B, L, heads, 64]
    int64_t B;
    int L, heads;
};

// Piece `piece` of row `row` of a plane: rows of 128 bytes, turned so that 16 rows' reads of one piece fall on different banks.
__device__ __forceinline__ int at_piece(int row, int piece) { return row * 8 + (piece ^ ((row >> 1) & 7)); }

// 2^e, -126 <= e <= 127
__device__ __forceinline__ float power_of_two(int e) { return __uint_as_float((127 + e) << 23); }

// eight numbers as hi and the rest
__device__ __forceinline__ void split8(const float (&v)[8], uint4 &hi, uint4 &lo) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        h[e] = split_hi(v[2 * e], v[2 * e + 1], 1.f);
        l[e] = split_rest(v[2 * e], v[2 * e + 1], h[e]);
    }
    hi = make_uint4(h[0], h[1], h[2], h[3]);
    lo = make_uint4(l[0], l[1], l[2], l[3]);
}

__global__ __launch_bounds__(256, 2) void attention_kernel(AttentionArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint4 lds[];
    float *const bias = reinterpret_cast<float *>(lds + 2 * BUF);        // [L rounded up to KT]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 31, half = lane >> 5;
    const int L = a.L, H = a.heads * HEAD, steps = (L + KT - 1) / KT;
    float *const unscale_k = bias + steps * KT;                          // [2][8] of a step's keys, eight to a scale
    float *const shrink = unscale_k + 2 * 8;                             // [2][HEAD] what a step's columns of the values have their sums
                                                                         // multiplied with before they are added to
    uint32_t *const shrunk = reinterpret_cast<uint32_t *>(shrink + 2 * HEAD);      // [2][4] whether there is one in a wavefront's columns
    float *const part = shrink;                                          // (4 words, before the first step)
    const int qtiles = (L + QT - 1) / QT;
    const int nblk = gridDim.x, xcd = blockIdx.x & 7, per = nblk >> 3, rem = nblk & 7;
    const int unit = xcd * per + min(xcd, rem) + (blockIdx.x >> 3);
    const int qt = unit % qtiles, bh = unit / qtiles, head = bh % a.heads;
    const int64_t b = bh / a.heads;
    const int64_t base = b * L * H + head * HEAD;
    const float *const kp = a.k + base, *const vp = a.v + base;

    // the thread's share of a step: two pieces of keys, sixteen keys of one column of the values (a wavefront has all keys of its
    // sixteen columns)
    const int krow = tid >> 3, kpiece = tid & 7, vcol = wave * 16 + (lane & 15), vgroup = lane >> 4;
    float kv[2][8], vv[16];
    auto fetch = [&](int step) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int key = step * KT + krow + 32 * i;
            const float *p = kp + int64_t(min(key, L - 1)) * H + kpiece * 8;
            *reinterpret_cast<float4 *>(&kv[i][0]) = *reinterpret_cast<const float4 *>(p);
            *reinterpret_cast<float4 *>(&kv[i][4]) = *reinterpret_cast<const float4 *>(p + 4);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) vv[i] = vp[int64_t(min(step * KT + vgroup * 16 + i, L - 1)) * H + vcol];
    };
    float vscale = 0.f;
    int vexponent = 0;
    auto place = [&](int step) {
        uint4 *const buf = lds + (step & 1) * BUF;
        const bool last = (step + 1) * KT > L;              // keys beyond the end: a value of one would be read as 0 x whatever it is
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float t[8], m = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(kv[i][e]));
            m = fmaxf(m, lane_xor<1>(m));
            m = fmaxf(m, lane_xor<2>(m));
            m = fmaxf(m, lane_xor<4>(m));
            m = fmaxf(m, lane_xor<8>(m));
            m = rows_most(m);
            int back;
            const float scale = scale_to(m, TOP, back);
#pragma unroll
            for (int e = 0; e < 8; ++e) t[e] = kv[i][e] * scale;
            uint4 hi, lo;
            split8(t, hi, lo);
            const int row = krow + 32 * i;
            buf[at_piece(row, kpiece)] = hi;
            buf[PLANE + at_piece(row, kpiece)] = lo;
            if (lane == 0) unscale_k[(step & 1) * 8 + 4 * i + wave] = power_of_two(back);
        }
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if (last && step * KT + vgroup * 16 + i >= L) vv[i] = 0.f;
            m = fmaxf(m, fabsf(vv[i]));
        }
        m = rows_most(m);
        const bool grown = step > 0 && m * vscale >= MOST_V && is_finite(m), any = __any(grown);
        if (step == 0) vscale = scale_to(m, TOP, vexponent);
        if (any) {
            const int was = vexponent;
            if (grown) vscale = scale_to(m, TOP, vexponent);
            if (vgroup == 0) shrink[(step & 1) * HEAD + vcol] = __builtin_amdgcn_ldexpf(1.f, was - vexponent);
        }
        if (lane == 0) shrunk[(step & 1) * 4 + wave] = any;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float t[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) t[e] = vv[4 * h + 8 * (e / 4) + e % 4] * vscale;
            uint4 hi, lo;
            split8(t, hi, lo);
            buf[2 * PLANE + at_piece(vcol, 2 * vgroup + h)] = hi;
            buf[3 * PLANE + at_piece(vcol, 2 * vgroup + h)] = lo;
        }
    };

    fetch(0);
    // the queries of this lane's column: 8 of every 16 columns of the head
    const int qrow = qt * QT + wave * 32 + r;
    uint4 fq[4][2];
    float qinv;
    {
        const float *p = a.q + base + int64_t(min(qrow, L - 1)) * H + 8 * half;
        float t[4][8], most = 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            *reinterpret_cast<float4 *>(&t[s][0]) = *reinterpret_cast<const float4 *>(p + 16 * s);
            *reinterpret_cast<float4 *>(&t[s][4]) = *reinterpret_cast<const float4 *>(p + 16 * s + 4);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(t[s][e]));
        most = fmaxf(most, lane_xor<32>(most));
        int back;
        const float scale = scale_to(most, TOP, back);
        qinv = power_of_two(back);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) t[s][e] *= scale;
            split8(t[s], fq[s][0], fq[s][1]);
        }
    }
    // the mask's part of the scores, times log2 e, less its largest (which takes nothing from a softmax)
    float most_b = -INFINITY;
    for (int key = tid; key < L; key += 256) most_b = fmaxf(most_b, -1000.f * (1.f - a.mask[b * L + key]));
    most_b = fmaxf(most_b, lane_xor<1>(most_b));
    most_b = fmaxf(most_b, lane_xor<2>(most_b));
    most_b = fmaxf(most_b, lane_xor<4>(most_b));
    most_b = fmaxf(most_b, lane_xor<8>(most_b));
    most_b = rows_most(most_b);
    if (lane == 0) part[wave] = most_b;
    __syncthreads();
    most_b = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    if (!is_finite(most_b)) most_b = 0.f;
    for (int key = tid; key < steps * KT; key += 256)
        bias[key] = key < L ? (-1000.f * (1.f - a.mask[b * L + key]) - most_b) * LOG2E : -INFINITY;
    const float scale = LOG2E / 8 * qinv;
    place(0);
    if (steps > 1) fetch(1);
    __syncthreads();

    f32x16_t o[2] = {};
    float most = -INFINITY, sum = 0.f;
#pragma unroll 1
    for (int step = 0; step < steps; ++step) {
        const uint4 *const buf = lds + (step & 1) * BUF;
        const uint4 any = *reinterpret_cast<const uint4 *>(shrunk + (step & 1) * 4);
        if (__builtin_amdgcn_readfirstlane(any.x | any.y | any.z | any.w)) {
            // values that have outgrown their columns' scales: the sums so far go by the new ones
            // (a wavefront without such columns has left its part of `shrink` as it was)
            const uint32_t of[4] = {any.x, any.y, any.z, any.w};
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    if (!of[2 * d + g / 2]) continue;
                    const float4 f = *reinterpret_cast<const float4 *>(shrink + (step & 1) * HEAD + d * 32 + 8 * g + 4 * half);
                    o[d][4 * g] *= f.x; o[d][4 * g + 1] *= f.y; o[d][4 * g + 2] *= f.z; o[d][4 * g + 3] *= f.w;
                }
        }
        f32x16_t s[2] = {};
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int at = at_piece(kb * 32 + r, 2 * c + half);
                const uint4 hi = buf[at], lo = buf[PLANE + at];
                s[kb] = mfma_f16(lo, fq[c][0], s[kb]);
                s[kb] = mfma_f16(hi, fq[c][1], s[kb]);
                s[kb] = mfma_f16(hi, fq[c][0], s[kb]);
            }
        // scores times log2 e, their largest so far
        float now = most;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const float4 uk = *reinterpret_cast<const float4 *>(unscale_k + (step & 1) * 8 + 4 * kb);
            const float by[4] = {uk.x * scale, uk.y * scale, uk.z * scale, uk.w * scale};
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 bb = *reinterpret_cast<const float4 *>(bias + step * KT + kb * 32 + 8 * g + 4 * half);
                s[kb][4 * g] = fmaf(s[kb][4 * g], by[g], bb.x);
                s[kb][4 * g + 1] = fmaf(s[kb][4 * g + 1], by[g], bb.y);
                s[kb][4 * g + 2] = fmaf(s[kb][4 * g + 2], by[g], bb.z);
                s[kb][4 * g + 3] = fmaf(s[kb][4 * g + 3], by[g], bb.w);
                now = fmaxf(fmaxf(now, s[kb][4 * g]), s[kb][4 * g + 1]);
                now = fmaxf(fmaxf(now, s[kb][4 * g + 2]), s[kb][4 * g + 3]);
            }
        }
        now = fmaxf(now, lane_xor<32>(now));
        if (__any(now > most)) {
            const float by = now > most ? __builtin_amdgcn_exp2f(most - now) : 1.f;
            sum *= by;
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[d][e] *= by;
            most = now;
        }
        // weights times 2^14 (behind the power: an exponent near 14 would be rounded to 2^-21)
        const float less = most == -INFINITY ? 0.f : most;               // (no key yet that is not masked by an infinity)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                s[kb][e] = __builtin_amdgcn_exp2f(s[kb][e] - less) * 16384.f;
                sum += s[kb][e];
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                float t[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) t[e] = s[kb][8 * c + e];
                uint4 ph, pl;
                split8(t, ph, pl);
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    const int at = at_piece(d * 32 + r, 2 * (2 * kb + c) + half);
                    const uint4 hi = buf[2 * PLANE + at], lo = buf[3 * PLANE + at];
                    o[d] = mfma_f16(lo, ph, o[d]);
                    o[d] = mfma_f16(hi, pl, o[d]);
                    o[d] = mfma_f16(hi, ph, o[d]);
                }
            }
        }
        if (step + 1 < steps) {
            place(step + 1);
            if (step + 2 < steps) fetch(step + 2);
        }
        __syncthreads();
    }
    sum += lane_xor<32>(sum);
    const float by = sum == 0.f ? 0.f : 1.f / sum;           // a query whose keys are all masked by an infinity: zero, as in torch
    if (vgroup == 0) shrink[vcol] = power_of_two(vexponent);             // (the loop's last barrier is behind its last reader)
    __syncthreads();
    bool bad = false;
    float *const op = a.out + base + int64_t(min(qrow, L - 1)) * H + 4 * half;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 uv = *reinterpret_cast<const float4 *>(shrink + d * 32 + 8 * g + 4 * half);
            const float back[4] = {uv.x, uv.y, uv.z, uv.w};
            float t[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                t[e] = o[d][4 * g + e] * by * back[e];
                bad |= !is_finite(t[e]);
            }
            if (qrow < L) *reinterpret_cast<float4 *>(op + d * 32 + 8 * g) = make_float4(t[0], t[1], t[2], t[3]);
        }
    if (__any(bad)) {
        // the split does not carry infinities: the wavefront's queries once more in fp32, half of the head's columns a lane
        float q[32], acc[32] = {};
        const float *const p = a.q + base + int64_t(min(qrow, L - 1)) * H + 32 * half;
#pragma unroll
        for (int e = 0; e < 32; ++e) q[e] = p[e];
        float m = -INFINITY, l = 0.f;
        for (int pass = 0; pass < 2; ++pass)
#pragma unroll 1
            for (int key = 0; key < L; ++key) {
                const float *const kr = kp + int64_t(key) * H + 32 * half, *const vr = vp + int64_t(key) * H + 32 * half;
                float d = 0.f;
#pragma unroll
                for (int e = 0; e < 32; ++e) d = fmaf(q[e], kr[e], d);
                d = (d + lane_xor<32>(d)) * 0.125f + (-1000.f * (1.f - a.mask[b * L + key]) - most_b);
                if (pass == 0) {
                    m = fmaxf(m, d);
                } else {
                    const float w = expf(d - (m == -INFINITY ? 0.f : m));
                    l += w;
#pragma unroll
                    for (int e = 0; e < 32; ++e) acc[e] = fmaf(w, vr[e], acc[e]);
                }
            }
        if (qrow < L) {
            float *const t = a.out + base + int64_t(qrow) * H + 32 * half;
#pragma unroll
            for (int e = 0; e < 32; ++e) t[e] = l == 0.f ? 0.f : acc[e] / l;
        }
    }
}

}  // namespace

extern "C" int lffn_attention_f32(const float *q, const float *k, const float *v, const float *mask, float *out, int64_t B, int64_t L,
                                  int64_t heads, void *stream) {
    LFFN_REQUIRE(q && k && v && mask && out, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(B >= 0 && L >= 0 && heads >= 0, LFFN_ERR_BAD_ARG);
    LFFN_REQUIRE(lffn_aligned16(q) && lffn_aligned16(k) && lffn_aligned16(v) && lffn_aligned16(out), LFFN_ERR_BAD_ARG);
    if (B == 0 || L == 0 || heads == 0) return LFFN_OK;
    LFFN_REQUIRE(L <= LFFN_ATTENTION_MAX_KEYS && heads <= 65536, LFFN_ERR_UNSUPPORTED);
    const int64_t tiles = heads * ((L + QT - 1) / QT);
    LFFN_REQUIRE(B <= INT32_MAX / tiles, LFFN_ERR_UNSUPPORTED);
    const size_t lds = 2 * BUF * 16 + ((L + KT - 1) / KT * KT + 2 * 8 + 2 * HEAD + 8) * 4;
    static LdsGrant granted;
    if (!lffn_grant_dynamic_lds(reinterpret_cast<const void *>(&attention_kernel), lds, granted)) return LFFN_ERR_LAUNCH;
    attention_kernel<<<dim3(B * tiles), dim3(256), lds, static_cast<hipStream_t>(stream)>>>({q, k, v, mask, out, B, (int)L, (int)heads});
    return lffn_launch_status();
}
