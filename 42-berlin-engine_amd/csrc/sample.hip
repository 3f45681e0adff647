// sample.hip -- temperature and top-p sampling of logits on gfx950.
//
// sample_temperature  src/compute/sampler_temp.c:57-114
// sample_top_p        src/compute/sampler_topp.c:17-158
//
// Both turn logits into probabilities p_i = expf((x_i - max) / temp) / sum
// (the temperature sampler starts its max at -1e9, top-p at x_0), then draw
// one index with a uniform number the caller supplies:
//   temperature: the first index whose running sum of p exceeds r
//                (sampler_random_float's draw);
//   top-p:       in the order of p descending (equal probabilities in
//                ascending index order, where the reference's qsort leaves
//                them unspecified), the shortest prefix whose running sum
//                exceeds top_p, r = u * that sum (u = rand() / RAND_MAX),
//                the first entry of the prefix whose running sum exceeds r.
// The temperature sampler's running sums are formed 64 entries at a time
// (lane prefix sums plus a carried sum), equal to the reference's
// sequential fp32 sums to rounding.  Where no running sum exceeds
// r (possible only through rounding) the reference returns n, an index past
// the vocabulary; here the last index is returned.
//
// Top-p never sorts: both cuts are weighted selections.  The entry at which
// the descending-order running sum first exceeds a threshold is found by a
// most-significant-first radix select over the bit patterns of the
// (non-negative) probabilities, where each pass sums the probabilities of the
// remaining candidates per value of a bit field (kSelBits) and keeps the one
// whose bucket holds the crossing; after three passes the crossing entry's
// value is known, and among the entries of that value (ascending index) the
// crossing is the (T - sum above) / value-th.  The sums are exact:
// probabilities as 62-bit fixed point (p * 2^62, truncated) in 64-bit integer
// additions, so they do not depend on the order of the atomic additions, and
// they are the float64 running sums to ~n * 2^-62 -- closer than the
// reference's fp32 sums.
#include <cstring>

#include "be42_common.h"

namespace be42 {

constexpr int kSampT = 1024;

// The loops below read a row with their loads issued U at a time (the
// values into registers first, then used in the same order as one at a
// time): a loop that uses each value as it arrives waits a full memory
// round trip per element, and one block walks a whole 128k-entry row.
//   strided: i = t, t + NT, ... (thread t of NT), f(i, v)
template <int U, int NT = kSampT, class Ld, class F>
__device__ __forceinline__ void strided_batches(int n, Ld &&ld, F &&f)
{
    for (int i0 = threadIdx.x; i0 < n; i0 += U * NT) {
        decltype(ld(0)) v[U];
#pragma unroll
        for (int j = 0; j < U; j++) {
            const int i = i0 + j * NT;
            v[j] = ld(i < n ? i : i0);
        }
#pragma unroll
        for (int j = 0; j < U; j++)
            if (i0 + j * NT < n)
                f(i0 + j * NT, v[j]);
    }
}
//   wave:    entries c0 .. c1 - 1 of one wave, 64 a step (lane l: entry
//            a + l, T(0) past c1), f(a, v) returns true (wave-uniform) to stop
template <int U, class T, class Ld, class F>
__device__ __forceinline__ void wave_steps(Ld &&ld, int c0, int c1, F &&f)
{
    const int lane = threadIdx.x & (kWave - 1);
    for (int a0 = c0; a0 < c1; a0 += kWave * U) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = a0 + kWave * u + lane;
            v[u] = i < c1 ? ld(i) : T(0);
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (a0 + kWave * u < c1 && f(a0 + kWave * u, v[u]))
                return;
    }
}

// the wave's number as a scalar, so that its ranges and loops are scalar too
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); }

// contiguous slice `part` of `parts` of a row, whole steps of `unit` entries
__device__ __forceinline__ void slice_of(int n, int part, int parts, int unit, int &c0, int &c1)
{
    const int cw = ((n + parts - 1) / parts + unit - 1) / unit * unit;
    c0 = min(n, part * cw);
    c1 = min(n, c0 + cw);
}

// inclusive prefix sum over the lanes (DPP row shifts, then row broadcasts)
__device__ __forceinline__ float wave_prefix_sum(float v)
{
    v = v + dpp_mov<0x111>(0.0f, v);         // row_shr:1
    v = v + dpp_mov<0x112>(0.0f, v);         // row_shr:2
    v = v + dpp_mov<0x114>(0.0f, v);         // row_shr:4
    v = v + dpp_mov<0x118>(0.0f, v);         // row_shr:8
    v = v + dpp_mov<0x142, 0xA>(0.0f, v);    // row_bcast:15 into rows 1, 3
    v = v + dpp_mov<0x143, 0xC>(0.0f, v);    // row_bcast:31 into rows 2, 3
    return v;
}
__device__ __forceinline__ float lane63(float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63)); }

__device__ __forceinline__ float block_reduce(float v, float *red, bool is_max)
{
    v = is_max ? wave_max(v) : wave_sum(v);
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
        red[wave] = v;
    __syncthreads();
    float r = red[0];
    for (int w = 1; w < kSampT / 64; w++)
        r = is_max ? fmaxf(r, red[w]) : r + red[w];
    return r;
}

// p[b][i] = expf((x - m) / temp) / sum for row b (one block per row)
template <bool BF16>
__global__ __launch_bounds__(kSampT) void k_probs(float *__restrict__ p, const void *__restrict__ logits, int n,
                                                  float temp, bool max_from_first)
{
    __shared__ float red[kSampT / 64];
    const int b = blockIdx.x;
    auto x = [&](int i) {
        return BF16 ? bf16_to_f32(((const uint16_t *)logits)[(size_t)b * n + i])
                    : ((const float *)logits)[(size_t)b * n + i];
    };
    float m = max_from_first ? x(0) : -1e9f;
    strided_batches<16>(n, x, [&](int, float v) { m = fmaxf(m, v); });
    m = block_reduce(m, red, true);
    float *pb = p + (size_t)b * n;
    float s = 0.0f;
    strided_batches<16>(n, x, [&](int i, float v) {
        const float e = expf(__fdiv_rn(v - m, temp));
        pb[i] = e;
        s += e;
    });
    s = block_reduce(s, red, false);
    strided_batches<16>(n, [&](int i) { return pb[i]; }, [&](int i, float v) { pb[i] = __fdiv_rn(v, s); });
}

// The first position i < lim whose running sum of q exceeds thr, or -1.
// Each wave walks its own contiguous range 64 entries a step; a step's
// running sums are the lanes' prefix sums plus the sum carried from the
// steps before (the range's first step carries the sum of the ranges before).
// sh: 2 * (kSampT / 64) floats.
__device__ int block_first_exceeding(const float *__restrict__ q, int lim, float thr, float *sh, int *found)
{
    constexpr int NW = kSampT / kWave;
    const int wave = wave_id(), lane = threadIdx.x & (kWave - 1);
    int c0, c1;
    slice_of(lim, wave, NW, kWave, c0, c1);
    auto ld = [&](int i) { return q[i]; };
    float carry = 0.0f;
    wave_steps<8, float>(ld, c0, c1, [&](int, float v) {
        carry += lane63(wave_prefix_sum(v));
        return false;
    });
    if (lane == 0)
        sh[wave] = carry;
    if (threadIdx.x == 0)
        *found = INT32_MAX;
    __syncthreads();
    if (threadIdx.x == 0) {
        float o = 0.0f;
        for (int w = 0; w < NW; w++) {
            const float t = sh[w];
            sh[NW + w] = o;
            o += t;
        }
    }
    __syncthreads();
    carry = sh[NW + wave];
    wave_steps<8, float>(ld, c0, c1, [&](int a, float v) {
        const float ps = wave_prefix_sum(v);
        const unsigned long long m = __ballot(carry + ps > thr);
        if (m) {
            if (lane == 0)
                atomicMin(found, a + __ffsll((unsigned long long)m) - 1);
            return true;
        }
        carry += lane63(ps);
        return false;
    });
    __syncthreads();
    const int f = *found;
    __syncthreads();
    return f == INT32_MAX ? -1 : f;
}

__global__ __launch_bounds__(kSampT) void k_pick_temperature(int *__restrict__ out, const float *__restrict__ p, int n,
                                                             const float *__restrict__ r)
{
    __shared__ float sh[2 * (kSampT / kWave)];
    __shared__ int found;
    const int b = blockIdx.x;
    const int i = block_first_exceeding(p + (size_t)b * n, n, r[b], sh, &found);
    if (threadIdx.x == 0)
        out[b] = i < 0 ? n - 1 : i;
}

// the bit fields of a probability's pattern the three passes resolve (12, 10
// and 8 bits; bits 30 and 31 are clear in [0, 1], other patterns weigh
// nothing): the first pass spreads over 7 exponent and 5 mantissa bits, so the
// atomic additions of one wave rarely meet in one bucket, and a bucket is
// 1/32 of a power of two wide
constexpr int kSelPasses = 3;
constexpr int kSelShift[kSelPasses] = {18, 8, 0};
constexpr int kSelBits[kSelPasses] = {12, 10, 8};
constexpr int kSelBins = 1 << 12;

// p as 62-bit fixed point, floor(p * 2^62), from the bits of p in [0, 1]:
// mantissa (with its leading 1) shifted by exponent - 88 (0 for zero,
// subnormal, negative or NaN patterns; those above 1 do not occur)
__device__ __forceinline__ unsigned long long fixp_bits(unsigned k)
{
    const int e = (int)(k >> 23);   // the sign bit makes negative patterns > 255
    if (e == 0 || e > 127)
        return 0ull;
    const unsigned long long m = (unsigned long long)((k & 0x7FFFFFu) | 0x800000u);
    const int sh = e - 88;
    return sh >= 0 ? m << sh : (sh > -64 ? m >> -sh : 0ull);
}
__device__ __forceinline__ unsigned long long fixp(float p) { return fixp_bits(__float_as_uint(p)); }

template <int BINS>
struct SelShared {
    unsigned long long hist[BINS];   // bucket sums of a pass
    unsigned long long scan[kSampT / kWave];
    int isum[kSampT / kWave];
    unsigned long long total, above[3];
    int pos[3], idx;
};
using TopPShared = SelShared<kSelBins>;

__device__ __forceinline__ unsigned long long shfl_u64(unsigned long long v, int l)
{
    return (unsigned long long)(unsigned)__shfl((int)(v >> 32), l, kWave) << 32 | (unsigned)__shfl((int)v, l, kWave);
}
__device__ __forceinline__ unsigned long long shfl_up_u64(unsigned long long v, int o)
{
    const unsigned lo = __shfl_up((unsigned)v, o, kWave), hi = __shfl_up((unsigned)(v >> 32), o, kWave);
    return (unsigned long long)hi << 32 | lo;
}

// inclusive prefix sum over the lanes, as wave_prefix_sum
template <int CTRL, int ROWMASK = 0xF>
__device__ __forceinline__ unsigned long long dpp_u64(unsigned long long v)
{
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)v, CTRL, ROWMASK, 0xF, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWMASK, 0xF, false);
    return (unsigned long long)hi << 32 | lo;
}
__device__ __forceinline__ unsigned long long wave_prefix_sum_u64(unsigned long long v)
{
    v += dpp_u64<0x111>(v);
    v += dpp_u64<0x112>(v);
    v += dpp_u64<0x114>(v);
    v += dpp_u64<0x118>(v);
    v += dpp_u64<0x142, 0xA>(v);
    v += dpp_u64<0x143, 0xC>(v);
    return v;
}

// Exclusive block scan of one value per thread (thread order of NT); sh: one
// word per wave, free again after the caller's next barrier.  Six passes of a
// top-p call each wait for one scan and one crossing_bin: through the LDS
// crossbar, and with four barriers a crossing, a call on a row of 4096 took
// 42.4 us; with lane moves and one barrier 32.5.
template <int NT>
__device__ __forceinline__ unsigned long long block_excl_scan(unsigned long long v, unsigned long long *sh)
{
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const unsigned long long incl = wave_prefix_sum_u64(v);
    if (lane == kWave - 1)
        sh[wave] = incl;
    __syncthreads();
    unsigned long long before = 0;
#pragma unroll
    for (int w = 0; w < NT / kWave; w++)
        before += w < wave ? sh[w] : 0ull;
    return before + incl - v;
}

// A pass's buckets in descending order: thread t holds those at descending
// positions 4t .. 4t + 3 (h) and the sum of every bucket before them (ex); NT
// threads hold at most 4 NT buckets.
struct BinScan {
    unsigned long long h[4], ex;
};
template <int NT, class Sh>
__device__ __forceinline__ BinScan scan_bins(const unsigned long long *hist, int nb, Sh &S)
{
    BinScan r;
    unsigned long long ts = 0;
    if (threadIdx.x < 3)
        S.pos[threadIdx.x] = INT32_MAX;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int d = 4 * (int)threadIdx.x + j;
        r.h[j] = d < nb ? hist[nb - 1 - d] : 0ull;
        ts += r.h[j];
    }
    r.ex = block_excl_scan<NT>(ts, S.scan);
    if (threadIdx.x == NT - 1)
        S.total = r.ex + ts;
    return r;
}

// The descending position of the bucket in which base (at most T) + the
// running sum first exceeds T (INT32_MAX: none does), *above the sum before
// that bucket.  Called by the whole block, once per `at` after a scan_bins (the
// sums do not decrease, so one thread at most has the crossing).
template <class Sh>
__device__ __forceinline__ int crossing_bin(const BinScan &r, unsigned long long base, unsigned long long T,
                                            Sh &S, int at, unsigned long long *above)
{
    unsigned long long acc = base + r.ex;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (acc <= T && acc + r.h[j] > T) {
            S.pos[at] = 4 * (int)threadIdx.x + j;
            S.above[at] = acc;
        }
        acc += r.h[j];
    }
    __syncthreads();
    *above = S.above[at];
    return S.pos[at];
}

// The entry of a list of n probabilities (ld(i): the bits of the i-th, in
// ascending index order) at which the running sum of fixp, taken in descending
// order of value with equal values in list order, first exceeds T; -1 if none
// does.  The passes before pass0 are done: `prefix` holds the bits they found
// and `base` the sum of every entry above them.  *above: the running sum
// before the entry; *all: the sum of every entry (from pass 0).  Called by the
// whole block.
template <int NT, class Ld, class Sh>
__device__ int weighted_select(Ld &&ld, int n, unsigned long long T, Sh &S, int pass0, unsigned prefix,
                               unsigned long long base, unsigned long long *above, unsigned long long *all)
{
    const int tid = threadIdx.x;
    unsigned pmask = 0;
    for (int pass = 0; pass < pass0; pass++)
        pmask |= ((1u << kSelBits[pass]) - 1) << kSelShift[pass];
    for (int pass = pass0; pass < kSelPasses; pass++) {
        const int shift = kSelShift[pass], nb = 1 << kSelBits[pass];
        for (int i = tid; i < nb; i += NT)
            S.hist[i] = 0ull;
        __syncthreads();
        strided_batches<16, NT>(n, ld, [&](int, unsigned k) {
            if ((k & pmask) == prefix) {
                const unsigned long long f = fixp_bits(k);
                if (f)
                    atomicAdd(&S.hist[(k >> shift) & (nb - 1)], f);
            }
        });
        __syncthreads();
        const BinScan r = scan_bins<NT>(S.hist, nb, S);
        const int pos = crossing_bin(r, base, T, S, 0, &base);
        if (pass == 0)
            *all = S.total;
        if (pos == INT32_MAX)
            return -1;
        prefix |= (unsigned)(nb - 1 - pos) << shift;
        pmask |= (unsigned)(nb - 1) << shift;
    }
    // the crossing entry has the value whose bits are `prefix`; among the
    // entries of that value (list order) it is the k-th
    const unsigned long long fv = fixp(__uint_as_float(prefix));   // > 0: its bucket's sum is positive
    const unsigned long long k = (T - base) / fv;
    const int wave = wave_id(), lane = tid & (kWave - 1);
    int c0, c1;
    slice_of(n, wave, NT / kWave, kWave, c0, c1);
    auto match = [&](int a, unsigned v) { return __ballot(a + lane < c1 && v == prefix); };
    int cnt = 0;   // entries of that value in this wave's range
    wave_steps<8, unsigned>(ld, c0, c1, [&](int a, unsigned v) {
        cnt += __popcll(match(a, v));
        return false;
    });
    if (lane == 0)
        S.isum[wave] = cnt;
    if (tid == 0)
        S.idx = -1;
    __syncthreads();
    int off = 0;
    for (int w = 0; w < wave; w++)
        off += S.isum[w];
    if ((unsigned long long)off <= k && k < (unsigned long long)(off + cnt)) {
        int rem = (int)(k - (unsigned long long)off);
        wave_steps<8, unsigned>(ld, c0, c1, [&](int a, unsigned v) {
            unsigned long long m = match(a, v);
            const int c = __popcll(m);
            if (rem < c) {
                for (int j = 0; j < rem; j++)
                    m &= m - 1;
                if (lane == 0)
                    S.idx = a + __ffsll(m) - 1;
                return true;
            }
            rem -= c;
            return false;
        });
    }
    __syncthreads();
    *above = base + k * fv;
    const int idx = S.idx;
    __syncthreads();
    return idx;
}

// The last entry in descending order: the smallest value, the largest index
// among equal ones.
template <int NT, class Sh>
__device__ int last_entry(const float *__restrict__ p, int n, Sh &S)
{
    const int tid = threadIdx.x;
    unsigned long long best = 0;   // (~key << 32 | index): the largest is the last entry
    strided_batches<16, NT>(n, [&](int i) { return __float_as_uint(p[i]); }, [&](int i, unsigned k) {
        const unsigned long long c = ((unsigned long long)~k << 32) | (unsigned)i;
        best = c > best ? c : best;
    });
    unsigned long long *words = S.hist;
    words[tid] = best;
    __syncthreads();
    if (tid == 0) {
        unsigned long long t = 0;
        for (int i = 0; i < NT; i++)
            t = words[i] > t ? words[i] : t;
        S.idx = (int)(unsigned)t;
    }
    __syncthreads();
    const int idx = S.idx;
    __syncthreads();
    return idx;
}

// top_p as a threshold on the fixed-point sums (which stay near 2^62: a
// threshold of 2 or more is never exceeded)
__device__ __forceinline__ unsigned long long cut_threshold(float top_p)
{
    return top_p >= 2.0f ? ~0ull : (top_p > 0.0f ? (unsigned long long)((double)top_p * 0x1p62) : 0ull);
}
// u * (the set's sum); non-decreasing in the sum
__device__ __forceinline__ unsigned long long draw_threshold(float u, unsigned long long total)
{
    return u > 0.0f ? (unsigned long long)fmin((double)u * (double)total, 1.8e19) : 0ull;
}

// One block per row of probabilities p: the set runs through the first entry
// whose running sum exceeds top_p; the pick is the first entry whose running
// sum exceeds u times the set's sum, or the set's last entry when none does.
__global__ __launch_bounds__(kSampT) void k_top_p(int *__restrict__ out, const float *__restrict__ p, int n,
                                                  float top_p, const float *__restrict__ u)
{
    __shared__ TopPShared S;
    const float *pb = p + (size_t)blockIdx.x * n;
    auto ld = [&](int i) { return __float_as_uint(pb[i]); };
    unsigned long long above, all;
    const int c = weighted_select<kSampT>(ld, n, cut_threshold(top_p), S, 0, 0u, 0ull, &above, &all);
    const unsigned long long total = c >= 0 ? above + fixp(pb[c]) : all;
    const unsigned long long R = draw_threshold(u[blockIdx.x], total);
    int pick = -1;
    if (R < total) {
        unsigned long long a2, all2;
        pick = weighted_select<kSampT>(ld, n, R, S, 0, 0u, 0ull, &a2, &all2);
    }
    if (pick < 0)
        pick = c >= 0 ? c : last_entry<kSampT>(pb, n, S);
    if (threadIdx.x == 0)
        out[blockIdx.x] = pick;
}

// ---- long rows: a row over kSlices blocks --------------------------------------
// Bound by latency (a 128k-entry row is 0.5 MB; the passes wait on loads,
// barriers and each other).  One block walks such a row ten times, at a
// fraction of what a CU can load, and leaves the other CUs idle; here each step
// of the same computation is a launch of kSlices blocks per row, and after the
// first pass only the few entries in the buckets of the two crossings are
// looked at again (8 rows of 128256: 194 us on one block each, 44 so, of which
// k_row_bins 6, k_row_gather 6 and k_row_pick 16).  The
// results are the same bits: the
// maximum and the 62-bit sums do not depend on the order, and the sum of the
// exponentials keeps k_probs's (block j sums, row by row of kSampT entries,
// the 64 columns that wave j of k_probs's block sums).
constexpr int kSlices = kSampT / kWave;
static_assert(kSlices == 16, "one block per wave of k_probs");

// The buckets that can hold the two crossing entries: at descending positions
// `cut` (the set's last entry; INT32_MAX: the set is every entry) and lo .. hi
// (the pick; lo > hi: the set's last entry).  The set's sum is known to within
// the cut bucket, so the draw's threshold, which grows with it, lies between
// those of the two ends.
struct PickBins {
    int cut, lo, hi, pad;
    unsigned long long all, cut_above, lo_above;   // the row's sum, the sums before those buckets
};

// a row's scratch besides its probabilities
struct alignas(16) RowScratch {
    unsigned long long hist[kSelBins];
    float pmax[kSlices], psum[kSlices];
    // candidates found by each wave of each block, their place in the row's
    // list, and the row's
    int cnt[kSlices * kSlices], at[kSlices * kSlices], total;
    PickBins bins;
};

template <bool BF16>
__device__ __forceinline__ float logit(const void *logits, size_t i)
{
    return BF16 ? bf16_to_f32(((const uint16_t *)logits)[i]) : ((const float *)logits)[i];
}

// the slices' maxima; clears the row's buckets for k_row_hist and the count of
// its candidates for k_row_gather
template <bool BF16>
__global__ __launch_bounds__(kSampT) void k_row_max(RowScratch *__restrict__ rs, const void *__restrict__ logits, int n)
{
    __shared__ float red[kSampT / 64];
    const int b = blockIdx.y, tid = threadIdx.x;
    RowScratch &R = rs[b];
    for (int i = blockIdx.x * (kSelBins / kSlices) + tid; i < (int)(blockIdx.x + 1) * (kSelBins / kSlices); i += kSampT)
        R.hist[i] = 0ull;
    if (blockIdx.x == 0 && tid == 0)
        R.total = 0;
    int c0, c1;
    slice_of(n, blockIdx.x, kSlices, kSampT, c0, c1);
    float m = -INFINITY;
    const size_t row = (size_t)b * n + c0;
    strided_batches<8>(c1 - c0, [&](int i) { return logit<BF16>(logits, row + i); },
                       [&](int, float v) { m = fmaxf(m, v); });
    m = block_reduce(m, red, true);
    if (tid == 0)
        R.pmax[blockIdx.x] = m;
}

// e_i = expf((x_i - max) / temp) and the sum over this block's 64 columns: for
// each column in ascending order, then over the columns as wave_sum does
constexpr int kExpRows = 128;   // rows of kSampT entries per round
template <bool BF16>
__global__ __launch_bounds__(kSampT) void k_row_exp(float *__restrict__ p, RowScratch *__restrict__ rs,
                                                    const void *__restrict__ logits, int n, float temp,
                                                    bool max_from_first)
{
    __shared__ float e[kExpRows][kWave];
    const int b = blockIdx.y, lane = threadIdx.x & (kWave - 1), wave = wave_id();
    RowScratch &R = rs[b];
    const size_t row = (size_t)b * n;
    float m = max_from_first ? logit<BF16>(logits, row) : -1e9f;
    for (int j = 0; j < kSlices; j++)
        m = fmaxf(m, R.pmax[j]);
    const int col = blockIdx.x * kWave + lane;
    float s = 0.0f;
    for (int r0 = 0; r0 * kSampT < n; r0 += kExpRows) {
        constexpr int U = kExpRows / kSlices;
        float v[U];
#pragma unroll
        for (int j = 0; j < U; j++) {
            const int i = (r0 + wave + kSlices * j) * kSampT + col;
            v[j] = logit<BF16>(logits, row + (i < n ? i : 0));
        }
#pragma unroll
        for (int j = 0; j < U; j++) {
            const int r = wave + kSlices * j, i = (r0 + r) * kSampT + col;
            if (i < n)
                p[row + i] = e[r][lane] = expf(__fdiv_rn(v[j] - m, temp));
        }
        __syncthreads();
        if (wave == 0) {
            const int rows = min(kExpRows, (n - col + kSampT - 1) / kSampT - r0);
#pragma unroll 16
            for (int r = 0; r < rows; r++)
                s += e[r][lane];
        }
        __syncthreads();
    }
    if (wave == 0) {
        s = wave_sum(s);
        if (lane == 0)
            R.psum[blockIdx.x] = s;
    }
}

__device__ __forceinline__ float row_sum(const RowScratch &R)
{
    float s = R.psum[0];
    for (int w = 1; w < kSlices; w++)
        s = s + R.psum[w];
    return s;
}

// p_i = e_i / sum, and the first pass's bucket sums of the row
__global__ __launch_bounds__(kSampT) void k_row_hist(float *__restrict__ p, RowScratch *__restrict__ rs, int n)
{
    __shared__ unsigned long long hist[kSelBins];
    const int b = blockIdx.y;
    RowScratch &R = rs[b];
    for (int i = threadIdx.x; i < kSelBins; i += kSampT)
        hist[i] = 0ull;
    const float s = row_sum(R);
    int c0, c1;
    slice_of(n, blockIdx.x, kSlices, kSampT, c0, c1);
    float *pb = p + (size_t)b * n + c0;
    __syncthreads();
    strided_batches<8>(c1 - c0, [&](int i) { return pb[i]; }, [&](int i, float v) {
        const float q = __fdiv_rn(v, s);
        pb[i] = q;
        const unsigned k = __float_as_uint(q);
        const unsigned long long f = fixp_bits(k);
        if (f)
            atomicAdd(&hist[(k >> kSelShift[0]) & (kSelBins - 1)], f);
    });
    __syncthreads();
    for (int i = threadIdx.x; i < kSelBins; i += kSampT)
        if (hist[i])
            atomicAdd(&R.hist[i], hist[i]);
}

__global__ __launch_bounds__(kSampT) void k_row_bins(RowScratch *__restrict__ rs, float top_p,
                                                     const float *__restrict__ u)
{
    __shared__ TopPShared S;
    RowScratch &R = rs[blockIdx.x];
    const float uu = u[blockIdx.x];
    const BinScan r = scan_bins<kSampT>(R.hist, kSelBins, S);
    __syncthreads();
    PickBins q;
    unsigned long long a;
    q.all = S.total;
    q.cut = crossing_bin(r, 0ull, cut_threshold(top_p), S, 0, &q.cut_above);
    unsigned long long least = q.all, most = q.all;
    if (q.cut != INT32_MAX) {
        if ((int)threadIdx.x == q.cut / 4)
            S.total = q.cut_above + r.h[q.cut & 3];
        __syncthreads();
        least = q.cut_above;
        most = S.total;
    }
    q.lo = crossing_bin(r, 0ull, draw_threshold(uu, least), S, 1, &q.lo_above);
    q.hi = min(crossing_bin(r, 0ull, draw_threshold(uu, most), S, 2, &a), q.cut);
    if (threadIdx.x == 0)
        R.bins = q;
}

// Each wave lists the entries of those buckets in its slice, in ascending
// order, as (bits << 32 | index), in a run of the row's list that it claims
// after it has counted them.  The list holds kCandMax entries, as many as
// k_row_pick takes: past that nothing is written.
constexpr int kCandMax = 4096;
__global__ __launch_bounds__(kSampT) void k_row_gather(unsigned long long *__restrict__ cand,
                                                       RowScratch *__restrict__ rs, const float *__restrict__ p,
                                                       int n)
{
    const int b = blockIdx.y, lane = threadIdx.x & (kWave - 1);
    RowScratch &R = rs[b];
    const int cut = R.bins.cut, lo = R.bins.lo, hi = R.bins.hi;
    const int part = blockIdx.x * kSlices + wave_id();
    int c0, c1, cnt = 0;
    slice_of(n, part, kSlices * kSlices, kWave, c0, c1);
    const float *pb = p + (size_t)b * n;
    auto ld = [&](int i) { return __float_as_uint(pb[i]); };
    auto wanted = [&](int a, unsigned k) {
        const int d = kSelBins - 1 - (int)(k >> kSelShift[0]);   // negative for patterns above 1
        return a + lane < c1 && d >= 0 && (d == cut || (d >= lo && d <= hi));
    };
    wave_steps<8, unsigned>(ld, c0, c1, [&](int a, unsigned k) {
        cnt += __popcll(__ballot(wanted(a, k)));
        return false;
    });
    int at = 0;
    if (lane == 0) {
        at = cnt ? atomicAdd(&R.total, cnt) : 0;
        R.cnt[part] = cnt;
        R.at[part] = at;
    }
    at = __builtin_amdgcn_readfirstlane(at);
    if (cnt == 0 || at + cnt > kCandMax)
        return;
    unsigned long long *cb = cand + (size_t)b * kCandMax + at;
    wave_steps<8, unsigned>(ld, c0, c1, [&](int a, unsigned k) {
        const bool in = wanted(a, k);
        const unsigned long long m = __ballot(in);
        if (in)
            cb[__popcll(m & ((1ull << lane) - 1))] = (unsigned long long)k << 32 | (unsigned)(a + lane);
        cb += __popcll(m);
        return false;
    });
}

// The draw over the listed entries, one block per row: few enough for LDS, and
// a small block, whose many barriers are cheap.  Where they are too many
// (equal or nearly equal logits) the passes read the whole row instead.
constexpr int kPickT = 512;
struct TopPPick : SelShared<1 << kSelBits[1]> {
    alignas(16) int start[kSlices * kSlices];
};
static_assert((1 << kSelBits[1]) >= kPickT && (1 << kSelBits[1]) <= 4 * kPickT && kSelBits[2] <= kSelBits[1], "buckets of the later passes");
__global__ __launch_bounds__(kPickT) void k_row_pick(int *__restrict__ out, const unsigned long long *__restrict__ cand,
                                                     const RowScratch *__restrict__ rs, const float *__restrict__ p,
                                                     int n, float top_p, const float *__restrict__ u)
{
    __shared__ unsigned bits[kCandMax], idx[kCandMax];
    __shared__ TopPPick S;
    constexpr int parts = kSlices * kSlices, NW = kPickT / kWave;
    const int b = blockIdx.x, lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const RowScratch &R = rs[b];
    const PickBins q = R.bins;
    const float uu = u[b];
    const float *pb = p + (size_t)b * n;
    const unsigned long long *cb = cand + (size_t)b * kCandMax;
    // the parts' places in the list; a wave copies parts wave, wave + NW, ...
    const int total = R.total;
    const bool listed = total <= kCandMax;
    if (wave == 0) {
        const int4 c = *(const int4 *)&R.cnt[4 * lane];
        int v = c.x + c.y + c.z + c.w, incl = v;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int a = __shfl_up(incl, o, kWave);
            incl += lane >= o ? a : 0;
        }
        *(int4 *)&S.start[4 * lane] = make_int4(incl - v, incl - v + c.x, incl - v + c.x + c.y, incl - c.w);
    }
    __syncthreads();
    if (listed)
        for (int i0 = wave; i0 < parts; i0 += NW * 8) {
            unsigned long long c[8];
            int cnt[8], c0[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                c0[j] = R.at[i0 + NW * j];
                cnt[j] = R.cnt[i0 + NW * j];
                c[j] = lane < cnt[j] ? cb[c0[j] + lane] : 0ull;
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int at = S.start[i0 + NW * j];
                for (int i = lane; i < cnt[j]; i += kWave) {
                    const unsigned long long e = i == lane ? c[j] : cb[c0[j] + i];
                    bits[at + i] = (unsigned)(e >> 32);
                    idx[at + i] = (unsigned)e;
                }
            }
        }
    __syncthreads();
    auto prefix = [&](int pos) { return (unsigned)(kSelBins - 1 - pos) << kSelShift[0]; };
    auto draw = [&](auto &&ld, int m) {
        unsigned long long above, unused, set = q.all;
        int c = -1;
        if (q.cut != INT32_MAX) {
            c = weighted_select<kPickT>(ld, m, cut_threshold(top_p), S, 1, prefix(q.cut), q.cut_above, &above, &unused);
            if (c < 0)
                return -1;
            set = above + fixp_bits(ld(c));
        }
        const unsigned long long T = draw_threshold(uu, set);
        if (T >= set)
            return c;
        // the pick's bucket among lo .. hi
        int pos = q.lo;
        unsigned long long base = q.lo_above;
        for (; pos < q.hi; pos += kWave) {
            const int d = min(pos + lane, q.hi);
            const unsigned long long h = pos + lane <= q.hi ? R.hist[kSelBins - 1 - d] : 0ull;
            unsigned long long incl = h;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const unsigned long long a = shfl_up_u64(incl, o);
                incl += lane >= o ? a : 0ull;
            }
            const unsigned long long over = __ballot(h && base + incl > T);
            if (over) {
                const int l = __ffsll(over) - 1;
                pos += l;
                base += shfl_u64(incl - h, l);
                break;
            }
            base += shfl_u64(incl, kWave - 1);
        }
        return weighted_select<kPickT>(ld, m, T, S, 1, prefix(pos), base, &above, &unused);
    };
    int pick;
    if (listed) {
        pick = draw([&](int i) { return bits[i]; }, total);
        if (pick >= 0)
            pick = (int)idx[pick];
    } else {
        pick = draw([&](int i) { return __float_as_uint(pb[i]); }, n);
    }
    if (pick < 0)   // no cut and the draw above every sum: the smallest entry
        pick = last_entry<kPickT>(pb, n, S);
    if (threadIdx.x == 0)
        out[b] = pick;
}

// p_i = e_i / sum and, for the running sums of block_first_exceeding, the sum
// of each step of 64 entries of each of its 16 ranges.
__global__ __launch_bounds__(kSampT) void k_row_steps(float *__restrict__ p, const RowScratch *__restrict__ rs,
                                                      float *__restrict__ steps, int n)
{
    const int b = blockIdx.y, lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const float s = row_sum(rs[b]);
    int c0, c1;
    slice_of(n, blockIdx.x, kSlices, kWave, c0, c1);
    float *pb = p + (size_t)b * n;
    const int per = (n + kWave - 1) / kWave + kSlices;   // steps of a row, the ranges' last ones short
    float *sb = steps + (size_t)b * per;
    for (int a = c0 + wave * kWave; a < c1; a += kSampT) {
        const int i = a + lane;
        float v = 0.0f;
        if (i < c1)
            pb[i] = v = __fdiv_rn(pb[i], s);
        const float t = lane63(wave_prefix_sum(v));
        if (lane == 0)
            sb[a / kWave] = t;
    }
}

// The temperature draw from the steps' sums: wave w carries its range's
// running sum from step to step as block_first_exceeding does and looks into
// the steps that can hold a crossing.  Their running sums differ from carry +
// step by a few roundings only.
__global__ __launch_bounds__(kSampT) void k_row_walk(int *__restrict__ out, const float *__restrict__ p,
                                                     const float *__restrict__ steps, int n,
                                                     const float *__restrict__ r)
{
    __shared__ float sh[kSlices];
    __shared__ int found;
    const int b = blockIdx.x, lane = threadIdx.x & (kWave - 1), wave = wave_id();
    int c0, c1;
    slice_of(n, wave, kSlices, kWave, c0, c1);
    const float *pb = p + (size_t)b * n;
    const int per = (n + kWave - 1) / kWave + kSlices;
    const float *sb = steps + (size_t)b * per + c0 / kWave;
    const int ns = (c1 - c0 + kWave - 1) / kWave;
    const float thr = r[b];
    // f(step, its sum): true to stop; 64 steps' sums are loaded at a time
    auto walk = [&](auto &&f) {
        for (int k0 = 0; k0 < ns; k0 += kWave) {
            const float t = k0 + lane < ns ? sb[k0 + lane] : 0.0f;
            const int m = min(kWave, ns - k0);
            for (int k = 0; k < m; k++)
                if (f(k0 + k, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t), k))))
                    return;
        }
    };
    float carry = 0.0f;
    walk([&](int, float t) {
        carry += t;
        return false;
    });
    if (lane == 0)
        sh[wave] = carry;
    if (threadIdx.x == 0)
        found = INT32_MAX;
    __syncthreads();
    carry = 0.0f;
    for (int w = 0; w < wave; w++)
        carry += sh[w];
    walk([&](int k, float t) {
        if (!(carry + t * 1.00001f < thr * 0.99999f)) {
            const int a = c0 + k * kWave;
            const float ps = wave_prefix_sum(a + lane < c1 ? pb[a + lane] : 0.0f);
            const unsigned long long m = __ballot(carry + ps > thr);
            if (m) {
                if (lane == 0)
                    atomicMin(&found, a + __ffsll(m) - 1);
                return true;
            }
        }
        carry += t;
        return false;
    });
    __syncthreads();
    if (threadIdx.x == 0)
        out[b] = found == INT32_MAX ? n - 1 : found;
}

// Rows go over kSlices blocks where the rows alone leave CUs idle and are long
// enough to pay for the launches: one block / kSlices blocks, top-p us a call,
// 16384 entries: 41 / 31 (1 row), 44 / 37 (16 rows), 45 / 54 (64); 32768: 61 / 33
// (1 row), 68 / 58 (64 rows); 65536: 104 / 35, 114 / 64; 128256: 186 / 38, 204 / 77
// (277 / 190 at 250 rows); temperature at 16384: 14 / 18, 32768: 25 / 18, 27.3 /
// 27.7, 128256: 86 / 31, 99 / 56.  One line for both, where no row count loses
// yet: it is temperature's, and top-p's for few rows lies lower.  The gain
// shrinks with the rows: at most one row per 512 entries.
static bool long_rows(int n, int batch) { return n >= 32768 && batch <= n / 512 && batch <= 65535; }

// maxima and exponentials of the rows (long_rows): p = e, not yet divided
static int row_exp_launch(float *p, RowScratch *rs, const void *logits, bool bf16, int n, int batch, float temp,
                          bool max_first, hipStream_t s)
{
    const dim3 g(kSlices, batch), t(kSampT);
    if (bf16) {
        hipLaunchKernelGGL(k_row_max<true>, g, t, 0, s, rs, logits, n);
        hipLaunchKernelGGL(k_row_exp<true>, g, t, 0, s, p, rs, logits, n, temp, max_first);
    } else {
        hipLaunchKernelGGL(k_row_max<false>, g, t, 0, s, rs, logits, n);
        hipLaunchKernelGGL(k_row_exp<false>, g, t, 0, s, p, rs, logits, n, temp, max_first);
    }
    BE42_LAUNCH_CHECK();
    return BE42_OK;
}

int probs_launch(float *p, const void *logits, bool bf16, int n, int batch, float temp, bool max_first,
                 hipStream_t s)
{
    if (bf16)
        hipLaunchKernelGGL(k_probs<true>, dim3(batch), dim3(kSampT), 0, s, p, logits, n, temp, max_first);
    else
        hipLaunchKernelGGL(k_probs<false>, dim3(batch), dim3(kSampT), 0, s, p, logits, n, temp, max_first);
    BE42_LAUNCH_CHECK();
    return BE42_OK;
}

}  // namespace be42

using namespace be42;

// logits_bf16: logits are bf16 (the reference's DTYPE_BF16 tensors)
extern "C" int be42_sample_temperature_dt(int *out, const void *logits, int logits_bf16, int n, int batch, float temp,
                                          const float *r, void *stream)
{
    BE42_CHECK(out && logits && r, "be42_sample_temperature: null pointer");
    BE42_CHECK(n > 0 && batch > 0, "be42_sample_temperature: n %d, batch %d", n, batch);
    hipStream_t s = as_stream(stream);
    const size_t rsb = sizeof(RowScratch) * (size_t)batch, pb = (size_t)n * batch * 4;
    const size_t per = (size_t)(n + kWave - 1) / kWave + kSlices;
    // without the memory: one block per row, which needs pb
    if (uint8_t *ws = long_rows(n, batch) ? (uint8_t *)workspace(rsb + pb + per * batch * 4, s) : nullptr) {
        RowScratch *rs = (RowScratch *)ws;
        float *p = (float *)(ws + rsb), *steps = (float *)(ws + rsb + pb);
        const int rc = row_exp_launch(p, rs, logits, logits_bf16 != 0, n, batch, temp, false, s);
        if (rc)
            return rc;
        hipLaunchKernelGGL(k_row_steps, dim3(kSlices, batch), dim3(kSampT), 0, s, p, rs, steps, n);
        hipLaunchKernelGGL(k_row_walk, dim3(batch), dim3(kSampT), 0, s, out, p, steps, n, r);
        BE42_LAUNCH_CHECK();
        return BE42_OK;
    }
    float *p = (float *)workspace(pb, s);
    if (!p)
        return BE42_ENOMEM;
    const int rc = probs_launch(p, logits, logits_bf16 != 0, n, batch, temp, false, s);
    if (rc)
        return rc;
    hipLaunchKernelGGL(k_pick_temperature, dim3(batch), dim3(kSampT), 0, s, out, p, n, r);
    BE42_LAUNCH_CHECK();
    return BE42_OK;
}

extern "C" int be42_sample_temperature(int *out, const float *logits, int n, int batch, float temp, const float *r,
                                       void *stream)
{
    return be42_sample_temperature_dt(out, logits, 0, n, batch, temp, r, stream);
}

extern "C" int be42_sample_top_p_dt(int *out, const void *logits, int logits_bf16, int n, int batch, float temp,
                                    float top_p, const float *u, void *stream)
{
    BE42_CHECK(out && logits && u, "be42_sample_top_p: null pointer");
    BE42_CHECK(n > 0 && batch > 0, "be42_sample_top_p: n %d, batch %d", n, batch);
    hipStream_t s = as_stream(stream);
    const size_t rsb = sizeof(RowScratch) * (size_t)batch, cb = (size_t)kCandMax * batch * 8, pb = (size_t)n * batch * 4;
    // without the memory: one block per row, which needs pb
    if (uint8_t *ws = long_rows(n, batch) ? (uint8_t *)workspace(rsb + cb + pb, s) : nullptr) {
        RowScratch *rs = (RowScratch *)ws;
        unsigned long long *cand = (unsigned long long *)(ws + rsb);
        float *p = (float *)(ws + rsb + cb);
        const int rc = row_exp_launch(p, rs, logits, logits_bf16 != 0, n, batch, temp, true, s);
        if (rc)
            return rc;
        const dim3 g(kSlices, batch), t(kSampT);
        hipLaunchKernelGGL(k_row_hist, g, t, 0, s, p, rs, n);
        hipLaunchKernelGGL(k_row_bins, dim3(batch), t, 0, s, rs, top_p, u);
        hipLaunchKernelGGL(k_row_gather, g, t, 0, s, cand, rs, p, n);
        hipLaunchKernelGGL(k_row_pick, dim3(batch), dim3(kPickT), 0, s, out, cand, rs, p, n, top_p, u);
        BE42_LAUNCH_CHECK();
        return BE42_OK;
    }
    float *p = (float *)workspace(pb, s);
    if (!p)
        return BE42_ENOMEM;
    const int rc = probs_launch(p, logits, logits_bf16 != 0, n, batch, temp, true, s);
    if (rc)
        return rc;
    hipLaunchKernelGGL(k_top_p, dim3(batch), dim3(kSampT), 0, s, out, p, n, top_p, u);
    BE42_LAUNCH_CHECK();
    return BE42_OK;
}

extern "C" int be42_sample_top_p(int *out, const float *logits, int n, int batch, float temp, float top_p,
                                 const float *u, void *stream)
{
    return be42_sample_top_p_dt(out, logits, 0, n, batch, temp, top_p, u, stream);
}
