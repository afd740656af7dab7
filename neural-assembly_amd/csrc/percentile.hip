// percentile.hip -- calibrate_percentile (quantize.c:89-132).
//
// The reference sorts a copy of the data with qsort and the comparator
// (a > b) - (a < b) (quantize.c:31-35, 99), takes clipped_min = sorted[lo],
// clipped_max = sorted[hi] with lo = (int64)(n p), hi = (int64)(n (1 - p))
// (clamped to [0, n - 1]; p outside [0, 0.5] taken as 0.01) and calibrates on
// that range with the same expressions as calibrate_minmax.
//
// Here the two order statistics are found on the device without sorting the
// data.  First a sampled select (select_sampled): 2048 sampled values, sorted
// by one block, bracket each rank; one pass over the data counts what lies
// below each bracket and copies the keys strictly inside it; a histogram over
// the copied keys narrows them to one bucket, which one block sorts.  The
// result is exact: the counts say where each rank lies, and a rank that its
// bracket missed, or copies that do not fit, send the call to the radix
// select below.  Data of up to 2048 values are sorted as they are.
//
// The radix select (select_ranks): each element maps to a 64-bit key that orders as the
// comparator does (-0 and +0 compare equal, so they share one key), and eight
// histogram passes -- 12 bits (sign and exponent), six of 8 bits, 4 bits; one
// histogram for each rank, counting only the elements that match the rank's
// prefix so far -- fix the keys digit by digit;
// once few elements match, their keys are copied out and the remaining
// passes read only those copies.  A one-block step after each pass picks the
// byte on the device, so the host waits once per call.
// Equal keys are equal doubles except for the zero key: the reference's qsort
// (glibc's merge sort, stable while its n * 8-byte copy fits in about a
// quarter of physical memory) keeps equal elements in input order, so a
// selected zero takes the sign of the j-th zero of the input, j the rank's
// position among the zeros; two more launches find it (zero counts per chunk,
// then one wave walks the chunk that holds it).  Beyond that size glibc falls
// back to an unstable in-place sort and the reference's zero sign no longer
// follows input order.  The parameter arithmetic then runs on the host in the
// reference's expressions.
//
// Divergences (the reference's behaviour is undefined there): a NaN
// percentile returns -1 (the reference indexes out of bounds); NaN data sort
// above +inf (the reference's comparator orders NaN inconsistently, so its
// result depends on the sort's internals).
#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "common.hpp"
#include "quant_common.hpp"
#include "reduce_impl.hpp"

namespace nh {

namespace {

constexpr int kPB = 256;               // threads per block
constexpr int64_t kZChunk = 1 << 16;   // elements per zero-count chunk

// Key ordering doubles as the comparator does; NaN takes the largest key.
// Integer selects only (no branch), so that loads can be hoisted past it.
__device__ __forceinline__ uint64_t pct_key_bits(uint64_t b)
{
    const uint64_t mag = b & ~(uint64_t(1) << 63);
    b = mag == 0 ? 0 : b;  // -0 -> +0: they compare equal
    const uint64_t k = (b >> 63) ? ~b : (b | (uint64_t(1) << 63));
    return mag > 0x7FF0000000000000ull ? ~uint64_t(0) : k;
}

constexpr uint64_t kZeroKey = uint64_t(1) << 63;  // key of +0 and of -0

double key_value(uint64_t k)
{
    if (k == ~uint64_t(0)) return std::nan("");
    const uint64_t b = (k >> 63) ? (k & ~(uint64_t(1) << 63)) : ~k;
    double v;
    std::memcpy(&v, &b, 8);
    return v;
}

constexpr int kPU = 8;                // elements per thread per tile (loads in flight)
constexpr int kTile = kPB * kPU;      // elements per block tile
constexpr int64_t kRegion = 2 * kTile; // copied keys per block, at most
constexpr int kPasses = 8;
constexpr int kMaxBins = 4096;

// Digits: the first pass takes the top 12 bits (sign and exponent), so that
// for most data few elements match after it; then 8-bit digits, and 4 last.
__host__ __device__ constexpr int pass_bits(int p) { return p == 0 ? 12 : (p == kPasses - 1 ? 4 : 8); }
__host__ __device__ constexpr int pass_shift(int p) { return p == 0 ? 52 : (p == kPasses - 1 ? 0 : 52 - 8 * p); }
static_assert(pass_shift(kPasses - 2) == 4 && pass_bits(kPasses - 2) == 8, "digits must tile the 64-bit key");

// h[d] += 1 for every lane with m set.  The first three distinct bytes of the
// wave each take one atomic for all their lanes (the leading passes see few
// distinct bytes: sign and exponent bits), the rest one atomic per lane.
__device__ __forceinline__ void hist_add(unsigned *h, bool m, unsigned d)
{
    uint64_t rem = __ballot(m);
#pragma unroll
    for (int it = 0; it < 3; it++) {
        if (rem == 0) return;
        const int leader = __builtin_ctzll(rem);
        const unsigned dl = __builtin_amdgcn_readlane(d, leader);
        const uint64_t same = __ballot(m && d == dl);
        if (int(threadIdx.x & 63) == leader) atomicAdd(&h[dl], unsigned(__popcll(same)));
        m = m && d != dl;
        rem &= ~same;
    }
    if (m) atomicAdd(&h[d], 1u);
}

// Select state, in device memory, carried from pass to pass.
struct PctState {
    uint64_t pre[2];   // key prefixes of the two ranks (bytes fixed so far)
    uint64_t mask;     // bits of the key fixed so far
    int64_t rem[2];    // rank within the elements matching pre[q]
    int64_t matched;   // elements matching either prefix
    int cur;           // key buffer holding every matching element, -1: none
    int copy;          // this pass copies its matches into buffer dst
    int dst;
    int err;           // a rank fell outside its histogram (cannot happen)
};

// Fixed-size record the host reads at the end.
struct PctResult {
    uint64_t key[2];
    int64_t within[2];
    int err;
};

// The pass body.  KEYS = false: the doubles, block b taking tiles b, b + grid,
// ... of kTile elements.  KEYS = true: keys copied out by an earlier pass,
// block b reading its own region [b R, b R + cnt_in[b]).  h[0..nb) counts
// digit (key >> shift) & (nb - 1) of the elements whose key matches pre0
// under mask, h[nb..2 nb) likewise for pre1 (left at zero when pre1 == pre0:
// the two would be equal).  With out set, the elements matching either prefix are
// also copied to block b's region of out (slots below R) and cnt_out[b] is
// how many matched; above R only on a first copy from the doubles, which is
// then discarded.
template <bool KEYS>
__device__ __forceinline__ void pct_pass_body(const void *__restrict__ src, int64_t n,
                                              const unsigned *__restrict__ cnt_in, int64_t R, int shift,
                                              unsigned dmask, uint64_t mask, uint64_t pre0, uint64_t pre1, unsigned *h,
                                              unsigned &nout, uint64_t *__restrict__ out)
{
    const int lane = int(threadIdx.x & 63);
    const bool two = pre1 != pre0;
    int64_t t0, hi, step;
    if (KEYS) {
        t0 = int64_t(blockIdx.x) * R;
        hi = t0 + int64_t(cnt_in[blockIdx.x]);
        step = kTile;
    } else {
        t0 = int64_t(blockIdx.x) * kTile;
        hi = n;
        step = int64_t(gridDim.x) * kTile;
    }
    for (; t0 < hi; t0 += step) {
        uint64_t k[kPU];
        bool v[kPU];
        // Past the end a lane re-reads the last element (hi > t0 >= 0 here) and
        // is masked by v: unconditional loads stay in flight together.
#pragma unroll
        for (int u = 0; u < kPU; u++) {
            const int64_t i = t0 + u * kPB + int64_t(threadIdx.x);
            v[u] = i < hi;
            const int64_t ic = v[u] ? i : hi - 1;
            k[u] = KEYS ? static_cast<const uint64_t *>(src)[ic]
                        : __builtin_nontemporal_load(static_cast<const uint64_t *>(src) + ic);
        }
        if (!KEYS) {
#pragma unroll
            for (int u = 0; u < kPU; u++) k[u] = pct_key_bits(k[u]);
        }
        uint64_t bal[kPU];
#pragma unroll
        for (int u = 0; u < kPU; u++) {
            const bool m0 = v[u] && (k[u] & mask) == pre0;
            const bool m1 = v[u] && (k[u] & mask) == pre1;
            const unsigned d = unsigned(k[u] >> shift) & dmask;
            hist_add(h, m0, d);
            if (two) hist_add(h + dmask + 1, m1, d);
            bal[u] = __ballot(m0 || m1);
        }
        if (out) {
            // one slot reservation per wave and tile
            unsigned total = 0u;
#pragma unroll
            for (int u = 0; u < kPU; u++) total += unsigned(__popcll(bal[u]));
            if (total) {
                unsigned base = 0u;
                if (lane == 0) base = atomicAdd(&nout, total);
                base = __builtin_amdgcn_readfirstlane(base);
                const uint64_t below = (uint64_t(1) << lane) - 1;
#pragma unroll
                for (int u = 0; u < kPU; u++) {
                    const int64_t slot = int64_t(base) + __popcll(bal[u] & below);
                    if (((bal[u] >> lane) & 1) && slot < R) out[int64_t(blockIdx.x) * R + slot] = k[u];
                    base += unsigned(__popcll(bal[u]));
                }
            }
        }
    }
}

// One radix pass over the doubles or, once they exist, the copied keys; the
// prefixes and the copy decision come from the state the previous select
// step wrote.  Adds the block's counts into hist and, when copying, stores
// the block's match count into cnt[dst][b].
__global__ __launch_bounds__(kPB) void k_pct_pass(const double *__restrict__ x, int64_t n, int64_t R, int pass,
                                                   const PctState *__restrict__ st,
                                                   unsigned long long *__restrict__ hist, uint64_t *keys0,
                                                   uint64_t *keys1, unsigned *cnt0, unsigned *cnt1)
{
    __shared__ unsigned h[kMaxBins];
    __shared__ unsigned nout;
    const int shift = pass_shift(pass);
    const int nb = 1 << pass_bits(pass);
    const int nh = st->pre[1] != st->pre[0] ? 2 * nb : nb;
    for (int i = threadIdx.x; i < nh; i += kPB) h[i] = 0u;
    if (threadIdx.x == 0) nout = 0u;
    __syncthreads();
    const int cur = st->cur, dst = st->dst;
    uint64_t *out = st->copy ? (dst ? keys1 : keys0) : nullptr;
    if (cur >= 0)
        pct_pass_body<true>(cur ? keys1 : keys0, n, cur ? cnt1 : cnt0, R, shift, unsigned(nb - 1), st->mask,
                            st->pre[0], st->pre[1], h, nout, out);
    else
        pct_pass_body<false>(x, n, nullptr, R, shift, unsigned(nb - 1), st->mask, st->pre[0], st->pre[1], h, nout,
                             out);
    __syncthreads();
    for (int i = threadIdx.x; i < nh; i += kPB)
        if (h[i]) atomicAdd(&hist[i], (unsigned long long)h[i]);
    if (out && threadIdx.x == 0) (dst ? cnt1 : cnt0)[blockIdx.x] = nout;
}

// Initial state for ranks r0, r1 of n elements; clears the histogram.
__global__ __launch_bounds__(64) void k_pct_init(PctState *st, unsigned long long *hist, int64_t r0, int64_t r1,
                                                 int64_t n)
{
    for (int i = threadIdx.x; i < kMaxBins; i += 64) hist[i] = 0ull;
    if (threadIdx.x == 0) {
        PctState s;
        s.pre[0] = s.pre[1] = 0;
        s.mask = 0;
        s.rem[0] = r0;
        s.rem[1] = r1;
        s.matched = n;
        s.cur = -1;
        s.copy = 0;
        s.dst = 0;
        s.err = 0;
        *st = s;
    }
}

// After pass `pass`: fix each rank's digit from the histogram, take over the
// copied keys if every block's matches fitted its region, decide whether the
// next pass copies, clear the histogram.  One wave; lane l holds bins
// [l PER, (l + 1) PER) of each histogram in registers (PER = nb / 64, or 1 for
// the 16-bin last digit, lanes past the bins holding none); every lane
// computes the same new state from a scan over the lanes and lane 0 stores
// it.  The last pass also writes the result record (res, host-visible memory).
template <int PER>
__global__ __launch_bounds__(64) void k_pct_select(PctState *st, unsigned long long *hist, const unsigned *cnt0,
                                                   const unsigned *cnt1, int64_t g, int64_t R, int pass,
                                                   PctResult *res)
{
    const int lane = int(threadIdx.x);
    const int shift = pass_shift(pass), nb = 1 << pass_bits(pass);
    const bool mine = lane * PER < nb;  // this lane holds bins
    PctState s = *st;
    const bool same = s.pre[1] == s.pre[0];  // the pass built one histogram for both
    int64_t hb[2][PER];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const unsigned long long *hq = hist + (same ? 0 : nb * q) + lane * PER;
#pragma unroll
        for (int j = 0; j < PER; j++) hb[q][j] = mine ? int64_t(hq[j]) : 0;
    }
    // first copy from the doubles: did every block's matches fit its region?
    bool fits = true;
    if (s.copy && s.cur < 0) {
        const unsigned *c = s.dst ? cnt1 : cnt0;
        for (int64_t b = lane; b < g; b += 64) fits = fits && int64_t(c[b]) <= R;
        fits = __ballot(!fits) == 0;
    }
    if (mine) {
#pragma unroll
        for (int j = 0; j < PER; j++) {
            hist[lane * PER + j] = 0ull;
            if (!same) hist[nb + lane * PER + j] = 0ull;
        }
    }
    if (s.copy && fits) s.cur = s.dst;
    int64_t c[2] = {0, 0};
#pragma unroll
    for (int q = 0; q < 2; q++) {
        int64_t ls = 0;
#pragma unroll
        for (int j = 0; j < PER; j++) ls += hb[q][j];
        int64_t inc = ls;  // inclusive scan over the lanes
        for (int off = 1; off < 64; off <<= 1) {
            const int64_t t = __shfl_up(inc, off);
            if (lane >= off) inc += t;
        }
        const uint64_t hit = __ballot(s.rem[q] < inc);
        int d = 0;
        int64_t cnt = 0, below = 0;
        if (hit == 0) {
            s.err = 1;  // counts lost: cannot happen for a valid rank
        } else {
            // the first lane whose bins reach the rank holds it
            const int L = __builtin_ctzll(hit);
            below = inc - ls;
            int jj = PER - 1;
            bool found = false;
#pragma unroll
            for (int j = 0; j < PER; j++) {
                const bool here = !found && s.rem[q] < below + hb[q][j];
                if (here) {
                    jj = j;
                    cnt = hb[q][j];
                    found = true;
                }
                if (!found) below += hb[q][j];
            }
            d = __shfl(L * PER + jj, L);
            cnt = __shfl(cnt, L);
            below = __shfl(below, L);
        }
        c[q] = cnt;
        s.pre[q] |= uint64_t(d) << shift;
        s.rem[q] -= below;
    }
    s.matched = s.pre[0] == s.pre[1] ? c[0] : c[0] + c[1];
    s.mask |= uint64_t(nb - 1) << shift;
    // A run of consecutive matches of at most g R / 2 <= g kTile elements
    // covers at most g + 1 tiles, dealt round-robin: at most 2 tiles per
    // block, within a region of 2 (or, for small n, regions that hold a
    // block's whole share).
    s.copy = s.cur >= 0 || s.matched <= g * R / 2;
    s.dst = s.cur >= 0 ? 1 - s.cur : 0;
    if (lane != 0) return;
    *st = s;
    if (res) {
        PctResult r;
        for (int q = 0; q < 2; q++) {
            r.key[q] = s.pre[q];
            r.within[q] = s.rem[q];
        }
        r.err = s.err;
        *res = r;
    }
}

// counts[c] = zeros (either sign) in elements [c * kZChunk, (c + 1) * kZChunk).
__global__ __launch_bounds__(kPB) void k_pct_zero_count(const double *__restrict__ x, int64_t n,
                                                        unsigned *__restrict__ counts)
{
    const int64_t c0 = int64_t(blockIdx.x) * kZChunk;
    const int64_t c1 = c0 + kZChunk < n ? c0 + kZChunk : n;
    unsigned s = 0u;
    for (int64_t i = c0 + threadIdx.x; i < c1; i += kPB) s += x[i] == 0.0 ? 1u : 0u;
    __shared__ unsigned sh[kPB];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int off = kPB / 2; off > 0; off >>= 1) {
        if (int(threadIdx.x) < off) sh[threadIdx.x] += sh[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) counts[blockIdx.x] = sh[0];
}

// One wave walks [c0, c1) in order and stores the sign bit (0 / 1) of its
// j-th zero into *sign (j < the chunk's zero count, so the walk finds it).
__global__ __launch_bounds__(64) void k_pct_zero_pick(const double *__restrict__ x, int64_t c0, int64_t c1,
                                                      unsigned j, int *__restrict__ sign)
{
    const int lane = threadIdx.x;
    for (int64_t base = c0; base < c1; base += 64) {
        const int64_t i = base + lane;
        const bool z = i < c1 && x[i] == 0.0;
        const uint64_t m = __ballot(z);
        const unsigned cnt = unsigned(__popcll(m));
        if (j < cnt) {
            // lane holding the j-th set bit of m
            const uint64_t below = lane == 0 ? 0 : (m & ((uint64_t(1) << lane) - 1));
            if (z && unsigned(__popcll(below)) == j) *sign = __builtin_signbit(x[i]) ? 1 : 0;
            return;
        }
        j -= cnt;
    }
}

}  // namespace

// ---- the sampled select --------------------------------------------------------------

namespace {

constexpr int kFB = 1024;        // lanes of the one-block steps
constexpr int kSample = 2 * kFB; // sampled values
constexpr int kList = 4096;      // the most keys the last step looks at per rank
constexpr int kFineBins = 8192;  // buckets of the histogram over the copied keys

constexpr int64_t kMaxCopies = int64_t(1) << 22;

// How far the bracket of the rank at fraction f reaches to either side, in
// sampled values.
__host__ __device__ inline double sample_margin(double f) { return 4.0 * sqrt(kSample * f * (1.0 - f)) + 3.0; }

struct PctFast {
    double l[2], u[2];  // bracket of each rank
    // elements below l, equal to l, strictly inside, equal to u
    unsigned long long lt[2], eql[2], in[2], equ[2];
    unsigned long long kmin[2], kmax[2];  // keys of the elements strictly inside
    int bucket[2];      // the rank's bucket, -1: none to search
    int64_t rem[2];     // the rank's place in its bucket
    int64_t count[2];   // elements in its bucket
    unsigned long long bmin[2], bmax[2];  // smallest and largest key of a bucket too full to list
    unsigned listed[2];
    int bad;            // give up: the radix select answers
};

// What each block of the pass over the data saw, per rank, one array per value:
// the counts, the range of the keys strictly inside (as doubles), and the keys
// it copied.  (8192 waves adding into one record by atomics took 500 us.)
struct PctSeen {
    double *mn[2], *mx[2];
    unsigned *n[8];  // lt, eql, in, equ: rank 0, rank 1 each
    unsigned *copied;
};

// Ascending bitonic sort of kSample keys by kFB lanes, lane t holding keys 2 t
// and 2 t + 1: neighbours meet in registers, partners up to 64 apart by lane
// shuffles, beyond in LDS (10 of the 66 steps).  4096 keys with every step in
// LDS took 42 us with the sampling, 18 now.
__device__ void block_sort(uint64_t (&k)[2], uint64_t *lds)
{
    static_assert(kSample == 2 * kFB, "two keys per lane");
    const int i0 = 2 * int(threadIdx.x);
    for (int w = 2; w <= kSample; w <<= 1) {
        const bool up = (i0 & w) == 0;
        for (int j = w >> 1; j >= 2; j >>= 1) {
            const bool keep_min = ((i0 & j) == 0) == up;
            uint64_t o[2];
            if (j >= 128) {
                __syncthreads();
                lds[i0] = k[0];
                lds[i0 + 1] = k[1];
                __syncthreads();
                o[0] = lds[i0 ^ j];
                o[1] = lds[(i0 ^ j) + 1];
            } else {
#pragma unroll
                for (int e = 0; e < 2; e++) o[e] = __shfl_xor(static_cast<unsigned long long>(k[e]), j >> 1, 64);
            }
#pragma unroll
            for (int e = 0; e < 2; e++) k[e] = (k[e] < o[e]) == keep_min ? k[e] : o[e];
        }
        const bool swap = (k[0] > k[1]) == up;
        const uint64_t x = swap ? k[1] : k[0];
        k[1] = swap ? k[0] : k[1];
        k[0] = x;
    }
    __syncthreads();
    lds[i0] = k[0];
    lds[i0 + 1] = k[1];
    __syncthreads();
}

__device__ __forceinline__ double key_double(uint64_t k)
{
    return __longlong_as_double(static_cast<long long>((k >> 63) ? (k & ~(uint64_t(1) << 63)) : ~k));
}

// One block: sample, sort, bracket.  Sample i is element h(i) of the i-th of
// kSample equal slices (h a hash, so that no period of the data meets the
// slices).  The bracket of rank r reaches 4 standard deviations of the sample
// rank and 3 more to either side; past the sample's ends it is unbounded.
// n <= kSample: the sample is the data, and the block answers (res).
__global__ __launch_bounds__(kFB) void k_pct_sample(const double *__restrict__ x, int64_t n, int64_t r0, int64_t r1,
                                                    PctFast *st, unsigned *hist, PctResult *res, Ticket tk)
{
    __shared__ uint64_t k[kSample];
    const bool all = n <= kSample;
    uint64_t mine[2];
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const int i = 2 * int(threadIdx.x) + e;
        int64_t at = i;
        if (!all) {
            const int64_t a = int64_t(double(n) * i / kSample), b = int64_t(double(n) * (i + 1) / kSample);
            uint32_t h = uint32_t(i) * 2654435761u;
            h ^= h >> 15;
            h *= 2246822519u;
            h ^= h >> 13;
            at = a + int64_t((double(h) * 0x1p-32) * double(b - a));
        }
        const double v = x[at < n ? at : n - 1];
        // past the end of short data: above everything
        mine[e] = i < n ? pct_key_bits(static_cast<uint64_t>(__double_as_longlong(v))) : ~uint64_t(0);
    }
    block_sort(mine, k);
    if (all) {
        if (threadIdx.x == 0) {
            PctResult r;
            r.err = 0;
            for (int q = 0; q < 2; q++) {
                const int at = int(q ? r1 : r0);
                int lo = 0, hi = at;  // first place of the key
                while (lo < hi) {
                    const int mid = (lo + hi) / 2;
                    if (k[mid] < k[at]) lo = mid + 1;
                    else hi = mid;
                }
                r.key[q] = k[at];
                r.within[q] = at - lo;
            }
            *res = r;
            publish(tk);
        }
        return;
    }
    for (int i = threadIdx.x; i < 2 * kFineBins; i += kFB) hist[i] = 0u;
    if (threadIdx.x < 2) {  // a lane per rank
        const int q = int(threadIdx.x);
        const double f = (double(q ? r1 : r0) + 0.5) / double(n);
        const double dev = sample_margin(f);
        const double lo = floor(kSample * f - dev), hi = ceil(kSample * f + dev);
        const uint64_t kl = lo < 0.0 ? 0 : k[int(lo)], ku = hi > kSample - 1 ? 0 : k[int(hi)];
        st->l[q] = lo < 0.0 ? -__builtin_inf() : key_double(kl);
        st->u[q] = hi > kSample - 1 ? __builtin_inf() : key_double(ku);
        st->bmin[q] = ~0ull;
        st->bmax[q] = 0ull;
        st->bucket[q] = -1;
        st->rem[q] = st->count[q] = 0;
        st->listed[q] = 0u;
        // NaN data around a rank: give up
        const uint64_t nan = __ballot(kl == ~uint64_t(0) || ku == ~uint64_t(0));
        if (q == 0) st->bad = nan ? 1 : 0;
    }
}

__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v)
{
    for (int off = 32; off >= 1; off >>= 1) {
        const uint64_t o = __shfl_xor(static_cast<unsigned long long>(v), off, 64);
        v = o < v ? o : v;
    }
    return v;
}
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) { return ~wave_min_u64(~v); }

// The one pass over the data, tiles dealt round-robin.  Most elements lie
// between the two brackets: two compares and a ballot count them.  The others
// (a few percent) are packed into the wave's LDS queue and looked at 64 at a
// time: counted per rank with ballots, and the keys strictly inside either
// bracket copied to the block's region.  A NaN compares false and counts as
// above every bracket, where the comparator's order puts it.
// Bound by HBM: 50 M values (400 MB) in 66 us at p = 0.001; looking at the
// others in place took 87 (half the waves have one).
__global__ __launch_bounds__(kPB) void k_pct_scan(const double *__restrict__ x, int64_t n, int64_t R,
                                                  const PctFast *__restrict__ st, uint64_t *__restrict__ keys,
                                                  PctSeen seen)
{
    constexpr int W = kPB / 64;
    __shared__ unsigned nout;
    __shared__ double queue[W][64 * (kPU + 1)];
    __shared__ unsigned sn[W][8];
    __shared__ double sr[W][4];
    if (st->bad) return;  // set by an earlier launch: uniform
    if (threadIdx.x == 0) nout = 0u;
    __syncthreads();
    const int lane = int(threadIdx.x & 63), w = int(threadIdx.x >> 6);
    double *wq = queue[w];
    const double l0 = st->l[0], u0 = st->u[0], l1 = st->l[1], u1 = st->u[1];
    // brackets that meet leave nothing between them: um = inf
    const double um = u0 < l1 ? u0 : __builtin_inf();
    unsigned c[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // lt, eql, in, equ per rank; uniform over the wave
    double mn[2] = {__builtin_inf(), __builtin_inf()}, mx[2] = {-__builtin_inf(), -__builtin_inf()};
    const auto look = [&](double v) {  // one element per lane, NaN: none
        uint64_t inside = 0;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const double l = q ? l1 : l0, h = q ? u1 : u0;
            const bool iq = v > l && v < h;
            const uint64_t bq = __ballot(iq), el = __ballot(v == l);
            c[q] += __popcll(__ballot(v < l));
            c[2 + q] += __popcll(el);
            c[4 + q] += __popcll(bq);
            c[6 + q] += __popcll(__ballot(v == h) & ~el);  // l == u: one atom, counted once
            inside |= bq;
            mn[q] = __builtin_fmin(mn[q], iq ? v : __builtin_inf());
            mx[q] = __builtin_fmax(mx[q], iq ? v : -__builtin_inf());
        }
        if (inside) {
            unsigned base = 0u;
            if (lane == 0) base = atomicAdd(&nout, unsigned(__popcll(inside)));
            base = __builtin_amdgcn_readfirstlane(base);
            const int64_t slot = int64_t(base) + __popcll(inside & ((uint64_t(1) << lane) - 1));
            if (((inside >> lane) & 1) && slot < R)
                keys[int64_t(blockIdx.x) * R + slot] =
                    pct_key_bits(static_cast<uint64_t>(__double_as_longlong(v)));
        }
    };
    const auto settle = [] {  // the wave's queue writes before its reads, and back
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    int qn = 0;  // queued, uniform; below 64 between tiles
    for (int64_t t0 = int64_t(blockIdx.x) * kTile; t0 < n; t0 += int64_t(gridDim.x) * kTile) {
        double v[kPU];
        const bool full = t0 + kTile <= n;
#pragma unroll
        for (int u = 0; u < kPU; u++) {
            const int64_t i = t0 + u * kPB + int64_t(threadIdx.x);
            if (full || i < n) v[u] = __builtin_nontemporal_load(x + i);
            else v[u] = __builtin_nan("");  // counts nowhere
        }
#pragma unroll
        for (int u = 0; u < kPU; u++) {
            const bool mid = v[u] > um && v[u] < l1;
            const uint64_t other = __ballot(!mid);
            c[1] += 64 - unsigned(__popcll(other));
            if (other) {
                if (!mid)
                    wq[qn + int(__builtin_amdgcn_mbcnt_hi(uint32_t(other >> 32),
                                                          __builtin_amdgcn_mbcnt_lo(uint32_t(other), 0u)))] = v[u];
                qn += __popcll(other);
            }
        }
        if (qn >= 64) {
            settle();
            while (qn >= 64) {
                qn -= 64;
                look(wq[qn + lane]);
            }
            settle();
        }
    }
    settle();
    look(lane < qn ? wq[lane] : __builtin_nan(""));
#pragma unroll
    for (int q = 0; q < 2; q++) {
        for (int off = 32; off >= 1; off >>= 1) {
            mn[q] = __builtin_fmin(mn[q], __shfl_xor(mn[q], off, 64));
            mx[q] = __builtin_fmax(mx[q], __shfl_xor(mx[q], off, 64));
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < 8; i++) sn[w][i] = c[i];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            sr[w][q] = mn[q];
            sr[w][2 + q] = mx[q];
        }
    }
    __syncthreads();
    const int t = int(threadIdx.x), q = t & 1;
    if (t < 8) {
        unsigned sum = 0;
        for (int k = 0; k < W; k++) sum += sn[k][t];
        seen.n[t][blockIdx.x] = sum;
    } else if (t < 10) {
        double m = sr[0][q];
        for (int k = 1; k < W; k++) m = __builtin_fmin(m, sr[k][q]);
        seen.mn[q][blockIdx.x] = m;
    } else if (t < 12) {
        double m = sr[0][2 + q];
        for (int k = 1; k < W; k++) m = __builtin_fmax(m, sr[k][2 + q]);
        seen.mx[q][blockIdx.x] = m;
    } else if (t == 12) {
        seen.copied[blockIdx.x] = nout;  // above R: the copies did not fit
    }
}

// One block: the blocks' records into the state, a wave per value.
__global__ __launch_bounds__(kFB) void k_pct_fold(PctFast *st, PctSeen seen, int g, int64_t R)
{
    if (st->bad) return;  // uniform: this launch writes it after the barrier below, when every wave has read it
    const int lane = int(threadIdx.x & 63), w = int(threadIdx.x >> 6), q = w & 1;
    __syncthreads();
    constexpr int U = 16;  // loads in flight per lane
    if (w < 8) {
        unsigned long long sum = 0;
        for (int b = lane; b < g; b += 64 * U) {
            unsigned v[U];
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = b + 64 * u < g ? seen.n[w][b + 64 * u] : 0u;
#pragma unroll
            for (int u = 0; u < U; u++) sum += v[u];
        }
        for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
        if (lane == 0) (w < 2 ? st->lt : w < 4 ? st->eql : w < 6 ? st->in : st->equ)[q] = sum;
    } else if (w < 12) {
        // the smallest, or minus the largest; nothing inside: kmin > kmax (+inf, -inf)
        const bool low = w < 10;
        const double *from = low ? seen.mn[q] : seen.mx[q];
        double m = __builtin_inf();
        for (int b = lane; b < g; b += 64 * U) {
            double v[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                v[u] = b + 64 * u < g ? from[b + 64 * u] : (low ? __builtin_inf() : -__builtin_inf());
#pragma unroll
            for (int u = 0; u < U; u++) m = __builtin_fmin(m, low ? v[u] : -v[u]);
        }
        for (int off = 32; off >= 1; off >>= 1) m = __builtin_fmin(m, __shfl_xor(m, off, 64));
        if (lane == 0)
            (low ? st->kmin : st->kmax)[q] = pct_key_bits(static_cast<uint64_t>(__double_as_longlong(low ? m : -m)));
    } else if (w == 12) {
        bool over = false;
        for (int b = lane; b < g; b += 64 * U) {
            unsigned v[U];
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = b + 64 * u < g ? seen.copied[b + 64 * u] : 0u;
#pragma unroll
            for (int u = 0; u < U; u++) over = over || int64_t(v[u]) > R;
        }
        const uint64_t any = __ballot(over);
        if (lane == 0) st->bad = any ? 1 : 0;
    }
}

// Where rank r lies: 0 at l, 1 strictly inside, 2 at u, -1 outside the
// bracket; rel: its place there.
__device__ __forceinline__ int pct_place(const PctFast &s, int q, int64_t r, int64_t &rel)
{
    rel = r - int64_t(s.lt[q]);
    if (rel < 0) return -1;
    if (rel < int64_t(s.eql[q])) return 0;
    rel -= int64_t(s.eql[q]);
    if (rel < int64_t(s.in[q])) return 1;
    rel -= int64_t(s.in[q]);
    return rel < int64_t(s.equ[q]) ? 2 : -1;
}

// Buckets: (key - kmin) >> shift, below kFineBins.
__device__ __forceinline__ int pct_shift(uint64_t kmin, uint64_t kmax)
{
    const uint64_t range = kmax - kmin;
    const int bits = range ? 64 - __builtin_clzll(range) : 0;
    return bits > 13 ? bits - 13 : 0;
}
static_assert(kFineBins == 1 << 13, "pct_shift");

// Histogram of the copied keys strictly inside each rank's bracket: LDS
// counters (64 KiB a block), so that a value that recurs does not queue at one
// address (25000 equal outliers among 0.8% of 50 M values: 309 us with one
// global atomic per key, 10 so).  A wave per region.
__global__ __launch_bounds__(kFB) void k_pct_fine(const PctFast *__restrict__ st, int64_t R, int g,
                                                  const uint64_t *__restrict__ keys, const unsigned *__restrict__ cnt,
                                                  unsigned *hist)
{
    __shared__ unsigned h[2 * kFineBins];
    if (st->bad) return;
    for (int i = threadIdx.x; i < 2 * kFineBins; i += kFB) h[i] = 0u;
    __syncthreads();
    const uint64_t k0 = st->kmin[0], e0 = st->kmax[0], k1 = st->kmin[1], e1 = st->kmax[1];
    const int s0 = pct_shift(k0, e0), s1 = pct_shift(k1, e1);
    const int lane = int(threadIdx.x & 63);
    for (int b = int(blockIdx.x) * (kFB / 64) + int(threadIdx.x >> 6); b < g; b += int(gridDim.x) * (kFB / 64)) {
        const uint64_t *from = keys + int64_t(b) * R;
        const int n = int(cnt[b]);
#pragma unroll 4
        for (int i = lane; i < n; i += 64) {
            const uint64_t k = from[i];
            if (k >= k0 && k <= e0) atomicAdd(&h[(k - k0) >> s0], 1u);
            if (k >= k1 && k <= e1) atomicAdd(&h[kFineBins + ((k - k1) >> s1)], 1u);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * kFineBins; i += kFB)
        if (h[i]) atomicAdd(&hist[i], h[i]);
}

// One block: the bucket of each rank that lies strictly inside its bracket.
__global__ __launch_bounds__(kFB) void k_pct_bucket(PctFast *st, const unsigned *__restrict__ hist, int64_t r0,
                                                    int64_t r1)
{
    __shared__ int64_t sums[kFB / 64];
    if (st->bad) return;
    constexpr int PER = kFineBins / kFB;
    const int lane = int(threadIdx.x & 63), w = int(threadIdx.x >> 6);
    for (int q = 0; q < 2; q++) {
        int64_t rel;
        if (pct_place(*st, q, q ? r1 : r0, rel) != 1) continue;  // uniform
        unsigned h[PER];
        int64_t mine = 0;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            h[j] = hist[q * kFineBins + int(threadIdx.x) * PER + j];
            mine += h[j];
        }
        int64_t inc = mine;
        for (int off = 1; off < 64; off <<= 1) {
            const int64_t o = __shfl_up(static_cast<long long>(inc), off, 64);
            if (lane >= off) inc += o;
        }
        if (lane == 63) sums[w] = inc;
        __syncthreads();
        for (int i = 0; i < w; i++) inc += sums[i];
        int64_t before = inc - mine;
        if (rel >= before && rel < inc) {
#pragma unroll
            for (int j = 0; j < PER; j++) {
                if (rel >= before && rel < before + int64_t(h[j])) {
                    st->bucket[q] = int(threadIdx.x) * PER + j;
                    st->rem[q] = rel - before;
                    st->count[q] = int64_t(h[j]);
                }
                before += int64_t(h[j]);
            }
        }
        __syncthreads();
    }
}

// The keys of each rank's bucket, listed where they fit (kList per rank), else
// their smallest and largest.  A wave per region, and few blocks: an atomic on
// one address of device memory takes about 35 ns, so each block gathers in LDS
// and makes one per rank (one per block of 2048 took 280 us).
constexpr int kListBlocks = 64;
__global__ __launch_bounds__(kFB) void k_pct_list(PctFast *st, int64_t R, int g, const uint64_t *__restrict__ keys,
                                                  const unsigned *__restrict__ cnt, uint64_t *list)
{
    constexpr int W = kFB / 64;
    __shared__ uint64_t buf[2][kList], smn[2][W], smx[2][W];
    __shared__ int have[2], base[2];
    if (st->bad) return;
    const int lane = int(threadIdx.x & 63), w = int(threadIdx.x >> 6);
    if (threadIdx.x < 2) have[threadIdx.x] = 0;
    __syncthreads();
    uint64_t k0[2], k1[2], mn[2] = {~uint64_t(0), ~uint64_t(0)}, mx[2] = {0, 0};
    int want[2], sh[2];
    bool fits[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        k0[q] = st->kmin[q];
        k1[q] = st->kmax[q];
        want[q] = st->bucket[q];  // -1: matches nothing
        sh[q] = pct_shift(k0[q], k1[q]);
        fits[q] = st->count[q] <= kList;
    }
    for (int b = int(blockIdx.x) * W + w; b < g; b += int(gridDim.x) * W) {
        const uint64_t *from = keys + int64_t(b) * R;
        const int n = int(cnt[b]);
#pragma unroll 4
        for (int i = lane; i < n; i += 64) {
            const uint64_t k = from[i];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                if (k < k0[q] || k > k1[q] || int((k - k0[q]) >> sh[q]) != want[q]) continue;
                if (fits[q]) {
                    buf[q][atomicAdd(&have[q], 1)] = k;  // the whole bucket fits
                } else {
                    mn[q] = k < mn[q] ? k : mn[q];
                    mx[q] = k > mx[q] ? k : mx[q];
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const uint64_t lo = wave_min_u64(mn[q]), hi = wave_max_u64(mx[q]);
        if (lane == 0) {
            smn[q][w] = lo;
            smx[q][w] = hi;
        }
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const int q = int(threadIdx.x);
        uint64_t lo = ~uint64_t(0), hi = 0;
        for (int i = 0; i < W; i++) {
            lo = smn[q][i] < lo ? smn[q][i] : lo;
            hi = smx[q][i] > hi ? smx[q][i] : hi;
        }
        if (lo <= hi) {
            atomicMin(&st->bmin[q], static_cast<unsigned long long>(lo));
            atomicMax(&st->bmax[q], static_cast<unsigned long long>(hi));
        }
        base[q] = have[q] ? int(atomicAdd(&st->listed[q], unsigned(have[q]))) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; q++)
        for (int i = threadIdx.x; i < have[q]; i += kFB) list[q * kList + base[q] + i] = buf[q][i];
}

// One block: each rank's key and its place among the equal keys.  A listed
// key is the answer when as many keys below it and equal to it surround the
// rank's place; each lane counts for its own keys, after a histogram over the
// bucket's width has left the keys of one of its kSub parts.
__global__ __launch_bounds__(kFB) void k_pct_answer(const PctFast *st, const uint64_t *__restrict__ list, int64_t r0,
                                                    int64_t r1, PctResult *res, Ticket tk)
{
    constexpr int kSubBits = 12, kSub = 1 << kSubBits;
    __shared__ uint64_t k[kList], smn[kFB / 64], smx[kFB / 64];
    __shared__ unsigned sub[kSub], wsum[kFB / 64];
    __shared__ int left, part, part_before;
    __shared__ PctResult r;
    const bool bad = st->bad;
    if (threadIdx.x == 0) r.err = bad ? 2 : 0;
    for (int q = 0; q < 2 && !bad; q++) {
        int64_t rel;
        const int place = pct_place(*st, q, q ? r1 : r0, rel);
        if (place == 1 && st->count[q] <= kList) {  // uniform
            const int all = int(st->count[q]);
            rel = st->rem[q];
            const int sh = pct_shift(st->kmin[q], st->kmax[q]), ss = sh > kSubBits ? sh - kSubBits : 0;
            const uint64_t lo = st->kmin[q] + (uint64_t(st->bucket[q]) << sh);
            __syncthreads();  // the first rank's LDS has been read
            for (int i = threadIdx.x; i < kSub; i += kFB) sub[i] = 0u;
            if (threadIdx.x == 0) left = 0;
            __syncthreads();
            for (int i = threadIdx.x; i < all; i += kFB) atomicAdd(&sub[(list[q * kList + i] - lo) >> ss], 1u);
            __syncthreads();
            // exclusive prefix over the parts: kSub / kFB per lane
            unsigned h[kSub / kFB], mine_n = 0u;
#pragma unroll
            for (int j = 0; j < kSub / kFB; j++) {
                h[j] = sub[int(threadIdx.x) * (kSub / kFB) + j];
                mine_n += h[j];
            }
            unsigned inc = mine_n;
            for (int off = 1; off < 64; off <<= 1) {
                const unsigned o = __shfl_up(inc, off, 64);
                if (int(threadIdx.x & 63) >= off) inc += o;
            }
            if ((threadIdx.x & 63) == 63) wsum[threadIdx.x >> 6] = inc;
            __syncthreads();
            for (int i = 0; i < int(threadIdx.x >> 6); i++) inc += wsum[i];
            int64_t before = int64_t(inc) - int64_t(mine_n);
#pragma unroll
            for (int j = 0; j < kSub / kFB; j++) {
                if (rel >= before && rel < before + int64_t(h[j])) {  // one lane
                    part = int(threadIdx.x) * (kSub / kFB) + j;
                    part_before = int(before);
                }
                before += int64_t(h[j]);
            }
            __syncthreads();
            rel -= part_before;
            for (int i = threadIdx.x; i < all; i += kFB) {
                const uint64_t key = list[q * kList + i];
                if (int((key - lo) >> ss) == part) k[atomicAdd(&left, 1)] = key;
            }
            __syncthreads();
            const int m = left;
            // One value that recurs answers at once: counting is quadratic (7 M
            // values of which 3500 equal ones hold the rank, 240 us by the radix
            // select, took 400).
            uint64_t mn = ~uint64_t(0), mx = 0;
            for (int i = threadIdx.x; i < m; i += kFB) {
                mn = k[i] < mn ? k[i] : mn;
                mx = k[i] > mx ? k[i] : mx;
            }
            mn = wave_min_u64(mn);
            mx = wave_max_u64(mx);
            if ((threadIdx.x & 63) == 0) {
                smn[threadIdx.x >> 6] = mn;
                smx[threadIdx.x >> 6] = mx;
            }
            __syncthreads();
            for (int i = 0; i < kFB / 64; i++) {
                mn = smn[i] < mn ? smn[i] : mn;
                mx = smx[i] > mx ? smx[i] : mx;
            }
            if (mn == mx) {  // uniform
                if (threadIdx.x == 0) {
                    r.key[q] = mn;
                    r.within[q] = rel;
                }
                continue;
            }
            for (int i = threadIdx.x; i < m; i += kFB) {
                const uint64_t mine = k[i];
                int less = 0, eq = 0;
                for (int o = 0; o < m; o++) {
                    less += k[o] < mine ? 1 : 0;
                    eq += k[o] == mine ? 1 : 0;
                }
                if (rel >= less && rel < less + eq) {  // equal keys write the same
                    r.key[q] = mine;
                    r.within[q] = rel - less;
                }
            }
        } else if (threadIdx.x == 0) {
            if (place == 1) {
                r.key[q] = st->bmin[q];
                r.within[q] = st->rem[q];
                if (st->bmin[q] != st->bmax[q]) r.err = 2;
            } else if (place >= 0) {
                r.key[q] = pct_key_bits(static_cast<uint64_t>(__double_as_longlong(place ? st->u[q] : st->l[q])));
                r.within[q] = rel;
            } else {
                r.err = 2;
            }
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        *res = r;
        publish(tk);
    }
}

}  // namespace

// The sampled select (seven launches, one for n <= kSample): 50 M Laplace values
// with outliers 318 -> 124 us per call at p = 0.001, 451 -> 151 at 0.01, 5 M 181 ->
// 68, 100 K 94 -> 52, 4096 91 -> 51, against the radix select alone (two full
// passes of 110 us and 15 short launches).  *done = false: the
// radix select has to answer.
static int select_sampled(const double *x, int64_t n, const int64_t r[2], uint64_t key[2], int64_t within[2],
                          bool *done)
{
    *done = false;
    const bool all = n <= kSample;
    const int64_t tiles = ceil_div(n, int64_t(kTile));
    int64_t g = int64_t(num_cus()) * 8;
    if (g > tiles) g = tiles;
    // The share of the data that the brackets are expected to hold: 0.5% at p =
    // 0.0001, 1% at 0.001, 4% at 0.01, 17% at 0.3.  Past kMaxCopies copied keys
    // a bucket outgrows the list and the call would be made twice (268 M values
    // at p = 0.01, some of them: 1210 us on average against 1966 for the radix
    // select; at p = 0.3 2718 against 2102), so the radix select takes it.
    double held = 0.0;
    for (int q = 0; q < 2; q++) held += 2.0 * sample_margin((double(r[q]) + 0.5) / double(n)) / kSample;
    if (!all && held * double(n) > double(kMaxCopies)) return NEURAL_OK;
    // A block's region: twice its expected copies and two tiles (a run of
    // matches in sorted data is dealt over the blocks tile by tile).
    const int64_t share = ceil_div(tiles, g);
    const int64_t reg = int64_t(double(share) * held * 2.0) + 2;
    const int64_t R = (reg < share ? reg : share) * kTile;
    // [state][hist 2 x kFineBins x u32][list 2 x kList x u64][records, counts: g each][keys g x R x u64]
    const size_t st_b = 512, hist_b = 2 * kFineBins * sizeof(unsigned), list_b = 2 * kList * sizeof(uint64_t);
    static_assert(sizeof(PctFast) <= 512, "state record");
    const size_t seen_off = st_b + hist_b + list_b;
    const size_t keys_off = (seen_off + size_t(g) * (4 * sizeof(double) + 9 * sizeof(unsigned)) + 255) / 256 * 256;
    char *ws = static_cast<char *>(dev_alloc(all ? st_b : keys_off + size_t(g * R) * sizeof(uint64_t)));
    if (!ws) return set_error(NEURAL_ERR_OUT_OF_MEMORY);
    auto *st = reinterpret_cast<PctFast *>(ws);
    auto *hist = reinterpret_cast<unsigned *>(ws + st_b);
    auto *list = reinterpret_cast<uint64_t *>(ws + st_b + hist_b);
    PctSeen seen;
    auto *sd = reinterpret_cast<double *>(ws + seen_off);
    auto *su = reinterpret_cast<unsigned *>(sd + 4 * g);
    for (int q = 0; q < 2; q++) {
        seen.mn[q] = sd + q * g;
        seen.mx[q] = sd + (2 + q) * g;
    }
    for (int i = 0; i < 8; i++) seen.n[i] = su + i * g;
    unsigned *cnt = seen.copied = su + 8 * g;
    auto *keys = reinterpret_cast<uint64_t *>(ws + keys_off);
    WsGuard wg;
    auto *res = static_cast<PctResult *>(workspace().host_result_dev);
    const Ticket tk = next_ticket();
    NH_LAUNCH(k_pct_sample, dim3(1), dim3(kFB), 0, stream(), x, n, r[0], r[1], st, hist, res, tk);
    if (!all) {
        NH_LAUNCH(k_pct_scan, dim3(unsigned(g)), dim3(kPB), 0, stream(), x, n, R, st, keys, seen);
        NH_LAUNCH(k_pct_fold, dim3(1), dim3(kFB), 0, stream(), st, seen, int(g), R);
        NH_LAUNCH(k_pct_fine, dim3(unsigned(ceil_div(g, int64_t(kFB / 64)))), dim3(kFB), 0, stream(), st, R, int(g), keys,
                  cnt, hist);
        NH_LAUNCH(k_pct_bucket, dim3(1), dim3(kFB), 0, stream(), st, hist, r[0], r[1]);
        NH_LAUNCH(k_pct_list, dim3(kListBlocks), dim3(kFB), 0, stream(), st, R, int(g), keys, cnt, list);
        NH_LAUNCH(k_pct_answer, dim3(1), dim3(kFB), 0, stream(), st, list, r[0], r[1], res, tk);
    }
    int rc = check_launch();
    PctResult out{};
    if (rc == NEURAL_OK) rc = host_result_wait(tk.value, &out, sizeof(out));
    dev_free(ws);
    if (rc != NEURAL_OK) return set_error(rc);
    *done = out.err == 0;
    for (int q = 0; q < 2; q++) {
        key[q] = out.key[q];
        within[q] = out.within[q];
    }
    return NEURAL_OK;
}

// Keys of the elements at ranks r[0], r[1] of the comparator's order, and the
// rank within its run of equal keys (rank - elements with a smaller key).
// Eight passes fix the keys a digit at a time, each followed by a one-block
// select step that updates the state on the device, so the host waits once.
// Once few enough elements match the two prefixes (at most half the copy
// area, so that a run of consecutive matches spread over the tiles fits every
// block's region), a pass also copies their keys out, and the later
// passes read only the copies, each copying its own matches on into the
// other buffer.
static int select_ranks(const double *x, int64_t n, const int64_t r[2], uint64_t key[2], int64_t within[2])
{
    const int64_t tiles = ceil_div(n, int64_t(kTile));
    int64_t g = int64_t(num_cus()) * 8;
    if (g > tiles) g = tiles;
    int64_t R = ceil_div(tiles, g) * kTile;
    if (R > kRegion) R = kRegion;
    // [state][hist kMaxBins x u64][counts 2 x g x u32][keys 2 x g x R x u64]
    const size_t st_b = 256, hist_b = kMaxBins * sizeof(unsigned long long), cnt_b = size_t(2 * g) * sizeof(unsigned);
    const size_t keys_off = (st_b + hist_b + cnt_b + 255) / 256 * 256;
    char *ws = static_cast<char *>(dev_alloc(keys_off + size_t(2 * g * R) * sizeof(uint64_t)));
    if (!ws) return set_error(NEURAL_ERR_OUT_OF_MEMORY);
    auto *st = reinterpret_cast<PctState *>(ws);
    auto *hist = reinterpret_cast<unsigned long long *>(ws + st_b);
    unsigned *cnt0 = reinterpret_cast<unsigned *>(ws + st_b + hist_b), *cnt1 = cnt0 + g;
    uint64_t *keys0 = reinterpret_cast<uint64_t *>(ws + keys_off), *keys1 = keys0 + g * R;
    static_assert(sizeof(PctResult) <= 256, "result record exceeds the host result area");
    WsGuard wg;
    auto *res = static_cast<PctResult *>(workspace().host_result_dev);
    NH_LAUNCH(k_pct_init, dim3(1), dim3(64), 0, stream(), st, hist, r[0], r[1], n);
    int rc = check_launch();
    for (int pass = 0; pass < kPasses && rc == NEURAL_OK; pass++) {
        NH_LAUNCH(k_pct_pass, dim3(unsigned(g)), dim3(kPB), 0, stream(), x, n, R, pass, st, hist, keys0,
                           keys1, cnt0, cnt1);
        rc = check_launch();
        if (rc != NEURAL_OK) break;
        PctResult *last = pass == kPasses - 1 ? res : nullptr;
        const int nb = 1 << pass_bits(pass);
        if (nb == 4096)
            NH_LAUNCH(k_pct_select<64>, dim3(1), dim3(64), 0, stream(), st, hist, cnt0, cnt1, g, R, pass, last);
        else if (nb == 256)
            NH_LAUNCH(k_pct_select<4>, dim3(1), dim3(64), 0, stream(), st, hist, cnt0, cnt1, g, R, pass, last);
        else
            NH_LAUNCH(k_pct_select<1>, dim3(1), dim3(64), 0, stream(), st, hist, cnt0, cnt1, g, R, pass, last);
        rc = check_launch();
    }
    PctResult out{};
    if (rc == NEURAL_OK) rc = host_result_fetch(&out, sizeof(out));
    dev_free(ws);
    if (rc != NEURAL_OK) return set_error(rc);
    if (out.err) return set_error(NEURAL_ERR_INTERNAL);  // counts lost: cannot happen for a valid rank
    for (int q = 0; q < 2; q++) {
        key[q] = out.key[q];
        within[q] = out.within[q];
    }
    return NEURAL_OK;
}

// Sign bit of the j-th zero of x in input order.
static int zero_sign(const double *x, int64_t n, int64_t j, int *sign_out)
{
    const int64_t nch = ceil_div(n, kZChunk);
    unsigned *counts = static_cast<unsigned *>(dev_alloc(size_t(nch) * sizeof(unsigned) + sizeof(int)));
    if (!counts) return set_error(NEURAL_ERR_OUT_OF_MEMORY);
    int *dsign = reinterpret_cast<int *>(counts + nch);
    std::vector<unsigned> c(static_cast<size_t>(nch));
    NH_LAUNCH(k_pct_zero_count, dim3(unsigned(nch)), dim3(kPB), 0, stream(), x, n, counts);
    int rc = check_launch();
    if (rc == NEURAL_OK &&
        hipMemcpyAsync(c.data(), counts, size_t(nch) * sizeof(unsigned), hipMemcpyDeviceToHost, stream()) != hipSuccess)
        rc = NEURAL_ERR_INTERNAL;
    if (rc == NEURAL_OK) rc = sync();
    int64_t ch = 0;
    if (rc == NEURAL_OK) {
        for (; ch < nch && j >= int64_t(c[size_t(ch)]); ch++) j -= int64_t(c[size_t(ch)]);
        if (ch == nch) rc = NEURAL_ERR_INTERNAL;
    }
    int sign = 0;
    if (rc == NEURAL_OK) {
        const int64_t c0 = ch * kZChunk, c1 = c0 + kZChunk < n ? c0 + kZChunk : n;
        NH_LAUNCH(k_pct_zero_pick, dim3(1), dim3(64), 0, stream(), x, c0, c1, unsigned(j), dsign);
        rc = check_launch();
        if (rc == NEURAL_OK && hipMemcpyAsync(&sign, dsign, sizeof(int), hipMemcpyDeviceToHost, stream()) != hipSuccess)
            rc = NEURAL_ERR_INTERNAL;
        if (rc == NEURAL_OK) rc = sync();
    }
    dev_free(counts);
    if (rc != NEURAL_OK) return set_error(rc);
    *sign_out = sign;
    return NEURAL_OK;
}

static int calibrate_pct(const double *data, int64_t n, double percentile, int symmetric, QuantParams *out)
{
    if (!data || n <= 0 || !out) return -1;
    if (percentile != percentile) return -1;
    if (percentile < 0.0 || percentile > 0.5) percentile = 0.01;
    if (ensure_init() != NEURAL_OK) return -1;
    if (stream_recording()) {  // the result cannot come back: refused before anything is recorded
        set_error(NEURAL_ERR_INTERNAL);
        return -1;
    }
    int64_t lo_idx = int64_t(double(n) * percentile);
    int64_t hi_idx = int64_t(double(n) * (1.0 - percentile));
    if (lo_idx < 0) lo_idx = 0;
    if (hi_idx >= n) hi_idx = n - 1;
    Staged s;
    if (s.open_n(data, uint64_t(n), sizeof(double), true) != NEURAL_OK) return -1;
    const double *x = static_cast<const double *>(s.dev);
    const int64_t ranks[2] = {lo_idx, hi_idx};
    uint64_t key[2];
    int64_t within[2];
    bool done = false;
    if (select_sampled(x, n, ranks, key, within, &done) != NEURAL_OK) return -1;
    if (!done && select_ranks(x, n, ranks, key, within) != NEURAL_OK) return -1;
    double v[2];
    for (int q = 0; q < 2; q++) {
        v[q] = key_value(key[q]);
        if (key[q] == kZeroKey) {
            int sign = 0;
            if (zero_sign(x, n, within[q], &sign) != NEURAL_OK) return -1;
            v[q] = sign ? -0.0 : 0.0;
        }
    }
    if (s.finish(false) != NEURAL_OK) return -1;
    // quantize.c:112-129: the epilogue shared with calibrate_minmax
    minmax_epilogue(v[0], v[1], symmetric, out);
    set_error(NEURAL_OK);
    return 0;
}

}  // namespace nh

extern "C" int calibrate_percentile(const double *data, int64_t n, double percentile, int symmetric,
                                    QuantParams *out)
{
    return nh::calibrate_pct(data, n, percentile, symmetric, out);
}
