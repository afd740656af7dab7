// losses.hip -- cross-entropy losses: label-smoothed CE forward / backward and
// a fused forward+backward, and the tensor cross-entropy loss.
//
// Reference: metrics_losses.c:28-125 (label_smoothing_ce_forward/backward,
// f64 logits, int64 targets):
//   m = max (strict compare from row[0]); lse = log(sum_c exp(x_c - m));
//   st_c = a/K + (c == t ? 1 - a : 0); loss_row = -sum_c st_c * ((x_c - m) - lse);
//   loss = sum_rows / B;   grad_c = (1/B) * (exp(x_c - m) / sum - st_c)
// and losses.asm:315-613 (cross_entropy_loss, intended semantics -- the C-ABI
// wrapper neural_api.asm:2546-2568 passes a Tensor* where a Node* is expected
// and never writes *loss): softmax per row, target index = truncation of the
// target tensor's value, loss = mean_rows(-log(p_target + 1e-7)); f32 rows
// keep the float roundings of e_j, of p_t and of each row's loss.
//
// A row sits in the VGPRs of 4 to 1024 lanes (one HBM read; the gradient
// written once), at any width and alignment up to 98304 f32 / 49152 f64
// classes; wider rows are read twice by a block of 1024.  Per-row losses land in a double buffer and are summed by the
// segmented reduction (fixed order, deterministic); the row sums of exp use a
// fixed wave tree instead of the reference's sequential order, so losses
// agree to a few ulps of the row terms, not bit for bit.  An invalid target
// sets a device flag and the call returns -1 (C API) / INVALID_ARGUMENT.
#include <cmath>

#include <type_traits>

#include "reduce_impl.hpp"
#include "row_group.hpp"

namespace nh {

enum { CE_LS_FWD = 1, CE_LS_BWD = 2, CE_LS_FUSED = 3, CE_ASM = 4 };

template <typename T>
NH_DEV bool loss_target(const int64_t *ti, const T *tv, int64_t r, int64_t cols, int64_t &t)
{
    if (ti) {
        t = ti[r];
        return t >= 0 && t < cols;
    }
    const T v = tv[r];
    if (!(v > T(-1) && v < T(cols))) return false;  // NaN fails too
    t = int64_t(v);                                  // truncation (cvttss2si / cvttsd2si)
    return true;
}

// e = exp(x - m) for one element: double exp for f64 rows; for f32 rows the
// hardware exp2 of (x - m) * log2(e) in float (m is the row's largest float,
// so float(m) is exact).  Relative error about (|x - m| + 1) * 1.2e-7 against
// the reference's float rounding of the exact value: the losses built on it
// stay within 2e-6 of the exact loss (the f32 bar), and the float gradients
// within 1e-5.  Exact-difference double range reduction was measured ~20%
// slower for the tensor loss kernel.
NH_DEV double row_exp_d(double x, double m) { return exp(x - m); }

// e^y for the one-wave-per-row forward's f64 rows, from a 64-entry table of
// 2^(j/64) that each block keeps in LDS: y = (64 k + j) ln2 / 64 + r with
// |r| <= ln2 / 128, e^r by its Taylor polynomial through r^5 (truncation
// below 4e-17 relative), scaled by 2^k with ldexp (exact, or rounded once
// into the denormal range).  About 3 ulp against the device library's ~1,
// in 17 instructions instead of ~24: the 1e-12 bars of the losses and
// gradients are 3e3 times wider.  y below -1100 is taken as -1100 (e^y is 0
// either way), +inf and overflow give +inf, a NaN stays NaN (through r).
constexpr double kLn2_64Hi = kLn2Hi / 64.0;  // n * kLn2_64Hi exact for |n| < 2^20
constexpr double kLn2_64Lo = kLn2Lo / 64.0;
NH_DEV double exp_tab(double y, const double *tab)
{
    y = y < -1100.0 ? -1100.0 : y;  // NaN compares false and stays
    const double n = __builtin_rint(y * 92.332482616893658);  // 64 / ln 2
    double r = __builtin_fma(-n, kLn2_64Hi, y);
    r = __builtin_fma(-n, kLn2_64Lo, r);
    const int ni = int(n);  // |n| <= 2^17 for finite y <= 1100; a NaN's r carries it
    double p = 1.0 / 120.0;
    p = __builtin_fma(p, r, 1.0 / 24.0);
    p = __builtin_fma(p, r, 1.0 / 6.0);
    p = __builtin_fma(p, r, 0.5);
    p = __builtin_fma(p, r, 1.0);
    p = __builtin_fma(p, r, 1.0);
    return __builtin_ldexp(tab[ni & 63] * p, ni >> 6);  // 2^floor(n / 64); beyond 2^1023: +inf
}
NH_DEV double row_exp_f(float x, double m)
{
    return double(__builtin_amdgcn_exp2f((x - float(m)) * 1.4426950408889634f));
}

struct CeArgs {
    const int64_t *tidx;   // int64 targets (label-smoothed API) or null
    const void *tval;      // target values of the logits' dtype (tensor API) or null
    int64_t rows, cols;
    double alpha, inv_n;
    double *row_loss;      // [rows] or null: p_t (tensor CE) or sum_c st_c (x_c - m) (label-smoothed)
    double *row_s;         // [rows] or null: sum_c exp(x_c - m) (label-smoothed forward)
    void *grad;            // [rows, cols] or null
    int *bad;              // set to 1 when a target is out of range
};

// The row loss is -sum_c st_c ((x_c - m) - lse) = lse * sum_c st_c - A with
// A = sum_c st_c (x_c - m) = st0 * sum_c (x_c - m) + (st1 - st0) (x_t - m)
// (st_c = st0 off the target, st1 on it): every term of the reference's sum
// has one sign (x_c - m <= 0, lse >= 0), and so have the two parts of A, so
// the regrouping changes only the last bits; the log moves out of the row
// kernel into the summing pass and the weights out of the element loop.

// Gradient element from e = exp(x_c - m): (1/B) (e / sum - st_c).  WIDE f32
// rows take it in double and round once; rows held by at most a wave in float.
template <typename T, bool WIDE>
struct CeGrad {
    double rs, st0, st1, inv_n;
    NH_DEV T operator()(T e, bool at_t) const
    {
        if constexpr (sizeof(T) == 4 && WIDE) {
            asm("" : "+v"(e));  // or the compiler keeps double(e) of the sum: two more registers per value
            return T(inv_n * (double(e) * rs - (at_t ? st1 : st0)));
        } else if constexpr (sizeof(T) == 4) {
            return float(inv_n) * (e * float(rs) - (at_t ? float(st1) : float(st0)));
        } else {
            return T(inv_n * (double(e) * rs - (at_t ? st1 : st0)));
        }
    }
};

// x_c - m as the row loss sums it.
template <typename T, bool WIDE>
NH_DEV double ce_diff(T x, double m)
{
    if constexpr (sizeof(T) == 4 && !WIDE) return double(x - float(m));
    else return double(x) - m;
}

// One row per group of NT lanes, VPT 16-byte vectors per lane and the values
// past the vectors in one scalar of the first lanes (RowCut; the
// other lanes' scalar is -inf and adds nothing).  FULL: the row is exactly NT * VPT vectors, so no
// element needs a bounds check (per-element checks around the exp turn into
// exec-mask branches).  e_c replaces x_c.  x_t is read again from memory, beside
// the row (a pick from the registers, with an exp of its own for the tensor
// loss: f64 [65536, 256] 44.0 us, now 40.0); the tensor loss's lane that holds the
// target keeps the e_t it computes.
//
// What bounds it: HBM where enough rows are in flight, so that one block loads
// or stores while another computes.  A 201 KB row of 50257 f32 classes is 25
// vectors for each of 512 lanes: 16 in registers and LV = 9 in LDS (72 KB; a
// lane reads and writes its own slots only), two blocks per CU.  With all 25
// in registers the compiler spilled 35-84 of them to scratch memory
// ([4096, 50257] fused f32 373 us against 318, both with stores cut at 64-byte
// boundaries; three passes of 4-byte accesses took 861); this form spills 4 in
// f32 and 11 in f64.  Rows of an odd width start anywhere, and a vector store
// that starts inside a 64-byte block is slower: 331 us there, 314 with each row
// cut at the first boundary of its own gradient.  But then the order of a row's
// sums, and so the result's last bits, went by the buffer's address; equal bits
// are promised.
//
// WAVES: the minimum waves per SIMD the compiler must fit (1: its own
// choice).  The f64 forward with rows of up to 1024 values takes 5 (no
// spills; 103 VGPRs and 4 waves otherwise when it was measured): 88.8-90.1 -> 82.9
// us at [65536,1024] (A/B in one run).  The fused and backward forms keep every
// exp for the gradient and spill under that bound (fused f64 180 -> 331 us),
// as do rows of 2048 doubles.
template <typename T, int NT, int VPT, int LV, int MODE, bool FULL, int WAVES>
__global__ __launch_bounds__(NT < 256 ? 256 : NT, WAVES) void k_ce_rows(const T *__restrict__ x, CeArgs a,
                                                                       int64_t r_base)
{
    using V = typename Vec16<T>::type;
    using U = typename VecU<T>::type;
    using G = RowGrp<NT>;
    constexpr int VN = Vec16<T>::n;
    constexpr int RPB = NT < 256 ? 256 / NT : 1;
    constexpr bool WIDE = NT > 64;
    constexpr bool LOSS = MODE == CE_LS_FWD || MODE == CE_LS_FUSED;
    constexpr bool GRAD = MODE == CE_LS_BWD || MODE == CE_LS_FUSED;
    // The f64 forward takes exp_tab (2^(j/64) by the device library's exp2,
    // in LDS): 85-90 -> 84-87 us at [65536,1024] (A/B in one run).  The modes
    // that keep every e for the gradient keep the library's exp: with the
    // table their longer-lived registers made the fused pass 177 -> 182 us.
    constexpr bool kTab = sizeof(T) == 8 && MODE == CE_LS_FWD && !WIDE;
    __shared__ double etab[kTab ? 64 : 1];
    __shared__ T lds_m[G::kWaves];
    __shared__ double lds_s[G::kWaves], lds_a[G::kWaves];
    __shared__ V more[LV > 0 ? LV : 1][LV > 0 ? NT : 1];
    __shared__ T lds_xt;
    if constexpr (kTab) {
        if (threadIdx.x < 64) etab[threadIdx.x] = exp2(double(threadIdx.x) * (1.0 / 64.0));
        __syncthreads();
    }
    const int lane = threadIdx.x % NT;
    const int64_t r = r_base + int64_t(blockIdx.x) * RPB + threadIdx.x / NT;
    if (RPB > 1 && r >= a.rows) return;  // uniform per group; a block of one row has one
    const int64_t cols = a.cols;
    const T *xr = x + r * cols;
    T *gr = GRAD ? static_cast<T *>(a.grad) + r * cols : nullptr;
    const RowCut<T> cut(cols);
    const int nsc = FULL ? 0 : cut.rem;
    const auto in_row = [&](int k) { return FULL || lane + k * NT < cut.ncv; };
    // the target first: its load overlaps the row's instead of following the reductions
    int64_t t = 0;
    const bool ok = loss_target(a.tidx, static_cast<const T *>(a.tval), r, cols, t);
    V v[VPT], w[LV > 0 ? LV : 1];
    T vt = -inf_t<T>();
    const U *xv = reinterpret_cast<const U *>(xr);
#pragma unroll
    for (int k = 0; k < VPT; k++)
        if (in_row(k)) v[k] = __builtin_nontemporal_load(xv + lane + k * NT);
#pragma unroll
    for (int k = 0; k < LV; k++)
        if (in_row(VPT + k)) w[k] = __builtin_nontemporal_load(xv + lane + (VPT + k) * NT);
    if (lane < nsc) vt = xr[cut.sc(lane)];
    T xt = LOSS && ok ? xr[t] : T(0);
    // the target's vector and slot, or the scalar that holds it (-1: neither)
    const bool t_vec = ok && t < int64_t(FULL ? NT * VPT : cut.ncv) * VN;
    const int tv = t_vec ? int(t / VN) : -1, tj = int(t % VN);
    const bool t_mine = ok && !t_vec && lane < nsc && cut.sc(lane) == t;  // in this lane's scalar
    T mx = vt == vt ? vt : -inf_t<T>();
#pragma unroll
    for (int k = 0; k < VPT; k++)
        if (in_row(k)) {
#pragma unroll
            for (int j = 0; j < VN; j++) mx = fmax_nn(mx, v[k][j]);
        }
#pragma unroll
    for (int k = 0; k < LV; k++)
        if (in_row(VPT + k)) {
#pragma unroll
            for (int j = 0; j < VN; j++) mx = fmax_nn(mx, w[k][j]);
            more[k][lane] = w[k];
        }
    // x_t waits in LDS where a block holds the row (a register kept for it spilled
    // others: fused f32 [256, 65536] 30.8 -> 43.4 us); lane 0 alone uses it
    if constexpr (LOSS && WIDE)
        if (lane == 0) lds_xt = xt;
    const double m = double(G::max(mx, lds_m));
    const auto row_exp = [&](T xv) {
        if constexpr (kTab) return exp_tab(double(xv) - m, etab);
        else if constexpr (sizeof(T) == 8) return row_exp_d(double(xv), m);
        else return row_exp_f(float(xv), m);
    };
    // Per-lane sums: double, except the f32 tensor loss of rows held by a
    // wave, whose reference sums its float e_c in float (a lane's 64 float
    // partial sums stay far inside that sum's own rounding); the group sum is
    // double either way.
    using Acc = typename std::conditional<MODE == CE_ASM && sizeof(T) == 4 && !WIDE, float, double>::type;
    Acc sl = Acc(0);
    double acc = 0.0;
    double e_t = 0.0;  // tensor CE: the lane that holds the target has its e here
    bool mine = t_mine;
    const auto sum_vec = [&](V &q, int k) {  // vector lane + k NT of the row
        double e[VN];
#pragma unroll
        for (int j = 0; j < VN; j++) {
            e[j] = row_exp(q[j]);
            if constexpr (LOSS) acc += ce_diff<T, WIDE>(q[j], m);
            if constexpr (GRAD) q[j] = T(e[j]);
            sl += Acc(e[j]);
        }
        if (MODE == CE_ASM && lane + k * NT == tv) {
            e_t = e[0];
#pragma unroll
            for (int j = 1; j < VN; j++) e_t = j == tj ? e[j] : e_t;
            mine = true;
        }
    };
#pragma unroll
    for (int k = 0; k < VPT; k++)
        if (in_row(k)) sum_vec(v[k], k);
#pragma unroll 1
    for (int k = 0; k < LV; k++)
        if (in_row(VPT + k)) {
            V q = more[k][lane];
            sum_vec(q, VPT + k);
            if constexpr (GRAD) more[k][lane] = q;
        }
    if (nsc) {  // uniform
        const double e = row_exp(vt);
        if (LOSS && lane < nsc) acc += ce_diff<T, WIDE>(vt, m);
        if (MODE == CE_ASM && t_mine) e_t = e;
        if constexpr (GRAD) vt = T(e);
        sl += Acc(e);
    }
    const double s = G::sum(double(sl), lds_s);
    // x_t is read before any gradient is written, which may be over the logits
    if constexpr (LOSS && GRAD && !WIDE) asm volatile("" : "+v"(xt) : : "memory");
    if (!ok) {
        if (lane == 0) {
            __hip_atomic_store(a.bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (a.row_loss) a.row_loss[r] = __builtin_nan("");
        }
        return;  // uniform per group
    }
    if constexpr (MODE == CE_ASM) {
        // p_t = e_t / sum (f32: e_t, sum and p_t rounded to float); the row's
        // loss -log(p_t + 1e-7) is taken in the summing pass (RedCeLoss), where
        // the double log runs on all lanes instead of on lane 0 of every row.
        if (mine) a.row_loss[r] = sizeof(T) == 4 ? double(float(e_t) / float(s)) : e_t / s;
        return;
    }
    const double st0 = a.alpha / double(cols), st1 = st0 + (1.0 - a.alpha);
    if constexpr (GRAD) {
        const CeGrad<T, WIDE> grad{1.0 / s, st0, st1, a.inv_n};
        const auto store_vec = [&](const V &q, int k) {
            V g;
#pragma unroll
            for (int j = 0; j < VN; j++) g[j] = grad(q[j], false);
            if (lane + k * NT == tv) {
#pragma unroll
                for (int j = 0; j < VN; j++)
                    if (j == tj) g[j] = grad(q[j], true);
            }
            __builtin_nontemporal_store(g, reinterpret_cast<U *>(gr) + lane + k * NT);
        };
#pragma unroll
        for (int k = 0; k < VPT; k++)
            if (in_row(k)) store_vec(v[k], k);
#pragma unroll 3
        for (int k = 0; k < LV; k++)
            if (in_row(VPT + k)) store_vec(more[k][lane], VPT + k);
        if (lane < nsc) gr[cut.sc(lane)] = grad(vt, t_mine);
    }
    if constexpr (LOSS) {
        acc = G::sum(acc, lds_a);
        if (lane == 0) {
            a.row_loss[r] = st0 * acc + (st1 - st0) * ce_diff<T, WIDE>(WIDE ? lds_xt : xt, m);
            a.row_s[r] = s;
        }
    }
}

// Rows wider than a block's registers: 1024 lanes per row and two reads, the
// first for the maximum and the sum of exp (a running maximum per lane, the
// lane's sum rescaled in double when a batch of vectors raises it), the second
// for the outputs.
constexpr int kCeWide = 1024;
template <typename T, int MODE>
__global__ __launch_bounds__(kCeWide) void k_ce_stream(const T *__restrict__ x, CeArgs a, int64_t r_base)
{
    using V = typename Vec16<T>::type;
    using U = typename VecU<T>::type;
    using G = RowGrp<kCeWide>;
    constexpr int VN = Vec16<T>::n, UN = 4;
    constexpr bool LOSS = MODE == CE_LS_FWD || MODE == CE_LS_FUSED;
    constexpr bool GRAD = MODE == CE_LS_BWD || MODE == CE_LS_FUSED;
    __shared__ T lds_m[G::kWaves];
    __shared__ double lds_s[G::kWaves], lds_a[G::kWaves];
    const int64_t r = r_base + blockIdx.x;
    const int64_t cols = a.cols, ncv = cols / VN;
    const T *xr = x + r * cols;
    const U *xv = reinterpret_cast<const U *>(xr);
    int64_t t = 0;
    const bool ok = loss_target(a.tidx, static_cast<const T *>(a.tval), r, cols, t);
    T xt = ok ? xr[t] : T(0);
    const auto row_exp = [](T xv, double m) {
        return sizeof(T) == 8 ? row_exp_d(double(xv), m) : row_exp_f(float(xv), m);
    };
    T mx = -inf_t<T>();
    double s = 0.0, mr = 0.0;  // mr: what the sum's exponents are relative to (0 while only -inf was seen)
    const auto rise = [&](T bm) {
        if (bm > mx) {
            if (s != 0.0) s *= exp(mr - double(bm));
            mx = bm;
            mr = double(bm);
        }
    };
    for (int64_t c = threadIdx.x; c < ncv; c += UN * kCeWide) {
        V v[UN];
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (c + u * kCeWide < ncv) v[u] = xv[c + u * kCeWide];
        T bm = -inf_t<T>();
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (c + u * kCeWide < ncv) {
#pragma unroll
                for (int j = 0; j < VN; j++) bm = fmax_nn(bm, v[u][j]);
            }
        rise(bm);
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (c + u * kCeWide < ncv) {
#pragma unroll
                for (int j = 0; j < VN; j++) s += row_exp(v[u][j], mr);
            }
    }
    const int64_t jt = ncv * VN + threadIdx.x;  // at most VN - 1 values past the vectors
    if (jt < cols) {
        rise(xr[jt]);
        s += row_exp(xr[jt], mr);
    }
    const double m = double(G::max(mx, lds_m));
    // a row of only -inf is NaN, as exp(-inf - -inf) makes it
    s = G::sum(s == 0.0 ? s : s * exp(mr - m), lds_s);
    if (m == -__builtin_inf()) s = __builtin_nan("");
    if constexpr (LOSS && GRAD) asm volatile("" : "+v"(xt) : : "memory");  // before any gradient is written
    if (!ok) {
        if (threadIdx.x == 0) {
            __hip_atomic_store(a.bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (a.row_loss) a.row_loss[r] = __builtin_nan("");
        }
        return;
    }
    if constexpr (MODE == CE_ASM) {
        const double e_t = row_exp(xt, m);
        if (threadIdx.x == 0) a.row_loss[r] = sizeof(T) == 4 ? double(float(e_t) / float(s)) : e_t / s;
        return;
    }
    const double st0 = a.alpha / double(cols), st1 = st0 + (1.0 - a.alpha);
    const CeGrad<T, true> grad{1.0 / s, st0, st1, a.inv_n};
    T *gr = static_cast<T *>(a.grad) + r * cols;
    double acc = 0.0;
    const int64_t tv = t / VN;
    const int tj = int(t % VN);
    for (int64_t c = threadIdx.x; c < ncv; c += UN * kCeWide) {
        V v[UN];
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (c + u * kCeWide < ncv) v[u] = xv[c + u * kCeWide];
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const int64_t i = c + u * kCeWide;
            if (i < ncv) {
                V g;
#pragma unroll
                for (int j = 0; j < VN; j++) {
                    if constexpr (LOSS) acc += ce_diff<T, true>(v[u][j], m);
                    if constexpr (GRAD) g[j] = grad(T(row_exp(v[u][j], m)), i == tv && j == tj);
                }
                if constexpr (GRAD) __builtin_nontemporal_store(g, reinterpret_cast<U *>(gr) + i);
            }
        }
    }
    if (jt < cols) {
        const T xj = xr[jt];
        if constexpr (LOSS) acc += ce_diff<T, true>(xj, m);
        if constexpr (GRAD) gr[jt] = grad(T(row_exp(xj, m)), jt == t);
    }
    if constexpr (LOSS) {
        acc = G::sum(acc, lds_a);
        if (threadIdx.x == 0) {
            a.row_loss[r] = st0 * acc + (st1 - st0) * ce_diff<T, true>(xt, m);
            a.row_s[r] = s;
        }
    }
}

template <typename T, int MODE, int NT, int VPT, int LV = 0>
static void launch_ce_rows(const T *x, const CeArgs &a)
{
    constexpr int W = NT == 512 ? 4 : (NT <= 64 && sizeof(T) == 8 && MODE == CE_LS_FWD && VPT <= 8 ? 5 : 1);
    constexpr int block = NT < 256 ? 256 : NT;
    for_row_launches(a.rows, block / NT, [&](unsigned g, int64_t base) {
        if constexpr (NT <= 64) {
            if (a.cols == int64_t(NT) * VPT * Vec16<T>::n) {
                // (the tensor loss, which stores nothing, wants it from 8 vectors: f32
                // [65536, 1024] 57.6 us with it, 50.4 without, [32768, 2048] 49.4, 51.1)
                constexpr unsigned lds = sizeof(T) == 4 && VPT >= (MODE == CE_ASM ? 8 : 4) ? kFullRowsLds : 0;
                NH_LAUNCH((k_ce_rows<T, NT, VPT, LV, MODE, true, W>), dim3(g), dim3(block), lds, stream(), x, a, base);
                return;
            }
        }
        NH_LAUNCH((k_ce_rows<T, NT, VPT, LV, MODE, false, W>), dim3(g), dim3(block), 0, stream(), x, a, base);
    });
}

// The smallest group whose registers hold the row (as launch_softmax).  A wave
// ends at exactly 4096 f32 / 2048 f64 values, without the few more that its
// scalars would hold: wider rows form every term in double (WIDE).  Before
// (a wave per row up to 4096 f32 / 2048 f64 values, element by element where
// the width was no multiple of the vector, then three passes) -> now, us,
// smoothed fused form with its summing launches:
//   f32 [65536, 10] 32.1 -> 10.7, [32768, 256] 24.3 -> 19.2, [30000, 1001] 84.3 -> 49.0, [65536, 1024] 93.2 -> 89.9
//       [8192, 3000] 107 -> 43.5, [4096, 8192] 115 -> 52.4, [2048, 32000] 267 -> 104, [4096, 50257] 861 -> 340
//       [600, 98000] 517 -> 110, [500, 131072] 682 -> 134 (two reads)
//   f64 [65536, 10] 33.7 -> 14.3, [30000, 1001] 104 -> 92, [4096, 8553] 203 -> 110, [2000, 24001] 332 -> 167
template <typename T, int MODE>
static int launch_ce(const T *x, const CeArgs &a)
{
    const int64_t ncv = a.cols / Vec16<T>::n;
    if (ncv <= 4) launch_ce_rows<T, MODE, 4, 1>(x, a);
    else if (ncv <= 16) launch_ce_rows<T, MODE, 16, 1>(x, a);
    else if (ncv <= 16 * 4) launch_ce_rows<T, MODE, 16, 4>(x, a);
    else if (ncv <= 64 * 2) launch_ce_rows<T, MODE, 64, 2>(x, a);
    else if (ncv <= 64 * 4) launch_ce_rows<T, MODE, 64, 4>(x, a);
    else if (ncv <= 64 * 8) launch_ce_rows<T, MODE, 64, 8>(x, a);
    else if (a.cols <= 64 * 16 * Vec16<T>::n) launch_ce_rows<T, MODE, 64, 16>(x, a);
    else if (ncv <= 256 * 8) launch_ce_rows<T, MODE, 256, 8>(x, a);
    else if (ncv <= 256 * 16) launch_ce_rows<T, MODE, 256, 16>(x, a);
    else if (ncv <= 512 * 16) launch_ce_rows<T, MODE, 512, 16>(x, a);
    else if (ncv <= 512 * 25) launch_ce_rows<T, MODE, 512, 16, 9>(x, a);
    else if (ncv <= 1024 * 24) launch_ce_rows<T, MODE, 1024, 24>(x, a);
    else
        for_row_launches(a.rows, 1, [&](unsigned g, int64_t base) {
            NH_LAUNCH((k_ce_stream<T, MODE>), dim3(g), dim3(kCeWide), 0, stream(), x, a, base);
        });
    return check_launch();
}

// Sum of the per-row losses of the tensor CE (losses.asm intended semantics):
// the rows hold p_t, the loss term is -log(p_t + 1e-7), rounded to float for
// f32 logits as the reference's float loss.  div != 0: the stored value is
// the sum / div (the mean, for a loss left in device memory), the division
// the host makes otherwise.
template <bool F32>
struct RedCeLoss {
    static constexpr bool kCostly = true;
    using L = double;
    using B = double;
    double div = 0.0;
    NH_DEV L linit() const { return 0.0; }
    NH_DEV void lacc(L &s, double p, int64_t) const
    {
        const double lt = -log(p + 1e-7);
        s += F32 ? double(float(lt)) : lt;
    }
    NH_DEV L lcomb(L a, L b) const { return a + b; }
    template <int TPR> NH_DEV B finish(L s, const double *, int64_t, int64_t) const { return s; }
    NH_DEV B bident() const { return 0.0; }
    NH_DEV B bcomb(B a, B b) const { return a + b; }
    NH_DEV void store(void *out, int64_t r, B s, const double *, int64_t) const
    {
        static_cast<double *>(out)[r] = div != 0.0 ? s / div : s;
    }
};

// Sum of the label-smoothed row losses: row r holds A_r = sum_c st_c (x_c - m)
// and s_r = sum_c exp(x_c - m); its loss is log(s_r) * S - A_r with
// S = sum_c st_c = st0 (cols - 1) + st1.  div as in RedCeLoss.
struct RedLsLoss {
    static constexpr bool kCostly = true;
    using L = double;
    using B = double;
    const double *s;
    double S;
    double div = 0.0;
    NH_DEV L linit() const { return 0.0; }
    NH_DEV void lacc(L &acc, double A, int64_t i) const
    {
        const double lse = log(s[i]);
        const double sl = lse * S;
        acc += sl - A;
    }
    NH_DEV L lcomb(L a, L b) const { return a + b; }
    template <int TPR> NH_DEV B finish(L v, const double *, int64_t, int64_t) const { return v; }
    NH_DEV B bident() const { return 0.0; }
    NH_DEV B bcomb(B a, B b) const { return a + b; }
    NH_DEV void store(void *out, int64_t r, B v, const double *, int64_t) const
    {
        static_cast<double *>(out)[r] = div != 0.0 ? v / div : v;
    }
};

// Runs MODE over [rows, cols] logits already on the device; sums the per-row
// losses into *loss_host (mean over rows) when wanted.  Returns NEURAL_OK,
// NEURAL_ERR_INVALID_ARGUMENT for a target out of range, or an error code.
// With loss_dev (device memory) instead, the mean loss is stored there by the
// last launch and the call returns once everything is enqueued: nothing is
// waited for, and a target out of range shows only as a NaN loss.
template <typename T, int MODE>
static int ce_run(const T *x, const int64_t *tidx, const T *tval, int64_t rows, int64_t cols, double alpha,
                  double *loss_host, T *grad_dev, double *loss_dev = nullptr)
{
    WsGuard wg;
    Workspace &ws = workspace();
    const bool on_dev = loss_dev != nullptr;
    const bool want_loss = MODE != CE_LS_BWD;
    constexpr bool kLs = MODE == CE_LS_FWD || MODE == CE_LS_FUSED;
    // The loss sum (word 0) and the out-of-range flag (int word 32) are stored
    // into the mapped host area.  The flag is zero at init and between calls
    // (a call that finds it set clears it on the host).  A call that leaves
    // its loss on the device points the flag at a spare word of its own row
    // buffer, which nothing reads.
    int *bad = static_cast<int *>(ws.host_result_dev) + 32;
    double *row_loss = nullptr, *row_s = nullptr;
    if (want_loss) {
        // one block: [rows] row values, then [rows] exp sums (label-smoothed),
        // then the spare flag word for a device-resident loss
        const size_t words = size_t(rows) * (kLs ? 2 : 1);
        row_loss = static_cast<double *>(dev_alloc((words + (on_dev ? 1 : 0)) * sizeof(double)));
        if (!row_loss) return set_error(NEURAL_ERR_OUT_OF_MEMORY);
        if (kLs) row_s = row_loss + rows;
        if (on_dev) bad = reinterpret_cast<int *>(row_loss + words);
    }
    CeArgs a{tidx, tval, rows, cols, alpha, 1.0 / double(rows), row_loss, row_s, grad_dev, bad};
    int rc = launch_ce<T, MODE>(x, a);
    // The loss sum's launch stores a ticket after the sum (and after the CE
    // kernel, earlier on the stream, has set the flag or not): the host waits
    // for the ticket instead of synchronising the stream.
    const Ticket tk = want_loss && !on_dev ? next_ticket() : Ticket{};
    if (rc == NEURAL_OK && want_loss) {
        void *dst = on_dev ? static_cast<void *>(loss_dev) : ws.host_result_dev;
        const double div = on_dev ? double(rows) : 0.0;
        if (MODE == CE_ASM) {
            rc = launch_reduce(row_loss, 1, rows, rows, RedCeLoss<sizeof(T) == 4>{div}, dst, nullptr, 0, tk);
        } else {
            const double st0 = alpha / double(cols), st1 = st0 + (1.0 - alpha);
            rc = launch_reduce(row_loss, 1, rows, rows, RedLsLoss{row_s, st0 * double(cols - 1) + st1, div}, dst,
                               nullptr, 0, tk);
        }
    }
    if (on_dev) {
        if (row_loss) dev_free(row_loss);  // reused only by work enqueued after these launches
        return rc;
    }
    struct { double sum; int pad[30]; int bad; } res;  // result area layout: sum at 0, flag at word 32
    static_assert(sizeof(res) == 136, "");
    if (rc == NEURAL_OK)
        rc = want_loss ? host_result_wait(tk.value, &res, sizeof(res)) : host_result_fetch(&res, sizeof(res));
    if (row_loss) dev_free(row_loss);
    if (rc != NEURAL_OK) return rc;
    if (res.bad) {
        // every launch of this call has finished writing the area (the
        // ticket, or the stream wait, comes after them)
        static_cast<int *>(ws.host_result)[32] = 0;
        return NEURAL_ERR_INVALID_ARGUMENT;
    }
    if (want_loss && loss_host) *loss_host = res.sum / double(rows);
    return NEURAL_OK;
}

// Raw-pointer label-smoothed CE (host or device pointers).
template <typename T, int MODE>
static int ls_ce(const T *logits, const int64_t *targets, int64_t batch, int64_t classes, double smoothing,
                 double *loss_out, T *grad_out)
{
    if (ensure_init() != NEURAL_OK) return -1;
    if (!logits || !targets) return -1;
    if ((MODE != CE_LS_BWD && !loss_out) || (MODE != CE_LS_FWD && !grad_out)) return -1;
    if (batch <= 0 || classes <= 0) return -1;
    if (!(smoothing >= 0.0 && smoothing <= 1.0)) return -1;
    int64_t n;
    if (__builtin_mul_overflow(batch, classes, &n)) return -1;
    Staged sx, st, sg;
    if (sx.open_n(logits, uint64_t(n), sizeof(T), true) != NEURAL_OK ||
        st.open_n(targets, uint64_t(batch), 8, true) != NEURAL_OK)
        return -1;
    if (MODE != CE_LS_FWD && sg.open_n(grad_out, uint64_t(n), sizeof(T), false) != NEURAL_OK) return -1;
    const int rc = ce_run<T, MODE>(static_cast<const T *>(sx.dev), static_cast<const int64_t *>(st.dev), nullptr,
                                   batch, classes, smoothing, loss_out, static_cast<T *>(sg.dev));
    if (rc != NEURAL_OK) return -1;
    if (MODE != CE_LS_FWD && sg.finish(true) != NEURAL_OK) return -1;
    set_error(NEURAL_OK);
    return 0;
}

// Label-smoothed CE on device pointers with the mean loss left in device
// memory (*loss_dev): every launch enqueued, nothing waited for.
template <typename T, int MODE>
static int ls_ce_dev(const T *logits, const int64_t *targets, int64_t batch, int64_t classes, double smoothing,
                     double *loss_dev, T *grad_dev)
{
    if (ensure_init() != NEURAL_OK) return -1;
    if (!logits || !targets || !loss_dev || (MODE == CE_LS_FUSED && !grad_dev)) {
        set_error(NEURAL_ERR_NULL_POINTER);
        return -1;
    }
    int64_t n;
    if (batch <= 0 || classes <= 0 || !(smoothing >= 0.0 && smoothing <= 1.0) ||
        __builtin_mul_overflow(batch, classes, &n) || uint64_t(n) > kMaxRawCount) {
        set_error(NEURAL_ERR_INVALID_ARGUMENT);
        return -1;
    }
    const auto misaligned = [](const void *p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) != 0; };
    if (!is_device_ptr(logits) || !is_device_ptr(targets) || !is_device_ptr(loss_dev) ||
        (grad_dev && !is_device_ptr(grad_dev)) || misaligned(logits, sizeof(T)) || misaligned(targets, 8) ||
        misaligned(loss_dev, 8) || (grad_dev && misaligned(grad_dev, sizeof(T)))) {
        set_error(NEURAL_ERR_INVALID_ARGUMENT);
        return -1;
    }
    if (ce_run<T, MODE>(logits, targets, nullptr, batch, classes, smoothing, nullptr, grad_dev, loss_dev) !=
        NEURAL_OK)
        return -1;
    set_error(NEURAL_OK);
    return 0;
}

}  // namespace nh

using namespace nh;

extern "C" {

int label_smoothing_ce_forward_dev(const double *logits, const int64_t *targets, int64_t batch_size,
                                   int64_t num_classes, double smoothing, double *loss_dev)
{
    return ls_ce_dev<double, CE_LS_FWD>(logits, targets, batch_size, num_classes, smoothing, loss_dev, nullptr);
}

int label_smoothing_ce_fused_dev(const double *logits, const int64_t *targets, int64_t batch_size,
                                 int64_t num_classes, double smoothing, double *loss_dev, double *grad_dev)
{
    return ls_ce_dev<double, CE_LS_FUSED>(logits, targets, batch_size, num_classes, smoothing, loss_dev, grad_dev);
}

int label_smoothing_ce_fused_f32_dev(const float *logits, const int64_t *targets, int64_t batch_size,
                                     int64_t num_classes, double smoothing, double *loss_dev, float *grad_dev)
{
    return ls_ce_dev<float, CE_LS_FUSED>(logits, targets, batch_size, num_classes, smoothing, loss_dev, grad_dev);
}

int label_smoothing_ce_forward(const double *logits, const int64_t *targets, int64_t batch_size,
                               int64_t num_classes, double smoothing, double *loss_out)
{
    return ls_ce<double, CE_LS_FWD>(logits, targets, batch_size, num_classes, smoothing, loss_out, nullptr);
}

int label_smoothing_ce_backward(const double *logits, const int64_t *targets, int64_t batch_size,
                                int64_t num_classes, double smoothing, double *grad_out)
{
    return ls_ce<double, CE_LS_BWD>(logits, targets, batch_size, num_classes, smoothing, nullptr, grad_out);
}

int label_smoothing_ce_fused(const double *logits, const int64_t *targets, int64_t batch_size, int64_t num_classes,
                             double smoothing, double *loss_out, double *grad_out)
{
    return ls_ce<double, CE_LS_FUSED>(logits, targets, batch_size, num_classes, smoothing, loss_out, grad_out);
}

int label_smoothing_ce_fused_f32(const float *logits, const int64_t *targets, int64_t batch_size,
                                 int64_t num_classes, double smoothing, double *loss_out, float *grad_out)
{
    return ls_ce<float, CE_LS_FUSED>(logits, targets, batch_size, num_classes, smoothing, loss_out, grad_out);
}

int neural_cross_entropy_loss(const NeuralTensor *prediction, const NeuralTensor *target, double *loss)
{
    NH_TRY(ensure_init());
    if (!prediction || !target || !loss) return set_error(NEURAL_ERR_NULL_POINTER);
    NH_TRY(check_tensor(prediction));
    NH_TRY(check_tensor(target));
    if (prediction->dtype != target->dtype) return set_error(NEURAL_ERR_DTYPE_MISMATCH);
    if (prediction->ndim != 2) return set_error(NEURAL_ERR_DIM_MISMATCH);
    const int64_t rows = prediction->shape[0], cols = prediction->shape[1];
    if (rows <= 0 || cols <= 0) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    if (numel(target) != rows) return set_error(NEURAL_ERR_SHAPE_MISMATCH);
    if (!is_contiguous(prediction) || !is_contiguous(target)) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    const void *px = nullptr, *pt = nullptr;
    NH_TRY(dev_read(prediction, &px));
    NH_TRY(dev_read(target, &pt));
    int rc;
    if (prediction->dtype == NEURAL_DTYPE_FLOAT32)
        rc = ce_run<float, CE_ASM>(static_cast<const float *>(px), nullptr, static_cast<const float *>(pt), rows, cols,
                                   0.0, loss, nullptr);
    else
        rc = ce_run<double, CE_ASM>(static_cast<const double *>(px), nullptr, static_cast<const double *>(pt), rows,
                                    cols, 0.0, loss, nullptr);
    return set_error(rc);
}

}  // extern "C"
