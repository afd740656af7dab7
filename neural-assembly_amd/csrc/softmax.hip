// softmax.hip -- row softmax and log-softmax over the last dimension.
//
// Softmax follows node_softmax (activations.asm:761-987) with its intended
// f32 semantics (the asm keeps the max and the running sum in one stack slot,
// activations.asm:900,927-929):
//   f32: m = row max; e_j = (float)exp((double)x_j - (double)m);
//        s = sum of e_j; y_j = e_j / s
//   f64: e_j = exp(x_j - m); y_j = e_j / s
// Here the f32 e_j come from the exact double difference x - m and the
// hardware exp2 (about 1.5e-7 relative, see exp_diff_f32) and y_j = e_j * (1/s).
// Log-softmax follows the formula of label_smoothing_ce_forward
// (metrics_losses.c:47-64) in double: y = (x - m) - log(sum exp(x - m)),
// rounded once for f32.
//
// The sum is accumulated in double with a fixed wave/block tree instead of the
// reference's sequential order; results are compared against the fp64-exact
// softmax.  A NaN anywhere in a row makes the whole row NaN, as in the
// reference (the NaN reaches the sum).
//
// A row is held in registers by one group of lanes -- part of a wave or a wave up
// to 2048 f32 / 1024 f64 values and at exactly twice that, else a block of 256 to
// 1024 lanes, up to 98304 / 49152 values -- so it is read once and written once at any width and alignment:
// 16-byte accesses at the element's own alignment and one scalar per lane for
// the values at the row's ends.  Wider rows are read twice.
#include <cmath>

#include <hip/hip_ext.h>

#include "row_group.hpp"

namespace nh {

constexpr int kSmBlock = 256;

template <typename T>
NH_DEV T neg_inf();
template <> NH_DEV float neg_inf<float>() { return -__builtin_inff(); }
template <> NH_DEV double neg_inf<double>() { return -__builtin_inf(); }

// exp(x - m) for f32 rows (x <= m, m the row max held in double): the
// difference is exact in double, so exp_d2f gives about 1.5e-7 relative
// against (float)exp((double)x - (double)m) for any spread of the row.  A NaN
// passes through and makes the row's sum NaN, as in the reference.
NH_DEV float exp_diff_f32(float x, double md) { return exp_d2f(double(x) - md); }

NH_DEV float row_exp(float x, double m) { return exp_diff_f32(x, m); }
NH_DEV double row_exp(double x, double m) { return exp(x - m); }

// One output value.  f32 takes its last step in double and rounds once; the
// softmax multiplies by the reciprocal of the sum there (a double division
// per value made the instruction count, not HBM, the bound).
template <typename T, bool LOG>
NH_DEV T row_out(T v, double md, double lse, double s, double rs)
{
    // hides the value's origin: the compiler would keep double(v) from the sum
    // (two more registers per value) instead of converting again here
    if constexpr (sizeof(T) == 4) asm("" : "+v"(v));
    if constexpr (LOG) return T((double(v) - md) - lse);
    else if constexpr (sizeof(T) == 4) return T(double(v) * rs);
    else return v / s;
}

// One row per group of NT lanes, held in VPT vectors per lane (and the values
// past the vectors in one scalar of the first lanes, see RowCut;
// the other lanes' scalar is -inf, which adds 0 to the sum, or NaN where the
// row is NaN anyway).  FULL: the
// row is exactly NT * VPT vectors, so no element needs a bounds check.
//
// What bounds it: HBM, one read and one write, while the rows in flight per
// CU cover the latency; hence VPT <= 25 (two 512-lane blocks per CU at 51200
// f32 values; __launch_bounds__ asks for them) and 1024 lanes only past that.
// f32, before (three passes of 4-byte accesses per row for odd or long rows)
// and after: see launch_softmax.
template <typename T, bool LOG, int NT, int VPT, bool FULL>
__global__ __launch_bounds__(NT < kSmBlock ? kSmBlock : NT, NT == 512 ? 4 : 1) void k_softmax_rows(
    const T *__restrict__ x, T *__restrict__ y, int64_t rows, int64_t cols, int64_t r_base)
{
    using V = typename Vec16<T>::type;
    using U = typename VecU<T>::type;
    using G = RowGrp<NT>;
    constexpr int VN = Vec16<T>::n;
    constexpr int RPB = NT < kSmBlock ? kSmBlock / NT : 1;
    __shared__ T lds_m[G::kWaves];
    __shared__ double lds_s[G::kWaves];
    const int lane = threadIdx.x % NT;
    const int64_t r = r_base + int64_t(blockIdx.x) * RPB + threadIdx.x / NT;
    if (RPB > 1 && r >= rows) return;  // uniform per group; a block of one row has one
    const T *xr = x + r * cols;
    T *yr = y + r * cols;
    const RowCut<T> cut(cols);
    const int nsc = FULL ? 0 : cut.rem;
    const auto in_row = [&](int k) { return FULL || lane + k * NT < cut.ncv; };
    V v[VPT];
    T vt = neg_inf<T>();
#pragma unroll
    for (int k = 0; k < VPT; k++)
        if (in_row(k)) v[k] = __builtin_nontemporal_load(reinterpret_cast<const U *>(xr) + lane + k * NT);
    if (lane < nsc) vt = xr[cut.sc(lane)];

    T m = vt == vt ? vt : neg_inf<T>();
#pragma unroll
    for (int k = 0; k < VPT; k++) {
        if (in_row(k)) {
#pragma unroll
            for (int j = 0; j < VN; j++) {
                if constexpr (sizeof(T) == 4) m = __builtin_fmaxf(m, v[k][j]);
                else m = v[k][j] > m ? v[k][j] : m;
            }
        }
    }
    const double md = double(G::max(m, lds_m));
    double s = 0.0;
    // softmax: e_j kept in the input registers, rounded to T as the reference does
#pragma unroll
    for (int k = 0; k < VPT; k++) {
        if (in_row(k)) {
#pragma unroll
            for (int j = 0; j < VN; j++) {
                const T e = row_exp(v[k][j], md);
                if (!LOG) v[k][j] = e;
                s += double(e);
            }
        }
    }
    if (nsc) {  // uniform
        const T e = row_exp(vt, md);
        if (!LOG) vt = e;
        s += double(e);
    }
    s = G::sum(s, lds_s);
    // s >= 1: the maximum contributes 1.  f64 rows of whole vectors within a wave
    // take log_ge1 (about 3 ulp, fewer instructions per row); the others, whose
    // rows are longer or were always logged by the library, its log.
    double lse = 0.0;
    if constexpr (LOG && sizeof(T) == 4) lse = log_ge1(s);
    else if constexpr (LOG) lse = NT <= 64 && cols % VN == 0 ? log_ge1(s) : log(s);
    const double rs = LOG ? 0.0 : 1.0 / s;
#pragma unroll
    for (int k = 0; k < VPT; k++) {
        if (in_row(k)) {
            V o;
#pragma unroll
            for (int j = 0; j < VN; j++) o[j] = row_out<T, LOG>(v[k][j], md, lse, s, rs);
            __builtin_nontemporal_store(o, reinterpret_cast<U *>(yr) + lane + k * NT);
        }
    }
    if (lane < nsc) yr[cut.sc(lane)] = row_out<T, LOG>(vt, md, lse, s, rs);
}

// Rows wider than the registers of a block: one 1024-lane block per row, two
// reads.  Each lane keeps a running maximum and the sum of exp(x - maximum),
// rescaled (in double) when a batch of four vectors raises the maximum; the
// block's sum is the rescaled total, and the second pass writes the outputs.
constexpr int kSmWide = 1024;
template <typename T, bool LOG>
__global__ __launch_bounds__(kSmWide) void k_softmax_stream(const T *__restrict__ x, T *__restrict__ y, int64_t cols,
                                                           int64_t r_base)
{
    using V = typename Vec16<T>::type;
    using U = typename VecU<T>::type;
    using G = RowGrp<kSmWide>;
    constexpr int VN = Vec16<T>::n, UN = 4;
    __shared__ T lds_m[G::kWaves];
    __shared__ double lds_s[G::kWaves];
    const int64_t r = r_base + blockIdx.x;
    const T *xr = x + r * cols;
    T *yr = y + r * cols;
    const U *xv = reinterpret_cast<const U *>(xr);
    U *yv = reinterpret_cast<U *>(yr);
    const int64_t ncv = cols / VN;
    T m = neg_inf<T>();
    double s = 0.0;
    double mr = 0.0;  // what the sum's exponents are relative to: m, or 0 while the lane has seen only -inf
    const auto rise = [&](T bm) {
        if (bm > m) {
            if (s != 0.0) s *= exp(mr - double(bm));
            m = bm;
            mr = double(bm);
        }
    };
    for (int64_t c = threadIdx.x; c < ncv; c += UN * kSmWide) {
        V v[UN];
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (c + u * kSmWide < ncv) v[u] = xv[c + u * kSmWide];
        T bm = neg_inf<T>();
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (c + u * kSmWide < ncv) {
#pragma unroll
                for (int j = 0; j < VN; j++) bm = v[u][j] > bm ? v[u][j] : bm;
            }
        rise(bm);
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (c + u * kSmWide < ncv) {
#pragma unroll
                for (int j = 0; j < VN; j++) s += double(row_exp(v[u][j], mr));
            }
    }
    const int64_t jt = ncv * VN + threadIdx.x;  // at most VN - 1 values past the vectors
    if (jt < cols) {
        rise(xr[jt]);
        s += double(row_exp(xr[jt], mr));
    }
    const double md = double(G::max(m, lds_m));
    // (s = 0: the lane saw only -inf; the outputs of a row of -inf are NaN below)
    s = G::sum(s == 0.0 ? 0.0 : s * exp(mr - md), lds_s);
    const double lse = LOG ? log(s) : 0.0;
    const double rs = LOG ? 0.0 : 1.0 / s;
    for (int64_t c = threadIdx.x; c < ncv; c += UN * kSmWide) {
        V v[UN];
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (c + u * kSmWide < ncv) v[u] = xv[c + u * kSmWide];
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (c + u * kSmWide < ncv) {
                V o;
#pragma unroll
                for (int j = 0; j < VN; j++)
                    o[j] = row_out<T, LOG>(LOG ? v[u][j] : T(row_exp(v[u][j], md)), md, lse, s, rs);
                __builtin_nontemporal_store(o, yv + c + u * kSmWide);
            }
    }
    if (jt < cols) yr[jt] = row_out<T, LOG>(LOG ? xr[jt] : T(row_exp(xr[jt], md)), md, lse, s, rs);
}

template <typename T, bool LOG, int NT, int VPT>
static void launch_rows(const T *x, T *y, int64_t rows, int64_t cols)
{
    for_row_launches(rows, NT < kSmBlock ? kSmBlock / NT : 1, [&](unsigned g, int64_t base) {
        constexpr int block = NT < kSmBlock ? kSmBlock : NT;
        if constexpr (NT <= 64 && sizeof(T) == 4) {
            if (cols == int64_t(NT) * VPT * Vec16<T>::n) {
                NH_LAUNCH((k_softmax_rows<T, LOG, NT, VPT, true>), dim3(g), dim3(block), VPT >= 4 ? kFullRowsLds : 0,
                          stream(), x, y, rows, cols, base);
                return;
            }
        }
        NH_LAUNCH((k_softmax_rows<T, LOG, NT, VPT, false>), dim3(g), dim3(block), 0, stream(), x, y, rows, cols, base);
    });
}

// The smallest group whose registers hold the row: its lanes stay busy and
// most rows are in flight.  Narrow rows share a wave, 16 rows of up to 4
// vectors, 4 of up to 64, 2 of up to 128; where the rows' ends are not vector
// ends the last take a whole wave (its longer stores: [100000, 511] 73 against
// 84 us).  16 vectors per lane only where every one is full: between 2048 and
// 4096 f32 values 256 lanes with up to 4 or 8 vectors answer few rows sooner and
// many alike (f32 [131, 4000] 6.2 -> 3.6 us, [4194, 4000] 24.5 -> 23.3, f64 [255, 2049]
// 8.1 -> 4.8).  Before (a wave per aligned row of up to 4096 values, else three
// passes of 4-byte accesses) -> now, us:
//   f32 [55392, 577] softmax / log-softmax  159 -> 45 / 160 -> 47 (256 MB, 5.7 TB/s)
//       [200000, 16] 42.2 -> 6.0, [200000, 64] 47.4 -> 18.1, [200000, 63] 203 -> 23.7
//       [100000, 197] 148 -> 37.4, [100000, 260] 43.2 -> 38.8, [100000, 400] 54.0 -> 53.4 (log 52.8 -> 54.5)
//       [65536, 1024] 87.8 -> 85.3, [8192, 4096] 52.0 -> 46.3, [8192, 4097] 129 -> 52, [4096, 8192] 116 -> 45.5
//   f64 [100000, 33] 118 -> 12.4, [32768, 1024] the same, [4096, 8191] log-softmax 179 -> 100
//   log-softmax and argmax, f32: [64, 32000] 77 -> 17.8, [100, 98000] 332 -> 41, [128, 131072] 429 -> 60
template <typename T, bool LOG>
static int launch_softmax(const T *x, T *y, int64_t rows, int64_t cols)
{
    const int64_t ncv = cols / Vec16<T>::n;
    if (ncv <= 4) launch_rows<T, LOG, 4, 1>(x, y, rows, cols);
    else if (ncv <= 16) launch_rows<T, LOG, 16, 1>(x, y, rows, cols);
    else if (ncv <= 16 * 2) launch_rows<T, LOG, 16, 2>(x, y, rows, cols);
    else if (ncv <= 16 * 4) launch_rows<T, LOG, 16, 4>(x, y, rows, cols);
    else if (ncv <= 32 * 4 && cols % Vec16<T>::n == 0) launch_rows<T, LOG, 32, 4>(x, y, rows, cols);
    else if (ncv <= 64 * 2) launch_rows<T, LOG, 64, 2>(x, y, rows, cols);
    else if (ncv <= 64 * 4) launch_rows<T, LOG, 64, 4>(x, y, rows, cols);
    else if (ncv <= 64 * 8) launch_rows<T, LOG, 64, 8>(x, y, rows, cols);
    else if (cols == 64 * 16 * Vec16<T>::n) launch_rows<T, LOG, 64, 16>(x, y, rows, cols);
    else if (ncv <= 256 * 4) launch_rows<T, LOG, 256, 4>(x, y, rows, cols);
    else if (ncv <= 256 * 8) launch_rows<T, LOG, 256, 8>(x, y, rows, cols);
    else if (ncv <= 256 * 16) launch_rows<T, LOG, 256, 16>(x, y, rows, cols);
    else if (ncv <= 512 * 16) launch_rows<T, LOG, 512, 16>(x, y, rows, cols);
    else if (ncv <= 512 * 25) launch_rows<T, LOG, 512, 25>(x, y, rows, cols);
    else if (ncv <= 1024 * 16) launch_rows<T, LOG, 1024, 16>(x, y, rows, cols);
    else if (ncv <= 1024 * 24) launch_rows<T, LOG, 1024, 24>(x, y, rows, cols);
    else
        for_row_launches(rows, 1, [&](unsigned g, int64_t base) {
            NH_LAUNCH((k_softmax_stream<T, LOG>), dim3(g), dim3(kSmWide), 0, stream(), x, y, cols, base);
        });
    return check_launch();
}

static int softmax_api(NeuralTensor *out, const NeuralTensor *in, bool log)
{
    NH_TRY(ensure_init());
    if (!out || !in) return set_error(NEURAL_ERR_NULL_POINTER);
    NH_TRY(check_tensor(in));
    NH_TRY(check_tensor(out));
    if (in->dtype != out->dtype) return set_error(NEURAL_ERR_DTYPE_MISMATCH);
    if (in->ndim < 1) return set_error(NEURAL_ERR_DIM_MISMATCH);
    const int64_t n = numel(in);
    if (numel(out) != n) return set_error(NEURAL_ERR_SHAPE_MISMATCH);
    if (!is_contiguous(in) || !is_contiguous(out)) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    const int64_t cols = in->shape[in->ndim - 1];
    if (n == 0 || cols == 0) return set_error(NEURAL_OK);
    const int64_t rows = n / cols;
    const void *src = nullptr;
    void *dst = nullptr;
    NH_TRY(dev_read(in, &src));
    NH_TRY(dev_write(out, &dst, true));
    if (in->dtype == NEURAL_DTYPE_FLOAT32) {
        if (log) NH_TRY((launch_softmax<float, true>(static_cast<const float *>(src), static_cast<float *>(dst), rows, cols)));
        else NH_TRY((launch_softmax<float, false>(static_cast<const float *>(src), static_cast<float *>(dst), rows, cols)));
    } else {
        if (log) NH_TRY((launch_softmax<double, true>(static_cast<const double *>(src), static_cast<double *>(dst), rows, cols)));
        else NH_TRY((launch_softmax<double, false>(static_cast<const double *>(src), static_cast<double *>(dst), rows, cols)));
    }
    NH_TRY(dev_written(out));
    return set_error(NEURAL_OK);
}

}  // namespace nh

extern "C" {

// neural_softmax (neural_api.asm:1340-1396): rows over the last dimension
// (the reference handles 2-D [batch, classes] only).
int neural_softmax(NeuralTensor *out, const NeuralTensor *in) { return nh::softmax_api(out, in, false); }

int neural_log_softmax(NeuralTensor *out, const NeuralTensor *in) { return nh::softmax_api(out, in, true); }

}  // extern "C"
