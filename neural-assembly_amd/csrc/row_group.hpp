// row_group.hpp -- reductions over the lanes that share one row, for the kernels
// that hold a row in registers (softmax, cross-entropy).
#pragma once

#include "common.hpp"

namespace nh {

// Group-wide max (NaN-ignoring) and sum over the NT lanes that share a row:
// 4, 16 or 32 lanes of a wave or the whole wave (DPP moves, and swizzles across
// 16 and 32), or a block of NT lanes through LDS.  (The f64 maximum by six
// swizzles and NaN tests per row: [65536, 256] forward loss 41.3 us, now 37.7.)
template <int NT>
struct RowGrp {
    static constexpr int kWaves = NT < 64 ? 1 : NT / 64;
    template <typename T> NH_DEV static T dpp(T v, int step)
    {
        if constexpr (sizeof(T) == 4)
            return step == 0 ? dpp_f<kDppXor1>(v) : step == 1 ? dpp_f<kDppXor2>(v)
                 : step == 2 ? dpp_f<kDppHalfMirror>(v) : dpp_f<kDppMirror>(v);
        else
            return step == 0 ? dpp_d<kDppXor1>(v) : step == 1 ? dpp_d<kDppXor2>(v)
                 : step == 2 ? dpp_d<kDppHalfMirror>(v) : dpp_d<kDppMirror>(v);
    }
    template <typename T, typename C>
    NH_DEV static T part(T v, C comb)
    {
#pragma unroll
        for (int i = 0; i < (NT == 4 ? 2 : 4); i++) v = comb(v, dpp(v, i));
        if constexpr (NT >= 32) v = comb(v, __shfl_xor(v, 16, 64));
        if constexpr (NT >= 64) v = comb(v, __shfl_xor(v, 32, 64));
        return v;
    }
    template <typename T, typename C>
    NH_DEV static T across(T w, T *lds, C comb)
    {
        if constexpr (kWaves == 1) {
            return w;
        } else {
            if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = w;
            __syncthreads();
            T r = lds[0];
#pragma unroll
            for (int i = 1; i < kWaves; i++) r = comb(r, lds[i]);
            return r;
        }
    }
    NH_DEV static float max(float v, float *lds)
    {
        const auto comb = [](float a, float b) { return __builtin_fmaxf(a, b); };
        return across(part(v, comb), lds, comb);
    }
    NH_DEV static double max(double v, double *lds)
    {
        const auto comb = [](double a, double b) { return __builtin_fmax(a, b); };
        return across(part(v, comb), lds, comb);
    }
    NH_DEV static double sum(double v, double *lds)
    {
        const auto comb = [](double a, double b) { return a + b; };
        return across(part(v, comb), lds, comb);
    }
};

// Unused dynamic LDS that the check-free f32 kernels of groups within a wave (4
// or more vectors per lane) are launched with: it holds residency to 4 blocks of
// 256 lanes (4, 8 or 16 rows) per CU.  Fewer rows in flight suit the memory here:
// [65536, 1024] softmax 85.6 us with 8 blocks, 84.2 with 6, 81.9 with 4, 83.8 with
// 3; fused cross-entropy 95.0 / 93.9 / 89.9 / 91.6 us.  8 -> 4 blocks elsewhere:
// [262144, 256] softmax 84.0 -> 81.2, fused 93.5 -> 90.5, [131072, 512] softmax 84.3
// -> 81.1, [32768, 2048] 87.3 -> 86.3, [16384, 4096] alike.
constexpr unsigned kFullRowsLds = 40000;

// How a row of `cols` values is cut: ncv vectors from its first value, `rem`
// values past them; lane l < rem holds value sc(l) as a scalar.  The cut goes
// by index alone: which lane holds a value, and so the order of the row's
// sums, does not depend on where the row lies in memory.
template <typename T>
struct RowCut {
    static constexpr int VN = Vec16<T>::n;
    int ncv, rem;
    NH_DEV explicit RowCut(int64_t cols) : ncv(int(cols / VN)), rem(int(cols % VN)) {}
    NH_DEV int64_t sc(int lane) const { return int64_t(ncv) * VN + lane; }
};

}  // namespace nh
