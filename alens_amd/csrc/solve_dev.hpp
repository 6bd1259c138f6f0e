// solve_dev.hpp -- device helpers shared by the BBPGD kernels (k_solve.hip, k_resident.hip): the
// partial-sum slots, the wave folds of the fixed reduction order and small vector types.
#pragma once
#include "alens_dev.hpp"
#include "alens_internal.hpp"

namespace alens {

// Polls before a wait of a solver kernel gives up, sets the abort word and leaves: a minute or so, since blocks may
// start late beside other work on the GPU, or be held up by it.
constexpr uint32_t kSpinLimit = 1u << 26;

// partial sums of a chunk: s.s, s.y, y.y, max residual, non-finite count; cold-start residual and count
enum : int { Q_SS = 0, Q_SY = 1, Q_YY = 2, Q_RMAX = 3, Q_NF = 4, Q_RC = 5, Q_NFC = 6 };
// state of a system, and the modes of the two phases
enum : int { S_ACTIVE = 0, S_CONVERGED = 1, S_NONFINITE = 2, S_NOCONV = 3 };
enum : int { A_PROJ = 0, A_GRAD = 1 };
enum : int { B_INIT = 0, B_ALPHA0 = 1, B_ITER = 2 };

template <typename T>
__device__ inline typename Vec2<T>::type mk2(T x, T y);
template <>
__device__ inline double2 mk2<double>(double x, double y) {
    return make_double2(x, y);
}
template <>
__device__ inline float2 mk2<float>(float x, float y) {
    return make_float2(x, y);
}

// Halving fold of one wave: lane l takes lane l + h for h = 32, 16, ..., 1 (sums: x + o; maxima:
// o > x ? o : x) and the result is read from lane 0.  The partner values come from the gfx950 lane
// swaps (h = 32 and 16) and DPP row shifts (h <= 8), register moves without the LDS round trip of a
// general shuffle; lanes at or above h receive values that never reach lane 0.
__device__ inline double lanes_up32(double x) {
    const unsigned lo = (unsigned)__double2loint(x), hi = (unsigned)__double2hiint(x);
    const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return __hiloint2double((int)b[1], (int)a[1]);
}
__device__ inline double lanes_up16(double x) {
    const unsigned lo = (unsigned)__double2loint(x), hi = (unsigned)__double2hiint(x);
    const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return __hiloint2double((int)b[1], (int)a[1]);
}
template <int H>
__device__ inline double lanes_up_row(double x) {  // DPP row_shl:H (H < 16)
    const unsigned lo = (unsigned)__double2loint(x), hi = (unsigned)__double2hiint(x);
    return __hiloint2double((int)__builtin_amdgcn_update_dpp(0u, hi, 0x100 + H, 0xF, 0xF, true),
                            (int)__builtin_amdgcn_update_dpp(0u, lo, 0x100 + H, 0xF, 0xF, true));
}
template <bool MAX>
__device__ inline double fold_step(double x, double o) {
    if (MAX) return o > x ? o : x;
    return x + o;
}
template <bool MAX>
__device__ inline double wave_fold(double x) {
    x = fold_step<MAX>(x, lanes_up32(x));
    x = fold_step<MAX>(x, lanes_up16(x));
    x = fold_step<MAX>(x, lanes_up_row<8>(x));
    x = fold_step<MAX>(x, lanes_up_row<4>(x));
    x = fold_step<MAX>(x, lanes_up_row<2>(x));
    x = fold_step<MAX>(x, lanes_up_row<1>(x));
    return x;
}

}  // namespace alens
