// The 2- and 3-body polynomials evaluated through their relabelling groups:
//   E(x) = R(x) + sum over the relabellings h of Q(x o h),
// one pass of Q per relabelling (pip_orbit_gen.h, generated by gen_pip.py; 8
// passes for a dimer, 24 for a trimer, R empty for the dimer).  Between passes
// the variable registers x and the gradient registers g are permuted by one of
// two fixed relabellings (steps a and b), along a cycle that visits every
// relabelling once and ends in the original labelling: after pass k the
// registers hold y[m] = x[h_k[m]], and g[m] holds dE/dx[h_k[m]] so far.  Q's
// code is one loop body of a few thousand instructions (it stays in the
// instruction cache) and reads its coefficients in order from a table.
//
// Shared by the device kernels and a host build (the CPU test compiles it with
// g++); the includer defines PIP_FENCE(v) and PIP_OPAQUE_PTR(p), empty asm
// statements on the device that keep the compiler from hoisting products of the
// variables out of their blocks and the coefficient loads out of the loop, and
// PIP_CONST_PTR(T), the type of a pointer to the coefficient table.
#pragma once
#include "pip_orbit_gen.h"

namespace mbpol {

// The coefficient tables; PIP_CONST_PTR(T) is the pointer type they are read
// through (on the device one into the constant address space, so that the
// reads are scalar loads).
template <typename T>
struct pip_orbit_tables;
template <>
struct pip_orbit_tables<double> {
    static __host__ __device__ __forceinline__ PIP_CONST_PTR(double) dimer() {
        return (PIP_CONST_PTR(double))pip2b_orbit_coef_f64;
    }
    static __host__ __device__ __forceinline__ PIP_CONST_PTR(double) trimer() {
        return (PIP_CONST_PTR(double))pip3b_orbit_coef_f64;
    }
};
template <>
struct pip_orbit_tables<float> {
    static __host__ __device__ __forceinline__ PIP_CONST_PTR(float) dimer() {
        return (PIP_CONST_PTR(float))pip2b_orbit_coef_f32;
    }
    static __host__ __device__ __forceinline__ PIP_CONST_PTR(float) trimer() {
        return (PIP_CONST_PTR(float))pip3b_orbit_coef_f32;
    }
};

// Passes k0 .. k1 - 1 of Q over the group.  On entry the registers hold the
// labelling before pass k0, on return the one after pass k1 - 1.
// Pass(x, g, cf) adds one pass's gradient into g and returns its energy.
template <typename T, int N, typename Pass, typename Table>
__host__ __device__ __forceinline__ T pip_orbit_passes(T (&x)[N], T (&g)[N], Pass pass, Table table, int k0, int k1,
                                                       unsigned step_mask, const int (&step_a)[N],
                                                       const int (&step_b)[N]) {
    T e = T(0);
#pragma nounroll
    for (int k = k0; k < k1; ++k) {
        auto cf = table();
        PIP_OPAQUE_PTR(cf);
        e += pass(x, g, cf);
        T tx[N], tg[N];
        if ((step_mask >> k) & 1u) {
#pragma unroll
            for (int m = 0; m < N; ++m) {
                tx[m] = x[step_a[m]];
                tg[m] = g[step_a[m]];
            }
        } else {
#pragma unroll
            for (int m = 0; m < N; ++m) {
                tx[m] = x[step_b[m]];
                tg[m] = g[step_b[m]];
            }
        }
#pragma unroll
        for (int m = 0; m < N; ++m) {
            x[m] = tx[m];
            g[m] = tg[m];
        }
    }
    return e;
}

template <typename T>
__host__ __device__ __forceinline__ T pip3b_orbit_passes(T (&x)[36], T (&g)[36], int k0, int k1) {
    return pip_orbit_passes<T, 36>(
        x, g, [](T (&y)[36], T (&h)[36], PIP_CONST_PTR(T) cf) { return pip3b_orbit_pass<T>(y, h, cf); },
        [] { return pip_orbit_tables<T>::trimer(); }, k0, k1, pip3b_step_mask, pip3b_step_a, pip3b_step_b);
}
template <typename T>
__host__ __device__ __forceinline__ T pip2b_orbit_passes(T (&x)[31], T (&g)[31], int k0, int k1) {
    return pip_orbit_passes<T, 31>(
        x, g, [](T (&y)[31], T (&h)[31], PIP_CONST_PTR(T) cf) { return pip2b_orbit_pass<T>(y, h, cf); },
        [] { return pip_orbit_tables<T>::dimer(); }, k0, k1, pip2b_step_mask, pip2b_step_a, pip2b_step_b);
}

// E(x) and dE/dx (into g, overwritten) of the 3-body polynomial; x is left as it was.
template <typename T>
__host__ __device__ __forceinline__ T pip3b_orbit_eval(T (&x)[36], T (&g)[36]) {
    const T e = pip3b_rest<T>(x, g);
    return e + pip3b_orbit_passes<T>(x, g, 0, pip3b_npass);
}

// the same for the 2-body polynomial (R is empty)
template <typename T>
__host__ __device__ __forceinline__ T pip2b_orbit_eval(T (&x)[31], T (&g)[31]) {
    const T e = pip2b_rest<T>(x, g);
    return e + pip2b_orbit_passes<T>(x, g, 0, pip2b_npass);
}

}  // namespace mbpol
