// 2-body and 3-body permutationally invariant polynomial kernels.
//
// One dimer (trimer) per lane.  Positions are read and minimum-imaged in FP64,
// then made relative to the first oxygen so that the arithmetic type T
// (float on the mixed-precision path, double on the FP64 path) only ever sees
// small coordinates.  The polynomial itself (generated, pip_eval_gen.h) keeps
// variables, gradients and coefficients in registers.  Per-atom forces are
// accumulated in T inside the lane and scattered once as 64-bit fixed point;
// the first molecule's are first summed over the lanes that share it (the
// lists are ordered by first molecule), one atomic per run of lanes.
//
// This file is compiled once per body order and arithmetic type:
//   -DPIP_BODY=2|3  -DPIP_REAL=float|double
// with -DPIP_ORBIT=1 the polynomial is evaluated through the relabelling group
// of the dimer or trimer (pip_orbit_loop.h) instead of term by term.
#include <algorithm>
#include <type_traits>

#include "device_common.h"
// an empty asm that re-defines a variable in its register: no instruction
#define PIP_FENCE(v) asm volatile("" : "+v"(v))
// the same for a uniform pointer in scalar registers
#define PIP_OPAQUE_PTR(p) asm volatile("" : "+s"(p))
// tables read through the constant address space: scalar loads
#define PIP_CONST_PTR(T) const __attribute__((address_space(4))) T*
#if PIP_ORBIT
#include "pip_orbit_loop.h"
#else
#include "pip_eval_gen.h"
#endif
#ifndef PIP_BODY
#error "PIP_BODY must be 2 or 3"
#endif
#ifndef PIP_REAL
#error "PIP_REAL must be float or double"
#endif

namespace mbpol {
namespace {  // kernels have internal linkage: this file is compiled once per body order and type
using namespace mbpol_params;
typedef PIP_REAL real;
typedef v3<real> vr;

// image_to by products with 1/L, for a hydrogen about its own oxygen: the image index differs from the one
// the quotient gives only where a separation is within rounding of half the box, which no O-H distance is.
// Oxygens take image_to: a third molecule half a box from the first has a switch of zero with it, but which
// of its images is taken decides its distance from the second.
__device__ __forceinline__ d3 image_near(const d3& ref, const d3& p, const d3& L, const d3& iL) {
    return d3{p.x + L.x * floor((ref.x - p.x) * iL.x + 0.5), p.y + L.y * floor((ref.y - p.y) * iL.y + 0.5),
              p.z + L.z * floor((ref.z - p.z) * iL.z + 0.5)};
}

#if !PIP_ORBIT
__device__ __forceinline__ vr rel(const d3& p, const d3& o) { return vr((real)(p.x - o.x), (real)(p.y - o.y), (real)(p.z - o.z)); }
#else
// Forces of one molecule {idx[3 mol ..]} added by the lane that holds its run's sums.
__device__ __forceinline__ void add_molecule(u64* __restrict__ force, const int* __restrict__ idx, long long mol,
                                             bool last, const u64 (&f)[9]) {
    if (!last || mol < 0) return;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int a = idx[3 * mol + q];
#pragma unroll
        for (int d = 0; d < 3; ++d) atomicAdd(&force[3 * a + d], f[3 * q + d]);
    }
}
#endif

#if PIP_BODY == 2
// ---------------------------------------------------------------------------
// 2-body: platforms/reference/src/MBPolReferenceTwoBodyForce.cpp:110-296 and
// mbpol_2body_constants.cpp:10-111.  Points (Angstrom, relative to Oa):
// 0 Oa 1 Ha1 2 Ha2 3 Ob 4 Hb1 5 Hb2 6 Xa1 7 Xa2 8 Xb1 9 Xb2.
// ---------------------------------------------------------------------------
struct Var2 {
    int a, b, coul;
    double k, r0;
};
// the 31 variables in reference order (:170-207)
#define V2(a, b, c, k, r) {a, b, c, k, r}
__host__ __device__ constexpr Var2 var2(int n) {
    const double di = tb_d0_intra, de = tb_d0_inter;
    switch (n) {
        case 0: return V2(1, 2, 0, tb_k_HH_intra, di);
        case 1: return V2(4, 5, 0, tb_k_HH_intra, di);
        case 2: return V2(0, 1, 0, tb_k_OH_intra, di);
        case 3: return V2(0, 2, 0, tb_k_OH_intra, di);
        case 4: return V2(3, 4, 0, tb_k_OH_intra, di);
        case 5: return V2(3, 5, 0, tb_k_OH_intra, di);
        case 6: return V2(1, 4, 1, tb_k_HH_coul, de);
        case 7: return V2(1, 5, 1, tb_k_HH_coul, de);
        case 8: return V2(2, 4, 1, tb_k_HH_coul, de);
        case 9: return V2(2, 5, 1, tb_k_HH_coul, de);
        case 10: return V2(0, 4, 1, tb_k_OH_coul, de);
        case 11: return V2(0, 5, 1, tb_k_OH_coul, de);
        case 12: return V2(3, 1, 1, tb_k_OH_coul, de);
        case 13: return V2(3, 2, 1, tb_k_OH_coul, de);
        case 14: return V2(0, 3, 1, tb_k_OO_coul, de);
        case 15: return V2(6, 4, 0, tb_k_XH_main, de);
        case 16: return V2(6, 5, 0, tb_k_XH_main, de);
        case 17: return V2(7, 4, 0, tb_k_XH_main, de);
        case 18: return V2(7, 5, 0, tb_k_XH_main, de);
        case 19: return V2(8, 1, 0, tb_k_XH_main, de);
        case 20: return V2(8, 2, 0, tb_k_XH_main, de);
        case 21: return V2(9, 1, 0, tb_k_XH_main, de);
        case 22: return V2(9, 2, 0, tb_k_XH_main, de);
        case 23: return V2(0, 8, 0, tb_k_XO_main, de);
        case 24: return V2(0, 9, 0, tb_k_XO_main, de);
        case 25: return V2(3, 6, 0, tb_k_XO_main, de);
        case 26: return V2(3, 7, 0, tb_k_XO_main, de);
        case 27: return V2(6, 8, 0, tb_k_XX_main, de);
        case 28: return V2(6, 9, 0, tb_k_XX_main, de);
        case 29: return V2(7, 8, 0, tb_k_XX_main, de);
        default: return V2(7, 9, 0, tb_k_XX_main, de);
    }
}
#undef V2

// extra points of one monomer (mbpol_2body_constants.cpp:62-76)
template <typename T>
__device__ __forceinline__ void extra_points(const v3<T>& O, const v3<T>& H1, const v3<T>& H2, v3<T>& x1, v3<T>& x2) {
    const v3<T> oh1 = H1 - O, oh2 = H2 - O;
    const v3<T> in_plane = O + (oh1 + oh2) * (T)(0.5 * tb_in_plane_gamma);
    const v3<T> out_of_plane = oh1.cross(oh2) * (T)tb_out_of_plane_gamma;
    x1 = in_plane + out_of_plane;
    x2 = in_plane - out_of_plane;
}

// back-propagation of the extra-point gradients (mbpol_2body_constants.cpp:80-96)
__device__ __forceinline__ void extra_grads(const vr& O, const vr& H1, const vr& H2, const vr& g1, const vr& g2, vr& fO,
                                            vr& fH1, vr& fH2) {
    const vr oh1 = H1 - O, oh2 = H2 - O;
    const vr gm = g1 - g2;
    const vr t1 = oh2.cross(gm), t2 = oh1.cross(gm);
    const vr gsum = g1 + g2;
    const vr in_plane = gsum * (real)(0.5 * tb_in_plane_gamma);
    const vr gh1 = in_plane + t1 * (real)tb_out_of_plane_gamma;
    const vr gh2 = in_plane - t2 * (real)tb_out_of_plane_gamma;
    fO += gsum - (gh1 + gh2);
    fH1 += gh1;
    fH2 += gh2;
}

#if !PIP_ORBIT
// Geometry of dimer t: atom indices, imaged positions (Angstrom) and, when the
// O-O distance is inside [2, r2f] Angstrom, the ten points relative to Oa.
// Returns whether the dimer contributes.
__device__ __forceinline__ bool dimer_geometry(long long t, const int2* __restrict__ pairs,
                                               const int* __restrict__ idx, const double* __restrict__ pos,
                                               int periodic, const d3& boxA, int (&at)[6], vr (&R)[10],
                                               d3& dOO, double& rOO) {
    const int2 pr = pairs[t];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        at[q] = idx[3 * pr.x + q];
        at[3 + q] = idx[3 * pr.y + q];
    }
    d3 P[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const d3 p = load_d3(pos, at[q]);
        P[q] = d3{p.x * 10., p.y * 10., p.z * 10.};
    }
    if (periodic) {  // imageMolecules (MBPolReferenceTwoBodyForce.cpp:78-100)
        const d3 iL{1.0 / boxA.x, 1.0 / boxA.y, 1.0 / boxA.z};
        P[1] = image_near(P[0], P[1], boxA, iL);
        P[2] = image_near(P[0], P[2], boxA, iL);
        P[3] = image_to(P[0], P[3], boxA);
        P[4] = image_near(P[3], P[4], boxA, iL);
        P[5] = image_near(P[3], P[5], boxA, iL);
    }
    dOO = d3{P[0].x - P[3].x, P[0].y - P[3].y, P[0].z - P[3].z};
    rOO = sqrt(dOO.x * dOO.x + dOO.y * dOO.y + dOO.z * dOO.z);
    if (!(rOO <= tb_r2f && rOO >= 2.)) return false;
#pragma unroll
    for (int q = 0; q < 6; ++q) R[q] = rel(P[q], P[0]);
    extra_points(R[0], R[1], R[2], R[6], R[7]);
    extra_points(R[3], R[4], R[5], R[8], R[9]);
    return true;
}
#endif

// switch and its derivative (mbpol_2body_constants.cpp:98-111), FP64
__device__ __forceinline__ void switch2(double rOO, double& sw, double& gsw) {
    if (rOO > tb_r2i) {
        constexpr double t1 = 1.0 / (tb_r2f - tb_r2i);
        double sn, cs;
        sincospi((rOO - tb_r2i) * t1, &sn, &cs);  // the argument in units of pi: no range reduction
        gsw = -sn * (0.5 * M_PI * t1);
        sw = (1.0 + cs) / 2.0;
    } else {
        sw = 1.0;
        gsw = 0.0;
    }
}

#if PIP_ORBIT
typedef v3<double> vd;
// the ten points of dimer t relative to Oa, Angstrom; whether it contributes
__device__ __forceinline__ bool unit_geometry(long long t, const int2* __restrict__ pairs, const int* __restrict__ idx,
                                              const double* __restrict__ pos, int periodic, const d3& box, vd (&R)[10]) {
    const int2 pr = pairs[t];
    d3 P[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const d3 p = load_d3(pos, idx[3 * (q < 3 ? pr.x : pr.y) + q % 3]);
        P[q] = d3{p.x * 10., p.y * 10., p.z * 10.};
    }
    if (periodic) {  // imageMolecules (MBPolReferenceTwoBodyForce.cpp:78-100)
        const d3 L{box.x * 10., box.y * 10., box.z * 10.}, iL{1.0 / L.x, 1.0 / L.y, 1.0 / L.z};
        P[1] = image_near(P[0], P[1], L, iL);
        P[2] = image_near(P[0], P[2], L, iL);
        P[3] = image_to(P[0], P[3], L);
        P[4] = image_near(P[3], P[4], L, iL);
        P[5] = image_near(P[3], P[5], L, iL);
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) R[q] = vd(P[q].x - P[0].x, P[q].y - P[0].y, P[q].z - P[0].z);
    extra_points(R[0], R[1], R[2], R[6], R[7]);
    extra_points(R[3], R[4], R[5], R[8], R[9]);
    const double r = sqrt(R[3].dot(R[3]));
    return r <= tb_r2f && r >= 2.;
}

__device__ __forceinline__ PIP_CONST_PTR(int) label_table() { return (PIP_CONST_PTR(int))pip2b_label; }
template <typename T>
__device__ __forceinline__ T passes(T (&x)[31], T (&g)[31], int k0, int k1) {
    return pip2b_orbit_passes<T>(x, g, k0, k1);
}

// step 5: forces of molecule `part` (0, 1) or the energy (2)
__device__ __forceinline__ void unit_end(int part, bool on, long long t, bool in, double E, const double (&rs)[30][64],
                                         const real (&fs)[30][64], const int2* __restrict__ pairs,
                                         const int* __restrict__ idx, u64* __restrict__ force,
                                         u64* __restrict__ energy, double* __restrict__ eunit, int lane) {
    const vd b(rs[9][lane], rs[10][lane], rs[11][lane]);  // Oa -> Ob
    double sw = 0.0, gsw = 0.0;
    const double r = sqrt(b.dot(b));
    if (on) switch2(r, sw, gsw);
    if (part == 2) {
        const double e = on ? sw * E * cal2joule : 0.0;
        if (eunit && in) eunit[t] = e;
        add_energy(energy, e);
        return;
    }
    u64 f[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    long long key = in ? (long long)(part ? pairs[t].y : pairs[t].x) : -1;
    if (on) {
        auto point = [&](const auto& v, int q) { return vr((real)v[3 * q][lane], (real)v[3 * q + 1][lane], (real)v[3 * q + 2][lane]); };
        const int o = 3 * part, x = 6 + 2 * part;
        vr F[3] = {point(fs, o), point(fs, o + 1), point(fs, o + 2)};
        extra_grads(point(rs, o), point(rs, o + 1), point(rs, o + 2), point(fs, x), point(fs, x + 1), F[0], F[1], F[2]);
        const double s = sw * cal2joule * -10.;
        // of the switch, on the oxygens along Oa - Ob
        const double gq = gsw * E / r * cal2joule * (part ? -10. : 10.);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            double fx = (double)F[q].x * s, fy = (double)F[q].y * s, fz = (double)F[q].z * s;
            if (q == 0) {
                fx += gq * b.x;
                fy += gq * b.y;
                fz += gq * b.z;
            }
            f[3 * q] = to_fix(fx);
            f[3 * q + 1] = to_fix(fy);
            f[3 * q + 2] = to_fix(fz);
        }
    }
    // the first molecule's forces over the wave's runs of dimers that share it, the second's after a sort
    const bool last = part == 0 ? wave_run_sum(key, f) : wave_sorted_run_sum(key, f);
    add_molecule(force, idx, key, last, f);
}
#endif

#if !PIP_ORBIT
__global__ void __launch_bounds__(64) k_twobody(long long np, const long long* __restrict__ ndev,
                                                const int2* __restrict__ pairs, const int* __restrict__ idx,
                                                const double* __restrict__ pos, int periodic, d3 boxA,
                                                u64* __restrict__ force, u64* __restrict__ energy,
                                                double* __restrict__ eunit) {
    // np: the list's capacity; ndev (when given): its length, known on the device only
    if (ndev) np = min(np, *ndev);
    // a capped grid strides over the list in whole waves
    for (long long t0 = (long long)blockIdx.x * blockDim.x; t0 < np; t0 += (long long)gridDim.x * blockDim.x) {
        const long long t = t0 + threadIdx.x;
        double e_out = 0.0;
        int at[6];
        vr R[10];
        d3 dOO;
        double rOO;
        // forces on the first molecule, summed over the wave's runs of dimers that share it, and
        // on the second, summed over the wave's dimers that share it after a sort by molecule
        u64 fa[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        u64 fb[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        const long long key = t < np ? (long long)pairs[t].x : -1;
        long long key2 = t < np ? (long long)pairs[t].y : -1;
        if (t < np && dimer_geometry(t, pairs, idx, pos, periodic, boxA, at, R, dOO, rOO)) {
            real x[31], g[31];
#pragma unroll
            for (int n = 0; n < 31; ++n) {
                const Var2 v = var2(n);
                const vr d = R[v.a] - R[v.b];
                const real r = sqrt(d.dot(d));
                const real e = exp_t<real>((real)v.k * ((real)v.r0 - r));
                x[n] = v.coul ? e / r : e;
            }
            real Ep = pip2b_eval<real>(x, g);
            // Only t, Ep and g stay live across the polynomial: the geometry is
            // reloaded from memory (the opaque copy of t keeps the compiler from
            // holding the first loads in registers through the polynomial).
            long long tt = t;
            asm volatile("" : "+v"(tt));
            asm volatile("" : "+v"(Ep));
#pragma unroll
            for (int n = 0; n < 31; ++n) asm volatile("" : "+v"(g[n]));
            dimer_geometry(tt, pairs, idx, pos, periodic, boxA, at, R, dOO, rOO);
            // chain rule through the variables
            vr F[10];
#pragma unroll
            for (int q = 0; q < 10; ++q) F[q] = vr(0, 0, 0);
#pragma unroll
            for (int n = 0; n < 31; ++n) {
                const Var2 v = var2(n);
                const vr d = R[v.a] - R[v.b];
                const real r = sqrt(d.dot(d));
                const real e = exp_t<real>((real)v.k * ((real)v.r0 - r));
                real gg;
                if (v.coul) {
                    const real ri = (real)1 / r, val = e * ri;
                    gg = -((real)v.k + ri) * val * ri;
                } else {
                    gg = -(real)v.k * e / r;
                }
                const vr dd = d * (gg * g[n]);
                F[v.a] += dd;
                F[v.b] -= dd;
            }
            extra_grads(R[0], R[1], R[2], F[6], F[7], F[0], F[1], F[2]);
            extra_grads(R[3], R[4], R[5], F[8], F[9], F[3], F[4], F[5]);
            double sw, gsw;
            switch2(rOO, sw, gsw);
            const double s = sw * cal2joule * -10.;
            const double gs = gsw * (double)Ep / rOO * cal2joule * -10.;
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                double fx = (double)F[q].x * s, fy = (double)F[q].y * s, fz = (double)F[q].z * s;
                if (q == 0) { fx += gs * dOO.x; fy += gs * dOO.y; fz += gs * dOO.z; }
                if (q == 3) { fx -= gs * dOO.x; fy -= gs * dOO.y; fz -= gs * dOO.z; }
                if (q < 3) {
                    fa[3 * q] = to_fix(fx);
                    fa[3 * q + 1] = to_fix(fy);
                    fa[3 * q + 2] = to_fix(fz);
                } else {
                    fb[3 * (q - 3)] = to_fix(fx);
                    fb[3 * (q - 3) + 1] = to_fix(fy);
                    fb[3 * (q - 3) + 2] = to_fix(fz);
                }
            }
            e_out = sw * (double)Ep * cal2joule;
        }
        if (wave_run_sum(key, fa) && key >= 0) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int a = idx[3 * key + q];
#pragma unroll
                for (int d = 0; d < 3; ++d) atomicAdd(&force[3 * a + d], fa[3 * q + d]);
            }
        }
        if (wave_sorted_run_sum(key2, fb) && key2 >= 0) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int a = idx[3 * key2 + q];
#pragma unroll
                for (int d = 0; d < 3; ++d) atomicAdd(&force[3 * a + d], fb[3 * q + d]);
            }
        }
        if (eunit && t < np) eunit[t] = e_out;
        add_energy(energy, e_out);
    }
}
#endif

#else
// ---------------------------------------------------------------------------
// 3-body: platforms/reference/src/MBPolReferenceThreeBodyForce.cpp:67-293.
// Points (nm, relative to Oa): 0 Oa 1 Ha1 2 Ha2 3 Ob 4 Hb1 5 Hb2 6 Oc 7 Hc1 8 Hc2.
// ---------------------------------------------------------------------------
struct Var3 {
    int a, b, coul;
    double k, r0;
};
#define V3(a, b, k, r) {a, b, 0, k, r}
__host__ __device__ constexpr Var3 var3(int n) {
    switch (n) {  // reference order (:170-206)
        case 0: return V3(1, 2, th_kHH_intra, th_dHH_intra);
        case 1: return V3(4, 5, th_kHH_intra, th_dHH_intra);
        case 2: return V3(7, 8, th_kHH_intra, th_dHH_intra);
        case 3: return V3(0, 1, th_kOH_intra, th_dOH_intra);
        case 4: return V3(0, 2, th_kOH_intra, th_dOH_intra);
        case 5: return V3(3, 4, th_kOH_intra, th_dOH_intra);
        case 6: return V3(3, 5, th_kOH_intra, th_dOH_intra);
        case 7: return V3(6, 7, th_kOH_intra, th_dOH_intra);
        case 8: return V3(6, 8, th_kOH_intra, th_dOH_intra);
        case 9: return V3(1, 4, th_kHH, th_dHH);
        case 10: return V3(1, 5, th_kHH, th_dHH);
        case 11: return V3(1, 7, th_kHH, th_dHH);
        case 12: return V3(1, 8, th_kHH, th_dHH);
        case 13: return V3(2, 4, th_kHH, th_dHH);
        case 14: return V3(2, 5, th_kHH, th_dHH);
        case 15: return V3(2, 7, th_kHH, th_dHH);
        case 16: return V3(2, 8, th_kHH, th_dHH);
        case 17: return V3(4, 7, th_kHH, th_dHH);
        case 18: return V3(4, 8, th_kHH, th_dHH);
        case 19: return V3(5, 7, th_kHH, th_dHH);
        case 20: return V3(5, 8, th_kHH, th_dHH);
        case 21: return V3(0, 4, th_kOH, th_dOH);
        case 22: return V3(0, 5, th_kOH, th_dOH);
        case 23: return V3(0, 7, th_kOH, th_dOH);
        case 24: return V3(0, 8, th_kOH, th_dOH);
        case 25: return V3(3, 1, th_kOH, th_dOH);
        case 26: return V3(3, 2, th_kOH, th_dOH);
        case 27: return V3(3, 7, th_kOH, th_dOH);
        case 28: return V3(3, 8, th_kOH, th_dOH);
        case 29: return V3(6, 1, th_kOH, th_dOH);
        case 30: return V3(6, 2, th_kOH, th_dOH);
        case 31: return V3(6, 4, th_kOH, th_dOH);
        case 32: return V3(6, 5, th_kOH, th_dOH);
        case 33: return V3(0, 3, th_kOO, th_dOO);
        case 34: return V3(0, 6, th_kOO, th_dOO);
        default: return V3(3, 6, th_kOO, th_dOO);
    }
}
#undef V3

__device__ __forceinline__ double switch3(double r, double& g) {  // (:103-120)
    if (r > th_r3f) { g = 0.0; return 0.0; }
    if (r > th_r3i) {
        constexpr double t1 = 1.0 / (th_r3f - th_r3i);
        double sn, cs;
        sincospi((r - th_r3i) * t1, &sn, &cs);  // the argument in units of pi: no range reduction
        g = -sn * (0.5 * M_PI * t1);
        return (1.0 + cs) / 2.0;
    }
    g = 0.0;
    return 1.0;
}

#if !PIP_ORBIT
// Geometry of trimer t: atom indices, imaged positions, the three O-O vectors
// (Angstrom) and, unless an O-O distance is below 2 Angstrom (:160-163), the
// nine points in Angstrom relative to Oa.  Returns whether the trimer contributes.
__device__ __forceinline__ bool trimer_geometry(long long t, const int* __restrict__ trip, const int* __restrict__ idx,
                                                const double* __restrict__ pos, int periodic, const d3& box,
                                                int (&at)[9], vr (&R)[9], d3 (&roo)[3], double (&doo)[3]) {
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const int mol = trip[3 * t + m];
#pragma unroll
        for (int q = 0; q < 3; ++q) at[3 * m + q] = idx[3 * mol + q];
    }
    d3 P[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) P[q] = load_d3(pos, at[q]);
    if (periodic) {  // imageMolecules in nm (MBPolReferenceTwoBodyForce.cpp:78-109)
        const d3 iL{1.0 / box.x, 1.0 / box.y, 1.0 / box.z};
        P[1] = image_near(P[0], P[1], box, iL);
        P[2] = image_near(P[0], P[2], box, iL);
        P[3] = image_to(P[0], P[3], box);
        P[4] = image_near(P[3], P[4], box, iL);
        P[5] = image_near(P[3], P[5], box, iL);
        P[6] = image_to(P[0], P[6], box);
        P[7] = image_near(P[6], P[7], box, iL);
        P[8] = image_near(P[6], P[8], box, iL);
    }
    roo[0] = d3{(P[0].x - P[3].x) * 10., (P[0].y - P[3].y) * 10., (P[0].z - P[3].z) * 10.};  // ab
    roo[1] = d3{(P[0].x - P[6].x) * 10., (P[0].y - P[6].y) * 10., (P[0].z - P[6].z) * 10.};  // ac
    roo[2] = d3{(P[3].x - P[6].x) * 10., (P[3].y - P[6].y) * 10., (P[3].z - P[6].z) * 10.};  // bc
#pragma unroll
    for (int q = 0; q < 3; ++q) doo[q] = sqrt(roo[q].x * roo[q].x + roo[q].y * roo[q].y + roo[q].z * roo[q].z);
    if (doo[0] < 2 || doo[1] < 2 || doo[2] < 2) return false;
    const d3 o{P[0].x * 10., P[0].y * 10., P[0].z * 10.};
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const d3 p{P[q].x * 10., P[q].y * 10., P[q].z * 10.};
        R[q] = rel(p, o);
    }
    return true;
}
#endif

#if PIP_ORBIT
typedef v3<double> vd;
// the nine points of trimer t relative to Oa, Angstrom; whether it contributes
__device__ __forceinline__ bool unit_geometry(long long t, const int* __restrict__ trip, const int* __restrict__ idx,
                                              const double* __restrict__ pos, int periodic, const d3& box, vd (&R)[9]) {
    d3 P[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) P[q] = load_d3(pos, idx[3 * trip[3 * t + q / 3] + q % 3]);
    if (periodic) {  // imageMolecules in nm (MBPolReferenceTwoBodyForce.cpp:78-109)
        const d3 iL{1.0 / box.x, 1.0 / box.y, 1.0 / box.z};
        P[1] = image_near(P[0], P[1], box, iL);
        P[2] = image_near(P[0], P[2], box, iL);
        P[3] = image_to(P[0], P[3], box);
        P[4] = image_near(P[3], P[4], box, iL);
        P[5] = image_near(P[3], P[5], box, iL);
        P[6] = image_to(P[0], P[6], box);
        P[7] = image_near(P[6], P[7], box, iL);
        P[8] = image_near(P[6], P[8], box, iL);
    }
#pragma unroll
    for (int q = 0; q < 9; ++q) R[q] = vd((P[q].x - P[0].x) * 10., (P[q].y - P[0].y) * 10., (P[q].z - P[0].z) * 10.);
    const vd bc = R[3] - R[6];
    // nothing below 2 Angstrom (:160-163)
    return !(R[3].dot(R[3]) < 4. || R[6].dot(R[6]) < 4. || bc.dot(bc) < 4.);
}

__device__ __forceinline__ PIP_CONST_PTR(int) label_table() { return (PIP_CONST_PTR(int))pip3b_label; }
template <typename T>
__device__ __forceinline__ T passes(T (&x)[36], T (&g)[36], int k0, int k1) {
    return pip3b_orbit_passes<T>(x, g, k0, k1);
}

// step 5: forces of molecule `part` (0 .. 2) or the energy (3)
__device__ __forceinline__ void unit_end(int part, bool on, long long t, bool in, double E, const double (&rs)[27][64],
                                         const real (&fs)[27][64], const int* __restrict__ trip,
                                         const int* __restrict__ idx, u64* __restrict__ force,
                                         u64* __restrict__ energy, double* __restrict__ eunit, int lane) {
    const vd b(rs[9][lane], rs[10][lane], rs[11][lane]), c(rs[18][lane], rs[19][lane], rs[20][lane]), bc = b - c;
    double sab = 0, sac = 0, sbc = 0, gab = 0, gac = 0, gbc = 0;
    const double rab = sqrt(b.dot(b)), rac = sqrt(c.dot(c)), rbc = sqrt(bc.dot(bc));
    if (on) {
        sab = switch3(rab, gab);
        sac = switch3(rac, gac);
        sbc = switch3(rbc, gbc);
    }
    const double s = sab * sac + sab * sbc + sac * sbc;
    if (part == 3) {
        const double e = on ? E * s * cal2joule : 0.0;
        if (eunit && in) eunit[t] = e;
        add_energy(energy, e);
        return;
    }
    u64 f[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    long long key = in ? (long long)trip[3 * t + part] : -1;
    if (on) {
        const double fsc = s * cal2joule * 10. * -1, u = cal2joule * -nm_to_A;
        gab *= (sac + sbc) * E / rab;
        gac *= (sab + sbc) * E / rac;
        gbc *= (sab + sac) * E / rbc;
        // of the switches, on the oxygens along Oa - Ob = -b, Oa - Oc = -c, Ob - Oc = bc
        const vd w = part == 0 ? b * -gab - c * gac : part == 1 ? bc * gbc + b * gab : c * gac - bc * gbc;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int p = 3 * (3 * part + q);
            double fx = (double)fs[p][lane] * fsc, fy = (double)fs[p + 1][lane] * fsc, fz = (double)fs[p + 2][lane] * fsc;
            if (q == 0) {
                fx += w.x * u;
                fy += w.y * u;
                fz += w.z * u;
            }
            f[3 * q] = to_fix(fx);
            f[3 * q + 1] = to_fix(fy);
            f[3 * q + 2] = to_fix(fz);
        }
    }
    // the list is ordered by first, then second molecule: their forces are summed over the wave's runs of
    // trimers that share them, the third's after a sort by molecule
    const bool last = part < 2 ? wave_run_sum(key, f) : wave_sorted_run_sum(key, f);
    add_molecule(force, idx, key, last, f);
}
#endif

#if !PIP_ORBIT
__global__ void __launch_bounds__(64) k_threebody(long long nt, const long long* __restrict__ ndev,
                                                                 const int* __restrict__ trip,
                                                                 const int* __restrict__ idx,
                                                                 const double* __restrict__ pos, int periodic, d3 box,
                                                                 u64* __restrict__ force, u64* __restrict__ energy,
                                                                 double* __restrict__ eunit) {
    // nt: the list's capacity; ndev (when given): its length, known on the device only
    if (ndev) nt = min(nt, *ndev);
    // a capped grid strides over the list in whole waves
    for (long long t0 = (long long)blockIdx.x * blockDim.x; t0 < nt; t0 += (long long)gridDim.x * blockDim.x) {
        const long long t = t0 + threadIdx.x;
        double e_out = 0.0;
        int at[9];
        vr R[9];
        d3 roo[3];
        double doo[3];
        // forces on the first and on the second molecule, each summed over the wave's runs of
        // trimers that share it (the list is ordered by first, then second molecule), and on the
        // third, summed over the wave's trimers that share it after a sort by molecule
        u64 fa[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        u64 fb[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        u64 fc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        const long long key = t < nt ? (long long)trip[3 * t] : -1;
        const long long key2 = t < nt ? (long long)trip[3 * t + 1] : -1;
        long long key3 = t < nt ? (long long)trip[3 * t + 2] : -1;
        if (t < nt && trimer_geometry(t, trip, idx, pos, periodic, box, at, R, roo, doo)) {
            real x[36], g[36];
#pragma unroll
            for (int n = 0; n < 36; ++n) {
                const Var3 v = var3(n);
                const vr d = R[v.a] - R[v.b];
                const real r = sqrt(d.dot(d));
                x[n] = exp_t<real>(-(real)v.k * (r - (real)v.r0));
            }
            real Ep = pip3b_eval<real>(x, g);
            // Only t, Ep and g stay live across the polynomial; the geometry is
            // reloaded (through an opaque copy of t, so that the first loads are
            // not kept in registers).
            long long tt = t;
            asm volatile("" : "+v"(tt));
            asm volatile("" : "+v"(Ep));
#pragma unroll
            for (int n = 0; n < 36; ++n) asm volatile("" : "+v"(g[n]));
            trimer_geometry(tt, trip, idx, pos, periodic, box, at, R, roo, doo);
            double gab, gac, gbc;
            const double sab = switch3(doo[0], gab), sac = switch3(doo[1], gac), sbc = switch3(doo[2], gbc);
            const double s = sab * sac + sab * sbc + sac * sbc;
            // g_var (:80-101): forces of the variables, times s; units kJ/mol/nm
            vr F[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) F[q] = vr(0, 0, 0);
#pragma unroll
            for (int n = 0; n < 36; ++n) {
                const Var3 v = var3(n);
                const vr d = R[v.a] - R[v.b];
                const real r = sqrt(d.dot(d));
                const real gg = -(real)v.k * g[n] * exp_t<real>(-(real)v.k * (r - (real)v.r0)) / r;
                const vr dd = d * gg;
                F[v.a] += dd;
                F[v.b] -= dd;
            }
            const double fs = s * cal2joule * 10. * -1;
            const double E = (double)Ep;
            gab *= (sac + sbc) * E / doo[0];
            gac *= (sab + sbc) * E / doo[1];
            gbc *= (sab + sac) * E / doo[2];
            const double u = cal2joule * -nm_to_A;
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                double fx = (double)F[q].x * fs, fy = (double)F[q].y * fs, fz = (double)F[q].z * fs;
                if (q == 0) {
                    fx += (gab * roo[0].x + gac * roo[1].x) * u;
                    fy += (gab * roo[0].y + gac * roo[1].y) * u;
                    fz += (gab * roo[0].z + gac * roo[1].z) * u;
                } else if (q == 3) {
                    fx += (gbc * roo[2].x - gab * roo[0].x) * u;
                    fy += (gbc * roo[2].y - gab * roo[0].y) * u;
                    fz += (gbc * roo[2].z - gab * roo[0].z) * u;
                } else if (q == 6) {
                    fx -= (gac * roo[1].x + gbc * roo[2].x) * u;
                    fy -= (gac * roo[1].y + gbc * roo[2].y) * u;
                    fz -= (gac * roo[1].z + gbc * roo[2].z) * u;
                }
                if (q < 3) {
                    fa[3 * q] = to_fix(fx);
                    fa[3 * q + 1] = to_fix(fy);
                    fa[3 * q + 2] = to_fix(fz);
                } else if (q < 6) {
                    fb[3 * (q - 3)] = to_fix(fx);
                    fb[3 * (q - 3) + 1] = to_fix(fy);
                    fb[3 * (q - 3) + 2] = to_fix(fz);
                } else {
                    fc[3 * (q - 6)] = to_fix(fx);
                    fc[3 * (q - 6) + 1] = to_fix(fy);
                    fc[3 * (q - 6) + 2] = to_fix(fz);
                }
            }
            e_out = E * s * cal2joule;
        }
        if (wave_run_sum(key, fa) && key >= 0) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int a = idx[3 * key + q];
#pragma unroll
                for (int d = 0; d < 3; ++d) atomicAdd(&force[3 * a + d], fa[3 * q + d]);
            }
        }
        if (wave_run_sum(key2, fb) && key2 >= 0) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int a = idx[3 * key2 + q];
#pragma unroll
                for (int d = 0; d < 3; ++d) atomicAdd(&force[3 * a + d], fb[3 * q + d]);
            }
        }
        if (wave_sorted_run_sum(key3, fc) && key3 >= 0) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int a = idx[3 * key3 + q];
#pragma unroll
                for (int d = 0; d < 3; ++d) atomicAdd(&force[3 * a + d], fc[3 * q + d]);
            }
        }
        if (eunit && t < nt) eunit[t] = e_out;
        add_energy(energy, e_out);
    }
}
#endif
#endif

#if PIP_ORBIT
// ---------------------------------------------------------------------------
// The polynomial through the unit's relabelling group: 64 dimers (trimers) a
// block, the 8 (24) passes shared out among its 4 waves -- for a short list among
// the 4 Q waves of Q blocks.
//   1. wave 0 reads the geometry into LDS;
//   2. the waves compute the variables (LDS);
//   3. each wave takes them in the labelling its passes start from, runs its
//      passes, and adds its gradient to the block's in the original labelling,
//      one wave after the other: the sums do not depend on scheduling;
//   4. the waves take the points in turn for the chain rule;
//   5. wave m sums and adds the forces of molecule m, the wave after them the energy.
// With Q > 1 the blocks write their shares of the points' gradient and of the energy to
// memory instead, and k_pip_join adds a unit's shares in their order before step 5: a
// unit's sums are formed in floating point and rounded to fixed point once.  (The last of
// the blocks doing so in this kernel, behind fences, took as long and put registers of
// the passes into scratch.)  Q follows from the list's length on the device, not from the
// capacity the host launches by, so that a configuration's results do not depend on those
// evaluated before it.
// Steps 2 and 4 are rolled loops over tables of the variables, so that a unit's
// code outside the passes is short and, for a short list, not fetched in vain.
//
// What bounds it: FP64 issue.  A wave alone on its SIMD issues one instruction in
// 4.9 cycles, two one in 4.3 between them, and a pass is 4200 (3-body) or 4600
// (2-body) instructions.  A long list fills two waves a SIMD, which 256 registers
// allow; a short one lasts as long as one wave's share of the passes, so it is cut
// finer until the waves would meet on a SIMD again (8 waves in one block on one CU
// gained nothing over 4).  One wave per unit through all passes (2-body: term by
// term) took 207 us for 101 trimers, 238 for 13,641, 566 for 139,535; 93 for 91 dimers,
// 93 for 4612, 105 for 42,250.  Here, with the join (4-5 us) where there is one: 101
// trimers 38-48 (beside the other terms, or alone), 776 40, 9204 84-91, 134,272 633 in a
// grid of one wave a SIMD; 91 dimers 37, 2016 42, 42,250 81.
// ---------------------------------------------------------------------------
#if PIP_BODY == 2
constexpr int kPoints = 10, kVars = 31, kMols = 2, kPassAll = pip2b_npass;
typedef Var2 Var;
typedef int2 Unit;
__host__ __device__ constexpr Var var_of(int n) { return var2(n); }
#else
constexpr int kPoints = 9, kVars = 36, kMols = 3, kPassAll = pip3b_npass;
typedef Var3 Var;
typedef int Unit;
__host__ __device__ constexpr Var var_of(int n) { return var3(n); }
#endif
// the variables, and for every point the variables it enters with the point at the other end
struct Partner {
    int n, other, coul, pad;
    double k;
};
struct PipTables {
    Var var[kVars];
    Partner with[kPoints][kPoints];
    int count[kPoints];
};
constexpr PipTables make_tables() {
    PipTables t{};
    for (int n = 0; n < kVars; ++n) {
        t.var[n] = var_of(n);
        const int a = t.var[n].a, b = t.var[n].b;
        t.with[a][t.count[a]++] = Partner{n, b, t.var[n].coul, 0, t.var[n].k};
        t.with[b][t.count[b]++] = Partner{n, a, t.var[n].coul, 0, t.var[n].k};
    }
    return t;
}
__constant__ PipTables pip_tables = make_tables();

__device__ __forceinline__ double rsqrt_pip(double v) { return rsqrt(v); }
__device__ __forceinline__ float rsqrt_pip(float v) { return 1.0f / sqrtf(v); }

constexpr int P = 4;  // waves of a block
constexpr int kXYZ = 3 * kPoints;
static_assert(kXYZ + 1 <= kPipRows, "the rows of a share: the points' gradient, the energy");

// Blocks a unit's passes are spread over: as many as still find a CU each, since
// only then does every wave have a SIMD to itself, and a short list takes as long
// as one wave's passes.
__host__ __device__ constexpr int unit_parts(long long units, int slots) {
    for (int q : {6, 3, 2})
        if (kPassAll % (P * q) == 0 && units * q <= slots) return q;
    return 1;
}
constexpr int kMostParts = unit_parts(1, 1 << 20);

__global__ void __launch_bounds__(64 * P) __attribute__((amdgpu_waves_per_eu(2)))
k_pip_split(PipScratch scratch, long long nu, const long long* __restrict__ ndev, const Unit* __restrict__ list,
            const int* __restrict__ idx, const double* __restrict__ pos, int periodic, d3 box,
            u64* __restrict__ force, u64* __restrict__ energy, double* __restrict__ eunit) {
    constexpr int N = kVars;
    static_assert(P > kMols, "a wave for each part of step 5");
    __shared__ double rs[kPoints * 3][64];          // points relative to the first oxygen, Angstrom
    __shared__ real xs[N][64], gs[N][64], es[P][64];  // variables, gradient, energies of the waves' passes
    __shared__ real fs[kPoints * 3][64];            // minus the gradient on the points (before switch and units)
    __shared__ int ons[64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    PIP_CONST_PTR(PipTables) tab = (PIP_CONST_PTR(PipTables))&pip_tables;
    if (ndev) nu = min(nu, *ndev);
    int parts = unit_parts((nu + 63) / 64, scratch.slots);
    PIP_OPAQUE_PTR(parts);  // one copy of the code for every value
    const int part = blockIdx.x % parts, npass = kPassAll / (P * parts), k0 = (part * P + wave) * npass;
    for (long long t0 = (long long)(blockIdx.x / parts) * 64; t0 < nu; t0 += (long long)gridDim.x * 64) {
        const long long t = t0 + lane;
        if (wave == 0) {
            bool on = false;
            if (t < nu) {
                vd R[kPoints];
                on = unit_geometry(t, list, idx, pos, periodic, box, R);
                if (on) {
#pragma unroll
                    for (int q = 0; q < kPoints; ++q) {
                        rs[3 * q][lane] = R[q].x;
                        rs[3 * q + 1][lane] = R[q].y;
                        rs[3 * q + 2][lane] = R[q].z;
                    }
                }
            }
            if (!on) {  // any points apart: the results are not used
#pragma unroll
                for (int q = 0; q < kPoints; ++q) rs[3 * q][lane] = rs[3 * q + 1][lane] = rs[3 * q + 2][lane] = (double)q;
            }
            ons[lane] = on;
        }
        __syncthreads();
        const bool on = ons[lane];
#pragma unroll 3
        for (int n = wave; n < N; n += P) {
            const int a = 3 * tab->var[n].a, b = 3 * tab->var[n].b;
            const vr d((real)(rs[a][lane] - rs[b][lane]), (real)(rs[a + 1][lane] - rs[b + 1][lane]),
                       (real)(rs[a + 2][lane] - rs[b + 2][lane]));
            const real r = sqrt(d.dot(d));
            const real e = exp_t<real>((real)tab->var[n].k * ((real)tab->var[n].r0 - r));
            xs[n][lane] = tab->var[n].coul ? e / r : e;
        }
        __syncthreads();
        {
            PIP_CONST_PTR(int) from = label_table() + N * k0;
            real x[N], g[N];
#pragma unroll
            for (int m = 0; m < N; ++m) x[m] = xs[from[m]][lane];
            real e = 0;
#if PIP_BODY == 3
            if (k0 == 0) {  // R: this wave starts from the original labelling
                e = pip3b_rest<real>(x, g);
            } else
#endif
            {
#pragma unroll
                for (int m = 0; m < N; ++m) g[m] = 0;
            }
            e += passes<real>(x, g, k0, k0 + npass);
            es[wave][lane] = e;
            PIP_CONST_PTR(int) to = label_table() + N * (k0 + npass);
            PIP_OPAQUE_PTR(to);  // read after the passes
            for (int w = 0; w < P; ++w) {
                if (w == wave) {
#pragma unroll
                    for (int m = 0; m < N; ++m) {
                        const int i = to[m];
                        gs[i][lane] = w == 0 ? g[m] : gs[i][lane] + g[m];
                    }
                }
                __syncthreads();
            }
        }
        for (int p = wave; p < kPoints; p += P) {
            vr F(0, 0, 0);
            const double px = rs[3 * p][lane], py = rs[3 * p + 1][lane], pz = rs[3 * p + 2][lane];
#pragma unroll 2
            for (int c = 0; c < tab->count[p]; ++c) {
                const int n = tab->with[p][c].n, o = 3 * tab->with[p][c].other;
                const vr d((real)(px - rs[o][lane]), (real)(py - rs[o + 1][lane]), (real)(pz - rs[o + 2][lane]));
                const real ri = rsqrt_pip(d.dot(d)), k = (real)tab->with[p][c].k;
                const real gg = -(tab->with[p][c].coul ? k + ri : k) * xs[n][lane] * ri;
                F += d * (gg * gs[n][lane]);
            }
            fs[3 * p][lane] = F.x;
            fs[3 * p + 1][lane] = F.y;
            fs[3 * p + 2][lane] = F.z;
        }
        __syncthreads();
        if (parts > 1) {  // the block's only unit: the grid has a block for every part of every unit
            int ln = lane;  // opaque copies: no address of this part is kept in registers through the passes
            asm volatile("" : "+v"(ln));
            real* share = static_cast<real*>(scratch.shares) + (size_t)blockIdx.x * (kPipRows * 64);
            double* points = scratch.points + (size_t)(blockIdx.x / parts) * (kPipRows * 64);
            PIP_OPAQUE_PTR(share);
            PIP_OPAQUE_PTR(points);
#pragma nounroll
            for (int r = wave; r < kXYZ; r += P) {
                share[r * 64 + ln] = fs[r][ln];
                if (part == 0) points[r * 64 + ln] = rs[r][ln];
            }
            if (wave == 0) {
                share[kXYZ * 64 + ln] = es[0][ln] + es[1][ln] + es[2][ln] + es[3][ln];
                if (part == 0) points[kXYZ * 64 + ln] = on ? 1.0 : 0.0;
            }
            return;
        }
        if (wave <= kMols) {
            real E = es[0][lane];
#pragma unroll
            for (int w = 1; w < P; ++w) E += es[w][lane];
            unit_end(wave, on, t, t < nu, (double)E, rs, fs, list, idx, force, energy, eunit, lane);
        }
        __syncthreads();  // the LDS arrays are written again
    }
}

// step 5 of the units whose passes were spread over several blocks, a block per unit
__global__ void __launch_bounds__(64 * P)
k_pip_join(PipScratch scratch, long long nu, const long long* __restrict__ ndev, const Unit* __restrict__ list,
           const int* __restrict__ idx, u64* __restrict__ force, u64* __restrict__ energy,
           double* __restrict__ eunit) {
    __shared__ double rs[kXYZ][64], ons[64];
    __shared__ real fs[kXYZ][64], es[64];
    if (ndev) nu = min(nu, *ndev);
    const int unit = blockIdx.x, parts = unit_parts((nu + 63) / 64, scratch.slots);
    const long long t = (long long)unit * 64 + (threadIdx.x & 63);
    if (parts == 1 || (long long)unit * 64 >= nu) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int R = (kXYZ + 1 + P - 1) / P;  // rows of a wave
    const real* shares = static_cast<const real*>(scratch.shares) + (size_t)unit * parts * (kPipRows * 64) + lane;
    const double* points = scratch.points + (size_t)unit * (kPipRows * 64) + lane;
    real v[kMostParts][R];
    double x[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {  // every load in flight at once (past the last part or row: that one again)
        const int r = min(wave + P * i, kXYZ);
        x[i] = points[r * 64];
#pragma unroll
        for (int p = 0; p < kMostParts; ++p) v[p][i] = shares[(min(p, parts - 1) * kPipRows + r) * 64];
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int r = wave + P * i;
        real sum = v[0][i];
#pragma unroll
        for (int p = 1; p < kMostParts; ++p)
            if (p < parts) sum += v[p][i];
        if (r <= kXYZ) {
            (r < kXYZ ? rs[r] : ons)[lane] = x[i];
            (r < kXYZ ? fs[r] : es)[lane] = sum;
        }
    }
    __syncthreads();
    if (wave <= kMols)
        unit_end(wave, ons[lane] != 0.0, t, t < nu, (double)es[lane], rs, fs, list, idx, force, energy, eunit, lane);
}
#endif

}  // namespace
}  // namespace mbpol

#define PIP_CAT2(a, b) a##b
#define PIP_CAT(a, b) PIP_CAT2(a, b)
namespace mbpol {
// one block of `waves` waves per 64 units, at most max_waves waves (when positive)
static inline int grid(long long n, int max_waves, int waves) {
    const long long b = (n + 63) / 64, cap = std::max(1, max_waves / waves);
    return (int)(max_waves > 0 && b > cap ? cap : b);
}
#if PIP_ORBIT
// One block per 64 units at most max_waves / P of them, but a block for every part of every unit of any list
// that unit_parts would split (units * parts <= slots of them); and those lists' second kernel.
static inline int split_grid(long long n, int max_waves, int slots) {
    return std::max(grid(n, max_waves, P), (int)std::min<long long>((n + 63) / 64 * kMostParts, slots));
}
static inline int join_grid(long long n, int slots) { return (int)std::min<long long>((n + 63) / 64, slots / 2); }
#define PIP_SCRATCH const PipScratch &scratch,
#define PIP_LAUNCH(kern, n, s, np, ndev, list, idx, ...)                                                             \
    do {                                                                                                             \
        const int blocks = split_grid(n, max_blocks, scratch.slots), joins = join_grid(n, scratch.slots);            \
        const hipEvent_t split_stop = scratch.join ? nullptr : ev.stop; /* a timed span ends with the last kernel */ \
        if (ev.start)                                                                                                \
            hipExtLaunchKernelGGL(k_pip_split, blocks, 64 * P, 0, s, ev.start, split_stop, 0, scratch, np, ndev,     \
                                  list, idx, __VA_ARGS__);                                                           \
        else                                                                                                         \
            hipLaunchKernelGGL(k_pip_split, blocks, 64 * P, 0, s, scratch, np, ndev, list, idx, __VA_ARGS__);        \
        if (!scratch.join) break;                                                                                    \
        if (ev.start)                                                                                                \
            hipExtLaunchKernelGGL(k_pip_join, joins, 64 * P, 0, s, nullptr, ev.stop, 0, scratch, np, ndev, list,     \
                                  idx, force, energy, eunit);                                                        \
        else                                                                                                         \
            hipLaunchKernelGGL(k_pip_join, joins, 64 * P, 0, s, scratch, np, ndev, list, idx, force, energy, eunit); \
    } while (0)
#else
#define PIP_SCRATCH
#define PIP_LAUNCH(kern, n, s, ...) MBPOL_LAUNCH(ev, kern, grid(n, max_blocks, 1), 64, 0, s, __VA_ARGS__)
#endif
#if PIP_BODY == 2
void PIP_CAT(launch_twobody_, PIP_SUFFIX)(hipStream_t s, long long npairs, const long long* ndev, const int2* pairs,
                                          const int* idx, const double* pos, int periodic, d3 box, u64* force,
                                          u64* energy, PIP_SCRATCH const KEvents& ev, double* eunit, int max_blocks) {
#if !PIP_ORBIT
    box = d3{box.x * 10., box.y * 10., box.z * 10.};
#endif
    if (npairs > 0)
        PIP_LAUNCH(k_twobody, npairs, s, npairs, ndev, pairs, idx, pos, periodic, box,
                     force, energy, eunit);
}
#else
void PIP_CAT(launch_threebody_, PIP_SUFFIX)(hipStream_t s, long long ntrip, const long long* ndev, const int* trip,
                                            const int* idx, const double* pos, int periodic, d3 box, u64* force,
                                            u64* energy, PIP_SCRATCH const KEvents& ev, double* eunit, int max_blocks) {
    if (ntrip > 0)
        PIP_LAUNCH(k_threebody, ntrip, s, ntrip, ndev, trip, idx, pos, periodic, box,
                     force, energy, eunit);
}
#endif
}  // namespace mbpol
