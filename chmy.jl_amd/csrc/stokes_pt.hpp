// Shared by the fused PT kernels (stokes_fused.hip, stokes_multi2d.hip): the
// arithmetic forms of the iteration, addressing, lane shifts and the 2D
// argument block.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace chmy {

constexpr int kFX = 64;
enum { LC = 0, LVX = 1, LVY = 2, LVZ = 3, LXY = 4, LXZ = 5, LYZ = 6, NLOC = 7 };

// Scalars shared by both arithmetic forms.
template <class T>
struct Kc {
    T Gs, dts, Gdt, dPr, dr, nu, eta_s, eve_s;   // reference inputs
    T iGdt, omdr, third, a_s, b_s, cv_s;         // fast-form constants (host computed)
};

struct LocStride {
    uint32_t sy, sz;     // element strides
    uint32_t o0;         // element offset of logical (0, 0, 0)
};

#ifndef CHMY_FUSED_NT_STORE
#define CHMY_FUSED_NT_STORE 0
#endif

template <class T>
__device__ __forceinline__ T ldo(const T* p, uint32_t boff) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + boff);
}
// Loads of the sweep's read-only forcing (tau_old, f_V, f_P): in the sweep
// precision, or (BF, FP32 sweeps only) from bf16 storage at half the byte
// offset of the FP32 layout.
template <class T, bool BF>
__device__ __forceinline__ T ldf(const T* p, uint32_t boff) {
    if constexpr (BF) {
        static_assert(sizeof(T) == 4, "bf16 forcing goes with FP32 sweeps");
        return T(bf16_to_f32(*reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(p) + (boff >> 1))));
    } else {
        return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + boff);
    }
}

template <class T>
__device__ __forceinline__ void sto(T* p, uint32_t boff, T v) {
#if CHMY_FUSED_NT_STORE
    // streaming store: the advanced state is not re-read in this launch
    __builtin_nontemporal_store(v, reinterpret_cast<T*>(reinterpret_cast<char*>(p) + boff));
#else
    *reinterpret_cast<T*>(reinterpret_cast<char*>(p) + boff) = v;
#endif
}

// EXACT: the reference's expressions (stokes_3d_inc_ve_T.jl:23-57), bitwise.
// FAST: the same update with eta_ve*(1/(G dt) + 1/eta) = 1 used to cancel
// tau/eta: tau_new = tau(1 - dtau_r) + eta_ve dtau_r (tau_old/(G dt) + 2 eps'),
// eta_ve = eta/(1 + eta/(G dt)), Pr_new = Pr - divV eta_ve dtau_Pr and
// V_new = V + r nudtau (1/eta_V + 1/(G dt)): 7 divisions per point instead
// of 31, results within a few ulp per iteration of the exact form.
template <class T, bool EXACT>
struct Arith;

template <class T>
struct Arith<T, true> {
    struct Loc { T eta, eve; };
    __device__ static Loc field(T eta, const Kc<T>& k) { return Loc{eta, visc_ve(eta, k.Gs, k.dts)}; }
    __device__ static Loc scalar(const Kc<T>& k) { return Loc{k.eta_s, k.eve_s}; }
    __device__ static T diag(T t, T to, T e, T dV, Loc L, const Kc<T>& k) {
        T r = ((-(t - to)) / k.Gdt - t / L.eta) + T(2) * (e - dV / T(3));
        return t + (r * L.eve) * k.dr;
    }
    __device__ static T off(T t, T to, T e, Loc L, const Kc<T>& k) {
        T r = ((-(t - to)) / k.Gdt - t / L.eta) + T(2) * e;
        return t + (r * L.eve) * k.dr;
    }
    __device__ static T pr(T P, T dv, Loc L, const Kc<T>& k) { return P - (dv * L.eve) * k.dPr; }
    __device__ static T vcoef_field(T em, const Kc<T>& k) { return visc_ve(em, k.Gs, k.dts); }
    __device__ static T vcoef_scalar(const Kc<T>& k) { return k.eve_s; }
    __device__ static T vel(T v, T r, T c, const Kc<T>& k) { return v + (r * k.nu) / c; }
};

// Divisions of the fast form: IEEE in FP64; in FP32 (the defect-correction
// sweeps) a times the hardware reciprocal of b (v_rcp_f32, 1 ulp), for its 7
// divisions per point
__device__ __forceinline__ double fast_div(double a, double b) { return a / b; }
__device__ __forceinline__ float fast_div(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

template <class T>
struct Arith<T, false> {
    struct Loc { T a, b; };   // a = eta_ve dtau_r, b = eta_ve dtau_Pr
    __device__ static Loc field(T eta, const Kc<T>& k) {
        const T eve = fast_div(eta, fma(eta, k.iGdt, T(1)));
        return Loc{eve * k.dr, eve * k.dPr};
    }
    __device__ static Loc scalar(const Kc<T>& k) { return Loc{k.a_s, k.b_s}; }
    __device__ static T diag(T t, T to, T e, T dV, Loc L, const Kc<T>& k) {
        return fma(t, k.omdr, L.a * fma(to, k.iGdt, T(2) * fma(-dV, k.third, e)));
    }
    __device__ static T off(T t, T to, T e, Loc L, const Kc<T>& k) {
        return fma(t, k.omdr, L.a * fma(to, k.iGdt, T(2) * e));
    }
    __device__ static T pr(T P, T dv, Loc L, const Kc<T>& k) { return fma(-dv, L.b, P); }
    __device__ static T vcoef_field(T em, const Kc<T>& k) { return k.nu * (fast_div(T(1), em) + k.iGdt); }
    __device__ static T vcoef_scalar(const Kc<T>& k) { return k.cv_s; }
    __device__ static T vel(T v, T r, T c, const Kc<T>& k) { return fma(r, c, v); }
};

template <class T>
__device__ __forceinline__ T lerp4(T a0, T a1, T b0, T b1) {
    // knots (lo,lo),(hi,lo),(lo,hi),(hi,hi); first dim innermost (interpolation.jl:37-56)
    T A = fma(T(0.5), a1 - a0, a0);
    T B = fma(T(0.5), b1 - b0, b0);
    return fma(T(0.5), B - A, A);
}

enum { L2C = 0, L2X = 1, L2Y = 2, L2XY = 3, NLOC2 = 4 };

template <class T>
struct Fused2 {
    const T *Vx, *Vy, *Pr, *txx, *tyy, *txy;
    T *oVx, *oVy, *oPr, *otxx, *otyy, *otxy;
    const T *Oxx, *Oyy, *Oxy;
    const T *eta, *eml, *rg;
    const T *fVx, *fVy, *fP;
    T *dV, *rVx, *rVy;
    LocStride L[NLOC2];
    int32_t n[2];
    int32_t ntx, nchunks, ychunk;
    int32_t has_rg, write_res, has_f;
    T ix, iy;
    Kc<T> k;
};

// Raw load of a forcing value (kept as bf16 bits until use, so the load can
// stay in flight across a row of the march) and its conversion.
template <class T, bool BF>
using Fraw = typename std::conditional<BF, uint16_t, T>::type;
template <class T, bool BF>
__device__ __forceinline__ Fraw<T, BF> ldr(const T* p, uint32_t boff) {
    if constexpr (BF) return *reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(p) + (boff >> 1));
    else return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + boff);
}
template <class T, bool BF>
__device__ __forceinline__ T cvf(Fraw<T, BF> v) {
    if constexpr (BF) return T(bf16_to_f32(v));
    else return v;
}

// x neighbours inside a row's wave by DPP whole-wave shifts: xm1 gives lane l
// the value of lane l-1, xp1 that of lane l+1 (lanes 0 / 63 receive 0, and
// reach no output).
__device__ __forceinline__ int dpp_shr1(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, false); }
__device__ __forceinline__ int dpp_shl1(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, false); }
__device__ __forceinline__ double xm1(double v) {
    return __hiloint2double(dpp_shr1(__double2hiint(v)), dpp_shr1(__double2loint(v)));
}
__device__ __forceinline__ double xp1(double v) {
    return __hiloint2double(dpp_shl1(__double2hiint(v)), dpp_shl1(__double2loint(v)));
}
__device__ __forceinline__ float xm1(float v) { return __int_as_float(dpp_shr1(__float_as_int(v))); }
__device__ __forceinline__ float xp1(float v) { return __int_as_float(dpp_shl1(__float_as_int(v))); }

// The V batch a 2D free-slip solve applies after every iteration
// (stokes_2d_inc_ve_T.jl's bc of update_velocity!): Vx Dirichlet on its x
// nodes 1 / n+1 and Neumann in y, Vy Neumann in x and Dirichlet on its y
// nodes 1 / n+1, scalar values [side 1, side 2]; h the spacings.
struct FreeSlip2 {
    double ax[2], qy[2], by[2], qx[2];
    double hx, hy;
    int32_t iters;   // iterations of the pass
    int32_t pre;     // the batch is still to be applied to the V the pass reads
};

// Iterations of the next 2D pass of a run (stokes_multi2d.hip); 0: none, the
// run goes on in passes of two and single iterations.
int multi2d_next(const chmy_grid_t* g, bool f32_exact, bool forced, int run);

// fs.iters (as multi2d_next gives them) iterations in one launch; `a` holds everything but the tiling.
template <class T>
void multi2d_launch(Fused2<T> a, const FreeSlip2& fs, bool fv, bool exact, bool bf, bool rg, hipStream_t s);

}  // namespace chmy
