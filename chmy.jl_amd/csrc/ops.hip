// Per-point Launcher kernels: diffusion, update_old!, thermal flux/update and
// the viscosity max-neighbourhood.  Each thread owns one logical index I of the
// box, 256 consecutive points of a plane a block (flat_point).  These are
// bandwidth-bound streaming kernels; the fused Stokes iteration lives in
// stokes_fused.hip.  In FP32 on large boxes the address arithmetic bounds them
// too, so the views carry a unit x stride (a 64-bit product a point and array
// less): us, 64 x 4 blocks -> flat ones -> with unit strides, a step of
// chmy_diffusion_iterate FP32 3000^2 44.2 -> 48.2 -> 43.4, 400^3 728 -> 777 ->
// 710; compute_q FP64 400^3 606 -> 630 -> 597.  159x143x127 FP64: thermal flux
// 36.2 -> 25.8 -> 25.9, update 26.8 -> 19.8 -> 19.3, update_old! (loads before
// stores) 69 -> 62, a step of the loop 44.4 -> 35 -> 33.7.
#include <cstring>

#include "stokes_pt.hpp"

namespace chmy {

struct Ix3 {
    int64_t i, j, k;
};

__device__ __forceinline__ Ix3 box_index(const Box3& b, bool& ok) {
    Ix3 I;
    ok = flat_point(b, I.i, I.j, I.k);
    return I;
}

template <class T>
__device__ __forceinline__ T& g_at(const DF<T>& f, Ix3 I) { return f(I.i, I.j, I.k); }
__device__ __forceinline__ Ix3 sh(Ix3 I, int d, int64_t s) {
    if (d == 0) I.i += s; else if (d == 1) I.j += s; else I.k += s;
    return I;
}
// ------------------------------------------------------------------ diffusion
template <class T>
__global__ void __launch_bounds__(256) diffusion_flux_kernel(Box3 b, DF<T> C, DF<T> q0, DF<T> q1, DF<T> q2,
                                                             int nd, T nchi, T i0, T i1, T i2) {
    bool ok;
    Ix3 I = box_index(b, ok);
    if (!ok) return;
    // q.x[I] = -χ * ∂x(C)[I] (diffusion_2d.jl:11-12): Center C -> (C[I] - C[I-e]) iΔ
    g_at(q0, I) = nchi * ((g_at(C, I) - g_at(C, sh(I, 0, -1))) * i0);
    if (nd > 1) g_at(q1, I) = nchi * ((g_at(C, I) - g_at(C, sh(I, 1, -1))) * i1);
    if (nd > 2) g_at(q2, I) = nchi * ((g_at(C, I) - g_at(C, sh(I, 2, -1))) * i2);
}

template <class T>
__global__ void __launch_bounds__(256) diffusion_update_kernel(Box3 b, DF<T> C, DF<T> q0, DF<T> q1, DF<T> q2,
                                                               int nd, T dt, T i0, T i1, T i2) {
    bool ok;
    Ix3 I = box_index(b, ok);
    if (!ok) return;
    // C[I] -= Δt * divg(q)[I] (diffusion_2d.jl:18); Vertex q_D -> (q[I+e] - q[I]) iΔ
    T dv = (g_at(q0, sh(I, 0, 1)) - g_at(q0, I)) * i0;
    if (nd > 1) dv = dv + (g_at(q1, sh(I, 1, 1)) - g_at(q1, I)) * i1;
    if (nd > 2) dv = dv + (g_at(q2, sh(I, 2, 1)) - g_at(q2, I)) * i2;
    g_at(C, I) = g_at(C, I) - dt * dv;
}

// compute_q! and update_C! in one launch (build extension): q at I from C at
// I, I-e (stored, as compute_q! stores it), q at I+e recomputed the same way
// when I+e is inside the box, else read from q's storage (what update_C! would
// read there); C_out[I] = C[I] - Δt divg(q)[I].  C and C_out are distinct
// buffers, so no thread reads a C value another has advanced.
// The step's new C at I (box b): q_D at I (stored when store_q, as
// compute_q! stores it), q_D at I+e recomputed when I+e is in the box, else
// read from q's storage; C[I] - Δt divg(q)[I].
template <class T>
__device__ __forceinline__ T diffusion_value(const Box3& b, const DF<T>& C, const DF<T>& q0, const DF<T>& q1,
                                             const DF<T>& q2, int nd, T nchi, T dt, const T* isp, Ix3 I,
                                             bool store_q) {
    const T c = g_at(C, I);
    const int64_t hi[3] = {b.lo[0] + b.len[0], b.lo[1] + b.len[1], b.lo[2] + b.len[2]};
    const int64_t at[3] = {I.i, I.j, I.k};
    T dv = T(0);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= nd) break;
        const DF<T>& qd = d == 0 ? q0 : (d == 1 ? q1 : q2);
        const T ql = nchi * ((c - g_at(C, sh(I, d, -1))) * isp[d]);
        if (store_q) g_at(qd, I) = ql;
        const Ix3 J = sh(I, d, 1);
        const T qr = at[d] + 1 < hi[d] ? nchi * ((g_at(C, J) - c) * isp[d]) : g_at(qd, J);
        const T t = (qr - ql) * isp[d];
        dv = d == 0 ? t : dv + t;
    }
    return c - dt * dv;
}

template <class T>
__global__ void __launch_bounds__(256) diffusion_step_kernel(Box3 b, DF<T> C, DF<T> Co, DF<T> q0, DF<T> q1,
                                                             DF<T> q2, int nd, T nchi, T dt, T i0, T i1, T i2) {
    bool ok;
    Ix3 I = box_index(b, ok);
    if (!ok) return;
    const T isp[3] = {i0, i1, i2};
    g_at(Co, I) = diffusion_value(b, C, q0, q1, q2, nd, nchi, dt, isp, I, true);
}

// One scalar rule per (dim, side) of a Center field's batch.
struct SideRules {
    int32_t kind[3][2];   // CHMY_DIRICHLET / CHMY_NEUMANN
    double val[3][2];
    double h[3];          // spacings (the Neumann step)
};

// The step and the C batch in one launch, when every (dim, side) carries one
// scalar rule: one thread per point of [0, n+2]^N, which holds everything the
// step (box [0, n+1]^N) and the batch (ghost planes 0 and n+1, tangential
// 0..n+2) write.  A point that no dim writes keeps the step's value (or is
// left alone outside the box).  A point that some dims write takes the
// batch's final value, the chain bc_set_kernel evaluates: its inner point Q
// (every ghost coordinate moved inward) as the step leaves it (recomputed
// here when Q is in the box, else read as stored: no thread writes it), then
// each writing dim's rule from the highest to the lowest, the batch's own fma
// steps.  q is stored on the box as the step stores it.
template <class T>
__global__ void __launch_bounds__(256) diffusion_step_bc_kernel(Box3 box, Box3 reg, DF<T> C, DF<T> Co, DF<T> q0,
                                                                DF<T> q1, DF<T> q2, int nd, T nchi, T dt, T i0,
                                                                T i1, T i2, SideRules r) {
    bool ok;
    const Ix3 P = box_index(reg, ok);
    if (!ok) return;
    const T isp[3] = {i0, i1, i2};
    const int64_t p[3] = {P.i, P.j, P.k};
    int64_t m[3], qc[3];
    int gs[3];
    bool in_box = true, ghost = false;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        m[d] = box.len[d] - 2;   // cells: the box is [0, n+1]
        qc[d] = p[d];
        gs[d] = -1;
        if (d >= nd) continue;
        in_box = in_box && p[d] <= m[d] + 1;
        if (p[d] == 0 || p[d] == m[d] + 1) {
            gs[d] = p[d] == 0 ? 0 : 1;
            qc[d] = p[d] == 0 ? 1 : m[d];
            ghost = true;
        }
    }
    T v = T(0);
    if (in_box) v = diffusion_value(box, C, q0, q1, q2, nd, nchi, dt, isp, P, true);
    if (!ghost) {
        if (in_box) g_at(Co, P) = v;
        return;
    }
    const Ix3 Q{qc[0], qc[1], qc[2]};
    bool q_in = true;
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (d < nd) q_in = q_in && qc[d] <= m[d] + 1;
    T w = q_in ? diffusion_value(box, C, q0, q1, q2, nd, nchi, dt, isp, Q, false) : g_at(Co, Q);
#pragma unroll
    for (int d = 2; d >= 0; --d) {
        if (d >= nd || gs[d] < 0) continue;
        const T val = T(r.val[d][gs[d]]);
        if (r.kind[d][gs[d]] == CHMY_DIRICHLET) w = fma(T(2), val - w, w);
        else w = fma(T(r.h[d]), gs[d] == 0 ? -val : val, w);
    }
    g_at(Co, P) = w;
}

// Up to KS steps of the loop in one launch (build extension), C and its face
// ghosts only: a block loads its TX x TY (x TZ) cells with a ring of KS and
// advances them on chip, the valid region shrinking by one ring a step; the
// ring is computed again by the neighbouring blocks.  A thread holds PT
// consecutive points of the last dim in registers and finds its neighbours
// along the other dims in LDS (two buffers, one barrier a step).  A cell's
// value is the expression of diffusion_value on the same operands; the
// neighbour beyond a boundary is the batch's own fma step of the cell (the
// stored ghost in the first step), so every stored value has the bits of as
// many launches of the step.  q is not stored, so the caller runs the last step
// by itself; in 3D the last two, since the edge and corner ghosts (which no
// cell reads, but q on the ghosts does) are left alone there.
//
// Why: a step of 256^2 cells is one 5 us launch for 0.5 MB of data, most of it
// the wait for the launch before it.  Measured, us per step of a 100-step call,
// one launch each -> now: 2D FP64 64^2 4.7 -> 0.88, 256^2 5.1 -> 0.87, 500x480
// 5.5 -> 1.4, 1024^2 11.4 -> 3.5 (FP32 10.0 -> 2.8); 3D 20^3 5.6 -> 3.5, 64^3
// 12.6 -> 3.7, 160^3 58.6 -> 25.7 (FP32 45 -> 15).  Bound by the chain of LDS
// reads and barriers (0.1 us a step) and the launches on small grids, by
// vector issue and LDS on large ones.
template <class T>
struct DiffTile {
    DF<T> C, Co;
    int32_t n[3], nb[3];
    int32_t steps;   // 1..KS
    T nchi, dt, isp[3];
    SideRules r;
};

template <class T>
__device__ __forceinline__ T ghost_of(const SideRules& r, int d, int side, T w) {
    const T val = T(r.val[d][side]);
    if (r.kind[d][side] == CHMY_DIRICHLET) return fma(T(2), val - w, w);
    return fma(T(r.h[d]), side == 0 ? -val : val, w);
}

template <class T, int ND, int TX, int TY, int TZ, int KS, int PT>
struct DiffShape {
    static constexpr int RX = TX + 2 * KS, RY = TY + 2 * KS, RZ = ND == 3 ? TZ + 2 * KS : 1;
    static constexpr int M = ND - 1, RM = ND == 3 ? RZ : RY, SM = ND == 3 ? RX * RY : RX;   // the last dim
    static constexpr int COLS = ND == 3 ? RX * RY : RX, NT = COLS * (RM / PT);
    static_assert(RM % PT == 0 && NT <= 1024, "strips tile the last dim");
};

template <class T, int ND, int TX, int TY, int TZ, int KS, int PT, int NT = DiffShape<T, ND, TX, TY, TZ, KS, PT>::NT>
__global__ void __launch_bounds__(NT) diffusion_tile_kernel(const DiffTile<T> p) {
    using Sh = DiffShape<T, ND, TX, TY, TZ, KS, PT>;
    constexpr int RX = Sh::RX, RY = Sh::RY, M = Sh::M, SM = Sh::SM;
    __shared__ T buf[2][Sh::COLS * Sh::RM];
    const int t = xcd_remap(line_id(), line_ids());
    const int row = t / p.nb[0], bx = t - row * p.nb[0], by = ND == 3 ? row % p.nb[1] : row, bz = ND == 3 ? row / p.nb[1] : 0;
    if (ND == 3 ? bz >= p.nb[2] : by >= p.nb[1]) return;   // no tile (whole block: no barrier passed)
    const int col = threadIdx.x % Sh::COLS, strip = threadIdx.x / Sh::COLS;
    const int a[3] = {col % RX, ND == 3 ? col / RX : strip * PT, strip * PT};
    const int org[3] = {1 + bx * TX - KS, 1 + by * TY - KS, ND == 3 ? 1 + bz * TZ - KS : 0};
    const int len[3] = {RX, RY, Sh::RZ};
    int ring0 = KS;
    bool cell0 = true, stored0 = true, edge = false, g0[2][2] = {};
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        edge = edge || org[d] < 1 || org[d] + len[d] > p.n[d] + 1;   // the region holds a boundary (block-uniform)
        if (d == M) continue;
        const int c = org[d] + a[d];
        stored0 = stored0 && c >= 0 && c <= p.n[d] + 1;
        cell0 = cell0 && c >= 1 && c <= p.n[d];
        ring0 = min(ring0, min(a[d], len[d] - 1 - a[d]));
        g0[d][0] = c == 1;
        g0[d][1] = c == p.n[d];
    }
    const int l0 = ND == 3 ? col + a[2] * SM : col + a[1] * SM;
    const int64_t base = (int64_t)(org[0] + a[0]) + (int64_t)(org[1] + a[1]) * p.C.sy +
                         (ND == 3 ? (int64_t)(org[2] + a[2]) * p.C.sz : 0);
    const int64_t sm = ND == 3 ? p.C.sz : p.C.sy;
    T c[PT];
    int ring[PT];   // steps the point is advanced: 0 where it is no cell of the region
#pragma unroll
    for (int q = 0; q < PT; ++q) {
        const int m = a[M] + q, i = org[M] + m;
        const bool in = i >= 1 && i <= p.n[M];
        ring[q] = cell0 && in ? min(ring0, min(m, Sh::RM - 1 - m)) - (KS - p.steps) : 0;
        c[q] = T(0);
        if (stored0 && i >= 0 && i <= p.n[M] + 1) c[q] = p.C.p[base + q * sm];
        buf[0][l0 + q * SM] = c[q];
    }
    __syncthreads();
    auto advance = [&](auto edge_) {
        constexpr bool EDGE = decltype(edge_)::value;
#pragma unroll 1
        for (int s = 1; s <= p.steps; ++s) {
            const T* in = buf[(s - 1) & 1];
            T* out = buf[s & 1];
            const bool by_rule = EDGE && s > 1;
            const T below = strip > 0 ? in[l0 - SM] : T(0), above = strip + 1 < Sh::RM / PT ? in[l0 + PT * SM] : T(0);
            T old = below;
#pragma unroll
            for (int q = 0; q < PT; ++q) {
                const T cq = c[q];
                const T next = q + 1 < PT ? c[q + 1] : above;
                if (ring[q] >= s) {
                    const int l = l0 + q * SM, i = org[M] + a[M] + q;
                    T dv = T(0);
#pragma unroll
                    for (int d = 0; d < ND; ++d) {
                        T lo = d == M ? old : in[l - (d == 0 ? 1 : RX)], hi = d == M ? next : in[l + (d == 0 ? 1 : RX)];
                        if (by_rule) {
                            if (d == M ? i == 1 : g0[d & 1][0]) lo = ghost_of(p.r, d, 0, cq);
                            if (d == M ? i == p.n[M] : g0[d & 1][1]) hi = ghost_of(p.r, d, 1, cq);
                        }
                        const T ql = p.nchi * ((cq - lo) * p.isp[d]);
                        const T qr = p.nchi * ((hi - cq) * p.isp[d]);
                        const T x = (qr - ql) * p.isp[d];
                        dv = d == 0 ? x : dv + x;
                    }
                    c[q] = cq - p.dt * dv;
                    out[l] = c[q];
                }
                old = cq;
            }
            __syncthreads();
        }
    };
    if (edge) advance(std::true_type{});
    else advance(std::false_type{});
#pragma unroll
    for (int q = 0; q < PT; ++q) {
        if (ring[q] < p.steps) continue;   // the tile's own cells
        const int64_t o = base + q * sm;
        p.Co.p[o] = c[q];
        if (!edge) continue;
        const int i = org[M] + a[M] + q;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            const int64_t st = d == 0 ? 1 : d == 1 ? p.C.sy : p.C.sz;
            if (d == M ? i == 1 : g0[d & 1][0]) p.Co.p[o - st] = ghost_of(p.r, d, 0, c[q]);
            if (d == M ? i == p.n[M] : g0[d & 1][1]) p.Co.p[o + st] = ghost_of(p.r, d, 1, c[q]);
        }
        if constexpr (ND == 2) {
            // what else the batch writes: the corners (y's rule, then x's), and its
            // tangential range's last index n + 2, from points that no step changes
            const bool gy[2] = {i == 1, i == p.n[1]};
            const int64_t sy = p.C.sy;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int a_ = k & 1, b_ = k >> 1;
                const int64_t dx = a_ ? 1 : -1, dy = b_ ? sy : -sy;
                if (g0[0][a_] && gy[b_]) p.Co.p[o + dx + dy] = ghost_of(p.r, 0, a_, ghost_of(p.r, 1, b_, c[q]));
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                if (g0[0][k] && gy[1]) p.Co.p[o + 2 * sy + (k ? 1 : -1)] = ghost_of(p.r, 0, k, p.Co.p[o + 2 * sy]);
                if (gy[k] && g0[0][1]) p.Co.p[o + 2 + (k ? sy : -sy)] = ghost_of(p.r, 1, k, p.Co.p[o + 2]);
            }
        }
    }
}

// ------------------------------------------------------------------ update_old!
template <class T>
struct Copy7 {
    DF<T> src[7], dst[7];
    int n;
};

template <class T>
__global__ void __launch_bounds__(256) copy_kernel(Box3 b, Copy7<T> c) {
    bool ok;
    Ix3 I = box_index(b, ok);
    if (!ok) return;
    T v[7];
#pragma unroll
    for (int q = 0; q < 7; ++q)
        if (q < c.n) v[q] = g_at(c.src[q], I);
#pragma unroll
    for (int q = 0; q < 7; ++q)
        if (q < c.n) g_at(c.dst[q], I) = v[q];
}

// ------------------------------------------------------------------ thermal
template <class T>
__global__ void __launch_bounds__(256) thermal_flux_kernel(Box3 b, DF<T> Tf, DF<T> V0, DF<T> V1, DF<T> V2,
                                                           DF<T> q0, DF<T> q1, DF<T> q2, int nd, T nlam, T i0,
                                                           T i1, T i2) {
    bool ok;
    Ix3 I = box_index(b, ok);
    if (!ok) return;
    const T isp[3] = {i0, i1, i2};
    const T tc = g_at(Tf, I);
#pragma unroll
    for (int d = 0; d < 3; ++d) {   // constant indices once unrolled: no stack arrays
        if (d >= nd) break;
        const DF<T>& Vd = d == 0 ? V0 : (d == 1 ? V1 : V2);
        const DF<T>& qd = d == 0 ? q0 : (d == 1 ? q1 : q2);
        // qT_D = ((-λ ∂_D T) + max(V_D,0) left_D T) + min(V_D,0) right_D T
        // (stokes_3d_inc_ve_T.jl:59-71); T Center: left = T[I-e], right = T[I]
        const T tl = g_at(Tf, sh(I, d, -1));
        const T v = g_at(Vd, I);
        g_at(qd, I) = (nlam * ((tc - tl) * isp[d]) + jmax0(v) * tl) + jmin0(v) * tc;
    }
}

// update_thermal_flux! and update_thermal! in one launch (build extension):
// qT at I from T at I, I-e and V at I (stored, as update_thermal_flux! stores
// it), qT at I+e recomputed the same way when I+e is inside the box, else
// read from qT's storage; T_out[I] = T_old[I] - Δt divg(qT)[I].  T and T_out
// are distinct buffers.
template <class T>
__global__ void __launch_bounds__(256) thermal_step_kernel(Box3 b, DF<T> Tf, DF<T> Tout, DF<T> To, DF<T> V0,
                                                           DF<T> V1, DF<T> V2, DF<T> q0, DF<T> q1, DF<T> q2,
                                                           int nd, T nlam, T dt, T i0, T i1, T i2) {
    bool ok;
    Ix3 I = box_index(b, ok);
    if (!ok) return;
    const int64_t hi[3] = {b.lo[0] + b.len[0], b.lo[1] + b.len[1], b.lo[2] + b.len[2]};
    const int64_t at[3] = {I.i, I.j, I.k};
    const T isp[3] = {i0, i1, i2};
    const T tc = g_at(Tf, I);
    T dv = T(0);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= nd) break;
        const DF<T>& Vd = d == 0 ? V0 : (d == 1 ? V1 : V2);
        const DF<T>& qd = d == 0 ? q0 : (d == 1 ? q1 : q2);
        const T tl = g_at(Tf, sh(I, d, -1));
        const T v = g_at(Vd, I);
        const T ql = (nlam * ((tc - tl) * isp[d]) + jmax0(v) * tl) + jmin0(v) * tc;
        g_at(qd, I) = ql;
        const Ix3 J = sh(I, d, 1);
        T qr;
        if (at[d] + 1 < hi[d]) {
            const T tr = g_at(Tf, J), vr = g_at(Vd, J);
            qr = (nlam * ((tr - tc) * isp[d]) + jmax0(vr) * tc) + jmin0(vr) * tr;
        } else {
            qr = g_at(qd, J);
        }
        const T t = (qr - ql) * isp[d];
        dv = d == 0 ? t : dv + t;
    }
    g_at(Tout, I) = g_at(To, I) - dt * dv;
}

// The same step in 3D as a z-march: a block is 64 (x, one wave) x kThY (y)
// points and walks a chunk of at most 16 planes, carrying T at the plane and z's flux
// (qT_z at k+1 computed at plane k is qT_z at plane k+1, the same
// expression on the same operands), so T and V_z stream from HBM once
// instead of being fetched again by the blocks of the neighbouring planes.
// x and y neighbours are loads of the same or adjacent rows, found in L2:
// blocks are remapped so that each XCD walks a contiguous run of tiles.
// Per point: the same expressions, association and stored qT as
// thermal_step_kernel; fields of one staggered location share strides
// (the host checks it).  Lanes outside the box load at clamped indices and
// store nothing.
constexpr int kThY = 4;   // rows per block; with 16-plane chunks the fastest of 1-16 rows x 8-64 planes

template <class T>
__device__ __forceinline__ T th_flux(T tc, T tl, T v, T nlam, T isp) {
    return (nlam * ((tc - tl) * isp) + jmax0(v) * tl) + jmin0(v) * tc;
}

template <class T>
__global__ void __launch_bounds__(64 * kThY) thermal_step3_kernel(Box3 b, DF<T> Tf, DF<T> Tout, DF<T> To, DF<T> V0,
                                                                  DF<T> V1, DF<T> V2, DF<T> q0, DF<T> q1, DF<T> q2,
                                                                  T nlam, T dt, T i0, T i1, T i2, int nbx, int nby,
                                                                  int kchunk) {
    const int lane = threadIdx.x, r = threadIdx.y;
    const int lt = xcd_remap(line_id(), line_ids());
    const int bx = lt % nbx, by = (lt / nbx) % nby, bz = lt / nbx / nby;
    const int64_t hi0 = b.lo[0] + b.len[0], hi1 = b.lo[1] + b.len[1], hi2 = b.lo[2] + b.len[2];
    const int64_t i = b.lo[0] + (int64_t)bx * 64 + lane, j = b.lo[1] + (int64_t)by * kThY + r;
    const int64_t kb = b.lo[2] + (int64_t)bz * kchunk;
    if (kb >= hi2) return;   // a last chunk past the box (whole block: no barrier follows)
    const int64_t ke = kb + kchunk < hi2 ? kb + kchunk : hi2;
    const bool act = i < hi0 && j < hi1;
    const int64_t ic = i < hi0 ? i : hi0 - 1, jc = j < hi1 ? j : hi1 - 1;
    const bool xr = ic + 1 < hi0, yr = jc + 1 < hi1;   // the right face's flux is computed, else read
    const int64_t sC = Tf.sz, sX = V0.sz, sY = V1.sz, sZ = V2.sz;
    const int64_t yC = Tf.sy, yY = V1.sy;
    int64_t oC = ic + jc * yC + kb * sC, oX = ic + jc * V0.sy + kb * sX;
    int64_t oY = ic + jc * yY + kb * sY, oZ = ic + jc * V2.sy + kb * sZ;
    T tc = Tf.p[oC];
    T qlz = th_flux(tc, Tf.p[oC - sC], V2.p[oZ], nlam, i2);
    for (int64_t k = kb; k < ke; ++k) {
        const T tp = Tf.p[oC + sC], vz1 = V2.p[oZ + sZ];
        const T txm = Tf.p[oC - 1], txp = Tf.p[oC + 1];
        const T tym = Tf.p[oC - yC], typ = Tf.p[oC + yC];
        const T vx = V0.p[oX], vx1 = V0.p[oX + 1];
        const T vy = V1.p[oY], vy1 = V1.p[oY + yY];
        const T to = To.p[oC];
        const T qlx = th_flux(tc, txm, vx, nlam, i0);
        const T qly = th_flux(tc, tym, vy, nlam, i1);
        const T qrx = xr ? th_flux(txp, tc, vx1, nlam, i0) : q0.p[oX + 1];
        const T qry = yr ? th_flux(typ, tc, vy1, nlam, i1) : q1.p[oY + yY];
        const T qrz = k + 1 < hi2 ? th_flux(tp, tc, vz1, nlam, i2) : q2.p[oZ + sZ];
        const T dv = ((qrx - qlx) * i0 + (qry - qly) * i1) + (qrz - qlz) * i2;
        if (act) {
            q0.p[oX] = qlx;
            q1.p[oY] = qly;
            q2.p[oZ] = qlz;
            Tout.p[oC] = to - dt * dv;
        }
        tc = tp;
        qlz = qrz;
        oC += sC;
        oX += sX;
        oY += sY;
        oZ += sZ;
    }
}

// Two thermal steps in one launch (3D), with T's Neumann(0) batch between
// them: T -> T1 (V of the first step) -> T_out at cells 1..n (V of the
// second).  T1 is never stored, nor any qT, so the two steps read T, T_old
// and both V once and write T_out once: 9 arrays where two
// thermal_step3_kernel launches move 18.  A block is 64 lanes x BY rows
// marching z: at plane s the first step forms T1(s) from T's planes in
// registers, and the second forms T_out(s - 1) from T1(s - 2 .. s) and T1's
// neighbouring rows in LDS (two planes by parity, one barrier a plane); x
// neighbours come by lane shifts.  T1 is exact on lanes 1..62 and all rows,
// T_out on lanes 2..61 and rows 1..BY-2.  A plane's loads are issued one
// plane ahead, since a block of one wave per row has few loads in flight.
// Same expressions as thermal_step3_kernel, so bitwise the two launches with
// chmy_bc_batchset between them.
// 175x159x143 FP64: 2 x 81 us -> 92 us (286 MB at least: 3.1 TB/s; 8, 10 and
// 12 rows a block and 2 to 4 blocks a CU were within 1%, so it runs at what
// the 12 strided streams give, not at its occupancy).
constexpr int kTh2Y = 16;

template <class T>
struct Thermal2 {
    DF<T> Tf, Tout, To, V1[3], V2[3];
    T nlam, dt, is[3];
    int n[3], nbx, nby, kchunk;
};

template <class T>
__global__ void __launch_bounds__(64 * kTh2Y) thermal_step2_kernel(Thermal2<T> a) {
    __shared__ T s1[2][kTh2Y][64];
    const int lane = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int lt = xcd_remap(line_id(), line_ids());
    const int bx = lt % a.nbx, by = (lt / a.nbx) % a.nby, bz = lt / a.nbx / a.nby;
    const int n0 = a.n[0], n1 = a.n[1], n2 = a.n[2];
    const int i = bx * 60 - 1 + lane, j = by * (kTh2Y - 2) + ty;   // lane 2 and row 1 of the first tile: cell 1
    const int kb = 1 + bz * a.kchunk, ke = min(kb + a.kchunk, n2 + 1);
    if (kb > n2) return;   // no tile (whole block: no barrier passed)
    const uint32_t ic = (uint32_t)min(max(i, 0), n0 + 1);
    const int jc = min(max(j, 0), n1 + 1);
    const bool own = lane >= 2 && lane <= 61 && i <= n0 && ty >= 1 && ty <= kTh2Y - 2 && j <= n1;
    const T nlam = a.nlam, dt = a.dt, ix = a.is[0], iy = a.is[1], iz = a.is[2];
    auto row = [](const DF<T>& f, int j, int k) -> T* { return f.p + ((int64_t)j * f.sy + (int64_t)k * f.sz); };
    const int s0 = max(kb - 1, 1);
    // plane s of T, its rows beside, V1 at the plane (z: the face above), T_old
    T tc = row(a.Tf, jc, s0)[ic];
    T qz = th_flux(tc, row(a.Tf, jc, s0 - 1)[ic], row(a.V1[2], jc, s0)[ic], nlam, iz);
    T tp, tym, typ, vx, vy, vy1, vz1, to;
    T wx, wy, wy1, wz1;   // V2 at the plane (z: the face above)
    T toc = T(0), wxc = T(0), wyc = T(0), wy1c = T(0), wz1c = T(0);   // of plane s - 1
    auto fetch = [&](int s) {
        tp = row(a.Tf, jc, s + 1)[ic];
        tym = row(a.Tf, jc - 1, s)[ic];
        typ = row(a.Tf, jc + 1, s)[ic];
        vx = row(a.V1[0], jc, s)[ic];
        vy = row(a.V1[1], jc, s)[ic];
        vy1 = row(a.V1[1], jc + 1, s)[ic];
        vz1 = row(a.V1[2], jc, s + 1)[ic];
        to = row(a.To, jc, s)[ic];
        wx = row(a.V2[0], jc, s)[ic];
        wy = row(a.V2[1], jc, s)[ic];
        wy1 = row(a.V2[1], jc + 1, s)[ic];
        wz1 = row(a.V2[2], jc, s + 1)[ic];
    };
    fetch(s0);
    T t1m = T(0), t1c = T(0), q2z = T(0);
    for (int s = s0; s <= ke; ++s) {
        T t1;
        if (s <= n2) {   // the first step at plane s
            const T qx = th_flux(tc, xm1(tc), vx, nlam, ix);
            const T qxr = xp1(qx);
            const T qy = th_flux(tc, tym, vy, nlam, iy), qyr = th_flux(typ, tc, vy1, nlam, iy);
            const T qzr = th_flux(tp, tc, vz1, nlam, iz);
            const T dv = ((qxr - qx) * ix + (qyr - qy) * iy) + (qzr - qz) * iz;
            t1 = to - dt * dv;
            tc = tp;
            qz = qzr;
            // x ghosts: the adjacent cell (fma(h, -0, f) and fma(h, 0, f) of the batch)
            const T up = xp1(t1), dn = xm1(t1) + T(0);
            t1 = i <= 0 ? up : i == n0 + 1 ? dn : t1;
        } else {
            t1 = t1c + T(0);   // z's upper ghost
        }
        const T to_s = to, wx_s = wx, wy_s = wy, wy1_s = wy1, wz1_s = wz1;
        if (s + 1 <= min(ke, n2)) fetch(s + 1);
        s1[s & 1][ty][lane] = t1;
        const int r = s - 1;
        if (r >= kb) {   // the second step at plane s - 1
            const int b = r & 1;
            const T lo = s1[b][ty > 0 ? ty - 1 : ty][lane], hi = s1[b][ty < kTh2Y - 1 ? ty + 1 : ty][lane];
            const T tm = j == 1 ? t1c : lo, tq = j == n1 ? t1c + T(0) : hi;
            if (r == kb) q2z = th_flux(t1c, r == 1 ? t1c : t1m, row(a.V2[2], jc, r)[ic], nlam, iz);
            const T qx = th_flux(t1c, xm1(t1c), wxc, nlam, ix);
            const T qxr = xp1(qx);
            const T qy = th_flux(t1c, tm, wyc, nlam, iy), qyr = th_flux(tq, t1c, wy1c, nlam, iy);
            const T qzr = th_flux(t1, t1c, wz1c, nlam, iz);
            const T dv = ((qxr - qx) * ix + (qyr - qy) * iy) + (qzr - q2z) * iz;
            if (own) row(a.Tout, j, r)[ic] = toc - dt * dv;
            q2z = qzr;
        }
        t1m = t1c;
        t1c = t1;
        toc = to_s;
        wxc = wx_s;
        wyc = wy_s;
        wy1c = wy1_s;
        wz1c = wz1_s;
        __syncthreads();
    }
}

template <class T>
__global__ void __launch_bounds__(256) thermal_update_kernel(Box3 b, DF<T> Tf, DF<T> To, DF<T> q0, DF<T> q1,
                                                             DF<T> q2, int nd, T dt, T i0, T i1, T i2) {
    bool ok;
    Ix3 I = box_index(b, ok);
    if (!ok) return;
    T dv = (g_at(q0, sh(I, 0, 1)) - g_at(q0, I)) * i0;
    if (nd > 1) dv = dv + (g_at(q1, sh(I, 1, 1)) - g_at(q1, I)) * i1;
    if (nd > 2) dv = dv + (g_at(q2, sh(I, 2, 1)) - g_at(q2, I)) * i2;
    g_at(Tf, I) = g_at(To, I) - dt * dv;
}

// ------------------------------------------------------------------ maxloc
template <class T>
__global__ void __launch_bounds__(256) maxloc_kernel(Box3 b, DF<T> dst, DF<T> src, int nd) {
    bool ok;
    Ix3 I = box_index(b, ok);
    if (!ok) return;
    T m = g_at(src, I);
    const int64_t rz = nd > 2 ? 1 : 0, ry = nd > 1 ? 1 : 0;
    for (int64_t c = -rz; c <= rz; ++c)
        for (int64_t bb = -ry; bb <= ry; ++bb)
            for (int64_t a = -1; a <= 1; ++a) m = jmax(m, g_at(src, Ix3{I.i + a, I.j + bb, I.k + c}));
    g_at(dst, I) = m;
}

// ------------------------------------------------------------------ host side
static dim3 blk2() { return dim3(kFlat, 1, 1); }

template <class T>
static int diffusion_launch(const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* q,
                            const chmy_field_t* Cf, double scalar, bool flux, hipStream_t s) {
    chmy_box_t bx;
    CHMY_TRY(check_box(g, box, &bx));
    Box3 b = box3(bx, g->nd);
    if (no_work(b)) return 0;
    DF<T> c = view<T>(*Cf);
    DF<T> q0 = view<T>(q[0]);
    DF<T> q1 = g->nd > 1 ? view<T>(q[1]) : q0, q2 = g->nd > 2 ? view<T>(q[2]) : q0;
    dim3 grd;
    CHMY_TRY(flat_grid(b, (1 + g->nd) * sizeof(T), &grd));
    if (flux)
        hipLaunchKernelGGL(diffusion_flux_kernel<T>, grd, blk2(), 0, s, b, c, q0, q1, q2, g->nd, -T(scalar),
                           T(g->inv_spacing[0]), T(g->inv_spacing[1]), T(g->inv_spacing[2]));
    else
        hipLaunchKernelGGL(diffusion_update_kernel<T>, grd, blk2(), 0, s, b, c, q0, q1, q2, g->nd, T(scalar),
                           T(g->inv_spacing[0]), T(g->inv_spacing[1]), T(g->inv_spacing[2]));
    CHMY_HIP(hipGetLastError());
    return 0;
}

template <class T, int ND, int TX, int TY, int TZ, int KS, int PT>
static int diffusion_tile_launch(const DiffTile<T>& base, int steps, const DF<T>* C, int p, hipStream_t s) {
    DiffTile<T> a = base;
    a.steps = steps;
    a.C = C[p];
    a.Co = C[1 - p];
    const int tile[3] = {TX, TY, TZ};
    int64_t nb = 1;
    for (int d = 0; d < 3; ++d) {
        const int64_t q = d < ND ? ((int64_t)a.n[d] + tile[d] - 1) / tile[d] : 1;
        a.nb[d] = (int32_t)q;
        nb *= q;
    }
    constexpr int NT = DiffShape<T, ND, TX, TY, TZ, KS, PT>::NT;
    dim3 grd;
    CHMY_TRY(line_grid(nb, NT, &grd));
    hipLaunchKernelGGL((diffusion_tile_kernel<T, ND, TX, TY, TZ, KS, PT>), grd, dim3(NT), 0, s, a);
    CHMY_HIP(hipGetLastError());
    return 0;
}

// Tiles.  Small grids, whose time is latency, take one point a thread (2D) or
// 3 (3D) and as many waves as a block holds; grids that fill the chip several
// times over take larger tiles, which compute less ring, with more points a
// thread.  The lines lie where the two cross (f64 us per step, small / large
// tile: 2D 240 k cells 1.75 / 1.50, 65 k 0.95 / 1.5; 3D 262 k cells 3.7 / 6.1,
// 4.1 M 35.9 / 25.7).
constexpr int kDiffK2 = 8, kDiffK3 = 2;
template <class T>
static int diffusion_tile_any(int nd, int k, int64_t cells, const DiffTile<T>& a, const DF<T>* C, int p,
                              hipStream_t s) {
    if (nd == 2)
        return cells < (1 << 17) ? diffusion_tile_launch<T, 2, 16, 16, 1, kDiffK2, 1>(a, k, C, p, s)
                                 : diffusion_tile_launch<T, 2, 32, 32, 1, kDiffK2, 3>(a, k, C, p, s);
    return cells < 3 * (1 << 18) ? diffusion_tile_launch<T, 3, 16, 8, 8, kDiffK3, 3>(a, k, C, p, s)
                                 : diffusion_tile_launch<T, 3, 28, 12, 12, kDiffK3, 8>(a, k, C, p, s);
}

// All but the last step (3D: two) in passes of up to 8 (2D) or 2 (3D) steps, as many
// passes as leave the buffers where single steps would (a pass flips the
// parity once); *done steps were taken.
template <class T>
static int diffusion_passes(const chmy_grid_t* g, const chmy_field_t* C0, const chmy_field_t* C1, const SideRules& r,
                            double chi, double dt, int niter, int* p, int* done, hipStream_t s) {
    const int nd = g->nd, steps = niter - (nd == 2 ? 1 : 2);
    int64_t cells = 1;
    for (int d = 0; d < nd; ++d) cells *= g->n[d];
    if (nd < 2 || steps < 2) return 0;
    DiffTile<T> a;
    std::memset(&a, 0, sizeof a);
    for (int d = 0; d < 3; ++d) {
        if (d < nd && g->n[d] > (int64_t(1) << 30)) return 0;
        a.n[d] = d < nd ? (int32_t)g->n[d] : 1;
        a.isp[d] = T(g->inv_spacing[d]);
    }
    a.nchi = -T(chi);
    a.dt = T(dt);
    a.r = r;
    const DF<T> C[2] = {view<T>(*C0), view<T>(*C1)};
    if (C[0].sy != C[1].sy || C[0].sz != C[1].sz) return 0;   // the kernel takes one stride set
    const int K = nd == 2 ? kDiffK2 : kDiffK3;
    int m = (steps + K - 1) / K;
    if ((m ^ steps) & 1) ++m;   // passes and steps of the same parity
    if (m > steps) return 0;
    for (int q = 0; q < m; ++q) {
        const int k = steps / m + (q < steps % m ? 1 : 0);
        CHMY_TRY(diffusion_tile_any<T>(nd, k, cells, a, C, *p, s));
        *p = 1 - *p;
        *done += k;
    }
    return 0;
}

template <class T>
static int copy_launch(const chmy_grid_t* g, const chmy_box_t& bx, const chmy_field_t* Tf, const chmy_field_t* tau,
                       const chmy_field_t* To, const chmy_field_t* tauo, hipStream_t s) {
    Copy7<T> c;
    int nt = g->nd == 2 ? 3 : 6;
    c.n = 0;
    if (Tf) { c.src[c.n] = view<T>(*Tf); c.dst[c.n] = view<T>(*To); ++c.n; }
    for (int q = 0; q < nt; ++q) { c.src[c.n] = view<T>(tau[q]); c.dst[c.n] = view<T>(tauo[q]); ++c.n; }
    Box3 b = box3(bx, g->nd);
    if (no_work(b)) return 0;
    dim3 grd;
    CHMY_TRY(flat_grid(b, 2 * c.n * sizeof(T), &grd));
    hipLaunchKernelGGL(copy_kernel<T>, grd, blk2(), 0, s, b, c);
    CHMY_HIP(hipGetLastError());
    return 0;
}

template <class T>
static int thermal_launch(const chmy_grid_t* g, const chmy_box_t& bx, const chmy_field_t* q, const chmy_field_t* Tf,
                          const chmy_field_t* other, double scalar, bool flux, hipStream_t s) {
    Box3 b = box3(bx, g->nd);
    if (no_work(b)) return 0;
    DF<T> t = view<T>(*Tf), o = view<T>(other[0]);
    DF<T> q0 = view<T>(q[0]);
    DF<T> q1 = g->nd > 1 ? view<T>(q[1]) : q0, q2 = g->nd > 2 ? view<T>(q[2]) : q0;
    dim3 grd;
    CHMY_TRY(flat_grid(b, (flux ? 1 + 2 * g->nd : 2 + g->nd) * sizeof(T), &grd));
    if (flux) {
        DF<T> v1 = g->nd > 1 ? view<T>(other[1]) : o, v2 = g->nd > 2 ? view<T>(other[2]) : o;
        hipLaunchKernelGGL(thermal_flux_kernel<T>, grd, blk2(), 0, s, b, t, o, v1, v2, q0, q1, q2, g->nd, -T(scalar),
                           T(g->inv_spacing[0]), T(g->inv_spacing[1]), T(g->inv_spacing[2]));
    } else {
        hipLaunchKernelGGL(thermal_update_kernel<T>, grd, blk2(), 0, s, b, t, o, q0, q1, q2, g->nd, T(scalar),
                           T(g->inv_spacing[0]), T(g->inv_spacing[1]), T(g->inv_spacing[2]));
    }
    CHMY_HIP(hipGetLastError());
    return 0;
}

}  // namespace chmy

using namespace chmy;

extern "C" {

int chmy_diffusion_flux(const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* q, const chmy_field_t* C,
                        double chi, void* stream) {
    CHMY_TRY(check_grid(g));
    CHMY_TRY(check_center(g, C, "C", -1));
    CHMY_TRY(check_vector(g, q, "q", C->dtype));
    return C->dtype == CHMY_F64 ? diffusion_launch<double>(g, box, q, C, chi, true, (hipStream_t)stream)
                                : diffusion_launch<float>(g, box, q, C, chi, true, (hipStream_t)stream);
}

int chmy_diffusion_update(const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* C,
                          const chmy_field_t* q, double dt, void* stream) {
    CHMY_TRY(check_grid(g));
    CHMY_TRY(check_center(g, C, "C", -1));
    CHMY_TRY(check_vector(g, q, "q", C->dtype));
    return C->dtype == CHMY_F64 ? diffusion_launch<double>(g, box, q, C, dt, false, (hipStream_t)stream)
                                : diffusion_launch<float>(g, box, q, C, dt, false, (hipStream_t)stream);
}

int chmy_diffusion_step(const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* C,
                        const chmy_field_t* C_out, const chmy_field_t* q, double chi, double dt, void* stream) {
    CHMY_TRY(check_grid(g));
    CHMY_TRY(check_center(g, C, "C", -1));
    CHMY_TRY(check_center(g, C_out, "C_out", C->dtype));
    CHMY_TRY(check_vector(g, q, "q", C->dtype));
    if (C->data == C_out->data) return set_error(CHMY_E_ARG, "C and C_out must be distinct buffers");
    chmy_box_t bx;
    CHMY_TRY(check_box(g, box, &bx));
    Box3 b = box3(bx, g->nd);
    if (no_work(b)) return 0;
    auto launch = [&](auto zero) -> int {
        using T = decltype(zero);
        DF<T> c = view<T>(*C), co = view<T>(*C_out);
        DF<T> q0 = view<T>(q[0]);
        DF<T> q1 = g->nd > 1 ? view<T>(q[1]) : q0, q2 = g->nd > 2 ? view<T>(q[2]) : q0;
        dim3 grd;
        CHMY_TRY(flat_grid(b, (2 + g->nd) * sizeof(T), &grd));
        hipLaunchKernelGGL(diffusion_step_kernel<T>, grd, blk2(), 0, (hipStream_t)stream, b, c, co, q0, q1, q2,
                           g->nd, -T(chi), T(dt), T(g->inv_spacing[0]), T(g->inv_spacing[1]),
                           T(g->inv_spacing[2]));
        CHMY_HIP(hipGetLastError());
        return 0;
    };
    return C->dtype == CHMY_F64 ? launch(0.0) : launch(0.0f);
}

int chmy_diffusion_iterate(const chmy_grid_t* g, const chmy_field_t* C0, const chmy_field_t* C1,
                           const chmy_field_t* q, const int32_t* bc_counts, const chmy_bc_t* bcs, double chi,
                           double dt, int niter, int* parity_inout, void* stream) {
    CHMY_TRY(check_grid(g));
    if (!parity_inout || (*parity_inout != 0 && *parity_inout != 1)) return set_error(CHMY_E_ARG, "parity must be 0/1");
    if (niter < 0) return set_error(CHMY_E_ARG, "niter < 0");
    if (!bc_counts || !bcs) return set_error(CHMY_E_ARG, "C batch is NULL");
    int total = 0;
    for (int k = 0; k < 2 * g->nd; ++k) {
        if (bc_counts[k] < 0 || bc_counts[k] > 1) return set_error(CHMY_E_ARG, "one C entry per (dim, side) at most");
        total += bc_counts[k];
    }
    const chmy_field_t* Cs[2] = {C0, C1};
    chmy_field_t fset[2][6];
    for (int s = 0; s < 2; ++s)
        for (int k = 0; k < total; ++k) fset[s][k] = *Cs[s];
    chmy_box_t box;
    for (int d = 0; d < 3; ++d) {
        box.lo[d] = 0;
        box.len[d] = d < g->nd ? g->n[d] + 2 : 1;
    }
    int p = *parity_inout;
    // one scalar rule on every (dim, side): the batch rides in the step's launch
    bool fold = total == 2 * g->nd;
    SideRules rules;
    std::memset(&rules, 0, sizeof rules);
    for (int k = 0; fold && k < total; ++k) {
        const chmy_bc_t& c = bcs[k];
        fold = (c.kind == CHMY_DIRICHLET || c.kind == CHMY_NEUMANN) &&
               (c.vkind == CHMY_VALUE_ZERO || c.vkind == CHMY_VALUE_SCALAR);   // else the batch set validates
        rules.kind[k / 2][k % 2] = c.kind;
        rules.val[k / 2][k % 2] = c.vkind == CHMY_VALUE_SCALAR ? c.value : 0.0;
    }
    if (fold && niter > 0) {
        for (int d = 0; d < 3; ++d) rules.h[d] = g->spacing[d];
        CHMY_TRY(check_center(g, C0, "C0", -1));
        CHMY_TRY(check_center(g, C1, "C1", C0->dtype));
        CHMY_TRY(check_vector(g, q, "q", C0->dtype));
        if (C0->data == C1->data) return set_error(CHMY_E_ARG, "C0 and C1 must be distinct buffers");
        chmy_box_t bx;
        CHMY_TRY(check_box(g, &box, &bx));
        const Box3 b = box3(bx, g->nd);
        Box3 reg = b;
        for (int d = 0; d < g->nd; ++d) reg.len[d] = b.len[d] + 1;   // [0, n+2]
        auto run = [&](auto zero) -> int {
            using T = decltype(zero);
            DF<T> c[2] = {view<T>(*C0), view<T>(*C1)};
            DF<T> q0 = view<T>(q[0]);
            DF<T> q1 = g->nd > 1 ? view<T>(q[1]) : q0, q2 = g->nd > 2 ? view<T>(q[2]) : q0;
            dim3 grd;
            CHMY_TRY(flat_grid(reg, (2 + g->nd) * sizeof(T), &grd));
            int it = 0;
            CHMY_TRY(diffusion_passes<T>(g, C0, C1, rules, chi, dt, niter, &p, &it, (hipStream_t)stream));
            for (; it < niter; ++it) {
                hipLaunchKernelGGL(diffusion_step_bc_kernel<T>, grd, blk2(), 0, (hipStream_t)stream, b, reg, c[p],
                                   c[1 - p], q0, q1, q2, g->nd, -T(chi), T(dt), T(g->inv_spacing[0]),
                                   T(g->inv_spacing[1]), T(g->inv_spacing[2]), rules);
                p = 1 - p;
            }
            CHMY_HIP(hipGetLastError());
            return 0;
        };
        CHMY_TRY(C0->dtype == CHMY_F64 ? run(0.0) : run(0.0f));
        *parity_inout = p;
        return 0;
    }
    for (int it = 0; it < niter; ++it) {
        CHMY_TRY(chmy_diffusion_step(g, &box, Cs[p], Cs[1 - p], q, chi, dt, stream));
        CHMY_TRY(chmy_bc_batchset(g, bc_counts, fset[1 - p], bcs, stream));
        p = 1 - p;
    }
    *parity_inout = p;
    return 0;
}

int chmy_stokes_update_old(const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* Tf,
                           const chmy_field_t* tau, const chmy_field_t* To, const chmy_field_t* tauo, void* stream) {
    CHMY_TRY(check_grid(g));
    chmy_box_t bx;
    CHMY_TRY(check_box(g, box, &bx));
    CHMY_TRY(check_tensor(g, tau, "tau", -1));
    const int dt = tau[0].dtype;
    CHMY_TRY(check_tensor(g, tauo, "tau_old", dt));
    if ((Tf == nullptr) != (To == nullptr)) return set_error(CHMY_E_ARG, "T and T_old must both be given or NULL");
    if (Tf) {
        CHMY_TRY(check_center(g, Tf, "T", dt));
        CHMY_TRY(check_center(g, To, "T_old", dt));
    }
    return dt == CHMY_F64 ? copy_launch<double>(g, bx, Tf, tau, To, tauo, (hipStream_t)stream)
                          : copy_launch<float>(g, bx, Tf, tau, To, tauo, (hipStream_t)stream);
}

int chmy_thermal_flux(const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* qT, const chmy_field_t* Tf,
                      const chmy_field_t* V, double lam, void* stream) {
    CHMY_TRY(check_grid(g));
    chmy_box_t bx;
    CHMY_TRY(check_box(g, box, &bx));
    CHMY_TRY(check_center(g, Tf, "T", -1));
    CHMY_TRY(check_vector(g, qT, "qT", Tf->dtype));
    CHMY_TRY(check_vector(g, V, "V", Tf->dtype));
    return Tf->dtype == CHMY_F64 ? thermal_launch<double>(g, bx, qT, Tf, V, lam, true, (hipStream_t)stream)
                                 : thermal_launch<float>(g, bx, qT, Tf, V, lam, true, (hipStream_t)stream);
}

int chmy_thermal_update(const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* Tf,
                        const chmy_field_t* To, const chmy_field_t* qT, double dt, void* stream) {
    CHMY_TRY(check_grid(g));
    chmy_box_t bx;
    CHMY_TRY(check_box(g, box, &bx));
    CHMY_TRY(check_center(g, Tf, "T", -1));
    CHMY_TRY(check_center(g, To, "T_old", Tf->dtype));
    CHMY_TRY(check_vector(g, qT, "qT", Tf->dtype));
    return Tf->dtype == CHMY_F64 ? thermal_launch<double>(g, bx, qT, Tf, To, dt, false, (hipStream_t)stream)
                                 : thermal_launch<float>(g, bx, qT, Tf, To, dt, false, (hipStream_t)stream);
}

int chmy_thermal_step(const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* Tf, const chmy_field_t* T_out,
                      const chmy_field_t* To, const chmy_field_t* qT, const chmy_field_t* V, double lam, double dt,
                      void* stream) {
    CHMY_TRY(check_grid(g));
    chmy_box_t bx;
    CHMY_TRY(check_box(g, box, &bx));
    CHMY_TRY(check_center(g, Tf, "T", -1));
    CHMY_TRY(check_center(g, T_out, "T_out", Tf->dtype));
    CHMY_TRY(check_center(g, To, "T_old", Tf->dtype));
    CHMY_TRY(check_vector(g, qT, "qT", Tf->dtype));
    CHMY_TRY(check_vector(g, V, "V", Tf->dtype));
    if (Tf->data == T_out->data) return set_error(CHMY_E_ARG, "T and T_out must be distinct buffers");
    Box3 b = box3(bx, g->nd);
    if (no_work(b)) return 0;
    auto launch = [&](auto zero) -> int {
        using T = decltype(zero);
        DF<T> t = view<T>(*Tf), to = view<T>(*T_out), o = view<T>(*To);
        DF<T> v0 = view<T>(V[0]), q0 = view<T>(qT[0]);
        DF<T> v1 = g->nd > 1 ? view<T>(V[1]) : v0, v2 = g->nd > 2 ? view<T>(V[2]) : v0;
        DF<T> q1 = g->nd > 1 ? view<T>(qT[1]) : q0, q2 = g->nd > 2 ? view<T>(qT[2]) : q0;
        // 3D with one stride set per location (Center; each V_D with qT_D): the z-march
        bool march = g->nd == 3;
        if (march) {
            const DF<T> c = view<T>(*Tf), c1 = view<T>(*T_out), c2 = view<T>(*To);
            march = c1.sy == c.sy && c1.sz == c.sz && c2.sy == c.sy && c2.sz == c.sz;
            for (int d = 0; d < 3; ++d) {
                const DF<T> a = view<T>(V[d]), q = view<T>(qT[d]);
                march = march && a.sy == q.sy && a.sz == q.sz;
            }
        }
        if (march) {
            const int nbx = (int)((b.len[0] + 63) / 64), nby = (int)((b.len[1] + kThY - 1) / kThY);
            const int64_t nch = (b.len[2] + 15) / 16;
            const int kchunk = (int)((b.len[2] + nch - 1) / nch);
            dim3 grd;
            CHMY_TRY(line_grid((int64_t)nbx * nby * nch, 64 * kThY, &grd));
            hipLaunchKernelGGL(thermal_step3_kernel<T>, grd, dim3(64, kThY, 1), 0, (hipStream_t)stream,
                               b, view<T>(*Tf), view<T>(*T_out), view<T>(*To), view<T>(V[0]), view<T>(V[1]),
                               view<T>(V[2]), view<T>(qT[0]), view<T>(qT[1]), view<T>(qT[2]), -T(lam), T(dt),
                               T(g->inv_spacing[0]), T(g->inv_spacing[1]), T(g->inv_spacing[2]), nbx, nby, kchunk);
            CHMY_HIP(hipGetLastError());
            return 0;
        }
        dim3 grd;
        CHMY_TRY(flat_grid(b, (3 + 2 * g->nd) * sizeof(T), &grd));
        hipLaunchKernelGGL(thermal_step_kernel<T>, grd, blk2(), 0, (hipStream_t)stream, b, t, to, o, v0, v1, v2, q0,
                           q1, q2, g->nd, -T(lam), T(dt), T(g->inv_spacing[0]), T(g->inv_spacing[1]),
                           T(g->inv_spacing[2]));
        CHMY_HIP(hipGetLastError());
        return 0;
    };
    return Tf->dtype == CHMY_F64 ? launch(0.0) : launch(0.0f);
}

int chmy_thermal_step2(const chmy_grid_t* g, const chmy_field_t* Tf, const chmy_field_t* T_out, const chmy_field_t* To,
                       const chmy_field_t* V1, const chmy_field_t* V2, double lam, double dt, void* stream) {
    CHMY_TRY(check_grid(g));
    if (g->nd != 3) return set_error(CHMY_E_ARG, "chmy_thermal_step2 is 3D");
    CHMY_TRY(check_center(g, Tf, "T", -1));
    CHMY_TRY(check_center(g, T_out, "T_out", Tf->dtype));
    CHMY_TRY(check_center(g, To, "T_old", Tf->dtype));
    CHMY_TRY(check_vector(g, V1, "V1", Tf->dtype));
    CHMY_TRY(check_vector(g, V2, "V2", Tf->dtype));
    if (T_out->data == Tf->data || T_out->data == To->data)
        return set_error(CHMY_E_ARG, "T_out must be distinct from T and T_old");
    auto launch = [&](auto zero) -> int {
        using T = decltype(zero);
        Thermal2<T> a;
        a.Tf = view<T>(*Tf);
        a.Tout = view<T>(*T_out);
        a.To = view<T>(*To);
        for (int d = 0; d < 3; ++d) {
            a.V1[d] = view<T>(V1[d]);
            a.V2[d] = view<T>(V2[d]);
            a.is[d] = T(g->inv_spacing[d]);
            a.n[d] = (int)g->n[d];
        }
        a.nlam = -T(lam);
        a.dt = T(dt);
        a.nbx = (a.n[0] + 59) / 60;
        a.nby = (a.n[1] + kTh2Y - 3) / (kTh2Y - 2);
        // chunks of z that fill whole rounds of the CUs (one block a CU, 2
        // planes a chunk recomputed), as the two-iteration Stokes pass picks its own
        const int64_t tiles = (int64_t)a.nbx * a.nby, slots = cu_count();
        int64_t best = INT64_MAX;
        a.kchunk = a.n[2];
        for (int nch = 1; nch <= a.n[2] && nch <= 64; ++nch) {
            const int k = (a.n[2] + nch - 1) / nch;
            const int64_t cost = (tiles * ((a.n[2] + k - 1) / k) + slots - 1) / slots * (k + 2);
            if (cost < best) {
                best = cost;
                a.kchunk = k;
            }
        }
        dim3 grd;
        CHMY_TRY(line_grid(tiles * ((a.n[2] + a.kchunk - 1) / a.kchunk), 64 * kTh2Y, &grd));
        hipLaunchKernelGGL(thermal_step2_kernel<T>, grd, dim3(64, kTh2Y, 1), 0, (hipStream_t)stream, a);
        CHMY_HIP(hipGetLastError());
        return 0;
    };
    return Tf->dtype == CHMY_F64 ? launch(0.0) : launch(0.0f);
}

int chmy_maxloc(const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* dst, const chmy_field_t* src,
                void* stream) {
    CHMY_TRY(check_grid(g));
    chmy_box_t bx;
    CHMY_TRY(check_box(g, box, &bx));
    CHMY_TRY(check_center(g, src, "src", -1));
    CHMY_TRY(check_center(g, dst, "dst", src->dtype));
    Box3 b = box3(bx, g->nd);
    if (no_work(b)) return 0;
    hipStream_t s = (hipStream_t)stream;
    dim3 grd;
    CHMY_TRY(flat_grid(b, 2 * (src->dtype == CHMY_F64 ? 8 : 4), &grd));
    if (src->dtype == CHMY_F64)
        hipLaunchKernelGGL(maxloc_kernel<double>, grd, blk2(), 0, s, b, view<double>(*dst), view<double>(*src),
                           g->nd);
    else
        hipLaunchKernelGGL(maxloc_kernel<float>, grd, blk2(), 0, s, b, view<float>(*dst), view<float>(*src), g->nd);
    CHMY_HIP(hipGetLastError());
    return 0;
}

}  // extern "C"
