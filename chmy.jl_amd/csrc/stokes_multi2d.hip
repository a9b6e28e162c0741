// Several PT iterations of a 2D free-slip solve per launch (chmy_stokes_iterate).
#include "stokes_pt.hpp"

namespace chmy {

// A pass's shape: iterations, waves per block, rows per thread.
template <int KM_, int W_, int PT_>
struct Shape2 {
    static constexpr int KM = KM_, W = W_, PT = PT_, TX = kFX - 2 * KM, TY = W * PT - 2 * KM;
};
using Small2 = Shape2<7, 16, 1>;
using Flat2 = Shape2<5, 16, 1>;
using Mid2 = Shape2<6, 16, 2>;
using Large2 = Shape2<8, 16, 3>;
using Dense2 = Shape2<5, 8, 3>;

// The first shape whose tiles all find a CU of their own is taken: the time is
// then one block's chain of iterations, and the flatter the tile, the shorter
// that chain.  Beyond, Dense2: two blocks of 8 waves a CU, so one computes
// while the other loads and stores (16 waves of 125 VGPRs fill a CU alone),
// at the same share of own points as Large2 (49% and 50%) but a pass of 5
// iterations.  FP64 us for 33 iterations, Mid2 / Large2 / Dense2: 600x512 272 /
// 231 / 246 (221 tiles of Large2), 800x640 340 / 313 / 297 (357 tiles),
// 1400x1200 693 / 633 / 592; 41 at 2047^2 1734 (Large2) / 1584; other waves,
// rows and lengths for the last one: <4, 8, 3> 1775, <6, 8, 3> 1668, <5, 16, 3>
// 1982, <6, 12, 4> 1840, <5, 6, 4> 2512.  400x380: Mid2 and Dense2 alike.  Mid2 /
// Flat2, 33 iterations: 200x150 188 / 152, 280x240 190 / 156, 160x150 in the
// exact form 250 / 184 (<5, 14, 1> 153 / 188 / 183, <6, 15, 1> 158 / 191 / 197).
static int64_t tiles2(int64_t nbx, int64_t nby, int tx, int ty) { return ((nbx + tx - 1) / tx) * ((nby + ty - 1) / ty); }
template <class Sh>
static bool one_round(int64_t nbx, int64_t nby) {
    return tiles2(nbx, nby, Sh::TX, Sh::TY) <= cu_count();
}
static int shape2(int64_t nbx, int64_t nby) {
    return one_round<Small2>(nbx, nby)  ? 0
           : one_round<Flat2>(nbx, nby) ? 1
           : one_round<Mid2>(nbx, nby)  ? 2
           : one_round<Large2>(nbx, nby) ? 3
                                         : 4;
}

// A run of iterations is cut into evenly long passes of at most the shape's
// iterations, three or more each (a remainder of one or two would take a launch
// that moves the state for itself).  FP32 in the exact form on large grids takes
// passes of five and two instead: there the two-iteration pass streams at its
// best while the divisions and the ring, five deep however short the pass,
// bound this one.  2047^2, variable eta, us per iteration: passes of 3 / 4 / 5 54 /
// 49 / 47, of 2 48, single 71; 4000^2 (6 iterations in 3 + 3 against 2 + 2 + 2) 198
// against 171 (and fives 174).  The line: at 1400^2 two passes of 3 and three of 2 take the same;
// with forcing, which a pass reads once for all its iterations, two of 4 and
// four of 2 do at 2500^2 (three of 2 10% less than two of 3).
int multi2d_next(const chmy_grid_t* g, bool f32_exact, bool forced, int run) {
    const int64_t nbx = g->n[0] + 2, nby = g->n[1] + 2;
    const int km[5] = {Small2::KM, Flat2::KM, Mid2::KM, Large2::KM, Dense2::KM};
    const int shape = shape2(nbx, nby), most = km[shape];
    if (run < 3) return 0;
    const int64_t line = (forced ? 10 : 5) * (int64_t(1) << 19);
    if (f32_exact && shape == 4 && nbx * nby >= line && run != 3)
        return run >= 2 * most || (run >= most && run % 2) ? most : 0;
    const int passes = (run + most - 1) / most;
    return (run + passes - 1) / passes;
}

// Up to KM PT iterations of a tile on chip (build extension): the state is
// read and written once for all of them, where a pass of two iterations moved
// it every second iteration (2047^2: 143 us a pass, near what its 17 arrays
// take at the copy rate; on small grids a serial march of 12 rows, 16 us).
// A block is W waves of 64 columns; a thread holds PT consecutive rows of the
// state, tau_old and the eta-derived coefficients (formed once per pass) in
// registers.  x neighbours are DPP lane shifts, y neighbours registers, and
// the rows at a wave's two ends go through LDS: V's after the velocity phase,
// the stresses' after the stress phase, two barriers an iteration.  Between
// iterations the free-slip V batch is applied as fused2d_tb_kernel applies it
// (blocks that hold no boundary skip it).  An iteration uses up one ring of
// the tile: after s iterations positions [s, 63 - s] x [s, W PT - 1 - s] are
// exact, and the tile's own are KM from each end.  Loads are clamped into the
// stored range; clamped values reach no output.  The expressions are row2's,
// so the results are bitwise those of single iterations with the batch
// between them; the batch after the last one is the caller's, or the next
// pass's, which applies it to the V it reads (fs.pre; 4.5 us a launch and its
// gap, a quarter of a pass at 127x95).
// Bound by FP64 issue: 16 waves of up to 128 VGPRs fill a CU (4 a SIMD, what
// the launch bounds ask for), as one block or as two.
template <class T, bool FVISC, bool EXACT, bool HF, bool BF, bool RG, int KM, int W, int PT>
__global__ void __launch_bounds__(kFX * W, 4) fused2d_multi_kernel(Fused2<T> a, FreeSlip2 fs, int iters) {
    using AR = Arith<T, EXACT>;
    using Loc = typename AR::Loc;
    constexpr int R = W * PT;
    __shared__ T sV[3][W][kFX], sS[3][W][kFX];   // V: Vx first row, Vx last, Vy first; stresses: txy first, P last, tyy last
    const Kc<T>& K = a.k;
    const int lane = threadIdx.x, w = threadIdx.y;
    const int t = xcd_remap(blockIdx.x, gridDim.x);
    const int xb = (t % a.ntx) * (kFX - 2 * KM) - KM, yb = (t / a.ntx) * (R - 2 * KM) - KM;
    const int i = xb + lane, j0 = yb + w * PT;
    const int n0 = a.n[0], n1 = a.n[1], nb0 = n0 + 1, nb1 = n1 + 1;
    const bool inx = i >= 0 && i <= nb0;
    const bool edge = xb <= 1 || xb + kFX - 1 >= n0 || yb <= 1 || yb + R - 1 >= n1;
    const int ic = min(max(i, -1), n0 + 2);
    const T ix = a.ix, iy = a.iy;
    constexpr uint32_t E = sizeof(T);
    auto off = [&](int c, int r) -> uint32_t {   // byte offset of (ic, row r clamped into the stored rows)
        const uint32_t k = (uint32_t)(min(max(r, -1), n1 + 2) + 1);
        return (a.L[c].o0 + (uint32_t)ic - a.L[c].sy + k * a.L[c].sy) * E;
    };
    T vx[PT], vy[PT], P[PT], txx[PT], tyy[PT], txy[PT], cx[PT], cy[PT];
    Fraw<T, BF> oxx[PT], oyy[PT], oxy[PT], fP[PT], fVx[PT], fVy[PT];
    T rg[PT];
    Loc Lc[PT], Le[PT];
    T eta_m = FVISC ? ldo(a.eta, off(L2C, j0 - 1)) : T(0), eml_m = FVISC ? ldo(a.eml, off(L2C, j0 - 1)) : T(0);
#pragma unroll
    for (int q = 0; q < PT; ++q) {
        const uint32_t oc = off(L2C, j0 + q), ox = off(L2X, j0 + q), oy = off(L2Y, j0 + q), oe = off(L2XY, j0 + q);
        vx[q] = ldo(a.Vx, ox);
        vy[q] = ldo(a.Vy, oy);
        P[q] = ldo(a.Pr, oc);
        txx[q] = ldo(a.txx, oc);
        tyy[q] = ldo(a.tyy, oc);
        txy[q] = ldo(a.txy, oe);
        oxx[q] = ldr<T, BF>(a.Oxx, oc);
        oyy[q] = ldr<T, BF>(a.Oyy, oc);
        oxy[q] = ldr<T, BF>(a.Oxy, oe);
        if constexpr (HF) {
            fP[q] = ldr<T, BF>(a.fP, oc);
            fVx[q] = ldr<T, BF>(a.fVx, ox);
            fVy[q] = ldr<T, BF>(a.fVy, oy);
        }
        if constexpr (RG) rg[q] = ldo(a.rg, oy);
        if constexpr (FVISC) {
            const T eta = ldo(a.eta, oc), eml = ldo(a.eml, oc);
            Lc[q] = AR::field(eta, K);
            Le[q] = AR::field(lerp4(xm1(eta_m), eta_m, xm1(eta), eta), K);
            cx[q] = AR::vcoef_field(jmax(xm1(eml), eml), K);
            cy[q] = AR::vcoef_field(jmax(eml_m, eml), K);
            eta_m = eta;
            eml_m = eml;
        } else {
            Lc[q] = Le[q] = AR::scalar(K);
            cx[q] = cy[q] = AR::vcoef_scalar(K);
        }
    }
    const T hx = T(fs.hx), hy = T(fs.hy);
    const bool i_in = i >= 0 && i <= n0 + 2;
    auto vx_bc = [&](int r, T rm, T r0, T rp) -> T {
        T v = r0;
        if (r == 0 && i_in) v = fma(hy, -T(fs.qy[0]), rp);
        else if (r == n1 + 1 && i_in) v = fma(hy, T(fs.qy[1]), rm);
        if ((i == 1 || i == n0 + 1) && r >= 0 && r <= n1 + 2) v = T(fs.ax[i == 1 ? 0 : 1]);
        return v;
    };
    auto vy_bc = [&](int r, T r0) -> T {
        T v = r0;
        if (i_in && r == 1) v = T(fs.by[0]);
        else if (i_in && r == n1 + 1) v = T(fs.by[1]);
        const T dn = xp1(v), up = xm1(v);
        const bool r_in = r >= 0 && r <= n1 + 2;
        if (i == 0 && r_in) return fma(hx, -T(fs.qx[0]), dn);
        if (i == n0 + 1 && r_in) return fma(hx, T(fs.qx[1]), up);
        return v;
    };
    const int wm = max(w - 1, 0), wp = min(w + 1, W - 1);   // (the region's own ends read a row that reaches no output)
    sV[0][w][lane] = vx[0];
    sV[1][w][lane] = vx[PT - 1];
    sV[2][w][lane] = vy[0];
#pragma unroll 1
    for (int it = 0; it < iters; ++it) {
        __syncthreads();
        T vxp = sV[1][wm][lane], vyn = sV[2][wp][lane];   // Vx at row j0 - 1, Vy at row j0 + PT
        if ((it > 0 || fs.pre) && edge) {
            const T first = vx[0];
            T rm = vxp;
#pragma unroll
            for (int q = 0; q < PT; ++q) {
                const T r0 = vx[q], rp = q + 1 < PT ? vx[q + 1] : sV[0][wp][lane];
                vx[q] = vx_bc(j0 + q, rm, r0, rp);
                vy[q] = vy_bc(j0 + q, vy[q]);
                rm = r0;
            }
            vxp = vx_bc(j0 - 1, vxp, vxp, first);
            vyn = vy_bc(j0 + PT, vyn);
        }
        // stresses and Pr
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            const bool in = inx && j0 + q >= 0 && j0 + q <= nb1;
            const T exx = (xp1(vx[q]) - vx[q]) * ix;
            const T eyy = ((q + 1 < PT ? vy[q + 1] : vyn) - vy[q]) * iy;
            const T dv = exx + eyy;
            const T Pn = AR::pr(P[q], HF ? dv - cvf<T, BF>(fP[q]) : dv, Lc[q], K);
            const T txxn = AR::diag(txx[q], cvf<T, BF>(oxx[q]), exx, dv, Lc[q], K);
            const T tyyn = AR::diag(tyy[q], cvf<T, BF>(oyy[q]), eyy, dv, Lc[q], K);
            const T exy = T(0.5) * ((vx[q] - (q > 0 ? vx[q - 1] : vxp)) * iy + (vy[q] - xm1(vy[q])) * ix);
            const T txyn = AR::off(txy[q], cvf<T, BF>(oxy[q]), exy, Le[q], K);
            P[q] = in ? Pn : P[q];
            txx[q] = in ? txxn : txx[q];
            tyy[q] = in ? tyyn : tyy[q];
            txy[q] = in ? txyn : txy[q];
        }
        sS[0][w][lane] = txy[0];
        sS[1][w][lane] = P[PT - 1];
        sS[2][w][lane] = tyy[PT - 1];
        __syncthreads();
        const T txyN = sS[0][wp][lane], Pp = sS[1][wm][lane], tyyp = sS[2][wm][lane];
        // velocities
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            const bool in = inx && j0 + q >= 0 && j0 + q <= nb1;
            const T txy1 = q + 1 < PT ? txy[q + 1] : txyN;
            T rx = (-((P[q] - xm1(P[q])) * ix) + (txx[q] - xm1(txx[q])) * ix) + (txy1 - txy[q]) * iy;
            T ry = (-((P[q] - (q > 0 ? P[q - 1] : Pp)) * iy) + (tyy[q] - (q > 0 ? tyy[q - 1] : tyyp)) * iy) +
                   (xp1(txy[q]) - txy[q]) * ix;
            if constexpr (RG) ry = ry - rg[q];
            if constexpr (HF) {
                rx = rx + cvf<T, BF>(fVx[q]);
                ry = ry + cvf<T, BF>(fVy[q]);
            }
            const T vxn = AR::vel(vx[q], rx, cx[q], K), vyn1 = AR::vel(vy[q], ry, cy[q], K);
            vx[q] = in ? vxn : vx[q];
            vy[q] = in ? vyn1 : vy[q];
        }
        sV[0][w][lane] = vx[0];
        sV[1][w][lane] = vx[PT - 1];
        sV[2][w][lane] = vy[0];
    }
    const bool own = lane >= KM && lane < kFX - KM && inx;
#pragma unroll
    for (int q = 0; q < PT; ++q) {
        const int pos = w * PT + q, j = j0 + q;
        if (!own || pos < KM || pos >= R - KM || j < 0 || j > nb1) continue;
        const uint32_t oc = off(L2C, j);
        sto(a.oPr, oc, P[q]);
        sto(a.otxx, oc, txx[q]);
        sto(a.otyy, oc, tyy[q]);
        sto(a.otxy, off(L2XY, j), txy[q]);
        sto(a.oVx, off(L2X, j), vx[q]);
        sto(a.oVy, off(L2Y, j), vy[q]);
    }
}

template <class T>
void multi2d_launch(Fused2<T> a, const FreeSlip2& fs, bool fv, bool exact, bool bf, bool rg, hipStream_t s) {
    const bool hf = a.has_f;
    const int64_t nbx = a.n[0] + 2, nby = a.n[1] + 2;
    auto go = [&](auto shape) {
        using Sh = decltype(shape);
        constexpr int KM = Sh::KM, W = Sh::W, PT = Sh::PT;
        a.ntx = (int32_t)((nbx + Sh::TX - 1) / Sh::TX);
        const dim3 blk(kFX, W, 1), grd((unsigned)tiles2(nbx, nby, Sh::TX, Sh::TY), 1, 1);
#define CHMY_M2(FV, EX, HF, BFF, RG) \
    hipLaunchKernelGGL((fused2d_multi_kernel<T, FV, EX, HF, BFF, RG, KM, W, PT>), grd, blk, 0, s, a, fs, fs.iters)
#define CHMY_M2R(FV, EX, RG)                                \
    do {                                                    \
        constexpr bool F32 = std::is_same<T, float>::value; \
        if (hf && bf) CHMY_M2(FV, EX, true, F32, RG);       \
        else if (hf) CHMY_M2(FV, EX, true, false, RG);      \
        else CHMY_M2(FV, EX, false, false, RG);             \
    } while (0)
#define CHMY_M2E(FV, EX)                \
    do {                                \
        if (rg) CHMY_M2R(FV, EX, true); \
        else CHMY_M2R(FV, EX, false);   \
    } while (0)
        if (fv && exact) CHMY_M2E(true, true);
        else if (fv) CHMY_M2E(true, false);
        else if (exact) CHMY_M2E(false, true);
        else CHMY_M2E(false, false);
#undef CHMY_M2E
#undef CHMY_M2R
#undef CHMY_M2
    };
    switch (shape2(nbx, nby)) {
        case 0: go(Small2{}); break;
        case 1: go(Flat2{}); break;
        case 2: go(Mid2{}); break;
        case 3: go(Large2{}); break;
        default: go(Dense2{}); break;
    }
}

template void multi2d_launch<double>(Fused2<double>, const FreeSlip2&, bool, bool, bool, bool, hipStream_t);
template void multi2d_launch<float>(Fused2<float>, const FreeSlip2&, bool, bool, bool, bool, hipStream_t);

}  // namespace chmy
