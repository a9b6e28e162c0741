// Shallow-ice (SIA) nonlinear diffusion: forward kernels of examples/sia.jl
// and a hand-written adjoint of one explicit step (build extension).
//
// Forward (sia.jl:7-16,30-54), on cells/vertices 1..n of a 2D grid:
//   S = B + H;  g_x = ∂x S (vertex);  a_x = lerp(g_x → centre);  vm = sqrt(a_x²+a_y²)
//   D = (A H^(n+2) + As H^n) vm^(n-1)          (A ≡ 1 reproduces sia.jl's D)
//   q_x = -lerp(D → x-vertex) g_x,  boundary vertices 0 (q Dirichlet on all sides)
//   M = min(mb_a (S - mb_b), mb_c);  H' = max(H + Δt(-divg q + M), 0)
// Powers are repeated products; lerp is fma(0.5, b - a, a) as in Chmy.  Lazy
// FunctionFields are evaluated at every access, so D is recomputed per use.
//
// Adjoint of one step H -> H' (reverse mode, exact derivative of the
// discrete map above; max(x,0) and min(..) take the branch they took):
//   A1 cells   mu = lam [x > 0]
//   A2 faces   qbar = Δt iΔ (mu_right - mu_left) on interior faces;
//              Dvbar = -g qbar,  gbar_direct = -lerp(D) qbar
//   A3 cells   Dbar = ½ Σ Dvbar of the 4 faces;  Abar → grad_logA += A Abar;
//              HDbar = Dbar ∂D/∂H;  abar = Dbar ∂D/∂a
//   A4 faces   gbar = gbar_direct + ½ (abar of the 2 cells sharing the face)
//   A5 cells   lam' = mu + HDbar + Sbar, Sbar = iΔ(gbar_left - gbar_right) (+ M branch);
//              halo cells fold into their neighbour (the Neumann copy H_0 = H_1).
// Each pass is a gather, so no float atomics and the result is deterministic.
#include <algorithm>
#include <mutex>

#include <vector>

#include "stokes_pt.hpp"

namespace chmy {

struct SiaPar {
    double As;
    int npow;
    double mb_a, mb_b, mb_c, dt;
};

template <class T>
__device__ __forceinline__ T ipow_(T x, int n) {
    T r = T(1);
    for (int i = 0; i < n; ++i) r = r * x;
    return r;
}

template <class T>
struct SiaF {
    DF<T> H, B, A;
    int hasA;
    T ix, iy, As, mba, mbb, mbc;
    int n;
    __device__ T S(int64_t i, int64_t j) const { return B(i, j, 0) + H(i, j, 0); }
    __device__ T gx(int64_t i, int64_t j) const { return (S(i, j) - S(i - 1, j)) * ix; }
    __device__ T gy(int64_t i, int64_t j) const { return (S(i, j) - S(i, j - 1)) * iy; }
    __device__ T ax(int64_t i, int64_t j) const { T l = gx(i, j), r = gx(i + 1, j); return fma(T(0.5), r - l, l); }
    __device__ T ay(int64_t i, int64_t j) const { T l = gy(i, j), r = gy(i, j + 1); return fma(T(0.5), r - l, l); }
    __device__ T D(int64_t i, int64_t j) const {
        const T h = H(i, j, 0);
        const T a = hasA ? A(i, j, 0) : T(1);
        const T u = ax(i, j), w = ay(i, j);
        const T vm = sqrt(u * u + w * w);
        return (a * ipow_(h, n + 2) + As * ipow_(h, n)) * ipow_(vm, n - 1);
    }
    __device__ T M(int64_t i, int64_t j) const {
        const T m = mba * (S(i, j) - mbb);
        return m < mbc ? m : mbc;
    }
    // fluxes of the reference kernel (sia.jl:14-15) at vertex (i, j)
    __device__ T qx(int64_t i, int64_t j) const {
        const T Dl = D(i - 1, j), Dr = D(i, j);
        return -fma(T(0.5), Dr - Dl, Dl) * gx(i, j);
    }
    __device__ T qy(int64_t i, int64_t j) const {
        const T Dl = D(i, j - 1), Dr = D(i, j);
        return -fma(T(0.5), Dr - Dl, Dl) * gy(i, j);
    }
    // flux after the Dirichlet batch: zero on boundary vertices 1 and n+1
    __device__ T qxb(int64_t i, int64_t j, int64_t nx) const { return (i <= 1 || i >= nx + 1) ? T(0) : qx(i, j); }
    __device__ T qyb(int64_t i, int64_t j, int64_t ny) const { return (j <= 1 || j >= ny + 1) ? T(0) : qy(i, j); }
};

template <class T>
__device__ __forceinline__ void cell_index(int64_t& i, int64_t& j, int64_t nx, int64_t ny, bool& ok) {
    i = 1 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    j = 1 + blockIdx.y * (int64_t)blockDim.y + threadIdx.y;
    ok = i <= nx && j <= ny;
}

// update_q! (sia.jl:12-16) over vertices 1..n in both dims
template <class T>
__global__ void __launch_bounds__(256) sia_flux_kernel(SiaF<T> s, DF<T> qx, DF<T> qy, int64_t nx, int64_t ny) {
    int64_t i, j;
    bool ok;
    cell_index<T>(i, j, nx, ny, ok);
    if (!ok) return;
    qx(i, j, 0) = s.qx(i, j);
    qy(i, j, 0) = s.qy(i, j);
}

// update_H! (sia.jl:7-10) over cells 1..n
template <class T>
__global__ void __launch_bounds__(256) sia_update_kernel(SiaF<T> s, DF<T> qx, DF<T> qy, DF<T> Ho, int64_t nx,
                                                         int64_t ny, T dt) {
    int64_t i, j;
    bool ok;
    cell_index<T>(i, j, nx, ny, ok);
    if (!ok) return;
    const T dv = (qx(i + 1, j, 0) - qx(i, j, 0)) * s.ix + (qy(i, j + 1, 0) - qy(i, j, 0)) * s.iy;
    Ho(i, j, 0) = jmax0(s.H(i, j, 0) + dt * (-dv + s.M(i, j)));
}

// D at cells 1..n (the lazy FunctionField of sia.jl:46-49 materialised)
template <class T>
__global__ void __launch_bounds__(256) sia_d_kernel(SiaF<T> s, DF<T> D, int64_t nx, int64_t ny) {
    int64_t i, j;
    bool ok;
    cell_index<T>(i, j, nx, ny, ok);
    if (!ok) return;
    D(i, j, 0) = s.D(i, j);
}

// update_q! + q Dirichlet batch + update_H! in one pass (no q storage)
template <class T>
__global__ void __launch_bounds__(256) sia_step_kernel(SiaF<T> s, DF<T> Ho, int64_t nx, int64_t ny, T dt) {
    int64_t i, j;
    bool ok;
    cell_index<T>(i, j, nx, ny, ok);
    if (!ok) return;
    const T dv = (s.qxb(i + 1, j, nx) - s.qxb(i, j, nx)) * s.ix + (s.qyb(i, j + 1, ny) - s.qyb(i, j, ny)) * s.iy;
    Ho(i, j, 0) = jmax0(s.H(i, j, 0) + dt * (-dv + s.M(i, j)));
}

// ---------------------------------------------------------------- adjoint
template <class T>
struct SiaW {   // workspace fields (Center / x-vertex / y-vertex)
    DF<T> mu, Dvx, gdx, Dvy, gdy, ax, ay, HD;
};

template <class T>
__global__ void __launch_bounds__(256) sia_adj1(SiaF<T> s, DF<T> lam, SiaW<T> w, int64_t nx, int64_t ny, T dt) {
    int64_t i, j;
    bool ok;
    cell_index<T>(i, j, nx, ny, ok);
    if (!ok) return;
    const T dv = (s.qxb(i + 1, j, nx) - s.qxb(i, j, nx)) * s.ix + (s.qyb(i, j + 1, ny) - s.qyb(i, j, ny)) * s.iy;
    const T x = s.H(i, j, 0) + dt * (-dv + s.M(i, j));
    w.mu(i, j, 0) = x > T(0) ? lam(i, j, 0) : T(0);
}

// faces: x-vertices (i in 1..nx+1, j in 1..ny) and y-vertices (i in 1..nx, j in 1..ny+1)
template <class T>
__global__ void __launch_bounds__(256) sia_adj2(SiaF<T> s, SiaW<T> w, int64_t nx, int64_t ny, T dt) {
    const int64_t i = 1 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t j = 1 + blockIdx.y * (int64_t)blockDim.y + threadIdx.y;
    if (i <= nx + 1 && j <= ny) {
        T Dv = T(0), gd = T(0);
        if (i >= 2 && i <= nx) {
            const T qb = dt * s.ix * (w.mu(i, j, 0) - w.mu(i - 1, j, 0));
            const T Dl = s.D(i - 1, j), Dr = s.D(i, j);
            Dv = -s.gx(i, j) * qb;
            gd = -fma(T(0.5), Dr - Dl, Dl) * qb;
        }
        w.Dvx(i, j, 0) = Dv;
        w.gdx(i, j, 0) = gd;
    }
    if (i <= nx && j <= ny + 1) {
        T Dv = T(0), gd = T(0);
        if (j >= 2 && j <= ny) {
            const T qb = dt * s.iy * (w.mu(i, j, 0) - w.mu(i, j - 1, 0));
            const T Dl = s.D(i, j - 1), Dr = s.D(i, j);
            Dv = -s.gy(i, j) * qb;
            gd = -fma(T(0.5), Dr - Dl, Dl) * qb;
        }
        w.Dvy(i, j, 0) = Dv;
        w.gdy(i, j, 0) = gd;
    }
}

template <class T>
__global__ void __launch_bounds__(256) sia_adj3(SiaF<T> s, SiaW<T> w, DF<T> gA, int64_t nx, int64_t ny) {
    int64_t i, j;
    bool ok;
    cell_index<T>(i, j, nx, ny, ok);
    if (!ok) return;
    const T Db = T(0.5) * (w.Dvx(i, j, 0) + w.Dvx(i + 1, j, 0)) + T(0.5) * (w.Dvy(i, j, 0) + w.Dvy(i, j + 1, 0));
    const int n = s.n;
    const T h = s.H(i, j, 0);
    const T a = s.hasA ? s.A(i, j, 0) : T(1);
    const T u = s.ax(i, j), v = s.ay(i, j);
    const T vm = sqrt(u * u + v * v);
    const T P = ipow_(vm, n - 1);
    const T C = a * ipow_(h, n + 2) + s.As * ipow_(h, n);
    if (s.hasA) gA(i, j, 0) = gA(i, j, 0) + a * (Db * ipow_(h, n + 2) * P);
    w.HD(i, j, 0) = Db * (T(n + 2) * a * ipow_(h, n + 1) + T(n) * s.As * ipow_(h, n - 1)) * P;
    // d(vm^(n-1))/du = coef * u with coef = (n-1) vm^(n-3) (n >= 3; n = 3 gives 2),
    // 1/vm for n = 2 (0 at vm = 0), 0 for n = 1
    T coef = T(0);
    if (n >= 3) coef = T(n - 1) * ipow_(vm, n - 3);
    else if (n == 2 && vm > T(0)) coef = T(1) / vm;
    const T Pb = Db * C;
    w.ax(i, j, 0) = Pb * coef * u;
    w.ay(i, j, 0) = Pb * coef * v;
}

template <class T>
__global__ void __launch_bounds__(256) sia_adj4(SiaW<T> w, int64_t nx, int64_t ny) {
    const int64_t i = 1 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t j = 1 + blockIdx.y * (int64_t)blockDim.y + threadIdx.y;
    if (i <= nx + 1 && j <= ny) {
        T g = w.gdx(i, j, 0);
        if (i - 1 >= 1) g = g + T(0.5) * w.ax(i - 1, j, 0);
        if (i <= nx) g = g + T(0.5) * w.ax(i, j, 0);
        w.gdx(i, j, 0) = g;
    }
    if (i <= nx && j <= ny + 1) {
        T g = w.gdy(i, j, 0);
        if (j - 1 >= 1) g = g + T(0.5) * w.ay(i, j - 1, 0);
        if (j <= ny) g = g + T(0.5) * w.ay(i, j, 0);
        w.gdy(i, j, 0) = g;
    }
}

template <class T>
__global__ void __launch_bounds__(256) sia_adj5(SiaF<T> s, SiaW<T> w, DF<T> lo, int64_t nx, int64_t ny, T dt) {
    int64_t i, j;
    bool ok;
    cell_index<T>(i, j, nx, ny, ok);
    if (!ok) return;
    auto Sb = [&](int64_t a, int64_t b) -> T {
        // Sbar of cell (a, b): gx(v) = (S_v - S_{v-1}) iΔx, faces v in 1..nx+1 (zero outside)
        T r = T(0);
        if (a >= 1 && a <= nx + 1) r = r + s.ix * w.gdx(a, b, 0);
        if (a + 1 >= 1 && a + 1 <= nx + 1) r = r - s.ix * w.gdx(a + 1, b, 0);
        if (b >= 1 && b <= ny + 1) r = r + s.iy * w.gdy(a, b, 0);
        if (b + 1 >= 1 && b + 1 <= ny + 1) r = r - s.iy * w.gdy(a, b + 1, 0);
        return r;
    };
    const T mu = w.mu(i, j, 0);
    T l = mu + w.HD(i, j, 0) + Sb(i, j);
    const T m = s.mba * (s.S(i, j) - s.mbb);
    if (m < s.mbc) l = l + dt * mu * s.mba;
    // halo cells feed through the Neumann copy H_0 = H_1, H_{n+1} = H_n: the halo
    // S enters only the boundary-face gradients, Sbar_0 = -iΔx gbar_1 and
    // Sbar_{n+1} = iΔx gbar_{n+1}
    if (i == 1) l = l + (-s.ix * w.gdx(1, j, 0));
    if (i == nx) l = l + s.ix * w.gdx(nx + 1, j, 0);
    if (j == 1) l = l + (-s.iy * w.gdy(i, 1, 0));
    if (j == ny) l = l + s.iy * w.gdy(i, ny + 1, 0);
    lo(i, j, 0) = l;
}

// ---------------------------------------------------------------- one-pass forms
// The forward steps and the adjoint step as one launch each.  A block is a
// region of 64 columns (one lane each) by NW x R rows: wave w holds rows
// w R .. w R + R - 1 of its column in registers.  x neighbours come by DPP
// lane shifts, y neighbours from the thread's own rows, and only a wave's
// first and last rows pass through LDS.  Every value of a cell is formed once
// per region and its row index is wave-uniform, so the row conditions and
// addresses are scalar.  The ring a stage cannot form right (2 cells per
// forward step, 1 more for the next state's D, 3 to 4 for the adjoint) is
// work that other blocks own.  The arithmetic of every value is the one of the
// per-point kernels above, so the results are bitwise equal to them.
template <int NW, int R>
struct SiaCol {
    static constexpr int NR = NW * R;
    using Edge = double[2][NW][64];   // first and last row of every wave
    int lane, w, i, jb;               // column, first row
    uint32_t ic;                      // column clamped into the stored 0..nx+1
    int rx, ry;                       // columns and rows around the owned ones
    int nx, ny;
    __device__ __forceinline__ SiaCol(int bx, int by, int rx_, int ry_, int64_t nx_, int64_t ny_) : rx(rx_), ry(ry_) {
        lane = threadIdx.x;
        w = __builtin_amdgcn_readfirstlane(threadIdx.y);
        nx = (int)nx_;
        ny = (int)ny_;
        i = 1 + bx * (64 - 2 * rx) - rx + lane;
        jb = 1 + by * (NR - 2 * ry) - ry + w * R;
        ic = (uint32_t)min(max(i, 0), nx + 1);
    }
    __device__ __forceinline__ int j(int r) const { return jb + r; }
    __device__ __forceinline__ int jc(int r) const { return min(max(jb + r, 0), ny + 1); }
    __device__ __forceinline__ bool inside(int r) const { return i >= 1 && i <= nx && j(r) >= 1 && j(r) <= ny; }
    __device__ __forceinline__ bool own(int r) const {
        const int y = w * R + r;
        return lane >= rx && lane < 64 - rx && y >= ry && y < NR - ry && inside(r);
    }
    __device__ __forceinline__ double ld(const DF<double>& f, int r) const {
        return (f.p + (int64_t)jc(r) * f.sy)[ic];
    }
    __device__ __forceinline__ double& at(const DF<double>& f, int r) const {   // owned cells only
        return (f.p + (int64_t)j(r) * f.sy)[ic];
    }
    __device__ __forceinline__ void put(Edge& e, const double* v) const {
        e[0][w][lane] = v[0];
        e[1][w][lane] = v[R - 1];
    }
    // the rows below the first and above the last (a row of the block's rim
    // gets its own value: it reaches ring cells only)
    __device__ __forceinline__ void get(const Edge& e, const double* v, double& lo, double& hi) const {
        lo = w > 0 ? e[1][w - 1][lane] : v[0];
        hi = w + 1 < NW ? e[0][w + 1][lane] : v[R - 1];
    }
};

template <class T>
struct SiaStep {   // forward steps H -> Ho, H's Neumann batch included
    SiaF<T> s;
    DF<T> Ho;
    int wd;        // also store D(H) of the cells into Dout (for a later adjoint step at H)
    DF<T> Dout;
};
struct SiaMid {    // two kept steps: the state between them and its D
    DF<double> H, D;
};

// Steps a launch may take: their time steps travel in its argument.
constexpr int kSiaSteps = 8;
struct SiaDts {
    double dt[kSiaSteps];
    int n;
};

// The time step from max(D) on the device (sia.jl:76-78): Δt =
// min(h2 / max(D) / 4.1, dt_max), with max(D) as the bits of its magnitude in
// *dmax.  Every block forms the same Δt; the first stores it.  next (or
// NULL) receives the new state's max(D) the same way.
struct SiaRule {
    const unsigned long long* dmax;
    unsigned long long* next;
    double h2, dt_max;
    double* dt_out;
};
__device__ __forceinline__ double sia_rule_dt(const SiaRule& r) {
    const double m = __longlong_as_double((long long)*r.dmax);
    const double d = m > 0.0 ? r.h2 / m / 4.1 : __longlong_as_double(0x7ff0000000000000ll);
    return r.dt_max < d ? r.dt_max : d;
}
__device__ __forceinline__ unsigned long long sia_mag(double d) {
    return (unsigned long long)__double_as_longlong(d) & 0x7fffffffffffffffull;
}

// One column's rows of H with B and A, and the surface gradients and D of the
// current H.  H's rows -1 and R (and the ghost cells) are kept with it.
template <int NW, int R>
struct SiaRows {
    using Col = SiaCol<NW, R>;
    double h[R + 2], b[R + 2], a[R];   // [r + 1]: row r
    double gx[R], gy[R + 1], u[R], v[R];
    __device__ __forceinline__ void load_h(const DF<double>& H, const Col& c) {
#pragma unroll
        for (int r = -1; r <= R; ++r) h[r + 1] = c.ld(H, r);
    }
    __device__ __forceinline__ void load(const SiaF<double>& s, const Col& c) {
#pragma unroll
        for (int r = -1; r <= R; ++r) {
            h[r + 1] = c.ld(s.H, r);
            b[r + 1] = c.ld(s.B, r);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = s.hasA ? c.ld(s.A, r) : 1.0;
    }
    __device__ __forceinline__ double S(int r) const { return b[r + 1] + h[r + 1]; }
    // after a step: the neighbouring waves' rows, then the Neumann(0) ghosts
    // (a ghost copies the adjacent cell: fma(Δ, -0, f) == f; corners are not read)
    __device__ __forceinline__ void refresh(const Col& c, typename Col::Edge& e) {
        c.put(e, h + 1);
        __syncthreads();
        c.get(e, h + 1, h[0], h[R + 1]);
#pragma unroll
        for (int r = -1; r < R; ++r)
            if (c.j(r) == 0) h[r + 1] = h[r + 2];
#pragma unroll
        for (int r = R; r >= 0; --r)
            if (c.j(r) == c.ny + 1) h[r + 1] = h[r];
        const int i0 = c.i - c.lane;
        if (i0 <= 0 || i0 + 63 > c.nx) {   // block-uniform
#pragma unroll
            for (int r = -1; r <= R; ++r) {
                const double up = xp1(h[r + 1]), dn = xm1(h[r + 1]);
                h[r + 1] = c.i == 0 ? up : c.i == c.nx + 1 ? dn : h[r + 1];
            }
        }
    }
    __device__ __forceinline__ void gradients(const SiaF<double>& s) {
#pragma unroll
        for (int r = 0; r <= R; ++r) gy[r] = (S(r) - S(r - 1)) * s.iy;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            gx[r] = (S(r) - xm1(S(r))) * s.ix;
            const double gr = xp1(gx[r]);
            u[r] = fma(0.5, gr - gx[r], gx[r]);
            v[r] = fma(0.5, gy[r + 1] - gy[r], gy[r]);
        }
    }
    __device__ __forceinline__ double D(const SiaF<double>& s, int r) const {
        const double vm = sqrt(u[r] * u[r] + v[r] * v[r]);
        return (a[r] * ipow_(h[r + 1], s.n + 2) + s.As * ipow_(h[r + 1], s.n)) * ipow_(vm, s.n - 1);
    }
    // H - Δt(divg q - M) of row r before max(., 0), from D's lerps on the faces
    __device__ __forceinline__ void update(const SiaF<double>& s, const Col& c, const double* fx, const double* fy,
                                           double dt, double* x) const {
        double qy[R + 1];
#pragma unroll
        for (int r = 0; r <= R; ++r) qy[r] = c.j(r) <= 1 || c.j(r) >= c.ny + 1 ? 0.0 : -fy[r] * gy[r];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const double q = c.i <= 1 || c.i >= c.nx + 1 ? 0.0 : -fx[r] * gx[r];
            const double dv = (xp1(q) - q) * s.ix + (qy[r + 1] - qy[r]) * s.iy;
            const double m = s.mba * (S(r) - s.mbb);
            x[r] = h[r + 1] + dt * (-dv + (m < s.mbc ? m : s.mbc));
        }
    }
};

// D's lerps on a column's x faces (left of each row's cell) and y faces
template <int NW, int R>
__device__ __forceinline__ void sia_face_d(const double* D, double lo, double hi, double* fx, double* fy) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const double l = xm1(D[r]);
        fx[r] = fma(0.5, D[r] - l, l);
    }
#pragma unroll
    for (int r = 0; r <= R; ++r) {
        const double l = r > 0 ? D[r - 1] : lo, g = r < R ? D[r] : hi;
        fy[r] = fma(0.5, g - l, l);
    }
}

// A state's owned cells and their Neumann(0) ghosts, dims y then x
// (batch.jl:20-29): ghosts copy the adjacent cell, corners the diagonal cell.
template <int NW, int R>
__device__ __forceinline__ void sia_store(const SiaCol<NW, R>& c, const DF<double>& f, const double* h) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (!c.own(r)) continue;
        double* row = &c.at(f, r);
        row[0] = h[r];
        const bool x0 = c.i == 1, x1 = c.i == c.nx;
        if (x0) row[-1] = h[r];
        if (x1) row[1] = h[r];
        if (c.j(r) == 1) {
            double* g = row - f.sy;
            g[0] = h[r];
            if (x0) g[-1] = h[r];
            if (x1) g[1] = h[r];
        }
        if (c.j(r) == c.ny) {
            double* g = row + f.sy;
            g[0] = h[r];
            if (x0) g[-1] = h[r];
            if (x1) g[1] = h[r];
        }
    }
}

// n forward steps on the region (a ring of 2 n); the owned cells' final H and
// its ghosts are stored; with KEEP (n at most 2) every state is.  With MAXD (a ring of 2 n + 1) the magnitude bits of
// the new state's largest owned D come back.
template <int NW, int R, bool MAXD, bool KEEP = false>
__device__ __forceinline__ unsigned long long sia_step_cols(const SiaStep<double>& p, const SiaMid& mid,
                                                            const SiaCol<NW, R>& c,
                                                            const double* dts, int n, double (*ldsH)[NW][64],
                                                            double (*ldsD)[NW][64]) {
    using Col = SiaCol<NW, R>;
    const SiaF<double>& s = p.s;
    typename Col::Edge& eH = *reinterpret_cast<typename Col::Edge*>(ldsH);
    typename Col::Edge& eD = *reinterpret_cast<typename Col::Edge*>(ldsD);
    SiaRows<NW, R> k;
    k.load(s, c);
    // (two kept steps are written out, so that no view is chosen at run time:
    // that puts the kernel's arguments in scratch)
    auto one = [&](int q, auto second) {
        if (q > 0) k.refresh(c, eH);
        k.gradients(s);
        double D[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            D[r] = c.inside(r) ? k.D(s, r) : 0.0;
            if (p.wd && c.own(r)) {
                if constexpr (decltype(second)::value) c.at(mid.D, r) = D[r];
                else c.at(p.Dout, r) = D[r];
            }
        }
        c.put(eD, D);
        __syncthreads();
        double lo, hi, fx[R], fy[R + 1], x[R];
        c.get(eD, D, lo, hi);
        sia_face_d<NW, R>(D, lo, hi, fx, fy);
        k.update(s, c, fx, fy, dts[q], x);
#pragma unroll
        for (int r = 0; r < R; ++r) k.h[r + 1] = c.inside(r) ? jmax0(x[r]) : k.h[r + 1];
    };
    if constexpr (MAXD) {
        one(0, std::false_type{});
    } else if constexpr (KEEP) {
        one(0, std::false_type{});
        if (n > 1) {
            sia_store(c, mid.H, k.h + 1);
            one(1, std::true_type{});
        }
    } else {
#pragma unroll 1
        for (int q = 0; q < n; ++q) one(q, std::false_type{});
    }
    sia_store(c, p.Ho, k.h + 1);
    unsigned long long m = 0;
    if constexpr (MAXD) {
        k.refresh(c, eH);
        k.gradients(s);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const unsigned long long d = c.own(r) ? sia_mag(k.D(s, r)) : 0ull;
            m = d > m ? d : m;
        }
    }
    return m;
}

template <class T>
struct SiaAdj {    // one adjoint step at state s.H, or two (then at H2): lam -> lo, gA += dJ/dlog A
    SiaF<T> s;
    DF<T> lam, lo, gA;
    T dt;
    int rd;        // D(s.H) read from Din (stored by the forward step at s.H) instead of evaluated
    DF<T> Din;
    int n;         // steps
    DF<T> H2, D2;  // the second step's state and its D (always stored)
    T dt2;
};

// lam' reaches D of the cells 3 away, and an evaluated D the surface of the
// cell beside that one: the rows -1 and R a wave holds cover it in y, one
// more lane in x.
constexpr int kAdjRing = 3;
__host__ __device__ constexpr int sia_adj_ring(int rd, int n) { return kAdjRing * n + (rd ? 0 : 1); }

// Between two steps lam stays in registers, exact 3 cells further in (a ring
// of 6 for both); B, A and the gradient's sum are read and written once.
template <int NW, int R, bool TWO>
__device__ __forceinline__ void sia_adj_cols(const SiaAdj<double>& p, const SiaCol<NW, R>& c, double (*lds0)[NW][64],
                                             double (*lds1)[NW][64]) {
    using Col = SiaCol<NW, R>;
    typename Col::Edge& e0 = *reinterpret_cast<typename Col::Edge*>(lds0);
    typename Col::Edge& e1 = *reinterpret_cast<typename Col::Edge*>(lds1);
    const SiaF<double>& s = p.s;
    const int nx = c.nx, ny = c.ny;
    SiaRows<NW, R> k;
    k.load(s, c);
    double lam[R], gA[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        lam[r] = c.ld(p.lam, r);
        gA[r] = s.hasA ? c.ld(p.gA, r) : 0.0;
    }
    auto one = [&](const DF<double>& Din, double dt, bool rd) {
        double D[R], Dlo, Dhi, fx[R], fy[R + 1];
        if (rd) {   // D of the wave's rows and the two beside them, stored by the forward step at this state
            const double lo = c.ld(Din, -1), hi = c.ld(Din, R);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const double d = c.ld(Din, r);
                D[r] = c.inside(r) ? d : 0.0;
            }
            Dlo = c.inside(-1) ? lo : 0.0;
            Dhi = c.inside(R) ? hi : 0.0;
            k.gradients(s);
        } else {
            k.gradients(s);
#pragma unroll
            for (int r = 0; r < R; ++r) D[r] = c.inside(r) ? k.D(s, r) : 0.0;
            c.put(e1, D);
            __syncthreads();
            c.get(e1, D, Dlo, Dhi);
        }
        sia_face_d<NW, R>(D, Dlo, Dhi, fx, fy);
        // A1: mu
        double mu[R], mlo, mhi;
        {
            double x[R];
            k.update(s, c, fx, fy, dt, x);
#pragma unroll
            for (int r = 0; r < R; ++r) mu[r] = c.inside(r) && x[r] > 0.0 ? lam[r] : 0.0;
        }
        c.put(e0, mu);
        __syncthreads();
        c.get(e0, mu, mlo, mhi);
        // A2 + A3: qbar on the faces, Dbar, abar; HD and the log A gradient
        const bool fxin = c.i >= 2 && c.i <= nx;
        double qbx[R], qby[R + 1], Dvy[R + 1], abx[R], aby[R], HD[R];
#pragma unroll
        for (int r = 0; r <= R; ++r) {
            qby[r] = dt * s.iy * ((r < R ? mu[r] : mhi) - (r > 0 ? mu[r - 1] : mlo));
            Dvy[r] = c.j(r) < 2 || c.j(r) > ny ? 0.0 : -k.gy[r] * qby[r];
        }
        const int n = s.n;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            qbx[r] = dt * s.ix * (mu[r] - xm1(mu[r]));
            const double Dvx = fxin ? -k.gx[r] * qbx[r] : 0.0;
            const double Db = 0.5 * (Dvx + xp1(Dvx)) + 0.5 * (Dvy[r] + Dvy[r + 1]);
            const double h = k.h[r + 1], av = k.a[r], u = k.u[r], v = k.v[r];
            const double vm = sqrt(u * u + v * v);
            const double P = ipow_(vm, n - 1);
            const double Cc = av * ipow_(h, n + 2) + s.As * ipow_(h, n);
            if (s.hasA) gA[r] = gA[r] + av * (Db * ipow_(h, n + 2) * P);
            HD[r] = Db * (double(n + 2) * av * ipow_(h, n + 1) + double(n) * s.As * ipow_(h, n - 1)) * P;
            double coef = 0.0;
            if (n >= 3) coef = double(n - 1) * ipow_(vm, n - 3);
            else if (n == 2 && vm > 0.0) coef = 1.0 / vm;
            const double Pb = Db * Cc;
            const bool in = c.inside(r);
            abx[r] = in ? Pb * coef * u : 0.0;
            aby[r] = in ? Pb * coef * v : 0.0;
        }
        double alo, ahi;
        c.put(e1, aby);
        __syncthreads();
        c.get(e1, aby, alo, ahi);
        // A4 + A5: gbar on the faces, then lam'
        double gby[R + 1];
#pragma unroll
        for (int r = 0; r <= R; ++r) {
            const int f = c.j(r);
            double g = f >= 2 && f <= ny ? -fy[r] * qby[r] : 0.0;
            if (f - 1 >= 1) g = g + 0.5 * (r > 0 ? aby[r - 1] : alo);
            if (f <= ny) g = g + 0.5 * (r < R ? aby[r] : ahi);
            gby[r] = g;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            double gx0 = fxin ? -fx[r] * qbx[r] : 0.0;
            const double al = xm1(abx[r]);
            gx0 = c.i - 1 >= 1 ? gx0 + 0.5 * al : gx0;
            gx0 = c.i <= nx ? gx0 + 0.5 * abx[r] : gx0;
            const double gx1 = xp1(gx0), gy0 = gby[r], gy1 = gby[r + 1];
            double t = 0.0;
            t = t + s.ix * gx0;
            t = t - s.ix * gx1;
            t = t + s.iy * gy0;
            t = t - s.iy * gy1;
            double l = mu[r] + HD[r] + t;
            const double m = s.mba * (k.S(r) - s.mbb);
            if (m < s.mbc) l = l + dt * mu[r] * s.mba;
            if (c.i == 1) l = l + (-s.ix * gx0);
            if (c.i == nx) l = l + s.ix * gx1;
            if (c.j(r) == 1) l = l + (-s.iy * gy0);
            if (c.j(r) == ny) l = l + s.iy * gy1;
            lam[r] = l;
        }
    };
    one(p.Din, p.dt, p.rd);
    if constexpr (TWO) {
        if (p.n > 1) {
            k.load_h(p.H2, c);
            one(p.D2, p.dt2, true);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (!c.own(r)) continue;
        c.at(p.lo, r) = lam[r];
        if (s.hasA) c.at(p.gA, r) = gA[r];
    }
}

// NP > 0: the Glen exponent as a compile-time constant (it must equal the
// run-time one), so that every power's product loop unrolls; the products
// and their order are the same as with NP = 0.
template <int NP, int NW, int R>
__global__ void __launch_bounds__(NW * 64) sia_steps_kernel(SiaStep<double> f, SiaDts d, int ntx, int64_t nx,
                                                            int64_t ny) {
    __shared__ double lds[2][2][NW][64];
    if constexpr (NP > 0) f.s.n = NP;
    const SiaCol<NW, R> c(blockIdx.x % ntx, blockIdx.x / ntx, 2 * d.n, 2 * d.n, nx, ny);
    sia_step_cols<NW, R, false>(f, SiaMid{}, c, d.dt, d.n, lds[0], lds[1]);
}

// The step whose Δt follows from its state's max(D), and the next state's.
template <int NP, int NW, int R, bool MAXD>
__global__ void __launch_bounds__(NW * 64) sia_rule_kernel(SiaStep<double> f, SiaRule rule, int ntx, int64_t nx,
                                                           int64_t ny) {
    __shared__ double lds[2][2][NW][64];
    __shared__ unsigned long long part[NW];
    if constexpr (NP > 0) f.s.n = NP;
    const double dt = sia_rule_dt(rule);
    if (blockIdx.x == 0 && threadIdx.x == 0 && threadIdx.y == 0) *rule.dt_out = dt;
    constexpr int ring = MAXD ? 3 : 2;
    const SiaCol<NW, R> c(blockIdx.x % ntx, blockIdx.x / ntx, ring, ring, nx, ny);
    unsigned long long m = sia_step_cols<NW, R, MAXD>(f, SiaMid{}, c, &dt, 1, lds[0], lds[1]);
    if constexpr (MAXD) {
        for (int o = 32; o > 0; o >>= 1) {
            const unsigned long long q = __shfl_xor(m, o, 64);
            m = q > m ? q : m;
        }
        if (threadIdx.x == 0) part[threadIdx.y] = m;
        __syncthreads();
        if (threadIdx.x == 0 && threadIdx.y == 0) {
            for (int q = 1; q < NW; ++q) m = part[q] > m ? part[q] : m;
            if (m > __hip_atomic_load(rule.next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(rule.next, m);
        }
    }
}

// D at cells 1..n and the maximum of its magnitude (bits; NaN above infinity)
template <class T, int NP>
__global__ void __launch_bounds__(256) sia_d_max_kernel(SiaF<T> s, DF<T> D, int64_t nx, int64_t ny,
                                                        unsigned long long* dmax) {
    __shared__ unsigned long long part[4];
    if constexpr (NP > 0) s.n = NP;
    int64_t i, j;
    bool ok;
    cell_index<T>(i, j, nx, ny, ok);
    unsigned long long m = 0;
    if (ok) {
        const T d = s.D(i, j);
        D(i, j, 0) = d;
        m = sia_mag((double)d);
    }
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long q = __shfl_xor(m, o, 64);
        m = q > m ? q : m;
    }
    if (threadIdx.x == 0) part[threadIdx.y] = m;
    __syncthreads();
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        for (int q = 1; q < 4; ++q) m = part[q] > m ? part[q] : m;
        if (m > __hip_atomic_load(dmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(dmax, m);
    }
}

// Blocks 0 .. na - 1: adjoint regions; the rest: as many independent forward
// steps (the recompute of the previous checkpoint segment rides along).
template <int NP, int NW, int RA, int RF, bool TWO>
__global__ void __launch_bounds__(NW * 64) sia_adj_kernel(SiaAdj<double> a, SiaStep<double> f, SiaMid mid, SiaDts fd, int na,
                                                          int ntxa, int ntxf, int64_t nx, int64_t ny) {
    __shared__ double lds[2][2][NW][64];
    if constexpr (NP > 0) {
        a.s.n = NP;
        f.s.n = NP;
    }
    const int bid = blockIdx.x;
    if (bid < na) {
        const SiaCol<NW, RA> c(bid % ntxa, bid / ntxa, sia_adj_ring(a.rd, a.n), kAdjRing * a.n, nx, ny);
        sia_adj_cols<NW, RA, TWO>(a, c, lds[0], lds[1]);
    } else {
        const SiaCol<NW, RF> c((bid - na) % ntxf, (bid - na) / ntxf, 2 * fd.n, 2 * fd.n, nx, ny);
        sia_step_cols<NW, RF, false, TWO>(f, mid, c, fd.dt, fd.n, lds[0], lds[1]);
    }
}

// Shapes, each the best measured of 4..16 waves by 1..6 rows.  A launch's floor
// is its serial chain (about 4.5 us a forward step, 5.4 us an adjoint step for
// one region alone), so forward steps go several to a launch: up to five while
// the regions' own 44 x 28 cells cover the grid in one round of the CUs, else
// three, where the ring's work counts (300 steps of 512^2 within the gradient,
// us a step: 5.1 singly, 4.3 in twos, 3.8 in threes, 3.1 in fives; gradient 4319
// -> 4098 from three to five, 64x51 935 -> 872, 250x177 1072 -> 1006), and adjoint steps
// two (the gradient with 1 -> 2 a launch, us: 64x51, 100 steps 1067 -> 928 with
// 8 waves of 2 rows, 1060 with 16; 250x177 1143 -> 1062 with 12 of 2, 1205 with
// 8; 512^2, 300 steps 4640 -> 4335 with 16 of 3, 4520 with 12 of 4, 6010 with
// 16 of 4).  Forward regions of 32 rows while they all fit the CUs at once,
// else 48 (250x177: 1.14 ms for the gradient of 100 steps with 32 rows, 1.20
// with 48; 512^2: 4.86 and 4.68 for 300).  A single adjoint step's regions are
// 16 rows with 24 for the step riding along: 3 blocks a CU hold them all at
// 512^2 (with 16 and 16 rows a second round starts: 5.04).
// A single forward step (every state kept, or recomputed for the adjoint) has a
// ring of 2, so smaller regions waste little and a block's waves wait for
// fewer others: 4 waves of 2 rows up to two blocks a CU, 8 of 2 up to one, then
// the shapes of several steps.  40 steps with every state kept, n = 3 / 8, us,
// a 256-thread tile a block -> 16 waves -> now: 64x64 162 / 193 -> 197 / 254 ->
// 155 / 190, 250x230 162 / 198 -> 203 / 254 -> 157 / 189, 400x390 185 / 222 -> 203 /
// 251 -> 167 / 197; 512x512 (unchanged) 211 / 249 -> 203 / 250.  (4 x 3 and 6 x 2:
// 4-15% more up to 250x230, 8 x 1: 5% more at n = 3.)
constexpr int kSiaMax = 5, kSiaMany = 3;          // forward steps per launch: one round, more
constexpr int kNWF = 16, kRF1 = 2, kRF2 = 3;      // forward: waves, rows per wave
constexpr int kNWS = 4, kNWT = 8, kRS = 2;        // a single forward step: waves up to two blocks a CU, up to one, rows
constexpr int kNWA = 8, kRA = 2, kRR = 3;         // adjoint, and the steps riding along
constexpr int kNWD = 8, kRD = 2;                  // the adaptive step (us for 24: 250x230 203, 400x390 243; 16 x 1: 206, 260)
static_assert(kSiaMax <= kSiaSteps && kNWF * kRF1 > 4 * kSiaMax && 64 > 4 * kSiaMax && kNWA * kRA > 2 * kAdjRing &&
                  kNWA * kRR > 4 && kNWD * kRD > 6 && kNWS * kRS > 4,
              "a region owns at least one row and column");

static int sia_regions(int64_t nx, int64_t ny, int rx, int ry, int rows, int* ntx) {
    const int64_t w = 64 - 2 * rx, h = rows - 2 * ry;
    *ntx = (int)((nx + w - 1) / w);
    return (int)(*ntx * ((ny + h - 1) / h));
}

// n = 3 (Glen's law as sia.jl uses it) takes the unrolled kernels
template <int NW, int R>
static void launch_steps_r(hipStream_t st, const SiaStep<double>& f, const SiaDts& d, int64_t nx, int64_t ny) {
    int ntx;
    const int nb = sia_regions(nx, ny, 2 * d.n, 2 * d.n, NW * R, &ntx);
    const dim3 blk(64, NW);
    if (f.s.n == 3) hipLaunchKernelGGL((sia_steps_kernel<3, NW, R>), dim3(nb), blk, 0, st, f, d, ntx, nx, ny);
    else hipLaunchKernelGGL((sia_steps_kernel<0, NW, R>), dim3(nb), blk, 0, st, f, d, ntx, nx, ny);
}

static void launch_steps(hipStream_t st, const SiaStep<double>& f, const double* dts, int n, int64_t nx, int64_t ny) {
    SiaDts d{};
    d.n = n;
    for (int q = 0; q < n; ++q) d.dt[q] = dts[q];
    auto fits = [&](int rows, int blocks) {
        int ntx;
        return sia_regions(nx, ny, 2 * n, 2 * n, rows, &ntx) <= blocks * cu_count();
    };
    if (n == 1 && fits(kNWS * kRS, 2)) launch_steps_r<kNWS, kRS>(st, f, d, nx, ny);
    else if (n == 1 && fits(kNWT * kRS, 1)) launch_steps_r<kNWT, kRS>(st, f, d, nx, ny);
    else if (fits(kNWF * kRF1, 1)) launch_steps_r<kNWF, kRF1>(st, f, d, nx, ny);
    else launch_steps_r<kNWF, kRF2>(st, f, d, nx, ny);
}

template <bool MAXD>
static void launch_rule(hipStream_t st, const SiaStep<double>& f, const SiaRule& r, int64_t nx, int64_t ny) {
    constexpr int NW = kNWD, R = kRD;
    int ntx;
    const int nb = sia_regions(nx, ny, MAXD ? 3 : 2, MAXD ? 3 : 2, NW * R, &ntx);
    const dim3 blk(64, NW);
    if (f.s.n == 3) hipLaunchKernelGGL((sia_rule_kernel<3, NW, R, MAXD>), dim3(nb), blk, 0, st, f, r, ntx, nx, ny);
    else hipLaunchKernelGGL((sia_rule_kernel<0, NW, R, MAXD>), dim3(nb), blk, 0, st, f, r, ntx, nx, ny);
}

template <int NW, int RA, int RF, bool TWO>
static void launch_adj_r(hipStream_t st, const SiaAdj<double>& a, const SiaStep<double>& f, const SiaMid& mid,
                         const SiaDts& fd, int64_t nx, int64_t ny) {
    int ntxa, ntxf = 1;
    const int na = sia_regions(nx, ny, sia_adj_ring(a.rd, a.n), kAdjRing * a.n, NW * RA, &ntxa);
    const int nf = fd.n ? sia_regions(nx, ny, 2 * fd.n, 2 * fd.n, NW * RF, &ntxf) : 0;
    const dim3 blk(64, NW), grd(na + nf);
    if (a.s.n == 3) hipLaunchKernelGGL((sia_adj_kernel<3, NW, RA, RF, TWO>), grd, blk, 0, st, a, f, mid, fd, na, ntxa, ntxf, nx, ny);
    else hipLaunchKernelGGL((sia_adj_kernel<0, NW, RA, RF, TWO>), grd, blk, 0, st, a, f, mid, fd, na, ntxa, ntxf, nx, ny);
}

// fd.n forward steps (0: none) ride along with a.n adjoint steps.  Two steps
// take the first shape whose blocks all find a CU of their own (the flatter,
// the shorter a block's chain), the largest regions beyond.
static void launch_adj(hipStream_t st, const SiaAdj<double>& a, const SiaStep<double>& f, const SiaMid& mid,
                       const SiaDts& fd, int64_t nx, int64_t ny) {
    if (a.n == 1 && fd.n <= 1) return launch_adj_r<kNWA, kRA, kRR, false>(st, a, f, mid, fd, nx, ny);
    auto fits = [&](int nw, int r) {
        int t;
        return sia_regions(nx, ny, 2 * kAdjRing, 2 * kAdjRing, nw * r, &t) + sia_regions(nx, ny, 4, 4, nw * (r + 1), &t) <=
               cu_count();
    };
    if (fits(8, 2)) launch_adj_r<8, 2, 3, true>(st, a, f, mid, fd, nx, ny);
    else if (fits(12, 2)) launch_adj_r<12, 2, 3, true>(st, a, f, mid, fd, nx, ny);
    else launch_adj_r<16, 3, 4, true>(st, a, f, mid, fd, nx, ny);
}

template <class T>
static SiaF<T> make_sia(const chmy_grid_t* g, const chmy_field_t* H, const chmy_field_t* B, const chmy_field_t* A,
                        const SiaPar& p) {
    SiaF<T> s;
    s.H = view<T>(*H);
    s.B = view<T>(*B);
    s.A = A ? view<T>(*A) : s.H;
    s.hasA = A != nullptr;
    s.ix = T(g->inv_spacing[0]);
    s.iy = T(g->inv_spacing[1]);
    s.As = T(p.As);
    s.mba = T(p.mb_a);
    s.mbb = T(p.mb_b);
    s.mbc = T(p.mb_c);
    s.n = p.npow;
    return s;
}

static int sia_check(const chmy_grid_t* g, const chmy_field_t* H, const chmy_field_t* B, const chmy_field_t* A,
                     int npow) {
    CHMY_TRY(check_grid(g));
    if (g->nd != 2) return set_error(CHMY_E_ARG, "SIA kernels are 2D");
    if (npow < 1 || npow > 12) return set_error(CHMY_E_ARG, "Glen exponent n=%d not in 1..12", npow);
    CHMY_TRY(check_center(g, H, "H", CHMY_F64));
    CHMY_TRY(check_center(g, B, "B", CHMY_F64));
    if (A) CHMY_TRY(check_center(g, A, "A", CHMY_F64));
    // D at cell 0 reads S at -1: halo 1 covers logical -1..n+2
    return 0;
}

static SiaStep<double> sia_stepper(const chmy_grid_t* g, const chmy_field_t* H, const chmy_field_t* Ho,
                                   const chmy_field_t* B, const chmy_field_t* A, const SiaPar& p) {
    SiaStep<double> f;
    f.s = make_sia<double>(g, H, B, A, p);
    f.Ho = view<double>(*Ho);
    f.wd = 0;
    f.Dout = f.Ho;
    return f;
}

static SiaAdj<double> sia_adjointer(const chmy_grid_t* g, const chmy_field_t* H, const chmy_field_t* lam,
                                    const chmy_field_t* lo, const chmy_field_t* gA, const chmy_field_t* B,
                                    const chmy_field_t* A, const SiaPar& p, double dt) {
    SiaAdj<double> a;
    a.s = make_sia<double>(g, H, B, A, p);
    a.lam = view<double>(*lam);
    a.lo = view<double>(*lo);
    a.gA = gA ? view<double>(*gA) : a.lo;
    a.dt = dt;
    a.rd = 0;
    a.n = 1;
    a.Din = a.H2 = a.D2 = a.lo;
    a.dt2 = 0.0;
    return a;
}

// Steps the launch that starts at state q takes: states between its first and
// its last are not stored, so each must have a later state in the same
// storage (looked for over the next 8), and the output must not touch the
// input (a block reads cells that its neighbours own).
static int sia_run_length(const chmy_field_t* st, int nstates, int q, int longest) {
    const auto same = [](const chmy_field_t& a, const chmy_field_t& b) {
        return a.data == b.data && a.halo[0] == b.halo[0] && a.halo[1] == b.halo[1];
    };
    const auto apart = [](const chmy_field_t& a, const chmy_field_t& b) {
        const char *pa = static_cast<const char*>(a.data), *pb = static_cast<const char*>(b.data);
        return pa + pad_of(a, 0) * pad_of(a, 1) * 8 <= pb || pb + pad_of(b, 0) * pad_of(b, 1) * 8 <= pa;
    };
    const auto replaced = [&](int m) {
        for (int t = m + 1; t < nstates && t <= m + 8; ++t)
            if (same(st[t], st[m])) return true;
        return false;
    };
    int most = 1;
    while (most < longest && q + most + 1 < nstates && replaced(q + most)) ++most;
    for (int n = most; n > 1; --n)
        if (apart(st[q], st[q + n])) return n;
    return 1;
}

static int sia_check_states(const chmy_grid_t* g, const chmy_field_t* st, int n, const char* what) {
    if (!st) return set_error(CHMY_E_ARG, "%s is NULL", what);
    for (int q = 0; q < n; ++q) CHMY_TRY(check_center(g, &st[q], what, CHMY_F64));
    return 0;
}

// Validation shared by both reverse-sweep entry points.
static int sia_reverse_check(const chmy_grid_t* g, const chmy_field_t* ckpt, int nckpt, int stride, int nsteps,
                             const chmy_field_t* lam, const chmy_field_t* grad_logA, const chmy_field_t* B,
                             const chmy_field_t* A, int npow, const double* dts) {
    if (nsteps < 1 || stride < 1) return set_error(CHMY_E_ARG, "nsteps=%d stride=%d", nsteps, stride);
    const int nseg = (nsteps + stride - 1) / stride;
    if (nckpt != nseg) return set_error(CHMY_E_ARG, "nckpt=%d, need ceil(nsteps/stride)=%d", nckpt, nseg);
    if (!dts) return set_error(CHMY_E_ARG, "dts is NULL");
    CHMY_TRY(check_grid(g));
    CHMY_TRY(sia_check_states(g, ckpt, nckpt, "ckpt"));
    CHMY_TRY(sia_check(g, &ckpt[0], B, A, npow));
    CHMY_TRY(check_center(g, lam, "lam_a", CHMY_F64));
    if (A) CHMY_TRY(check_center(g, grad_logA, "grad_logA", CHMY_F64));
    return 0;
}

// The reverse sweep on the stream: seg(i) gives segment state buffer i
// (0 <= i < 2 (stride - 1)) by value; with dbuf (2 stride Center fields, or
// NULL) the recompute steps also store D of the state they start from, and
// the adjoint step at that state reads it instead of evaluating it (every
// state of a segment but its last).  Returns the slot that holds dJ/dH_0
// (0 = lam_a, 1 = lam_b).
template <class SegF>
static int sia_reverse_sweep(const chmy_grid_t* g, const chmy_field_t* ckpt, int stride, int nsteps, SegF seg,
                             const chmy_field_t* lam_a, const chmy_field_t* lam_b, const chmy_field_t* grad_logA,
                             const chmy_field_t* B, const chmy_field_t* A, const SiaPar& p, const double* dts,
                             hipStream_t st, const chmy_field_t* dbuf = nullptr) {
    const int nseg = (nsteps + stride - 1) / stride;
    const int64_t nx = g->n[0], ny = g->n[1];
    // state q of segment s: q = 0 its checkpoint, q >= 1 seg((s % 2)(stride - 1) + q - 1)
    auto state = [&](int sg, int q) -> chmy_field_t {
        return q == 0 ? ckpt[sg] : seg((sg % 2) * (stride - 1) + q - 1);
    };
    // D of state q of segment s: dbuf[(s % 2) stride + q]
    auto dfield = [&](int sg, int q) -> DF<double> { return view<double>(dbuf[(sg % 2) * stride + q]); };
    auto len = [&](int sg) { return std::min(stride, nsteps - sg * stride); };
    // recompute the last segment on its own
    for (int q = 1; q < len(nseg - 1); ++q) {
        const chmy_field_t s0 = state(nseg - 1, q - 1), s1 = state(nseg - 1, q);
        SiaStep<double> f = sia_stepper(g, &s0, &s1, B, A, p);
        if (dbuf) {
            f.wd = 1;
            f.Dout = dfield(nseg - 1, q - 1);
        }
        launch_steps(st, f, &dts[(nseg - 1) * stride + q - 1], 1, nx, ny);
    }
    int slot = 0;   // lam_in of the next adjoint step: 0 = lam_a, 1 = lam_b
    for (int sg = nseg - 1; sg >= 0; --sg) {
        const int L = len(sg), Lp = sg > 0 ? len(sg - 1) : 0;
        for (int r = 0; r < std::max(L, Lp - 1);) {
            // the recompute of segment sg - 1 (state r -> r + 1) rides along with
            // adjoint step q = L - 1 - r of segment sg, two of each to a launch
            // where the second step's D is stored
            const int na = r >= L ? 0 : dbuf && r + 2 <= L ? 2 : 1, take = std::max(na, 1);
            const int nf = std::max(0, std::min(take, Lp - 1 - r));
            SiaStep<double> f{};
            SiaMid mid{};
            SiaDts fd{};
            fd.n = nf;
            if (nf > 0) {
                const chmy_field_t s0 = state(sg - 1, r), s1 = state(sg - 1, r + nf);
                f = sia_stepper(g, &s0, &s1, B, A, p);
                for (int k = 0; k < nf; ++k) fd.dt[k] = dts[(sg - 1) * stride + r + k];
                if (dbuf) {
                    f.wd = 1;
                    f.Dout = dfield(sg - 1, r);
                }
                if (nf == 2) {
                    mid.H = view<double>(state(sg - 1, r + 1));
                    mid.D = dfield(sg - 1, r + 1);
                }
            }
            if (na == 0) {
                launch_steps(st, f, fd.dt, 1, nx, ny);
                r += 1;
                continue;
            }
            const int q = L - 1 - r;
            const chmy_field_t* li = slot ? lam_b : lam_a;
            const chmy_field_t* lo = slot ? lam_a : lam_b;
            const chmy_field_t sq = state(sg, q);
            SiaAdj<double> a = sia_adjointer(g, &sq, li, lo, A ? grad_logA : nullptr, B, A, p,
                                             dts[sg * stride + q]);
            if (dbuf && q + 1 < L) {   // stored by the recompute step q -> q + 1
                a.rd = 1;
                a.Din = dfield(sg, q);
            }
            a.n = na;
            if (na == 2) {
                a.H2 = view<double>(state(sg, q - 1));
                a.D2 = dfield(sg, q - 1);
                a.dt2 = dts[sg * stride + q - 1];
            }
            launch_adj(st, a, f, mid, fd, nx, ny);
            slot ^= 1;
            r += na;
        }
    }
    return slot;
}

// Device scratch of chmy_sia_reverse_noalloc: the segment states and the
// second adjoint buffer in one file-scope array, which each GPU holds until
// the process ends.  48 MiB covers 512 x 512 cells (516 x 516 Center storage,
// 2.13 MB a field) at 10 steps per checkpoint: 2 x 9 segment states + 1.
// In host code `scratch` is not a device address: its address on a device
// comes from hipGetSymbolAddress with that device current.
constexpr size_t kSiaScratchBytes = size_t(48) << 20;
static __device__ __align__(256) double scratch[kSiaScratchBytes / sizeof(double)];

static std::mutex g_scratch_mu;
static void* g_scratch_dev[64] = {nullptr};   // scratch's address on each device

__global__ void __launch_bounds__(256) sia_fill_zero(double* p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0.0;
}

}  // namespace chmy

// Resolves scratch's address on the current device (chmy_init calls it; the
// no-allocation entry point calls it on its first use on a device).
int chmy::sia_scratch_ptr(void** p) {
    int dev = 0;
    CHMY_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return set_error(CHMY_E_ARG, "device index %d", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void* q = nullptr;
        const hipError_t e = hipGetSymbolAddress(&q, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !q)
            return set_error(CHMY_E_NODEV, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
        g_scratch_dev[dev] = q;
    }
    if (p) *p = g_scratch_dev[dev];
    return 0;
}

namespace chmy {

// Device memory for the D fields of chmy_sia_reverse: one buffer per device,
// grown on demand and kept until the process ends (calls on one device that
// overlap race, as with any shared workspace).
static std::mutex g_dcache_mu;
static void* g_dcache[64] = {nullptr};
static size_t g_dcache_sz[64] = {0};

static int sia_dcache(size_t bytes, void** p) {
    int dev = 0;
    CHMY_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return set_error(CHMY_E_ARG, "device index %d", dev);
    std::lock_guard<std::mutex> lk(g_dcache_mu);
    if (g_dcache_sz[dev] < bytes) {
        if (g_dcache[dev]) CHMY_HIP(hipFree(g_dcache[dev]));
        g_dcache[dev] = nullptr;
        g_dcache_sz[dev] = 0;
        CHMY_HIP(hipMalloc(&g_dcache[dev], bytes));
        g_dcache_sz[dev] = bytes;
    }
    *p = g_dcache[dev];
    return 0;
}

static dim3 sia_blk() { return dim3(64, 4, 1); }
static dim3 sia_grid(int64_t nx, int64_t ny) {
    return dim3((unsigned)((nx + 1 + 63) / 64), (unsigned)((ny + 1 + 3) / 4), 1);
}

}  // namespace chmy

using namespace chmy;

extern "C" {

int chmy_sia_flux(const chmy_grid_t* g, const chmy_field_t* q, const chmy_field_t* H, const chmy_field_t* B,
                  const chmy_field_t* A, double As, int npow, void* stream) {
    CHMY_TRY(sia_check(g, H, B, A, npow));
    CHMY_TRY(check_vector(g, q, "q", CHMY_F64));
    SiaPar p{As, npow, 0, 0, 0, 0};
    SiaF<double> s = make_sia<double>(g, H, B, A, p);
    hipLaunchKernelGGL(sia_flux_kernel<double>, sia_grid(g->n[0], g->n[1]), sia_blk(), 0, (hipStream_t)stream, s,
                       view<double>(q[0]), view<double>(q[1]), g->n[0], g->n[1]);
    CHMY_HIP(hipGetLastError());
    return 0;
}

int chmy_sia_update(const chmy_grid_t* g, const chmy_field_t* H, const chmy_field_t* H_out, const chmy_field_t* q,
                    const chmy_field_t* B, double mb_a, double mb_b, double mb_c, double dt, void* stream) {
    CHMY_TRY(sia_check(g, H, B, nullptr, 1));
    CHMY_TRY(check_center(g, H_out, "H_out", CHMY_F64));
    CHMY_TRY(check_vector(g, q, "q", CHMY_F64));
    SiaPar p{0, 1, mb_a, mb_b, mb_c, dt};
    SiaF<double> s = make_sia<double>(g, H, B, nullptr, p);
    hipLaunchKernelGGL(sia_update_kernel<double>, sia_grid(g->n[0], g->n[1]), sia_blk(), 0, (hipStream_t)stream, s,
                       view<double>(q[0]), view<double>(q[1]), view<double>(*H_out), g->n[0], g->n[1], dt);
    CHMY_HIP(hipGetLastError());
    return 0;
}

int chmy_sia_diffusivity(const chmy_grid_t* g, const chmy_field_t* D, const chmy_field_t* H, const chmy_field_t* B,
                         const chmy_field_t* A, double As, int npow, void* stream) {
    CHMY_TRY(sia_check(g, H, B, A, npow));
    CHMY_TRY(check_center(g, D, "D", CHMY_F64));
    SiaPar p{As, npow, 0, 0, 0, 0};
    SiaF<double> s = make_sia<double>(g, H, B, A, p);
    hipLaunchKernelGGL(sia_d_kernel<double>, sia_grid(g->n[0], g->n[1]), sia_blk(), 0, (hipStream_t)stream, s,
                       view<double>(*D), g->n[0], g->n[1]);
    CHMY_HIP(hipGetLastError());
    return 0;
}

int chmy_sia_step(const chmy_grid_t* g, const chmy_field_t* H, const chmy_field_t* H_out, const chmy_field_t* B,
                  const chmy_field_t* A, double As, int npow, double mb_a, double mb_b, double mb_c, double dt,
                  void* stream) {
    CHMY_TRY(sia_check(g, H, B, A, npow));
    CHMY_TRY(check_center(g, H_out, "H_out", CHMY_F64));
    if (H_out->data == H->data) return set_error(CHMY_E_ARG, "chmy_sia_step needs distinct H and H_out");
    SiaPar p{As, npow, mb_a, mb_b, mb_c, dt};
    SiaF<double> s = make_sia<double>(g, H, B, A, p);
    hipLaunchKernelGGL(sia_step_kernel<double>, sia_grid(g->n[0], g->n[1]), sia_blk(), 0, (hipStream_t)stream, s,
                       view<double>(*H_out), g->n[0], g->n[1], dt);
    CHMY_HIP(hipGetLastError());
    return 0;
}

int chmy_sia_step_adjoint(const chmy_grid_t* g, const chmy_field_t* H, const chmy_field_t* lam_in,
                          const chmy_field_t* lam_out, const chmy_field_t* grad_logA, const chmy_field_t* B,
                          const chmy_field_t* A, double As, int npow, double mb_a, double mb_b, double mb_c,
                          double dt, const chmy_field_t* work, void* stream) {
    CHMY_TRY(sia_check(g, H, B, A, npow));
    CHMY_TRY(check_center(g, lam_in, "lam_in", CHMY_F64));
    CHMY_TRY(check_center(g, lam_out, "lam_out", CHMY_F64));
    if (lam_in->data == lam_out->data) return set_error(CHMY_E_ARG, "lam_in and lam_out must differ");
    if (A) CHMY_TRY(check_center(g, grad_logA, "grad_logA", CHMY_F64));
    SiaPar p{As, npow, mb_a, mb_b, mb_c, dt};
    if (!work) {   // one tiled pass
        SiaAdj<double> a = sia_adjointer(g, H, lam_in, lam_out, A ? grad_logA : nullptr, B, A, p, dt);
        launch_adj((hipStream_t)stream, a, SiaStep<double>{}, SiaMid{}, SiaDts{}, g->n[0], g->n[1]);
        CHMY_HIP(hipGetLastError());
        return 0;
    }
    const int vx[3] = {1, 0, 0}, vy[3] = {0, 1, 0};
    CHMY_TRY(check_center(g, &work[0], "work.mu", CHMY_F64));
    CHMY_TRY(check_field(g, &work[1], "work.Dvx", vx, CHMY_F64));
    CHMY_TRY(check_field(g, &work[2], "work.gdx", vx, CHMY_F64));
    CHMY_TRY(check_field(g, &work[3], "work.Dvy", vy, CHMY_F64));
    CHMY_TRY(check_field(g, &work[4], "work.gdy", vy, CHMY_F64));
    for (int q = 5; q < 8; ++q) CHMY_TRY(check_center(g, &work[q], "work", CHMY_F64));
    SiaF<double> s = make_sia<double>(g, H, B, A, p);
    SiaW<double> w{view<double>(work[0]), view<double>(work[1]), view<double>(work[2]), view<double>(work[3]),
                   view<double>(work[4]), view<double>(work[5]), view<double>(work[6]), view<double>(work[7])};
    hipStream_t st = (hipStream_t)stream;
    const int64_t nx = g->n[0], ny = g->n[1];
    const DF<double> gA = A ? view<double>(*grad_logA) : view<double>(*lam_out);
    hipLaunchKernelGGL(sia_adj1<double>, sia_grid(nx, ny), sia_blk(), 0, st, s, view<double>(*lam_in), w, nx, ny, dt);
    hipLaunchKernelGGL(sia_adj2<double>, sia_grid(nx, ny), sia_blk(), 0, st, s, w, nx, ny, dt);
    hipLaunchKernelGGL(sia_adj3<double>, sia_grid(nx, ny), sia_blk(), 0, st, s, w, gA, nx, ny);
    hipLaunchKernelGGL(sia_adj4<double>, sia_grid(nx, ny), sia_blk(), 0, st, w, nx, ny);
    hipLaunchKernelGGL(sia_adj5<double>, sia_grid(nx, ny), sia_blk(), 0, st, s, w, view<double>(*lam_out), nx, ny, dt);
    CHMY_HIP(hipGetLastError());
    return 0;
}

int chmy_sia_run(const chmy_grid_t* g, const chmy_field_t* states, int nstates, const chmy_field_t* B,
                 const chmy_field_t* A, double As, int npow, double mb_a, double mb_b, double mb_c,
                 const double* dts, void* stream) {
    if (nstates < 1) return set_error(CHMY_E_ARG, "nstates=%d < 1", nstates);
    CHMY_TRY(check_grid(g));
    CHMY_TRY(sia_check_states(g, states, nstates, "states"));
    CHMY_TRY(sia_check(g, &states[0], B, A, npow));
    if (nstates > 1 && !dts) return set_error(CHMY_E_ARG, "dts is NULL");
    for (int q = 0; q + 1 < nstates; ++q)
        if (states[q].data == states[q + 1].data)
            return set_error(CHMY_E_ARG, "states[%d] and states[%d] share storage", q, q + 1);
    const SiaPar p{As, npow, mb_a, mb_b, mb_c, 0.0};
    hipStream_t st = (hipStream_t)stream;
    int ntx;
    const int longest = sia_regions(g->n[0], g->n[1], 2 * kSiaMax, 2 * kSiaMax, kNWF * kRF2, &ntx) <= cu_count() ? kSiaMax
                                                                                                               : kSiaMany;
    for (int q = 0; q + 1 < nstates;) {
        const int n = sia_run_length(states, nstates, q, longest);
        const SiaStep<double> f = sia_stepper(g, &states[q], &states[q + n], B, A, p);
        launch_steps(st, f, dts + q, n, g->n[0], g->n[1]);
        q += n;
    }
    CHMY_HIP(hipGetLastError());
    return 0;
}

// One launch per step: the step with the Δt of its state's max(D), then the new
// state's max(D); no host wait until the caller reads the Δt.  The host-side rule took three launches, a
// copy and a wait per step (57 us a step at 250x230; now 11).
int chmy_sia_run_adaptive(const chmy_grid_t* g, const chmy_field_t* states, int nstates, const chmy_field_t* B,
                          const chmy_field_t* A, double As, int npow, double mb_a, double mb_b, double mb_c, double h2,
                          double dt_max, const chmy_field_t* D, double* work_dev, void* stream) {
    if (nstates < 1) return set_error(CHMY_E_ARG, "nstates=%d < 1", nstates);
    CHMY_TRY(check_grid(g));
    CHMY_TRY(sia_check_states(g, states, nstates, "states"));
    CHMY_TRY(sia_check(g, &states[0], B, A, npow));
    CHMY_TRY(check_center(g, D, "D", CHMY_F64));
    if (nstates > 1 && !work_dev) return set_error(CHMY_E_ARG, "work_dev is NULL");
    for (int q = 0; q + 1 < nstates; ++q)
        if (states[q].data == states[q + 1].data)
            return set_error(CHMY_E_ARG, "states[%d] and states[%d] share storage", q, q + 1);
    for (int q = 0; q < nstates; ++q)
        if (states[q].data == D->data) return set_error(CHMY_E_ARG, "D shares storage with states[%d]", q);
    if (nstates == 1) return 0;
    const SiaPar p{As, npow, mb_a, mb_b, mb_c, 0.0};
    hipStream_t st = (hipStream_t)stream;
    const int64_t nx = g->n[0], ny = g->n[1];
    const int n = nstates - 1;
    unsigned long long* dmax = reinterpret_cast<unsigned long long*>(work_dev + n);
    hipLaunchKernelGGL(sia_fill_zero, dim3((unsigned)std::min((n + 255) / 256, 64)), dim3(256), 0, st, work_dev + n,
                       (int64_t)n);
    const dim3 grd((unsigned)((nx + 63) / 64), (unsigned)((ny + 3) / 4), 1);
    for (int q = 0; q < n; ++q) {
        SiaStep<double> f = sia_stepper(g, &states[q], &states[q + 1], B, A, p);
        f.Dout = view<double>(*D);
        if (q == 0) {   // the first state's D and maximum
            if (npow == 3)
                hipLaunchKernelGGL((sia_d_max_kernel<double, 3>), grd, sia_blk(), 0, st, f.s, f.Dout, nx, ny, dmax);
            else
                hipLaunchKernelGGL((sia_d_max_kernel<double, 0>), grd, sia_blk(), 0, st, f.s, f.Dout, nx, ny, dmax);
        }
        const bool last = q + 1 == n;
        f.wd = last;   // D keeps the last evaluated state's, as the rule leaves it
        const SiaRule r{dmax + q, last ? nullptr : dmax + q + 1, h2, dt_max, work_dev + q};
        if (last) launch_rule<false>(st, f, r, nx, ny);
        else launch_rule<true>(st, f, r, nx, ny);
    }
    CHMY_HIP(hipGetLastError());
    return 0;
}

int chmy_sia_reverse(const chmy_grid_t* g, const chmy_field_t* ckpt, int nckpt, int stride, int nsteps,
                     const chmy_field_t* seg, const chmy_field_t* lam_a, const chmy_field_t* lam_b,
                     const chmy_field_t* grad_logA, const chmy_field_t* B, const chmy_field_t* A, double As, int npow,
                     double mb_a, double mb_b, double mb_c, const double* dts, int* lam_slot, void* stream) {
    CHMY_TRY(sia_reverse_check(g, ckpt, nckpt, stride, nsteps, lam_a, grad_logA, B, A, npow, dts));
    if (!lam_slot) return set_error(CHMY_E_ARG, "lam_slot is NULL");
    if (stride > 1) CHMY_TRY(sia_check_states(g, seg, 2 * (stride - 1), "seg"));
    CHMY_TRY(check_center(g, lam_b, "lam_b", CHMY_F64));
    if (lam_a->data == lam_b->data) return set_error(CHMY_E_ARG, "lam_a and lam_b must differ");
    const SiaPar p{As, npow, mb_a, mb_b, mb_c, 0.0};
    // D of the segments' states (2 stride Center fields) in library-held device
    // memory, so that the adjoint steps read what the recompute steps evaluated
    std::vector<chmy_field_t> dbuf;
    if (stride > 1) {
        const size_t fbytes = (size_t)(pad_of(*lam_a, 0) * pad_of(*lam_a, 1)) * sizeof(double);
        const size_t fstride = (fbytes + 255) / 256 * 256;
        char* base = nullptr;
        CHMY_TRY(sia_dcache(2 * (size_t)stride * fstride, reinterpret_cast<void**>(&base)));
        for (int i = 0; i < 2 * stride; ++i) {
            chmy_field_t f = *lam_a;
            f.data = base + (size_t)i * fstride;
            dbuf.push_back(f);
        }
    }
    *lam_slot = sia_reverse_sweep(g, ckpt, stride, nsteps, [&](int i) { return seg[i]; }, lam_a, lam_b, grad_logA,
                                  B, A, p, dts, (hipStream_t)stream, dbuf.empty() ? nullptr : dbuf.data());
    CHMY_HIP(hipGetLastError());
    return 0;
}

int chmy_sia_reverse_noalloc(const chmy_grid_t* g, const chmy_field_t* ckpt, int nckpt, int stride, int nsteps,
                             const chmy_field_t* lam, const chmy_field_t* grad_logA, const chmy_field_t* B,
                             const chmy_field_t* A, double As, int npow, double mb_a, double mb_b, double mb_c,
                             const double* dts, void* stream) {
    CHMY_TRY(sia_reverse_check(g, ckpt, nckpt, stride, nsteps, lam, grad_logA, B, A, npow, dts));
    // 2 (stride - 1) segment states and the second adjoint buffer, one Center
    // storage each, every one starting on a 256 B boundary
    const int nbuf = 2 * (stride - 1) + 1;
    const size_t fbytes = (size_t)(pad_of(*lam, 0) * pad_of(*lam, 1)) * sizeof(double);
    const size_t fstride = (fbytes + 255) / 256 * 256;
    if ((size_t)nbuf > kSiaScratchBytes / fstride)
        return set_error(CHMY_E_SIZE,
                         "chmy_sia_reverse_noalloc: %d Center fields of %zu bytes (stride %d) exceed its %zu-byte "
                         "device scratch; use chmy_sia_reverse with caller-allocated seg and lam_b",
                         nbuf, fstride, stride, kSiaScratchBytes);
    char* base = nullptr;
    CHMY_TRY(sia_scratch_ptr(reinterpret_cast<void**>(&base)));
    hipStream_t st = (hipStream_t)stream;
    // the caller-allocated workspace of chmy_sia_reverse starts at zero; so
    // does this one, whatever the previous call on this device left in it
    const int64_t nz = (int64_t)(nbuf * fstride / sizeof(double));
    hipLaunchKernelGGL(sia_fill_zero, dim3((unsigned)std::min<int64_t>((nz + 255) / 256, 2048)), dim3(256), 0, st,
                       reinterpret_cast<double*>(base), nz);
    auto buf = [&](int i) {
        chmy_field_t f = *lam;
        f.data = base + (size_t)i * fstride;
        return f;
    };
    const chmy_field_t lam_b = buf(nbuf - 1);
    const SiaPar p{As, npow, mb_a, mb_b, mb_c, 0.0};
    const int slot = sia_reverse_sweep(g, ckpt, stride, nsteps, buf, lam, &lam_b, grad_logA, B, A, p, dts, st);
    if (slot == 1) CHMY_HIP(hipMemcpyAsync(lam->data, lam_b.data, fbytes, hipMemcpyDeviceToDevice, st));
    CHMY_HIP(hipGetLastError());
    return 0;
}

}  // extern "C"
