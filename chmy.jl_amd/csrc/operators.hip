// GridOperators over a box (chmy_op, chmy_op_masked): left/right, δ, ∂, ∂²,
// ∂k∂, lerp, hlerp, divg, lapl, divg_grad, vmag; plain and masked; uniform
// and FunctionAxis grids.
//
// Each operator is a functor that holds, per source field, the view and the
// element offsets of its knots, formed on the host from the field's location
// and strides; the operator, the number of dims, the number of interpolated
// dims, the mask and the axis kind are template parameters.  So the device
// code is the loads, the arithmetic and one store: no location is looked up
// per point, and no array is indexed at run time (with one kernel switching
// on the operator, the knots and the kernel's own arguments lived in scratch
// memory, 224-368 B a lane, and that traffic was the time).
//
// One kernel walks the box for all of them: a block is 256 consecutive points
// of a plane, counted along x and on into the next row, and marches up to 4
// planes in z, so that an operator's z neighbour is still in L1 or L2; blocks
// are remapped so that each XCD gets a contiguous run and the rows that y
// neighbours share stay in its L2.  With one wave per 64 columns instead, a
// row of 193 points took 4 waves, the last with one lane (1.33 times the
// instructions).  The result is stored past the caches (non-temporal): no
// point of it is read again.  Bound by HBM (∂, divg, lerp, vmag), by loads
// served from L2 (lapl, divg_grad: 7 and 21 loads a point) and by division
// (hlerp: 9 at an edge).
// Measured, FP64 191x175x167, fields not in the caches, us a launch, 64 x 4
// blocks -> flat -> and non-temporal (the bytes at 4.94 TB/s): ∂ 24 -> 20 -> 20
// (18), lerp 33 -> 27 -> 27 (18), divg 48 -> 42 -> 39 (36), vmag 36 -> 31 ->
// 29 (36), lapl 34 -> 29 -> 28 (18), hlerp 53 -> 37 -> 36 (18); masked ∂ 39 ->
// 32 -> 31 (27), divg 91 -> 83 -> 68 (63), divg_grad 107 -> 85 -> 85 (63).
// Chunks of 2 and 8 planes: divg_grad 84 and 93, ∂ 22 and 22.
#include "common.hpp"

namespace chmy {

// ------------------------------------------------------------------ knots
// Point index, for the rows of a FunctionAxis table.
struct Pt {
    int64_t i[3];
};
__device__ __forceinline__ Pt moved(Pt p, int d, int64_t s) {
    if (d == 0) p.i[0] += s;
    else if (d == 1) p.i[1] += s;
    else p.i[2] += s;
    return p;
}

// il/ir of an operator on a field at its own location along D
// (GridOperators.jl:23-36): offsets of the left and right knots, of the
// mask's at the same points, and iΔ along D at the source's location
// (partial_derivatives.jl:5; on a FunctionAxis read at the output index).
template <class T>
struct Axis1 {
    const T* f;
    const T* w;              // the mask component at f's location (masked forms)
    int64_t fy, fz, wy, wz;  // strides
    int64_t l, r, wl, wr;    // knot offsets
    T isp;
    AxisT ax;
    int32_t D, row;
};

template <class T>
__device__ __forceinline__ int64_t at_f(const Axis1<T>& a, const Pt& p) { return p.i[0] + p.i[1] * a.fy + p.i[2] * a.fz; }
template <class T>
__device__ __forceinline__ int64_t at_w(const Axis1<T>& a, const Pt& p) { return p.i[0] + p.i[1] * a.wy + p.i[2] * a.wz; }

template <class T, bool NU>
__device__ __forceinline__ T isp1(const Axis1<T>& a, const Pt& p) {
    if (!NU || !a.ax.p) return a.isp;
    return T(a.ax.at(a.row, a.D == 0 ? p.i[0] : a.D == 1 ? p.i[1] : p.i[2]));
}
// masked left/right read f[Il]·ω[Il] (masked_operators.jl:11-19)
template <class T, bool M>
__device__ __forceinline__ T left1(const Axis1<T>& a, int64_t o, int64_t ow) {
    const T v = a.f[o + a.l];
    return M ? v * a.w[ow + a.wl] : v;
}
template <class T, bool M>
__device__ __forceinline__ T right1(const Axis1<T>& a, int64_t o, int64_t ow) {
    const T v = a.f[o + a.r];
    return M ? v * a.w[ow + a.wr] : v;
}
template <class T, bool M, bool NU>
__device__ __forceinline__ T dd1(const Axis1<T>& a, const Pt& p) {
    const int64_t o = at_f(a, p), ow = M ? at_w(a, p) : 0;
    return (right1<T, M>(a, o, ow) - left1<T, M>(a, o, ow)) * isp1<T, NU>(a, p);
}

// lerp/hlerp (interpolation.jl:14-101): the 2^m knots over the dims whose
// location differs, reduced with fma(t, b - a, a) (harmonic: of the
// inverses), first differing dim innermost.  t is 0.5; Center -> Vertex on a
// FunctionAxis reads the axis's weight at the output index (:28-29).
template <class T>
struct Itp {
    const T* f;
    int64_t fy, fz;
    int64_t lo[3], hi[3];   // knot offsets of the q-th differing dim
    AxisT ax[3];            // table of that dim when its weight is not 0.5, else p == nullptr
    int32_t dim[3], m;
};

template <class T, int M, bool NU, bool HARM>
__device__ __forceinline__ T itp_m(const Itp<T>& a, const Pt& p) {
    const T* f = a.f + (p.i[0] + p.i[1] * a.fy + p.i[2] * a.fz);
    T v[1 << M];
#pragma unroll
    for (int q = 0; q < (1 << M); ++q) {
        int64_t o = 0;
#pragma unroll
        for (int b = 0; b < M; ++b) o += (q >> b) & 1 ? a.hi[b] : a.lo[b];
        v[q] = f[o];
    }
#pragma unroll
    for (int b = 0; b < M; ++b) {
        T t = T(0.5);
        if (NU && a.ax[b].p) {
            const int64_t i = a.dim[b] == 0 ? p.i[0] : a.dim[b] == 1 ? p.i[1] : p.i[2];
            t = T(a.ax[b].at(CHMY_AX_WCV, i));
        }
#pragma unroll
        for (int q = 0; q < (1 << (M - b - 1)); ++q) {
            const T x = v[2 * q], y = v[2 * q + 1];
            v[q] = HARM ? T(1) / fma(t, T(1) / y - T(1) / x, T(1) / x) : fma(t, y - x, x);
        }
    }
    return v[0];
}
// the coefficient of ∂k∂ at a knot, over as many dims as its location differs in
template <class T, bool NU>
__device__ __forceinline__ T coef(const Itp<T>& a, const Pt& p) {
    switch (a.m) {   // uniform
        case 0: return itp_m<T, 0, NU, false>(a, p);
        case 1: return itp_m<T, 1, NU, false>(a, p);
        case 2: return itp_m<T, 2, NU, false>(a, p);
        default: return itp_m<T, 3, NU, false>(a, p);
    }
}

// ------------------------------------------------------------------ operators
template <class T, bool M>
struct OpLeft {
    Axis1<T> a;
    __device__ T operator()(const Pt& p) const { return left1<T, M>(a, at_f(a, p), M ? at_w(a, p) : 0); }
};
template <class T, bool M>
struct OpRight {
    Axis1<T> a;
    __device__ T operator()(const Pt& p) const { return right1<T, M>(a, at_f(a, p), M ? at_w(a, p) : 0); }
};
template <class T, bool M>
struct OpDelta {
    Axis1<T> a;
    __device__ T operator()(const Pt& p) const {
        const int64_t o = at_f(a, p), ow = M ? at_w(a, p) : 0;
        return right1<T, M>(a, o, ow) - left1<T, M>(a, o, ow);
    }
};
template <class T, bool M, bool NU>
struct OpPartial {
    Axis1<T> a;
    __device__ T operator()(const Pt& p) const { return dd1<T, M, NU>(a, p); }
};
template <class T, int ND, bool M, bool NU>
struct OpDivg {
    Axis1<T> a[ND];
    __device__ T operator()(const Pt& p) const {
        T v = dd1<T, M, NU>(a[0], p);
#pragma unroll
        for (int d = 1; d < ND; ++d) v = v + dd1<T, M, NU>(a[d], p);
        return v;
    }
};
// The second differences read f·ω at I and at I ± e_D only, whichever
// location f has: the flipped location's knots are (I, I+e) for a Center dim
// and (I-e, I) for a Vertex dim, and δ at them spans (I-1, I) and (I, I+1) in
// both.  So the point's own value is loaded once for all dims.
template <class T>
struct Src2 {
    const T *f, *w;
    int64_t fy, fz, wy, wz;
};
template <class T>
struct Axis2 {
    int64_t st, sw;       // strides of f and ω along the dim
    int64_t pl, pr;       // index of the left and right flipped knots, relative to I
    T isp;
    AxisT ax;
    int32_t D, row;
};
template <class T, bool NU>
__device__ __forceinline__ T isp2(const Axis2<T>& a, const Pt& p, int64_t shift) {
    if (!NU || !a.ax.p) return a.isp;
    const int64_t i = a.D == 0 ? p.i[0] : a.D == 1 ? p.i[1] : p.i[2];
    return T(a.ax.at(a.row, i + shift));
}
template <class T, bool M>
struct Pt2 {              // the point's addresses and value of f·ω
    const T *f, *w;
    T c;
    __device__ __forceinline__ Pt2(const Src2<T>& s, const Pt& p)
        : f(s.f + (p.i[0] + p.i[1] * s.fy + p.i[2] * s.fz)), w(M ? s.w + (p.i[0] + p.i[1] * s.wy + p.i[2] * s.wz) : f) {
        c = M ? f[0] * w[0] : f[0];
    }
    __device__ __forceinline__ T at(int64_t o, int64_t ow) const { return M ? f[o] * w[ow] : f[o]; }
};

// Σ_D ∂²_D over the given dims (ND = 1: ∂² along one dim)
template <class T, int ND, bool M, bool NU>
struct OpLapl {
    Src2<T> s;
    Axis2<T> a[ND];
    __device__ T operator()(const Pt& p) const {
        const Pt2<T, M> q(s, p);
        T v = T(0);
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            const Axis2<T>& x = a[d];
            const T t = ((q.at(x.st, x.sw) - q.c) * isp2<T, NU>(x, p, x.pr) -
                         (q.c - q.at(-x.st, -x.sw)) * isp2<T, NU>(x, p, x.pl)) * isp2<T, NU>(x, p, 0);
            v = d == 0 ? t : v + t;
        }
        return v;
    }
};
// Σ_D ∂k∂_D (ND = 1: one dim); the coefficient is never masked.  CC: f and k
// are Center along every dim taken, so k at the left and right knots is
// lerped from k at (I-e, I) and (I, I+e), and k at I is loaded once.
template <class T, int ND, bool M, bool NU, bool CC>
struct OpDkd {
    Src2<T> s;
    Axis2<T> a[ND];
    Itp<T> k[ND];
    __device__ T operator()(const Pt& p) const {
        const Pt2<T, M> q(s, p);
        const T* kp = CC ? k[0].f + (p.i[0] + p.i[1] * k[0].fy + p.i[2] * k[0].fz) : nullptr;
        const T kc = CC ? kp[0] : T(0);
        T v = T(0);
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            const Axis2<T>& x = a[d];
            T kr, kl;
            if constexpr (CC) {
                const int64_t st = k[d].lo[0];   // -stride of k
                T tr = T(0.5), tl = T(0.5);
                if (NU && x.ax.p) {
                    const int64_t i = x.D == 0 ? p.i[0] : x.D == 1 ? p.i[1] : p.i[2];
                    tr = T(x.ax.at(CHMY_AX_WCV, i + 1));
                    tl = T(x.ax.at(CHMY_AX_WCV, i));
                }
                const T km = kp[st];
                kr = fma(tr, kp[-st] - kc, kc);
                kl = fma(tl, kc - km, km);
            } else {
                kr = coef<T, NU>(k[d], moved(p, x.D, x.pr));
                kl = coef<T, NU>(k[d], moved(p, x.D, x.pl));
            }
            const T t = (kr * ((q.at(x.st, x.sw) - q.c) * isp2<T, NU>(x, p, x.pr)) -
                         kl * ((q.c - q.at(-x.st, -x.sw)) * isp2<T, NU>(x, p, x.pl))) * isp2<T, NU>(x, p, 0);
            v = d == 0 ? t : v + t;
        }
        return v;
    }
};
template <class T, int NI, bool NU, bool HARM>
struct OpItp {
    Itp<T> a;
    __device__ T operator()(const Pt& p) const { return itp_m<T, NI, NU, HARM>(a, p); }
};
// vmag: V_D is Vertex along D only, so each component interpolates one dim
// with weight 0.5 on any axis
template <class T, int ND>
struct OpVmag {
    Itp<T> a[ND];
    __device__ T operator()(const Pt& p) const {
        const T x = itp_m<T, 1, false, false>(a[0], p);
        T acc = x * x;
#pragma unroll
        for (int d = 1; d < ND; ++d) {
            const T y = itp_m<T, 1, false, false>(a[d], p);
            acc = acc + y * y;
        }
        return sqrt(acc);
    }
};

// ------------------------------------------------------------------ kernel
constexpr int kOpB = 256, kOpZ = 4;

template <class T, class Op>
__global__ void __launch_bounds__(kOpB) op_kernel(Box3 b, DF<T> dst, Op op, int nbx, int kchunk) {
    const int t = xcd_remap(line_id(), line_ids());   // past the last tile: bz past the last chunk
    const int bx = t % nbx, bz = t / nbx;
    int64_t a, c;
    plane_index((int64_t)bx * kOpB + threadIdx.x, b.len[0], b.len[1], a, c);
    if (c >= b.len[1]) return;
    const int64_t e0 = (int64_t)bz * kchunk, e1 = e0 + kchunk < b.len[2] ? e0 + kchunk : b.len[2];
    for (int64_t e = e0; e < e1; ++e) {
        const Pt p{{b.lo[0] + a, b.lo[1] + c, b.lo[2] + e}};
        __builtin_nontemporal_store(op(p), &dst(p.i[0], p.i[1], p.i[2]));
    }
}

// ------------------------------------------------------------------ host side
template <class T>
static Axis1<T> axis1(const chmy_grid_t* g, const chmy_field_t& f, const chmy_field_t* w, int D) {
    Axis1<T> a;
    const DF<T> v = view<T>(f), m = w ? view<T>(*w) : v;
    const int64_t st = D == 0 ? 1 : D == 1 ? v.sy : v.sz, sw = D == 0 ? 1 : D == 1 ? m.sy : m.sz;
    const int vertex = f.loc[D];
    a.f = v.p;
    a.w = m.p;
    a.fy = v.sy;
    a.fz = v.sz;
    a.wy = m.sy;
    a.wz = m.sz;
    const int l = vertex ? 0 : -1;   // Center: knots (I-e, I); Vertex: (I, I+e)
    a.l = l * st;
    a.r = (l + 1) * st;
    a.wl = l * sw;
    a.wr = (l + 1) * sw;
    a.isp = T(g->inv_spacing[D]);
    a.ax = axes_of(g).a[D];
    a.D = D;
    a.row = vertex ? CHMY_AX_IDV : CHMY_AX_IDC;
    return a;
}

template <class T>
static Src2<T> src2(const chmy_field_t& f, const chmy_field_t* w) {
    const DF<T> v = view<T>(f), m = w ? view<T>(*w) : v;
    return Src2<T>{v.p, m.p, v.sy, v.sz, m.sy, m.sz};
}
template <class T>
static Axis2<T> axis2(const chmy_grid_t* g, const chmy_field_t& f, const chmy_field_t* w, int D) {
    const DF<T> v = view<T>(f), m = w ? view<T>(*w) : v;
    Axis2<T> a;
    a.st = D == 0 ? 1 : D == 1 ? v.sy : v.sz;
    a.sw = D == 0 ? 1 : D == 1 ? m.sy : m.sz;
    a.pl = f.loc[D] ? -1 : 0;   // the flipped knots: Center (I, I+e); Vertex (I-e, I)
    a.pr = a.pl + 1;
    a.isp = T(g->inv_spacing[D]);
    a.ax = axes_of(g).a[D];
    a.D = D;
    a.row = f.loc[D] ? CHMY_AX_IDV : CHMY_AX_IDC;
    return a;
}

template <class T>
static Itp<T> itp(const chmy_grid_t* g, const chmy_field_t& f, const int32_t* to) {
    Itp<T> a;
    std::memset(&a, 0, sizeof a);
    const DF<T> v = view<T>(f);
    a.f = v.p;
    a.fy = v.sy;
    a.fz = v.sz;
    const int64_t st[3] = {1, v.sy, v.sz};
    const Axes3 ax = axes_of(g);
    for (int d = 0; d < g->nd; ++d) {
        if (f.loc[d] == to[d]) continue;
        const int l = f.loc[d] ? 0 : -1;   // Center -> Vertex (I-e, I); Vertex -> Center (I, I+e)
        a.lo[a.m] = l * st[d];
        a.hi[a.m] = (l + 1) * st[d];
        a.dim[a.m] = d;
        if (!f.loc[d]) a.ax[a.m] = ax.a[d];
        ++a.m;
    }
    return a;
}

struct OpCall {
    int op;
    const chmy_grid_t* g;
    Box3 b;
    const chmy_field_t *dst, *src, *masks, *k;
    int dim;
    hipStream_t s;
};

// z planes a block walks: 4 where that leaves 16 blocks a CU, fewer on
// smaller boxes, where blocks in flight count for more than reuse.
template <class T, class Op>
static int op_launch(const OpCall& c, const Op& op) {
    const int64_t nbx = (c.b.len[0] * c.b.len[1] + kOpB - 1) / kOpB;
    int kz = kOpZ;
    while (kz > 1 && nbx * ((c.b.len[2] + kz - 1) / kz) < 4096) kz /= 2;
    dim3 grd;
    CHMY_TRY(line_grid(nbx * ((c.b.len[2] + kz - 1) / kz), kOpB, &grd));
    hipLaunchKernelGGL((op_kernel<T, Op>), grd, dim3(kOpB, 1, 1), 0, c.s, c.b, view<T>(*c.dst), op, (int)nbx, kz);
    CHMY_HIP(hipGetLastError());
    return 0;
}

template <class T, bool M, bool NU>
static int op_dispatch(const OpCall& c) {
    const chmy_grid_t* g = c.g;
    auto ax = [&](int q, int D) { return axis1<T>(g, c.src[q], M ? &c.masks[q] : nullptr, D); };
    const chmy_field_t* w0 = M ? &c.masks[0] : nullptr;
    auto lapl = [&](auto nd) -> int {
        constexpr int ND = decltype(nd)::value;
        OpLapl<T, ND, M, NU> op;
        op.s = src2<T>(c.src[0], w0);
        for (int d = 0; d < ND; ++d) op.a[d] = axis2<T>(g, c.src[0], w0, c.op == CHMY_OP_D2 ? c.dim : d);
        return op_launch<T>(c, op);
    };
    auto divg = [&](auto nd) -> int {
        constexpr int ND = decltype(nd)::value;
        OpDivg<T, ND, M, NU> op;
        for (int d = 0; d < ND; ++d) op.a[d] = ax(d, d);
        return op_launch<T>(c, op);
    };
    auto dkd = [&](auto nd) -> int {
        constexpr int ND = decltype(nd)::value;
        auto with = [&](auto cc) -> int {
            OpDkd<T, ND, M, NU, decltype(cc)::value> op;
            op.s = src2<T>(c.src[0], w0);
            for (int d = 0; d < ND; ++d) {
                const int D = c.op == CHMY_OP_DKD ? c.dim : d;
                int32_t to[3] = {c.src[0].loc[0], c.src[0].loc[1], c.src[0].loc[2]};
                to[D] = 1 - to[D];
                op.a[d] = axis2<T>(g, c.src[0], w0, D);
                op.k[d] = itp<T>(g, *c.k, to);
            }
            return op_launch<T>(c, op);
        };
        // Center f and k: the one-load form of the coefficient
        bool cc = true;
        for (int d = 0; d < g->nd; ++d) cc = cc && !c.src[0].loc[d] && !c.k->loc[d];
        return cc ? with(std::true_type{}) : with(std::false_type{});
    };
    using N1 = std::integral_constant<int, 1>;
    using N2 = std::integral_constant<int, 2>;
    using N3 = std::integral_constant<int, 3>;
    auto by_nd = [&](auto f) -> int { return g->nd == 1 ? f(N1{}) : g->nd == 2 ? f(N2{}) : f(N3{}); };
    switch (c.op) {
        case CHMY_OP_LEFT: return op_launch<T>(c, OpLeft<T, M>{ax(0, c.dim)});
        case CHMY_OP_RIGHT: return op_launch<T>(c, OpRight<T, M>{ax(0, c.dim)});
        case CHMY_OP_DELTA: return op_launch<T>(c, OpDelta<T, M>{ax(0, c.dim)});
        case CHMY_OP_PARTIAL: return op_launch<T>(c, OpPartial<T, M, NU>{ax(0, c.dim)});
        case CHMY_OP_D2: return lapl(N1{});
        case CHMY_OP_DKD: return dkd(N1{});
        case CHMY_OP_DIVG: return by_nd(divg);
        case CHMY_OP_LAPL: return by_nd(lapl);
        case CHMY_OP_DIVG_GRAD: return by_nd(dkd);
        default: break;
    }
    if constexpr (!M) {   // lerp, hlerp and vmag have no masked form
        const Itp<T> a = itp<T>(g, c.src[0], c.dst->loc);
        auto harm = [&](auto h) -> int {
            constexpr bool H = decltype(h)::value;
            switch (a.m) {
                case 0: return op_launch<T>(c, OpItp<T, 0, NU, H>{a});
                case 1: return op_launch<T>(c, OpItp<T, 1, NU, H>{a});
                case 2: return op_launch<T>(c, OpItp<T, 2, NU, H>{a});
                default: return op_launch<T>(c, OpItp<T, 3, NU, H>{a});
            }
        };
        auto vmag = [&](auto nd) -> int {
            constexpr int ND = decltype(nd)::value;
            const int32_t to[3] = {0, 0, 0};
            OpVmag<T, ND> op;
            for (int d = 0; d < ND; ++d) op.a[d] = itp<T>(g, c.src[d], to);
            return op_launch<T>(c, op);
        };
        switch (c.op) {
            case CHMY_OP_LERP: return harm(std::false_type{});
            case CHMY_OP_HLERP: return harm(std::true_type{});
            case CHMY_OP_VMAG: return by_nd(vmag);
            default: break;
        }
    }
    return set_error(CHMY_E_ARG, "unknown operator %d", c.op);
}

}  // namespace chmy

using namespace chmy;

extern "C" {

int chmy_op(int op, const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* dst, int nsrc,
            const chmy_field_t* src, int dim, void* stream) {
    if (op != CHMY_OP_PARTIAL && op != CHMY_OP_LERP && op != CHMY_OP_DIVG && op != CHMY_OP_VMAG &&
        op != CHMY_OP_LEFT && op != CHMY_OP_RIGHT) {
        CHMY_TRY(check_grid_any(g));
        if (!nonuniform(g)) return set_error(CHMY_E_ARG, "unknown operator %d", op);
    }
    return chmy_op_masked(op, g, box, dst, nsrc, src, nullptr, nullptr, dim, stream);
}

int chmy_op_masked(int op, const chmy_grid_t* g, const chmy_box_t* box, const chmy_field_t* dst, int nsrc,
                   const chmy_field_t* src, const chmy_field_t* masks, const chmy_field_t* k, int dim, void* stream) {
    CHMY_TRY(check_grid_any(g));
    chmy_box_t bx;
    CHMY_TRY(check_box(g, box, &bx));
    CHMY_TRY(check_field(g, dst, "dst", nullptr, -1));
    const int dt = dst->dtype;
    const bool vec = op == CHMY_OP_DIVG || op == CHMY_OP_VMAG;
    const bool per_dim = op == CHMY_OP_PARTIAL || op == CHMY_OP_DELTA || op == CHMY_OP_LEFT || op == CHMY_OP_RIGHT ||
                         op == CHMY_OP_D2 || op == CHMY_OP_DKD;
    const bool known = per_dim || vec || op == CHMY_OP_LERP || op == CHMY_OP_HLERP || op == CHMY_OP_LAPL ||
                       op == CHMY_OP_DIVG_GRAD;
    if (!known) return set_error(CHMY_E_ARG, "unknown operator %d", op);
    const bool maskable = op != CHMY_OP_LERP && op != CHMY_OP_HLERP && op != CHMY_OP_VMAG;
    const bool needs_k = op == CHMY_OP_DKD || op == CHMY_OP_DIVG_GRAD;
    if (vec && nsrc != g->nd) return set_error(CHMY_E_ARG, "divg/vmag need nd source fields");
    if (!vec && nsrc != 1) return set_error(CHMY_E_ARG, "operator needs one source field");
    if (!src) return set_error(CHMY_E_ARG, "src is NULL");
    if (per_dim && (dim < 0 || dim >= g->nd)) return set_error(CHMY_E_ARG, "dim %d out of range", dim);
    if (masks && !maskable) return set_error(CHMY_E_ARG, "operator %d has no masked form", op);
    if (needs_k != (k != nullptr))
        return set_error(CHMY_E_ARG, needs_k ? "k is NULL" : "k is given to an operator without a coefficient");
    for (int q = 0; q < nsrc; ++q) {
        const int* want = nullptr;
        int loc[3];
        if (vec) {
            for (int d = 0; d < 3; ++d) loc[d] = d == q ? 1 : 0;
            want = loc;
        }
        CHMY_TRY(check_field(g, &src[q], "src", want, dt));
        // the mask component read with src[q] is the one at src[q]'s location
        if (masks) CHMY_TRY(check_field(g, &masks[q], "mask", src[q].loc, dt));
    }
    if (k) CHMY_TRY(check_field(g, k, "k", nullptr, dt));
    Box3 b = box3(bx, g->nd);
    if (no_work(b)) return 0;
    const OpCall c{op, g, b, dst, src, masks, k, dim, (hipStream_t)stream};
    auto run = [&](auto tag) -> int {
        using T = decltype(tag);
        if (nonuniform(g)) return masks ? op_dispatch<T, true, true>(c) : op_dispatch<T, false, true>(c);
        return masks ? op_dispatch<T, true, false>(c) : op_dispatch<T, false, false>(c);
    };
    return dt == CHMY_F64 ? run(double{}) : run(float{});
}

}  // extern "C"
