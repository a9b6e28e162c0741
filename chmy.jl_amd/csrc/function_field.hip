// Device evaluation of set!(f, grid, fun) and of FunctionField values
// (src/Fields/field.jl:119-142, src/Fields/function_field.jl:51-61).
//
// The reference compiles the user's function into its own GPU kernel.  Here
// the host turns the function into a point program: a straight-line list of
// operations in SSA form (operation q writes register q and reads only
// registers < q).  One kernel runs the program at every point of a box of the
// destination's logical indices and stores the last register, converted to
// the field's dtype.  Program, constants and source descriptors travel in the
// kernel argument, so every wave runs the same operation at the same time
// (the switch is uniform) and the only per-lane state is the register file.
//
// Before the launch the host lowers the program (plan_program):
//  - constants become operands instead of operations;
//  - a wave owns 64 x points of one row and marches a chunk of the last dim;
//    operations that do not depend on the last dim (the x and y parts of a
//    distance, say) run once per chunk, the others at every plane;
//  - registers are assigned to slots by their last use.  8 or 16 slots are a
//    vector in VGPRs addressed by a uniform index, so no register lives in
//    memory (with one f64 per SSA register the file was 1 KB a lane of
//    scratch, and that traffic was the time);
//  - each operation runs on 4 (8 slots) or 2 (16 slots) planes at once, which
//    shares its decoding and gives independent work to overlap.
// Programs that need more slots keep the file in LDS; those, and the ones that
// call sin, cos, tanh or pow, whose code is large, run one plane at a time (two
// runs of a line: 141 VGPRs).
//  - sums, products, negations and squares become FMA with constant operands
//    that give the same bits, so most operations take the first branch.
// Bound by instruction issue: per operation and 4 planes about 65 vector and 83
// scalar instructions (counters), most of them operand moves and decoding.
// Measured, one launch, us, before -> now (register file in scratch, one
// point a lane): 160x144x127 FP64, 42 operations with two exp 295 -> 64, 27
// operations with one exp 188 -> 46, 11 operations with two loads 96 -> 32;
// 255^3: 1503 -> 212, 980 -> 154, 689 -> 148.
//
// Continuous functions read the coordinates at the destination's location,
// coord(grid, loc, I...) with the fma forms of uniform_axis.jl:18-19;
// discrete ones read logical indices and other fields at constant index
// offsets (the reference's discrete FunctionFields index their parameter
// fields at ix, iy, iz, e.g. examples/sia.jl:38-53).  Arithmetic is IEEE f64
// operation by operation with no contraction (FMA is an operation of its own),
// so programs made of + - * / sqrt, comparisons and ifelse give the bits of
// the same expressions evaluated on the host; exp, log, sin, cos, tanh and
// pow are the device math library's and may differ from the host's by an ulp.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"

namespace chmy {

constexpr int kPMaxOps = 128;
constexpr int kPMaxConst = 64;
constexpr int kPMaxSrc = 8;

struct PSrc {
    const char* p;       // logical index (0,0,0)
    int64_t st[3];       // element strides
    int32_t dtype;
    int32_t esize;
};

// A lowered operation: operands are slots (>= 0) or constants (-1 - index),
// or the fields of the leaf operations as in chmy_pop_t.
struct PIns {
    int16_t op, dst;
    int32_t a, b, c;
};

struct PProg {
    int32_t npro, n;     // operations [0, npro) once per chunk, [npro, n) per plane
    int32_t out;         // the stored value's operand
    int32_t m;           // the marched dim (nd - 1; in 1D x, 64 points at a time)
    double o[3], h[3], ih[3];
    Axes3 ax;            // FunctionAxis tables (p == nullptr: uniform dim)
    PIns op[kPMaxOps + 1];   // (one past the end is read ahead)
    double k[kPMaxConst + 3];   // the program's, then 1, -1 and -0.0
    PSrc src[kPMaxSrc];
};

__host__ __device__ __forceinline__ int off8(int32_t packed, int d) { return (int)(int8_t)((packed >> (8 * d)) & 0xff); }

// Julia's min/max on IEEE floats: NaN wins, -0.0 < 0.0
__device__ __forceinline__ double jl_min(double x, double y) {
    if (x != x || y != y) return x + y;
    return (y < x || (signbit(y) && !signbit(x))) ? y : x;
}
__device__ __forceinline__ double jl_max(double x, double y) {
    if (x != x || y != y) return x + y;
    return (y > x || (!signbit(y) && signbit(x))) ? y : x;
}

// The register file of one plane: a VGPR vector of S slots, or (S = 0) the
// block's LDS, one f64 a lane and slot.
typedef double slots8 __attribute__((ext_vector_type(8)));
typedef double slots16 __attribute__((ext_vector_type(16)));
extern __shared__ double slot_lds[];
template <int S>
struct Slots {
    __device__ __forceinline__ double get(int s) const { return slot_lds[64 * s + threadIdx.x]; }
    __device__ __forceinline__ void set(int s, double x) { slot_lds[64 * s + threadIdx.x] = x; }
};
template <>
struct Slots<8> {
    slots8 v;
    __device__ __forceinline__ double get(int s) const { return v[s]; }
    __device__ __forceinline__ void set(int s, double x) { v[s] = x; }
};
template <>
struct Slots<16> {
    slots16 v;
    __device__ __forceinline__ double get(int s) const { return v[s]; }
    __device__ __forceinline__ void set(int s, double x) { v[s] = x; }
};

// x^n as repeated products, left to right (Julia's literal powers x^2 = x*x,
// x^3 = x*x*x; x^-1 = inv(x), x^-2 = inv(x)^2)
__device__ __forceinline__ double powi(double r, int e) {
    const double x = e < 0 ? 1.0 / r : r;
    const int n = e < 0 ? -e : e;
    double v = n == 0 ? 1.0 : x;
    for (int q = 1; q < n; ++q) v = v * x;
    return v;
}

template <int S, int N, bool HEAVY>
__device__ __forceinline__ void program_run(const PProg& P, int q0, int q1, Slots<S>* r, const int64_t* I,
                                            const int64_t* Im) {
    PIns next = P.op[q0];
    for (int q = q0; q < q1; ++q) {
        const PIns o = next;
        next = P.op[q + 1];   // in flight while this one runs
        double v[N], x[N], y[N], z[N];
        auto get = [&](int s, double* t) {
            if (s >= 0) {
#pragma unroll
                for (int u = 0; u < N; ++u) t[u] = r[u].get(s);
            } else {
                const double k = P.k[-1 - s];
#pragma unroll
                for (int u = 0; u < N; ++u) t[u] = k;
            }
        };
        // index of plane u along dim d
        auto at = [&](int d, int u) -> int64_t {
            return d == P.m ? Im[u] : (d == 0 ? I[0] : d == 1 ? I[1] : I[2]);
        };
#define CHMY_P_EACH(expr)                      \
    do {                                       \
        _Pragma("unroll") for (int u = 0; u < N; ++u) v[u] = (expr); \
    } while (0)
        // the operations that fill most programs first, each one branch away
        if (o.op == CHMY_P_FMA) {
            get(o.a, x);
            get(o.b, y);
            get(o.c, z);
            CHMY_P_EACH(fma(x[u], y[u], z[u]));
        } else if (o.op == CHMY_P_LOAD) {
            const PSrc& s = P.src[o.a];
            const int64_t off = off8(o.b, 0) * s.st[0] + off8(o.b, 1) * s.st[1] + off8(o.b, 2) * s.st[2];
            int64_t w[N];
#pragma unroll
            for (int u = 0; u < N; ++u) w[u] = off + at(0, u) * s.st[0] + at(1, u) * s.st[1] + at(2, u) * s.st[2];
            if (s.dtype == CHMY_F64) CHMY_P_EACH(reinterpret_cast<const double*>(s.p)[w[u]]);
            else if (s.dtype == CHMY_F32) CHMY_P_EACH((double)reinterpret_cast<const float*>(s.p)[w[u]]);
            else CHMY_P_EACH((double)bf16_to_f32(reinterpret_cast<const uint16_t*>(s.p)[w[u]]));
        } else if (o.op == CHMY_P_SELECT) {
            get(o.a, x);
            get(o.b, y);
            get(o.c, z);
            CHMY_P_EACH(x[u] != 0.0 ? y[u] : z[u]);
        } else if (o.op == CHMY_P_LT) {
            get(o.a, x);
            get(o.b, y);
            CHMY_P_EACH(x[u] < y[u] ? 1.0 : 0.0);
        } else if (o.op == CHMY_P_COORD) {
            const AxisT ax = P.ax.a[o.a];
            if (ax.p) {
                CHMY_P_EACH(ax.at(o.b == CHMY_VERTEX ? CHMY_AX_VERTEX : CHMY_AX_CENTER, at(o.a, u) + o.c));
            } else {
                const double h = P.h[o.a], og = P.o[o.a];
                const double o1 = o.b == CHMY_VERTEX ? og : fma(0.5, h, og);
                CHMY_P_EACH(fma((double)(at(o.a, u) + o.c - 1), h, o1));
            }
        } else if (o.op == CHMY_P_EXP) {
            get(o.a, x);
            CHMY_P_EACH(exp(x[u]));
        } else if (o.op < CHMY_P_NEG) {
            const AxisT ax = P.ax.a[o.a];
            if (o.op == CHMY_P_INDEX) CHMY_P_EACH((double)(at(o.a, u) + o.b));
            else if (o.op == CHMY_P_SPACING)
                CHMY_P_EACH(ax.p ? ax.at(o.b == CHMY_VERTEX ? CHMY_AX_DV : CHMY_AX_DC, at(o.a, u) + o.c) : P.h[o.a]);
            else
                CHMY_P_EACH(ax.p ? ax.at(o.b == CHMY_VERTEX ? CHMY_AX_IDV : CHMY_AX_IDC, at(o.a, u) + o.c)
                                 : P.ih[o.a]);
        } else {
            get(o.a, x);
            if (o.op >= CHMY_P_ADD && o.op != CHMY_P_POWI) get(o.b, y);
            switch (o.op) {
                case CHMY_P_ABS: CHMY_P_EACH(fabs(x[u])); break;
                case CHMY_P_SQRT: CHMY_P_EACH(sqrt(x[u])); break;
                case CHMY_P_LOG: CHMY_P_EACH(log(x[u])); break;
                case CHMY_P_FLOOR: CHMY_P_EACH(floor(x[u])); break;
                case CHMY_P_NOT: CHMY_P_EACH(x[u] == 0.0 ? 1.0 : 0.0); break;
                case CHMY_P_DIV: CHMY_P_EACH(x[u] / y[u]); break;
                case CHMY_P_MIN: CHMY_P_EACH(jl_min(x[u], y[u])); break;
                case CHMY_P_MAX: CHMY_P_EACH(jl_max(x[u], y[u])); break;
                case CHMY_P_LE: CHMY_P_EACH(x[u] <= y[u] ? 1.0 : 0.0); break;
                case CHMY_P_EQ: CHMY_P_EACH(x[u] == y[u] ? 1.0 : 0.0); break;
                case CHMY_P_NE: CHMY_P_EACH(x[u] != y[u] ? 1.0 : 0.0); break;
                case CHMY_P_AND: CHMY_P_EACH((x[u] != 0.0 && y[u] != 0.0) ? 1.0 : 0.0); break;
                case CHMY_P_OR: CHMY_P_EACH((x[u] != 0.0 || y[u] != 0.0) ? 1.0 : 0.0); break;
                case CHMY_P_POWI: CHMY_P_EACH(powi(x[u], o.b)); break;
                default:
                    if constexpr (HEAVY) {
                        if (o.op == CHMY_P_SIN) CHMY_P_EACH(sin(x[u]));
                        else if (o.op == CHMY_P_COS) CHMY_P_EACH(cos(x[u]));
                        else if (o.op == CHMY_P_TANH) CHMY_P_EACH(tanh(x[u]));
                        else CHMY_P_EACH(pow(x[u], y[u]));
                    }
                    break;
            }
        }
#undef CHMY_P_EACH
#pragma unroll
        for (int u = 0; u < N; ++u) r[u].set(o.dst, v[u]);
    }
}

// One wave: 64 consecutive points of a plane (of a row where y is marched; in
// 1D, ROW, of the line), a chunk of planes of the marched dim (ROW: of runs of
// 64 points), N at a time.  Lanes and planes past the box evaluate its first or
// last indices and store nothing.  With 64 columns of one row a wave instead,
// 160 points took three waves: us at 160x144x127 FP64 66 -> 53 (42 operations),
// 46 -> 42 (27), 36 -> 29 (11 with loads); all three and their host side at
// 140x187x170 FP32 238 -> 187, 191x187x189 FP64 271 -> 256 (160x144x127 waits
// for the host: 161 both).
template <class T, int S, int N, bool HEAVY, bool ROW>
__global__ void __launch_bounds__(64) program_kernel(const PProg P, DF<T> dst, Box3 b, int nbx, int chunk) {
    const int t = line_id();
    const int bx = ROW ? 0 : t % nbx, bc = ROW ? t : t / nbx;
    const int m = P.m;
    // z marched: 64 consecutive points of a plane, counted along its rows; y
    // marched: of the row
    int64_t i = b.lo[0] + threadIdx.x, j = b.lo[1];
    bool in = true;
    if constexpr (!ROW) {
        plane_index((int64_t)bx * 64 + threadIdx.x, b.len[0], m == 2 ? b.len[1] : 1, i, j);
        in = j < (m == 2 ? b.len[1] : 1);
        i = in ? b.lo[0] + i : b.lo[0];
        j = in ? b.lo[1] + j : b.lo[1];
    }
    const int64_t m0 = (ROW ? 0 : b.lo[m]) + (int64_t)bc * chunk;
    const int64_t hm = ROW ? (b.len[0] + 63) / 64 : b.lo[m] + b.len[m], m1 = m0 + chunk < hm ? m0 + chunk : hm;
    // (a block past the last chunk, m0 >= hm, marches no plane; its part per chunk loads no field)
    const int64_t I[3] = {i, j, b.lo[2]}, last = b.lo[0] + b.len[0] - 1;   // (the line's last point)
    Slots<S> r[N];
    int64_t Im[N];
    // the index along the marched dim at step p of the march
    auto along = [&](int64_t p) -> int64_t {
        if (!ROW) return p < m1 ? p : m1 - 1;
        const int64_t x = i + 64 * p;
        return x < last ? x : last;
    };
#pragma unroll
    for (int u = 0; u < N; ++u) Im[u] = along(m0);
    program_run<S, N, HEAVY>(P, 0, P.npro, r, I, Im);
    for (int64_t p = m0; p < m1; p += N) {
#pragma unroll
        for (int u = 0; u < N; ++u) Im[u] = along(p + u);
        program_run<S, N, HEAVY>(P, P.npro, P.n, r, I, Im);
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const double v = P.out >= 0 ? r[u].get(P.out) : P.k[-1 - P.out];
            if constexpr (ROW) {
                if (p + u < m1 && i + 64 * (p + u) <= last) put(dst(Im[u], 0, 0), v);
            } else {
                if (in && p + u < m1) put(m == 2 ? dst(i, j, p + u) : dst(i, p + u, 0), v);
            }
        }
    }
}

static bool unary(int op) { return op >= CHMY_P_NEG && op <= CHMY_P_NOT; }
static bool binary(int op) { return op >= CHMY_P_ADD && op <= CHMY_P_OR; }

static int check_program(const chmy_grid_t* g, const chmy_pop_t* prog, int nprog, int nconst, const chmy_field_t* srcs,
                         int nsrc, const Box3& b) {
    if (!prog || nprog < 1 || nprog > kPMaxOps)
        return set_error(CHMY_E_SIZE, "point program: %d operations, need 1..%d", nprog, kPMaxOps);
    for (int q = 0; q < nprog; ++q) {
        const chmy_pop_t& o = prog[q];
        auto reg = [&](int r) { return r >= 0 && r < q; };
        bool ok;
        switch (o.op) {
            case CHMY_P_CONST: ok = o.a >= 0 && o.a < nconst; break;
            case CHMY_P_INDEX: ok = o.a >= 0 && o.a < g->nd && o.b >= -64 && o.b <= 64; break;
            case CHMY_P_COORD:
            case CHMY_P_SPACING:
            case CHMY_P_INV_SPACING:
                ok = o.a >= 0 && o.a < g->nd && (o.b == CHMY_CENTER || o.b == CHMY_VERTEX) && o.c >= -64 && o.c <= 64;
                // a FunctionAxis table covers logical -PAD .. n+1+PAD
                if (ok && g->axis[o.a])
                    ok = b.lo[o.a] + o.c >= -CHMY_AXIS_PAD &&
                         b.lo[o.a] + b.len[o.a] - 1 + o.c <= g->n[o.a] + 1 + CHMY_AXIS_PAD;
                break;
            case CHMY_P_LOAD: {
                ok = o.a >= 0 && o.a < nsrc && o.b >= 0 && o.b < (1 << 24);
                if (!ok) break;
                const chmy_field_t& s = srcs[o.a];
                // every point of the box plus the offset stays in the source's storage
                for (int d = 0; d < 3 && ok; ++d) {
                    const int off = off8(o.b, d);
                    if (d >= g->nd) {
                        ok = off == 0;
                        break;
                    }
                    const int64_t H = 2 * (int64_t)s.halo[d];
                    ok = b.lo[d] + off >= 1 - H && b.lo[d] + b.len[d] - 1 + off <= s.n[d] + H;
                }
                if (!ok)
                    return set_error(CHMY_E_BOX, "point program op %d: load of source %d at offset (%d, %d, %d) leaves "
                                     "its storage over the box", q, o.a, off8(o.b, 0), off8(o.b, 1), off8(o.b, 2));
                break;
            }
            case CHMY_P_POWI: ok = reg(o.a) && o.b >= -64 && o.b <= 64; break;
            case CHMY_P_SELECT:
            case CHMY_P_FMA: ok = reg(o.a) && reg(o.b) && reg(o.c); break;
            default:
                if (unary(o.op)) ok = reg(o.a);
                else if (binary(o.op)) ok = reg(o.a) && reg(o.b);
                else ok = false;
        }
        if (!ok) return set_error(CHMY_E_ARG, "point program op %d (code %d, %d, %d, %d) is malformed", q, o.op, o.a, o.b, o.c);
    }
    return 0;
}

static int nargs_of(int op) {
    if (op == CHMY_P_SELECT || op == CHMY_P_FMA) return 3;
    return binary(op) ? 2 : unary(op) || op == CHMY_P_POWI ? 1 : 0;
}

// Lowers a checked program into P (operations, split point, output operand);
// returns the number of slots it needs, and whether it calls sin, cos, tanh
// or pow.  Slots are reused after a register's last use; a value that the
// per-plane part reads from the per-chunk part keeps its slot to the end.
static int plan_program(const chmy_pop_t* prog, int n, PProg* P, bool* heavy) {
    bool plane[kPMaxOps], live[kPMaxOps] = {};
    int last[kPMaxOps];          // position of the last use in the lowered order
    int order[kPMaxOps], no = 0;
    *heavy = false;
    auto arg = [](const chmy_pop_t& o, int k) { return k == 0 ? o.a : k == 1 ? o.b : o.c; };
    live[n - 1] = true;
    for (int q = n - 1; q >= 0; --q)
        for (int k = 0; live[q] && k < nargs_of(prog[q].op); ++k) live[arg(prog[q], k)] = true;
    for (int q = 0; q < n; ++q) {
        const chmy_pop_t& o = prog[q];
        if (o.op == CHMY_P_LOAD) plane[q] = true;
        else if (o.op >= CHMY_P_INDEX && o.op <= CHMY_P_INV_SPACING) plane[q] = o.a == P->m;
        else plane[q] = false;
        for (int k = 0; k < nargs_of(o.op); ++k) plane[q] = plane[q] || plane[arg(o, k)];
    }
    for (int part = 0; part < 2; ++part) {
        if (part == 1) P->npro = no;
        for (int q = 0; q < n; ++q)
            if (live[q] && prog[q].op != CHMY_P_CONST && plane[q] == (part == 1)) order[no++] = q;
    }
    P->n = no;
    for (int q = 0; q < n; ++q) last[q] = -1;
    for (int p = 0; p < no; ++p) {
        const chmy_pop_t& o = prog[order[p]];
        for (int k = 0; k < nargs_of(o.op); ++k) {
            const int r = arg(o, k);
            last[r] = !plane[r] && p >= P->npro ? no : std::max(last[r], p);
        }
    }
    last[n - 1] = no;
    int slot[kPMaxOps], used = 0;
    bool busy[kPMaxOps] = {};
    auto operand = [&](int r) { return prog[r].op == CHMY_P_CONST ? -1 - prog[r].a : slot[r]; };
    for (int p = 0; p < no; ++p) {
        const int q = order[p];
        const chmy_pop_t& o = prog[q];
        const int na = nargs_of(o.op);
        PIns& w = P->op[p];
        w.op = (int16_t)o.op;
        w.a = na > 0 ? operand(o.a) : o.a;
        w.b = na > 1 ? operand(o.b) : o.b;
        w.c = na > 2 ? operand(o.c) : o.c;
        for (int k = 0; k < na; ++k) {
            const int r = arg(o, k);
            if (prog[r].op != CHMY_P_CONST && last[r] == p) busy[slot[r]] = false;
        }
        int s = 0;
        while (busy[s]) ++s;
        busy[s] = true;
        slot[q] = s;
        used = std::max(used, s + 1);
        w.dst = (int16_t)s;
        *heavy = *heavy || o.op == CHMY_P_SIN || o.op == CHMY_P_COS || o.op == CHMY_P_TANH || o.op == CHMY_P_POW;
    }
    P->out = operand(n - 1);
    // the sums, products and negations as the FMA that gives the same bits:
    // a + b = fma(a, 1, b), a - b = fma(b, -1, a), a b = fma(a, b, -0.0),
    // -a = fma(a, -1, -0.0); a > b and a >= b as b < a and b <= a
    const int one = -1 - kPMaxConst, minus = one - 1, nzero = one - 2;
    for (int p = 0; p < no; ++p) {
        PIns& w = P->op[p];
        const int32_t a = w.a, b = w.b;
        auto as_fma = [&w](int32_t x, int32_t y, int32_t z) {
            w.op = CHMY_P_FMA;
            w.a = x;
            w.b = y;
            w.c = z;
        };
        switch (w.op) {
            case CHMY_P_ADD: as_fma(a, one, b); break;
            case CHMY_P_SUB: as_fma(b, minus, a); break;
            case CHMY_P_MUL: as_fma(a, b, nzero); break;
            case CHMY_P_NEG: as_fma(a, minus, nzero); break;
            case CHMY_P_POWI:
                if (b == 2) as_fma(a, a, nzero);
                break;
            case CHMY_P_GT:
            case CHMY_P_GE:
                w.op = w.op == CHMY_P_GT ? CHMY_P_LT : CHMY_P_LE;
                w.a = b;
                w.b = a;
                break;
            default: break;
        }
    }
    P->k[kPMaxConst] = 1.0;
    P->k[kPMaxConst + 1] = -1.0;
    P->k[kPMaxConst + 2] = -0.0;
    return used;
}

template <class T>
static int program_launch(const PProg& P, const chmy_field_t* dst, const Box3& b, int slots, bool heavy,
                          hipStream_t st) {
    const bool row = P.m == 0;
    const int64_t nbx = row ? 1 : (b.len[0] * (P.m == 2 ? b.len[1] : 1) + 63) / 64;
    const int64_t nm = row ? (b.len[0] + 63) / 64 : b.len[P.m];
    const DF<T> d = view<T>(*dst);
    auto go = [&](auto s, auto n, auto h, auto line) -> int {
        constexpr int S = decltype(s)::value, N = decltype(n)::value;
        constexpr bool HEAVY = decltype(h)::value, ROW = decltype(line)::value;
        // planes per wave: fill whole rounds of the waves the chip holds (12 a CU
        // at these kernels' registers); a wave also spends about two planes' time
        // on the per-chunk operations.  160x144x127: 20 planes, one round.  On a
        // line no operation is per chunk, so short chunks that balance: twice the
        // runs that share the decoding (four times: 3-5% more below 10^6 points,
        // whole rounds: 10-60% more at 2 10^6), one run with the file in LDS
        int64_t chunk = S ? 2 * N : 1, best = INT64_MAX;
        const int64_t room = 12 * (int64_t)cu_count();
        for (int64_t c = 4; !ROW && c <= 64; c += 4) {
            const int64_t waves = nbx * ((nm + c - 1) / c), cost = (waves + room - 1) / room * (c + 2);
            if (cost < best) {
                best = cost;
                chunk = c;
            }
        }
        dim3 grd;
        CHMY_TRY(line_grid(nbx * ((nm + chunk - 1) / chunk), 64, &grd));
        const size_t lds = S ? 0 : (size_t)slots * 64 * sizeof(double);
        hipLaunchKernelGGL((program_kernel<T, S, N, HEAVY, ROW>), grd, dim3(64), lds, st, P, d, b, (int)nbx, (int)chunk);
        CHMY_HIP(hipGetLastError());
        return 0;
    };
    auto by_slots = [&](auto line) -> int {
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I4 = std::integral_constant<int, 4>;
        using I8 = std::integral_constant<int, 8>;
        using I16 = std::integral_constant<int, 16>;
        if (slots > 16) return go(I0{}, I1{}, std::true_type{}, line);
        if (heavy) return go(I16{}, std::conditional_t<decltype(line)::value, I2, I1>{}, std::true_type{}, line);
        if (slots > 8) return go(I16{}, I2{}, std::false_type{}, line);
        return go(I8{}, I4{}, std::false_type{}, line);
    };
    return row ? by_slots(std::true_type{}) : by_slots(std::false_type{});
}

}  // namespace chmy

using namespace chmy;

extern "C" {

int chmy_set_program(const chmy_grid_t* g, const chmy_field_t* dst, const chmy_box_t* box, const chmy_pop_t* prog,
                     int nprog, const double* consts, int nconst, const chmy_field_t* srcs, int nsrc, void* stream) {
    CHMY_TRY(check_grid_any(g));
    CHMY_TRY(check_field(g, dst, "dst", nullptr, -1, true));
    if (nconst < 0 || nconst > kPMaxConst || (nconst > 0 && !consts))
        return set_error(CHMY_E_SIZE, "point program: %d constants, at most %d", nconst, kPMaxConst);
    if (nsrc < 0 || nsrc > kPMaxSrc || (nsrc > 0 && !srcs))
        return set_error(CHMY_E_SIZE, "point program: %d source fields, at most %d", nsrc, kPMaxSrc);
    for (int s = 0; s < nsrc; ++s) CHMY_TRY(check_field(g, &srcs[s], "source", nullptr, -1, true));
    // the box: logical indices of dst, default its interior; within its storage
    chmy_box_t bb;
    for (int d = 0; d < 3; ++d) { bb.lo[d] = 1; bb.len[d] = d < g->nd ? dst->n[d] : 1; }
    if (box) bb = *box;
    for (int d = 0; d < g->nd; ++d) {
        const int64_t H = 2 * (int64_t)dst->halo[d];
        if (bb.len[d] < 0 || bb.lo[d] < 1 - H || bb.lo[d] + bb.len[d] - 1 > dst->n[d] + H)
            return set_error(CHMY_E_BOX, "point program: box outside the storage of dst along dim %d", d);
    }
    const Box3 b = box3(bb, g->nd);
    CHMY_TRY(check_program(g, prog, nprog, nconst, srcs, nsrc, b));
    if (b.len[0] == 0 || b.len[1] == 0 || b.len[2] == 0) return 0;
    PProg P;
    std::memset(&P, 0, sizeof P);
    P.m = g->nd - 1;
    for (int d = 0; d < 3; ++d) {
        P.o[d] = d < g->nd ? g->origin[d] : 0.0;
        P.h[d] = d < g->nd ? g->spacing[d] : 0.0;
        P.ih[d] = d < g->nd ? g->inv_spacing[d] : 0.0;
    }
    P.ax = axes_of(g);
    bool heavy;
    const int slots = plan_program(prog, nprog, &P, &heavy);
    if (nconst) std::memcpy(P.k, consts, sizeof(double) * nconst);
    for (int s = 0; s < nsrc; ++s) {
        const chmy_field_t& f = srcs[s];
        const int es = f.dtype == CHMY_F64 ? 8 : f.dtype == CHMY_F32 ? 4 : 2;
        // element strides and the element offset of logical (0,0,0): I + 2H - 1 per dim
        int64_t st[3] = {1, 0, 0}, off = 0;
        for (int d = 0; d < f.nd; ++d) {
            if (d > 0) st[d] = st[d - 1] * pad_of(f, d - 1);
            off += (2 * (int64_t)f.halo[d] - 1) * st[d];
        }
        P.src[s].p = static_cast<const char*>(f.data) + off * es;
        for (int d = 0; d < 3; ++d) P.src[s].st[d] = st[d];
        P.src[s].dtype = f.dtype;
        P.src[s].esize = es;
    }
    hipStream_t st = (hipStream_t)stream;
    if (dst->dtype == CHMY_F64) return program_launch<double>(P, dst, b, slots, heavy, st);
    if (dst->dtype == CHMY_F32) return program_launch<float>(P, dst, b, slots, heavy, st);
    return program_launch<bf16s>(P, dst, b, slots, heavy, st);
}

}  // extern "C"
