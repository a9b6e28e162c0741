// Shared device/host helpers of the gfx950 stencil library.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>

#include "../../include/chmy_mi355x.h"

namespace chmy {

// ------------------------------------------------------------------ errors
int set_error(int code, const char* fmt, ...);
int hip_status(hipError_t e, const char* what);

#define CHMY_HIP(call)                                   \
    do {                                                 \
        hipError_t e_ = (call);                          \
        if (e_ != hipSuccess) return hip_status(e_, #call); \
    } while (0)
#define CHMY_TRY(expr)               \
    do {                             \
        int rc_ = (expr);            \
        if (rc_ != 0) return rc_;    \
    } while (0)

// ------------------------------------------------------------------ bfloat16
// Storage type of bf16 fields (the forcing of FP32 correction sweeps):
// f32 -> bf16 rounds to nearest even, bf16 -> f32 is exact.
struct bf16s {
    uint16_t u;
};
__device__ __forceinline__ float bf16_to_f32(uint16_t u) { return __uint_as_float((uint32_t)u << 16); }
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
    uint32_t x = __float_as_uint(f);
    if ((x & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((x >> 16) | 0x40u);   // NaN stays a quiet NaN
    x += 0x7fffu + ((x >> 16) & 1u);
    return (uint16_t)(x >> 16);
}
// value conversions used by kernels that write in a chosen precision
template <class TO, class T>
__device__ __forceinline__ void put(TO& dst, T v) { dst = TO(v); }
template <class T>
__device__ __forceinline__ void put(bf16s& dst, T v) { dst.u = f32_to_bf16(float(v)); }
template <class T>
__device__ __forceinline__ double as_double(T v) { return (double)v; }
__device__ __forceinline__ double as_double(bf16s v) { return (double)bf16_to_f32(v.u); }

// ------------------------------------------------------------------ views
// Device view of a Field: p points at logical index (0,0,0), so logical I is
// p[i + j*sy + k*sz] (storage offset I + 2H - 1 per dim, field.jl:18).
template <class T>
struct DF {
    T* p;
    int64_t sy, sz;
    __device__ __forceinline__ T& operator()(int64_t i, int64_t j, int64_t k) const {
        return p[i + j * sy + k * sz];
    }
    __device__ __forceinline__ T& at(int64_t o) const { return p[o]; }
};

inline int64_t pad_of(const chmy_field_t& f, int d) { return f.n[d] + 4 * (int64_t)f.halo[d]; }

template <class T>
DF<T> view(const chmy_field_t& f) {
    DF<T> v;
    int64_t s1 = pad_of(f, 0);
    int64_t s2 = f.nd >= 2 ? s1 * pad_of(f, 1) : 0;
    v.sy = f.nd >= 2 ? s1 : 0;
    v.sz = f.nd >= 3 ? s2 : 0;
    int64_t off = (2 * (int64_t)f.halo[0] - 1);
    if (f.nd >= 2) off += (2 * (int64_t)f.halo[1] - 1) * v.sy;
    if (f.nd >= 3) off += (2 * (int64_t)f.halo[2] - 1) * v.sz;
    v.p = static_cast<T*>(f.data) + off;
    return v;
}

// ------------------------------------------------------------------ validation
// All descriptors are checked on the host before any launch, so that every
// access a kernel makes (box ± 1 in each dim) lies inside the field storage.
// check_grid accepts uniform grids only; check_grid_any also grids with a
// FunctionAxis (the operators, bc! and set!).
int check_grid(const chmy_grid_t* g);
int check_grid_any(const chmy_grid_t* g);

// A FunctionAxis metric table on the device (chmy_grid_t.axis): entry (row, i)
// at p[row * rs + i + CHMY_AXIS_PAD]; p == nullptr on a uniform dim.
struct AxisT {
    const double* p;
    int64_t rs;
    __host__ __device__ __forceinline__ double at(int row, int64_t i) const { return p[row * rs + i + CHMY_AXIS_PAD]; }
};
struct Axes3 {
    AxisT a[3];
};
inline Axes3 axes_of(const chmy_grid_t* g) {
    Axes3 r;
    for (int d = 0; d < 3; ++d) {
        r.a[d].p = d < g->nd ? g->axis[d] : nullptr;
        r.a[d].rs = d < g->nd ? g->n[d] + 2 + 2 * CHMY_AXIS_PAD : 0;
    }
    return r;
}
inline bool nonuniform(const chmy_grid_t* g) {
    for (int d = 0; d < g->nd; ++d)
        if (g->axis[d]) return true;
    return false;
}
int check_box(const chmy_grid_t* g, const chmy_box_t* b, chmy_box_t* out);
// loc: expected location per dim (-1 = any); dtype: expected (-1 = any).
// bf16 storage is rejected unless allow_bf16 (only the forcing of FP32
// correction sweeps and the reductions read it).
int check_field(const chmy_grid_t* g, const chmy_field_t* f, const char* name, const int* loc, int dtype,
                bool allow_bf16 = false);
int check_center(const chmy_grid_t* g, const chmy_field_t* f, const char* name, int dtype, bool allow_bf16 = false);
int check_vector(const chmy_grid_t* g, const chmy_field_t* V, const char* name, int dtype, bool allow_bf16 = false);
int check_tensor(const chmy_grid_t* g, const chmy_field_t* tau, const char* name, int dtype, bool allow_bf16 = false);
void tensor_loc(int nd, int c, int* loc);
// Address on the current device of the SIA reverse sweep's file-scope device
// scratch (sia.hip), resolved once per device; p may be NULL.
int sia_scratch_ptr(void** p);

struct Box3 {
    int64_t lo[3];
    int64_t len[3];
    int32_t spread = 0;   // flat_at's order of blocks
};
inline Box3 box3(const chmy_box_t& b, int nd) {
    Box3 r;
    for (int d = 0; d < 3; ++d) {
        r.lo[d] = d < nd ? b.lo[d] : 0;
        r.len[d] = d < nd ? b.len[d] : 1;
    }
    return r;
}

// A box with no points: the entry point launches nothing and returns 0 (a
// KernelAbstractions launch over an empty worksize does no work).
inline bool no_work(const Box3& b) { return b.len[0] <= 0 || b.len[1] <= 0 || b.len[2] <= 0; }

// A line of nb blocks as a grid.  HIP launches fewer than 2^32 work-items in a
// grid dimension, so a line of that many or more is folded into rows of
// kLineRow blocks (whole rounds of the 8 XCDs); the ids that the last row has
// too many name no tile, and their blocks do nothing.
constexpr int64_t kLineRow = int64_t(1) << 21, kLineMost = int64_t(1) << 30;
inline int line_grid(int64_t nb, int threads, dim3* grd) {
    if (nb > kLineMost) return set_error(CHMY_E_SIZE, "box too large: %lld blocks", (long long)nb);
    const bool one = nb * threads <= INT64_C(0xffffffff);
    *grd = one ? dim3((unsigned)nb, 1, 1) : dim3((unsigned)kLineRow, (unsigned)((nb + kLineRow - 1) / kLineRow), 1);
    return 0;
}
// (rows have kLineRow blocks whenever there are several: no read of the grid's size)
__device__ __forceinline__ uint32_t line_id() { return blockIdx.y * (uint32_t)kLineRow + blockIdx.x; }
__device__ __forceinline__ uint32_t line_ids() { return gridDim.y * gridDim.x; }

// The q-th point of a plane of rows of len0 points, counted along the rows:
// column a, row c (c >= len1 past the plane).  The 32-bit division unless the
// plane has 2^32 points (uniform).
__host__ __device__ __forceinline__ void plane_index(int64_t q, int64_t len0, int64_t len1, int64_t& a, int64_t& c) {
    if (len0 * len1 + 0x10000 < 0x100000000ll) {
        const uint32_t r = (uint32_t)q, n = (uint32_t)len0, k = r / n;
        c = k;
        a = r - k * n;
    } else {
        c = q / len0;
        a = q - c * len0;
    }
}

// Per-point kernels: blocks of 256 consecutive points of a plane (counted along
// x and on into the next row, so no lane idles at a row's end), plane after
// plane.  Which XCD takes which blocks (ids congruent mod 8 go to one XCD)
// depends on what the launch's arrays hold together:
//  - up to the 256 MB cache behind the L2s, each XCD one contiguous run: the
//    planes and rows that a neighbour's point shares are found in its L2;
//  - beyond, runs of 32 blocks, so that the XCDs work side by side.  Eight runs
//    far apart are eight places of HBM read and written at once, and a plane of
//    every array is more than an L2 holds anyway.
// Measured, FP64, us, 64 x 4 grid -> one run an XCD -> runs of 32: diffusion
// step (5 arrays) 159x143x127 33 -> 23 -> 28, 207x191x175 (277 MB) 81 -> 93 -> 67,
// 250^3 216 -> 237 -> 186, 400^3 842 -> 980 -> 750; compute_q (4 arrays)
// 207x191x175 (221 MB) 59 -> 38 -> 42, 400^3 605 -> 690 -> 628; update_C
// 1000x1000x60 497 -> 548 -> 487.  Runs of 16, 64 and 128: within 3% of 32,
// 128 up to 9% slower (one step of chmy_diffusion_iterate, 250^3).
constexpr int kFlat = 256;
constexpr uint32_t kFlatRun = 32;
constexpr int64_t kFlatCache = int64_t(256) << 20;
// point_bytes: what a point of the box keeps in the caches, over all arrays
// that the launch reads or writes (not those stored past them).
inline int flat_grid(Box3& b, int64_t point_bytes, dim3* grd) {
    int64_t plane, nb;
    if (__builtin_mul_overflow(b.len[0], b.len[1], &plane) ||
        __builtin_mul_overflow(plane / kFlat + (plane % kFlat != 0), b.len[2], &nb))
        nb = INT64_MAX;
    CHMY_TRY(line_grid(nb, kFlat, grd));
    b.spread = nb * kFlat > kFlatCache / point_bytes;
    return 0;
}
// Lane `lane` of block `bid` of nb: its point, or false.
__host__ __device__ __forceinline__ bool flat_at(const Box3& b, uint32_t bid, uint32_t nb, uint32_t lane, int64_t& i,
                                                 int64_t& j, int64_t& k) {
    const uint32_t per = (uint32_t)((b.len[0] * b.len[1] + kFlat - 1) / kFlat);
    uint32_t id = bid;   // the blocks past the last whole round of the XCDs keep theirs
    if (b.spread) {
        constexpr uint32_t G = 8 * kFlatRun;
        if ((bid | (G - 1)) < nb) id = bid / G * G + bid % 8 * kFlatRun + bid % G / 8;
    } else if (bid < nb / 8 * 8) {
        id = bid % 8 * (nb / 8) + bid / 8;
    }
    const uint32_t e = id / per;
    int64_t a, c;
    plane_index((int64_t)(id - e * per) * kFlat + lane, b.len[0], b.len[1], a, c);
    i = b.lo[0] + a;
    j = b.lo[1] + c;
    k = b.lo[2] + e;
    return c < b.len[1] && e < b.len[2];
}
__device__ __forceinline__ bool flat_point(const Box3& b, int64_t& i, int64_t& j, int64_t& k) {
    return flat_at(b, line_id(), line_ids(), threadIdx.x, i, j, k);
}

// Compute units of the current device, read once per device (api.hip).
int cu_count();

// Block id -> tile, so that the blocks an XCD receives (ids congruent mod 8,
// dispatched round-robin over the 8 XCDs) form one contiguous run of tiles and
// share halo rows in that XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int nb) {
    const int per = nb / 8;
    if (bid >= 8 * per) return bid;
    return (bid % 8) * per + bid / 8;
}

// Julia max/min against zero for floats (NaN propagates, max(-0.0, 0.0) = 0.0).
template <class T>
__device__ __forceinline__ T jmax0(T x) { return x != x ? x : (x > T(0) ? x : T(0)); }
template <class T>
__device__ __forceinline__ T jmin0(T x) { return x != x ? x : (x <= T(0) ? x : T(0)); }
template <class T>
__device__ __forceinline__ T jmax(T a, T b) {
    if (a != a) return a;
    if (b != b) return b;
    return a > b ? a : b;
}
template <class T>
__device__ __forceinline__ T visc_ve(T eta, T G, T dt) { return T(1) / (T(1) / eta + T(1) / (G * dt)); }

}  // namespace chmy
